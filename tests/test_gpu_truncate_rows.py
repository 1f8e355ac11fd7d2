"""GPU: truncation statistics of rows that start anywhere in a 16-byte line, end inside a tile of the streaming pass
(8192 elements, segments of tiles 0 mod 16, 4 mod 16, 2 mod 4 and the odd ones), or keep their likely tokens where
the pass sees them last; against the fp64 oracle."""
import numpy as np
import pytest
import torch

from oracle import accept as A
from trida_stack_amd import kernels as TK

pytestmark = pytest.mark.gpu

TILE = 8192


def check(x, T, k, p, ban=-1):
    """x: fp32 rows [B, R, V] on the GPU, any strides. The kept set matches but for a boundary within 1e-6 of top_p;
    the normaliser to 1e-6 (the 24-bit exponentials of the histogram)."""
    m, thr, zk, st, _ = (t.cpu().numpy() for t in TK.truncate_stats(x, temperature=T, top_k=k, top_p=p, ban_id=ban,
                                                                    want_passes=True))
    logits = x.cpu().numpy()
    _, info = A.truncated_probs(logits, T, k, p, ban, return_info=True)
    y = logits.copy()
    if ban >= 0:
        y[..., ban] = -np.inf
    y = (y / np.float32(T)).astype(np.float32).astype(np.float64)
    assert (st == 0).all() and (m == y.max(-1).astype(np.float32)).all()
    for at in np.ndindex(m.shape):
        if info.boundary_gap[at] < 1e-6:
            continue
        kept = info.kept[at] & np.isfinite(y[at])
        assert (kept == (np.isfinite(y[at]) & (y[at] >= thr[at]))).all(), (at, kept.sum())
        z = np.exp(y[at][kept] - y[at].max()).sum()
        assert abs(zk[at] / z - 1) < 1e-6, (at, zk[at], z)


@pytest.mark.parametrize("V", [1, 3, 7, 2051, TILE - 1, TILE + 1, 2 * TILE + 6, 5 * TILE - 3, 17 * TILE + 2])
@pytest.mark.parametrize("T,k,p", [(0.7, 0, 0.95), (1.0, 20, 0.9), (1.2, 0, 1.0)])
def test_unaligned_rows(gpu, V, T, k, p):
    g = torch.Generator(device=gpu).manual_seed(V)
    buf = torch.randn(4 * (V + 5), generator=g, device=gpu) * 3
    x = buf[1: 1 + 4 * (V + 1)].view(1, 4, V + 1)[..., :V]  # rows at every offset within a line, for odd V + 1
    check(x, T, k, p, ban=V // 2 if V > 1 else -1)


@pytest.mark.parametrize("T,k,p", [(0.7, 0, 0.95), (0.5, 0, 0.8), (1.2, 0, 0.98), (1.0, 50, 0.95), (1.0, 0, 1.0)])
def test_late_tokens(gpu, T, k, p):
    """Likely tokens in the last segment only, the first one only, a vocabulary sorted by frequency, a row whose
    whole mass is one token, and one with more values in the boundary bin than are ranked against each other."""
    V, g = 20 * TILE + 5, torch.Generator(device=gpu).manual_seed(3)
    x = torch.randn(6, V, generator=g, device=gpu) * 2
    x[0, 19 * TILE: 19 * TILE + 20] += 14 * torch.rand(20, generator=g, device=gpu)
    x[1, 5: 25] += 14 * torch.rand(20, generator=g, device=gpu)
    x[2] = x[2].sort(descending=True).values
    x[3, 3 * TILE + 7] = 25.0
    x[4] = x[4].mul(8).round().div(8)   # massive ties
    x[5] = x[5].mul(0.05)               # a flat row: everything within a few bins
    check(x.view(2, 3, V), T, k, p)


@pytest.mark.parametrize("V", [1, 5, 1027, 4 * TILE + 1, 33 * 4096 + 7])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_draw_unaligned_rows(gpu, V, dtype):
    """The gathered rows, the draws and the probability rows of rows at any offset within a line: exact copies, the
    inverse CDF of the fp64 distribution outside 1e-6 of a step, probabilities to 4e-6 (the rounding of
    an fp32 exponent of up to 24, times log2(e))."""
    g = torch.Generator(device=gpu).manual_seed(V)
    B, R = 2, 3
    src = (torch.randn(B, R, V + 3, generator=g, device=gpu) * 3).to(dtype)[..., 1: 1 + V]
    sel = torch.tensor([[2, 0, 1], [1, 1, 0]], device=gpu)
    out = torch.full((B, R, V + 2), -7.0, device=gpu)
    lf = TK.gather_rows(src, sel, out=out[..., 1: 1 + V])
    assert torch.equal(lf, torch.stack([src[b, sel[b]].float() for b in range(B)]))
    assert (out[..., 0] == -7).all() and (out[..., -1] == -7).all()
    stats = TK.truncate_stats(lf, temperature=0.8, top_k=0, top_p=0.9)[:3]
    u = torch.rand(B * R, generator=g, device=gpu)
    tok = TK.sample_rows(lf, stats, u, temperature=0.8).view(-1).tolist()
    q = torch.full((B, R, V + 2), -7.0, device=gpu)
    rows = torch.arange(R, device=gpu).repeat(B, 1).contiguous()
    TK.truncated_probs_rows(lf, stats, rows, rows, q[..., 1: 1 + V], temperature=0.8)
    y = (lf.cpu() / torch.tensor(0.8)).double().to(gpu)  # the CPU's division rounds correctly
    P = torch.where(y >= stats[1][..., None].double(), torch.exp(y - stats[0][..., None]), torch.zeros_like(y))
    P = P / P.sum(-1, keepdim=True)
    torch.testing.assert_close(q[..., 1: 1 + V].double(), P, rtol=4e-6, atol=0)
    assert (q[..., 0] == -7).all() and (q[..., -1] == -7).all()
    cdf = P.view(B * R, V).cumsum(-1)
    for i in range(B * R):
        lo = cdf[i, tok[i] - 1].item() if tok[i] else 0.0
        assert lo - 1e-6 <= u[i].item() < cdf[i, tok[i]].item() + 1e-6
        assert P.view(B * R, V)[i, tok[i]] > 0


def offset_rows(gpu, V, off):
    """Broad rows, every other one with 20 likely tokens, all shifted by `off` (exactly: multiples of 2^-7 below 2^17)."""
    g = torch.Generator(device=gpu).manual_seed(17)
    x = torch.randn(8, V, generator=g, device=gpu) * 2
    at = torch.randint(0, V, (4, 20), generator=g, device=gpu)
    x[::2].scatter_add_(1, at, torch.rand(4, 20, generator=g, device=gpu) * 8 + 8)
    return x.mul(128).round().div(128) + off


@pytest.mark.parametrize("off", [0.0, 100.0, -1000.0, 1e5])
@pytest.mark.parametrize("T", [1.0, 0.5, 2.0])
def test_offset_untruncated(gpu, T, off):
    """The normaliser does not depend on a shift of the row. y = x / T is exact at these temperatures, so what is left are
    roundings at random signs: the exponents' (2^-24 |d log2(e)| ln 2, |d| <= 8 where the mass is), exp2's and the
    fp32 sums of 16 (2^-24 each), 4e-7 for an entry and less by the root of the 5 or more that carry the mass of the broad
    rows at T = 0.5; the likely tokens' masses are exact to 2^-26."""
    x = offset_rows(gpu, 248320, off)
    m, _, zk, st = TK.truncate_stats(x[None], temperature=T)
    y = (x.double() / T)
    z = torch.exp(y - y.amax(-1, keepdim=True)).sum(-1)
    assert (st == 0).all() and (m[0].double() == y.amax(-1)).all()
    assert ((zk[0] / z - 1).abs() < 2e-7).all(), (zk[0] / z - 1).tolist()


@pytest.mark.parametrize("off", [0.0, 5e4, -8e4, 1e5])
def test_offset_restreamed(gpu, off):
    """Rows whose likely tokens sit in one tile of the last segment, so that the windows of the earlier ones miss the
    boundary and their segments are streamed again, shifted by up to 10^5."""
    g = torch.Generator(device=gpu).manual_seed(5)
    x = torch.randn(8, 30 * TILE, generator=g, device=gpu) * 2
    at = 19 * TILE + torch.randint(0, TILE, (8, 20), generator=g, device=gpu)
    x = (x.scatter_add_(1, at, torch.rand(8, 20, generator=g, device=gpu) * 8 + 4) + off).view(1, 8, -1)
    assert (TK.truncate_stats(x, temperature=1.0, top_p=0.9, want_passes=True)[4] > 4).all()
    check(x, 1.0, 0, 0.9)


@pytest.mark.parametrize("T,k,p", [(1.0, 0, 1.0), (1.0, 0, 0.95), (2.0, 0, 0.9), (0.7, 50, 0.95), (1.0, 4, 1.0)])
def test_far_rows(gpu, T, k, p):
    """Rows masked with the type's lowest value but for 20 tokens that the sample does not see (and one more that it may),
    ties and steps at 10^8, and at T < 1 the whole row at the lowest value (y = -inf: status 2; else all kept)."""
    V, g = 25 * TILE + 3, torch.Generator(device=gpu).manual_seed(9)
    x = torch.full((4, V), torch.finfo(torch.float32).min, device=gpu)
    x[0, 11 * TILE + 1: 11 * TILE + 41: 2] = torch.randn(20, generator=g, device=gpu) * 3
    x[1, 5::512] = torch.randn(V // 512 + (V % 512 > 5), generator=g, device=gpu) * 3
    x[2] = 1e8
    x[2, : V // 3] -= 8.0
    check(x[:3].view(1, 3, V), T, k, p)
    m, thr, zk, st = TK.truncate_stats(x[3].view(1, 1, V), temperature=T, top_k=k, top_p=p)
    assert st.item() == (2 if T < 1 else 0)
    if T >= 1:
        y = x[3, 0] / T
        assert m.item() == y.item() and zk.item() == V and thr.item() in (y.item(), -float("inf"))


@pytest.mark.parametrize("T,p", [(0.7, 0.95), (1.2, 0.98), (1.0, 0.5)])
def test_boundary_ties(gpu, T, p):
    """Widened bf16 rows: the value at the boundary has hundreds of copies; and rows of such values each beside its
    fp32 neighbour (two values of hundreds of copies in a sub-bin)."""
    g = torch.Generator(device=gpu).manual_seed(21)
    x = (torch.randn(4, 30 * TILE + 1, generator=g, device=gpu) * 2).bfloat16().float()
    x[2:] = torch.where(torch.rand(2, x.shape[1], generator=g, device=gpu) < 0.5, x[2:],
                        torch.nextafter(x[2:], torch.full_like(x[2:], 9.0)))
    thr = TK.truncate_stats(x[None], temperature=T, top_p=p)[1][0].cpu()
    y = x.cpu() / torch.tensor(T)
    assert (((y - thr[:, None]).abs() < 2e-6).sum(-1) > 64).all()  # more than a wave ranks
    check(x.view(2, 2, -1), T, 0, p)


@pytest.mark.parametrize("T,p", [(1.0, 0.95), (0.7, 0.8), (1.2, 0.3)])
def test_flat_rows(gpu, T, p):
    """Rows from near-flat to broad: the two bins at the boundary hold from all of the row down to a few thousand values,
    across the collection's 12288, the 8192 that are sorted and the rule that skips the streaming pass."""
    g = torch.Generator(device=gpu).manual_seed(31)
    std = torch.tensor([0.002, 0.05, 0.1, 0.2, 0.25, 0.3, 0.35, 0.4, 0.5, 0.6, 0.8, 1.0], device=gpu) * T
    x = torch.randn(12, 30 * TILE, generator=g, device=gpu) * std[:, None]
    x[1, 2::3] = -float("inf")
    check(x.view(2, 6, -1), T, 0, p)
