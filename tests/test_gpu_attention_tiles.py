"""GPU: canvas attention at the edges of its tiles: query rows around one and two row tiles per wave and the extra
rows of a last tile, keys around a 64-key step, scales of either sign and zero, scores that keep rising (the
running max moves at every step) and rows of very different magnitude in one tile; against the oracle."""
import pytest
import torch

from oracle import attention as A
from trida_stack_amd import kernels as K

pytestmark = pytest.mark.gpu
TOL = 2e-2  # normwise max-abs of bf16 products, as the other attention tests


def rel(a, b):
    a, b = a.float().cpu(), b.float().cpu()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-30))


def check(gpu, B, T, Hq, Hkv, D, prefix, mode, scale=None, shape=lambda q, k, v: (q, k, v), splits=0):
    g = torch.Generator().manual_seed(T * 7 + D + mode)
    L = max(prefix) + T
    q, k, v = shape(torch.randn(B, T, Hq, D, generator=g), torch.randn(B, Hkv, L, D, generator=g),
                    torch.randn(B, Hkv, L, D, generator=g))
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    # the oracle's scale is D^-0.5: the factor beyond it goes into its fp32 queries
    f = 1.0 if scale is None else scale * D ** 0.5
    ref = A.canvas_attention(q.float() * f, k.float(), v.float(), prefix, mode, T // 2)
    kw = {} if scale is None else dict(scale=scale)
    out = K.attn_canvas(q.to(gpu), k.to(gpu), v.to(gpu), torch.tensor(prefix, dtype=torch.int32, device=gpu), mask_mode=mode,
                        n_clean=T // 2, splits=splits, **kw)
    assert rel(out, ref) < TOL


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 64, 65, 96, 127, 128, 129, 144, 145, 256, 260])
def test_query_rows(gpu, D, rows):
    check(gpu, 1, rows, 1, 1, D, [100], 0)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("rows", [129, 144, 272])
def test_extra_rows(gpu, D, rows):
    B = 140  # more query tiles than CUs: the last one of <= 16 rows joins the tile before it
    check(gpu, B, rows, 2, 2, D, [(13 * i) % 90 for i in range(B)], 2)


@pytest.mark.parametrize("T", [65, 68, 97])
@pytest.mark.parametrize("splits", [1, 3])
def test_extra_rows_of_the_last_tile(gpu, T, splits):
    """Several query tiles of which the last has extra rows (4 T = 260, 272, 388): the rows before the last tile are bit by
    bit those of the same sequence alone, whose tiles have no extra rows."""
    B, G, D = 100, 4, 256
    g = torch.Generator(device=gpu).manual_seed(T)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu).to(torch.bfloat16)
    pre = torch.tensor([(13 * i) % 190 for i in range(B)], dtype=torch.int32, device=gpu)
    q, k, v = rnd(B, T, G, D), rnd(B, 1, 190 + T, D), rnd(B, 1, 190 + T, D)
    out = K.attn_canvas(q, k, v, pre, mask_mode=0, splits=splits)
    ref = A.canvas_attention(q[:9].float().cpu(), k[:9].float().cpu(), v[:9].float().cpu(), pre[:9].tolist(), 0, 0)
    assert rel(out[:9], ref) < TOL
    n = (4 * T - 1) // 128 - 1  # whole tiles before the last
    for b in (0, 1, 8, B - 1):
        one = K.attn_canvas(q[b:b + 1], k[b:b + 1], v[b:b + 1], pre[b:b + 1], mask_mode=0, splits=splits)
        assert torch.equal(out[b, :32 * n], one[0, :32 * n]) and rel(out[b], one[0]) < TOL


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("B,rows", [(2, 1), (2, 17), (2, 63), (2, 65), (2, 127), (140, 129), (140, 144), (140, 260)])
def test_gate_of_the_only_split(gpu, D, B, rows):
    """The gated output of one split against the ungated one: bf16(o) sigmoid(gate), rounded to bf16 (2^-8; the hardware
    exponential is within 2^-20)."""
    g = torch.Generator(device=gpu).manual_seed(rows + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu).to(torch.bfloat16)
    q, k, v, gate = rnd(B, rows, 2, D), rnd(B, 2, 300, D), rnd(B, 2, 300, D), rnd(B, rows, 2, 2 * D)[..., D:]
    pre = torch.tensor([(7 * i) % 40 for i in range(B)], dtype=torch.int32, device=gpu)
    plain = K.attn_canvas(q, k, v, pre, mask_mode=0, splits=1)
    out = K.attn_canvas(q, k, v, pre, mask_mode=0, splits=1, gate=gate)
    want = plain.double() * torch.sigmoid(gate.double())
    assert ((out.double() - want).abs() <= want.abs() * 2 ** -8).all()


@pytest.mark.parametrize("keys", [1, 63, 64, 65, 127, 128, 129, 193])
@pytest.mark.parametrize("splits", [1, 2, 0])
def test_key_steps(gpu, keys, splits):
    check(gpu, 2, 1, 4, 2, 256, [keys - 1, max(keys - 2, 0)], 1, splits=splits)


@pytest.mark.parametrize("scale", [0.0, -0.0625, 0.25])
def test_scales(gpu, scale):
    check(gpu, 1, 33, 8, 2, 128, [150], 0, scale=scale)


@pytest.mark.parametrize("T", [4, 33])
def test_rising_scores(gpu, T):
    def shape(q, k, v):
        ramp = torch.linspace(0.01, 3.0, k.shape[2])[None, None, :, None]
        rows = torch.logspace(-2, 1, q.shape[1])[None, :, None, None]
        return q.abs() * rows, k.abs() * ramp, v

    check(gpu, 1, T, 4, 1, 256, [500], 0, shape=shape, splits=1)
