"""GPU: the GDN front half in blocks of several rows (grids of >= 512 rows) is bitwise the one-row-per-block form:
every row and window of a batch equals that of its sequence run alone, at chunk lengths and remainders of either."""
import pytest
import torch

from trida_stack_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T", [(512, 1), (256, 2), (103, 5), (40, 13), (17, 31), (16, 33), (64, 33)])
@pytest.mark.parametrize("Hk,Hv,Dk,Kc", [(2, 4, 32, 4), (2, 2, 64, 3), (4, 4, 128, 4), (1, 3, 128, 2)])
def test_rows_match_single_sequences(gpu, B, T, Hk, Hv, Dk, Kc):
    C = 2 * Hk * Dk + Hv * 64
    g = torch.Generator(device=gpu).manual_seed(B * T)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    x, window, conv, a, b = rn(B, T, C + 8)[..., :C], rn(B, Kc - 1, C), rn(C, Kc), rn(B, T, Hv), rn(B, T, Hv)
    A_log, dt = torch.rand(Hv, generator=g, device=gpu), torch.rand(Hv, generator=g, device=gpu)

    def prep(s):
        win, pre = torch.empty_like(window[s]), torch.empty(x[s].shape, dtype=torch.bfloat16, device=gpu)
        out = K.gdn_prep(x[s], window[s], conv, a[s], b[s], A_log, dt, Hk=Hk, Hv=Hv, Dk=Dk, Dv=64, window_out=win,
                         pre_out=pre)
        return *out, win, pre

    many = prep(slice(0, B))
    for i in (0, 1, B // 2, B - 1):
        for m, o in zip(many, prep(slice(i, i + 1))):
            assert torch.equal(m[i], o[0])


@pytest.mark.parametrize("T", [31, 33, 129])
@pytest.mark.parametrize("lens", ["ragged", "past"])
def test_packed_rows(gpu, T, lens):
    """The same for packed sequences with a window pool, a pre-conv pool and a conv bias: lengths of 0, 1, around a chunk
    and the whole max_rows; and ("past") lengths above max_rows, of which the first max_rows rows are the sequence. Rows past
    it and pool rows that no sequence owns stay untouched."""
    Hk, Hv, Dk, Dv, Kc, B = 1, 2, 32, 64, 4, 24
    C = 2 * Hk * Dk + Hv * Dv
    g = torch.Generator(device=gpu).manual_seed(T)
    rn = lambda *s: torch.randn(*s, generator=g, device=gpu).to(torch.bfloat16)  # noqa: E731
    ns = [[0, 1, 3, 4, 5, 16, T - 1, T][i % 8] for i in range(B)]
    if lens == "past":
        ns = [n + T - 2 if i % 3 == 0 else n for i, n in enumerate(ns)]
    cu = torch.tensor([0] + ns, device=gpu).cumsum(0)
    total = int(cu[-1])
    x, window, conv, bias, a, b = rn(total, C + 8)[:, :C], rn(B + 2, Kc - 1, C), rn(C, Kc), rn(C), rn(total, Hv), rn(total, Hv)
    A_log, dt = torch.rand(Hv, generator=g, device=gpu), torch.rand(Hv, generator=g, device=gpu)
    perm = torch.randperm(B, generator=g, device=gpu).int()
    win_idx, pre_idx = (perm + 1).contiguous(), (perm.flip(0) + 1).contiguous()
    win, pre = torch.full_like(window, -7.0), torch.full((B + 2, T, C), -7.0, dtype=torch.bfloat16, device=gpu)
    out = tuple(torch.full((total, *s), -7.0, dtype=d, device=gpu) for s, d in
                (((Hk, Dk), torch.bfloat16), ((Hk, Dk), torch.bfloat16), ((Hv, Dv), torch.bfloat16), ((Hv,), torch.float32),
                 ((Hv,), torch.float32)))
    kw = dict(Hk=Hk, Hv=Hv, Dk=Dk, Dv=Dv, conv_bias=bias)
    assert B * T >= 512  # several rows per block
    K.gdn_prep(x, window, conv, a, b, A_log, dt, window_out=win, pre_out=pre, win_idx=win_idx, pre_idx=pre_idx,
               cu_seqlens=cu.int(), max_rows=T, out=out, **kw)
    for i, n in enumerate(ns):
        r0, m, wi, pi = int(cu[i]), min(n, T), int(win_idx[i]), int(pre_idx[i])
        assert all((o[r0 + m: r0 + n] == -7).all() for o in out) and (pre[pi, m:] == -7).all(), i
        if m == 0:
            assert (win[wi] == -7).all(), i
            continue
        w1 = torch.empty_like(window[:1])
        ref = K.gdn_prep(x[None, r0: r0 + m], window[wi][None], conv, a[None, r0: r0 + m], b[None, r0: r0 + m], A_log, dt,
                         window_out=w1, **kw)
        assert all(torch.equal(o[r0: r0 + m], r[0]) for o, r in zip(out, ref)), i
        assert torch.equal(pre[pi, :m], x[r0: r0 + m]) and torch.equal(win[wi], w1[0]), i
    for pool, own in ((win, win_idx), (pre, pre_idx)):
        assert all((pool[r] == -7).all() for r in set(range(B + 2)) - set(own.tolist()))
