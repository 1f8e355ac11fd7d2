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
