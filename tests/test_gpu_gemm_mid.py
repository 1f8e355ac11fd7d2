"""GPU: the mid-size weight-streaming GEMM against fp64 products of the same bf16 operands: row counts around its tiles of
16 and its rounds of 8 of them, K around its stages of 8 k-steps, column tiles that do not fill a workgroup, every
epilogue, row-major and fragment-order outputs; and the residual that writes its input."""
from dataclasses import replace

import pytest
import torch

from trida_stack_amd import kernels as K
from trida_stack_amd.model import HybridConfig, TridaRuntime, init_weights

pytestmark = pytest.mark.gpu


def frag(x):
    """Row-major [M, K] to fragment order, the rows past M NaN."""
    M, Kd = x.shape
    mt = (M + 15) // 16
    p = torch.full((mt * 16, Kd), float("nan"), dtype=x.dtype, device=x.device)
    p[:M] = x
    return p.view(mt, 16, Kd // 32, 4, 8).permute(2, 0, 3, 1, 4).contiguous().view(-1)


def unfrag(f, M, Kd):
    mt = (M + 15) // 16
    return f.view(Kd // 32, mt, 4, 16, 8).permute(1, 3, 0, 2, 4).reshape(mt * 16, Kd)[:M]


def rel(got, ref):
    return ((got.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("M", [49, 64, 65, 127, 128, 129, 144, 264, 385, 512])
@pytest.mark.parametrize("N,Kd", [(16, 32), (48, 256), (160, 288), (1040, 512), (2560, 2080)])
def test_products(gpu, M, N, Kd):
    g = torch.Generator(device=gpu).manual_seed(M * N + Kd)
    x = torch.randn(M, Kd, generator=g, device=gpu).to(torch.bfloat16)
    w = (torch.randn(N, Kd, generator=g, device=gpu) * Kd ** -0.5).to(torch.bfloat16)
    ref, xf = x.double() @ w.double().t(), frag(x)
    wp = K.ws_shuffle(w)
    out = torch.full((M, N + 4), -7.0, dtype=torch.bfloat16, device=gpu)
    K.ws_gemm_mid(xf, M, wp, N, out[:, :N])
    assert rel(out[:, :N], ref) < 2 ** -8 and (out[:, N:] == -7).all()  # one bf16 rounding
    parts = torch.empty(K.ws_mid_planes(M, N, Kd), M, N, device=gpu)
    assert K.ws_gemm_mid(xf, M, wp, N, parts, epilogue=K.WS_PARTS) == parts.shape[0]
    assert rel(parts.double().sum(0), ref) < 2e-6  # fp32 sums of K <= 2080 products
    if N % 64 == 0 or N == 160:
        h = torch.randn(M, Kd, generator=g, device=gpu).to(torch.bfloat16)
        r = torch.randn(M, Kd, generator=g, device=gpu).to(torch.bfloat16)
        ss, hf = torch.empty(M, K.ss_chunks(Kd), device=gpu), torch.empty_like(xf)
        want = (h.float() + r.float()).to(torch.bfloat16)
        K.residual_mid(h, r, ss, hf)
        assert torch.equal(h, want) and torch.equal(unfrag(hf, M, Kd), want)
        n = want.double() * torch.rsqrt((want.double() ** 2).mean(-1, keepdim=True) + 1e-6)
        gate, up = (n @ w.double().t()).to(torch.bfloat16).double().split(N // 2, -1)
        y = torch.nn.functional.silu(gate) * up
        act = torch.empty(M, N // 2, dtype=torch.bfloat16, device=gpu)
        wq = K.ws_shuffle(w, pair_halves=True)
        K.ws_gemm_mid(hf, M, wq, N, act, ss=ss, epilogue=K.WS_SILU)
        assert rel(act, y) < 2 ** -7  # the roundings of gate, up and the product
        if N // 2 % 32 == 0:
            af = torch.empty(K.ws_mid_numel(M, N // 2), dtype=torch.bfloat16, device=gpu)
            K.ws_gemm_mid(hf, M, wq, N, af, ss=ss, epilogue=K.WS_SILU, out_frag=True)
            assert torch.equal(unfrag(af, M, N // 2), act)


@pytest.mark.parametrize("M", [49, 128, 129, 264, 385, 512])
def test_wide_plans(gpu, M):
    """The products of the 4B-shape MLP, whose plans take 3 to 5 column tiles per workgroup (1216 tiles in fives: the
    last workgroup has one) and split K over up to 6 groups, where the shapes above take 2 tiles and at most 3 groups."""
    g = torch.Generator(device=gpu).manual_seed(M)
    N, Kd = 19456, 2560
    h = torch.randn(M, Kd, generator=g, device=gpu).to(torch.bfloat16)
    w = (torch.randn(N, Kd, generator=g, device=gpu) * Kd ** -0.5).to(torch.bfloat16)
    ss, hf, wp = torch.empty(M, K.ss_chunks(Kd), device=gpu), frag(h), K.ws_shuffle(w)
    K.residual_mid(h, torch.zeros_like(h), ss, torch.empty_like(hf))
    out = torch.full((M, N + 4), -7.0, dtype=torch.bfloat16, device=gpu)
    K.ws_gemm_mid(hf, M, wp, N, out[:, :N])
    assert rel(out[:, :N], h.double() @ w.double().t()) < 2 ** -8 and (out[:, N:] == -7).all()
    n = h.double() * torch.rsqrt((h.double() ** 2).mean(-1, keepdim=True) + 1e-6)
    gate, up = (n @ w.double().t()).to(torch.bfloat16).double().split(N // 2, -1)
    y = torch.nn.functional.silu(gate) * up
    wq = K.ws_shuffle(w, pair_halves=True)
    act = torch.full((M, N // 2 + 4), -7.0, dtype=torch.bfloat16, device=gpu)
    K.ws_gemm_mid(hf, M, wq, N, act[:, :N // 2], ss=ss, epilogue=K.WS_SILU)
    assert rel(act[:, :N // 2], y) < 2 ** -7 and (act[:, N // 2:] == -7).all()
    af = torch.empty(K.ws_mid_numel(M, N // 2), dtype=torch.bfloat16, device=gpu)
    K.ws_gemm_mid(hf, M, wq, N, af, ss=ss, epilogue=K.WS_SILU, out_frag=True)
    assert torch.equal(unfrag(af, M, N // 2), act[:, :N // 2])

    w2 = (torch.randn(Kd, N // 2, generator=g, device=gpu) * (N // 2) ** -0.5).to(torch.bfloat16)
    kg = K.ws_mid_planes(M, Kd, N // 2)
    parts = torch.empty(kg, M, Kd, device=gpu)
    assert K.ws_gemm_mid(af, M, K.ws_shuffle(w2), Kd, parts, epilogue=K.WS_PARTS) == kg
    ref = act[:, :N // 2].double() @ w2.double().t()
    assert rel(parts.double().sum(0), ref) < 2e-6  # fp32 sums of 32 products at a time, at most 9728 / 32 of them


@pytest.mark.parametrize("B,T", [(7, 7), (4, 33), (16, 32), (1, 300)])
@pytest.mark.parametrize("mid", [True, False])
def test_forward_mlp(gpu, B, T, mid):
    """Every layer's MLP branch of a forward against fp64 on the layer's own input rows, on this path and on the
    library's. Roundings to bf16 on the way: the normed rows or the normed weights, gate, up, their product and the
    branch, each at most 2^-9 of the value and at random signs: 2^-7 in the norm covers the five."""
    cfg = replace(HybridConfig.tiny(vocab=320), lin_v_heads=8)  # every projection in whole tiles
    w = init_weights(cfg, seed=5)
    g = torch.Generator().manual_seed(1)
    for i in range(cfg.n_layers):
        w[f"l{i}.post_norm"] = (torch.randn(cfg.hidden, generator=g) * 0.1).to(torch.bfloat16)
    rt = TridaRuntime(cfg, w, device=gpu)
    assert rt._mid(B * T)
    if not mid:
        rt._mid = lambda N: False
    seen = {}

    def probe(i, where, h, r):
        if where != "gdn":
            seen[i, where] = (h.clone(), None if r is None else r.clone())

    rt.layer_probe = probe
    ids = torch.randint(0, 300, (B, T), generator=g).to(gpu)
    rt.forward(ids, rt.make_cache(B, T + 8), "verify")
    for i in range(cfg.n_layers):
        h = seen[i, "mid"][0].double()
        n = h * torch.rsqrt((h * h).mean(-1, keepdim=True) + cfg.rms_eps) * (1 + rt.w[f"l{i}.post_norm"].double())
        gate, up = (n @ rt.w[f"l{i}.w_gu"].double().t()).split(cfg.intermediate, -1)
        ref = (torch.nn.functional.silu(gate) * up) @ rt.w[f"l{i}.w_down"].double().t()
        assert rel(seen[i + 1, "in"][1], ref) < 2 ** -7, i
