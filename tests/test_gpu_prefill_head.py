"""GPU: TridaRuntime.prefill runs the LM head on the prompt's last row alone (its chunks before the last one run
none); its logits and caches are those of the full causal forwards."""
import pytest
import torch

from trida_stack_amd.model import HybridConfig, TridaRuntime, init_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wsgemm", [True, False])
@pytest.mark.parametrize("n,chunk", [(1, 64), (64, 64), (65, 64), (130, 64), (131, 512)])
def test_prefill_logits_are_the_last_row(gpu, wsgemm, n, chunk):
    cfg = HybridConfig.tiny(vocab=320)
    rt = TridaRuntime.__new__(TridaRuntime)
    rt.use_wsgemm = wsgemm
    rt.__init__(cfg, init_weights(cfg, seed=3), device=gpu, prefill_chunk=chunk)
    prompt = torch.randint(0, 300, (n,), generator=torch.Generator().manual_seed(n)).tolist()
    cache, full = rt.make_cache(1, 256), rt.make_cache(1, 256)
    got = rt.prefill(cache, prompt)
    for s0 in range(0, n, chunk):
        part = prompt[s0: s0 + chunk]
        ref = rt.forward(rt._ids(part), full, "causal")
    ref = ref[0, -1].float()
    # both are bf16 roundings of the same fp32 products, summed in another order where the head of one row and
    # of many run on different GEMMs: one bf16 unit (2^-8) of the largest logit
    assert (got - ref).abs().max() <= 2.0 ** -8 * ref.abs().max()
    for a, b in ((cache.kv_k, full.kv_k), (cache.kv_v, full.kv_v), (cache.state, full.state), (cache.window, full.window)):
        assert torch.equal(a, b)
    assert cache.length.tolist() == full.length.tolist() == [n]


def test_forward_without_head(gpu):
    cfg = HybridConfig.tiny(vocab=320)
    rt = TridaRuntime(cfg, init_weights(cfg, seed=4), device=gpu)
    cache = rt.make_cache(1, 64)
    ids = torch.randint(0, 300, (1, 9), generator=torch.Generator().manual_seed(1)).to(gpu)
    assert rt.forward(ids, cache, "causal", head="none") is None
    assert cache.length.tolist() == [9]
