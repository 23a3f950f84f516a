"""The decoder's cache after a prefill (cqgdn_prefill_cache): a pure move of data, so every word
must equal torch's transpose and row lookup."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("docs,H,HK,K,n", [
    (1, 16, 16, 4, 0), (1, 16, 16, 4, 1), (1, 4, 4, 4, 2), (2, 4, 4, 4, 3), (1, 8, 4, 4, 4), (3, 16, 8, 2, 9),
    (5, 32, 32, 3, 300), (0, 16, 16, 4, 5)])
def test_prefill_cache_equals_torch(gdn, docs, H, HK, K, n):
    from cqgdn import gated_delta_net as core

    print(f"case prefill cache: {docs} documents, {H} heads ({HK} key heads), K={K}, {n} content rows", flush=True)
    gen = torch.Generator().manual_seed(17 * docs + H + n)
    C = (2 * HK + H) * 128
    P = C + H * 128 + 2 * H
    state = torch.randn(docs, H, 128, 128, generator=gen)
    state.view(-1)[:3] = torch.tensor([float("inf"), -0.0, 1e-42])[:min(3, state.numel())]
    proj = torch.randn(n + 7, P, generator=gen).bfloat16()
    order = torch.randperm(n + 7, generator=gen)[:n].to(torch.int32)
    ds, dp, do = state.to(DEV), proj.to(DEV), order.to(DEV)
    out = torch.full_like(ds, 7.0)
    hist = torch.full((K - 1, C), 7.0, dtype=torch.bfloat16, device=DEV)
    core.call("cqgdn_prefill_cache", core._ptr(ds), docs, H, HK, core._ptr(dp), P, core._ptr(do) if n else None, n, K,
              core._ptr(out), core._ptr(hist), core._stream(ds.device))
    torch.cuda.synchronize()
    want = torch.zeros(K - 1, C, dtype=torch.bfloat16)
    tail = order[max(0, n - K):max(n - 1, 0)].long()
    if tail.numel():
        want[K - 1 - tail.numel():] = proj[tail, :C]
    bits = lambda t: t.cpu().contiguous().view(torch.int16 if t.dtype == torch.bfloat16 else torch.int32)
    assert torch.equal(bits(out), bits(state.transpose(-1, -2)))
    assert torch.equal(bits(hist), bits(want))
