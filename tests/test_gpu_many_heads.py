"""cqgdn_fwd and cqgdn_bwd at head counts far past the layers': heads do not see each other, so some of
many heads must give bitwise what the same heads give in a call of their own.  20000 heads: a round of
the scans spans more than 2 GB; 26304: more than the 4 GB a raw buffer reaches, where the scans take a
buffer per step."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,dtype", [(20000, torch.bfloat16), (26304, torch.bfloat16), (26304, torch.float16)])
def test_many_heads_equal_the_same_heads_alone(gdn, H, dtype):
    bounds = (0, 6 * 64 - 9, 6 * 64 + 55)  # 6 chunks, a round and two steps; then one chunk
    T, scale = bounds[-1], 128 ** -0.5
    print(f"case many heads: H={H} {dtype} T={T}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(H)
    q, k, v, dy = (torch.randn(1, T, H, 128, generator=gen, device=DEV, dtype=dtype) for _ in range(4))
    v[0, 0, 0, 0] = 7.0  # the largest |v| and |dO| among the heads compared: the fp16 scales are a call's
    dy[0, 0, 0, 0] = 7.0
    v.clamp_(-7, 7)
    dy.clamp_(-7, 7)
    b = torch.rand(1, T, H, generator=gen, device=DEV)
    g = -0.1 * torch.rand(1, T, H, generator=gen, device=DEV)
    heads = torch.tensor([0, 1, 13107, H // 2, H - 2, H - 1], device=DEV)

    def run(q, k, v, g, b, dy):
        o, _, ws = gdn._forward(q, k, v, g, b, bounds, True, scale, training=True)
        return [o, *gdn._backward(q, k, v, g, b, ws, dy, bounds, True, scale)]

    alone = run(*(x.index_select(2, heads).contiguous() for x in (q, k, v, g, b, dy)))
    for name, x, want in zip(("o", "dq", "dk", "dv", "dg", "dbeta"), run(q, k, v, g, b, dy), alone):
        assert torch.isfinite(want.float()).all(), name
        assert torch.equal(x.index_select(2, heads), want), name
