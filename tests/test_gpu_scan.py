"""The state scans at every document length around their four-step rounds.

The scans run four chunk steps a round, the first round apart, and up to three steps after the
last; operands are requested four steps ahead.  One packed batch holds documents of 0 to 9 and 13
chunks, each ending in a chunk of another length, so every combination of rounds and last steps
occurs, and no document may see its neighbour's chunks.  Bars as in the parity tests: 2e-2 for
bf16 operands, 2e-3 for fp16 ones (four times what they measure), 1e-3 for the fp32 final states."""

import pytest
import torch

from gdn_testlib import TOL_BF16, TOL_STATE, assert_close_bf16, rel_l2
from oracle import gdn_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
LENGTHS = [1, 128, 129 + 63, 256, 0, 257, 6 * 64 - 31, 448, 7 * 64 + 5, 9 * 64 - 1, 13 * 64 - 47]


@pytest.mark.parametrize("H,dtype", [(4, torch.bfloat16), (8, torch.float16), (32, torch.bfloat16)])
def test_scans_at_every_round_remainder(gdn, H, dtype):
    bounds = [0]
    for n in LENGTHS:
        bounds.append(bounds[-1] + n)
    T = bounds[-1]
    print(f"case documents of {LENGTHS} events, H={H} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(77 + H)
    q, k, v, do = (torch.randn(1, T, H, 128, generator=gen).to(dtype) for _ in range(4))
    beta = torch.randn(1, T, H, generator=gen).sigmoid()
    g = -0.05 * torch.nn.functional.softplus(torch.randn(1, T, H, generator=gen))
    s0 = torch.randn(len(LENGTHS), H, 128, 128, generator=gen) * 0.1
    xd = [x.to(DEV).requires_grad_() for x in (q, k, v, g, beta)]
    y, _ = gdn.delta(*xd, use_qk_l2norm_in_kernel=True, cu_seqlens=torch.tensor(bounds, device=DEV),
                     cu_seqlens_cpu=bounds)
    y.backward(do.to(DEV))
    _, states = gdn.prefill(*(x.detach() for x in xd), bounds, initial_state=s0.to(DEV))
    torch.cuda.synchronize()
    ref = [x.double() for x in (q, k, v, g, beta)]
    tol = TOL_BF16 if dtype == torch.bfloat16 else 2e-3
    assert_close_bf16("o", y.detach().cpu(), O.chunk_delta(*ref, bounds), tol=tol)
    grads = O.chunk_delta_backward(*ref, do.double(), bounds)
    for name, x, r in zip(("dq", "dk", "dv", "dg", "dbeta"), xd, grads):
        assert_close_bf16(name, x.grad.cpu(), r, tol=tol)
    _, ref_states = O.chunk_delta(*ref, bounds, initial_state=s0.double(), output_final_state=True)
    for d, n in enumerate(LENGTHS):
        assert rel_l2(states[d].cpu(), ref_states[d]) <= TOL_STATE, (d, n)
