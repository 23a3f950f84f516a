"""The backward of the query convolutions alone (content events with zero gradients) against float64:
the queries' own rows, the history rows they share, and the taps' gradient."""
import ctypes
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K,n_q,n_c", [(2, 1, 1), (3, 130, 9), (4, 515, 200), (4, 33000, 40)])
def test_query_backward(gdn, K, n_q, n_c):
    """One query; workgroups with idle waves; rows read by 1 to 9 pairs and by thousands; and more
    queries than the 64 per wave whose indices are held at once (32768 over the 128 workgroups)."""
    from cqgdn import _lib, events

    H, S = 4, 512
    P, C = 4 * S + 2 * H, 3 * S
    print(f"case query backward: K={K}, {n_q} queries over {n_c} content rows", flush=True)
    gen = torch.Generator().manual_seed(K * n_q)
    hist = torch.randint(0, n_c + 1, (n_q, K - 1), generator=gen)
    ids = torch.arange(n_c + n_q)
    plan = SimpleNamespace(content_order=ids[:n_c], event_q=ids, event_write=torch.clamp(ids, max=n_c),
                           query_source=ids[n_c:], query_history=hist, content_bounds=(0, n_c),
                           event_bounds=(0, n_c + n_q), hidden_length=n_c + n_q, hidden_event=ids)
    ep = events.event_plan(plan, K, torch.device(DEV))
    proj = torch.randn(n_c + n_q, P, generator=gen).bfloat16()
    w = (torch.rand(C, K, generator=gen) - 0.5).bfloat16()
    dq = torch.randn(n_c + n_q, S, generator=gen).bfloat16()
    dq[:n_c] = 0
    gproj, gw, gdq = proj.to(DEV), w.to(DEV), dq.to(DEV)
    zero = torch.zeros_like(gdq)
    one = torch.zeros(H, device=DEV)
    gate = torch.zeros(n_c + n_q, H, device=DEV)
    dproj = torch.full_like(gproj, 7.0)
    dw = torch.full((C, K), 7.0, device=DEV)
    dgate = torch.full((2 * H,), 7.0, device=DEV)
    ws = torch.empty(_lib.lib().cqgdn_event_inputs_bwd_workspace_size(ctypes.byref(ep.cstruct), H, H),
                     dtype=torch.uint8, device=DEV)
    p = gdn._ptr
    gdn.call("cqgdn_event_inputs_bwd", ctypes.byref(ep.cstruct), H, H, p(gproj), P, gproj[:, 4 * S:].data_ptr(), P,
             gproj[:, 4 * S + H:].data_ptr(), P, p(gw), p(one), p(one), p(gdq), p(zero), p(zero), p(gate), p(gate),
             p(dproj), P, dproj[:, 4 * S:].data_ptr(), P, dproj[:, 4 * S + H:].data_ptr(), P, p(dw), p(dgate), p(ws),
             ws.numel(), gdn._stream(gproj.device))
    torch.cuda.synchronize()
    rows = torch.cat((proj[:n_c, :S], torch.zeros(1, S).bfloat16())).double()
    x = torch.cat((rows[hist], proj[n_c:, None, :S].double()), 1)  # [n_q][K][S]
    taps = w[:S].double()
    pre = (x * taps.T).sum(1)
    sg = torch.sigmoid(pre)
    dpre = dq[n_c:].double() * sg * (1 + pre * (1 - sg))
    want = torch.zeros(n_c + 1, S, dtype=torch.float64)
    size = torch.zeros(n_c + 1, S, dtype=torch.float64)
    for i in range(K - 1):
        term = dpre * taps[:, i]
        want.index_add_(0, hist[:, i], term)
        size.index_add_(0, hist[:, i], term.abs())
    want[n_c:], size[n_c:] = 0, 0
    own = dpre * taps[:, K - 1]
    got = dproj.cpu().double()
    # one bf16 rounding (2^-9) of an fp32 sum; the fast exp and reciprocal and the sums' order stay under 2^-15 of
    # the terms' size
    for name, g, e, s in (("own rows", got[n_c:, :S], own, own.abs()), ("history rows", got[:n_c, :S], want[:n_c], size[:n_c])):
        assert ((g - e).abs() <= 2.0 ** -8 * e.abs() + 2.0 ** -15 * s + 1e-6).all(), name
    terms = [(dpre * x[:, i], i) for i in range(K)]
    for t, i in terms:
        err = (dw[:S, i].cpu().double() - t.sum(0)).abs()
        assert (err <= 2.0 ** -15 * t.abs().sum(0) + 1e-6).all(), f"tap {i}: {err.max()}"
    assert not dw[S:].any() and not got[n_c:, S:C].any()
