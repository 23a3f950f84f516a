"""The conv backward's split of the rows into strips (csrc/gdn_conv.hip): enough workgroups for the
chip whatever the channels, and right at the strips' edges."""

import pytest
import torch

DEV = "cuda:0"


@pytest.mark.parametrize("K", [2, 4])
@pytest.mark.parametrize("C", [8, 128, 512, 1536, 2048, 3072, 6144])
def test_long_conv_backward_has_a_workgroup_per_cu(C, K):
    """A workgroup takes 256 channels of one part of the rows and writes one dw partial [C][K], so the
    workspace holds the number of parts; 256 workgroups give every CU one."""
    from cqgdn import _lib

    parts, rest = divmod(_lib.lib().cqgdn_conv1d_bwd_workspace_size(65536, C, K), C * K * 4)
    assert rest == 0
    assert parts * ((C + 255) // 256) >= 256, parts


def test_workspace_size_takes_any_channels():
    from cqgdn import _lib

    for C in range(1, 10):
        assert _lib.lib().cqgdn_conv1d_bwd_workspace_size(5, C, 4) == C * 4 * 4  # one part


@pytest.mark.gpu
@pytest.mark.parametrize("T,C,K,bounds", [
    (8192, 256, 4, (0, 8192)),              # 512 strips of 16 rows, the last part whole
    (8192 * 4 + 1, 64, 2, (0, 32769)),      # 17 rows a strip, the last parts short
    (20011, 512, 4, (0, 1, 9000, 20011)),   # documents ending inside strips
    (9000, 1544, 3, (0, 4500, 9000)),       # a channel block of 8
])
def test_conv_backward_over_many_strips(gdn, T, C, K, bounds):
    """dx and dw against float64.  dx is one bf16 rounding (2^-9) of K products; dw an fp32 sum of T
    products in strips, rounded to bf16 once (2^-9 of it): 2^-8 of the value, and for dw 2^-15 of the terms'
    size for the order of the sum and the fast exp."""
    print(f"case conv strips T={T} C={C} K={K} bounds={bounds}", flush=True)
    gen = torch.Generator().manual_seed(T + C)
    x, dy = (torch.randn(1, T, C, generator=gen).bfloat16() for _ in range(2))
    w = (torch.randn(C, K, generator=gen) * 0.5).bfloat16()
    xd, wd = x.to(DEV).requires_grad_(), w.to(DEV).requires_grad_()
    y, _ = gdn.conv(xd, wd, activation="silu", cu_seqlens=torch.tensor(bounds, device=DEV), cu_seqlens_cpu=bounds)
    y.backward(dy.to(DEV))
    pad = torch.zeros(K - 1, C, dtype=torch.float64)
    dx, dw, size = torch.zeros(T, C, dtype=torch.float64), torch.zeros(C, K, dtype=torch.float64), \
        torch.zeros(C, K, dtype=torch.float64)
    dx_size = torch.zeros_like(dx)
    taps = w.double()
    for a, b in zip(bounds, bounds[1:]):
        rows = torch.cat((pad, x[0, a:b].double()))
        shifted = [rows[i:i + b - a] for i in range(K)]
        pre = sum(s * taps[:, i] for i, s in enumerate(shifted))
        sg = torch.sigmoid(pre)
        dpre = dy[0, a:b].double() * sg * (1 + pre * (1 - sg))
        for i, s in enumerate(shifted):
            dw[:, i] += (dpre * s).sum(0)
            size[:, i] += (dpre * s).abs().sum(0)
            back = K - 1 - i
            if back < b - a:
                dx[a:b - back] += dpre[back:] * taps[:, i]
                dx_size[a:b - back] += (dpre[back:] * taps[:, i]).abs()
    for name, got, want, terms in (("dx", xd.grad[0], dx, dx_size), ("dw", wd.grad, dw, size)):
        err = (got.cpu().double() - want).abs()
        assert (err <= 2.0 ** -8 * want.abs() + 2.0 ** -15 * terms + 1e-6).all(), (name, float(err.max()))
