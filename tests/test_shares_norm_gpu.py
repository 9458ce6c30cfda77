"""GPU: a projection's shares of K, the residual and the next norm in one launch."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shares", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("rows,H", [(1, 512), (5, 4096), (3, 8 * 1024 + 8), (130, 2560)])
def test_shares_in_order_then_the_norm(gpu, oracle, shares, rows, H):
    """Every number of shares that is asked for at once and one that is not, rows of less than a wave's vectors up to two rounds of a block: the residual
    row is the bf16 of the shares' float32 sum in order, plus the row, and the norm is pie_hip_rmsnorm's of it, both bit for bit (the norm's float32 sum
    runs in another order: one bf16 step where it rounds the other way)."""
    import torch
    from pie_amd import ops
    from pie_amd.ops import _ptr, _stream, kernels

    g = torch.Generator(device=gpu).manual_seed(7 * shares + rows)
    part = torch.randn(shares, rows, H, generator=g, device=gpu)
    x = torch.randn(rows, H, generator=g, device=gpu).bfloat16()
    w = (torch.rand(H, generator=g, device=gpu) + 0.5).bfloat16()
    want = part[0].clone()
    for z in range(1, shares):
        want += part[z]
    want = (want + x.float()).bfloat16()
    y = torch.empty_like(x)
    st = kernels().pie_hip_shares_rmsnorm(_ptr(part), shares, _ptr(x), _ptr(w), _ptr(y), rows, H, C.c_float(1e-5), _stream())
    assert st == 0
    assert torch.equal(x.view(torch.int16), want.view(torch.int16))
    norm = ops.rmsnorm_bf16(want, w, 1e-5)
    step = np.abs(y.view(torch.int16).cpu().numpy().astype(np.int32) - norm.view(torch.int16).cpu().numpy().astype(np.int32))
    assert step.max() <= 1 and (step == 0).mean() > 0.97
