"""Operators and conversions on the (H,W,T) layout, where blocks of pixels, the
vector accesses and the LDS budget begin and end.  Every result is exact: the
forward model is one rounding of an FP64 sum in frame order, the rest are
single products and copies."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _flat(a, off):
    """`a` on the device, `off` floats behind a 16-byte boundary."""
    import torch
    buf = torch.empty(a.size + off, dtype=torch.float32, device="cuda")
    v = buf[off:].view(a.shape)
    v.copy_(torch.from_numpy(a))
    return v


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("T", [1, 2, 3, 8, 20, 21, 32, 40, 61, 79, 121, 160, 161, 241])
@pytest.mark.parametrize("H,W", [(1, 1), (1, 63), (8, 8), (5, 13), (16, 16), (1, 257), (37, 28)])
def test_hwt_operators_and_conversions_are_exact(gpu, H, W, T, off):
    import torch
    from pnp_sci.device import hwt_to_thw, thw_to_hwt
    from pnp_sci.utils import A_, At_
    g = np.random.default_rng(H * 1000 + T)
    x = g.standard_normal((H, W, T)).astype(np.float32)
    phi = g.random((H, W, T)).astype(np.float32)
    y = g.standard_normal((H, W)).astype(np.float32)
    s = np.zeros((H, W))
    for t in range(T):
        s += x[:, :, t].astype(np.float64) * phi[:, :, t]
    xd, pd = _flat(x, off), _flat(phi, off)
    assert np.array_equal(A_(xd, pd).cpu().numpy(), s.astype(np.float32))
    assert np.array_equal(At_(_flat(y, off), pd).cpu().numpy(), y[:, :, None] * phi)
    thw = np.ascontiguousarray(x.transpose(2, 0, 1))
    assert np.array_equal(hwt_to_thw(xd).cpu().numpy(), thw)
    assert np.array_equal(thw_to_hwt(_flat(thw, off)).cpu().numpy(), x)


def test_operators_agree_over_memory_orders(gpu):
    """NumPy arrays C-ordered, frame-major and Fortran-ordered, in any mix, give
    the same bits."""
    from pnp_sci.utils import A_, At_
    g = np.random.default_rng(3)
    x, phi = (g.random((9, 14, 6)).astype(np.float32) for _ in range(2))
    y = A_(x, phi)
    back = At_(y, phi)
    orders = (np.ascontiguousarray, np.asfortranarray,
              lambda a: np.ascontiguousarray(a.transpose(2, 0, 1)).transpose(1, 2, 0))
    for fx in orders:
        for fp in orders:
            assert np.array_equal(A_(fx(x), fp(phi)), y)
            assert np.array_equal(At_(y, fp(phi)), back)
