"""SSIM where a lane's walk down a column ends: after each of its rows, at the end
of a wave's and of a workgroup's rows."""

import numpy as np
import pytest

import pnp_sci_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [7, 8, 9, 10, 11, 12, 13, 14, 15, 21, 22, 23, 37, 38, 39, 45, 46, 47])
def test_ssim_of_every_last_row(gpu, H):
    """FP64 in another order: differences of about 49 roundings over the smallest
    denominator, 9e-4, stay below 1e-11."""
    from pnp_sci.device import hwt_to_thw, to_device
    from pnp_sci.metrics import ssim_frames
    g = np.random.default_rng(H)
    a = g.random((H, 11, 3)).astype(np.float32)
    b = (a + 0.1 * g.standard_normal(a.shape)).astype(np.float32)
    got = ssim_frames(hwt_to_thw(to_device(a)), hwt_to_thw(to_device(b)))
    for t in range(3):
        assert abs(got[t] - O.compare_ssim(a[..., t], b[..., t])) <= 1e-11
