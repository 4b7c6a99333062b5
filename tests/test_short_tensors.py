"""Tensors smaller than what a kernel reads are refused before any device work
(no GPU)."""

import pytest
import torch

from pnp_sci.device import sq_error
from pnp_sci.metrics import ssim_frames
from pnp_sci.pnp_sci_algo import solve_device

H, W, T = 9, 8, 3


@pytest.mark.parametrize("short", [dict(y=(H, W - 1)), dict(phi_sum=(H - 1, W)),
                                   dict(x0=(T - 1, H, W)), dict(truth=(T, H - 1, W))])
def test_a_solve_refuses_short_tensors(short):
    kw = dict(y=torch.ones(H, W), phi=torch.ones(T, H, W), phi_sum=torch.ones(H, W))
    kw.update({k: torch.ones(v) for k, v in short.items()})
    with pytest.raises(ValueError):
        solve_device(kw.pop("y"), kw.pop("phi"), kw.pop("phi_sum"), iters=1, **kw)


def test_metrics_refuse_short_tensors():
    x, fewer = torch.ones(T, H, W), torch.ones(T - 1, H, W)
    for per_frame in (False, True):
        with pytest.raises(ValueError):
            sq_error(x, fewer, per_frame)
    with pytest.raises(ValueError):
        ssim_frames(fewer, x)
