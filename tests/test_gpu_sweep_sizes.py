"""The deep TV at every height of its strips, with few strips a frame (each wave
takes the exit test) and many (a launch of its own), against the FP64 oracle:
frames that stop in the first, a middle and the last pass, and ones that do not."""

import numpy as np
import pytest

from test_sweep_geometry import SIZES

pytestmark = pytest.mark.gpu

UNIQUE = 6


@pytest.mark.parametrize("H,W,T,n", list(SIZES))
def test_every_strip_height_matches_oracle(gpu, H, W, T, n):
    """Image (2e-5, the bound of the TV tests) and exit iteration of up to six
    different frames; the others repeat them and give the same bits."""
    import torch
    import oracle_c
    from pnp_sci.tv import tv_device
    g = np.random.default_rng(H + W)
    r, c = np.arange(H)[:, None], np.arange(W)[None]
    base = 0.5 + 0.3 * np.cos(2 * np.pi * (r / 50 + c / 70))
    k = min(UNIQUE, T)
    img = np.stack([base + (0.02 + 0.1 * t) * g.standard_normal((H, W))
                    for t in range(k)]).astype(np.float32)
    dev = torch.tensor(img, device="cuda")[torch.arange(T, device="cuda") % k].contiguous()
    passes = -(-(n - 1) // 6)
    met = set()
    for eps in (2e-4, 1e-2, 0.0):
        got, stop = tv_device(dev, 0.1, eps, n, return_stop=True)
        want, stops = oracle_c.tv(np.moveaxis(img, 0, -1), 0.1, eps, n)
        assert stop[:k].cpu().tolist() == stops.tolist(), eps
        assert np.max(np.abs(got[:k].cpu().numpy() - np.moveaxis(want, -1, 0))) <= 2e-5, eps
        assert torch.equal(got, got[torch.arange(T, device="cuda") % k]), eps
        assert torch.equal(stop, stop[torch.arange(T, device="cuda") % k]), eps
        met |= {min(s * passes // (n - 1), passes) for s in stops.tolist()}
    if k == UNIQUE:
        assert {0, passes - 1, passes} <= met, met   # pass that the frame stopped in
