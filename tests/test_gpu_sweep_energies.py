"""Energies of the deep TV, the sums its early exit compares: their error does not
grow with the rows of a strip."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _align(n):
    return (n + 255) // 256 * 256


@pytest.mark.parametrize("weight", [0.007, 0.051, 0.1, 0.171, 0.217, 0.283])
@pytest.mark.parametrize("H,T", [(64, 4096), (64, 2)])   # strips of 64 rows, of 8
def test_first_energy_of_a_ramp(gpu, H, T, weight):
    """A ramp of slope 1/64: E_0 = weight |g| over H x (W-1) pixels, every term the
    same number, so that roundings do not cancel.  A sum of m equal terms is off
    by up to (m + 1)/2 roundings of 2^-24: 4.5 for the 8 terms of 4 rows of two
    columns, 8.5 for the 16 such sums of a strip, one for each of the 6 levels
    over the lanes: 19.  A sum of all 128 terms reaches 32 at these weights."""
    import torch
    from pnp_sci import _lib
    W = 100
    img = (torch.arange(W, device="cuda", dtype=torch.float32) / 64).expand(T, H, W).contiguous()
    out = torch.empty_like(img)
    nb = gpu.scigap_tv_workspace_bytes(H, W, T, 8)
    ws = torch.zeros(nb, dtype=torch.uint8, device="cuda")
    _lib.check(gpu.scigap_tv_chambolle(img.data_ptr(), out.data_ptr(), H, W, T, weight, 0.0, 8, None,
                                       ws.data_ptr(), nb, _lib.stream_ptr()))
    torch.cuda.synchronize()
    # the slots of the first pass follow the two dual fields: [frame][6 updates][strips]
    off = 2 * _align(8 * T * H * W)
    rows = {4096: 64, 2: 8}[T]
    strips = H // rows
    slots = ws[off:off + T * 6 * strips * 4].view(torch.float32).view(T, 6, strips)[:, 0].double()
    want = float(np.float32(weight)) / 64 * rows * (W - 1)
    rel = (slots / want - 1).abs().max().item()
    assert rel <= 19 * 2.0 ** -24, rel / 2.0 ** -24
