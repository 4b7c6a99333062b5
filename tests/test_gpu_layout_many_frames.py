"""Layout conversions and forward model at the frame counts where their kernels
or block sizes change, with and without 16-byte accesses.  Conversions move
floats: equal bits.  The forward model sums exact products in fp64 and rounds
once: within one fp32 rounding of the fp64 sum."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [10, 11, 20, 21, 41, 64, 96, 112, 113, 160, 240, 241, 300])
@pytest.mark.parametrize("H,W", [(1, 1), (5, 13), (8, 8), (9, 29), (16, 36)])
def test_conversions_at_every_block_size(gpu, H, W, T):
    import torch
    from pnp_sci.device import hwt_to_thw, thw_to_hwt
    v = torch.rand((H, W, T), device="cuda")
    w = hwt_to_thw(v)
    assert torch.equal(w, v.permute(2, 0, 1))
    assert torch.equal(thw_to_hwt(w), v)


@pytest.mark.parametrize("T", [20, 21, 40, 41, 120, 121, 128, 129, 300])
@pytest.mark.parametrize("H,W", [(1, 1), (15, 17), (16, 16), (9, 29), (16, 36)])
def test_forward_model_of_many_frames(gpu, H, W, T):
    import torch
    from pnp_sci.utils import A_, At_
    x, phi = torch.rand((H, W, T), device="cuda"), torch.rand((H, W, T), device="cuda")
    y = A_(x, phi)
    want = (x.double() * phi.double()).sum(2)
    # half an ulp of fp32, and the fp64 sum's own order (2^-53 per term)
    assert float((y.double() - want).abs().max()) <= float(want.max()) * (2.0 ** -24 + T * 2.0 ** -52)
    assert torch.equal(At_(y, phi), y[:, :, None] * phi)
