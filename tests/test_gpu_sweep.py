"""Row-sweep kernels on the device against the FP64 oracle, at the sizes where
strips, blocks of rows and passes begin and end."""

import numpy as np
import pytest

import pnp_sci_oracle as O

pytestmark = pytest.mark.gpu


def _frames(H, W, T, seed):
    """Frames that stop at different depths: a smooth image under growing noise."""
    g = np.random.default_rng(seed)
    r, c = np.arange(H)[:, None], np.arange(W)[None]
    base = 0.5 + 0.3 * np.cos(2 * np.pi * (r / 50 + c / 70))
    return np.stack([base + (0.02 + 0.1 * t) * g.standard_normal((H, W)) for t in range(T)])


@pytest.mark.parametrize("n", [8, 13, 14, 30])       # passes 4+3, 6+6, 5+4+4, 6+6+6+6+5
@pytest.mark.parametrize("H,W", [(1, 300), (300, 1), (7, 9), (8, 127), (9, 128), (63, 129),
                                 (64, 232), (65, 243), (130, 518)])
def test_deep_tv_passes_match_oracle(gpu, H, W, n):
    """The default deep TV: image and exit iteration of every frame, for frames
    that stop inside the first, a middle and the last pass and for ones that
    run to the end (max abs error 2e-5, the bound of the TV tests)."""
    import torch
    from pnp_sci.tv import tv_device
    img = _frames(H, W, 3, 1000 * H + W).astype(np.float32)
    for eps in (2e-4, 1e-2):
        got, stop = tv_device(torch.tensor(img, device="cuda"), 0.1, eps, n, return_stop=True)
        got, stop = got.cpu().numpy(), stop.cpu().tolist()
        for t in range(img.shape[0]):
            st = {}
            want = O.tv_chambolle_nd(img[t].astype(np.float64), 0.1, eps, n, _stats=st)
            assert stop[t] == st["returned"], (eps, t)
            assert np.max(np.abs(got[t] - want)) <= 2e-5, (eps, t)


@pytest.mark.parametrize("n", [2, 3, 4, 5])          # 1..4 dual updates
@pytest.mark.parametrize("H,W", [(1, 130), (7, 113), (8, 112), (9, 128), (16, 127), (33, 226),
                                 (65, 240)])
def test_reverse_sweep_matches_fp64_autograd(gpu, H, W, n):
    """The reverse TV at the edges of strips and blocks of rows: gradients of
    the mask, lambda and weights against FP64 autograd (the bounds of the
    unrolled tests: 1e-4 forward, 1e-3 gradients)."""
    from pnp_sci.synthetic import unrolled_batch
    from test_gpu_unrolled import _hip, _ref, _schedules, rel
    truth, mask = unrolled_batch(1, H, W, 3, seed=H * W, mask="logits")
    lam, w = _schedules(2, n)
    got = _hip(mask, truth, lam, w, n, True)
    want = _ref(mask, truth, lam, w, n, True)
    assert rel(got["x"], want["x"]) <= 1e-4
    for k in ("mask", "lam", "w"):
        assert rel(got[k], want[k]) <= 1e-3, k


@pytest.mark.parametrize("H,W", [(7, 7), (7, 71), (14, 70), (15, 9), (38, 134), (39, 135)])
def test_ssim_column_walk_matches_oracle(gpu, H, W):
    """Window centres at the ends of rows of lanes, of a lane's walk and of a
    workgroup (FP64 in another order: differences of about 49 roundings over the
    smallest denominator, 9e-4, stay below 1e-11)."""
    from pnp_sci.device import hwt_to_thw, to_device
    from pnp_sci.metrics import ssim_frames
    g = np.random.default_rng(H * W)
    a = g.random((H, W, 2)).astype(np.float32)
    b = (a + 0.1 * g.standard_normal(a.shape)).astype(np.float32)
    got = ssim_frames(hwt_to_thw(to_device(a)), hwt_to_thw(to_device(b)))
    for t in range(2):
        assert abs(got[t] - O.compare_ssim(a[..., t], b[..., t])) <= 1e-11
