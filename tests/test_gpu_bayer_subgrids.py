"""The two ways of the Bayer solver (sub-grids that share their launches, and
one at a time above a size) give the same mosaic.  Sub-grids of odd height and
width begin at odd elements of a packed array, where a single solve, which wants
8-byte alignment, would be refused."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,T", [(10, 14, 3), (10, 14, 2), (18, 30, 1), (16, 20, 3)])
@pytest.mark.parametrize("warm,iqa,n", [(False, False, 5), (True, True, 5), (True, False, 9)])
def test_subgrids_in_turn_match_shared_launches(gpu, monkeypatch, H, W, T, warm, iqa, n):
    import pnp_sci
    from pnp_sci import pnp_sci_algo as algo
    from pnp_sci.synthetic import truth_video
    g = np.random.default_rng(H + T)
    truth = truth_video(g, H, W, T)
    mask = (g.random((H, W, T)) < 0.5).astype(np.float32)
    y = (truth * mask).sum(2)
    x0 = g.random((H, W, T + 1)).astype(np.float32) if warm else None  # (one frame is not read)
    runs = []
    for voxels in (algo._SHARED_SOLVE_VOXELS, 0):
        monkeypatch.setattr(algo, "_SHARED_SOLVE_VOXELS", voxels)
        runs.append(pnp_sci.gap_denoise_bayer(y, mask, iter_max=6, tv_iter_max=n, x0_bayer=x0,
                                              X_orig=truth if iqa else None))
    (x, p, s, pa), (xt, pt, st, pat) = runs
    assert x.shape == xt.shape == (H, W, T)
    # (the frames may be split differently over workgroups: A x rounds differently)
    assert np.max(np.abs(x - xt)) <= 1e-5
    assert len(p) == len(pt) == len(s) == len(st) == (T if iqa else 0)
    assert np.allclose(p, pt, atol=1e-2) and np.allclose(s, st, atol=1e-4)
    assert len(pa) == len(pat) == (6 if iqa else 0) and np.allclose(pa, pat, atol=1e-2)


def test_short_warm_start_or_truth_is_refused(gpu, monkeypatch):
    import pnp_sci
    from pnp_sci import pnp_sci_algo as algo
    mask = np.ones((16, 20, 3), np.float32)
    for voxels in (algo._SHARED_SOLVE_VOXELS, 0):
        monkeypatch.setattr(algo, "_SHARED_SOLVE_VOXELS", voxels)
        for short in (dict(x0_bayer=mask[..., :2]), dict(X_orig=mask[..., :2])):
            with pytest.raises(ValueError):
                pnp_sci.gap_denoise_bayer(mask.sum(2), mask, iter_max=2, **short)
