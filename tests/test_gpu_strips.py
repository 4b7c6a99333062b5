"""Strips of the fused outer iteration: the default launch chooses masks and row
updates strip by strip, the launches split by tile class (engine 3) mask whole
tiles and update every row.  Both give the same bits, at the sizes where strips
begin, end, cross the image's edges or lie beyond them."""

import pytest

pytestmark = pytest.mark.gpu


def _solve(L, H, W, T, method, accelerate, engine, truth, pr):
    import torch
    from pnp_sci import _lib
    p = _lib.Params()
    L.scigap_default_params(p, H, W, T)
    p.method = _lib.METHOD_ADMM if method == "admm" else _lib.METHOD_GAP
    p.accelerate = 1 if accelerate else 0
    p.iters, p.tv_weight, p.tv_iter_max, p.tile_rows, p.engine = 4, 0.1, 5, 8, engine
    y, phi, ps = (torch.as_tensor(a, device="cuda").contiguous()
                  for a in (pr.y, pr.mask_thw, pr.phi_sum))
    tr = torch.as_tensor(pr.truth, device="cuda").permute(2, 0, 1).contiguous() if truth else None
    nb = L.scigap_solve_workspace_bytes(p)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    x = torch.empty((T, H, W), device="cuda")
    err = torch.zeros(4, dtype=torch.float64, device="cuda")
    stats = torch.zeros(4, dtype=torch.int32, device="cuda")
    _lib.check(L.scigap_solve(p, y.data_ptr(), phi.data_ptr(), ps.data_ptr(), None, x.data_ptr(),
                              tr.data_ptr() if truth else None, err.data_ptr() if truth else None,
                              stats.data_ptr(), ws.data_ptr(), nb, _lib.stream_ptr()))
    return x.cpu(), err.cpu(), stats.cpu()


@pytest.mark.parametrize("H,W", [
    (1, 1), (1, 130), (130, 1), (3, 2), (4, 127), (5, 128), (20, 129), (23, 130), (24, 131),
    (25, 248), (28, 249), (29, 250), (47, 127), (48, 128), (49, 256), (52, 317), (53, 368),
    (71, 369), (72, 376), (97, 490)])
@pytest.mark.parametrize("method,accelerate,truth", [("gap", True, False), ("gap", False, True),
                                                     ("admm", True, False), ("admm", True, True)])
def test_strip_bodies_match_whole_tiles(gpu, H, W, method, accelerate, truth):
    import torch
    from pnp_sci.synthetic import make_problem
    pr = make_problem(H, W, 3, seed=H * 1000 + W, p=0.5)
    x, err, stats = _solve(gpu, H, W, 3, method, accelerate, 1, truth, pr)
    xw, errw, statsw = _solve(gpu, H, W, 3, method, accelerate, 3, truth, pr)
    assert torch.equal(x, xw)
    assert torch.equal(stats, statsw)
    # (fp64 sums of the same fp32 terms, added by atomics in any order)
    assert torch.allclose(err, errw, rtol=1e-12, atol=0)


@pytest.mark.parametrize("H,W,T", [(1, 1, 1), (5, 7, 3), (24, 130, 2), (70, 317, 5)])
@pytest.mark.parametrize("method,engine,iters,n", [("gap", 0, 7, 5), ("admm", 6, 7, 5),
                                                   ("gap", 1, 4, 3), ("admm", 0, 1, 5),
                                                   ("gap", 3, 3, 5), ("gap", 0, 3, 9),
                                                   ("gap", 0, 2, 1), ("gap", 0, 0, 5)])
def test_solves_that_share_launches_match_single_ones(gpu, H, W, T, method, engine, iters, n):
    """Three solves together against one at a time, with a loose exit tolerance
    (frames stop early) and with a truth.  The frame split may differ, so yb may
    round differently: 1e-5, a few hundred fp32 roundings over the iterations."""
    import torch
    from pnp_sci import _lib
    from pnp_sci.synthetic import make_problem
    prs = [make_problem(H, W, T, seed=H + W + i, p=0.5) for i in range(3)]
    cat = lambda f: torch.stack([torch.as_tensor(f(q), device="cuda") for q in prs])  # noqa: E731
    y, phi, ps, tr = (cat(f).contiguous() for f in (lambda q: q.y, lambda q: q.mask_thw,
                                                    lambda q: q.phi_sum, lambda q: q.truth_thw))
    p = _lib.Params()
    gpu.scigap_default_params(p, H, W, T)
    p.method = _lib.METHOD_ADMM if method == "admm" else _lib.METHOD_GAP
    p.iters, p.tv_iter_max, p.tv_eps, p.engine = iters, n, 2e-2, engine
    x = torch.empty_like(phi)
    err = torch.zeros((3, max(iters, 1)), dtype=torch.float64, device="cuda")
    stats = torch.zeros((3, max(iters, 1)), dtype=torch.int32, device="cuda")
    nb = gpu.scigap_solve_many_workspace_bytes(p, 3)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    _lib.check(gpu.scigap_solve_many(p, 3, y.data_ptr(), phi.data_ptr(), ps.data_ptr(), None,
                                     x.data_ptr(), tr.data_ptr(), err.data_ptr(),
                                     stats.data_ptr(), ws.data_ptr(), nb, _lib.stream_ptr()))
    for i in range(3):
        # (single solves want 8-byte aligned arrays: copies of the slices)
        yi, fi, si, ti = (v[i].clone() for v in (y, phi, ps, tr))
        xi, ei = torch.empty_like(fi), torch.zeros_like(err[i])
        sti = torch.zeros_like(stats[i])
        _lib.check(gpu.scigap_solve(p, yi.data_ptr(), fi.data_ptr(), si.data_ptr(), None,
                                    xi.data_ptr(), ti.data_ptr(), ei.data_ptr(), sti.data_ptr(),
                                    ws.data_ptr(), nb, _lib.stream_ptr()))
        assert torch.equal(stats[i], sti)
        assert float((x[i] - xi).abs().max()) <= 1e-5
        assert torch.allclose(err[i], ei, rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("projmeth,direction", [("gap", "plain"), ("admm", "updown"),
                                                ("gap", "downup")])
@pytest.mark.parametrize("H,W,T,F", [(24, 130, 3, 1), (7, 9, 2, 5), (33, 40, 4, 3)])
def test_coded_frame_blocks_together_match_one_at_a_time(gpu, capsys, monkeypatch, projmeth,
                                                         direction, H, W, T, F):
    """The driver with groups of blocks against the same driver one block at a
    time: results, progress lines and their order."""
    import numpy as np
    import pnp_sci
    from pnp_sci import pnp_sci_algo
    from pnp_sci.synthetic import truth_video
    rng = np.random.default_rng(H + F)
    mask = (rng.random((H, W, T)) < 0.5).astype(np.float32)
    orig = (truth_video(rng, H, W, T * F) * 255).astype(np.float32)
    meas = np.stack([(orig[..., f * T:(f + 1) * T] * mask).sum(2) for f in range(F)], -1)
    v0 = rng.random((H, W, T * F)).astype(np.float32)
    for warm in (None, v0):
        runs = []
        for voxels in (1 << 25, 0):
            monkeypatch.setattr(pnp_sci_algo, "_SHARED_SOLVE_VOXELS", voxels)
            runs.append((pnp_sci.admmdenoise_cacti(
                meas, mask, lambda v: pnp_sci.A_(v, mask), lambda v: pnp_sci.At_(v, mask),
                projmeth=projmeth, v0=warm, orig=orig, nframe=F, MAXB=255.,
                maskdirection=direction, denoiser="tv", iter_max=6), capsys.readouterr().out))
        (x, _, p, s, pa), text = runs[0]
        (xw, _, pw, sw, paw), textw = runs[1]
        assert x.shape == xw.shape and x.dtype == xw.dtype and x.flags.c_contiguous
        assert np.max(np.abs(x - xw)) <= 1e-5
        assert np.allclose(p, pw, atol=1e-2) and np.allclose(s, sw, atol=1e-4)
        assert np.allclose(pa, paw, atol=1e-2)
        strip = lambda t: [line.split("PSNR")[0] for line in t.splitlines()]  # noqa: E731
        assert strip(text) == strip(textw)
