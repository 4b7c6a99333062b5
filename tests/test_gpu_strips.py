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
