"""Tuning the deep TV with the workspace the header asks for: what depth 0 runs
afterwards is what the result says."""

import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,T,n", [(96, 200, 3, 14), (256, 256, 8, 30)])
def test_depth_zero_runs_the_fastest_of_sweeps_and_depths(gpu, H, W, T, n):
    import torch
    from pnp_sci import _lib, tune
    from pnp_sci.tv import tv_device
    tune.clear()
    img = torch.rand((T, H, W), device="cuda")
    untuned = tv_device(img, 0.1, 2e-4, n)
    out = torch.empty_like(img)
    nb = gpu.scigap_tv_workspace_bytes_depth(H, W, T, n, 1)  # as scigap.h says
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    r = _lib.TuneResult()

    def autotune(nbytes):
        return gpu.scigap_autotune_tv(img.data_ptr(), out.data_ptr(), H, W, T, 0.1, 2e-4, n,
                                      ws.data_ptr(), nbytes, _lib.stream_ptr(), ctypes.byref(r))

    def kernels():
        return set(_lib.kernel_profile(lambda: tv_device(img, 0.1, 2e-4, n)))

    try:
        _lib.check(autotune(nb))
        assert r.candidates == 6 and 1 <= r.tv_depth <= 6 and r.best_ms <= r.default_ms
        names = kernels()
        assert ("tv_pass" in names) == (r.best_ms == r.default_ms), (names, r.best_ms, r.default_ms)
        assert float((tv_device(img, 0.1, 2e-4, n) - untuned).abs().max()) <= 2e-5
        # a tune that fails keeps the choice
        assert autotune(16) != 0
        assert kernels() == names
    finally:
        tune.clear()
