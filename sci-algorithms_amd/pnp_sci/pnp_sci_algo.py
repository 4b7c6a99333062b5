"""GAP-TV / ADMM-TV reconstruction for video SCI on MI355X.

Drop-in mirror of the TV path of ``PnP_SCI/python/pnp_sci_algo.py``:
``gap_denoise`` (:536-706), ``admm_denoise`` (:708-864),
``gap_denoise_bayer`` (:20-265), ``admmdenoise_cacti`` (:479-534) and the legacy ``GAP_TV_rec`` /
``ADMM_TV_rec`` (:866-907), plus the clipped ADMM of
``joint_pnp_sci_algo.py:502-663`` as ``admm_denoise(..., clip=True)``.
Same argument names, defaults, return tuples and error behaviour; every outer
iteration runs as fused HIP kernels (scigap_solve) in fp32.

Differences a caller can observe:
  * Arithmetic is fp32 whatever the input dtype; results are returned in the
    input's dtype and container (NumPy or torch).
  * ``denoiser`` must be 'tv'.  The deep and wavelet denoisers of the
    reference are not part of this path and raise NotImplementedError.
  * ``multichannel=False`` (3-D TV over (H,W,T)) is not implemented.
  * The operators ``A``/``At`` must be the SCI mask operators (any callables
    equal to ``A_(x, Phi)`` / ``At_(y, Phi)``): the mask is recovered once as
    ``At(ones)`` and checked against ``A`` on a random probe.
"""

from __future__ import annotations

import math
import time

import numpy as np

from . import _lib
from .device import hwt_to_thw, is_torch, thw_to_hwt, to_device, to_device_thw, to_host_like
from .metrics import psnr_frames, ssim_frames

__all__ = ["gap_denoise", "admm_denoise", "admmdenoise_cacti", "GAP_TV_rec", "ADMM_TV_rec",
           "gap_denoise_bayer", "recover_mask", "solve_device"]

_OTHER_DENOISERS = ("wavelet", "ffdnet", "fastdvdnet", "vnlnet")


def _torch():
    import torch
    return torch


# ---------------------------------------------------------------------------
# Operator recovery
# ---------------------------------------------------------------------------

def recover_mask(A, At, y, check: bool = True):
    """Device (T,H,W) mask behind the opaque operators A, At.

    ``At_(y, Phi)`` is ``y*Phi`` per frame, so ``At(ones) = Phi`` exactly
    (utils.py:17-26).  ``A`` is then checked on a random probe against
    ``sum_t x*Phi``; a mismatch means the callables are not SCI operators.
    """
    phi = getattr(At, "scigap_phi", None)
    if phi is not None:
        return phi
    torch = _torch()
    ones = torch.ones_like(y) if is_torch(y) else np.ones(np.shape(y), dtype=np.asarray(y).dtype)
    mask_hwt = At(ones)
    if len(np.shape(mask_hwt)) != 3 or tuple(np.shape(mask_hwt)[:2]) != tuple(np.shape(y)):
        raise ValueError("At(ones) must return an (H,W,T) mask, got shape %s"
                         % (tuple(np.shape(mask_hwt)),))
    phi = to_device_thw(mask_hwt, "At(ones)")
    if check:
        H, W, T = np.shape(mask_hwt)
        rng = np.random.default_rng(12345)
        probe = rng.random((H, W, T), dtype=np.float32)
        if is_torch(y):
            probe_in = torch.from_numpy(probe).to(device=y.device, dtype=y.dtype)
        else:
            probe_in = probe.astype(np.asarray(y).dtype, copy=False)
        got = to_device(A(probe_in), "A(probe)")
        pd = to_device_thw(probe, "probe")
        want = torch.empty((H, W), dtype=torch.float32, device=pd.device)
        L = _lib.lib()
        _lib.check(L.scigap_forward(pd.data_ptr(), phi.data_ptr(), want.data_ptr(), H, W, T,
                                    _lib.stream_ptr()))
        scale = float(want.abs().max().item()) + 1e-30
        if got.shape != want.shape or float((got - want).abs().max().item()) > 1e-4 * scale:
            raise ValueError("A and At are not the SCI forward model and its transpose "
                             "(A(x) != sum_t x*At(1)); only A_(x,Phi)/At_(y,Phi) are supported")
    return phi


# ---------------------------------------------------------------------------
# Device solve
# ---------------------------------------------------------------------------

def solve_device(y, phi, phi_sum, *, method="gap", iters=50, _lambda=1.0, accelerate=True,
                 gamma=0.01, clip=False, tv_weight=0.1, tv_iter_max=5, tv_eps=2e-4,
                 x0=None, truth=None, tv_weight_decay=1.0, gamma_decay=1.0, stream=None):
    """One GAP/ADMM-TV solve on device tensors already in library layout.

    y, phi_sum: (H,W) float32; phi, x0, truth: (T,H,W) float32, all on the
    device.  Returns (x (T,H,W), sq_err (iters,) fp64 or None,
    early_exits (iters,) int32).  With a leading dimension on every tensor,
    that many solves share their launches (scigap_solve_many) and the results
    have it too.
    """
    torch = _torch()
    lead = tuple(phi.shape[:-3])
    T, H, W = phi.shape[-3:]
    if lead:  # the solves' arrays are addressed by their distance: all of it must be there
        for v, want in ((y, (H, W)), (phi, (T, H, W)), (phi_sum, (H, W)), (x0, (T, H, W)),
                        (truth, (T, H, W))):
            if v is not None and (len(lead) > 1 or tuple(v.shape) != lead + want or
                                  not v.is_contiguous()):
                raise ValueError("solves that share launches need contiguous tensors with one "
                                 "leading dimension: got %s, expected %s"
                                 % (tuple(v.shape), lead + want))
    for name, v, n in (("y", y, H * W), ("phi_sum", phi_sum, H * W), ("x0", x0, T * H * W),
                       ("truth", truth, T * H * W)):
        if v is not None and v.numel() < n:  # would be read past its end
            raise ValueError("%s has %d elements, a %dx%dx%d solve reads %d"
                             % (name, v.numel(), H, W, T, n))
    p = _lib.Params()
    L = _lib.lib()
    L.scigap_default_params(p, H, W, T)
    p.method = _lib.METHOD_ADMM if method == "admm" else _lib.METHOD_GAP
    p.accelerate = 1 if accelerate else 0
    p.clip = 1 if clip else 0
    p.iters = int(iters)
    p.lambda_ = float(_lambda)
    p.gamma = float(gamma)
    p.tv_weight = float(tv_weight)
    p.tv_eps = float(tv_eps)
    p.tv_iter_max = int(tv_iter_max)
    p.tv_weight_decay = float(tv_weight_decay)
    p.gamma_decay = float(gamma_decay)
    solves = lead[0] if lead else 1
    nbytes = L.scigap_solve_many_workspace_bytes(p, solves)
    if nbytes == 0:
        raise _lib.ScigapError(-1, L.scigap_last_error().decode(errors="replace"))
    dev = phi.device
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    x = torch.empty(phi.shape, dtype=torch.float32, device=dev)
    sq = torch.empty(lead + (max(iters, 1),), dtype=torch.float64,
                     device=dev) if truth is not None else None
    stats = torch.empty(lead + (max(iters, 1),), dtype=torch.int32, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None  # noqa: E731
    args = (ptr(y), ptr(phi), ptr(phi_sum), ptr(x0), ptr(x), ptr(truth), ptr(sq), ptr(stats),
            ptr(ws), nbytes, _lib.stream_ptr(stream))
    _lib.check(L.scigap_solve_many(p, solves, *args) if lead else L.scigap_solve(p, *args))
    return x, (sq[..., :iters] if sq is not None else None), stats[..., :iters]


# ---------------------------------------------------------------------------
# Reference-shaped entry points
# ---------------------------------------------------------------------------

def _check_denoiser(denoiser, multichannel):
    d = denoiser.lower()
    if d in _OTHER_DENOISERS:
        raise NotImplementedError("denoiser %r is outside the GAP/ADMM-TV path" % denoiser)
    if d != "tv":
        raise ValueError('Unsupported denoiser {}!'.format(denoiser))
    if not multichannel:
        raise NotImplementedError("multichannel=False (3-D TV) is not implemented")


def _stages(sigma, iter_max):
    """Noise-level stages (pnp_sci_algo.py:628-631); for TV they only add up."""
    if not isinstance(sigma, list):
        sigma = [sigma]
    if not isinstance(iter_max, list):
        iter_max = [iter_max] * len(sigma)
    return sigma, iter_max


def _psnr_from_sq(sq, n):
    out = []
    for s in sq:
        mse = s / n
        out.append(100 if mse == 0 else 20 * math.log10(1.0 / math.sqrt(mse)))
    return out


def _print_progress(tag, psnr_all, sigma, iter_max):
    """Progress lines of pnp_sci_algo.py:683-696 (every fifth iteration)."""
    k = 0
    for idx, nsig in enumerate(sigma):
        for _ in range(iter_max[idx]):
            if (k + 1) % 5 == 0 and k < len(psnr_all):
                if nsig is not None:
                    if nsig < 1:
                        print('  {0}-TV iteration {1: 3d}, sigma {2: 3g}/255, '
                              'PSNR {3:2.2f} dB.'.format(tag, k + 1, nsig * 255, psnr_all[k]))
                    else:
                        print('  {0}-TV iteration {1: 3d}, sigma {2: 3g}, '
                              'PSNR {3:2.2f} dB.'.format(tag, k + 1, nsig, psnr_all[k]))
                else:
                    print('  {0}-TV iteration {1: 3d}, PSNR {2:2.2f} dB.'.format(
                        tag, k + 1, psnr_all[k]))
            k += 1


def _run(method, y, Phi_sum, A, At, *, _lambda, accelerate, gamma, clip, denoiser, iter_max,
         sigma, tv_weight, tv_iter_max, multichannel, x0, X_orig, show_iqa, tvm="tv_chambolle",
         tv_weight_decay=1.0, gamma_decay=1.0, tv_eps=2e-4):
    _check_denoiser(denoiser, multichannel)
    if tvm in ("ITV3D_FGP", "ITV2D_cham") and method == "gap":
        # pnp_sci_algo.py:651-654 call functions that are never defined.
        raise NameError("name of the TV denoiser for tvm=%r is not defined" % tvm)
    if tvm != "tv_chambolle" and method == "gap":
        # pnp_sci_algo.py:655-658: TypeError raised and printed, TV skipped.
        print("Exception: ", repr(TypeError("no such tv denoiser")))
        tv_iter_max = 1  # identity denoiser
    sigma, iter_max = _stages(sigma, iter_max)
    iters = int(sum(iter_max))
    torch = _torch()
    group = y if isinstance(y, _Blocks) else None
    phi = recover_mask(A, At, y)
    T, H, W = phi.shape
    yd = hwt_to_thw(to_device(y.array, "y")) if group else to_device(y, "y")
    psd = to_device(Phi_sum, "Phi_sum")
    lead = (group.n,) if group else ()
    if tuple(yd.shape) != lead + (H, W) or tuple(psd.shape) != (H, W):
        raise ValueError("y and Phi_sum must be (H,W) = (%d,%d)" % (H, W))

    def volume(v, name):  # (T,H,W), or the group's [block][T][H][W]
        if not group:
            return to_device_thw(v, name)
        vd = to_device_thw(v.array, name)
        if tuple(vd.shape) != (group.n * T, H, W):
            raise ValueError("%s must hold %d frames of %dx%d" % (name, group.n * T, H, W))
        return vd.reshape(group.n, T, H, W)

    x0d = volume(x0, "x0") if x0 is not None else None
    want_iqa = show_iqa and X_orig is not None
    truth = volume(X_orig, "X_orig") if X_orig is not None else None
    n = group.n if group else 1
    if group:
        phi = phi.expand(n, T, H, W).contiguous()
        psd = psd.expand(n, H, W).contiguous()
    x, sq, _ = solve_device(yd, phi, psd, method=method, iters=iters, _lambda=_lambda,
                            accelerate=accelerate, gamma=gamma, clip=clip, tv_weight=tv_weight,
                            tv_iter_max=tv_iter_max, tv_eps=tv_eps, x0=x0d,
                            truth=truth if want_iqa else None,
                            tv_weight_decay=tv_weight_decay, gamma_decay=gamma_decay)
    psnr_all = []
    if want_iqa:
        sq = sq.cpu().tolist()
        psnr_all = [_psnr_from_sq(e, T * H * W) for e in (sq if group else [sq])]
        _print_progress(method.upper(), psnr_all[0], sigma, iter_max)
    psnr_, ssim_ = [], []
    x, truth = (None if v is None else v.reshape(n * T, H, W) for v in (x, truth))
    if X_orig is not None:
        psnr_ = psnr_frames(truth, x)
        ssim_ = ssim_frames(truth, x)  # raises for frames under 7x7, as the reference does
    for i in range(1, n):
        group.on_block(i)
        if want_iqa:
            _print_progress(method.upper(), psnr_all[i], sigma, iter_max)
    out = to_host_like(thw_to_hwt(x), y.array if group else y)
    return out, psnr_, ssim_, (psnr_all if group else psnr_all[0] if psnr_all else [])


class _Blocks:
    """The arrays of `n` coded-frame blocks of one shape and mask, side by side in
    the last dimension, which `_run` solves together (as `y`, `x0` and
    `X_orig`).  Its results are side by side too, psnr_all a list per block;
    ``on_block(i)`` runs before the progress lines of block i > 0."""

    def __init__(self, array, n, on_block=None):
        self.array, self.n, self.on_block = array, n, on_block


def gap_denoise(y, Phi_sum, A, At, _lambda=1, accelerate=True,
                denoiser='tv', iter_max=50, noise_estimate=False, sigma=None,
                tv_weight=0.1, tv_iter_max=5, multichannel=True, x0=None,
                X_orig=None, model=None, show_iqa=True, tvm='tv_chambolle'):
    """GAP-TV (pnp_sci_algo.py:536-706).  Returns (x, psnr_, ssim_, psnr_all)."""
    return _run("gap", y, Phi_sum, A, At, _lambda=_lambda, accelerate=accelerate, gamma=0.0,
                clip=False, denoiser=denoiser, iter_max=iter_max, sigma=sigma,
                tv_weight=tv_weight, tv_iter_max=tv_iter_max, multichannel=multichannel,
                x0=x0, X_orig=X_orig, show_iqa=show_iqa, tvm=tvm)


def admm_denoise(y, Phi_sum, A, At, _lambda=1, gamma=0.01,
                 denoiser='tv', iter_max=50, noise_estimate=False, sigma=None,
                 tv_weight=0.1, tv_iter_max=5, multichannel=True, x0=None, model=None,
                 X_orig=None, show_iqa=True, clip=False):
    """ADMM-TV (pnp_sci_algo.py:708-864).  ``clip=True`` is the variant of
    joint_pnp_sci_algo.py:502-663 (theta clipped to [0,1] after TV; that
    function defaults gamma to 0).  Returns (x, psnr_, ssim_, psnr_all)."""
    return _run("admm", y, Phi_sum, A, At, _lambda=_lambda, accelerate=False, gamma=gamma,
                clip=clip, denoiser=denoiser, iter_max=iter_max, sigma=sigma,
                tv_weight=tv_weight, tv_iter_max=tv_iter_max, multichannel=multichannel,
                x0=x0, X_orig=X_orig, show_iqa=show_iqa)


# Sub-grids of up to this many voxels (H*W*T) are solved together.  A larger one
# fills the GPU by itself, and one workspace is enough for all four in turn.
# (20 iterations, together / in turn: 0.73 / 1.6 ms for sub-grids of 256x256x8,
# 1.40 / 2.34 of 512x512x10, 7.8 / 8.7 of 2048x1024x8, 10.0 / 9.3 of
# 1024x1024x20, 14.7 / 12.9 of 2048x2048x8.)
_SHARED_SOLVE_VOXELS = 1 << 24


def gap_denoise_bayer(y_bayer, Phi_bayer, _lambda=1, accelerate=True, denoiser='tv',
                      iter_max=50, noise_estimate=True, sigma=None, tv_weight=0.1,
                      tv_iter_max=5, multichannel=True, x0_bayer=None, X_orig=None,
                      model=None, show_iqa=True):
    """GAP-TV on a Bayer-mosaic measurement (pnp_sci_algo.py:20-265).

    The reference splits the mosaic into its four 2x2 sub-grids, applies the
    GAP update to each and one multichannel TV to all nmask*4 sub-grid frames
    per outer iteration.  The TV is per frame, so the four sub-grids are
    independent GAP-TV solves, which share their launches here, and the
    results are written back into the mosaic.  y_bayer (H,W), Phi_bayer
    (H,W,nmask) with H and W even.  Returns (x_bayer, psnr_, ssim_, psnr_all),
    psnr_all on the whole mosaic per iteration.
    """
    torch = _torch()
    _check_denoiser(denoiser, multichannel)
    sigma, iter_max = _stages(sigma, iter_max)
    iters = int(sum(iter_max))
    yd = to_device(y_bayer, "y_bayer")
    phid = to_device(Phi_bayer, "Phi_bayer")
    nrow, ncol, nmask = phid.shape
    if nrow % 2 or ncol % 2 or tuple(yd.shape) != (nrow, ncol):
        raise ValueError("y_bayer (H,W) and Phi_bayer (H,W,nmask) need equal, even H and W")
    want_iqa = show_iqa and X_orig is not None
    truth = to_device(X_orig, "X_orig") if X_orig is not None else None
    x0d = to_device(x0_bayer, "x0_bayer") if x0_bayer is not None else None
    L = _lib.lib()
    H, W, T = nrow // 2, ncol // 2, nmask

    def split(v):  # (H,W[,T]) mosaic -> four sub-grids, frame-major
        v = v.reshape((H, 2, W, 2) + tuple(v.shape[2:]))
        v = v.permute((1, 3, 4, 0, 2) if v.dim() == 5 else (1, 3, 0, 2))
        return v.reshape((4,) + tuple(v.shape[2:])).contiguous()

    def take(v, c):  # one sub-grid, frame-major, in a tensor of its own
        v = v[c >> 1::2, c & 1::2].contiguous()
        return hwt_to_thw(v) if v.dim() == 3 else v

    def frame_sum(phi):
        ps = torch.empty((H, W), dtype=torch.float32, device=phid.device)
        _lib.check(L.scigap_phi_sum(phi.data_ptr(), ps.data_ptr(), H, W, T, _lib.stream_ptr()))
        return ps

    x0d = x0d[..., :nmask] if x0d is not None else None
    opts = dict(method="gap", iters=iters, _lambda=_lambda, accelerate=accelerate,
                tv_weight=tv_weight, tv_iter_max=tv_iter_max)
    if T * H * W <= _SHARED_SOLVE_VOXELS:
        phi_c = split(phid)
        x_c, sq, _ = solve_device(split(yd), phi_c, torch.stack([frame_sum(f) for f in phi_c]),
                                  x0=split(x0d) if x0d is not None else None,
                                  truth=split(truth) if want_iqa else None, **opts)
        sq_total = sq.sum(0) if sq is not None else None
        x_bayer = x_c.reshape(2, 2, T, H, W).permute(3, 0, 4, 1, 2).reshape(nrow, ncol, nmask)
    else:
        x_bayer = torch.empty((nrow, ncol, nmask), dtype=torch.float32, device=phid.device)
        sq_total = None
        for c in range(4):
            phi_c = take(phid, c)
            x_c, sq, _ = solve_device(take(yd, c), phi_c, frame_sum(phi_c),
                                      x0=take(x0d, c) if x0d is not None else None,
                                      truth=take(truth, c) if want_iqa else None, **opts)
            x_bayer[c >> 1::2, c & 1::2] = thw_to_hwt(x_c)
            if sq is not None:
                sq_total = sq if sq_total is None else sq_total + sq
    psnr_all = []
    if want_iqa:
        psnr_all = _psnr_from_sq(sq_total.cpu().tolist(), nrow * ncol * nmask)
        stages = [None] * len(sigma) if noise_estimate else sigma
        _print_progress("GAP", psnr_all, stages, iter_max)
    psnr_, ssim_ = [], []
    if X_orig is not None:
        xt = hwt_to_thw(x_bayer)
        tt = hwt_to_thw(truth)
        psnr_ = psnr_frames(tt, xt)
        ssim_ = ssim_frames(tt, xt)
    return to_host_like(x_bayer, Phi_bayer), psnr_, ssim_, psnr_all


def _planes(stack, lo, hi):
    """Planes lo to hi - 1 of the last axis by the rules of an index: beyond the
    stack is an IndexError (a slice would end short), negative counts from its
    end."""
    planes = [stack[..., i] for i in range(lo, hi)]
    if lo >= 0:
        return np.asarray(stack[..., lo:hi])
    return np.stack([np.asarray(v) for v in planes], axis=-1)


def admmdenoise_cacti(meas, mask, A, At, projmeth='admm', v0=None, orig=None,
                      iframe=0, nframe=1, MAXB=1., maskdirection='plain', **args):
    """Per-coded-frame driver (pnp_sci_algo.py:479-534).

    Divides measurement and truth by MAXB, computes Phi_sum once with the
    zero fix (:491-492, on the device), flips warm starts and results for
    'updown'/'downup' masks, and returns (x_, t_, psnr_, ssim_, psnrall_)
    with x_ float32 (H,W,nmask*nframe) and t_ the wall time in seconds.
    """
    torch = _torch()
    nmask = mask.shape[-1]
    md = to_device(mask, "mask")
    phi = hwt_to_thw(md)
    T, H, W = phi.shape
    msum = torch.empty((H, W), dtype=torch.float32, device=phi.device)
    L = _lib.lib()
    _lib.check(L.scigap_phi_sum(phi.data_ptr(), msum.data_ptr(), H, W, T, _lib.stream_ptr()))
    if getattr(At, "scigap_phi", None) is None:
        # Probe the caller's operators once, then reuse the recovered mask.
        phi = recover_mask(A, At, meas[..., iframe] if not is_torch(meas) else meas[..., iframe])

    class _Bound:
        scigap_phi = phi

        def __call__(self, v):  # pragma: no cover - never called by the solvers
            raise RuntimeError("bound operator is not callable")

    A_b, At_b = _Bound(), _Bound()
    x_ = np.zeros((*mask.shape[:-1], nmask * nframe), dtype=np.float32)
    psnr_, ssim_, psnrall_ = [], [], []
    begin = time.time()
    t_ = 0.0
    msum_host = msum.cpu().numpy()

    def announce(kf):
        print('%s-%s Reconstruction coded frame block %2d of %2d ...'
              % (projmeth.upper(), args['denoiser'].upper(), kf + 1, nframe))

    def flipped(kf):
        return ((maskdirection.lower() == 'updown' and (kf + iframe) % 2 == 1) or
                (maskdirection.lower() == 'downup' and (kf + iframe) % 2 == 0))

    # Blocks are independent solves of one shape: groups of them share their
    # launches (one block of 256x256x8 fills a tenth of the GPU) and their
    # transfers and conversions, which gain at larger sizes too (20 iterations
    # of two blocks of 2048x1024x8: 21 ms, one at a time 42).
    voxels = H * W * T
    per_group = 1
    if voxels <= 2 * _SHARED_SOLVE_VOXELS:
        per_group = max(1, min(4 * _SHARED_SOLVE_VOXELS // voxels, 4096 // T))
    for k0 in range(0, nframe, per_group):
        ks = range(k0, min(k0 + per_group, nframe))
        announce(k0)
        n, lo, hi = len(ks), iframe + k0, iframe + ks[-1] + 1
        pack = lambda v: v if n == 1 else _Blocks(  # noqa: E731
            v, n, lambda i: announce(k0 + i))
        orig_k = None
        if orig is not None:
            orig_k = pack(np.asarray(orig[..., lo * nmask:hi * nmask]) / MAXB)
        y_k = np.asarray(meas[..., lo] if n == 1 else _planes(meas, lo, hi)) / MAXB
        v0_k = None
        if v0 is not None:
            v0_k = np.asarray(v0[:, :, k0 * nmask:(ks[-1] + 1) * nmask])
            if any(flipped(kf) for kf in ks):
                v0_k = np.concatenate(
                    [v0_k[..., i * nmask:(i + 1) * nmask][..., ::-1 if flipped(kf) else 1]
                     for i, kf in enumerate(ks)], axis=-1)
            v0_k = pack(v0_k)
        if projmeth.lower() == 'admm':
            res = admm_denoise(pack(y_k), msum_host, A_b, At_b, x0=v0_k, X_orig=orig_k, **args)
        elif projmeth.lower() == 'gap':
            res = gap_denoise(pack(y_k), msum_host, A_b, At_b, x0=v0_k, X_orig=orig_k, **args)
        else:
            # The reference prints this and then reads the unbound result of
            # the solve (pnp_sci_algo.py:518-529): UnboundLocalError.
            print('Unsupported projection method %s' % projmeth.upper())
            raise UnboundLocalError("local variable 'x_k' referenced before assignment")
        x_k, psnr_k, ssim_k, psnrall_k = res
        if n == nframe and x_k.dtype == x_.dtype:
            x_ = x_k  # the whole result as it came from the device
        else:
            x_[..., k0 * nmask:(k0 + n) * nmask] = x_k
        for i, kf in enumerate(ks):
            part = slice(i * nmask, (i + 1) * nmask)
            step = -1 if flipped(kf) else 1
            if step < 0:
                cols = slice(kf * nmask, (kf + 1) * nmask)
                x_[..., cols] = x_[..., cols][..., ::-1].copy()
            psnr_.extend(psnr_k[part][::step])
            ssim_.extend(ssim_k[part][::step])
            psnrall_.append((psnrall_k if n == 1 else psnrall_k[i] if psnrall_k else [])[::step])
        t_ = time.time() - begin
    return x_, t_, psnr_, ssim_, psnrall_


def GAP_TV_rec(y, Phi, A, At, Phi_sum, maxiter, step_size, weight, row, col, ColT, X_ori):
    """Legacy accelerated GAP-TV with 30 TV iterations per call
    (pnp_sci_algo.py:866-882); ``A(f, Phi)``/``At(y, Phi)`` are not called,
    the mask ``Phi`` is used directly.  Progress printing is omitted."""
    x, _, _, _ = _run("gap", y, Phi_sum, _MaskOnly(Phi), _MaskOnly(Phi), _lambda=step_size,
                      accelerate=True, gamma=0.0, clip=False, denoiser='tv', iter_max=maxiter,
                      sigma=None, tv_weight=weight, tv_iter_max=30, multichannel=True, x0=None,
                      X_orig=None, show_iqa=False)
    return x


def ADMM_TV_rec(y, Phi, A, At, Phi_sum, maxiter, step_size, weight, row, col, ColT, eta, X_ori):
    """Legacy ADMM-TV (pnp_sci_algo.py:884-907): 30 TV iterations per call,
    TV weight x0.999 and eta x0.998 after every iteration."""
    x, _, _, _ = _run("admm", y, Phi_sum, _MaskOnly(Phi), _MaskOnly(Phi), _lambda=step_size,
                      accelerate=False, gamma=eta, clip=False, denoiser='tv', iter_max=maxiter,
                      sigma=None, tv_weight=weight, tv_iter_max=30, multichannel=True, x0=None,
                      X_orig=None, show_iqa=False, tv_weight_decay=0.999, gamma_decay=0.998)
    return x


class _MaskOnly:
    """Operator stand-in carrying an explicit (H,W,T) mask."""

    def __init__(self, Phi):
        self.scigap_phi = to_device_thw(Phi, "Phi")

    def __call__(self, v):  # pragma: no cover
        raise RuntimeError("mask-only operator is not callable")
