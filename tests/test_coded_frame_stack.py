"""Shapes of the grouped solves, without a GPU: the coded-frame driver hands
solve_device one plane, warm start and truth per block of a group, by the rules
of an index into the measurement stack, and solve_device refuses tensors whose
leading dimensions differ before any device work."""

import types

import numpy as np
import pytest
import torch

from pnp_sci import pnp_sci_algo as algo

H, W, T = 16, 12, 2


@pytest.fixture
def solves(monkeypatch):
    """Device helpers on the CPU; returns the list of solve_device calls."""
    calls = []
    dev = lambda a, name="": torch.as_tensor(np.array(a, dtype=np.float32))  # noqa: E731
    monkeypatch.setattr(algo, "to_device", dev)
    monkeypatch.setattr(algo, "to_device_thw", lambda a, name="": dev(a).permute(2, 0, 1).contiguous())
    monkeypatch.setattr(algo, "hwt_to_thw", lambda v: v.permute(2, 0, 1).contiguous())
    monkeypatch.setattr(algo, "thw_to_hwt", lambda v: v.permute(1, 2, 0).contiguous())
    monkeypatch.setattr(algo, "to_host_like", lambda t, like: t.numpy().astype(np.float32))
    lib = types.SimpleNamespace(scigap_phi_sum=lambda *a: 0)
    monkeypatch.setattr(algo, "_lib", types.SimpleNamespace(
        lib=lambda: lib, check=lambda rc: None, stream_ptr=lambda stream=None: None))

    def solve(y, phi, phi_sum, **kw):
        calls.append((y, phi, phi_sum, kw))
        # the "result" of a block is its measurement in every frame
        return y[..., None, :, :].expand(phi.shape).contiguous(), None, None

    monkeypatch.setattr(algo, "solve_device", solve)
    return calls


def _run(meas, nframe, iframe=0, **kw):
    mask = np.ones((H, W, T), np.float32)
    op = types.SimpleNamespace(scigap_phi=torch.ones(T, H, W))
    return algo.admmdenoise_cacti(meas, mask, op, op, projmeth="gap", nframe=nframe, iframe=iframe,
                                  denoiser="tv", iter_max=2, **kw)


def _stack(n):
    return np.random.default_rng(n).random((H, W, n)).astype(np.float32)


@pytest.mark.parametrize("container", [np.asarray, torch.as_tensor])
@pytest.mark.parametrize("n,nframe,iframe", [(3, 4, 0), (3, 3, 1), (3, 2, 2), (1, 2, 0), (3, 2, 3),
                                             (3, 2, 7), (3, 2, -4), (2, 2, -3)])
def test_stack_without_all_the_blocks_raises_index_error(solves, container, n, nframe, iframe):
    with pytest.raises(IndexError):
        _run(container(_stack(n)), nframe, iframe)
    assert not solves


def test_short_truth_and_warm_start_are_refused(solves):
    meas = _stack(3)
    for short in (dict(orig=_stack(3 * T - 1)), dict(v0=_stack(2 * T)), dict(v0=_stack(3 * T - 1)),
                  dict(v0=_stack(3 * T).transpose(1, 0, 2))):
        with pytest.raises((ValueError, IndexError, RuntimeError)):
            _run(meas, 3, **short)
    with pytest.raises(IndexError):
        _run(meas, 4, orig=_stack(4 * T))
    assert not solves


@pytest.mark.parametrize("n,nframe,iframe", [(3, 3, 0), (5, 2, 3), (3, 1, 2), (3, 2, -2), (3, 2, -3),
                                             (3, 3, -1), (3, 1, -1)])
def test_blocks_are_the_planes_an_index_names(solves, n, nframe, iframe):
    meas = _stack(n)
    x = _run(meas, nframe, iframe)[0]
    assert len(solves) == 1
    y, phi, psd, _ = solves[0]
    lead = (nframe,) if nframe > 1 else ()
    assert tuple(y.shape) == lead + (H, W) and tuple(phi.shape) == lead + (T, H, W)
    assert tuple(psd.shape) == lead + (H, W)
    for k in range(nframe):
        for t in range(T):
            assert np.array_equal(x[..., k * T + t], meas[..., iframe + k])


def test_solve_device_refuses_leading_dimensions_that_differ():
    full = dict(y=torch.ones(3, H, W), phi=torch.ones(3, T, H, W), phi_sum=torch.ones(3, H, W))
    bad = [dict(y=torch.ones(2, H, W)), dict(y=torch.ones(H, W)), dict(phi_sum=torch.ones(H, W)),
           dict(phi_sum=torch.ones(1, H, W)), dict(x0=torch.ones(T, H, W)),
           dict(truth=torch.ones(2, T, H, W)), dict(y=torch.ones(1, H, W).expand(3, H, W)),
           dict(phi=torch.ones(1, 3, T, H, W))]
    for change in bad:
        kw = dict(full, **change)
        with pytest.raises(ValueError):
            algo.solve_device(kw.pop("y"), kw.pop("phi"), kw.pop("phi_sum"), iters=1, **kw)
