"""The autotuner's file of choices, without a GPU: a TV depth is used in place of
the row sweeps only if it was timed against them."""

import os
import subprocess
import sys

import pytest

from pnp_sci.build import LIB_PATH

# The choice for depth 0 (an internal function, by its C++ name):
# tuned_tv_depth(int64_t H, int64_t W, int64_t T, int n, bool sweep_fits).
CODE = """
import ctypes, sys
import torch
lib = ctypes.CDLL(sys.argv[1])
f = lib._ZN6scigap14tuned_tv_depthElllib
f.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_bool]
print([f(64, 96, int(t), 30, fits) for t in sys.argv[2].split(",") for fits in (True, False)])
"""


def _choices(tmp_path, lines, frames):
    path = tmp_path / "choices.txt"
    path.write_text("".join("%s\n" % line for line in lines))
    env = dict(os.environ, SCIGAP_TUNE_CACHE=str(path))
    r = subprocess.run([sys.executable, "-c", CODE, LIB_PATH, ",".join(map(str, frames))], env=env,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return eval(r.stdout.strip().splitlines()[-1])


def test_depths_of_older_files_do_not_replace_the_sweeps(tmp_path):
    if not os.path.exists(LIB_PATH):
        pytest.fail("libscigap.so is not built (run __graft_entry__.build())")
    # kind H W T a b tile_rows engine depth ms; a TV entry's engine column is 1
    # where the depth was faster than the sweeps
    lines = ["1 64 96 2 0 30 0 0 4 0.100000",   # written before there were sweeps
             "1 64 96 3 0 30 0 0 0 0.100000",   # the sweeps were faster, no depth kept
             "1 64 96 4 0 30 0 1 5 0.100000",   # a depth that beat the sweeps
             "1 64 96 5 0 30 0 0 2 0.100000"]   # the sweeps were faster
    got = _choices(tmp_path, lines, (1, 2, 3, 4, 5))
    # sweeps (0) unless beaten; in a workspace too small for them the depth, 6 untuned
    assert got == [0, 6, 0, 4, 0, 6, 5, 5, 0, 2]
