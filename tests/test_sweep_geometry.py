"""How the deep TV cuts images into strips, checked on the CPU: tests/host/sweep_rows.hip
evaluates the rules of sweep.h for the sizes at which test_gpu_sweep_sizes.py runs
them, so that those keep meeting every height of a strip, with the exit test in
the waves and as a launch of its own."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# (H, W, T, n_iter_max): rows of a strip, strips of a frame in each pass
SIZES = {
    (203, 130, 2, 8): (8, [52, 52]),
    (520, 518, 2, 8): (8, [325, 325]),
    (1030, 130, 2, 30): (8, [258] * 5),
    (203, 130, 301, 30): (16, [26] * 5),
    (310, 700, 16, 30): (16, [140] * 4 + [120]),   # the last pass within the limit
    (700, 700, 9, 30): (16, [308] * 4 + [264]),
    (131, 150, 600, 8): (32, [10, 10]),
    (203, 130, 120, 30): (32, [14] * 5),
    (1030, 700, 9, 30): (32, [231] * 4 + [198]),
    (515, 518, 41, 30): (64, [45] * 5),
    (1500, 600, 20, 30): (64, [144] * 5),
}


def test_sizes_meet_every_strip_height_and_both_exit_tests(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is needed to build the host-side check")
    exe = str(tmp_path / "sweep_rows")
    cmd = [hipcc, "--offload-arch=gfx950", "-O2", "-std=c++17",
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "sci-algorithms_amd", "csrc"),
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-Wno-unused-command-line-argument", os.path.join(HERE, "host", "sweep_rows.hip"),
           "-o", exe]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    args = [str(v) for size in SIZES for v in size]
    run = subprocess.run([exe] + args, capture_output=True, text=True, timeout=300)
    lines = run.stdout.split("\n")
    limit = int(lines[len(SIZES)].split()[1])
    seen = set()
    for line, (size, (rows, strips)) in zip(lines, SIZES.items()):
        got = [int(v) for v in line.split()]
        assert (got[0], got[1:]) == (rows, strips), size
        seen |= {(rows, s > limit) for s in strips}
    assert seen == {(r, many) for r in (8, 16, 32, 64) for many in (False, True)}
