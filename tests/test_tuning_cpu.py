"""The part of a batch that the autotuner times (no GPU): bounded, whatever the shots, and with as full a queue."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHUNK = 256
QUEUE = 8192 * 64 * 64  # pixels of a full queue


@pytest.fixture(scope="module")
def cut(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the ROCm headers")
    exe = str(tmp_path_factory.mktemp("tuning") / "tuning_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-unknown-pragmas",
                    os.path.join(ROOT, "tests", "host_asan", "tuning_check.cpp"), "-o", exe], check=True)

    def run(npix, cap, offsets):
        text = "%r %r %d %s\n" % (float(npix), float(cap), len(offsets) - 1, " ".join(str(int(o)) for o in offsets))
        return np.array(subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split(),
                        dtype=np.int64)

    return run


SHOTS = [
    (512**2, np.random.default_rng(1).integers(300, 1001, 10000)),  # many small shots
    (256**2, np.full(100000, 200)),
    (256**2, np.full(100000, 3)),
    (64**2, np.random.default_rng(2).integers(0, 3, 50000)),        # empty ones among them
    (1024**2, np.array([1000000, 1000000])),
    (1024**2, np.array([2000000])),
    (256**2, np.random.default_rng(3).integers(1000, 50001, 64)),
    (2048**2, np.full(500, 100000)),
    (4096**2, np.full(300, 257)),
    (256**2, np.full(3000, 100000)),
    (100, np.full(200000, 5000)),
    (1, np.array([0])),
    (1, np.array([7])),
]


@pytest.mark.parametrize("cap", [2e11, 2e10])
@pytest.mark.parametrize("npix,sizes", SHOTS)
def test_the_timed_part(cut, npix, sizes, cap):
    off = np.concatenate([[0], np.cumsum(sizes)])
    t = cut(npix, cap, off)
    ts = len(t) - 1
    kept = np.diff(t)
    assert 1 <= ts <= len(sizes) and t[0] == 0
    assert np.all(kept >= 0) and np.all(kept <= sizes[:ts])
    # at most the cap, and a chunk for each shot of a full queue
    assert t[-1] * npix <= cap + (QUEUE + npix) * CHUNK
    # as many items as the whole batch has, up to a full queue
    assert ts * npix >= min(QUEUE, len(sizes) * npix)
    if off[-1] * npix <= cap:
        assert np.array_equal(t, off)
    else:
        # no less than a quarter of the cap is timed (a batch of whole, equal shares)
        assert t[-1] * npix >= 0.25 * min(cap, off[-1] * npix)
        if ts * npix <= QUEUE:  # the cut ones: the same share of each
            big = sizes[:ts] > 4 * CHUNK
            assert np.all(np.abs(kept[big] / sizes[:ts][big] - kept[big].sum() / sizes[:ts][big].sum()) <=
                          CHUNK / sizes[:ts][big])
