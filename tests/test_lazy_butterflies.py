"""The NTT kernels' butterflies and their compile-time bound schedule, on the
CPU: congruence and range of each butterfly with unbounded integers at the
edges of its stated inputs, and that no stage of any pass can exceed the lazy
range (LIM q, below 2^64)."""
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "fhe-mamba_amd", "csrc")
R64 = 1 << 64
# LIM 16 takes moduli in [2^33, 2^60), LIM 8 any below 2^61
MODS = {16: [(1 << 33) + 1, (1 << 45) + 59, (1 << 59) - 55, (1 << 59) + 21, (1 << 60) - 93],
        8: [(1 << 20) + 7, (1 << 60) + 33, (1 << 61) - 1]}


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("lazy") / "lazy_driver")
    subprocess.run([cxx, "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, os.path.join(HERE, "lazy_driver.cpp"), "-o", exe], check=True,
                   capture_output=True)
    return exe


def records(lim, x_bound, y_bound):
    rng = random.Random(x_bound * 100 + lim)
    out = []
    for q in MODS[lim]:
        xt, yt = min(x_bound * q, R64), min(y_bound * q, R64)
        for i in range(600):
            x = [0, 1, xt - 1, q, xt - q][i] if i < 5 else rng.randrange(xt)
            y = [yt - 1, 0, yt - 1, q - 1, yt - q][i] if i < 5 else rng.randrange(yt)
            out.append((q, x, y, [0, 1, q - 1, rng.randrange(q)][i % 4]))
    return out


def run(exe, args, recs):
    res = subprocess.run([exe, *map(str, args)], input=np.asarray(recs, dtype=np.uint64).tobytes(),
                         capture_output=True, check=True)
    return np.frombuffer(res.stdout, dtype=np.uint64).reshape(-1, 4).tolist()


@pytest.mark.parametrize("lim", [16, 8])
@pytest.mark.parametrize("red", [0, 1])
def test_forward_butterfly(driver, lim, red):
    bound = lim if red else lim - 4
    left = lim // 2 if red else bound
    recs = records(lim, bound, lim)
    for (q, x, y, w), (u, v, _, _) in zip(recs, run(driver, ["fwd", lim, red], recs)):
        assert u < (left + 4) * q and v <= (left + 4) * q and (left + 4) * q <= R64
        assert (u - x - y * w) % q == 0 and (v - x + y * w) % q == 0


@pytest.mark.parametrize("lim,bx,by", [(16, 1, 1), (16, 2, 2), (16, 4, 4), (16, 8, 4), (16, 8, 8),
                                       (8, 1, 1), (8, 2, 2), (8, 4, 4)])
def test_inverse_butterfly(driver, lim, bx, by):
    recs = records(lim, bx, by)
    for (q, x, y, w), (u, v, cx, cy) in zip(recs, run(driver, ["inv", lim, bx, by], recs)):
        assert u < cx * q and v < cy * q and max(cx, cy) <= lim // 2
        assert (u - x - y) % q == 0 and (v - (x - y) * w) % q == 0


@pytest.mark.parametrize("lim,b", [(16, 1), (16, 2), (16, 3), (16, 4), (16, 12), (8, 1), (8, 4),
                                   (8, 8)])
def test_forward_schedule(driver, lim, b):
    """Entering bounds as the butterfly test assumes them, and the bound each
    pass promises the next."""
    for stages in range(4, 13):
        text = subprocess.run([driver, "schedule", str(lim), str(b), str(stages)],
                              capture_output=True, check=True, text=True).stdout
        rows = [tuple(map(int, line.split())) for line in text.split("\n") if line]
        cur = b
        for bound, red in rows[:-1]:
            assert bound == cur and bound <= (lim if red else lim - 4)
            cur = (lim // 2 if red else bound) + 4
        assert rows[-1][0] == cur <= (12 if lim == 16 else 8)
