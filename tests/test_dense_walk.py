"""The dense build at record counts near 2^32: the rounds of its scatter end
and take every record once (pyrit_amd/csrc/dense_walk.h, compiled for the host
with g++), and counts that no build takes are refused before any device work,
on small grids as on large ones (no GPU)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
THREADS, UNROLL = 2048 * 256, 4  # the largest grid of the launch, records per round


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("dw") / "dense_walk_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT}/pyrit_amd/csrc",
                    os.path.join(ROOT, "tests", "dense_walk_driver.cpp"), "-o", exe], check=True)

    def run(n, threads, thread):
        r = subprocess.run([exe, str(n), str(threads), str(UNROLL), str(thread)], capture_output=True, text=True)
        assert r.returncode == 0, "the rounds do not end"
        return [int(w) for w in r.stdout.split()]
    return run


@pytest.mark.parametrize("n", [1, 255, 256, 257, 2 ** 21, 2 ** 31 + 5, 2 ** 32 - 2 ** 21, 2 ** 32 - 2 ** 21 + 1,
                               2 ** 32 - 5121, 2 ** 32 - 2])
def test_rounds_end(walk, n):
    threads = min(THREADS, (n + 1023) // 1024 * 256)
    for thread in (0, 1, threads // 2, threads - 1):
        rounds, taken, first, last, regular = walk(n, threads, thread)
        want = max(0, (n - thread + threads - 1) // threads)
        assert taken == want and regular
        if taken:
            assert first == n - 1 - thread and last == (n - 1 - thread) % threads


@pytest.mark.parametrize("log2", [3, 5, 6, 7, 8, 12])
def test_counts_refused(log2):
    from pyrit_amd import abi, lib

    L = lib()
    out, t = abi.PyrhipBuilt(), abi.PyrhipBuildTuning()
    # (the addresses are never used: the count is refused first)
    for n_old, n_new in ((0, 2 ** 32 - 2), (0, 2 ** 32 - 3000), (2 ** 31, 2 ** 31 - 2)):
        code = L.pyrhip_build(log2, 4096 if n_old else 0, 4096 if n_old else 0, n_old, 4096, n_new, C.byref(t), None,
                              C.byref(out))
        assert code == abi.PYR_ERROR_INVALID_ARGUMENT, (n_old, n_new, code)
