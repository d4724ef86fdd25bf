"""The dense build at record counts near 2^32: the rounds of its scatter end
and take every record once (pyrit_amd/csrc/dense_walk.h, compiled for the host
with g++; no GPU)."""
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
