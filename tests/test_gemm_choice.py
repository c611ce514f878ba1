"""The tile that the library itself picks for a large GEMM (gemm_choice.h), on
the host: the sizes that test_gpu_tile_rows takes for its 192 and 128 rows, the
rounds rule on both sides of its lines, and what every choice must hold."""
import os
import random
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "gemm_choice_host_check.cpp")


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("choice") / "gemm_choice")
    subprocess.run(["g++", "-O1", "-std=c++17", SRC, "-o", exe], check=True)

    def run(sizes):
        args = []
        for m, n, k in sizes:  # padded as Linears are
            args += [m, -(-m // 256) * 256, -(-n // 256) * 256, -(-k // 64) * 64]
        out = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return run


CASES = [
    # the cases of test_gpu_tile_rows
    ((2890, 4096, 130), (192, 256, 1)), ((5900, 4096, 64), (192, 256, 1)),
    ((2570, 2972, 200), (128, 256, 1)), ((2600, 3002, 330), (128, 256, 1)),
    # 1.25 and 1.5 rounds of 256 rows, not 2.5 and 3 of 128
    ((5100, 4096, 4096), (256, 256, 1)), ((8192, 3000, 2000), (256, 256, 1)),
    ((8192, 4096, 4096), (256, 256, 1)), ((3000, 4096, 4096), (192, 256, 1)),
    # 128 x 128 tiles; K split below 128 of them
    ((1500, 4096, 4096), (128, 128, 1)), ((100, 4096, 4096), (128, 128, 8)),
]


def test_choices(choose):
    assert choose([c for c, _ in CASES]) == [w for _, w in CASES]


def test_tiles_stay_within_the_padded_rows(choose):
    rng = random.Random(1)
    sizes = [(rng.randint(1, 20000), rng.randint(1, 9000), rng.randint(1, 20000)) for _ in range(400)]
    for (m, n, k), (bm, bn, splits) in zip(sizes, choose(sizes)):
        assert -(-m // bm) * bm <= -(-m // 256) * 256, (m, bm)
        assert (-(-n // 256) * 256) % bn == 0 and 1 <= splits <= max(1, -(-k // 64) // 4), (n, k, bn, splits)
