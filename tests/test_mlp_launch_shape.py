"""The network's launch shapes over every accepted size (host arithmetic, no GPU).

rie_mlp_shape.hpp is compiled by itself and asked for the grid at the limits:
y and z hold at most 65535 blocks, every dimension's threads fit 32 bits, the
blocks are exactly the tiles (spare ones only past the last row), and the loss
partials hold the tiles of every smaller row count.
"""

from __future__ import annotations

import os
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "gpu_simulation_amd" / "csrc"
SIZES = [1, 15, 16, 17, 31, 33, 257, 4095, 4096]
ROWS = [1, 16, 33, 4099, 65535 * 16 + 1, (1 << 21) - 31, (1 << 21) + 1, (1 << 22) - 1, 1 << 22]

PROGRAM = r"""
#include <cstdio>
#include "rie_mlp_shape.hpp"
int main() {
    int m, n;
    while (std::scanf("%d %d", &m, &n) == 2) {
        const rie::MlpGrid g = rie::mlp_grid(m, n);
        std::printf("%d %u %u %u %u %zu %lld\n", g.sub, g.rows, g.x, g.y, g.z,
                    rie::mlp_mse_partials(m, n), rie::mlp_elements(m, n));
    }
}
"""


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    work = tmp_path_factory.mktemp("mlp_shape")
    src, exe = work / "shape.cpp", work / "shape"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", f"-I{CSRC}", str(src), "-o",
                    str(exe)], check=True)

    def ask(pairs):
        text = "".join(f"{m} {n}\n" for m, n in pairs)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True)
        return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]

    return ask


def test_grids_stay_within_the_launch_limits(shapes):
    # row calls (rows x width) and weight gradients (width + 1 x width)
    pairs = [(m, n) for m in ROWS for n in SIZES] + [(m + 1, n) for m in SIZES for n in SIZES]
    for (m, n), (sub, row_tiles, x, y, z, _, _) in zip(pairs, shapes(pairs)):
        tile = 16 * sub
        assert 1 <= y <= 65535 and 1 <= z <= 65535 and x * 256 < 1 << 32, (m, n)
        assert (row_tiles - 1) * tile < m <= row_tiles * tile, (m, n)
        assert (x - 1) * tile < n <= x * tile, (m, n)
        assert (z - 1) * y < row_tiles <= z * y, (m, n)


@pytest.mark.parametrize("cols", [1, 30, 81, 4096])
def test_loss_partials_hold_every_smaller_grid(shapes, cols):
    rows = sorted({1, 2, 511, 512, 513, 8191, 8192, 16384, 16385, *ROWS})
    out = shapes([(m, cols) for m in rows])
    for k, (*_, room, _) in enumerate(out):
        for _, row_tiles, x, *_ in out[:k + 1]:
            assert row_tiles * x <= room, (rows[k], cols)


def test_the_loss_is_a_mean_over_all_values(shapes):
    # 2^22 rows of 4096 outputs: more values than 32 bits count
    pairs = [(m, n) for m in ROWS for n in SIZES]
    for (m, n), (*_, elements) in zip(pairs, shapes(pairs)):
        assert elements == m * n
