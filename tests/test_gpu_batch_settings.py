"""What a batch's settings change, and what they only check and report.

structured_grid bounds the workgroups of the 14-qubit adjoint launch and
dense_max_qubits splits the circuits between the strategies; both are held to the
CPU oracle at the project's 1e-10.  threads, chunk_by_n and dense_tile are
checked and reported: the kernels have one shape per qubit count.
"""

from __future__ import annotations

import numpy as np
import pytest

from gpu_simulation_amd.batch import CircuitSpec, RingIsingBatch

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.mark.parametrize("dense_max", [0, 2, 5, 8])
@pytest.mark.parametrize("grid", [0, 1, 5])
def test_grid_and_split_keep_results(oracle, dense_max, grid):
    specs = [CircuitSpec(n, 2 + n % 3, 0.7 + 0.05 * n) for n in (14, 2, 3, 5, 8, 9, 13, 14, 14)]
    rng = np.random.default_rng(71)
    params = [rng.uniform(0, 2 * np.pi, (s.layers, s.num_qubits, 2)) for s in specs]
    batch = RingIsingBatch(specs, dense_max_qubits=dense_max)
    batch.native.set_config(512, None, 64, grid)
    print(f"case dense_max={dense_max} grid={grid}", flush=True)
    assert batch.config()["grid"] == (3 if grid == 0 else min(grid, 3))
    energies, grads = batch.energy_and_grad(params)
    for s, p, e, g in zip(specs, params, energies, grads):
        e_ref, g_ref = oracle.energy_and_grad(s.num_qubits, s.layers, s.field, p)
        assert abs(e - e_ref) <= TOL, s
        assert np.max(np.abs(np.ravel(g) - np.ravel(g_ref))) <= TOL, s


@pytest.mark.parametrize("threads,widest", [(256, 4), (512, 3), (1024, 2)])
def test_reported_widths_are_those_of_the_workgroup_size(threads, widest):
    batch = RingIsingBatch([CircuitSpec(4, 2, 1.0)], dense_max_qubits=0)
    for width in (1, 2, 3, 4):
        batch.native.set_config(threads, [width] * 15, 32, 0)
        cfg = batch.config()
        assert cfg["threads"] == threads and cfg["dense_tile"] == 32
        assert set(cfg["chunk_by_n"].values()) == {min(width, widest)}


@pytest.mark.parametrize("args", [(128, None, 64, 0), (512, None, 16, 0), (512, None, 64, -1),
                                  (512, [3] * 14, 64, 0), (512, [5] * 15, 64, 0),
                                  (512, [0] * 15, 64, 0)])
def test_settings_out_of_range_are_refused(args):
    batch = RingIsingBatch([CircuitSpec(4, 2, 1.0)], dense_max_qubits=0)
    with pytest.raises((RuntimeError, ValueError)):
        batch.native.set_config(*args)
