"""Large batches run in slices that share the memory of records and 14-qubit states.

A slice ends at a gigabyte once it has sixteen circuits for each CU, in any case
at a quarter of the free memory.  Memory stays bounded and every circuit's
result is what it is alone: a few distinct circuits, held to the CPU oracle at the
project's 1e-10, repeat over the slices bit by bit.
"""

from __future__ import annotations

import numpy as np
import pytest

from gpu_simulation_amd.batch import CircuitSpec, RingIsingBatch

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _hold(oracle, distinct, repeats, energies, grads):
    for k, (spec, p) in enumerate(distinct):
        e_ref, g_ref = oracle.energy_and_grad(spec.num_qubits, spec.layers, spec.field, p)
        assert abs(energies[k] - e_ref) <= TOL, spec
        assert np.max(np.abs(np.ravel(grads[k]) - np.ravel(g_ref))) <= TOL, spec
        for r in range(1, repeats):
            at = r * len(distinct) + k
            assert energies[at] == energies[k], (r, spec)
            assert np.array_equal(grads[at], grads[k]), (r, spec)


@pytest.mark.parametrize("sizes,repeats,free", [
    # 4,300 circuits of 14 qubits (states), smaller ones in the last slice
    ([(14, 1), (14, 2), (14, 1), (9, 3), (14, 3)], 1075, None),
    # records alone: 4,200 x 512 layers
    ([(4, 512), (5, 512)], 2100, None),
    # a gigabyte of records and little memory free
    ([(4, 8192), (5, 8192)], 130, 3 << 30),
])
def test_slices_repeat_the_results(oracle, sizes, repeats, free):
    import torch

    hold = None
    if free is not None:
        torch.cuda.empty_cache()
        hold = torch.empty(torch.cuda.mem_get_info()[0] - free, dtype=torch.uint8, device="cuda")
    rng = np.random.default_rng([41, repeats])
    distinct = [(CircuitSpec(n, layers, 0.5 + 0.05 * k),
                 rng.uniform(0, 2 * np.pi, (layers, n, 2))) for k, (n, layers) in enumerate(sizes)]
    batch = RingIsingBatch([s for s, _ in distinct] * repeats, dense_max_qubits=0)
    params = [p for _, p in distinct] * repeats
    print(f"case slices {sizes} x {repeats}", flush=True)
    energies, grads = batch.energy_and_grad(params)
    _hold(oracle, distinct, repeats, energies, grads)
    batch.native.set_use_graph(True)
    for _ in range(3):
        again, grads2 = batch.energy_and_grad(params)
        assert np.array_equal(again, energies)
        assert all(np.array_equal(a, b) for a, b in zip(grads, grads2))
    batch.native.set_use_graph(False)
    batch.native.run_per_circuit(True, 0)
    single, grads3 = batch.results()
    assert np.array_equal(single, energies)
    assert all(np.array_equal(a, b) for a, b in zip(grads, grads3))
    del hold
    torch.cuda.empty_cache()


def test_memory_of_many_fourteen_qubit_circuits_is_bounded():
    import torch

    torch.zeros(1, device="cuda")
    torch.cuda.synchronize()
    before, _ = torch.cuda.mem_get_info()
    batch = RingIsingBatch([CircuitSpec(14, 1, 1.0)] * 16384)
    after, _ = torch.cuda.mem_get_info()
    # 1 GiB of a slice, 256 workgroups' scratch of 1 MiB, a few MB of parameters and
    # jobs; a state each would be 4 GiB
    assert before - after < 3 << 29
    del batch
