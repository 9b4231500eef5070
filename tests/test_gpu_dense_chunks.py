"""dense_scan over chunks of layers: one chunk, several, ragged last ones.

A circuit is cut into a power of two of chunks of at least 16 layers (fewer
when many circuits run together), whose products meet in the FP64-MFMA tree.
Every case is held to the CPU oracle at the project's 1e-10: depths around the
switch from one chunk to four, depths that leave a short or an empty last
chunk, the padded sizes (n = 2, 3), and circuits of several sizes together.
"""

from __future__ import annotations

import numpy as np
import pytest

from gpu_simulation_amd.batch import CircuitSpec, RingIsingBatch

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.mark.parametrize("n,layers", [(2, 64), (3, 67), (4, 63), (4, 64), (5, 129), (6, 255),
                                      (7, 65), (7, 131), (8, 1), (8, 64), (8, 145), (8, 530)])
def test_engine_depths(oracle, backend_module, n, layers):
    p = np.random.default_rng([21, n, layers]).uniform(0, 2 * np.pi, (layers, n, 2))
    print(f"case dense n={n} L={layers}", flush=True)
    eng = backend_module.RingIsingCudaBackend(n, layers, 0.9, "dense_scan", 8, False)
    out = eng.energy_and_grad(p.reshape(-1))
    e_ref, g_ref = oracle.energy_and_grad(n, layers, 0.9, p)
    assert abs(out["energy"] - e_ref) <= TOL
    assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(g_ref))) <= TOL
    assert abs(eng.energy_and_grad(p.reshape(-1), False)["energy"] - e_ref) <= TOL


def test_batch_of_trees_and_single_chunks(oracle):
    specs = [CircuitSpec(n, layers, 0.5 + 0.1 * n)
             for n, layers in [(8, 70), (4, 200), (8, 3), (2, 90), (6, 64), (4, 17), (7, 97)]]
    rng = np.random.default_rng(22)
    params = [rng.uniform(0, 2 * np.pi, (s.layers, s.num_qubits, 2)) for s in specs]
    batch = RingIsingBatch(specs, dense_max_qubits=8)
    batch.set_params(params)
    batch.native.run_device(True, 0)
    energies, grads = batch.results()
    for s, p, e, g in zip(specs, params, energies, grads):
        e_ref, g_ref = oracle.energy_and_grad(s.num_qubits, s.layers, s.field, p)
        assert abs(e - e_ref) <= TOL, s
        assert np.max(np.abs(np.ravel(g) - np.ravel(g_ref))) <= TOL, s
    batch.native.run_per_circuit(True, 0)
    e_single, g_single = batch.results()
    assert np.array_equal(energies, e_single)
    assert all(np.array_equal(a, b) for a, b in zip(grads, g_single))
