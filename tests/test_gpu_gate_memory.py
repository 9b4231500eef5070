"""The gate-level strategy where the tile passes' buffers are not free.

Up to 26 qubits it runs on the tile passes (four state buffers and tables); with
less memory free it runs gate by gate on two, so an engine that fitted before
still does.  Three layers gate by gate against the CPU oracle at the project's
1e-10: the walk back carries psi and lambda from layer to layer.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10


@pytest.mark.parametrize("n,layers", [(23, 3)])
def test_gate_by_gate_where_memory_is_short(oracle, backend_module, n, layers):
    import torch

    p = np.random.default_rng([51, n]).uniform(0, 2 * np.pi, 2 * n * layers)
    strategy = "inverse_walk_cuQuantum"
    tiles = backend_module.RingIsingCudaBackend(n, layers, 0.8, strategy, 8, False)
    first = tiles.energy_and_grad(p)  # kernels loaded before memory runs short
    assert tiles.fused_hamiltonian  # only evaluations on the tile passes are
    del tiles
    state = 16 << n
    torch.cuda.empty_cache()
    hold = []
    for left in (8 * state, 7 * state // 2):  # what is reported free differs after the first
        free, _ = torch.cuda.mem_get_info()
        hold.append(torch.empty(max(1, free - left), dtype=torch.uint8, device="cuda"))
    print(f"case gate by gate n={n} L={layers}", flush=True)
    try:
        eng = backend_module.RingIsingCudaBackend(n, layers, 0.8, strategy, 8, False)
        assert not eng.fused_hamiltonian
        out = eng.energy_and_grad(p)
        energy_only = eng.energy_and_grad(p, False)["energy"]
        del eng
    finally:
        del hold
        torch.cuda.empty_cache()
    e_ref, g_ref = oracle.energy_and_grad(n, layers, 0.8, p.reshape(layers, n, 2))
    for e, g in ((out["energy"], out["gradient"]), (first["energy"], first["gradient"])):
        assert abs(e - e_ref) <= TOL
        assert np.max(np.abs(np.asarray(g) - np.ravel(g_ref))) <= TOL
    assert abs(energy_only - e_ref) <= TOL


def test_gate_by_gate_layers_above_the_limit(backend_module):
    # 27 qubits against the structured engine, which the headline tests hold to
    # the oracle
    n, layers = 27, 2
    p = np.random.default_rng([52, n]).uniform(0, 2 * np.pi, 2 * n * layers)
    print(f"case gate by gate n={n} L={layers}", flush=True)
    gate = backend_module.RingIsingCudaBackend(n, layers, 1.1, "inverse_walk_cuQuantum", 8, False)
    out = gate.energy_and_grad(p)
    del gate
    ref = backend_module.RingIsingCudaBackend(n, layers, 1.1, "structured_adjoint", 8, False)
    want = ref.energy_and_grad(p)
    assert abs(out["energy"] - want["energy"]) <= TOL
    assert np.max(np.abs(np.asarray(out["gradient"]) - np.asarray(want["gradient"]))) <= TOL
