"""Whole-circuit kernels with the state in registers (2..13 qubits; 14 in halves).

Each qubit count has its own layout (register, lane and wave wires) and its own
unrolled layer, so every one is checked against the FP64 CPU oracle: one, two
and several layers, generic angles and those where the tangent form changes
(half angles at 0, pi/4, pi/2, pi and their negatives, on every wire in turn).
FP64 rounding over a few hundred gates is below 1e-13; the bound is the
project's 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

from gpu_simulation_amd.batch import CircuitSpec, RingIsingBatch

pytestmark = pytest.mark.gpu

TOL = 1e-10
# the last pair straddles the switch of the tangent form at a half angle of pi/4
SPECIAL = np.array([0.0, np.pi, -np.pi, 2 * np.pi, np.pi / 2, -np.pi / 2, 3 * np.pi / 2,
                    np.nextafter(np.pi / 2, 4.0)])


def _params(kind, layers, n, rng):
    p = rng.uniform(-2 * np.pi, 4 * np.pi, (layers, n, 2))
    if kind == "special":
        k = np.arange(layers * n).reshape(layers, n)
        p[..., 0] = SPECIAL[(k * 5 + k // 8) % len(SPECIAL)]
        p[..., 1] = np.where(k % 3 == 0, SPECIAL[(k * 3) % len(SPECIAL)], p[..., 1])
    return p


@pytest.mark.parametrize("n", range(2, 15))
def test_every_layout_matches_oracle(oracle, n):
    rng = np.random.default_rng([9, n])
    specs, params = [], []
    for kind in ("generic", "special"):
        for layers in (1, 2, 3, 6):
            specs.append(CircuitSpec(n, layers, 0.6 + 0.1 * layers))
            params.append(_params(kind, layers, n, rng))
    print(f"case n={n}", flush=True)
    batch = RingIsingBatch(specs, dense_max_qubits=0)
    energies, grads = batch.energy_and_grad(params)
    energy_only, _ = batch.energy_and_grad(params, compute_gradient=False)
    assert np.array_equal(energy_only, energies)
    for s, p, e, g in zip(specs, params, energies, grads):
        e_ref, g_ref = oracle.energy_and_grad(n, s.layers, s.field, p)
        assert abs(e - e_ref) <= TOL, (n, s.layers)
        assert np.max(np.abs(np.ravel(g) - np.ravel(g_ref))) <= TOL, (n, s.layers)


def test_fourteen_qubit_circuits_share_workgroups(oracle):
    # more circuits than workgroups of the adjoint launch: each workgroup takes
    # several of different depths in turn, on one scratch
    specs = [CircuitSpec(14, layers, 0.4 + 0.1 * layers) for layers in (5, 1, 2, 4, 1, 3, 2)]
    rng = np.random.default_rng(11)
    params = [_params("generic", s.layers, 14, rng) for s in specs]
    batch = RingIsingBatch(specs)
    batch.native.set_config(512, None, 64, 3)
    print("case 14 qubits, 7 circuits on 3 workgroups", flush=True)
    energies, grads = batch.energy_and_grad(params)
    for s, p, e, g in zip(specs, params, energies, grads):
        e_ref, g_ref = oracle.energy_and_grad(14, s.layers, s.field, p)
        assert abs(e - e_ref) <= TOL, s
        assert np.max(np.abs(np.ravel(g) - np.ravel(g_ref))) <= TOL, s


@pytest.mark.parametrize("n", [2, 5, 6, 7, 8, 9, 11, 12])
def test_engine_calls_agree(oracle, backend_module, n):
    # host call, device calls (one and two step), walk back to |0...0>
    import torch

    layers = 40 if n <= 8 else 9
    p = np.random.default_rng([10, n]).uniform(0, 2 * np.pi, (layers, n, 2))
    eng = backend_module.RingIsingCudaBackend(n, layers, 0.8, "structured_adjoint", 8, False)
    print(f"case engine n={n}", flush=True)
    out = eng.energy_and_grad(p.reshape(-1))
    e_ref, g_ref = oracle.energy_and_grad(n, layers, 0.8, p)
    assert abs(out["energy"] - e_ref) <= TOL
    assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(g_ref))) <= TOL
    assert eng.inverse_walk_drift(p.reshape(-1)) <= 1e-12
    d = torch.from_numpy(p.reshape(-1)).cuda()
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    g = torch.zeros_like(d)
    scale = torch.full((1,), -2.0, dtype=torch.float64, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    eng.energy_and_grad_device(d.data_ptr(), e.data_ptr(), g.data_ptr(), stream)
    torch.cuda.synchronize()
    assert e.item() == out["energy"] and np.array_equal(g.cpu().numpy(), out["gradient"])
    eng.forward_device(d.data_ptr(), e.data_ptr(), stream)
    eng.backward_device(d.data_ptr(), scale.data_ptr(), g.data_ptr(), stream)
    torch.cuda.synchronize()
    assert e.item() == out["energy"]
    assert np.array_equal(g.cpu().numpy(), -2.0 * np.asarray(out["gradient"]))


@pytest.mark.parametrize("n,layers", [(2, 1), (9, 3), (14, 1), (14, 3), (17, 2), (27, 1)])
def test_gate_level_strategy_over_its_paths(oracle, backend_module, n, layers):
    # whole circuit, tile passes, and above 26 qubits gate by gate; at that size
    # against the structured engine, which the headline tests hold to the oracle
    p = np.random.default_rng([12, n]).uniform(0, 2 * np.pi, 2 * n * layers)
    print(f"case gate n={n} L={layers}", flush=True)
    eng = backend_module.RingIsingCudaBackend(n, layers, 1.1, "inverse_walk_cuQuantum", 8, False)
    out = eng.energy_and_grad(p, True, True)
    assert {"forward_apply_ms", "hamiltonian_ms", "energy_dot_ms",
            "backward_sweep_ms"} <= set(out["timings_ms"])
    if n <= 17:
        e_ref, g_ref = oracle.energy_and_grad(n, layers, 1.1, p.reshape(layers, n, 2))
    else:
        ref = backend_module.RingIsingCudaBackend(n, layers, 1.1, "structured_adjoint", 8, False)
        r = ref.energy_and_grad(p)
        e_ref, g_ref = r["energy"], r["gradient"]
    assert abs(out["energy"] - e_ref) <= TOL
    assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(g_ref))) <= TOL
    assert abs(eng.energy_and_grad(p, False)["energy"] - e_ref) <= TOL
    with pytest.raises((RuntimeError, ValueError)):
        eng.final_state()
