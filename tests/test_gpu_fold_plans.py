"""Evaluations of three and more layers in the plans that the other tests leave out.

The next tile prefetched (double_buffer) at the default register shapes, where the
adjoint passes form H psi: it changes no arithmetic, so energies and gradients are
bitwise equal with it on and off, and they are the CPU oracle's.  Three high
groups (31 qubits): the middle group's terms reach the pass below and above it;
against the evaluation with separate Hamiltonian passes.  FP64 rounding is far
below the project's 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _engine(module, n, layers, double_buffer=False):
    return module.RingIsingCudaBackend(n, layers, 0.9, "structured_adjoint", 8, double_buffer)


@pytest.mark.parametrize("schedule", ["stored", "inverse_walk"])
@pytest.mark.parametrize("n,layers", [(20, 3), (22, 4), (23, 3)])
def test_prefetch_at_the_default_shapes(oracle, backend_module, n, layers, schedule):
    p = np.random.default_rng([81, n]).uniform(0, 2 * np.pi, 2 * n * layers)
    outs = []
    for double_buffer in (False, True):
        print(f"case prefetch={double_buffer} n={n} L={layers} {schedule}", flush=True)
        eng = _engine(backend_module, n, layers, double_buffer)
        eng.set_schedule(schedule)
        out = eng.energy_and_grad(p)
        outs.append((out["energy"], np.asarray(out["gradient"])))
    assert outs[0][0] == outs[1][0]
    assert np.array_equal(outs[0][1], outs[1][1])
    if n == 20:
        e_ref, g_ref = oracle.energy_and_grad(n, layers, 0.9, p.reshape(layers, n, 2))
        assert abs(outs[1][0] - e_ref) <= TOL
        assert np.max(np.abs(outs[1][1] - np.ravel(g_ref))) <= TOL


@pytest.mark.parametrize("schedule", ["default", "inverse_walk"])
def test_three_groups_match_separate_hamiltonian_passes(backend_module, schedule):
    n, layers = 31, 3
    p = np.random.default_rng([82, n]).uniform(0, 2 * np.pi, 2 * n * layers)
    eng = _engine(backend_module, n, layers)
    if schedule != "default":
        eng.set_schedule(schedule)
    print(f"case three groups {eng.schedule}", flush=True)
    eng.set_fused_hamiltonian(0)
    want = eng.energy_and_grad(p)
    energy = eng.energy_and_grad(p, False)["energy"]
    eng.set_fused_hamiltonian(1)
    assert abs(eng.energy_and_grad(p, False)["energy"] - energy) <= TOL
    for double_buffer in (0, 1):
        eng.set_double_buffer(double_buffer)
        got = eng.energy_and_grad(p)
        assert abs(got["energy"] - want["energy"]) <= TOL
        assert np.max(np.abs(np.asarray(got["gradient"]) - np.asarray(want["gradient"]))) <= TOL
