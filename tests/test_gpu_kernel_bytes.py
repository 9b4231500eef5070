"""Algorithmic bytes that the per-launch kernel timing reports.

From three layers on (20, 22 to 28 qubits) the last layer's low adjoint pass starts
lambda from the state alone: it reads one state array less than the other
layers' low passes, and no Hamiltonian pass runs.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule,walk", [("stored", 0), ("inverse_walk", 1)])
def test_low_adjoint_pass_that_starts_lambda(backend_module, schedule, walk):
    n, layers = 20, 4
    state = 16 << n
    p = np.random.default_rng(101).uniform(0, 2 * np.pi, 2 * n * layers)
    eng = backend_module.RingIsingCudaBackend(n, layers, 1.0, "structured_adjoint", 8, False)
    eng.set_schedule(schedule)
    for fused, arrays in ((1, 2 + 3 + 3), (0, 3 + 3 + 3)):
        eng.set_fused_hamiltonian(fused)
        eng.energy_and_grad(p)
        eng.set_kernel_timing(1)
        eng.reset_kernel_stats()
        eng.energy_and_grad(p)
        stats = {k["name"]: k for k in eng.kernel_stats()}
        eng.set_kernel_timing(0)
        low = stats["bwd_pass_low_cnot"]
        # the walk rewrites the state of the layers above the first
        assert low["launches"] == 3
        assert low["total_bytes"] == state * (arrays + 2 * walk)
        assert any(name.startswith("ham_pass") for name in stats) == (not fused)
