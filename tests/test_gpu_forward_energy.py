"""Energies from the last layer's forward passes (20, 22 to 28 and 31 to 34 qubits,
three layers and more), against the passes over the finished state and against the
gradient evaluation's energy.  FP64 rounding is far below the project's 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10
FWD_LOW = 2  # place in pass_shapes


@pytest.mark.parametrize("schedule", ["stored", "inverse_walk"])
@pytest.mark.parametrize("shape", [3, 4])
@pytest.mark.parametrize("n,layers", [(19, 3), (20, 3), (21, 3), (22, 4), (23, 3), (27, 3), (28, 3)])
def test_energy_without_hamiltonian_passes(backend_module, n, layers, shape, schedule):
    import torch

    p = np.random.default_rng([16, n]).uniform(0, 2 * np.pi, layers * n * 2)
    eng = backend_module.RingIsingCudaBackend(n, layers, 0.7, "structured_adjoint", 8, False)
    eng.set_schedule(schedule)
    shapes = list(eng.pass_shapes)
    shapes[FWD_LOW] = shape
    eng.set_pass_shapes(shapes)
    print(f"case n={n} L={layers} shape={shape} {schedule}", flush=True)
    eng.set_fused_hamiltonian(0)
    ref = eng.energy_and_grad(p, False)["energy"]
    eng.set_fused_hamiltonian(1)
    assert abs(eng.energy_and_grad(p, False)["energy"] - ref) <= TOL
    assert abs(eng.energy_and_grad(p)["energy"] - ref) <= TOL
    d = torch.from_numpy(p).cuda()
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    eng.forward_device(d.data_ptr(), e.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert abs(e.item() - ref) <= TOL
