"""Gradient evaluations whose adjoint passes form H psi by themselves (three
layers and more): every register shape, order of the high passes (down in the
stored schedule, up in the walk) and group split, against the oracle where it is
quick and against the evaluation with separate Hamiltonian passes elsewhere.
21 qubits have a group of nine wires and keep the Hamiltonian pass.  FP64
rounding is far below the project's 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10
BWD_LOW, BWD_HIGH = 4, 5  # places in pass_shapes


def _check(out, e_ref, g_ref):
    assert abs(out["energy"] - e_ref) <= TOL
    assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(g_ref))) <= TOL


@pytest.mark.parametrize("schedule", ["stored", "inverse_walk"])
@pytest.mark.parametrize("shape", [3, 4])
@pytest.mark.parametrize("n,layers", [(13, 3), (15, 4), (17, 3), (20, 3), (21, 3), (22, 3), (25, 3)])
def test_adjoint_passes_form_the_hamiltonian(oracle, backend_module, n, layers, shape, schedule):
    import torch

    p = np.random.default_rng([15, n]).uniform(0, 2 * np.pi, (layers, n, 2))
    eng = backend_module.RingIsingCudaBackend(n, layers, 1.3, "structured_adjoint", 8, False)
    eng.set_schedule(schedule)
    shapes = list(eng.pass_shapes)
    shapes[BWD_LOW] = shapes[BWD_HIGH] = shape
    eng.set_pass_shapes(shapes)
    print(f"case n={n} L={layers} shape={shape} {schedule}", flush=True)
    if n <= 17:
        e_ref, g_ref = oracle.energy_and_grad(n, layers, 1.3, p)
    else:
        eng.set_fused_hamiltonian(0)
        r = eng.energy_and_grad(p.reshape(-1))
        e_ref, g_ref = r["energy"], r["gradient"]
        eng.set_fused_hamiltonian(1)
    _check(eng.energy_and_grad(p.reshape(-1)), e_ref, g_ref)
    # the two device calls, the second with a scale
    d = torch.from_numpy(p.reshape(-1)).cuda()
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    g = torch.zeros_like(d)
    scale = torch.full((1,), -2.0, dtype=torch.float64, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for _ in range(2):
        eng.forward_device(d.data_ptr(), e.data_ptr(), stream)
        eng.backward_device(d.data_ptr(), scale.data_ptr(), g.data_ptr(), stream)
    torch.cuda.synchronize()
    _check({"energy": e.item(), "gradient": g.cpu().numpy() / -2.0}, e_ref, g_ref)
