"""The launches that begin and end a tile-path evaluation.

One launch prepares coefficients, chain tables and addresses (from 24 qubits on
the coefficient table is a launch of its own), one reduces every pass's gradient
partials and the layer-0 sums (two when the tiles take more than one chunk, from
21 qubits on; several when more than 16 passes ran).  FP64 rounding is far below
the project's 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10
BWD_HIGH = 5  # place in pass_shapes


def _engine(module, n, layers):
    return module.RingIsingCudaBackend(n, layers, 0.9, "structured_adjoint", 8, False)


@pytest.mark.parametrize("n,layers", [(13, 1), (13, 9), (16, 6), (17, 2)])
@pytest.mark.parametrize("schedule", ["stored", "inverse_walk"])
def test_small_tile_paths_match_oracle(oracle, backend_module, n, layers, schedule):
    # 9 layers of two passes and 6 of two: past and below 16 waiting passes
    p = np.random.default_rng([13, n]).uniform(0, 2 * np.pi, (layers, n, 2))
    eng = _engine(backend_module, n, layers)
    if layers > 1:
        eng.set_schedule(schedule)
    print(f"case n={n} L={layers} schedule={schedule}", flush=True)
    e_ref, g_ref = oracle.energy_and_grad(n, layers, 0.9, p)
    for _ in range(2):
        out = eng.energy_and_grad(p.reshape(-1))
        assert abs(out["energy"] - e_ref) <= TOL
        assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(g_ref))) <= TOL
    assert eng.inverse_walk_drift(p.reshape(-1)) <= 1e-12


@pytest.mark.parametrize("n,layers", [(20, 2), (21, 2), (21, 3), (23, 2), (24, 2)])
def test_generated_and_walked_evaluations_agree(backend_module, n, layers):
    # each way prepares and ends differently: generated start, generated layer 1
    # over the two device calls (the backward keeps or rebuilds the tables), walk
    import torch

    p = np.random.default_rng([14, n]).uniform(0, 2 * np.pi, 2 * n * layers)
    eng = _engine(backend_module, n, layers)
    print(f"case n={n} L={layers}", flush=True)
    first = eng.energy_and_grad(p)
    d = torch.from_numpy(p).cuda()
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    g = torch.zeros_like(d)
    stream = torch.cuda.current_stream().cuda_stream
    for shape in (None, 3):  # the adjoint's register shape changed between the two calls
        eng.forward_device(d.data_ptr(), e.data_ptr(), stream)
        if shape is not None:
            shapes = list(eng.pass_shapes)
            shapes[BWD_HIGH] = shape
            eng.set_pass_shapes(shapes)
        eng.backward_device(d.data_ptr(), 0, g.data_ptr(), stream)
        torch.cuda.synchronize()
        assert abs(e.item() - first["energy"]) <= TOL
        assert np.max(np.abs(g.cpu().numpy() - np.asarray(first["gradient"]))) <= TOL, shape
    eng.set_layer1_generation(0)
    walked = eng.energy_and_grad(p)
    assert abs(walked["energy"] - first["energy"]) <= TOL
    assert np.max(np.abs(np.asarray(walked["gradient"]) - np.asarray(first["gradient"]))) <= TOL
