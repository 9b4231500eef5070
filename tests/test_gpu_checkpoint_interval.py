"""Checkpoint intervals on engines that keep no checkpoints, and out of range.

The gate-level strategy accepts an interval and keeps none, also where it runs on
the tile passes; an interval beyond the layers keeps none either.  Against the CPU
oracle at the project's 1e-10.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _check(out, ref):
    assert abs(out["energy"] - ref[0]) <= TOL
    assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(ref[1]))) <= TOL


@pytest.mark.parametrize("strategy,n,layers", [
    ("inverse_walk_cuQuantum", 5, 4), ("inverse_walk_cuQuantum", 13, 4),
    ("inverse_walk_cuQuantum", 17, 3), ("dense_scan", 5, 4), ("structured_adjoint", 13, 4),
    ("structured_adjoint", 17, 3)])
def test_any_interval_keeps_results(oracle, backend_module, strategy, n, layers):
    import torch

    p = np.random.default_rng([91, n]).uniform(0, 2 * np.pi, (layers, n, 2))
    ref = oracle.energy_and_grad(n, layers, 0.9, p)
    eng = backend_module.RingIsingCudaBackend(n, layers, 0.9, strategy, 8, False)
    if strategy == "structured_adjoint":
        eng.set_schedule("inverse_walk")
    d = torch.from_numpy(p.reshape(-1)).cuda()
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    g = torch.zeros_like(d)
    stream = torch.cuda.current_stream().cuda_stream
    for every in (1, 2, layers - 1, layers, 1 << 32, 0):
        print(f"case {strategy} n={n} L={layers} every {every}", flush=True)
        eng.set_checkpoint_interval(every)
        _check(eng.energy_and_grad(p.reshape(-1)), ref)
        assert abs(eng.energy_and_grad(p.reshape(-1), False)["energy"] - ref[0]) <= TOL
        eng.forward_device(d.data_ptr(), e.data_ptr(), stream)
        eng.backward_device(d.data_ptr(), 0, g.data_ptr(), stream)
        torch.cuda.synchronize()
        _check({"energy": e.item(), "gradient": g.cpu().numpy()}, ref)


def test_gate_level_module_with_checkpoints(oracle):
    import torch

    from gpu_simulation_amd.autograd import RingIsingEnergy

    n, layers = 14, 5
    p = np.random.default_rng(92).uniform(0, 2 * np.pi, (layers, n, 2))
    e_ref, g_ref = oracle.energy_and_grad(n, layers, 1.0, p)
    params = torch.from_numpy(p).cuda().requires_grad_(True)
    print("case gate-level module, checkpoint_every 2", flush=True)
    energy = RingIsingEnergy(n, layers, 1.0, "inverse_walk_cuQuantum", checkpoint_every=2)(params)
    energy.backward()
    _check({"energy": energy.item(), "gradient": params.grad.cpu().numpy().reshape(-1)},
           (e_ref, g_ref))


def test_interval_set_between_forward_and_backward(oracle, backend_module):
    import torch

    n, layers = 16, 5
    p = np.random.default_rng(93).uniform(0, 2 * np.pi, (layers, n, 2))
    ref = oracle.energy_and_grad(n, layers, 1.0, p)
    eng = backend_module.RingIsingCudaBackend(n, layers, 1.0, "structured_adjoint", 8, False)
    eng.set_schedule("inverse_walk")
    d = torch.from_numpy(p.reshape(-1)).cuda()
    e = torch.zeros(1, dtype=torch.float64, device="cuda")
    g = torch.zeros_like(d)
    stream = torch.cuda.current_stream().cuda_stream
    for every in (2, 0, 1):
        print(f"case interval {every} between forward and backward", flush=True)
        eng.forward_device(d.data_ptr(), e.data_ptr(), stream)
        eng.set_checkpoint_interval(every)
        eng.backward_device(d.data_ptr(), 0, g.data_ptr(), stream)
        torch.cuda.synchronize()
        _check({"energy": e.item(), "gradient": g.cpu().numpy()}, ref)
