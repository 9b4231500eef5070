"""Row counts up to the accepted 2^22: one launch each, the row tiles on grid y and z.

Against the same network in float64 torch.  Outputs and loss are held to the 1e-5
of the other MLP tests.  A gradient entry is four FP32 chains of 2^18 sums of four
terms: independent roundings of at most 2^-24 of the chain each leave about
2^9 * 2^-24 / sqrt(3) = 2e-5 of it, so 1e-4 of the largest entry is five times the
expected error; the targets' offsets vary and have one sign, so the terms neither
repeat nor cancel.
"""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [(1 << 21) + 1, 1 << 22])
def test_rows_up_to_the_limit(backend_module, rows):
    import torch

    net = backend_module.WarmStartMLP(1, 2, 1, 5)
    rng = np.random.default_rng([32, rows])
    x = rng.uniform(-1, 2, (rows, 1)).astype(np.float32)
    flat = torch.tensor(np.asarray(net.get_params()), dtype=torch.float64, requires_grad=True)
    w1, b1, w2, b2, w3, b3 = torch.split(flat, [2, 2, 4, 2, 2, 1])
    a = torch.nn.functional.gelu(torch.from_numpy(x).double() @ w1.view(1, 2) + b1)
    a = torch.nn.functional.gelu(a @ w2.view(2, 2) + b2)
    y_ref = a @ w3.view(2, 1) + b3
    y_top = float(y_ref.detach().abs().max())
    print(f"case mlp 1-2-2-1 rows {rows}", flush=True)
    y = np.asarray(net.forward(x))
    assert np.max(np.abs(y - y_ref.detach().numpy())) <= 1e-5 * max(1.0, y_top)
    t = (y_ref.detach().numpy() + rng.uniform(0.5, 1.5, (rows, 1))).astype(np.float32)
    loss, g = net.loss_and_grad(x, t)
    loss_ref = ((y_ref - torch.from_numpy(t).double()) ** 2).mean()
    (g_ref,) = torch.autograd.grad(loss_ref, flat)
    assert abs(loss - loss_ref.item()) <= 1e-5 * loss_ref.item()
    assert np.max(np.abs(np.asarray(g, dtype=np.float64) - g_ref.numpy())) <= \
        1e-4 * float(g_ref.abs().max())


def test_more_rows_are_refused(backend_module):
    net = backend_module.WarmStartMLP(1, 2, 1, 5)
    with pytest.raises((RuntimeError, ValueError)):
        net.forward(np.zeros(((1 << 22) + 1, 1), dtype=np.float32))
