"""MLP products on the FP32 matrix cores at ragged and large shapes.

Sizes that are no multiple of the 16 x 16 and 32 x 32 tiles or of the 16-wide k
blocks, operands whose rows are not 16-byte aligned, one row, and enough rows for
the larger tile.  Against the FP64 oracle with the bounds of the other MLP test:
1e-5 of the largest output and of the loss, 1e-4 of the largest gradient entry
(FP32 sums of a few hundred to a few thousand terms).
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import mlp_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inputs,hidden,outputs,rows", [
    (1, 1, 1, 1), (3, 17, 5, 1), (3, 33, 30, 47), (2, 100, 7, 130), (5, 64, 81, 257),
    (3, 255, 80, 64), (3, 256, 80, 4099), (16, 512, 112, 1100),
])
def test_ragged_shapes_match_fp64_oracle(backend_module, inputs, hidden, outputs, rows):
    net = backend_module.WarmStartMLP(inputs, hidden, outputs, 5)
    rng = np.random.default_rng([31, hidden, rows])
    x = rng.uniform(-1, 2, (rows, inputs)).astype(np.float32)
    t = rng.standard_normal((rows, outputs)).astype(np.float32)
    p = np.asarray(net.get_params(), dtype=np.float64)
    print(f"case mlp {inputs}-{hidden}-{hidden}-{outputs} rows {rows}", flush=True)
    y = np.asarray(net.forward(x))
    y_ref, _ = mlp_oracle.forward(p, x, inputs, hidden, outputs)
    assert np.max(np.abs(y - y_ref)) <= 1e-5 * max(1.0, np.max(np.abs(y_ref)))
    loss, g = net.loss_and_grad(x, t)
    loss_ref, g_ref = mlp_oracle.loss_and_grad(p, x, t, inputs, hidden, outputs)
    assert abs(loss - loss_ref) <= 1e-5 * loss_ref
    assert np.max(np.abs(np.asarray(g, dtype=np.float64) - g_ref)) <= 1e-4 * np.max(np.abs(g_ref))
    # fewer rows on the same buffers
    few = max(1, rows // 3)
    loss2, _ = net.loss_and_grad(x[:few], t[:few])
    ref2, _ = mlp_oracle.loss_and_grad(p, x[:few], t[:few], inputs, hidden, outputs)
    assert abs(loss2 - ref2) <= 1e-5 * ref2
