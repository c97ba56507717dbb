"""Row counts at which the closure network's forward and training kernels can go wrong.

One row, the edges of a 32-row chunk, a block's second chunk (more than 512 chunks), and rows that start on no
16-byte boundary.  Reference and tolerances of test_gpu_closure.py: the FP64 restatement with the same bf16
roundings; z relative L2 2e-3; a gradient entry is a product of at most three bf16-rounded factors, 3 * 2^-8 =
1.2e-2, and 3e-2 per parameter block holds it with the activations' rounding.
"""

import numpy as np
import pytest

from mlp_ref import bf16_round, forward, loss_and_gradient
from test_gpu_closure import BLOCKS, _net, _rel, _rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shift", [(1, 0), (31, 0), (33, 1), (512 * 32 + 5, 0)])
def test_rows_match_fp64(gpu, n, shift):
    import torch

    print(f"[closure] {n} rows, {shift} elements off alignment", flush=True)
    net, theta = _net(gpu)
    X, T = _rows(n, 5 + n)
    flat = torch.zeros(n * 64 + 8, dtype=torch.bfloat16, device=gpu)
    x = flat[shift:shift + n * 64].view(n, 64)
    x.copy_(torch.tensor(X, device=gpu))
    th = theta.astype(np.float32).astype(np.float64)
    zr, _ = forward(th, bf16_round(X))
    assert _rel(net.z(x), zr) < 2e-3
    loss, g = net.gradient(x, torch.tensor(T, device=gpu), 1.0 / n)
    lr, gr = loss_and_gradient(th, X, T, 1.0 / n, 150.0)
    assert abs(loss - lr) <= 1e-3 * abs(lr), (loss, lr)
    for name, (a, b) in BLOCKS.items():
        assert _rel(g[a:b], gr[a:b]) < 3e-2, name
