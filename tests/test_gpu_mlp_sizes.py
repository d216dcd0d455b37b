"""The scheduler network's training kernels at the sizes where their split has
edges: tiles of 32 rows, sums over 128 tiles at a time.  The gradient equals
the tiles' own gradients added one after the other in FP32, bit for bit; an
Adam step equals the same formula in NumPy; the loss after training equals the
gradient's."""
import numpy as np
import pytest

from hidem_amd import _abi as A
from oracle import mlp_oracle as M
from test_gpu_sched import rand_inputs, weights_struct

pytestmark = pytest.mark.gpu


def data(n):
    r = np.random.default_rng(n)
    return (rand_inputs(n, n), r.normal(2.0, 1.0, n).astype(np.float32), (r.random(n) < 0.3).astype(np.uint8))


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 4064, 4096, 4097, 8192, 8200, 12320])
def test_gradient_is_the_sum_of_its_tiles(n):
    print("  rows", n, flush=True)
    w = weights_struct(M.init_weights(22, mean=np.full(M.NF, 0.3), std=np.full(M.NF, 1.5)))
    X, t, cen = data(n)
    with A.Context(A.HDM_PREC_FP64) as c:
        g, loss = c.mlp_gradient(w, X, t, cen)
        want, wl = np.zeros_like(g), 0.0
        for o in range(0, n, 32):
            gt, lt = c.mlp_gradient(w, X[o:o + 32], t[o:o + 32], cen[o:o + 32])
            want += gt
            wl += lt
    assert np.array_equal(g.view(np.uint32), want.view(np.uint32))
    assert loss == wl


@pytest.mark.parametrize("n,batch", [(1, 1), (33, 32), (100, 64), (4100, 4096), (4100, 8192)])
def test_adam_steps(n, batch):
    print("  rows", n, "batch", batch, flush=True)
    lr, b1, b2, eps = 1e-3, 0.9, 0.999, 1e-8
    X, t, cen = data(n)
    w0 = M.init_weights(22, mean=np.full(M.NF, 0.3), std=np.full(M.NF, 1.5))
    with A.Context(A.HDM_PREC_FP64) as c:
        ref = weights_struct(w0)
        P = None
        for k, o in enumerate(range(0, n, batch), 1):
            g, _ = c.mlp_gradient(ref, X[o:o + batch], t[o:o + batch], cen[o:o + batch])
            if P is None:
                P, m, v = g.size, np.zeros(g.size), np.zeros(g.size)
            g = g.astype(np.float64) / len(X[o:o + batch])
            m = b1 * m + (1 - b1) * g
            v = b2 * v + (1 - b2) * g * g
            flat = np.frombuffer(bytearray(ref), np.float32).copy()
            flat[:P] -= (lr * (m / (1 - b1 ** k)) / (np.sqrt(v / (1 - b2 ** k)) + eps)).astype(np.float32)
            ref = type(ref).from_buffer_copy(flat.tobytes())
            # one more step from the same start, on the device
            w = weights_struct(w0)
            last = c.mlp_train(w, X[:o + batch], t[:o + batch], cen[:o + batch], epochs=1, batch=batch, lr=lr)
            got = np.frombuffer(bytearray(w), np.float32)
            # ten FP32 roundings in the update (at most lr each way) and one of the weight;
            # 1 - beta^k loses up to 3 more digits for small k
            assert np.all(np.abs(got[:P] - flat[:P]) <= k * (lr * 2e-4 + np.abs(flat[:P]) * 2.0 ** -23))
            assert np.array_equal(got[P:], flat[P:])
            _, loss = c.mlp_gradient(w, X[:o + batch], t[:o + batch], cen[:o + batch])
            assert last == loss / len(X[:o + batch])
            ref = w   # the next gradient at the device's weights
