"""The surrogate's row-tile kernels where tiles end: layer widths around 16,
32, 64, 256 and the widest one the kernels take (and one past it, which runs
a product a launch), rows around the 16 of a workgroup, minibatches with a
remainder; against the float64 numpy network.

Tolerances.  A product of operands split into bf16 halves drops lo*lo and
rounds each lo: at most 3 * 2^-18 = 1.2e-5 of |A||B| per product.  A forward
pass has up to five products in series (6e-5): 1e-4 of the result's norm.  A
gradient has up to ten and the derivatives of GELU (at most 1.13) between
them: 10 * 1.2e-5 * 4 = 5e-4, tested at 1e-3.  An Adam update from zero
moments is lr * sign(g) to leading order, so entries within the gradient's
error of zero may take either sign: a fraction below 1e-3 of them, each
twice the update, sqrt(4 * 1e-3) = 0.063 of the update's norm, tested at 0.1."""
import numpy as np
import pytest

from arbo_gpu_fit_amd.surrogate import Surrogate
from tests.mlp_ref import backward64, flatten, forward64, loss_grad64, random_layers
from tests.test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

WIDTHS = [[1, 1], [6, 16, 17], [6, 15, 33, 31], [5, 64, 65, 64, 1], [6, 256, 256, 257], [40, 200, 260],
          [6, 256, 256, 256, 256, 260], [7, 300, 512, 12], [513, 30, 20], [6, 520, 30]]


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-30))


@pytest.mark.parametrize("widths", WIDTHS, ids=lambda w: "-".join(map(str, w)))
def test_passes_at_the_tile_edges(hip_lib, widths):
    hip = Hip()
    layers = random_layers(widths, 21)
    s = Surrogate(widths, max_batch=70, seed=3, lib=hip_lib)
    s.set_params(flatten(layers))
    rng = np.random.default_rng(22)
    for n in (1, 15, 16, 17, 70):
        print(f"[tiles] widths={widths} rows={n}", flush=True)
        x = rng.normal(size=(n, widths[0])).astype(np.float32)
        f = forward64(layers, x)[0]
        out = s.forward(x)
        assert rel(out, f) < 1e-4
        dev_x, dev_out = hip.upload(x), hip.upload(np.full((n + 1, widths[-1]), 7.0, np.float32))
        assert s.lib.arbo_sur_forward_noalloc(s._h, n, dev_x, dev_out, None) == 0
        hip.check(hip.lib.hipDeviceSynchronize(), "hipDeviceSynchronize")
        got = hip.download(dev_out, (n + 1, widths[-1]))
        assert np.array_equal(got[:n], out) and np.all(got[n] == 7.0)   # nothing past the last row
        hip.check(hip.lib.hipFree(dev_x), "hipFree")
        hip.check(hip.lib.hipFree(dev_out), "hipFree")
        dout = rng.normal(size=f.shape).astype(np.float32)
        out2, dx = s.input_grad(x, dout)
        assert np.array_equal(out2, out)
        assert rel(dx, backward64(layers, x, dout)[1]) < 1e-3
        y = rng.poisson(np.exp(np.clip(f, -5, 3))).astype(np.float32)
        loss, g = s.loss_grad(x, y)
        l64, g64 = loss_grad64(layers, x, y)
        assert abs(loss - l64) < 1e-4 * max(abs(l64), 1.0)
        assert rel(g, g64) < 1e-3
    s.close()


def test_a_row_does_not_depend_on_its_batch(hip_lib):
    widths = [6, 96, 96, 40]
    s = Surrogate(widths, max_batch=300, seed=4, lib=hip_lib)
    x = np.random.default_rng(5).normal(size=(300, 6)).astype(np.float32)
    whole = s.forward(x)
    for lo, hi in ((0, 1), (3, 20), (100, 300)):
        assert np.array_equal(s.forward(x[lo:hi]), whole[lo:hi])
    s.close()


@pytest.mark.parametrize("widths", [[6, 16, 17], [6, 65, 64, 31], [6, 256, 260], [6, 520, 30]],
                         ids=lambda w: "-".join(map(str, w)))
def test_training_steps_and_packed_weights(hip_lib, widths):
    """Three Adam steps of one epoch (16, 16 and 8 rows): the update against
    float64 over the documented row order, and the weights the next passes
    read against the parameters read back."""
    n, batch, lr, seed = 40, 16, 1e-3, 9
    print(f"[tiles] training widths={widths}", flush=True)
    layers = random_layers(widths, 31)
    rng = np.random.default_rng(32)
    x = rng.normal(size=(n, widths[0])).astype(np.float32)
    y = rng.poisson(np.exp(np.clip(forward64(layers, x)[0], -5, 3))).astype(np.float32)
    s = Surrogate(widths, max_batch=64, seed=3, lib=hip_lib)
    p0 = flatten(layers)
    s.set_params(p0)
    hist = s.train(x, y, epochs=1, batch=batch, lr=lr, seed=seed)
    p1 = s.get_params()

    from arbo_gpu_fit_amd.configs import philox4x32
    r = philox4x32(np.arange(n), 0, 7, 0, seed, 0)[0].astype(np.uint64)
    perm = list(range(n))
    for i in range(n - 1, 0, -1):
        j = int((int(r[i]) * (i + 1)) >> 32)
        perm[i], perm[j] = perm[j], perm[i]
    p, m, v, total = p0.astype(np.float64), 0.0, 0.0, 0.0
    for t, b0 in enumerate(range(0, n, batch), 1):
        rows = perm[b0:b0 + batch]
        l, g = loss_grad64(s.layers(p), x[rows], y[rows])
        total += l * len(rows)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    assert rel(p1 - p0, p - p0) < 0.1
    assert abs(hist[0] - total / n) < 1e-3 * max(abs(total / n), 1.0)
    after = s.layers(p1)
    assert rel(s.forward(x), forward64(after, x)[0]) < 1e-4
    dout = rng.normal(size=(n, widths[-1])).astype(np.float32)
    assert rel(s.input_grad(x, dout)[1], backward64(after, x, dout)[1]) < 1e-3
    s.close()
