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
import ctypes

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


@pytest.mark.parametrize("widths,max_batch,rows", [([6, 64, 20], 2100, (1023, 1024, 1025, 2049, 2100)),
                                                   ([512, 16, 511], 4200, (2047, 2051, 4200)),
                                                   ([3, 300, 7], 1030, (1030,))],
                         ids=lambda w: "-".join(map(str, w)) if isinstance(w, list) else None)
def test_host_rows_in_chunks(hip_lib, widths, max_batch, rows):
    """Host calls around the 1,024 rows of a chunk, and of more rows than the
    pinned ones hold: every row as in a call of 64 rows."""
    s = Surrogate(widths, max_batch=max_batch, seed=6, lib=hip_lib)
    rng = np.random.default_rng(7)
    x = rng.normal(size=(max_batch, widths[0])).astype(np.float32)
    dout = rng.normal(size=(max_batch, widths[-1])).astype(np.float32)
    parts = [s.input_grad(x[i:i + 64], dout[i:i + 64]) for i in range(0, max_batch, 64)]
    out, dx = (np.concatenate([p[k] for p in parts]) for k in (0, 1))
    for n in rows:
        print(f"[tiles] host rows widths={widths} rows={n}", flush=True)
        assert np.array_equal(s.forward(x[:n]), out[:n])
        got_out, got_dx = s.input_grad(x[:n], dout[:n])
        assert np.array_equal(got_out, out[:n]) and np.array_equal(got_dx, dx[:n])
    s.close()


@pytest.mark.parametrize("outputs", [16, 19, 20])
def test_device_rows_at_any_float_address(hip_lib, outputs):
    """x and out one to three floats past a 16-byte boundary."""
    hip = Hip()
    s = Surrogate([6, 32, outputs], max_batch=64, seed=8, lib=hip_lib)
    x = np.random.default_rng(9).normal(size=(33, 6)).astype(np.float32)
    ref = s.forward(x)
    for k in (1, 2, 3):
        dev_x = hip.upload(np.concatenate([np.zeros(k, np.float32), x.ravel()]))
        dev_out = hip.upload(np.full(k + ref.size + 1, 7.0, np.float32))
        at = [p.value + 4 * k for p in (dev_x, dev_out)]
        print(f"[tiles] offset {k} outputs={outputs}", flush=True)
        assert s.lib.arbo_sur_forward_noalloc(s._h, 33, at[0], at[1], None) == 0
        hip.check(hip.lib.hipDeviceSynchronize(), "hipDeviceSynchronize")
        got = hip.download(dev_out, (k + ref.size + 1,))
        assert np.array_equal(got[k:-1].reshape(ref.shape), ref)
        assert np.all(got[:k] == 7.0) and got[-1] == 7.0
        hip.check(hip.lib.hipFree(dev_x), "hipFree")
        hip.check(hip.lib.hipFree(dev_out), "hipFree")
    s.close()


@pytest.mark.parametrize("widths", [[6, 33, 12], [6, 520, 9]], ids=lambda w: "-".join(map(str, w)))
def test_epochs_take_their_own_row_orders(hip_lib, widths):
    """Two epochs in one call give the weights of two calls of one, the second
    on rows laid out so that the first epoch's order reads the second's."""
    from arbo_gpu_fit_amd.configs import philox4x32
    n, seed = 50, 11
    rng = np.random.default_rng(12)
    x = rng.normal(size=(n, 6)).astype(np.float32)
    y = rng.poisson(2.0, size=(n, widths[-1])).astype(np.float32)
    order = []
    for e in (0, 1):
        r = philox4x32(np.arange(n), e, 7, 0, seed, 0)[0].astype(np.uint64)
        perm = list(range(n))
        for i in range(n - 1, 0, -1):
            j = int((int(r[i]) * (i + 1)) >> 32)
            perm[i], perm[j] = perm[j], perm[i]
        order.append(perm)
    x2, y2 = np.empty_like(x), np.empty_like(y)
    x2[order[0]], y2[order[0]] = x[order[1]], y[order[1]]
    got = []
    for calls in ([(x, y, 2)], [(x, y, 1), (x2, y2, 1)]):
        s = Surrogate(widths, max_batch=64, seed=13, lib=hip_lib)
        for cx, cy, epochs in calls:
            s.train(cx, cy, epochs=epochs, batch=16, lr=1e-3, seed=seed)
        got.append(s.get_params())
        s.close()
    assert np.array_equal(got[0], got[1])


def _place(kind, n_in, n_out):
    """Element offsets of an input and an output of n_in and n_out elements
    that overlap, and the buffer's size."""
    at = {"output first": (n_out // 3, 0), "input first": (0, n_in // 2), "same start": (0, 0)}[kind]
    return *at, max(at[0] + n_in, at[1] + n_out)


OVERLAPS = ["output first", "input first", "same start"]


@pytest.mark.parametrize("kind", OVERLAPS)
@pytest.mark.parametrize("widths,n", [([6, 64, 64, 20], 4000), ([20, 33, 20], 2500), ([200, 16, 16, 30], 12000),
                                      ([6, 520, 30], 300)],
                         ids=lambda w: "-".join(map(str, w)) if isinstance(w, list) else None)
def test_results_over_the_inputs(hip_lib, widths, n, kind):
    """Calls whose results lie over their inputs give what they give apart
    from them: rows of several chunks, of one width and of two, and more
    inputs than the scratch holds (products of other rounding)."""
    print(f"[tiles] overlap {kind} {widths}", flush=True)
    hip = Hip()
    f32p = ctypes.POINTER(ctypes.c_float)
    s = Surrogate(widths, max_batch=n, seed=7, lib=hip_lib)
    rng = np.random.default_rng(8)
    x = rng.normal(size=(n, widths[0])).astype(np.float32)
    dout = rng.normal(size=(n, widths[-1])).astype(np.float32)
    want, want_dx = s.input_grad(x, dout)
    at_x, at_o, size = _place(kind, x.size, want.size)

    def ptr(a, at):
        return a[at:].ctypes.data_as(f32p)
    buf = np.zeros(size, np.float32)
    buf[at_x:at_x + x.size] = x.ravel()
    assert s.lib.arbo_sur_forward(s._h, n, ptr(buf, at_x), ptr(buf, at_o)) == 0
    assert np.array_equal(buf[at_o:at_o + want.size], want.ravel())

    dev = hip.upload(np.concatenate([np.zeros(at_x, np.float32), x.ravel(),
                                     np.zeros(size - at_x - x.size, np.float32)]))
    base = dev.value
    assert s.lib.arbo_sur_forward_noalloc(s._h, n, ctypes.c_void_p(base + 4 * at_x), ctypes.c_void_p(base + 4 * at_o), None) == 0
    hip.check(hip.lib.hipDeviceSynchronize(), "hipDeviceSynchronize")
    got = hip.download(dev, (size,))[at_o:at_o + want.size]
    if n * widths[0] > 1 << 21 and not (at_x == at_o and widths[0] == widths[-1]):
        assert rel(got, want) < 1e-4
    else:
        assert np.array_equal(got, want.ravel())
    hip.check(hip.lib.hipFree(dev), "hipFree")

    # the gradient in the inputs' place and the outputs in dout's, outputs over
    # the inputs, the gradient over dout
    buf = np.zeros(size, np.float32)
    buf[at_x:at_x + x.size] = x.ravel()
    y = dout.ravel().copy()
    assert s.lib.arbo_sur_input_grad(s._h, n, ptr(buf, at_x), ptr(y, 0), ptr(y, 0), ptr(buf, at_x)) == 0
    assert np.array_equal(y, want.ravel()) and np.array_equal(buf[at_x:at_x + x.size], want_dx.ravel())
    buf[at_x:at_x + x.size] = x.ravel()
    dx = np.empty_like(x)
    assert s.lib.arbo_sur_input_grad(s._h, n, ptr(buf, at_x), ptr(dout.ravel(), 0), ptr(buf, at_o), ptr(dx.ravel(), 0)) == 0
    assert np.array_equal(buf[at_o:at_o + want.size], want.ravel()) and np.array_equal(dx, want_dx)
    at_y, at_d, size = _place(kind, want.size, x.size)
    buf = np.zeros(size, np.float32)
    buf[at_y:at_y + want.size] = dout.ravel()
    assert s.lib.arbo_sur_input_grad(s._h, n, ptr(x.ravel(), 0), ptr(buf, at_y), None, ptr(buf, at_d)) == 0
    assert np.array_equal(buf[at_d:at_d + x.size], want_dx.ravel())
    s.close()


@pytest.mark.parametrize("widths,rows", [([6, 16, 4], (43679, 43680, 43681, 87365)), ([20, 16, 260], (1007, 1009, 2017)),
                                         ([300, 33, 74], (1747, 1748, 2500)), ([300, 33, 75], (1748,)),
                                         ([301, 33, 1], (869, 870, 871, 1741, 1742, 6000))],
                         ids=lambda w: "-".join(map(str, w)) if isinstance(w, list) else None)
def test_host_rows_in_chunks_of_bytes(hip_lib, widths, rows):
    """Host calls around the rows of a 1 MB chunk (2^20 / (4 x the wider of
    inputs and outputs), a multiple of 16), and around the 2 MB of inputs from
    which a forward call of few outputs copies them: every row as in calls of
    fewer rows."""
    s = Surrogate(widths, max_batch=rows[-1], seed=6, lib=hip_lib)
    rng = np.random.default_rng(7)
    x = rng.normal(size=(rows[-1], widths[0])).astype(np.float32)
    dout = rng.normal(size=(rows[-1], widths[-1])).astype(np.float32)
    parts = [s.input_grad(x[i:i + 800], dout[i:i + 800]) for i in range(0, rows[-1], 800)]
    out, dx = (np.concatenate([p[k] for p in parts]) for k in (0, 1))
    for n in rows:
        print(f"[tiles] host chunks widths={widths} rows={n}", flush=True)
        assert np.array_equal(s.forward(x[:n]), out[:n])
        got_out, got_dx = s.input_grad(x[:n], dout[:n])
        assert np.array_equal(got_out, out[:n]) and np.array_equal(got_dx, dx[:n])
    s.close()


@pytest.mark.parametrize("widths", [[1, 1], [6, 33, 12], [5, 17, 300, 64, 7], [6, 520, 9]], ids=lambda w: "-".join(map(str, w)))
def test_new_parameters_start_afresh(hip_lib, widths):
    """set_params after a training: its weights are the ones the next calls
    read, and the next training starts from zero moments, as a surrogate's
    first one does."""
    rng = np.random.default_rng(14)
    x = rng.normal(size=(40, widths[0])).astype(np.float32)
    y = rng.poisson(2.0, size=(40, widths[-1])).astype(np.float32)
    p = flatten(random_layers(widths, 15))
    got = []
    for before in (False, True):
        s = Surrogate(widths, max_batch=64, seed=16, lib=hip_lib)
        if before:
            s.train(x, y, epochs=2, batch=16, lr=1e-2, seed=17)
        s.set_params(p)
        out = s.forward(x)
        s.train(x, y, epochs=1, batch=16, lr=1e-3, seed=18)
        got.append((out, s.get_params(), s.forward(x)))
        s.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("inputs", [1, 31, 32, 33, 63, 64, 65, 255, 256, 257, 319, 320, 511, 512])
def test_rows_of_any_width_are_read(hip_lib, inputs):
    """Input widths around the columns that a row's loads take at once; a NaN
    in a row's first column, which loads past the last column read, stays in
    its row."""
    print(f"[tiles] inputs={inputs}", flush=True)
    layers = random_layers([inputs, 24, 9], 23)
    s = Surrogate([inputs, 24, 9], max_batch=64, seed=24, lib=hip_lib)
    s.set_params(flatten(layers))
    x = np.random.default_rng(25).normal(size=(37, inputs)).astype(np.float32)
    out = s.forward(x)
    assert rel(out, forward64(layers, x)[0]) < 1e-4
    x[5, 0] = np.nan
    bad = s.forward(x)
    assert np.all(np.isnan(bad[5])) and np.array_equal(np.delete(bad, 5, 0), np.delete(out, 5, 0))
    s.close()
