"""How far FP16 and FP32 sums are from 64 bits.

Every row (image) of the input is the same and the bias is minus the exact
sum, so an output is the error of its f32 sum (in FP16 to 11 bits of it).

A chain of n f32 additions of random terms errs by 0.415 u sqrt(n / 2) of its
result (u = 2^-24; a rounding is uniform, 0.415 u of what the sum holds, which
grows evenly); m runs of n that join a total by 0.415 u sqrt((n + m) / 2).  The
limits take that for the longest slice of K (a quarter of it), four more for
the slices' sums and the bias, and half as much again.  A chain over all of
the slice is past them.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _limit(run, runs):
    return 1.5 * 0.415 * U * np.sqrt((run + runs) / 2 + 4)


def _best(roundings):
    return _limit(np.sqrt(roundings), np.sqrt(roundings))


def _error(rg, make, x_row, w, shape, precision):
    """rms error of the sums over rms of the sums; `make` builds the layer from its bias."""
    exact = w.astype(np.float64) @ x_row.astype(np.float64).reshape(-1)
    bias = (-exact).astype(np.float32)
    x = np.ascontiguousarray(np.broadcast_to(x_row, shape), np.float32)
    provider = rg.ExecutionProvider.Gpu(0) if precision == "f32" else rg.ExecutionProvider.mi355x_fp16()
    sess = rg.InferenceSession.from_layers([make(bias)], provider)
    y = np.asarray(sess.run(x), np.float64).reshape(shape[0], -1)
    sess.close()
    assert np.array_equal(y, np.broadcast_to(y[0], y.shape)), "equal rows, equal sums"
    err = y - (exact + bias.astype(np.float64))
    return np.mean(err ** 2), np.mean(exact ** 2)


def _values(rng, precision, shape, scale):
    v = rng.uniform(-scale, scale, shape)
    if precision == "f16":  # what lies below 2^-14 counts as zero there
        v = np.where(np.abs(v) < 2.0 ** -13, 0, v).astype(np.float16)
    return v.astype(np.float32)


@pytest.mark.parametrize("precision", ["f32", "f16"])
@pytest.mark.parametrize("rows,k,n", [(16, 512, 10), (33, 1024, 10), (17, 4096, 16), (40, 8192, 5), (3, 14336, 640),
                                      (5, 8192, 1040), (12, 4096, 512), (100, 4096, 256), (100, 2048, 515),
                                      (300, 1024, 1024), (64, 14336, 300)])
def test_linear(rg, precision, rows, k, n):
    from rustgears_amd.inference import LayerSpec
    rng = np.random.default_rng(rows + k + n)
    sums = []
    for _ in range(max(1, 400 // n)):  # 400 sums or more
        # of ~2e4: their errors are above binary16's smallest, 2^-14
        x, w = _values(rng, precision, (k,), 6e4 / k ** 0.5), _values(rng, precision, (n, k), 1.0)
        sums.append(_error(rg, lambda b: LayerSpec.Linear(k, n, np.ascontiguousarray(w.T), b), x, w, (rows, k),
                           precision))
    e = np.sqrt(np.mean([a for a, _ in sums]) / np.mean([b for _, b in sums]))
    if precision == "f16":  # 8 products at a time
        limit = _best(k / 4 / 8)
    elif n <= 16 or rows <= 8:  # two chains
        limit = _best(k / 4 / 2)
    else:  # runs of 64 in each of two chains
        limit = _limit(64, k / 4 / 2 / 64)
    print(f"[sums lin] {precision} {rows}x{k}x{n} {e / U:.2f} u limit {limit / U:.2f} u", flush=True)
    assert e <= limit


@pytest.mark.parametrize("precision", ["f32", "f16"])
@pytest.mark.parametrize("images", [20, 3000])
@pytest.mark.parametrize("c,o,k", [(32, 64, 3), (60, 64, 3), (128, 40, 3), (16, 64, 5), (64, 33, 5), (64, 64, 7),
                                   (16, 40, 7), (256, 64, 1), (256, 96, 3)])
def test_conv(rg, precision, c, o, k, images):
    from rustgears_amd.inference import LayerSpec
    rng = np.random.default_rng(c + o + k)
    sums = []
    for _ in range(6):
        x = _values(rng, precision, (c, k, k), 6e4 / (c * k * k) ** 0.5)
        w = _values(rng, precision, (o, c * k * k), 1.0)
        sums.append(_error(rg, lambda b: LayerSpec.Conv2d(c, o, k, 1, 0, w.reshape(o, c, k, k), b), x, w,
                           (images, c, k, k), precision))
    e = np.sqrt(np.mean([a for a, _ in sums]) / np.mean([b for _, b in sums]))
    # FP32: runs of three taps of 16 products; FP16: of nine taps, every other one, 32 products 8 at a time
    if precision == "f32":
        limit = _limit(48, -(-c // 16) * -(-k * k // 3))
    else:
        limit = _limit(5 * 4, 2 * -(-c // 32) * -(-k * k // 9))
    print(f"[sums conv] {precision} conv {c}->{o} k {k} {images} images {e / U:.2f} u limit {limit / U:.2f} u", flush=True)
    assert e <= limit
