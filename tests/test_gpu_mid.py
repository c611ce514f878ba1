"""The small-tile GEMM (mid.hip gemm_mid_kernel): Linears on more than 8 rows
whose 128 x 128 tiles would not fill the chip.

Every tile shape (forced with RGNPU_MID_TILE, RGNPU_MID=2) on rows and columns
one below, at and one above its edges, K shorter than one 64-byte block, in
the last block of a stage, at and past a stage, and more stages than the ring
holds, against the oracle: INT8 bit for bit (with and without capture), FP32
and FP16 within the bound of a reordered f32 sum.  Each f32 summation of K
products is within K u sum|p| of the exact sum (u = 2^-24), so two orders are
within 2K u sum|p|; the bias and the activation add a rounding each, FP16 at
most one binary16 step where the sums round differently.  The FP16 hand-off
must equal the separate conversion bit for bit, and a FP32 Linear that applies
the Act op after it the separate Act kernel (capture keeps that one).
"""
import numpy as np
import pytest

from conftest import assert_bitexact_f32
from test_gpu_fp16 import check_per_op as check_fp16
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

TILES = [(16, 16), (16, 32), (16, 64), (32, 32), (64, 32), (32, 64), (64, 64), (128, 64), (64, 128)]
KS = [5, 64, 128, 252, 516, 2052]


def _layers(rg, k, n, n2, relu=False):
    from rustgears_amd import nn
    rg.manual_seed(k * 7 + n)
    a, b = (nn.Relu(), nn.Relu()) if relu else (nn.Gelu(), nn.LeakyRelu(0.05))
    return nn.Sequential().add(nn.Linear(k, n)).add(a).add(nn.Linear(n, n2)).add(b).export()


def _shapes(tile):
    tm, tn = TILES[tile]
    for i, k in enumerate(KS):
        rows = max(9, (tm - 1, tm, tm + 1)[i % 3])
        yield rows, k, (tn + 1, max(17, tn - 1), 2 * tn)[i % 3], (20, 33)[i % 2]


@pytest.mark.parametrize("tile", range(len(TILES)), ids=[f"{a}x{b}" for a, b in TILES])
def test_int8_tiles(rg, ref, monkeypatch, tile):
    monkeypatch.setenv("RGNPU_MID", "2")
    monkeypatch.setenv("RGNPU_MID_TILE", str(tile))
    for rows, k, n, n2 in _shapes(tile):
        layers, x = _layers(rg, k, n, n2), rg.randn([rows, k])
        what = f"tile {TILES[tile]} {rows}x{k}x{n}x{n2}"
        print(f"[mid i8] {what}", flush=True)
        want = ref.RefProgram(layers).run(x, parallel=True)
        for small in ("0", "1"):  # the second Linear here, or quantizing as it reads
            monkeypatch.setenv("RGNPU_SMALL_XQ", small)
            sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_int8())
            assert_bitexact_f32(sess.run(x), want, what)
            assert_bitexact_f32(sess.run(x), want, what + " (second run)")
            sess.close()
        check_against_oracle(rg, ref, layers, x, what + " capture")


@pytest.mark.parametrize("tile", range(len(TILES)), ids=[f"{a}x{b}" for a, b in TILES])
def test_fp16_tiles(rg, ref, monkeypatch, tile):
    monkeypatch.setenv("RGNPU_MID", "2")
    monkeypatch.setenv("RGNPU_MID_TILE", str(tile))
    for rows, k, n, n2 in _shapes(tile):
        # ReLU: check_fp16 takes the binary16 step at the output, and only where
        # the activation is the identity is that the step of the rounded sum (a
        # GELU output of 0.86 has a step of 2^-11, the sum 1.04 before it 2^-10)
        layers, x = _layers(rg, k, n, n2, relu=True), rg.randn([rows, k])
        what = f"f16 tile {TILES[tile]} {rows}x{k}x{n}x{n2}"
        check_fp16(rg, ref, layers, x, what)
        outs = []
        for handoff in ("0", "1"):
            monkeypatch.setenv("RGNPU_F16_HANDOFF", handoff)
            sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_fp16())
            outs.append(sess.run(x))
            sess.close()
        monkeypatch.delenv("RGNPU_F16_HANDOFF")
        assert_bitexact_f32(outs[1], outs[0], what + " hand-off")


@pytest.mark.parametrize("tile", range(len(TILES)), ids=[f"{a}x{b}" for a, b in TILES])
def test_fp32_tiles(rg, ref, monkeypatch, tile):
    monkeypatch.setenv("RGNPU_MID", "2")
    monkeypatch.setenv("RGNPU_MID_TILE", str(tile))
    for rows, k, n, n2 in _shapes(tile):
        layers, x = _layers(rg, k, n, n2), rg.randn([rows, k])
        what = f"f32 tile {TILES[tile]} {rows}x{k}x{n}x{n2}"
        print(f"[mid f32] {what}", flush=True)
        sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.Gpu(0))
        y = sess.run(x)
        sess.set_capture(True)
        assert_bitexact_f32(sess.run(x), y, what + " separate Act kernels")
        outs = [sess.capture(i, 3) for i in range(4)]
        sess.close()
        u, a = 2.0 ** -24, x
        for op in (0, 2):  # each Linear on its own captured input
            w, b = layers[op].weight.reshape(a.shape[1], -1).astype(np.float64), layers[op].bias.astype(np.float64)
            got, a64 = outs[op].reshape(rows, -1), a.astype(np.float64)
            want, mass = a64 @ w + b, np.abs(a64) @ np.abs(w) + np.abs(b)
            assert np.all(np.abs(got - want) <= (2 * a.shape[1] + 4) * u * mass), (what, op)
            a = outs[op + 1].reshape(rows, -1)


@pytest.mark.parametrize("rows,dims", [(100, (512, 1024, 1024, 300)), (777, (784, 1024, 1024, 10)),
                                       (33, (1024, 2048, 515, 9)), (300, (1200, 4096, 64))])
def test_default_choice(rg, ref, rows, dims):
    """What the plan picks by itself, INT8 bit for bit and FP16 per op."""
    from rustgears_amd import nn
    rg.manual_seed(rows)
    m = nn.Sequential()
    for a, b in zip(dims[:-1], dims[1:]):
        m.add(nn.Linear(a, b)).add(nn.Relu())
    layers, x = m.export(), rg.randn([rows, dims[0]])
    print(f"[mid] default {rows} {dims}", flush=True)
    sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_int8())
    assert_bitexact_f32(sess.run(x), ref.RefProgram(layers).run(x, parallel=True), f"default {rows} {dims}")
    sess.close()
    check_fp16(rg, ref, layers, x, f"f16 default {rows} {dims}")
