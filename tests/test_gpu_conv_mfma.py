"""FP16 and FP32 convolutions in one implicit GEMM kernel (conv_mfma.hip).

Shapes on the edges of its tiling: channels below, at and past a 64-byte block
(32 binary16, 16 f32) and over several, output channels at and past the 16, 32
and 64 of a workgroup, images narrower and wider than the 64-pixel tile, odd
sizes, strides, paddings, windows of 1 to 7 (more taps than are staged at
once), one image and many.  Each op is checked on its own captured input
within the bound of a reordered f32 sum (test_gpu_fp16 / test_gpu_fp32), the
production plan (pool, activation and operand hand-off in the kernel) must give
the bits of the separate kernels, and im2col + GEMM stays within the same bound.
"""
import numpy as np
import pytest

from conftest import assert_bitexact_f32
from test_gpu_fp16 import check_per_op as check_fp16
from test_gpu_fp32 import check_per_op as check_fp32

pytestmark = pytest.mark.gpu

CASES = [
    # name, images, C, O, (H, W), k, stride, pad, pool, tail
    ("cnn conv2", 5, 32, 64, (16, 16), 3, 1, 1, True, "linear"),
    ("one channel over a block, odd size", 3, 33, 17, (13, 11), 3, 1, 1, True, "linear"),
    ("two blocks, 65 outputs", 2, 64, 65, (12, 24), 3, 1, 1, True, "conv"),
    ("wide image", 1, 5, 20, (6, 131), 3, 1, 1, True, None),
    ("direct taps, too many outputs", 2, 3, 70, (18, 18), 3, 1, 1, True, "linear"),
    ("stride 2", 3, 17, 32, (15, 21), 3, 2, 1, False, None),
    ("window 1", 4, 48, 16, (19, 7), 1, 1, 0, True, "linear"),
    ("window 7", 2, 16, 40, (20, 14), 7, 1, 3, True, None),
    ("window 5, stride 3, no padding", 2, 9, 33, (23, 17), 5, 3, 0, False, "conv"),
    ("many images of one pixel", 70, 40, 24, (3, 3), 3, 1, 0, False, "linear"),
    ("two rows", 9, 24, 100, (2, 66), 3, 1, 1, True, "linear"),
]
IDS = [c[0] for c in CASES]


def _model(rg, c, o, hw, k, stride, pad, pool, tail):
    from rustgears_amd import nn
    rg.manual_seed(c * 100 + o)
    m = nn.Sequential().add(nn.Conv2d(c, o, k).stride(stride).padding(pad)).add(nn.Relu())
    h, w = ((d + 2 * pad - k) // stride + 1 for d in hw)
    if pool:
        m.add(nn.MaxPool2d(2))
        h, w = h // 2, w // 2
    if tail == "linear":
        m.add(nn.Flatten()).add(nn.Linear(o * h * w, 21)).add(nn.Relu()).add(nn.Linear(21, 9))
    elif tail == "conv":
        m.add(nn.Conv2d(o, 20, 3).padding(1)).add(nn.Relu())
    return m.export()


def _run(rg, layers, x, provider, monkeypatch, **env):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    sess = rg.InferenceSession.from_layers(layers, provider)
    y = sess.run(x)
    assert_bitexact_f32(sess.run(x), y, "second run")
    sess.close()
    for k in env:
        monkeypatch.delenv(k)
    return y


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_fp16(rg, ref, monkeypatch, case):
    name, n, c, o, hw, k, stride, pad, pool, tail = case
    layers = _model(rg, c, o, hw, k, stride, pad, pool, tail)
    x = rg.randn([n, c, *hw])
    check_fp16(rg, ref, layers, x, f"conv mfma fp16 {name}")
    monkeypatch.setenv("RGNPU_CONV_MFMA", "0")
    check_fp16(rg, ref, layers, x, f"im2col fp16 {name}")
    monkeypatch.delenv("RGNPU_CONV_MFMA")
    p = rg.ExecutionProvider.mi355x_fp16()
    y = _run(rg, layers, x, p, monkeypatch)
    y0 = _run(rg, layers, x, p, monkeypatch, RGNPU_CONV_POOL="0", RGNPU_F16_HANDOFF="0")
    assert_bitexact_f32(y, y0, f"{name}: fused")


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_fp32(rg, ref, monkeypatch, case):
    name, n, c, o, hw, k, stride, pad, pool, tail = case
    layers = _model(rg, c, o, hw, k, stride, pad, pool, tail)
    x = rg.randn([n, c, *hw])
    check_fp32(rg, ref, layers, x, f"conv mfma fp32 {name}")
    p = rg.ExecutionProvider.Gpu(0)
    y = _run(rg, layers, x, p, monkeypatch)
    y0 = _run(rg, layers, x, p, monkeypatch, RGNPU_CONV_POOL="0")
    assert_bitexact_f32(y, y0, f"{name}: fused")


def test_special_values(rg, monkeypatch):
    """FP32: NaN and infinite inputs and bias channels through the fused
    activation and pool give what the separate kernels give."""
    layers = _model(rg, 20, 40, (10, 14), 3, 1, 1, True, None)
    layers[0].bias[[1, 30]] = np.float32(np.nan)
    layers[0].bias[[2, 39]] = np.float32(-np.inf)
    x = rg.randn([3, 20, 10, 14])
    x[0, 3, 4, 5], x[1, 7, 0, 0], x[2, 19, 9, 13] = np.nan, np.inf, -np.inf
    p = rg.ExecutionProvider.Gpu(0)
    y = _run(rg, layers, x, p, monkeypatch)
    assert_bitexact_f32(y, _run(rg, layers, x, p, monkeypatch, RGNPU_CONV_POOL="0"), "special values")
