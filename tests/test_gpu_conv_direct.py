"""Direct FP16 and FP32 convolutions (conv_direct.hip): windows of at most 32
taps and at most 64 output channels, bit-exact with the oracle, which sums in
the same serial order.

The tap count is rounded up to a compiled one (9, 18, 27 or 32), so every
count between has taps that must add nothing whatever the input holds.
"""
import numpy as np
import pytest

from conftest import assert_bitexact_f32

pytestmark = pytest.mark.gpu


def _run(rg, ref, c, o, k, stride, pad, x, relu, pool, precision="f32"):
    from rustgears_amd import nn
    rg.manual_seed(c * 100 + o * 10 + k)
    m = nn.Sequential().add(nn.Conv2d(c, o, k).stride(stride).padding(pad))
    if relu:
        m.add(nn.Relu())
    if pool:
        m.add(nn.MaxPool2d(2))
    layers = m.export()
    provider = rg.ExecutionProvider.Gpu(0) if precision == "f32" else rg.ExecutionProvider.mi355x_fp16()
    sess = rg.InferenceSession.from_layers(layers, provider)
    y = sess.run(x)
    sess.close()
    want = ref.RefProgram(layers, precision=ref.FP32 if precision == "f32" else ref.FP16).run(x, parallel=True)
    what = f"{precision} {c}->{o} k {k} stride {stride} pad {pad} {x.shape} relu {relu} pool {pool}"
    assert_bitexact_f32(y, want, what)
    return np.asarray(y)


@pytest.mark.parametrize("relu", [False, True], ids=["none", "relu"])
@pytest.mark.parametrize("hw", [(6, 12), (16, 16), (4, 32), (6, 2900)], ids=["band", "pool 16", "pool 32", "no band"])
@pytest.mark.parametrize("c,k", [(1, 5), (2, 2), (1, 2), (3, 2), (3, 1), (1, 1), (7, 2), (3, 3)],
                         ids=["25 taps", "8", "4", "12", "3", "1", "28", "27"])
def test_fp32_infinite_inputs(rg, ref, c, k, hw, relu):
    """+-Inf and NaN at the last tap of a window, alone and beside finite and
    other infinite values: the sums of the oracle, not NaN for infinity times the
    zero weight of a tap that does not exist."""
    x = rg.randn([3, c, *hw])
    h, w = hw
    x[0, c - 1, h - 1, w - 1] = np.inf
    x[0, 0, 2, 3] = -np.inf
    x[1, c - 1, 3, 4], x[1, c - 1, 3, 7] = -np.inf, np.nan
    x[2, c - 1, 2, 2:4] = np.inf, -np.inf
    pad = k // 2
    oh, ow = h + 2 * pad - k + 1, w + 2 * pad - k + 1
    for pool in (False, True) if oh % 2 == 0 and ow in (16, 32) else (False,):
        y = _run(rg, ref, c, 20, k, 1, pad, x, relu, pool)
    assert relu or np.isinf(y).any()


@pytest.mark.parametrize("precision", ["f32", "f16"])
@pytest.mark.parametrize("n,c,o,k,stride,pad,hw,relu,pool", [
    # images too wide for the LDS band (32 KiB)
    (2, 3, 20, 3, 1, 1, (6, 700), True, False), (2, 3, 64, 3, 2, 1, (7, 1500), False, False),
    (1, 1, 17, 5, 1, 2, (5, 1400), True, False),
    # 32 channels per thread (768 workgroups or more), the second block of them partly past the last channel
    (400, 3, 40, 3, 1, 1, (16, 16), True, True), (400, 3, 60, 3, 1, 1, (16, 16), False, False),
    (200, 3, 60, 3, 1, 1, (16, 32), True, True), (400, 2, 33, 3, 1, 1, (13, 19), False, False),
    (800, 1, 64, 2, 1, 0, (9, 17), True, False),
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_wide_images_and_many_channels(rg, ref, precision, n, c, o, k, stride, pad, hw, relu, pool):
    rg.manual_seed(n)
    _run(rg, ref, c, o, k, stride, pad, rg.randn([n, c, *hw]), relu, pool, precision)
