"""Convolutions of more workgroups than one grid dimension holds (2^32 threads):
2^24 images of one pixel on the direct kernel, and 2^24 tiles of images and output
channels, which im2col + GEMM takes over from the MFMA kernel."""
import numpy as np
import pytest

from conftest import assert_bitexact_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f32", "f16"])
def test_direct_conv(rg, precision):
    from rustgears_amd import nn
    rg.manual_seed(1)
    layers = nn.Sequential().add(nn.Conv2d(1, 2, 1)).add(nn.Relu()).export()
    provider = rg.ExecutionProvider.Gpu(0) if precision == "f32" else rg.ExecutionProvider.mi355x_fp16()
    sess = rg.InferenceSession.from_layers(layers, provider)
    n = (1 << 24) + 300
    x = np.tile(rg.randn([4099, 1, 1, 1]), (n // 4099 + 1, 1, 1, 1))[:n]
    want = np.asarray(sess.run(x[:4099]))
    print(f"[limits] direct {precision} {n}", flush=True)
    y = np.asarray(sess.run(x)).reshape(n, 2)
    sess.close()
    for at in range(0, n - 4099, 4099 * 400):
        assert_bitexact_f32(y[at:at + 4099], want, f"image {at}")
    assert_bitexact_f32(y[-300:], want.reshape(-1, 2)[np.arange(n - 300, n) % 4099], "last images")


def test_mfma_conv(rg):
    from rustgears_amd import _native as N
    from rustgears_amd.inference import DeviceBuffer, LayerSpec
    n, c, o = 1 << 18, 33, 4096
    rg.manual_seed(2)
    w, b, x = rg.randn([o, c, 1, 1]), rg.randn([o]), rg.randn([n, c, 1, 1])
    sess = rg.InferenceSession.from_layers([LayerSpec.Conv2d(c, o, 1, 1, 0, w, b)], rg.ExecutionProvider.Gpu(0))
    d_x, d_y = DeviceBuffer.from_array(x), DeviceBuffer(n * o * 4)
    print("[limits] mfma", flush=True)
    sess.run_device(d_x, x.shape, d_y)
    sess.synchronize()
    sess.close()
    w64, b64 = np.asarray(w, np.float64).reshape(o, c), np.asarray(b, np.float64)
    y = np.empty((256, o), np.float32)
    for at in [*range(0, n, n // 8), n - 256]:
        N.check(N.lib().rgnpu_memcpy_d2h(y.ctypes.data, d_y.ptr + at * o * 4, y.nbytes))
        rows = np.asarray(x[at:at + 256], np.float64).reshape(256, c)
        want, mass = rows @ w64.T + b64, np.abs(rows) @ np.abs(w64).T + np.abs(b64)
        assert np.all(np.abs(y - want) <= (c + 2) * 2.0 ** -24 * mass), at
    d_x.free()
    d_y.free()
