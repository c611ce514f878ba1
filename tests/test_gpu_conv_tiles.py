"""The tiles of the MFMA convolution (conv_mfma.hip conv_mfma_tile): 64, 128 or
256 pixels x 16, 32 or 64 channels by image size, batch and channels, each op
within the bound of a reordered f32 sum and the plan with the fused pool equal
to the separate kernels; and the deep layers on few pixels that im2col + GEMM
takes."""
import pytest

from conftest import assert_bitexact_f32
from test_gpu_fp16 import check_per_op as check_fp16
from test_gpu_fp32 import check_per_op as check_fp32

pytestmark = pytest.mark.gpu

CASES = [
    # images, C, O, (H, W), k, pad: pixels x channels of a workgroup
    (1, 40, 64, (6, 6), 3, 1),      # 64 x 16: one workgroup per 16 channels
    (9, 33, 130, (7, 7), 3, 1),     # 64 x 16, ragged channels
    (130, 20, 64, (8, 8), 3, 1),    # 64 x 16
    (300, 17, 64, (7, 7), 3, 1),    # 64 x 32 or 64: the image fits the smallest tile
    (400, 17, 70, (5, 9), 3, 1),    # 64 x 64, two channel blocks
    (130, 33, 200, (11, 11), 3, 1),  # 128: rows of 11 fill no 64
    (40, 12, 64, (30, 40), 3, 1),   # 256: 6 rows of 40
    (2, 24, 96, (5, 64), 3, 1),     # 128 with a pool (one row of 64 has no pair), 16 channels
    (3, 20, 30, (9, 100), 5, 2),    # two column tiles
]


def _model(rg, c, o, k, pad, pool):
    from rustgears_amd import nn
    rg.manual_seed(c * 100 + o)
    m = nn.Sequential().add(nn.Conv2d(c, o, k).padding(pad)).add(nn.Relu())
    return (m.add(nn.MaxPool2d(2)) if pool else m).export()


@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c[:3] + c[3])) for c in CASES])
def test_tiles(rg, ref, monkeypatch, case):
    n, c, o, hw, k, pad = case
    x = rg.randn([n, c, *hw])
    for provider, check in ((rg.ExecutionProvider.mi355x_fp16(), check_fp16), (rg.ExecutionProvider.Gpu(0), check_fp32)):
        check(rg, ref, _model(rg, c, o, k, pad, False), x, f"{case}")
        layers, outs = _model(rg, c, o, k, pad, True), []
        for fused in ("1", "0"):
            monkeypatch.setenv("RGNPU_CONV_POOL", fused)
            sess = rg.InferenceSession.from_layers(layers, provider)
            outs.append(sess.run(x))
            sess.close()
        monkeypatch.delenv("RGNPU_CONV_POOL")
        assert_bitexact_f32(outs[0], outs[1], f"{case} pool")


@pytest.mark.parametrize("n,c,hw,im2col", [(1, 512, 7, True), (4, 512, 7, True), (64, 512, 7, False),
                                           (16, 256, 7, False), (1, 1024, 3, True)])
def test_deep_layers_on_few_pixels(rg, ref, n, c, hw, im2col):
    layers = _model(rg, c, c, 3, 1, False)
    x = rg.randn([n, c, hw, hw])
    check_fp16(rg, ref, layers, x, f"{n} x {c} x {hw}")
    sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_fp16())
    sess.run(x)
    r = sess.last_npu_profile().records[0]
    sess.close()
    # im2col runs before the op's main kernel
    assert (r.duration_ns > r.kernel_ns) == im2col, r


@pytest.mark.parametrize("hw", [4, 6, 8, 11])
def test_small_images_pool_in_the_convolution(rg, hw):
    """Images of fewer than 128 pixels too: the pool launches nothing and the
    Linear after it converts nothing."""
    from rustgears_amd import nn
    rg.manual_seed(hw)
    layers = (nn.Sequential().add(nn.Conv2d(32, 64, 3).padding(1)).add(nn.Relu()).add(nn.MaxPool2d(2))
              .add(nn.Flatten()).add(nn.Linear(64 * (hw // 2) ** 2, 64))).export()
    sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_fp16())
    sess.run(rg.randn([20, 32, hw, hw]))
    conv, pool, _, linear = sess.last_npu_profile().records
    sess.close()
    assert conv.kernel_ns > 0 and pool.duration_ns == 0, (conv, pool)
    assert linear.duration_ns == linear.kernel_ns > 0, linear
