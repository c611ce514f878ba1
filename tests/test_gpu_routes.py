"""Which kernel a Linear takes where two can do it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(rg, monkeypatch, layers, x, mid):
    if mid is None:
        monkeypatch.delenv("RGNPU_MID", raising=False)
    else:
        monkeypatch.setenv("RGNPU_MID", mid)
    sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.Gpu(0))
    y = sess.run(x)
    sess.close()
    return y


@pytest.mark.parametrize("rows,k,n,small_tiles", [(777, 4096, 4096, False), (1300, 1024, 8192, False),
                                                  (1300, 4096, 4096, True), (400, 4096, 4096, True),
                                                  (1000, 1024, 1024, True), (2000, 1024, 1024, True)])
def test_fp32_small_tiles_or_large(rg, monkeypatch, rows, k, n, small_tiles):
    """FP32 on the small-tile GEMM only where it is the faster one; the two sum
    in different orders, so the bits tell which one ran."""
    from rustgears_amd.inference import LayerSpec
    rg.manual_seed(rows)
    layers = [LayerSpec.Linear(k, n, rg.randn([k * n]), rg.randn([n]))]
    x = rg.randn([rows, k])
    y, large, small = (_run(rg, monkeypatch, layers, x, mid) for mid in (None, "0", "2"))
    assert not np.array_equal(large, small)
    assert np.array_equal(y, small if small_tiles else large)


@pytest.mark.parametrize("rows,k,n,small_tiles", [(9, 1024, 8192, True), (128, 512, 8192, True), (12, 512, 14000, True),
                                                  (128, 512, 14000, False), (9, 384, 8192, False),
                                                  (300, 512, 4096, False)])
def test_int8_up_to_128_rows(rg, ref, monkeypatch, rows, k, n, small_tiles):
    """An INT8 Linear on up to 128 rows has half of the tiles of its padded 256;
    on the small-tile GEMM the next Linear quantizes its input in a pass of its
    own, on the tile GEMM it comes quantized."""
    from conftest import assert_bitexact_f32
    from rustgears_amd import nn
    monkeypatch.setenv("RGNPU_SMALL_XQ", "0")  # which would quantize as it reads
    rg.manual_seed(rows + n)
    layers = nn.Sequential().add(nn.Linear(k, n)).add(nn.Relu()).add(nn.Linear(n, 40)).export()
    x = rg.randn([rows, k])
    sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_int8())
    assert_bitexact_f32(sess.run(x), ref.RefProgram(layers).run(x, parallel=True), f"{rows} {k} {n}")
    second = sess.last_npu_profile().records[1]
    sess.close()
    assert (second.duration_ns > second.kernel_ns) == small_tiles, second


def test_the_tile_is_chosen_with_the_plan(rg, monkeypatch):
    """The environment is read when a plan is made, not by each run: another
    thread may be setting a variable then."""
    from rustgears_amd.inference import LayerSpec
    rg.manual_seed(3)
    layers = [LayerSpec.Linear(3000, 200, rg.randn([600000]), rg.randn([200]))]
    x = rg.randn([40, 3000])
    sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.Gpu(0))
    monkeypatch.setenv("RGNPU_MID_TILE", "0")
    y = sess.run(x)
    monkeypatch.setenv("RGNPU_MID_TILE", "6")  # sums over half as many slices of K
    assert np.array_equal(sess.run(x), y)
    other = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.Gpu(0))
    assert not np.array_equal(other.run(x), y)
    sess.close()
    other.close()
