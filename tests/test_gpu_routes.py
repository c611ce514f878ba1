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
