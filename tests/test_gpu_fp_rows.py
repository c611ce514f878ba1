"""FP16 and FP32 Linears on 1 to 8 rows: the GEMV and, from 2 rows and 16 MB of
weights on, the small-tile GEMM (mid.hip), with the FP16 operand hand-off from
either (the GEMV's only where the operand has no padding columns)."""
import pytest

from conftest import assert_bitexact_f32
from test_gpu_fp16 import check_per_op as check_fp16
from test_gpu_fp32 import check_per_op as check_fp32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 5, 8])
@pytest.mark.parametrize("dims", [(96, 4096, 2080, 33), (130, 515, 64, 7), (2052, 4100, 50)],
                         ids=["16 MB", "small", "ragged 33 MB"])
def test_rows(rg, ref, monkeypatch, rows, dims):
    from rustgears_amd import nn
    rg.manual_seed(rows + dims[0])
    m = nn.Sequential()
    for a, b in zip(dims[:-1], dims[1:]):
        m.add(nn.Linear(a, b)).add(nn.Relu())
    layers, x = m.export(), rg.randn([rows, dims[0]])
    what = f"{rows} rows {dims}"
    for mid in ("1", "2"):
        monkeypatch.setenv("RGNPU_MID", mid)
        check_fp16(rg, ref, layers, x, f"fp16 {what} mid {mid}")
        check_fp32(rg, ref, layers, x, f"fp32 {what} mid {mid}")
        outs = []
        for handoff in ("0", "1"):
            monkeypatch.setenv("RGNPU_F16_HANDOFF", handoff)
            sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_fp16())
            outs.append(sess.run(x))
            sess.close()
        monkeypatch.delenv("RGNPU_F16_HANDOFF")
        assert_bitexact_f32(outs[1], outs[0], f"{what}: hand-off")
