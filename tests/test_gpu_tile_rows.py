"""The large GEMM's tiles of 192 and 128 rows (kernels.hip choose_gemm,
gemm_core.h alternating_kloop): row counts that take them in one round of the
CUs and in several, with a ragged last tile, few and odd K steps, N not a
multiple of 256 and of 4.  INT8 bit for bit with the oracle, with the fused
requantization (certified GELU and plain), its deferral and capture; FP16
per op, and its operand hand-off against the separate conversion; FP32 per op."""
import pytest

from conftest import assert_bitexact_f32
from test_gpu_fp16 import check_per_op as check_fp16
from test_gpu_fp32 import check_per_op as check_fp32
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

CASES = [
    # rows, dims, tile rows of the wide layer
    (2890, (130, 4096, 40), 192),   # 16 x 16 tiles, the last one of 10 rows; 3 K steps
    (5900, (64, 4096, 24), 192),    # 31 x 16 = 496: two rounds
    (2570, (200, 2972, 33), 128),   # 21 x 12 = 252 tiles
    (2600, (330, 3002, 20), 128),   # N % 4: no fused requantization
]


def _rows_of(m, n):
    best = None
    mpad, npad = -(-m // 256) * 256, -(-n // 256) * 256
    for bm in (256, 192, 128):
        tm = -(-m // bm)
        if tm * bm > mpad:
            continue
        cost = -(-tm * (npad // 256) // 256) * (bm + 104)
        if best is None or cost < best[0]:
            best = (cost, bm)
    return best[1]


def _layers(rg, dims, act):
    from rustgears_amd import nn
    rg.manual_seed(sum(dims))
    m = nn.Sequential()
    for a, b in zip(dims[:-1], dims[1:]):
        m.add(nn.Linear(a, b)).add(act())
    return m.export()


@pytest.mark.parametrize("rows,dims,bm", CASES, ids=[f"{r}x{d[1]}" for r, d, _ in CASES])
def test_int8(rg, ref, monkeypatch, rows, dims, bm):
    from rustgears_amd import nn
    assert _rows_of(rows, dims[1]) == bm
    x = rg.randn([rows, dims[0]])
    for act in (nn.Gelu, nn.Tanh):
        layers = _layers(rg, dims, act)
        want = ref.RefProgram(layers).run(x, parallel=True)
        for spin in (None, "0"):
            if spin:
                monkeypatch.setenv("RGNPU_REQUANT_SPIN_LIMIT", spin)
            print(f"[tile rows] int8 {rows} {dims} {act.__name__} spin {spin}", flush=True)
            sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_int8())
            assert_bitexact_f32(sess.run(x), want, f"{rows} {dims}")
            sess.close()
            monkeypatch.delenv("RGNPU_REQUANT_SPIN_LIMIT", raising=False)
    check_against_oracle(rg, ref, _layers(rg, dims, nn.Relu), x, f"{rows} {dims} capture")


@pytest.mark.parametrize("rows,dims,bm", CASES, ids=[f"{r}x{d[1]}" for r, d, _ in CASES])
def test_fp16(rg, ref, monkeypatch, rows, dims, bm):
    from rustgears_amd import nn
    layers, x = _layers(rg, dims, nn.Relu), rg.randn([rows, dims[0]])
    check_fp16(rg, ref, layers, x, f"fp16 {rows} {dims}")
    outs = []
    for handoff in ("0", "1"):
        monkeypatch.setenv("RGNPU_F16_HANDOFF", handoff)
        sess = rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_fp16())
        outs.append(sess.run(x))
        sess.close()
    assert_bitexact_f32(outs[1], outs[0], "hand-off")


@pytest.mark.parametrize("rows,dims", [(2890, (36, 4096)), (2570, (36, 2972))], ids=["192", "128"])
def test_fp32(rg, ref, monkeypatch, rows, dims):
    from rustgears_amd import nn
    monkeypatch.setenv("RGNPU_MID", "0")  # FP32 takes smaller tiles at these shapes by itself
    check_fp32(rg, ref, _layers(rg, dims, nn.Relu), rg.randn([rows, dims[0]]), f"fp32 {rows} {dims}")

