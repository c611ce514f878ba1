"""rgmath::half_bits (devmath.h) equals fp16_bits(round_fp16(x)) -- the binary16
operand of an FP16 value (quantize.rs:50-64) -- on every 7th f32 bit pattern;
all 2^32 with RG_EXHAUSTIVE=1."""
import os
import subprocess


def test_half_bits_equals_the_two_steps(tmp_path):
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "half_host_check.cpp")
    exe = str(tmp_path / "half_host_check")
    subprocess.run(["g++", "-O2", "-std=c++17", src, "-o", exe], check=True)
    stride = "1" if os.environ.get("RG_EXHAUSTIVE") == "1" else "7"
    out = subprocess.run([exe, stride], capture_output=True, text=True)
    checked, bad, first = out.stdout.split()
    assert int(checked) >= (1 << 32) // 7 and int(bad) == 0, (out.stdout, first)
