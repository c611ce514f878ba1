"""The profile of a run among others: two event sets are used in turn, and a run
behind one still under way takes that one's last kernel as its start."""
import pytest

from conftest import assert_bitexact_f32

pytestmark = pytest.mark.gpu

DIMS = (1024, 4096, 4096, 300)


def _session(rg):
    from rustgears_amd import nn
    rg.manual_seed(5)
    m = nn.Sequential()
    for a, b in zip(DIMS[:-1], DIMS[1:]):
        m.add(nn.Linear(a, b)).add(nn.Relu())
    layers = m.export()
    return layers, rg.InferenceSession.from_layers(layers, rg.ExecutionProvider.mi355x_int8())


def _buffers(rg, rows):
    from rustgears_amd.inference import DeviceBuffer
    x = rg.randn([rows, DIMS[0]])
    return x, DeviceBuffer.from_array(x), DeviceBuffer(rows * DIMS[-1] * 4)


def _check(prof, rows):
    assert [r.macs for r in prof.records] == [rows * a * b for a, b in zip(DIMS[:-1], DIMS[1:])]
    ops = sum(r.duration_ns for r in prof.records)
    assert all(r.duration_ns >= r.kernel_ns > 0 for r in prof.records), prof.records
    # the ops follow one another from the run's start to its end (float ms, rounded per op)
    assert abs(prof.total_time_ns - ops) <= 200 + 1e-3 * ops, (prof.total_time_ns, ops)
    assert prof.total_time_ns < 5_000_000, prof.total_time_ns


def test_profile_after_queued_runs(rg):
    _, sess = _session(rg)
    x, d_x, d_y = _buffers(rg, 2000)
    for queued in (1, 2, 3, 8, 9):
        for _ in range(queued):
            sess.run_device(d_x, x.shape, d_y)
        _check(sess.last_npu_profile(), 2000)
    for _ in range(4):  # each on an idle stream
        sess.run_device(d_x, x.shape, d_y)
        sess.synchronize()
        _check(sess.last_npu_profile(), 2000)
    sess.close()


def test_profile_after_shape_changes_and_host_runs(rg, ref):
    layers, sess = _session(rg)
    small, big = _buffers(rg, 40), _buffers(rg, 2000)
    for x, d_x, d_y in (big, small, big, big, small, small, big):
        sess.run_device(d_x, x.shape, d_y)
        sess.run_device(d_x, x.shape, d_y)
    _check(sess.last_npu_profile(), 2000)
    y = sess.run(small[0])
    _check(sess.last_npu_profile(), 40)
    sess.run_device(big[1], big[0].shape, big[2])
    sess.run_device(small[1], small[0].shape, small[2])
    _check(sess.last_npu_profile(), 40)
    want = ref.RefProgram(layers).run(small[0], parallel=True)
    assert_bitexact_f32(y, want, "host run")
    assert_bitexact_f32(small[2].download((40, DIMS[-1])), want, "device run")
    sess.close()


def test_profile_after_a_run_that_failed(rg):
    from rustgears_amd._native import RgnpuError
    from rustgears_amd.inference import DeviceBuffer
    _, sess = _session(rg)
    x, d_x, d_y = _buffers(rg, 2000)
    sess.run_device(d_x, x.shape, d_y)
    with pytest.raises(RgnpuError):
        sess.run_device(d_x, x.shape, DeviceBuffer(64))
    _check(sess.last_npu_profile(), 2000)
    with pytest.raises(RgnpuError):
        sess.run_device(d_x, (2000, 1000), d_y)
    for _ in range(3):
        sess.run_device(d_x, x.shape, d_y)
    _check(sess.last_npu_profile(), 2000)
    sess.close()


def test_profiling_off_times_the_run_alone(rg, ref):
    layers, sess = _session(rg)
    x, d_x, d_y = _buffers(rg, 2000)
    other = _buffers(rg, 40)
    sess.run_device(d_x, x.shape, d_y)
    full = sess.last_npu_profile().total_time_ns
    sess.set_profiling(0)
    for n in (1, 2, 5):
        for _ in range(n):
            sess.run_device(d_x, x.shape, d_y)
        sess.set_profiling(1)  # by the time it is read, profiling is on again
        prof = sess.last_npu_profile()
        sess.set_profiling(0)
        assert all(r.duration_ns == 0 and r.kernel_ns == 0 for r in prof.records), prof.records
        assert 0.3 * full < prof.total_time_ns < 3 * full + 50_000, (prof.total_time_ns, full)
        sess.run_device(other[1], other[0].shape, other[2])
    sess.run_device(d_x, x.shape, d_y)
    sess.set_profiling(1)
    sess.run_device(d_x, x.shape, d_y)
    _check(sess.last_npu_profile(), 2000)
    assert_bitexact_f32(d_y.download((2000, DIMS[-1])), ref.RefProgram(layers).run(x, parallel=True), "profiling off")
    sess.close()
