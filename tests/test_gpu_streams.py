"""Executions on streams of the caller: captured into a graph and replayed, and on a stream that is
destroyed before the object is.  Counts, so every volume must EQUAL the first one."""
import ctypes

import numpy as np
import pytest

from test_gpu_count_rows import basis, pairs_of

pytestmark = pytest.mark.gpu
f32 = np.float32
POINTER = ctypes.c_void_p


@pytest.fixture
def hip(gpu):
    h = ctypes.CDLL("libamdhip64.so.7")
    for name, args in dict(hipStreamCreate=[ctypes.POINTER(POINTER)], hipStreamSynchronize=[POINTER], hipStreamDestroy=[POINTER],
                           hipStreamBeginCapture=[POINTER, ctypes.c_int],
                           hipStreamEndCapture=[POINTER, ctypes.POINTER(POINTER)],
                           hipGraphInstantiate=[ctypes.POINTER(POINTER), POINTER, POINTER, POINTER, ctypes.c_size_t],
                           hipGraphLaunch=[POINTER, POINTER], hipGraphExecDestroy=[POINTER], hipGraphDestroy=[POINTER]).items():
        getattr(h, name).argtypes = args
    return h


def stream(hip):
    s = POINTER()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    return s


def capture_args(N, samples, seed=0):
    pr = pairs_of(13, 12)
    rng = np.random.default_rng(seed)
    H = rng.integers(0, 9, (len(pr), 900)).astype(f32)
    if samples == "real":
        H += f32(0.25)
    return (H, pr, N, *basis(N, (0.02, 0.0, 0.7), (0.4, 0.4, 0.4)), 0.5, 0.003)


@pytest.mark.parametrize("samples", ["counts", "real"])
@pytest.mark.parametrize("N", [(32, 32, 32), (20, 18, 5)])   # the LDS-staged gather, the split texture path
def test_captured_execution(gpu, hip, N, samples):
    """The calls after the capture neither wait for events that were recorded into it nor miss replays."""
    with gpu.Plan(*capture_args(N, samples)) as plan, gpu.Plan(*capture_args(N, samples, 1)) as other:
        plan.execute()
        ref = plan.volume()
        s = stream(hip)
        graph, exec_ = POINTER(), POINTER()
        assert hip.hipStreamBeginCapture(s, 2) == 0     # relaxed
        plan.execute(s.value)
        assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
        plan.synchronize()
        assert np.array_equal(plan.volume(), ref)
        assert hip.hipGraphInstantiate(ctypes.byref(exec_), graph, None, None, 0) == 0
        for _ in range(3):
            other.execute()
            other.synchronize()
            assert hip.hipGraphLaunch(exec_, s) == 0
            assert hip.hipStreamSynchronize(s) == 0
            assert np.array_equal(plan.volume(), ref)
        plan.execute(s.value)                           # and eagerly, on the same stream and its own
        plan.execute()
        assert np.array_equal(plan.volume(), ref)
        assert hip.hipGraphExecDestroy(exec_) == 0 and hip.hipGraphDestroy(graph) == 0
        assert hip.hipStreamSynchronize(s) == 0 and hip.hipStreamDestroy(s) == 0


@pytest.mark.parametrize("kind", ["plan", "octree", "batch"])
def test_stream_destroyed_before_the_object(gpu, hip, kind):
    args = capture_args((32, 32, 32), "counts")
    for _ in range(2):   # the second object may get the first one's memory and stream
        obj = gpu.Batch([args]) if kind == "batch" else gpu.Plan.octree(*args, levels=3) if kind == "octree" else gpu.Plan(*args)
        read = (lambda: obj.volume(0)) if kind == "batch" else (lambda: obj.volume())
        with obj:
            obj.execute()
            ref = read()
            for _ in range(2):
                s = stream(hip)
                obj.execute(s.value)
                assert hip.hipStreamSynchronize(s) == 0 and hip.hipStreamDestroy(s) == 0
                obj.synchronize()
                assert np.array_equal(read(), ref)
            obj.execute()
            assert np.array_equal(read(), ref)
