"""Host transfers in chunks, reused device blocks and streams.  Counts, so every volume must EQUAL
the oracle's exactly accumulated one."""
import threading

import numpy as np
import pytest

from test_gpu_count_rows import basis, pairs_of

pytestmark = pytest.mark.gpu
f32 = np.float32


def capture(scan, T, seed):
    pr = pairs_of(*scan)
    return np.random.default_rng(seed).integers(0, 9, (len(pr), T)).astype(f32), pr


# volumes of 16 MiB less a row (one plain copy), of 16 MiB, of 32 MiB and 4 bytes * 7 more (a second
# round with one short chunk), and of an odd size in between
@pytest.mark.parametrize("N", [(256, 256, 63), (256, 256, 64), (7, 13, 92183), (211, 173, 149)])
def test_volume_in_chunks(gpu, oracle, N):
    H, pr = capture((2, 2), 700, N[2])
    zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    with gpu.Plan(H, pr, N, zero, inc, 0.5, 0.005) as plan:
        plan.execute()
        got = plan.volume()
    assert np.array_equal(got, oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.5, 0.005).astype(f32))


# transients just under, at and past the 64 MiB from which they go through the ring
@pytest.mark.parametrize("T", [16381, 16384, 16389, 40001])
def test_transient_in_chunks(gpu, oracle, T):
    H, pr = capture((32, 32), T, T)
    N = (5, 4, 3)
    zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    dT = 4.0 / T
    with gpu.Plan(H, pr, N, zero, inc, 0.5, dT) as plan:
        plan.execute()
        got = plan.volume()
    assert np.array_equal(got, oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.5, dT).astype(f32))


def test_plans_of_several_threads(gpu, oracle):
    """Blocks and streams released by one thread's plans are taken by another's at once."""
    shapes = [((9, 8, 11), (5, 7), 400), ((16, 16, 16), (8, 8), 500), ((33, 20, 24), (16, 9), 300), ((4, 4, 40), (3, 3), 900)]
    cases = []
    for k, (N, scan, T) in enumerate(shapes):
        H, pr = capture(scan, T, k)
        zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
        cases.append((H, pr, N, zero, inc, oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.5, 0.005).astype(f32)))
    bad = []

    def work(first):
        for r in range(6):
            H, pr, N, zero, inc, ref = cases[(first + r) % len(cases)]
            with gpu.Plan(H, pr, N, zero, inc, 0.5, 0.005) as plan:
                plan.execute()
                if not np.array_equal(plan.volume(), ref):
                    bad.append((first, r))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def hip_memory(n, pinned):
    """(runtime, address) of n bytes of pinned host memory or of device memory."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so.7")
    p = ctypes.c_void_p()
    hip.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipHostFree.argtypes = hip.hipFree.argtypes = [ctypes.c_void_p]
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    assert (hip.hipHostMalloc(ctypes.byref(p), n, 0) if pinned else hip.hipMalloc(ctypes.byref(p), n)) == 0
    return hip, p


@pytest.mark.parametrize("N", [(256, 256, 64), (512, 512, 128)])
def test_volume_into_pinned_and_device_memory(gpu, N):
    """Destinations that the copy engine reaches by itself take one copy: the pinned one in less than
    0.8 of the time of pageable memory (0.63 measured at 128 MiB; chunks would take both alike)."""
    import ctypes
    import time
    H, pr = capture((3, 2), 700, 1)
    zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    n = 4 * int(np.prod(N))
    from backprojector_amd._native import lib
    read = lib().bpx_plan_read_volume
    with gpu.Plan(H, pr, N, zero, inc, 0.5, 0.005) as plan:
        plan.execute()
        ref = plan.volume()

        def into(address, reps):
            best = np.inf
            for _ in range(reps):
                t = time.perf_counter()
                assert read(plan._h, ctypes.cast(address, ctypes.POINTER(ctypes.c_float))) == 0
                best = min(best, time.perf_counter() - t)
            return best

        hip, p = hip_memory(n, True)
        host = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), N)
        host[...] = -1
        pinned = into(p.value, 8)
        assert np.array_equal(host, ref)
        del host
        assert hip.hipHostFree(p) == 0
        back = np.full(N, -1, f32)
        pageable = into(back.ctypes.data, 8)
        assert np.array_equal(back, ref)
        if n >= 128 << 20:
            assert pinned < 0.8 * pageable, (pinned, pageable)
        hip, p = hip_memory(n, False)
        into(p.value, 1)
        back[...] = -1
        assert hip.hipMemcpy(back.ctypes.data, p, n, 2) == 0 and hip.hipFree(p) == 0
        assert np.array_equal(back, ref)


def test_transient_from_pinned_memory(gpu, oracle):
    import ctypes
    H, pr = capture((32, 32), 16389, 5)
    N = (5, 4, 3)
    zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    hip, p = hip_memory(H.nbytes, True)
    pinned = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), H.shape)
    pinned[...] = H
    with gpu.Plan(pinned, pr, N, zero, inc, 0.5, 4.0 / 16389) as plan:
        plan.execute()
        got = plan.volume()
    del pinned
    assert hip.hipHostFree(p) == 0
    assert np.array_equal(got, oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.5, 4.0 / 16389).astype(f32))


def test_transfers_of_several_threads(gpu, oracle):
    """Volumes out of and a transient into the library from several threads at once: one thread has the
    staging chunks of a direction, the others wait for them."""
    N = (256, 255, 97)   # 24 MiB, no round number of chunks
    zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    plans, refs = [], []
    for k in range(3):
        H, pr = capture((3, 2), 700, k)
        plans.append(gpu.Plan(H, pr, N, zero, inc, 0.5, 0.005))
        plans[-1].execute()
        refs.append(oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.5, 0.005).astype(f32))
    H, pr = capture((32, 32), 16389, 9)
    small = (5, 4, 3)
    grid = basis(small, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    up = oracle.a1_volume_f64acc(H, pr, small, *grid, 0.5, 4.0 / 16389).astype(f32)
    bad = []

    def down(k):
        for r in range(6):
            if not np.array_equal(plans[k].volume(), refs[k]):
                bad.append((k, r))

    def upload():
        for r in range(4):
            with gpu.Plan(H, pr, small, *grid, 0.5, 4.0 / 16389) as plan:
                plan.execute()
                if not np.array_equal(plan.volume(), up):
                    bad.append(("up", r))

    threads = [threading.Thread(target=down, args=(k,)) for k in range(3)] + [threading.Thread(target=upload)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for p in plans:
        p.close()
    assert not bad


def test_transfers_on_a_second_device(gpu, oracle):
    """The staging chunks serve every device of the process, each with its own events."""
    import torch
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs")
    N = (256, 255, 97)
    zero, inc = basis(N, (0.0, 0.0, 0.9), (0.5, 0.5, 0.5))
    H, pr = capture((32, 32), 16389, 5)
    ref = oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.5, 4.0 / 16389).astype(f32)
    for device in (0, 1, 0):
        with torch.cuda.device(device), gpu.Plan(H, pr, N, zero, inc, 0.5, 4.0 / 16389) as plan:
            plan.execute()
            assert np.array_equal(plan.volume(), ref), device
