"""Calls when the device's memory runs short: what fails says so, leaves nothing behind and takes nothing
along; what a faster kernel would need beside its general form is given up instead.  Counts, so every
volume must EQUAL the oracle's exactly accumulated one."""
import ctypes
from contextlib import contextmanager, nullcontext

import numpy as np
import pytest

from backprojector_amd._native import BpxError
from test_gpu_count_rows import basis, pairs_of

pytestmark = pytest.mark.gpu
f32 = np.float32


def capture(scan=(9, 8), T=900, seed=0):
    pr = pairs_of(*scan)
    return np.random.default_rng(seed).integers(0, 9, (len(pr), T)).astype(f32), pr


def test_failed_allocation_leaves_no_error(gpu, oracle):
    """Volumes of 16 GiB until one does not fit: the call says so, and the next launches do not report its
    error as theirs."""
    H, pr = capture()
    N = (20, 18, 17)
    grid = basis(N, (0.0, 0.0, 0.7), (0.4, 0.4, 0.4))
    ref = oracle.a1_volume_f64acc(H, pr, N, *grid, 0.5, 0.003).astype(f32)
    big = (2048, 2048, 1024)
    big_grid = basis(big, (0.0, 0.0, 0.7), (0.4, 0.4, 0.4))
    held = []
    try:
        with gpu.Plan(H, pr, N, *grid, 0.5, 0.003) as plan:
            with pytest.raises(BpxError, match="OUT_OF_MEMORY"):
                for _ in range(32):
                    held.append(gpu.Plan(H, pr, big, *big_grid, 0.5, 0.003))
            assert len(held) > 8
            plan.execute()
            assert np.array_equal(plan.volume(), ref)
    finally:
        for p in held:
            p.close()


@contextmanager
def memory_left(n):
    """All of the device's free memory but n bytes taken."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2
    hip.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    free, total, p = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_void_p()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    assert free.value > n and hip.hipMalloc(ctypes.byref(p), free.value - n) == 0
    try:
        yield
    finally:
        assert hip.hipFree(p) == 0


def long_rows(scan, T):
    pr = pairs_of(*scan)
    rows = np.random.default_rng(T).integers(0, 9, (64, T)).astype(f32)
    return np.tile(rows, (len(pr) // 64, 1)), pr


def test_window_tables_that_do_not_fit(gpu):
    """8,192 rows of 16,384 bins: 0.5 GiB of samples and 1 of prefix sums for the general kernel, 2 more for
    the LDS-staged one's tables."""
    T, N = 16384, (32, 32, 32)
    H, pr = long_rows((128, 64), T)
    args = (H, pr, N, (0.0, 0.0, 0.8), (0.15, 0.15, 0.15), 0.0, 4.0 / T)
    ref = gpu.window_backprojection(*args)
    assert ref.max() > 0
    with memory_left(5 << 29):
        assert np.array_equal(gpu.window_backprojection(*args), ref)


def octree_args(samples):
    """16,384 rows of 8,192 bins: 0.5 GiB of samples, 1 GiB of fused rows."""
    T, N = 8192, (32, 32, 32)
    H, pr = long_rows((128, 128), T)
    if samples == "real":
        H += f32(0.25)
    return (H, pr, N, *basis(N, (0.0, 0.0, 0.8), (0.2, 0.2, 0.2)), 0.0, 4.0 / T)


def memory_of(make):
    """(object, bytes of device memory that making it took)."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    free, after, total = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    obj = make()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ctypes.byref(after), ctypes.byref(total)) == 0
    return obj, free.value - after.value


def test_octree_count_rows_only_where_they_serve(gpu):
    """Real samples take no count rows (as large as the fused rows, 1 GiB); counts that find no room for
    them give the volume of those that do."""
    counts, real = octree_args("counts"), octree_args("real")
    rows = 8 * counts[0].size
    plan, with_rows = memory_of(lambda: gpu.Plan.octree(*counts, levels=2))
    with plan:
        plan.execute()
        ref = plan.volume()
        other, without = memory_of(lambda: gpu.Plan.octree(*real, levels=2))
        other.close()
    # blocks released by earlier plans, at most 0.5 GiB, may serve either
    assert without < with_rows - rows // 2, (with_rows, without)
    with memory_left(without + (3 << 27)):
        with gpu.Plan.octree(*counts, levels=2) as plan:
            plan.execute()
            assert np.array_equal(plan.volume(), ref)


def test_octree_tile_sums_that_do_not_fit(gpu):
    """1024 x 1024 x 512 voxels, every one listed: 131,072 tiles take 2 GiB of partial sums at the first
    execution; without them the voxels are gathered one by one."""
    H, pr = capture((8, 8), 1200)
    N = (1024, 1024, 512)
    args = (H, pr, N, *basis(N, (0.0, 0.0, 0.8), (0.5, 0.5, 0.25)), 0.5, 0.0025)
    with gpu.Plan.octree(*args, levels=2, threshold=0.0) as plan:
        plan.execute()
        ref = plan.volume()
    assert ref.max() > 0
    with gpu.Plan.octree(*args, levels=2, threshold=0.0) as plan, memory_left(1 << 30):
        plan.execute()
        assert np.array_equal(plan.volume(), ref)
        plan.execute()
        assert np.array_equal(plan.volume(), ref)


def test_batch_sums_that_do_not_fit(gpu):
    """70 captures of 64 MiB of partial sums each, split texture-path captures among them: at most 4 GiB at a
    time, and where they do not fit either, in smaller waves.  Every volume is its own plan's bit for bit."""
    N, T = (64, 64, 64), 300
    grid = basis(N, (0.0, 0.0, 0.7), (0.4, 0.4, 0.4))
    kinds = []
    for k in range(5):
        H, pr = capture((64, 64), T, k)
        kinds.append(((H + f32(0.25) if k % 2 else H), pr, N, *grid, 1.0, 0.006))
    refs = []
    for a in kinds:
        with gpu.Plan(*a) as plan:
            plan.execute()
            refs.append(plan.volume())
            assert int(plan.info()["kernel"].split("tiles, ")[1].split()[0]) >= 32
    H, pr = capture((31, 33), 2000, 9)
    kinds.append((H, pr, (24, 24, 24), *basis((24, 24, 24), (0.0, 0.0, 0.7), (0.8, 0.8, 0.6)), 0.5, 0.0015))
    with gpu.Plan(*kinds[-1]) as plan:
        plan.execute()
        refs.append(plan.volume())
        assert plan.info()["kernel"].startswith("confocal_kernel_split<")
    args = [kinds[i % 6] for i in range(84)]
    b, taken = memory_of(lambda: gpu.Batch(args))
    rows = 70 * (T * 4096 * 4 + 8 * 4096 * 384 + 4 * 64 ** 3) + 14 * 12 * H.size
    assert taken < rows + (4 << 30) + (256 << 20), taken
    for room in (None, 5 << 29):
        with memory_left(room) if room else nullcontext(), b or gpu.Batch(args) as batch:
            for rep in range(2):
                batch.execute()
                for i in range(84):
                    assert np.array_equal(batch.volume(i), refs[i % 6]), (room, rep, i)
            assert np.all(batch.latencies() > 0)
        b = None


def test_kept_blocks_can_be_given_back(gpu, oracle):
    """What destroyed plans leave with the library is bounded, and a call returns it to the device."""
    H, pr = capture((64, 64), 2000)
    N = (128, 128, 128)
    args = (H, pr, N, *basis(N, (0.0, 0.0, 0.7), (0.4, 0.4, 0.4)), 0.5, 0.003)
    gpu.release_memory()
    assert gpu.release_memory() == 0
    with gpu.Plan(*args) as plan:
        plan.execute()
        ref = plan.volume()
    kept = []
    _, taken = memory_of(lambda: kept.append(gpu.release_memory()))
    assert 100 << 20 < kept[0] <= 512 << 20
    assert -taken >= kept[0] // 2 and gpu.release_memory() == 0
    with gpu.Plan(*args) as plan:
        plan.execute()
        assert np.array_equal(plan.volume(), ref)
