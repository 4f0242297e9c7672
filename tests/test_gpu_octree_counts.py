"""Octree executions of count captures: fine voxels of well-filled tiles computed tile by tile, the
others one by one with the pairs split over lanes -- integer sums either way, so every computed
voxel must EQUAL the dense reconstruction and the oracle.  (Learned executions, with both their lists:
test_gpu_learned_octree.py.)"""
import numpy as np
import pytest

from backprojector_amd import scenes

pytestmark = pytest.mark.gpu
f32 = np.float32


def capture(side, T, real=False, seed=0):
    cg = scenes.wall_grid(side)
    pr = scenes.wall_pairs(cg, cg, True)
    rng = np.random.default_rng(seed)
    # positive samples (a computed voxel is 0 only without any in-range bin), brighter around one
    # bin per pair
    b = np.arange(T)[None, :]
    peak = rng.integers(T // 2, T // 2 + T // 8, len(pr))[:, None]
    H = rng.integers(1, 9, (len(pr), T)) + 200 * (np.abs(b - peak) < 12)
    return (H + 0.25 if real else H).astype(f32), pr


def basis(N, pos, size):
    pos, size = np.asarray(pos, f32), np.asarray(size, f32)
    return pos - size / f32(2), np.diag([size[k] / f32(N[k] - 1) for k in range(3)]).astype(f32).ravel()


# columns of 16 and of 8 voxels, tiles cut by every face, a last slab reaching back, few and many
# voxels per tile (the threshold decides), one to many pair parts
@pytest.mark.parametrize("N,levels,size,side,tau", [
    ((64, 64, 64), 3, (0.5, 0.5, 0.5), 16, 0.1), ((64, 64, 64), 3, (0.5, 0.5, 0.5), 16, 0.6),
    ((40, 24, 56), 3, (0.4, 0.3, 0.5), 12, 0.3), ((36, 20, 28), 2, (0.9, 0.9, 0.7), 20, 0.5),
    ((16, 16, 8), 1, (0.1, 0.1, 0.05), 6, 0.05), ((32, 32, 32), 4, (0.3, 0.3, 0.3), 9, 0.9)])
@pytest.mark.parametrize("real", [False, True])
def test_octree_counts_equal_dense(gpu, oracle, N, levels, size, side, tau, real):
    T, dT = 1024, 0.003
    H, pr = capture(side, T, real)
    zero, inc = basis(N, (0.0, 0.0, 0.75), size)
    t0 = 0.4
    ref = oracle.a1_volume_f64acc(H, pr, N, zero, inc, t0, dT)
    dense = gpu.backprojection(H, pr, N, zero, inc, t0, dT)
    if not real:
        assert np.array_equal(dense, ref.astype(f32))
    with gpu.Plan.octree(H, pr, N, zero, inc, t0, dT, levels=levels, threshold=tau) as plan:
        for _ in range(2):   # the second execution reuses lists, masks and partial sums
            plan.execute()
            vol, st = plan.volume(), plan.octree_stats()
            c = vol != 0
            assert np.array_equal(vol[c], dense[c])
            assert c[dense >= tau * dense.max()].all()
            # every listed voxel is written (some hold no in-range bin at all: value 0)
            assert 0 <= st["active"][-1] - c.sum() <= (dense == 0).sum()
        plan.set_octree_options(threshold=0.02)
        plan.execute()
        vol = plan.volume()
        assert np.array_equal(vol, dense) if (dense >= 0.02 * dense.max()).all() else np.array_equal(vol[vol != 0], dense[vol != 0])

