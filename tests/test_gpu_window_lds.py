"""CPU-path semantics of real confocal captures through the LDS-staged window kernel.  Complex
samples keep the general window kernel, so a capture is compared with itself as complex samples:
integer samples exactly (every prefix sum and volume value is an integer below 2^24), real samples
within one unit in the last place (double sums in another order, rounded once to float)."""
import numpy as np
import pytest

from backprojector_amd import scenes

pytestmark = pytest.mark.gpu
f32 = np.float32


def pairs_of(nx, ny, seed):
    gx, gy = np.linspace(-1, 1, nx), np.linspace(-1, 1, ny)
    X, Y = np.meshgrid(gx, gy, indexing="ij")
    cg = np.stack([X, Y, np.zeros_like(X)], -1).astype(f32)
    cg += np.random.default_rng(seed).uniform(-0.01, 0.01, cg.shape).astype(f32) * np.array([1, 1, 0], f32)
    return scenes.wall_pairs(cg, cg, True)


# volume, centre and size (m), bins, bin width, t0, scan: columns of 8 and 16 voxels, slabs reaching
# back, wide windows (anisotropic voxels), rows shorter than the windows' reach, starts before bin 0
# and ends past the last, every window past the row, one part and many
CASES = [
    ((20, 18, 16), (0, 0, 0.8), (1, 1, 1), 2600, 0.001, 2.0, (16, 16)),
    ((33, 17, 38), (0.1, 0, 0.7), (0.5, 0.3, 0.4), 1500, 0.002, 1.9, (23, 19)),
    ((40, 40, 40), (0, 0, 0.8), (1, 1, 1), 1024, 0.004, 0.0, (31, 33)),
    ((16, 16, 8), (0, 0, 0.6), (0.1, 0.8, 0.1), 700, 0.003, 2.0, (7, 5)),
    ((12, 35, 23), (0, 0.2, 0.9), (0.3, 0.6, 0.5), 300, 0.003, 3.1, (14, 9)),
    ((12, 35, 23), (0, 0.2, 0.9), (0.3, 0.6, 0.5), 64, 0.003, 3.9, (14, 9)),
    ((12, 20, 17), (0, 0.2, 0.9), (0.3, 0.6, 0.5), 2, 0.003, 3.6, (14, 9)),
    ((12, 20, 17), (0, 0.2, 0.9), (0.3, 0.6, 0.5), 500, 0.003, 9.0, (5, 9)),
]


@pytest.mark.parametrize("N,pos,size,T,dT,t0,scan", CASES)
def test_window_lds_equals_general_kernel(gpu, oracle, N, pos, size, T, dT, t0, scan):
    pr = pairs_of(*scan, seed=N[2])
    rng = np.random.default_rng(T)
    pr["camera_wall"] += rng.uniform(0, 0.2, len(pr)).astype(f32)
    pos, size = np.array(pos, f32), np.array(size, f32)
    H = rng.integers(0, 60, (len(pr), T)).astype(f32)
    got = gpu.window_backprojection(H, pr, N, pos, size, t0, dT)
    want = gpu.window_backprojection(H.astype(np.complex64), pr, N, pos, size, t0, dT).real
    assert want.max() < 2 ** 24
    assert np.array_equal(got, want)
    assert np.array_equal(got, oracle.a2_volume(H, pr, N, pos, size, t0, dT).astype(f32))
    Hr = rng.gamma(0.5, 2.0, H.shape).astype(f32)
    got = gpu.window_backprojection(Hr, pr, N, pos, size, t0, dT)
    want = gpu.window_backprojection(Hr.astype(np.complex64), pr, N, pos, size, t0, dT).real
    assert np.all(np.abs(got - want) <= np.spacing(np.maximum(np.abs(got), np.abs(want))))


def test_window_geometries_that_keep_the_general_kernel(gpu, oracle):
    """A wall that is not flat and a volume across the wall plane: the general kernel, as before."""
    pr = pairs_of(9, 8, 1)
    H = np.random.default_rng(2).integers(0, 60, (len(pr), 900)).astype(f32)
    tilted = pr.copy()
    tilted["laser_point"][:, 2] = np.linspace(0, 0.05, len(pr)).astype(f32)
    tilted["camera_point"] = tilted["laser_point"]
    for q, z in ((tilted, 0.7), (pr, 0.1)):
        pos, size = np.array([0, 0, z], f32), np.array([0.4, 0.4, 0.4], f32)
        got = gpu.window_backprojection(H, q, (20, 18, 24), pos, size, 1.5, 0.003)
        assert np.array_equal(got, gpu.window_backprojection(H.astype(np.complex64), q, (20, 18, 24), pos, size, 1.5, 0.003).real)
