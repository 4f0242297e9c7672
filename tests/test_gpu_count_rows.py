"""Confocal captures of photon counts (integers 0 .. 2048): integer sums through the LDS-staged
kernel with polynomial quotients.  Volumes are sums of integers below 2^24, so they must EQUAL the
oracle's exactly accumulated ones, the fp32 rows' (keep_f32_rows) and every other kernel's."""
import numpy as np
import pytest

from backprojector_amd import scenes

pytestmark = pytest.mark.gpu
f32 = np.float32


def pairs_of(nx, ny):
    gx, gy = np.linspace(-1, 1, nx), np.linspace(-1, 1, ny)
    X, Y = np.meshgrid(gx, gy, indexing="ij")
    cg = np.stack([X, Y, np.zeros_like(X)], -1).astype(f32)
    cg += np.random.default_rng(nx).uniform(-0.01, 0.01, cg.shape).astype(f32) * np.array([1, 1, 0], f32)
    return scenes.wall_pairs(cg, cg, True)


def basis(N, pos, size):
    pos, size = np.asarray(pos, f32), np.asarray(size, f32)
    return pos - size / f32(2), np.diag([size[k] / f32(max(N[k] - 1, 1)) for k in range(3)]).astype(f32).ravel()


# volume, its size (m), bins, bin width, t0, scan: columns of 8 (the shortest) and 16 voxels, the
# last slab reaching back over its neighbour (nz = 17, 23, 38), a z axis running towards the wall,
# quadratic and cubic polynomials, long windows (1.5 mm bins on a coarse grid), windows that start
# before bin 0 and end past the last, one part and many, pair counts that no stage divides
CASES = [
    ((16, 16, 16), (0.1, 0.1, 0.1), 3000, 0.001, 1.2, (15, 15)),
    ((35, 33, 17), (0.25, 0.22, 0.12), 3000, 0.001, 1.2, (16, 16)),
    ((40, 20, 23), (0.9, 0.6, 0.4), 1501, 0.004, 0.0, (31, 17)),
    ((33, 30, 38), (1.0, 1.0, 0.8), 2731, 0.0015, 0.0, (13, 11)),
    ((3, 5, 8), (0.02, 0.05, 0.05), 2000, 0.001, 1.6, (9, 7)),
    ((17, 16, 31), (0.3, 0.3, -0.3), 2000, 0.001, 2.4, (20, 21)),
    ((20, 24, 28), (0.3, 0.3, 0.3), 900, 0.001, 3.3, (37, 29)),
]


@pytest.mark.parametrize("N,size,T,dT,t0,scan", CASES)
def test_count_rows_equal_oracle(gpu, oracle, N, size, T, dT, t0, scan):
    pr = pairs_of(*scan)
    rng = np.random.default_rng(N[2])
    H = rng.integers(0, 2049, (len(pr), T)).astype(f32)
    H[rng.random(H.shape) < 0.3] = 0
    H[:, 0] = H[:, -1] = 2048
    zero, inc = basis(N, (0.03, -0.02, 0.75), size)
    ref = oracle.a1_volume_f64acc(H, pr, N, zero, inc, t0, dT)
    assert ref.max() < 2 ** 24
    for variant in (-1, 8):
        with gpu.Plan(H, pr, N, zero, inc, t0, dT, variant=variant) as plan:
            plan.execute()
            plan.execute()   # partial sums are rewritten by every execution
            info = plan.info()
            assert info["kernel"].startswith("confocal_lds_kernel_poly"), info
            assert info["row_storage"] == "f16"
            assert np.array_equal(plan.volume(), ref.astype(f32)), variant
    with gpu.Plan(H, pr, N, zero, inc, t0, dT, keep_f32_rows=True) as plan:
        plan.execute()
        assert "poly" not in plan.info()["kernel"]
        assert np.array_equal(plan.volume(), ref.astype(f32))


@pytest.mark.parametrize("value", [-1.0, 0.5, 2049.0, np.nan, np.inf, -0.0])
def test_one_sample_that_is_no_count(gpu, value):
    """One such sample (in the middle, at either end) takes the whole execution off count rows, and
    -0.0 is the count 0; the volume is the fp32 rows' either way."""
    N, T = (35, 33, 17), 2001
    pr = pairs_of(15, 15)
    zero, inc = basis(N, (0.03, -0.02, 0.75), (0.25, 0.22, 0.12))
    H = np.random.default_rng(3).integers(0, 60, (len(pr), T)).astype(f32)
    for p, b in [(0, 0), (100, 700), (len(pr) - 1, T - 1)]:
        Hb = H.copy()
        Hb[p, b] = value
        vols = {}
        for variant, keep in ((-1, False), (7, False), (8, False), (-1, True)):
            with gpu.Plan(Hb, pr, N, zero, inc, 1.2, 0.001, variant=variant, keep_f32_rows=keep) as plan:
                plan.execute()
                info = plan.info()
                counts = value == 0.0 and not keep
                assert info["kernel"].startswith("confocal_lds_kernel_poly") == counts, (variant, info)
                f16 = counts or (value == -1.0 and variant > 0)
                assert info["row_storage"] == ("f16" if f16 else "f32"), (variant, info)
                vols[variant, keep] = plan.volume()
        for k, v in vols.items():
            assert np.array_equal(v, vols[-1, True], equal_nan=True), (p, b, k)


def test_geometries_that_keep_the_other_kernels(gpu, oracle):
    """A volume that touches the wall, a wall that is not flat, a rotated basis, fewer than 8 voxels
    along z and an integer block above the exact range keep the kernels they had, exact as before."""
    T, dT = 2000, 0.002
    pr = pairs_of(9, 8)
    H = np.random.default_rng(5).integers(0, 61, (len(pr), T)).astype(f32)
    tilted = pr.copy()
    tilted["laser_point"][:, 2] = np.linspace(0, 0.05, len(pr)).astype(f32)
    tilted["camera_point"] = tilted["laser_point"]
    rot = np.array([0.01, 0, 0.002, 0, 0.01, 0, -0.002, 0, 0.01], f32)
    base = basis((20, 18, 24), (0, 0, 0.7), (0.4, 0.4, 0.4))
    cases = [(pr, (20, 18, 24), *basis((20, 18, 24), (0, 0, 0.2), (0.4, 0.4, 0.4)), 0),
             (tilted, (20, 18, 24), *base, 0),
             (pr, (20, 18, 24), base[0], rot, 0),
             (pr, (20, 18, 7), *basis((20, 18, 7), (0, 0, 0.7), (0.4, 0.4, 0.1)), 0),
             (pr, (20, 18, 24), *base, 5000)]
    for q, N, zero, inc, kahan in cases:
        with gpu.Plan(H, q, N, zero, inc, 0.5, dT, kahan_block=kahan) as plan:
            plan.execute()
            assert "poly" not in plan.info()["kernel"], (N, kahan)
            vol = plan.volume()
        assert np.array_equal(vol, oracle.a1_volume_f64acc(H, q, N, zero, inc, 0.5, dT).astype(f32))
