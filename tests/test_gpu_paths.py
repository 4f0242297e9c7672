"""Non-confocal captures (exhaustive grids, pair lists) through the LDS-staged paths kernel: exact
bins against the oracle with integer samples (every sum an integer below 2^24), real and 16-bit
samples against the general kernels (an explicit variant keeps those)."""
import numpy as np
import pytest

from backprojector_amd import scenes

pytestmark = pytest.mark.gpu
f32 = np.float32


def grid_pairs(oracle, nl, nc, seed=0):
    lg, cg = scenes.wall_grid(nl), (scenes.wall_grid(nc) * f32(0.9)).astype(f32)
    cg[..., 2] += np.random.default_rng(seed).uniform(0, 0.02, cg.shape[:2]).astype(f32)   # not flat
    return oracle.precompute_pairs(scenes.ORIGIN, lg, scenes.ORIGIN, cg, confocal=False)


def basis(N, pos, size):
    pos, size = np.asarray(pos, f32), np.asarray(size, f32)
    return pos - size / f32(2), np.diag([size[k] / f32(max(N[k] - 1, 1)) for k in range(3)]).astype(f32).ravel()


# volume, size (m), bins, bin width, t0, lasers, SPADs: partial tiles, slabs reaching back, SPAD counts
# that 8 does and does not divide, windows before bin 0 and past the row, wholly outside it, rows
# whose length no 4 divides, one part and many
CASES = [
    ((32, 32, 16), (0.5, 0.5, 0.3), 2500, 0.001, 2.0, 5, 4),
    ((17, 20, 23), (0.4, 0.5, 0.6), 1999, 0.002, 1.2, 6, 3),
    ((40, 33, 8), (1.0, 1.0, 0.2), 1021, 0.004, 0.0, 9, 5),
    ((5, 3, 9), (0.1, 0.1, 0.1), 700, 0.001, 3.6, 3, 2),
    ((20, 16, 17), (0.3, 0.3, 0.3), 300, 0.003, 9.0, 3, 3),
    ((20, 16, 17), (0.3, 0.3, 0.3), 3, 0.003, 4.0, 4, 3),
]


@pytest.mark.parametrize("N,size,T,dT,t0,nl,nc", CASES)
@pytest.mark.parametrize("shuffled", [False, True])
def test_paths_bins_bit_exact(gpu, oracle, N, size, T, dT, t0, nl, nc, shuffled):
    pr = grid_pairs(oracle, nl, nc, seed=nl)
    rng = np.random.default_rng(T)
    if shuffled:
        pr = pr[rng.permutation(len(pr))]
    H = rng.integers(1, 62, (len(pr), T)).astype(f32)
    zero, inc = basis(N, (0.05, -0.02, 0.75), size)
    with gpu.Plan(H, pr, N, zero, inc, t0, dT) as plan:
        plan.execute()
        plan.execute()
        info = plan.info()
        assert info["kernel"].startswith("paths_lds_kernel") and info["path"] == ("pairs" if shuffled else "grid"), info
        vol = plan.volume()
    ref = oracle.a1_volume_f64acc(H, pr, N, zero, inc, t0, dT)
    assert ref.max() < 2 ** 24 and np.array_equal(vol, ref.astype(f32))


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("shuffled", [False, True])
def test_paths_formats(gpu, oracle, storage, shuffled):
    """Real samples, every storage: within the reference order's tolerance of the exact sum of the
    stored samples, and no further from it than the general kernel is, but for one rounding."""
    pr = grid_pairs(oracle, 7, 5)
    rng = np.random.default_rng(4)
    if shuffled:
        pr = pr[rng.permutation(len(pr))]
    T, N = 2000, (33, 18, 21)
    H = rng.gamma(0.5, 2.0, (len(pr), T)).astype(f32)
    zero, inc = basis(N, (0.05, -0.02, 0.75), (0.5, 0.5, 0.5))
    vols = {}
    for v in (-1, 2):
        with gpu.Plan(H, pr, N, zero, inc, 1.8, 0.0015, storage=storage, variant=v) as plan:
            plan.execute()
            assert plan.info()["kernel"].startswith("paths_lds") == (v < 0)
            vols[v] = plan.volume().astype(np.float64)
            scale = plan.info()["scale"]
    x = H / f32(scale)
    if storage == "f16":
        x = x.astype(np.float16).astype(f32)
    elif storage == "bf16":
        u = x.view(np.uint32)
        x = ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(f32)
    exact = oracle.a1_volume_f64acc(x * f32(scale), pr, N, zero, inc, 1.8, 0.0015)
    err = {v: np.abs(vols[v] - exact) for v in vols}
    ulp = np.spacing(exact.astype(f32)).astype(np.float64)
    assert np.all(err[-1] <= 2 * ulp)          # block sums of 32 and one final rounding
    assert np.linalg.norm(err[-1]) <= 1.05 * np.linalg.norm(err[2])


def test_paths_that_keep_the_general_kernels(gpu, oracle):
    """A volume around a laser point, a rotated basis, fewer than 8 voxels along z, windows too long,
    complex samples and an explicit variant: the general kernels, exact as before."""
    pr = grid_pairs(oracle, 4, 3)
    H = np.random.default_rng(1).integers(1, 62, (len(pr), 1500)).astype(f32)
    rot = np.array([0.01, 0, 0.002, 0, 0.01, 0, -0.002, 0, 0.01], f32)
    base = basis((20, 18, 16), (0, 0, 0.7), (0.4, 0.4, 0.4))
    for N, zero, inc, dT, v, cplx in [((20, 18, 16), *basis((20, 18, 16), (0, 0, 0.1), (2.2, 2.2, 0.4)), 0.002, -1, False),
                                      ((20, 18, 16), base[0], rot, 0.002, -1, False),
                                      ((20, 18, 7), *basis((20, 18, 7), (0, 0, 0.7), (0.4, 0.4, 0.1)), 0.002, -1, False),
                                      ((8, 8, 8), *basis((8, 8, 8), (0, 0, 0.8), (1, 1, 1)), 0.001, -1, False),
                                      ((20, 18, 16), *base, 0.002, 0, False), ((20, 18, 16), *base, 0.002, -1, True)]:
        with gpu.Plan(H.astype(np.complex64) if cplx else H, pr, N, zero, inc, 2.0, dT, variant=v) as plan:
            plan.execute()
            assert "paths" not in plan.info()["kernel"], (N, v, cplx)
            vol = plan.volume()
        ref = oracle.a1_volume_f64acc(H, pr, N, zero, inc, 2.0, dT).astype(f32)
        assert np.array_equal(vol.real if cplx else vol, ref), (N, v, cplx)


@pytest.mark.parametrize("variant", [-1, 2])
@pytest.mark.parametrize("kahan", [1, 2])
@pytest.mark.parametrize("nl,nc", [(9, 4), (7, 5)])
def test_grid_blocks_shorter_than_a_stage(gpu, oracle, nl, nc, kahan, variant):
    """Every sample 1.6000018: 8 of them summed plainly are 2.5 units (of 2^-24, relative) off, 1 or 2 are
    exact.  Blocks of 1 or 2 leave the compensated sum's n 2^-48 and the final rounding, at most 1 unit;
    blocks of 8 would end 1.8 to 2.9 off."""
    pr = grid_pairs(oracle, nl, nc)
    N, T = (32, 20, 16), 2500
    zero, inc = basis(N, (0.05, -0.02, 0.75), (0.5, 0.4, 0.3))
    H = np.full((len(pr), T), 1.6000018, f32)
    exact = oracle.a1_volume_f64acc(H, pr, N, zero, inc, 0.0, 0.004)
    assert np.allclose(exact, len(pr) * float(H[0, 0]), rtol=1e-12)
    with gpu.Plan(H, pr, N, zero, inc, 0.0, 0.004, kahan_block=kahan, variant=variant) as plan:
        plan.execute()
        assert plan.info()["path"] == "grid" and plan.info()["kernel"].startswith("paths_lds") == (variant < 0)
        vol = plan.volume().astype(np.float64)
    assert np.abs(vol / exact - 1).max() <= 1.1 * 2.0 ** -24
