"""Confocal captures that are no counts (fp32, 16-bit and complex rows): the LDS-staged kernel with
polynomial quotients against the texture-path kernel of an explicit variant, and exact sums against
the oracle."""
import numpy as np
import pytest

from test_gpu_count_rows import CASES, basis, pairs_of

pytestmark = pytest.mark.gpu
f32 = np.float32
EPS = 2.0 ** -24


@pytest.mark.parametrize("storage,cplx", [("f32", False), ("f16", False), ("bf16", False), ("f32", True)])
@pytest.mark.parametrize("N,size,T,dT,t0,scan", CASES)
def test_real_rows_equal_the_texture_path(gpu, N, size, T, dT, t0, scan, storage, cplx):
    """One part: the same sums in the same order, bit for bit.  More parts: every voxel is a sum of the
    same non-negative samples in other groups.  A group of 32 added in turn is off by at most 31
    roundings, its compensated sum by 2 and the end by 1, on either side: |a - b| <= 68 eps sum."""
    pr = pairs_of(*scan)
    rng = np.random.default_rng(N[2])
    H = rng.gamma(0.5, 2.0, (len(pr), T)).astype(f32)
    if cplx:
        H = (H + 1j * rng.gamma(0.5, 2.0, H.shape)).astype(np.complex64)
    zero, inc = basis(N, (0.03, -0.02, 0.75), size)
    vols, parts = [], 0
    for variant in (-1, 5):
        with gpu.Plan(H, pr, N, zero, inc, t0, dT, variant=variant, storage=storage) as plan:
            plan.execute()
            plan.execute()   # partial sums are rewritten by every execution
            name = plan.info()["kernel"]
            assert ("degree=" in name) == (variant == -1), name
            if variant == -1:
                parts = int(name.split("tiles, ")[1].split()[0])
                th = plan.thresholds()
            else:
                assert np.array_equal(th, plan.thresholds())
            vols.append(plan.volume())
    a, b = vols
    assert np.abs(b).max() > 0
    if parts == 1:
        assert np.array_equal(a, b)
    for x, y in ((a.real, b.real), (a.imag, b.imag)):
        assert np.all(np.abs(x.astype(np.float64) - y) <= 68 * EPS * np.abs(y).astype(np.float64))


@pytest.mark.parametrize("kahan", [1, 5, 32, 5000])
@pytest.mark.parametrize("N,size,T,dT,t0,scan", CASES[1:4])
def test_complex_integer_rows_equal_oracle(gpu, oracle, N, size, T, dT, t0, scan, kahan):
    pr = pairs_of(*scan)
    rng = np.random.default_rng(N[2])
    re, im = (rng.integers(-60, 61, (len(pr), T)).astype(f32) for _ in range(2))
    zero, inc = basis(N, (0.03, -0.02, 0.75), size)
    with gpu.Plan((re + 1j * im).astype(np.complex64), pr, N, zero, inc, t0, dT, kahan_block=kahan) as plan:
        plan.execute()
        assert "degree=" in plan.info()["kernel"]
        vol = plan.volume()
    assert np.array_equal(vol.real, oracle.a1_volume_f64acc(re, pr, N, zero, inc, t0, dT).astype(f32))
    assert np.array_equal(vol.imag, oracle.a1_volume_f64acc(im, pr, N, zero, inc, t0, dT).astype(f32))


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_values_that_are_no_numbers(gpu, value):
    """They reach the voxels that the texture path gives them to, and no other."""
    N, T = (35, 33, 17), 2001
    pr = pairs_of(15, 15)
    zero, inc = basis(N, (0.03, -0.02, 0.75), (0.25, 0.22, 0.12))
    H = np.full((len(pr), T), 0.5, f32)
    H[::7, 100::211] = value
    vols = []
    for variant in (-1, 5):
        with gpu.Plan(H, pr, N, zero, inc, 1.2, 0.001, variant=variant) as plan:
            plan.execute()
            vols.append(plan.volume())
    bad = ~np.isfinite(vols[1])
    assert 0 < bad.sum() < bad.size
    assert np.array_equal(~np.isfinite(vols[0]), bad) and np.array_equal(vols[0][~bad], vols[1][~bad])


def test_tune_may_keep_the_default_kernel(gpu):
    N, T = (48, 48, 48), 2000
    pr = pairs_of(24, 24)
    zero, inc = basis(N, (0.03, -0.02, 0.75), (0.5, 0.5, 0.5))
    H = np.random.default_rng(2).gamma(0.5, 2.0, (len(pr), T)).astype(f32)
    with gpu.Plan(H, pr, N, zero, inc, 0.5, 0.002) as plan:
        plan.execute()
        before = plan.volume().astype(np.float64)
        got = plan.tune(reps=2)
        plan.execute()
        assert plan.info()["kernel"] == got["kernel"]
        assert np.all(np.abs(plan.volume() - before) <= 68 * EPS * before)


# coarse grids and long time axes, whose tiles' bin windows or column polynomials are out of the LDS
# kernel's range: non-round volumes, one voxel, a wall that is not flat, a rotated basis
SPLIT_CASES = [((9, 7, 5), False, False), ((24, 24, 24), False, False), ((1, 1, 1), False, False),
               ((16, 8, 9), True, False), ((11, 17, 8), False, True)]


@pytest.mark.parametrize("storage,cplx", [("f32", False), ("bf16", False), ("f32", True), ("f16", True)])
@pytest.mark.parametrize("N,tilted,rotated", SPLIT_CASES)
def test_split_pairs_equal_the_whole(gpu, N, tilted, rotated, storage, cplx):
    """Pairs split over work-groups on the texture path, against the unsplit kernel of the explicit
    variant; tolerance as above."""
    pr = pairs_of(31, 33)
    if tilted:
        pr["laser_point"][:, 2] = np.linspace(0, 0.05, len(pr)).astype(f32)
        pr["camera_point"] = pr["laser_point"]
    T, dT = 3000, 0.0012
    rng = np.random.default_rng(N[0])
    H = rng.gamma(0.5, 2.0, (len(pr), T)).astype(f32)
    if cplx:
        H = (H + 1j * rng.gamma(0.5, 2.0, H.shape)).astype(np.complex64)
    zero, inc = basis(N, (0.03, -0.02, 0.75), (0.8, 0.8, 0.6))
    if rotated:
        inc = inc + np.array([0, 0, 0.004, 0, 0, 0.002, -0.004, 0.001, 0], f32)
    vols = []
    for variant in (-1, 5):
        with gpu.Plan(H, pr, N, zero, inc, 0.8, dT, variant=variant, storage=storage) as plan:
            plan.execute()
            plan.execute()
            assert plan.info()["kernel"].startswith("confocal_kernel"), plan.info()
            vols.append(plan.volume())
    a, b = vols
    assert np.abs(b).min() > 0
    for x, y in ((a.real, b.real), (a.imag, b.imag)):
        assert np.all(np.abs(x.astype(np.float64) - y) <= 68 * EPS * np.abs(y).astype(np.float64))


@pytest.mark.parametrize("storage,cplx,rows", [("f32", False, "F32Rows"), ("f16", False, "Half16Rows<false>"),
                                               ("bf16", False, "Half16Rows<true>"), ("f32", True, "ComplexRows")])
def test_reported_kernel_names_its_rows(gpu, storage, cplx, rows):
    N, size, T, dT, t0, scan = CASES[1]
    pr = pairs_of(*scan)
    H = np.random.default_rng(1).gamma(0.5, 2.0, (len(pr), T)).astype(np.complex64 if cplx else f32)
    grid = basis(N, (0.03, -0.02, 0.75), size)
    with gpu.Plan(H, pr, N, *grid, t0, dT, storage=storage) as plan:
        plan.execute()
        info = plan.info()
    kz = int(info["kernel"].split("KZ=")[1].split(",")[0])
    assert info["kernel"].startswith(f"confocal_lds_kernel_column<{rows}, KZ=") and info["lane_voxels"] == kz, info


@pytest.mark.parametrize("N,tilted,rotated", SPLIT_CASES)
def test_split_pairs_are_reported(gpu, N, tilted, rotated):
    """The plans of the test above: more than one part, and none with an explicit variant."""
    pr = pairs_of(31, 33)
    if tilted:
        pr["laser_point"][:, 2] = np.linspace(0, 0.05, len(pr)).astype(f32)
        pr["camera_point"] = pr["laser_point"]
    zero, inc = basis(N, (0.03, -0.02, 0.75), (0.8, 0.8, 0.6))
    if rotated:
        inc = inc + np.array([0, 0, 0.004, 0, 0, 0.002, -0.004, 0.001, 0], f32)
    H = np.random.default_rng(1).gamma(0.5, 2.0, (len(pr), 3000)).astype(f32)
    for variant in (-1, 5):
        with gpu.Plan(H, pr, N, zero, inc, 0.8, 0.0012, variant=variant) as plan:
            plan.execute()
            name = plan.info()["kernel"]
        assert name.startswith("confocal_kernel_split<") == (variant == -1), name
        assert variant == 5 or int(name.split("tiles, ")[1].split()[0]) > 1, name


def test_tune_may_keep_split_pairs(gpu):
    """27 tiles for 256 CUs: no kernel that leaves the pairs whole comes near the split default, so a tuned
    plan runs it still, and its volume is the untuned plan's bit for bit."""
    pr = pairs_of(61, 67)
    N, grid = (24, 24, 24), basis((24, 24, 24), (0.03, -0.02, 0.75), (0.8, 0.8, 0.6))
    H = np.random.default_rng(2).gamma(0.5, 2.0, (len(pr), 3000)).astype(f32)
    with gpu.Plan(H, pr, N, *grid, 0.8, 0.0012) as plan:
        plan.execute()
        ref, name = plan.volume(), plan.info()["kernel"]
        assert name.startswith("confocal_kernel_split<")
        got = plan.tune(reps=4)
        assert got["kernel"] == name, got
        plan.execute()
        assert plan.info()["kernel"] == name and np.array_equal(plan.volume(), ref)
