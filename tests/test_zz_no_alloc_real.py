"""bpx_backprojection_noalloc on real samples, whose sums round: the explicit texture-path variant's volume
bit for bit, the default kernel's within the rounding of both (68 units: a group of 32 added in turn is off
by at most 31 roundings, its compensated sum by 2 and the end by 1, on either side)."""
import numpy as np
import pytest

from test_gpu_count_rows import basis, pairs_of
from test_zz_no_alloc import dev, noalloc  # noqa: F401

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("N,size", [((40, 33, 38), (0.4, 0.4, 0.4)), ((9, 7, 5), (0.8, 0.8, 0.6))])
def test_noalloc_of_real_samples(gpu, dev, N, size):  # noqa: F811
    pr = pairs_of(31, 33)
    H = np.random.default_rng(8).gamma(0.5, 2.0, (len(pr), 2000)).astype(f32)
    args = (H, pr, N, *basis(N, (0.03, -0.02, 0.75), size), 0.8, 0.0015)
    got = noalloc(dev, *args)
    assert np.array_equal(got, gpu.backprojection(*args, variant=5))
    default = gpu.backprojection(*args).astype(np.float64)
    assert default.max() > 0 and np.all(np.abs(got - default) <= 68 * 2.0 ** -24 * default)
