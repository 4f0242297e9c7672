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
