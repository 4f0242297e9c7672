"""Calls when the device's memory runs short: what fails says so, leaves nothing behind and takes nothing
along; what a faster kernel would need beside its general form is given up instead.  Counts, so every
volume must EQUAL the oracle's exactly accumulated one."""
import ctypes
from contextlib import contextmanager

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
