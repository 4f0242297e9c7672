"""The phasor filter at the edges of its tiles: 8 outputs per lane, up to 2,048 per work-group, taps
in blocks of 8; rows shorter than the pulse, values that are no numbers.  Bit for bit the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.mark.parametrize("wl", [0.0011, 0.0023, 0.004, 0.0405, 0.9])
@pytest.mark.parametrize("rows,T", [(1, 1), (3, 7), (5, 8), (2, 9), (4, 511), (3, 512), (2, 513), (3, 2047), (2, 2048),
                                    (2, 2049), (1, 5000)])
def test_filter_equals_oracle(gpu, oracle, rows, T, wl):
    x = np.random.default_rng(T).normal(0.0, 3.0, (rows, T)).astype(f32)
    assert np.array_equal(gpu.phasor_pulse(x, wl, 0.001), oracle.phasor_filter(x, wl, 0.001))


def test_infinite_samples(gpu, oracle):
    x = np.zeros((2, 700), f32)
    x[0, 0] = np.inf            # bin 0 is never read
    x[0, 699] = np.inf
    x[1, 300] = np.nan
    with np.errstate(invalid="ignore"):
        want = oracle.phasor_filter(x, 0.004, 0.001)
    assert np.isnan(want[1]).any() and not np.isnan(want[0, :600]).any()
    got = gpu.phasor_pulse(x, 0.004, 0.001)
    for a, b in ((got.real, want.real), (got.imag, want.imag)):
        assert np.array_equal(a, b, equal_nan=True)
