"""The Fourier transform of the observables with 1, 4, 8 and 16 frequencies per
workgroup, a last workgroup that is not full, and fewer, as many and more times
than threads, against the oracle (the tolerance of its other test)."""
import numpy as np
import pytest

import pyoracle as po
from mattohf_amd import tdhf as T


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 1])
@pytest.mark.parametrize("nt,nomega", [(2, 1), (513, 256), (512, 257), (511, 1023), (600, 2047),
                                       (40, 2049), (300, 4001)])
def test_fourier_splits_match_oracle(nt, nomega, window):
    rng = np.random.default_rng(nt)
    dt = 0.8
    t = dt * (np.arange(nt) + 0.3 * rng.random(nt))
    J, E, A = rng.standard_normal((3, nt))
    args = (t, J, 0.2, E, A, dt, nomega, 2.0)
    got = T.fourier(*args, window=window, tpulse=0.7 * dt * nt, nenvelope=3)
    want = po.fourier(*args, window=window, tpulse=0.7 * dt * nt, nenvelope=3)
    np.testing.assert_array_equal(got[:, 0], want[:, 0])
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-11 * np.abs(want).max())
