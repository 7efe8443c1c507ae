"""The Fourier transform of the observables at phases omega t on both sides of
2^26, from where each sine and cosine is taken by itself, and far beyond: against
the oracle.  Tolerance: 600 terms of three roundings each against a sum of the
size of their root, 600^(1/2) 3 2^-53 < 1e-13 of the largest value; 1e-12."""
import numpy as np
import pytest

import pyoracle as po
from mattohf_amd import tdhf as T


@pytest.mark.gpu
@pytest.mark.parametrize("nomega", [257, 1025, 2049, 4001])  # 1, 4, 8 and 16 at a time, and one left
@pytest.mark.parametrize("phase", [0.9 * 2.0 ** 26, 1.5 * 2.0 ** 26, 1e11, 1e14, -1e11])
def test_large_phases_match_oracle(nomega, phase):
    nt, omegam = 600, 2.0
    rng = np.random.default_rng(nomega)
    t = abs(phase) / omegam * np.sort(rng.random(nt))
    J, E, A = rng.standard_normal((3, nt))
    args = (t, J, 0.2, E, A, 0.8, nomega, np.copysign(omegam, phase))
    got, want = T.fourier(*args), po.fourier(*args)
    np.testing.assert_allclose(got[:, 1:], want[:, 1:], rtol=0, atol=1e-12 * np.abs(want[:, 1:]).max())


@pytest.mark.gpu
@pytest.mark.parametrize("nomega", [257, 741, 1025, 2049, 4001])
@pytest.mark.parametrize("omegam", [2.5, -1.7, 0.057])
def test_frequencies_that_are_rounded(nomega, omegam):
    """Largest frequencies of more than one bit: i/nomega omegam is rounded, and the
    phases are of the rounded ones.  A unit of omega t in its last place is 1e-12
    at phases of 1e4; 600 terms of ten roundings each, at worst all of one sign,
    600 10 2^-53 against a largest value of over 10: 1e-13."""
    rng = np.random.default_rng(nomega)
    t = 2e4 / abs(omegam) * np.sort(rng.random(600))
    J, E, A = rng.standard_normal((3, 600))
    args = (t, J, 0.2, E, A, 0.8, nomega, omegam)
    got, want = T.fourier(*args), po.fourier(*args)
    np.testing.assert_array_equal(got[:, 0], want[:, 0])
    np.testing.assert_allclose(got[:, 1:], want[:, 1:], rtol=0, atol=1e-13 * np.abs(want[:, 1:]).max())
