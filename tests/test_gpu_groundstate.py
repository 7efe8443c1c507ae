"""The ground-state kernels at the edges of their ranges against the oracle: one
column, odd numbers of columns, 64 columns (the columns of the Rayleigh-Ritz
step no longer fit LDS), more columns than waves, and more bands than
Gram_Schmidt holds in LDS; and energies read together as when read one by one.
Tolerances: energies |dE| < 1e-10 Ha, orthonormal columns 1e-12, eigenvalues
1e-10 Ha (as the other parity tests)."""
import numpy as np
import pytest

import pyoracle as po
from mattohf_amd import tdhf as T

pytestmark = pytest.mark.gpu


def orbitals(S, seed):
    rng = np.random.default_rng(seed)
    u = rng.standard_normal(S.shape) + 1j * rng.standard_normal(S.shape)
    return np.asfortranarray(u)


# (ng, nk, nb, nbocc, ncg, acell, Z)
@pytest.mark.parametrize("ng,nk,nb,nbocc,ncg,acell,Z", [
    (16, 1, 1, 1, 1, 8.0, 2.0),
    (16, 3, 1, 1, 3, 8.0, 2.0),
    (32, 5, 3, 2, 1, 8.0, 4.0),
    (32, 2, 5, 4, 3, 8.0, 4.0),
    (64, 2, 16, 3, 4, 10.0, 6.0),
    (64, 65, 3, 3, 3, 10.0, 6.0),
    (128, 2, 32, 5, 2, 12.0, 6.0),
    (128, 16, 11, 11, 2, 12.0, 6.0),
])
def test_gs_edges_match_oracle(ng, nk, nb, nbocc, ncg, acell, Z):
    S = po.System(ng, nk, nb, nbocc, acell)
    vion = S.ion_potential(Z, 1.0, 0.5 * acell)
    O = po.Oracle(S, vion)
    u0 = S.gram_schmidt(orbitals(S, ng + nk))
    ub, eh, eps, _ = O.GS_calculation(u0, 2, ncg)
    with T.TDHF(ng, nk, nb, nbocc, acell, 0.01, vion) as G:
        ua, eh2, eps2, _ = G.GS_calculation(u0, 2, ncg)[:4]
    assert np.abs(np.asarray(eh2) - eh).max() < 1e-10
    assert np.abs(np.asarray(eps2) - eps).max() < 1e-10
    dv = acell / ng
    for k in range(nk):
        g = dv * ua[:, :, k].conj().T @ ua[:, :, k]
        assert np.abs(g - np.eye(nb)).max() < 1e-12


# 16, 17 columns: at and over the number of waves; 80 and 78: either side of
# the LDS at NG=128 (79 columns of 129 points)
@pytest.mark.parametrize("ng,nb", [(16, 1), (16, 16), (64, 17), (128, 78), (128, 80)])
def test_gram_schmidt_edges(ng, nb):
    S = po.System(ng, 2, nb, 1, 10.0)
    u = orbitals(S, nb)
    with T.TDHF(ng, 2, nb, 1, 10.0, 0.01, np.zeros(ng)) as G:
        g = G.Gram_Schmidt(u)
    assert np.abs(g - S.gram_schmidt(u)).max() < 1e-12 * max(1.0, np.abs(g).max()) * nb


def test_energies_read_together():
    """More iterations than are read at a time: the history is that of a run
    that reads each energy, and its state too."""
    S = po.System(16, 2, 2, 1, 8.0)
    vion = S.ion_potential(2.0, 1.0, 4.0)
    u0 = S.gram_schmidt(orbitals(S, 1))
    with T.TDHF(16, 2, 2, 1, 8.0, 0.01, vion) as G:
        a = G.GS_calculation(u0, 300, 2)
        b = G.GS_calculation(u0, 300, 2, tol=1e-300)
    ea, eb = np.asarray(a[1]), np.asarray(b[1])
    n = int(np.count_nonzero(eb)) if eb.size == ea.size else eb.size
    assert n > 1
    assert np.array_equal(ea[:n], eb[:n])
