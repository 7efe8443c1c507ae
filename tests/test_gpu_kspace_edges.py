"""Calls at the edges of the density-matrix path (tdhf_kspace.h): launch shapes,
numbers of columns and trajectories, memory, timing.  The systems are well over
the line from which the library takes the path (twice the row-wise cost or
more, except where a test says otherwise).  Tolerances as in
test_gpu_kspace.py."""
import numpy as np
import pytest

from mattohf_amd import tdhf as T
from test_gpu_kspace import orbitals, rel, system

pytestmark = pytest.mark.gpu

CELL = {16: (3.6, 1.0), 32: (8.0, 4.0), 64: (10.0, 6.0), 128: (12.0, 6.0)}


@pytest.mark.parametrize("ng,nk,nb,ntraj", [(64, 64, 4, 9), (16, 16, 4, 300)])
def test_waves_that_are_no_power_of_two(ng, nk, nb, ntraj):
    """3, 5, 6 and 7 waves of the product launch: the points do not divide among
    them, the results are those of 1, 2, 4 and 8."""
    a, z = CELL[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    A = 0.1 * np.random.default_rng(1).standard_normal((ntraj, 2))
    us = [orbitals((ng, nk, nb, nb, a, z), t) for t in range(ntraj)]
    with T.Batch(ng, nb, nb, a, 0.004, [nk] * ntraj, np.array([vion] * ntraj)) as B:
        out = {}
        for nw in (4, 3, 5, 6, 7):
            B.set_waves(nw)
            B.upload(us)
            out[nw] = B.propagate(A, A)[0], B.download()
    for nw in (3, 5, 6, 7):
        assert rel(out[nw][0], out[4][0]) < 1e-12
        for u, v in zip(out[nw][1], out[4][1]):
            assert rel(u, v) < 1e-12


# the density-matrix path (pinned memory, and a state too large for it) and the
# row-wise one
@pytest.mark.parametrize("case", [(16, 128, 8, 8), (64, 64, 8, 8), (32, 4, 2, 2)],
                         ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_launches_are_timed(case):
    """Four launches a step; in the ground state every product with H."""
    a, z = CELL[case[0]]
    vion = T.ion_potential(case[0], case[1], a, [z], [1.0], [0.0])
    u = orbitals(case + (a, z), 1)
    with T.TDHF(*case, a, 0.004, vion) as G:
        G.set_kernel_timing(True)
        for _ in range(2):
            u = G.RT_RK4_ubk(u, 0.1, 0.1)
        n, ms = G.kernel_stats()
        assert n == 8 and ms > 0.0
        G.set_kernel_timing(True)
        G.GS_calculation(u, 1, 2)
        assert G.kernel_stats()[0] >= 6  # energies 2, Krylov products 2, subspace 1, residuals 1


def test_many_pulses_of_a_row_wise_system():
    """One trajectory is row-wise, twenty-four go through the matrices, whose tables
    their first forward call makes: batch against single runs, twice."""
    ng, nk, nb, nt, ntraj = 64, 32, 4, 3, 24
    a, z = CELL[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    us = [orbitals((ng, nk, nb, nb, a, z), t) for t in range(ntraj)]
    A = 0.1 * np.random.default_rng(4).standard_normal((ntraj, nt))
    with T.TDHF(ng, nk, nb, nb, a, 0.004, vion) as G:
        for objective in ("energy", "jsq"):
            L, fin, _, _, _ = G.fwd_batch(us, A, objective=objective)
            g, gu = G.bwd_batch()
            for t in (0, 11, 23):
                L1, f1, _, _, _ = G.fwd_batch([us[t]], A[t:t + 1], objective=objective)
                g1, gu1 = G.bwd_batch()
                assert abs(L[t] - L1[0]) < 1e-11 * max(1.0, abs(L1[0])) and rel(fin[t], f1[0]) < 1e-12
                assert rel(g[t], g1[0]) < 1e-9 and rel(gu[t], gu1[0]) < 1e-9


# either side of where one H application of host arrays takes the path, beside
# steps of the same context, which do
@pytest.mark.parametrize("case", [(64, 33, 9, 8), (64, 64, 13, 13), (128, 16, 13, 13), (128, 33, 12, 12),
                                  (32, 65, 17, 17), (16, 128, 9, 9)],
                         ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_one_application_between_steps(case):
    case = case + CELL[case[0]]
    S, O, G, _ = system(case)
    u, w = orbitals(case, 1), orbitals(case, 2)
    h, s = O.ubkwbk_hwbk(u, w, 0.2), O.RT_RK4_ubk(u, G.dt, 0.05, 0.1)
    with G:
        for _ in range(2):
            assert rel(G.ubkwbk_hwbk(u, w, 0.2), h) < 1e-12
            assert rel(G.RT_RK4_ubk(u, 0.05, 0.1), s) < 1e-12


@pytest.mark.parametrize("case", [(16, 3, 2, 1), (64, 64, 8, 8)], ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_ground_state_ends_soon_after_a_bad_energy(case):
    """Orbitals that are not numbers: the first iteration's energy is none, and the
    run of 200 ends by it (launches counted on the row-wise and the
    density-matrix path; at most 7 and 9 an iteration)."""
    a, z = CELL[case[0]]
    vion = T.ion_potential(case[0], case[1], a, [z], [1.0], [0.0])
    u = orbitals(case + (a, z), 1)
    u[0, 0, 0] = np.nan
    with T.TDHF(*case, a, 0.004, vion) as G:
        G.set_kernel_timing(True)
        with pytest.raises(T.TDHFError, match="iteration 1"):
            G.GS_calculation(u, 200, 2)
        assert G.kernel_stats()[0] <= 16 * 9
        # and one that is: the energies of a run longer than is read at a time
        u[0, 0, 0] = 0.0
        long, short = G.GS_calculation(u, 33, 2)[1], G.GS_calculation(u, 33, 2, tol=1e-300)[1]
        n = np.count_nonzero(short)
        assert n > 17 and np.array_equal(long[:n], short[:n])


def test_ground_state_of_more_columns_than_bands():
    """Twelve Krylov columns of four bands: the product kernel's variant of eight
    columns and two grid points (64 KB of LDS and more), which no other call of
    the context launches, against the oracle."""
    case = (128, 96, 4, 4) + CELL[128]
    S, O, G, _ = system(case)
    u = orbitals(case, 1)
    with G:
        _, eh, eps, _ = G.GS_calculation(u, 1, 3)
    _, eo, epso, _ = O.GS_calculation(u, 1, 3)
    assert np.abs(np.asarray(eh) - eo).max() < 1e-10 and np.abs(np.asarray(eps) - epso).max() < 1e-10


def test_states_beyond_32_bit_offsets():
    """1.2 million bands of two k-points, 4.9 GB with the k-points padded to
    sixteen: row-wise.  Every band's H w is that of a system of few bands."""
    ng, nk, nb = 16, 2, 1200000
    a, z = CELL[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    u = orbitals((ng, nk, 4, 1, a, z), 1)
    with T.TDHF(ng, nk, 4, 1, a, 0.004, vion) as G:
        ref = G.ubkwbk_hwbk(u, u, 0.2)
    many = np.empty((ng, nb, nk), dtype=complex, order="F")
    many.reshape(ng, 4, nb // 4, nk, order="F")[:] = u[:, :, None, :]
    with T.TDHF(ng, nk, nb, 1, a, 0.004, vion) as G:
        h = G.ubkwbk_hwbk(many, many, 0.2)
    d = np.abs(h.reshape(ng, 4, nb // 4, nk, order="F") - ref[:, :, None, :])
    assert d.max() < 1e-12 * np.abs(ref).max()
