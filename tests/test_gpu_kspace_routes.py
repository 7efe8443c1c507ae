"""Calls on the density-matrix path (tdhf_kspace.h) that no other module runs
there, and the reverse pair tiles over several pulses and steps.  Tolerances as in
test_gpu_kspace.py."""
import numpy as np
import pytest

from mattohf_amd import tdhf as T
from test_gpu_kspace import SYSTEMS, orbitals, rel, system

pytestmark = pytest.mark.gpu

CELL = {16: (3.6, 1.0), 32: (8.0, 4.0), 64: (10.0, 6.0), 128: (12.0, 6.0)}
SECOND_BLOCK = (128, 17, 13, 12) + CELL[128]


def test_more_columns_than_a_grid_has_in_z():
    """H and a step of 100000 bands: every band's are those of a system of few."""
    ng, nk, nb = 16, 4, 100000
    a, z = CELL[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    u = orbitals((ng, nk, 4, 1, a, z), 1)
    with T.TDHF(ng, nk, 4, 1, a, 0.004, vion) as G:
        h, s = G.ubkwbk_hwbk(u, u, 0.2), G.RT_RK4_ubk(u, 0.05, 0.1)
    many = np.empty((ng, nb, nk), dtype=complex, order="F")
    many.reshape(ng, 4, nb // 4, nk, order="F")[:] = u[:, :, None, :]
    with T.TDHF(ng, nk, nb, 1, a, 0.004, vion) as G:
        for got, ref in ((G.ubkwbk_hwbk(many, many, 0.2), h), (G.RT_RK4_ubk(many, 0.05, 0.1), s)):
            d = np.abs(got.reshape(ng, 4, nb // 4, nk, order="F") - ref[:, :, None, :])
            assert d.max() < 1e-12 * np.abs(ref).max()


def test_more_trajectories_than_a_grid_has_in_z():
    """8200 trajectories of eight bands, as a batch and as pulses of one gradient,
    against single runs (row-wise)."""
    ng, nk, nb, ntraj = 16, 16, 8, 8200
    a, z = CELL[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    us = [orbitals((ng, nk, nb, nb, a, z), t) for t in range(3)]
    A = 0.1 * np.random.default_rng(2).standard_normal((3, 2))
    many = [us[t % 3] for t in range(ntraj)]
    field = np.array([A[t % 3] for t in range(ntraj)])
    with T.TDHF(ng, nk, nb, nb, a, 0.004, vion) as G:
        ref = [G.RT_calculation(us[t], A[t], A[t]) for t in range(3)]
        gref = []
        for t in range(3):
            G.fwd_batch([us[t]], A[t:t + 1])
            gref.append([x[0] for x in G.bwd_batch()])
        G.fwd_batch(many, field)
        g, gu = G.bwd_batch()
    with T.Batch(ng, nb, nb, a, 0.004, [nk] * ntraj, np.array([vion] * ntraj)) as B:
        B.upload(many)
        e = B.propagate(field, field)[0]
        out = B.download()
    for t in (0, 1, 2, 8190, 8191, 8192, ntraj - 1):
        assert rel(out[t], ref[t % 3][0]) < 1e-12 and rel(e[t], ref[t % 3][1]) < 1e-12
        assert rel(g[t], gref[t % 3][0]) < 1e-9 and rel(gu[t], gref[t % 3][1]) < 1e-9


def launches(case):
    """Of a ground-state iteration with one Krylov block."""
    ng, nk, nb, nbocc, a, z = case
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    with T.TDHF(ng, nk, nb, nbocc, a, 0.004, vion) as G:
        G.set_kernel_timing(True)
        G.GS_calculation(orbitals(case, 1), 1, 1)
        return G.kernel_stats()[0]


@pytest.mark.parametrize("case", [c for c in SYSTEMS if c[:4] != (128, 17, 11, 10)] + [SECOND_BLOCK],
                         ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_systems_take_the_path(case):
    """The systems of test_gpu_kspace.py are there for the path (of NG=128, NK=17 the
    one with 13 bands; with 11 it is row-wise): a ground-state iteration makes the
    matrices apart from their products, three launches more than the row-wise
    five."""
    assert launches(case) == 8


@pytest.mark.parametrize("case", [(64, 32, 8, 8), (64, 16, 16, 16), (128, 40, 6, 6), (128, 16, 16, 8)],
                         ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_one_round_of_rows_is_row_wise(case):
    """Up to 256 rows, one for each CU: the row-wise kernel is the faster one."""
    assert launches(case + CELL[case[0]]) == 5


def test_largest_pinned_state():
    """16384 elements, the most that go through pinned memory, on the path."""
    case = (32, 64, 8, 8) + CELL[32]
    assert launches(case) == 8
    S, O, G, _ = system(case)
    with G:
        for seed in (1, 2):  # (the memory is used again)
            u, w = orbitals(case, seed), orbitals(case, 10 + seed)
            assert rel(G.ubkwbk_hwbk(u, w, 0.2), O.ubkwbk_hwbk(u, w, 0.2)) < 1e-12
            assert rel(G.RT_RK4_ubk(u, 0.05, 0.1), O.RT_RK4_ubk(u, G.dt, 0.05, 0.1)) < 1e-12
            np.testing.assert_array_equal(G.download(), G.RT_RK4_ubk(u, 0.05, 0.1))


def test_just_past_a_transform_length_with_an_empty_band():
    """NG=128, one k-point past the transforms of length 16, thirteen bands in two
    blocks, one of them empty."""
    S, O, G, _ = system(SECOND_BLOCK)
    u, w = orbitals(SECOND_BLOCK, 1), orbitals(SECOND_BLOCK, 2)
    A = np.array([0.1, -0.05])
    with G:
        assert rel(G.ubkwbk_hwbk(u, w, 0.2), O.ubkwbk_hwbk(u, w, 0.2)) < 1e-12
        ug, eg, _, jg, _ = G.RT_calculation(u, A, A)
    uo, eo, _, jo, _ = O.RT_calculation(u, 0.004, A, A)
    assert rel(ug, uo) < 1e-12 and np.abs(eg - eo).max() < 1e-10 and rel(jg, jo) < 1e-8


@pytest.mark.parametrize("variant", [0, 1, 2], ids=["TE", "TEPC", "TEPC2"])
@pytest.mark.parametrize("case", [SYSTEMS[3], SYSTEMS[5]], ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_taylor_steps_match_oracle(case, variant):
    S, O, G, _ = system(case)
    ug = uo = orbitals(case, 1)
    with G:
        for aave in (0.05, -0.07):
            ug, uo = G.TE_step(ug, aave, variant), O.TE_step(uo, G.dt, aave, variant)
            assert rel(ug, uo) < 1e-12
        np.testing.assert_array_equal(G.download(), ug)


def test_ground_state_columns_match_oracle():
    case = (32, 65, 7, 6, 8.0, 4.0)
    S, O, G, _ = system(case)
    u = orbitals(case, 1)
    with G:
        _, eh, eps, err, dg = G.GS_calculation_diag(u, 3, 4)
    _, eho, epso, erro, dgo = O.GS_calculation_diag(u, 3, 4)
    np.testing.assert_allclose(eh, eho, rtol=0, atol=1e-10)
    np.testing.assert_allclose(eps, epso, rtol=0, atol=1e-10)
    np.testing.assert_allclose(err, erro, rtol=1e-6, atol=1e-9)
    np.testing.assert_allclose(dg, dgo, rtol=1e-6, atol=1e-9)


@pytest.mark.parametrize("objective", ["energy", "jsq"])
def test_pair_tiles_of_many_pulses(objective):
    """44 pulses of a system whose tiles (six each; one pulse is row-wise) fill half
    the CUs only together: each pulse's own gradient, over three steps."""
    ng, nk, nb, nt, ntraj = 128, 8, 6, 3, 44
    a, z = CELL[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    us = [orbitals((ng, nk, nb, nb, a, z), t) for t in range(ntraj)]
    A = 0.1 * np.random.default_rng(4).standard_normal((ntraj, nt))
    with T.TDHF(ng, nk, nb, nb, a, 0.004, vion) as G:
        L, fin, _, _, _ = G.fwd_batch(us, A, objective=objective)
        g, gu = G.bwd_batch()
        for t in (0, 21, 43):
            L1, f1, _, _, _ = G.fwd_batch([us[t]], A[t:t + 1], objective=objective)
            g1, gu1 = G.bwd_batch()
            assert abs(L[t] - L1[0]) < 1e-11 * max(1.0, abs(L1[0])) and rel(fin[t], f1[0]) < 1e-12
            assert rel(g[t], g1[0]) < 1e-9 and rel(gu[t], gu1[0]) < 1e-9
