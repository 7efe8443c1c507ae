"""The row-wise kernels at the edges of their split: every number of waves, a
last pass in which one or all but one of the lane groups of a wave have a pair,
one pair in all, more bands than are occupied.  Against the oracle, at the
tolerances of the density-matrix path's tests."""
import numpy as np
import pytest

from mattohf_amd import tdhf as T
from test_gpu_kspace import orbitals, rel, system

pytestmark = pytest.mark.gpu

A16, A32, A64, A128 = (3.6, 1.0), (8.0, 4.0), (10.0, 6.0), (12.0, 6.0)
# (ng, nk, nb, nbocc, acell, Z): NG = 16 and 32 hold 16 pairs per wave, 64
# eight, 128 four
CASES = [(16, 1, 1, 1) + A16, (16, 17, 2, 1) + A16, (16, 11, 3, 3) + A16, (16, 43, 3, 3) + A16,
         (32, 1, 1, 1) + A32, (32, 16, 2, 1) + A32, (32, 7, 5, 5) + A32, (32, 19, 5, 5) + A32,
         (64, 1, 2, 1) + A64, (64, 3, 3, 3) + A64, (64, 21, 3, 3) + A64, (64, 13, 5, 5) + A64,
         (64, 5, 13, 13) + A64, (128, 1, 1, 1) + A128, (128, 3, 3, 3) + A128, (128, 7, 3, 3) + A128,
         (128, 11, 3, 3) + A128]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"ng{c[0]}_nk{c[1]}_nb{c[2]}_{c[3]}")
def test_rows_match_oracle(case):
    S, O, G, _ = system(case)
    u, w = orbitals(case, 1), orbitals(case, 2)
    with G:
        assert rel(G.ubkwbk_hwbk(u, w, 0.23), O.ubkwbk_hwbk(u, w, 0.23)) < 1e-12
        _, ec, n, j = G.observables(u, -0.17)
        assert rel(ec, O.ubk_Ecomps(u, -0.17)) < 1e-12
        assert abs(n - O.nele(u)) < 1e-12 and abs(j - O.ubk_Je(u, -0.17)) < 1e-12 * max(1.0, abs(j))
        A, Aave = np.array([0.1, 0.25, -0.1]), np.array([0.05, 0.175, 0.075])
        ug, eg, _, jg, i3 = G.RT_calculation(u, A, Aave)
        uo, eo, _, jo, i3o = O.RT_calculation(u, G.dt, A, Aave)
        assert rel(ug, uo) < 1e-12 and np.abs(eg - eo).max() < 1e-10
        assert rel(jg, jo) < 1e-8 and np.abs(i3 - i3o).max() < 1e-10


# (the adjoint takes occupied bands only; the last case is large enough for the
# pair tiles and, with over 128 k-points, outside the density-matrix path)
@pytest.mark.parametrize("case", [c for c in CASES if c[2] == c[3]] +
                         [(128, 130, 4, 4) + A128],
                         ids=lambda c: f"ng{c[0]}_nk{c[1]}_nb{c[2]}_{c[3]}")
def test_row_adjoint_matches_oracle(case):
    S, O, G, _ = system(case)
    big = case[1] > 128  # (seconds in the oracle: one step, one objective)
    u, A = orbitals(case, 3), np.array([0.1] if big else [0.1, -0.05])
    for objective, oracle in (("energy", "adjoint_energy"), ("jsq", "adjoint_jsq"))[:1 if big else 2]:
        L, _, _, _, _ = G.fwd_batch([u], A[None], objective=objective)
        g, gu = G.bwd_batch()
        ref = getattr(O, oracle)(u, G.dt, A)
        assert abs(L[0] - ref[0]) < 1e-11 * max(1.0, abs(ref[0]))
        assert np.abs(g[0] - ref[1]).max() < 1e-9 * np.abs(ref[1]).max()
        assert np.abs(gu[0] - ref[2]).max() < 1e-9 * np.abs(ref[2]).max()
    G.close()


# 16384 elements, the largest state that goes through pinned memory, row-wise
# and on the density-matrix path, and one beyond
@pytest.mark.parametrize("case", [(128, 16, 8, 2) + A128, (64, 32, 8, 8) + A64,
                                  (128, 17, 8, 2) + A128], ids=lambda c: f"ng{c[0]}_nk{c[1]}")
def test_staged_calls_match_oracle(case):
    S, O, G, _ = system(case)
    with G:
        for seed in (1, 2):  # (the memory is used again)
            u, w = orbitals(case, seed), orbitals(case, 10 + seed)
            assert rel(G.ubkwbk_hwbk(u, w, 0.2), O.ubkwbk_hwbk(u, w, 0.2)) < 1e-12
            ref = O.RT_RK4_ubk(u, G.dt, 0.05, 0.1)
            assert rel(G.RT_RK4_ubk(u, 0.05, 0.1), ref) < 1e-12
            np.testing.assert_array_equal(G.download(), G.RT_RK4_ubk(u, 0.05, 0.1))


# up to two rows per CU (512), up to four, more; one pair in all; NG = 128, which
# needs two waves
@pytest.mark.parametrize("ng,nb,nks,ntraj", [(32, 2, [7, 12, 20], 6), (32, 2, [7, 12, 20], 30),
                                             (16, 3, [5, 9, 4], 80), (64, 1, [1], 3),
                                             (128, 2, [3, 5], 40)])
def test_default_batch_shape(ng, nb, nks, ntraj):
    a, z = {16: A16, 32: A32, 64: A64, 128: A128}[ng]
    nk = [nks[t % len(nks)] for t in range(ntraj)]
    vi = {k: T.ion_potential(ng, k, a, [z], [1.0], [0.0]) for k in nks}
    rng = np.random.default_rng(3)
    A = 0.1 * rng.standard_normal((ntraj, 3))
    us = [orbitals((ng, k, nb, nb, a, z), t) for t, k in enumerate(nk)]
    with T.Batch(ng, nb, nb, a, 0.004, nk, np.array([vi[k] for k in nk])) as B:
        out = []
        for shape in (None, (ng + 63) // 64):
            if shape:
                B.set_schedule(0)
                B.set_waves(shape)
            B.upload(us)
            e, n, j, _ = B.propagate(A, A)
            out.append((B.download(), e, j))
    for u, v in zip(out[0][0], out[1][0]):
        assert rel(u, v) < 1e-12
    assert np.abs(out[0][1] - out[1][1]).max() < 1e-10 and rel(out[0][2], out[1][2]) < 1e-8


# waves of the product launch (density matrices) or of a row, by the rows of the
# fullest XCD: 5 per CU, 6, 9 (12 at NG = 16); 480 workgroups of matrices at NG = 16;
# 14 pairs a row at NG = 128, on more rows than CUs and on as many
@pytest.mark.parametrize("ng,nk,nb,ntraj,waves", [(64, 40, 4, 5, 2), (32, 48, 4, 4, 1),
                                                  (32, 140, 2, 2, 2), (16, 96, 4, 2, 1),
                                                  (16, 21, 6, 30, 4), (128, 7, 2, 19, 2),
                                                  (128, 7, 2, 18, 4)])
def test_default_batch_waves(ng, nk, nb, ntraj, waves):
    a, z = {16: A16, 32: A32, 64: A64, 128: A128}[ng]
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    u = orbitals((ng, nk, nb, nb, a, z), 1)
    A = np.tile([0.05, 0.1], (ntraj, 1))
    with T.TDHF(ng, nk, nb, nb, a, 0.004, vion) as G:
        ref = G.RT_calculation(u, A[0], A[0])
    with T.Batch(ng, nb, nb, a, 0.004, [nk] * ntraj, np.array([vion] * ntraj)) as B:
        assert B.waves() == waves
        B.upload([u] * ntraj)
        e = B.propagate(A, A)[0]
        out = B.download()
    for t in (0, ntraj - 1):
        assert rel(out[t], ref[0]) < 1e-12 and np.abs(e[t] - ref[1]).max() < 1e-10


@pytest.mark.parametrize("nk,nb,nw", [(64, 3, 1), (64, 3, 2), (65, 4, 1), (191, 1, 1), (201, 1, 1)])
def test_rows_of_one_wave(nk, nb, nw):
    """NG=32: from 192 pairs a row of one wave runs a variant of its own; even and
    odd numbers of passes, with groups that have no last pair, against single runs."""
    ng, ntraj = 32, 3
    a, z = A32
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.0])
    us = [orbitals((ng, nk, nb, nb, a, z), t) for t in range(ntraj)]
    A = 0.1 * np.random.default_rng(5).standard_normal((ntraj, 2))
    ref = []
    with T.TDHF(ng, nk, nb, nb, a, 0.004, vion) as G:
        ref = [G.RT_calculation(u, A[t], A[t]) for t, u in enumerate(us)]
    # one trajectory of few k-points besides: the largest one decides
    v2 = T.ion_potential(ng, 2, a, [z], [1.0], [0.0])
    u2 = orbitals((ng, 2, nb, nb, a, z), 9)
    with T.Batch(ng, nb, nb, a, 0.004, [nk] * ntraj + [2], np.array([vion] * ntraj + [v2])) as B:
        B.set_waves(nw)
        B.upload(us + [u2])
        F = np.concatenate([A, A[:1]])
        e, _, j, _ = B.propagate(F, F)
        out = B.download()
    for t in range(ntraj):
        assert rel(out[t], ref[t][0]) < 1e-12
        assert np.abs(e[t] - ref[t][1]).max() < 1e-10 and rel(j[t], ref[t][3]) < 1e-8
