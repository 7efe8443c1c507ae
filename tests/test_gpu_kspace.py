"""The density-matrix path (tdhf_kspace.h, tdhf_kadjoint.h): its Toeplitz
product on the CPU against the pair convolutions it stands for, and the GPU
path against the oracle at the edges of its k transforms (16, 32, 64, 128),
with empty bands, more bands than a workgroup holds and every grid size.  The
systems are large enough for the library to choose the path.
Tolerances: operators max|d| / max|ref| < 1e-12, energies 1e-10 Ha, gradients
1e-9 of the largest component (as the other parity tests)."""
import numpy as np
import pytest

import pyoracle as po
from mattohf_amd import tdhf as T


def rel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("nk", [1, 5, 16, 17, 32])
def test_toeplitz_product_equals_pair_convolutions(nk):
    """K_k(x,x') = sum_q T_{k-q}(x-x') rho_q(x,x') by a circulant and a
    skew-circulant product of length N >= NK, for a table with no symmetry at
    all, equals sum_qj IFFT[t_kq FFT[w conj(u_qj)]] u_qj."""
    ng, nb, rng = 8, 2, np.random.default_rng(nk)
    n = 16 if nk <= 16 else 32
    t = rng.standard_normal((2 * nk - 1, ng))
    u = rng.standard_normal((nk, nb, ng)) + 1j * rng.standard_normal((nk, nb, ng))
    w = rng.standard_normal((nk, nb, ng)) + 1j * rng.standard_normal((nk, nb, ng))
    ref = np.zeros_like(w)
    for k in range(nk):
        for q in range(nk):
            for j in range(nb):
                p = np.fft.fft(w[k] * u[q, j].conj(), axis=1)
                ref[k] += np.fft.ifft(t[k - q + nk - 1] * p, axis=1) * u[q, j]
    ty = np.fft.ifft(t, axis=1)  # T_d(y), d = row - (nk - 1)
    td = np.zeros((2 * n, ng), complex)  # d = -n .. n-1
    for d in range(-(nk - 1), nk):
        td[d + n] = ty[d + nk - 1]
    tw = np.exp(-1j * np.pi * np.arange(n) / n)[:, None, None]
    c, s = 0.5 * (td[n:] + td[:n]), 0.5 * (td[n:] - td[:n])
    y = (np.arange(ng)[:, None] - np.arange(ng)[None, :]) % ng
    rho = np.zeros((n, ng, ng), complex)
    rho[:nk] = np.einsum("qjx,qjy->qxy", u, u.conj())
    f = lambda m, z: np.fft.ifft(np.fft.fft(m, axis=0)[:, y] * np.fft.fft(z, axis=0), axis=0)  # noqa: E731
    K = f(c, rho) + tw.conj() * f(s * tw[:, :, 0], tw * rho)
    got = np.einsum("kxy,kiy->kix", K[:nk], w)
    assert rel(got, ref) < 1e-13
    assert rel(K[:nk], K[:nk].conj().transpose(0, 2, 1)) < 1e-13


# (ng, nk, nb, nbocc, acell, Z): both sides of the transform lengths, more
# than 8 bands (two blocks of bands), odd band counts, empty bands
SYSTEMS = [
    (128, 16, 11, 11, 12.0, 6.0),
    (128, 17, 11, 10, 12.0, 6.0),
    (64, 32, 9, 8, 10.0, 6.0),
    (64, 33, 8, 8, 10.0, 6.0),
    (64, 64, 5, 5, 10.0, 6.0),
    (32, 65, 6, 6, 8.0, 4.0),
    (16, 128, 5, 4, 3.6, 1.0),
]


def system(case, dt=0.004):
    ng, nk, nb, nbocc, a, z = case
    S = po.System(ng, nk, nb, nbocc, a)
    vion = T.ion_potential(ng, nk, a, [z], [1.0], [0.1])
    G = T.TDHF(ng, nk, nb, nbocc, a, dt, vion)
    _, vq = G.tables()
    full = np.empty((nk * nk, ng))
    for r in range(nk):
        for c in range(nk):
            full[r * nk + c] = vq[r - c + nk - 1]
    return S, po.Oracle(S, vion, full), G, vion


def orbitals(case, seed):
    ng, nk, nb, _, a, _ = case
    rng = np.random.default_rng(seed)
    g = np.abs(np.fft.fftfreq(ng, 1.0 / ng))
    c = np.exp(-0.4 * g) * (rng.standard_normal((nk, nb, ng)) + 1j * rng.standard_normal((nk, nb, ng)))
    q, _ = np.linalg.qr(np.fft.ifft(c, axis=2).transpose(0, 2, 1))
    return np.asfortranarray(q.transpose(1, 2, 0) / np.sqrt(a / ng))


@pytest.mark.gpu
@pytest.mark.parametrize("case", SYSTEMS, ids=lambda c: f"ng{c[0]}_nk{c[1]}_nb{c[2]}_{c[3]}")
def test_operators_and_steps_match_oracle(case):
    S, O, G, _ = system(case)
    u, w = orbitals(case, 1), orbitals(case, 2)
    with G:
        assert rel(G.ubkwbk_hwbk(u, w, 0.23), O.ubkwbk_hwbk(u, w, 0.23)) < 1e-12
        e, ec, n, j = G.observables(u, -0.17)
        assert rel(ec, O.ubk_Ecomps(u, -0.17)) < 1e-12
        assert abs(n - O.nele(u)) < 1e-12 and abs(j - O.ubk_Je(u, -0.17)) < 1e-12 * max(1.0, abs(j))
        A = np.array([0.1, 0.25])
        Aave = np.array([0.05, 0.175])
        ug, eg, _, jg, i3 = G.RT_calculation(u, A, Aave)
        uo, eo, _, jo, i3o = O.RT_calculation(u, G.dt, A, Aave)
        assert rel(ug, uo) < 1e-12 and np.abs(eg - eo).max() < 1e-10
        assert rel(jg, jo) < 1e-8 and np.abs(i3 - i3o).max() < 1e-10
        np.testing.assert_array_equal(G.RT_RK4_ubk(u, 0.05, 0.1), G.RT_calculation(u, A[:1], Aave[:1])[0])


@pytest.mark.gpu
@pytest.mark.parametrize("objective", ["energy", "jsq"])
@pytest.mark.parametrize("case", [SYSTEMS[0], SYSTEMS[3], SYSTEMS[5]],
                         ids=lambda c: f"ng{c[0]}_nk{c[1]}_nb{c[2]}")
def test_adjoint_matches_oracle(case, objective):
    S, O, G, _ = system(case)
    u, A = orbitals(case, 3), np.array([0.1, -0.05])
    with G:
        L, _, _, _, _ = G.fwd_batch([u], A[None], objective=objective)
        g, gu = G.bwd_batch()
    ref = O.adjoint_energy(u, G.dt, A) if objective == "energy" else O.adjoint_jsq(u, G.dt, A)
    assert abs(L[0] - ref[0]) < 1e-11 * max(1.0, abs(ref[0]))
    assert np.abs(g[0] - ref[1]).max() < 1e-9 * np.abs(ref[1]).max()
    assert np.abs(gu[0] - ref[2]).max() < 1e-9 * np.abs(ref[2]).max()


@pytest.mark.gpu
@pytest.mark.parametrize("ng,nks,nb", [(64, [16, 32, 64] * 4, 4), (16, [128, 3, 40, 17] * 3, 5),
                                       (64, [48] * 9, 3)])
def test_batch_matches_single_runs(ng, nks, nb):
    """Mixed and uniform k-meshes through one batch, in every schedule and
    launch shape, against each trajectory's own run; uploads of one trajectory
    and downloads between calls keep the layouts apart."""
    a, nt, dt = {16: 3.6, 64: 10.0}[ng], 3, 0.004
    rng = np.random.default_rng(5)
    A = 0.1 * rng.standard_normal((len(nks), nt))
    Aave = 0.5 * (A + np.concatenate([np.zeros((len(nks), 1)), A[:, :-1]], 1))
    vi = {k: T.ion_potential(ng, k, a, [4.0], [1.0], [0.0]) for k in set(nks)}
    us = [orbitals((ng, k, nb, nb, a, 0), 10 + t) for t, k in enumerate(nks)]
    ref = {}
    for t in (0, 1, len(nks) - 1):
        with T.TDHF(ng, nks[t], nb, nb, a, dt, vi[nks[t]]) as G:
            ref[t] = G.RT_calculation(us[t], A[t], Aave[t])
    with T.Batch(ng, nb, nb, a, dt, nks, np.array([vi[k] for k in nks])) as B:
        for sched, nw in ((0, 1), (1, 4), (2, 8)):
            B.set_schedule(sched)
            B.set_waves(nw)
            B.upload(us)
            B.propagate(A[:, :1], Aave[:, :1])
            B.upload(B.download())
            flat = np.asfortranarray(us[1])
            assert T.load().tdhf_batch_upload(B.h, 1, flat.ctypes.data) == 0
            B.upload(us)
            e, n, j, i3 = B.propagate(A, Aave)
            finals = B.download()
            for t, (u1, e1, n1, j1, i31) in ref.items():
                np.testing.assert_allclose(finals[t], u1, rtol=0, atol=1e-12)
                np.testing.assert_allclose(e[t], e1, rtol=0, atol=1e-12 * np.abs(e1).max())
                np.testing.assert_allclose(j[t], j1, rtol=0, atol=1e-12 * max(1.0, np.abs(j1).max()))
