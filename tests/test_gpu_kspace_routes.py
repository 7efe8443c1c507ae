"""Calls on the density-matrix path (tdhf_kspace.h) that no other module runs
there.  Tolerances as in test_gpu_kspace.py."""
import numpy as np
import pytest

from mattohf_amd import tdhf as T
from test_gpu_kspace import orbitals, rel

pytestmark = pytest.mark.gpu

CELL = {16: (3.6, 1.0), 32: (8.0, 4.0), 64: (10.0, 6.0), 128: (12.0, 6.0)}


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
