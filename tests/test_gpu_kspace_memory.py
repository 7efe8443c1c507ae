"""Calls that would take the density-matrix path (tdhf_kspace.h) on a device
whose memory holds the row-wise form only: they run row-wise.  The rest of the
memory is held by one allocation during the call; a gigabyte or more stays
free."""
import ctypes as C
from contextlib import contextmanager

import numpy as np
import pytest

from mattohf_amd import tdhf as T
from test_gpu_kspace import orbitals, rel

pytestmark = pytest.mark.gpu

GIB = 1 << 30
NG, NK, NB, NTRAJ, ACELL = 16, 33, 3, 8000, 3.6


@contextmanager
def free_memory(leave):
    """All device memory but `leave` bytes allocated meanwhile."""
    hip = C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    free, total, p = C.c_size_t(), C.c_size_t(), C.c_void_p()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    assert free.value > leave and hip.hipMalloc(C.byref(p), free.value - leave) == 0
    try:
        yield
    finally:
        hip.hipDeviceSynchronize()
        hip.hipFree(p)


def batch():
    vion = T.ion_potential(NG, NK, ACELL, [1.0], [1.0], [0.0])
    us = [orbitals((NG, NK, NB, NB, ACELL, 1.0), t) for t in range(3)]
    A = 0.1 * np.random.default_rng(2).standard_normal((3, 80))
    return vion, us, A


def test_context():
    """Padded states of 9.8 GB, 1.2 GB as they are."""
    nb = 400000
    vion = T.ion_potential(NG, 2, ACELL, [1.0], [1.0], [0.0])
    u = orbitals((NG, 2, 4, 1, ACELL, 1.0), 1)
    with T.TDHF(NG, 2, 4, 1, ACELL, 0.004, vion) as G:
        ref = G.ubkwbk_hwbk(u, u, 0.2)
    big = np.asfortranarray(np.concatenate([u] * (nb // 4), axis=1))
    with free_memory(4 * GIB), T.TDHF(NG, 2, nb, 1, ACELL, 0.004, vion) as G:
        h = G.ubkwbk_hwbk(big, big, 0.2)
    for i in (0, nb // 2, nb - 4):
        assert rel(h[:, i:i + 4], ref) < 1e-12


def test_gradients():
    """The matrices (4.5 GB) fit, the padded states and the tape beside them do
    not."""
    vion, us, A = batch()
    with T.TDHF(NG, NK, NB, NB, ACELL, 0.004, vion) as G:
        G.fwd_batch(us, A[:, :1])
        ref = G.bwd_batch()
        many = [us[t % 3] for t in range(NTRAJ)]
        field = np.array([A[t % 3, :1] for t in range(NTRAJ)])
        with free_memory(6 * GIB):
            G.fwd_batch(many, field)
            g, gu = G.bwd_batch()
    for t in (0, 1, 2, NTRAJ - 1):
        assert rel(g[t], ref[0][t % 3]) < 1e-11 and rel(gu[t], ref[1][t % 3]) < 1e-11


@pytest.mark.parametrize("when", ["create", "propagate"])
def test_batch_memory(when):
    """The matrices (2.2 GB) fit, the padded states (1.6 GB) or the observables of
    80 steps (1.6 GB) beside them do not."""
    vion, us, A = batch()
    nt = 2 if when == "create" else 80
    many = [us[t % 3] for t in range(NTRAJ)]
    field = np.array([A[t % 3, :nt] for t in range(NTRAJ)])
    args = (NG, NB, NB, ACELL, 0.004, [NK] * NTRAJ, np.array([vion] * NTRAJ))
    if when == "create":
        with free_memory(3 * GIB):
            B = T.Batch(*args)
            B.upload(many)
            e = B.propagate(field, field)[0]
    else:
        B = T.Batch(*args)
        B.upload(many)
        B.propagate(field[:, :1], field[:, :1])  # the states are padded now
        B.upload(B.download())
        with free_memory(int(1.2 * GIB)):
            e = B.propagate(field, field)[0]
    out = B.download()
    B.close()
    for t in range(3):
        with T.TDHF(NG, NK, NB, NB, ACELL, 0.004, vion) as G:
            u = us[t]
            if when == "propagate":
                u = G.RT_calculation(u, A[t, :1], A[t, :1])[0]
            u, e1 = G.RT_calculation(u, A[t, :nt], A[t, :nt])[:2]
        for k in (t, t + 3 * 2665):
            assert rel(out[k], u) < 1e-11 and rel(e[k], e1) < 1e-11


def used(call):
    """Bytes of device memory that call() leaves allocated."""
    hip = C.CDLL("libamdhip64.so")
    free, total = [C.c_size_t(), C.c_size_t()], C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free[0]), C.byref(total)) == 0
    call()
    assert hip.hipMemGetInfo(C.byref(free[1]), C.byref(total)) == 0
    return free[0].value - free[1].value


def test_observables_slots_of_row_wise_runs():
    """15 doubles a step at NG=128, NK=4, NB=1 (the other path's slots are of
    768): 24 MB and 56 MB of observables, with the reduced values and the field
    under 100 and 200 MB."""
    ng, nk, a, nt = 128, 4, 12.0, 200000
    vion = T.ion_potential(ng, nk, a, [6.0], [1.0], [0.0])
    field = np.zeros(nt)
    with T.TDHF(ng, nk, 1, 1, a, 0.004, vion) as G:
        G.upload(orbitals((ng, nk, 1, 1, a, 6.0), 1))
        assert used(lambda: G.rt_begin(field, field)) < 100e6
    ntraj, nt = 200, 2000
    with T.Batch(ng, 1, 1, a, 0.004, [nk] * ntraj, np.array([vion] * ntraj)) as B:
        B.upload([orbitals((ng, nk, 1, 1, a, 6.0), 1)] * ntraj)
        field = np.zeros((ntraj, nt))
        assert used(lambda: B.propagate(field, field)) < 200e6


def test_tables_of_a_batch():
    """Twelve k-meshes of NG=128: tables of 0.6 MB each beside the trajectories'
    states (four of 2 MB each) and matrices (34 MB), 510 MB in all; with states and
    matrices for runs of their own the tables alone would hold 970 MB more."""
    ng, nb, a, nks = 128, 8, 12.0, list(range(117, 129))
    vion = np.array([T.ion_potential(ng, k, a, [6.0], [1.0], [0.0]) for k in nks])
    B = []
    assert used(lambda: B.append(T.Batch(ng, nb, nb, a, 0.004, nks, vion))) < 700e6
    us = [orbitals((ng, k, nb, nb, a, 6.0), k) for k in nks]
    A = np.full((12, 2), 0.05)
    B[0].upload(us)
    e = B[0].propagate(A, A)[0]
    out = B[0].download()
    B[0].close()
    for t in (0, 11):
        with T.TDHF(ng, nks[t], nb, nb, a, 0.004, vion[t]) as G:
            u, e1 = G.RT_calculation(us[t], A[t], A[t])[:2]
        assert rel(out[t], u) < 1e-11 and rel(e[t], e1) < 1e-11
