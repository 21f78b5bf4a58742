"""The batched band Lanczos against the one-sector form (qed_band_lanczos): the same
Lehmann form from the same start vectors, with deflated start vectors, with more start
vectors than one pass over a vector serves, and through a cluster instance that takes it."""
import numpy as np
import pytest

from oracle import oracle as O
from tests import models as TM

pytestmark = pytest.mark.gpu


def _lehmann(e, Q, zs):
    return np.einsum("am,zm,bm->zab", Q, 1.0 / (zs[:, None] - e[None]), Q)


def _instance_green(model, vals, sector, zs, name):
    from pyqcm_amd import qcm
    qcm.new_model(name, model.n_sites if hasattr(model, "n_sites") else model.L, 0)
    for nm, op in model.operators.items():
        qcm.new_operator(name, nm, op.kind, [(r + 1, c + 1, v) for r, c, v in op.elements])
    qcm.new_model_instanceC(name, vals, sector, 8801)
    E0, _ = qcm.ground_state_solve(8801)
    G = qcm.Green_function(zs, 0, 8801)
    qcm.erase_model_instance(8801)
    return E0, G


@pytest.mark.parametrize("n,nup,ndn", [(6, 3, 3), (7, 3, 3), (8, 4, 4)])
def test_instance_green_function_matches_one_sector_form(gpu_lib, n, nup, ndn):
    """G of a cluster (8 vectors at most: one pass; the 8-site instance is batched) against
    c and c+ applied to the ground state and one band Lanczos per part"""
    from pyqcm_amd._lib import DeviceArray
    from pyqcm_amd.sector import Sector, apply_c
    m, vals = TM.chain(n, tp=-0.3, U=4.0, mu=1.7)
    zs = 1j * np.array([0.3, 1.0, 3.0, 10.0])
    E0, G = _instance_green(m, vals, "R0:N%d:S%d" % (nup + ndn, nup - ndn), zs, "band_batch_%d" % n)
    S = Sector(n, nup, ndn, m.flat(vals))
    e0, psi, *_ = S.lanczos_gs()
    assert abs(E0 - e0) <= 1e-10 * abs(e0)
    ref = np.zeros_like(G)
    for pm in (1, -1):
        T = Sector(n, nup + pm, ndn, m.flat(vals))
        phi = DeviceArray(n * T.dim).zeros()
        for a in range(n):
            class V:  # a view of one start vector
                ptr = phi.offset(a * T.dim)
            apply_c(n, nup, ndn, a, pm, psi, V)
        e, Q = T.band_lanczos(phi, n, M0=int(14 * n * np.log(T.dim)))
        ref += _lehmann(pm * (e - e0), Q, zs)
    # both stop where the lowest Ritz value is stationary to 1e-12; G has converged there to
    # about the square root of the residual weight, 1e-8 at these frequencies
    np.testing.assert_allclose(G, ref, rtol=0, atol=1e-7)


def test_start_vectors_that_deflate_and_many_of_them(gpu_lib):
    """A decoupled orbital makes start vectors eigenvectors (deflation); 12 orbitals need a
    second pass for the pending block (1 + 12 + 11 vectors)."""
    from pyqcm_amd import qcm
    zs = 1j * np.array([0.5, 2.0, 8.0])
    # two decoupled chains of 3: the Green function is block diagonal and its blocks equal
    bonds = [(0, 1), (1, 2), (3, 4), (4, 5)]
    m, vals = O.hubbard_cluster(6, bonds, U=4.0, mu=2.1)
    E0, G = _instance_green(m, vals, "R0:N6:S0", zs, "band_defl")
    assert np.abs(G[:, :3, 3:]).max() <= 1e-8
    # the sum rule Q Q^T = 1 (G ~ 1/z) through the 12-orbital instance, 12 start vectors
    m, vals = TM.chain(12, U=4.0, mu=2.0)
    big = 1j * np.array([1e4])
    E0, G = _instance_green(m, vals, "R0:N2:S0", big, "band_many")
    np.testing.assert_allclose(G[0] * big[0], np.eye(12), rtol=0, atol=1e-3)


@pytest.mark.parametrize("n,nup,ndn", [(9, 5, 4), (10, 5, 5), (11, 5, 5)])
def test_few_and_many_chunks(gpu_lib, n, nup, ndn):
    """Sums over few chunks (14 and 52 of 2048 amplitudes in the two parts: vectors split over
    blocks) and over many (180: one block per chunk), against the one-sector form as above"""
    test_instance_green_function_matches_one_sector_form(gpu_lib, n, nup, ndn)
