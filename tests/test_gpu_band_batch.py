"""The batched band Lanczos through the cluster instances that take it: the Green function
against the one-sector form (qed_band_lanczos) from the same start vectors; and, with deflated
start vectors and with more of them than one pass over a vector serves, the Green function
and its poles against exact diagonalization."""
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
    poles = qcm.qmatrix(8801)
    qcm.erase_model_instance(8801)
    return E0, G, poles


def _exact_green(m, vals, n, nup, ndn, zs):
    """E0, the gap and G of the spin-up orbitals from the oracle's dense sectors"""
    def dense(nu):
        S = O.Sector(m, vals, nu, ndn)
        return np.stack([S.hv(c) for c in np.eye(S.dim)], 1)
    e, U = np.linalg.eigh(dense(nup))
    G = np.zeros((len(zs), n, n), complex)
    for pm in (1, -1):
        ep, Up = np.linalg.eigh(dense(nup + pm))
        Q = np.array([O.create_destroy(n, nup, ndn, a, pm, U[:, 0]) for a in range(n)]) @ Up
        G += _lehmann(pm * (ep - e[0]), Q, zs)
    return e[0], e[1] - e[0], G


@pytest.mark.parametrize("n,nup,ndn", [(6, 3, 3), (7, 3, 3), (8, 4, 4)])
def test_instance_green_function_matches_one_sector_form(gpu_lib, n, nup, ndn):
    """G of a cluster (8 vectors at most: one pass; the 8-site instance is batched) against
    c and c+ applied to the ground state and one band Lanczos per part"""
    from pyqcm_amd._lib import DeviceArray
    from pyqcm_amd.sector import Sector, apply_c
    m, vals = TM.chain(n, tp=-0.3, U=4.0, mu=1.7)
    zs = 1j * np.array([0.3, 1.0, 3.0, 10.0])
    E0, G, _ = _instance_green(m, vals, "R0:N%d:S%d" % (nup + ndn, nup - ndn), zs, "band_batch_%d" % n)
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


def test_start_vectors_that_deflate(gpu_lib):
    """A chain of 6 and a decoupled, doubly occupied orbital (a non-degenerate ground state):
    c of that orbital makes an eigenvector of H, whose successor vanishes (a deflated vector,
    kept for the later steps), and c+ makes nothing (a deflated start vector)."""
    zs = np.array([0.4 + 0.3j, -1.0 + 0.5j, 1j, 3j])
    m, vals = O.hubbard_cluster(7, [(i, i + 1) for i in range(5)], tp_bonds=[(i, i + 2) for i in range(4)],
                                U=4.0, mu=1.7, tp=-0.3)
    m.add("deep", "one-body", [(6, 6, 1.0), (13, 13, 1.0)])
    vals["deep"] = -8.0
    E0, G, (e, Q) = _instance_green(m, vals, "R0:N8:S0", zs, "band_defl")
    e0, gap, ref = _exact_green(m, vals, 7, 4, 4, zs)
    assert gap > 0.1 and abs(E0 - e0) <= 1e-10 * abs(e0)
    np.testing.assert_allclose(G, ref, rtol=0, atol=1e-7)  # as above
    # the decoupled orbital: one pole at mu' + U below the ground state, of weight 1, and
    # nothing of it in any other (a vector that was not deflated would spread over them)
    own = np.abs(Q[:, 6]) > 1e-6
    assert own.sum() == 1
    np.testing.assert_allclose(e[own], vals["deep"] - vals["mu"] + vals["U"], rtol=0, atol=1e-9)
    np.testing.assert_allclose(np.abs(Q[own]), np.eye(7)[6:], rtol=0, atol=1e-7)


def test_deflated_vector_that_overlaps_later_ones(gpu_lib):
    """The same orbital coupled by 0.03 and a deflation threshold of 0.05: the deflated vector
    has overlaps with every later one, which enter the projected matrix. Against the oracle's
    recurrence with that threshold: its G moves by 5e-10 with perturbations of 1e-13, and by
    1.1e-7 to 2.5e-7 without the overlaps, their transpose or their subtraction."""
    from pyqcm_amd import qcm
    zs = 1j * np.array([0.5, 1.0, 3.0])
    m, vals = O.hubbard_cluster(7, [(i, i + 1) for i in range(5)], tp_bonds=[(i, i + 2) for i in range(4)],
                                U=4.0, mu=1.7, tp=-0.3)
    m.add("deep", "one-body", [(6, 6, 1.0), (13, 13, 1.0)])
    m.add("weak", "one-body", [(0, 6, 1.0), (7, 13, 1.0)])
    vals.update(deep=-8.0, weak=0.03)
    qcm.set_global_parameter("accur_deflation", 0.05)
    try:
        E0, G, _ = _instance_green(m, vals, "R0:N8:S0", zs, "band_overlap")
    finally:
        qcm.set_global_parameter("accur_deflation", 1e-7)
    e0, psi, *_ = O.Sector(m, vals, 4, 4).lanczos_gs()
    ref = np.zeros_like(G)
    for pm in (1, -1):
        T = O.Sector(m, vals, 4 + pm, 4)
        e, Q = O.band_lanczos(T.hv, [O.create_destroy(7, 4, 4, a, pm, psi) for a in range(7)], accur_deflation=0.05)
        ref += _lehmann(pm * (e - e0), Q, zs)
    assert abs(E0 - e0) <= 1e-10 * abs(e0)
    np.testing.assert_allclose(G, ref, rtol=0, atol=2e-8)


def test_more_start_vectors_than_one_pass_serves(gpu_lib):
    """12 orbitals, 2 electrons: the norm, 12 start-vector and 11 pending-block overlaps take
    two descriptors (1 + 12 + 11 > 20). The particle part (792 states) is the batched one; the
    hole part (12 states) is diagonalized."""
    zs = 1j * np.array([1.0, 3.0, 10.0])
    m, vals = TM.chain(12, U=4.0, mu=2.0, tp=-0.3)
    E0, G, (e, Q) = _instance_green(m, vals, "R0:N2:S0", zs, "band_many")
    e0, gap, ref = _exact_green(m, vals, 12, 1, 1, zs)
    assert gap > 0.01 and abs(E0 - e0) <= 1e-10 * abs(e0)
    # the recurrence stops by its lowest value, with G converged to 2e-8 at i and 1e-15 at 3 i
    np.testing.assert_allclose(G, ref, rtol=0, atol=1e-7)
    np.testing.assert_allclose(Q.T @ Q, np.eye(12), rtol=0, atol=1e-7)


@pytest.mark.parametrize("n,nup,ndn", [(9, 5, 4), (10, 5, 5), (11, 5, 5)])
def test_few_and_many_chunks(gpu_lib, n, nup, ndn):
    """Sums over few chunks (14 and 52 of 2048 amplitudes in the two parts: vectors split over
    blocks) and over many (180: one block per chunk), against the one-sector form as above"""
    test_instance_green_function_matches_one_sector_form(gpu_lib, n, nup, ndn)
