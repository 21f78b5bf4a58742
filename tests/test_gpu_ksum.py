"""The batched k-sums at every matrix dimension: M = Gc^-1 - V(k) needs row exchanges (its
diagonal vanishes in places), the k points exceed one device chunk, and a singular Gc is
refused."""
import numpy as np
import pytest

from pyqcm_amd import lattice as LT

pytestmark = pytest.mark.gpu


def _inputs(n, nw, nk, nterm, seed):
    rng = np.random.default_rng(seed)
    # Gc^-1 with a zero diagonal: the first pivots are off the diagonal where V(k)_ii = 0 too
    gi = rng.standard_normal((nw, n, n)) + 1j * rng.standard_normal((nw, n, n))
    if n > 1:
        gi[:, np.arange(n), np.arange(n)] = 0.0
    nv = rng.integers(-2, 3, (nterm, 3)).astype(float)
    mats = rng.standard_normal((nterm, n, n)) + 1j * rng.standard_normal((nterm, n, n))
    if n > 1 and nterm:
        mats[:, np.arange(n // 2), np.arange(n // 2)] = 0.0
    return np.linalg.inv(gi), rng.standard_normal((n, n)) * (1 - np.eye(n) * (n > 1)), nv, mats, rng.random((nk, 3))


def _reference(G, V0, nv, mats, k):
    V = V0 + np.einsum("kt,tab->kab", np.exp(2j * np.pi * (k @ nv.T)), mats)
    M = np.linalg.inv(G)[:, None] - V[None]
    inv = np.linalg.inv(M)
    # the terms of M may cancel and a phase 2 pi k.n carries an absolute error of its own
    # size times eps, so that M is known to eps times the sum below; the inverse amplifies it
    # by |M^-1|, Gc^-1 (inverted on both sides) by the condition number of Gc
    norm = lambda a: np.linalg.norm(a, axis=(-2, -1))
    size = (norm(np.linalg.inv(G)) * np.linalg.cond(G)).max() + norm(V0) + \
        (norm(mats) * (1 + 2 * np.pi * np.abs(nv).sum(1))).sum()
    return inv, np.linalg.slogdet(G)[1] + np.linalg.slogdet(M)[1].mean(1), norm(inv).max() * size


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 16])
@pytest.mark.parametrize("nw,nk,nterm", [(1, 1, 0), (3, 17, 5), (9, 130, 40)])
def test_modes_at_every_dimension(gpu_lib, n, nw, nk, nterm):
    args = _inputs(n, nw, nk, nterm, 100 * n + nk)
    inv, sef, cond = _reference(*args)
    # backward-stable elimination on both sides: a few n eps times that amplification
    tol = 10 * n * np.finfo(float).eps * cond
    scale = np.abs(inv).max()
    np.testing.assert_allclose(LT.cpt_batch(*args, mode="full"), inv, rtol=0, atol=tol * scale)
    np.testing.assert_allclose(LT.cpt_batch(*args, mode="trace"), np.trace(inv, axis1=2, axis2=3), rtol=0,
                               atol=n * tol * scale)
    np.testing.assert_allclose(LT.cpt_batch(*args, mode="average"), inv.mean(1), rtol=0, atol=tol * scale)
    np.testing.assert_allclose(LT.sef_batch(*args), sef, rtol=0, atol=tol)


@pytest.mark.parametrize("n,nk", [(16, 65537), (12, 116509)])
def test_k_points_beyond_one_chunk(gpu_lib, n, nk):
    args = _inputs(n, 2, nk, 3, 5)
    inv, sef, cond = _reference(*args)
    tol = 10 * n * np.finfo(float).eps * cond
    np.testing.assert_allclose(LT.cpt_batch(*args, mode="average"), inv.mean(1), rtol=0, atol=tol * np.abs(inv).max())
    np.testing.assert_allclose(LT.cpt_batch(*args, mode="trace")[:, -5:], np.trace(inv, axis1=2, axis2=3)[:, -5:], rtol=0,
                               atol=n * tol * np.abs(inv).max())
    np.testing.assert_allclose(LT.sef_batch(*args), sef, rtol=0, atol=tol)


@pytest.mark.parametrize("n", [1, 3, 12])
def test_singular_cluster_green_function_is_refused(gpu_lib, n):
    G, V0, nv, mats, k = _inputs(n, 3, 4, 2, 7)
    G[1] = 0.0
    for call in (lambda: LT.cpt_batch(G, V0, nv, mats, k, mode="trace"), lambda: LT.sef_batch(G, V0, nv, mats, k)):
        with pytest.raises(gpu_lib.QEDError, match="singular at a requested frequency"):
            call()
