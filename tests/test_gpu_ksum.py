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


def _gauss_jordan(M, real):
    """Inverses of a batch of matrices by Gauss-Jordan with partial pivoting, in real
    arithmetic of type `real` without fused multiply-adds."""
    B, n = M.shape[:2]
    re = np.concatenate([M.real.astype(real), np.broadcast_to(np.eye(n, dtype=real), M.shape)], 2)
    im = np.concatenate([M.imag.astype(real), np.zeros(M.shape, real)], 2)
    r = np.arange(B)
    for k in range(n):
        p = k + (re[:, k:, k] ** 2 + im[:, k:, k] ** 2).argmax(1)
        for a in (re, im):
            a[r, k], a[r, p] = a[r, p].copy(), a[r, k].copy()
        c, s = re[:, k, k][:, None], im[:, k, k][:, None]
        d = c * c + s * s
        c, s = c / d, -s / d
        re[:, k], im[:, k] = re[:, k] * c - im[:, k] * s, re[:, k] * s + im[:, k] * c
        fr, fi = re[:, :, k].copy()[:, :, None], im[:, :, k].copy()[:, :, None]
        fr[:, k] = fi[:, k] = 0.0
        pr, pi = re[:, None, k], im[:, None, k]
        re, im = re - (fr * pr - fi * pi), im - (fr * pi + fi * pr)
    return re[:, :, n:] + 1j * im[:, :, n:]


@pytest.mark.parametrize("n", [2, 4, 8, 12, 16])
def test_rounding_error_of_the_inverse(gpu_lib, n):
    """Geometric mean over 4096 matrices, known exactly, of the relative error of their
    inverses. In 64 bits the same elimination without fused multiply-adds rounds each product
    once more than the device, whose error is 0.91 to 0.93 of that one's; with two products
    added to the accumulator in turn, two roundings of its size, it is 1.02 to 1.04 of it.
    (The mean of 4096 logarithms is good to 1%.)"""
    rng = np.random.default_rng(n)
    k = np.stack(np.meshgrid(*[np.arange(4) / 4.0] * 3), -1).reshape(64, 3)  # phases 1, i, -1, -i
    nv = np.concatenate([np.eye(3), np.eye(3)[[1, 2, 0]] + np.eye(3)])
    exact = lambda *s: (rng.integers(-2**22, 2**22, s) + 1j * rng.integers(-2**22, 2**22, s)) / 2.0**20
    log_dev, log_ref = [], []
    for _ in range(64):
        V0, mats = exact(n, n), exact(6, n, n)
        ph = np.round(np.exp(2j * np.pi * (k @ nv.T)))
        M = np.eye(n) - (V0 + np.einsum("kt,tab->kab", ph, mats))
        dev = LT.cpt_batch(np.eye(n, dtype=complex)[None], V0, nv, mats, k, mode="full")[0]
        inv = _gauss_jordan(M, np.longdouble)
        norm = lambda a: np.sqrt((np.abs(a) ** 2).sum((1, 2)))
        log_dev.append(np.log(norm(dev - inv) / norm(inv)))
        log_ref.append(np.log(norm(_gauss_jordan(M, np.float64) - inv) / norm(inv)))
    ratio = float(np.exp(np.mean(log_dev) - np.mean(log_ref)))
    print("n = %d: error %.3e, %.3f of the unfused form's" % (n, np.exp(np.mean(log_dev)), ratio), flush=True)
    assert ratio <= 0.98


@pytest.mark.parametrize("n", [3, 8, 13])
def test_cluster_green_function_beyond_the_range_of_a_square(gpu_lib, n):
    """One orbital of Gc so small or so large that the square of its pivot leaves the range of
    a double: it drops out of the lattice Green function, and its logarithm stays finite."""
    _, V0, nv, mats, k = _inputs(n, 2, 3, 2, 11)
    rng = np.random.default_rng(n)
    G = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
    V = V0 + np.einsum("kt,tab->kab", np.exp(2j * np.pi * (k @ nv.T)), mats)
    Gc = G.copy()
    Gc[:, 0] = Gc[:, :, 0] = 0.0
    Gc[:, 0, 0] = 1e-160 * (1 + 1j)
    inv = np.linalg.inv(np.linalg.inv(Gc[:, 1:, 1:])[:, None] - V[:, 1:, 1:])
    dev = LT.cpt_batch(Gc, V0, nv, mats, k, mode="full")
    np.testing.assert_allclose(dev[:, :, 1:, 1:], inv, rtol=0, atol=1e-10 * np.abs(inv).max())
    assert np.abs(dev[:, :, 0]).max() < 1e-100 and np.abs(dev[:, :, :, 0]).max() < 1e-100
    Gc[:, 0, 0] = 1e160 * (1 + 1j)
    ref = np.linalg.slogdet(V[None] @ Gc[:, None] - np.eye(n))[1].mean(1)
    np.testing.assert_allclose(LT.sef_batch(Gc, V0, nv, mats, k), ref, rtol=1e-12)
