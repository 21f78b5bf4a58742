"""The chunked Lanczos ground state on every kind of sector and kernel it takes: values,
vector and step count against the plain recurrence in numpy, the iteration limit at and
around a chunk's end, and Krylov spaces that are exhausted inside the first chunk."""
import numpy as np
import pytest

from tests import models as TM

pytestmark = pytest.mark.gpu


def _plain(hv, x, accur, max_iter):
    """alpha, beta of the textbook recurrence up to the first step with |beta e_last| <= accur"""
    a, b = [], []
    r, q = x.copy(), np.zeros_like(x)
    while True:
        if b:
            r, q = r / b[-1], -b[-1] * q
        q = q + hv(r)
        r, q = q, r
        a.append(q @ r)
        r = r - a[-1] * q
        b.append(np.linalg.norm(r))
        T = np.diag(a) + np.diag(b[:-1], 1) + np.diag(b[:-1], -1)
        e, u = np.linalg.eigh(T)
        if abs(u[-1, 0] * b[-1]) <= accur or len(a) > max_iter:
            return np.array(a), np.array(b), e[0]


def _sectors():
    from pyqcm_amd.sector import GeneralSector, MixedSector, Sector
    m, v = TM.square(2, 3, tp=-0.3)
    yield "factorized 6 sites", Sector(6, 3, 3, m.flat(v)), 1e-12
    yield "factorized one state", Sector(6, 6, 0, m.flat(v)), 1e-12
    yield "factorized six states", Sector(6, 1, 6, m.flat(v)), 1e-12
    yield "mirror basis", MixedSector(6, 3, 3, m.flat(v), 6, [[1, 0, 3, 2, 5, 4]], 0), 1e-12
    m, v = TM.chain(13, U=4.0, mu=2.0)
    yield "odd rows", Sector(13, 6, 1, m.flat(v)), 1e-11
    m, v = TM.square(4, 4, tp=-0.3)
    yield "long rows", Sector(16, 8, 1, m.flat(v)), 1e-11
    m, v = TM.square(2, 2, tp=-0.3)
    m.add("hx", "one-body", [(i, i + 4, 1.0) for i in range(4)])
    v["hx"] = 0.4
    yield "spin flip", GeneralSector(4, [(nu, 4 - nu) for nu in range(5)], m.flat(v)), 1e-12


def test_steps_values_and_vector(gpu_lib):
    rng = np.random.default_rng(3)
    for name, S, accur in _sectors():
        x = rng.standard_normal(S.dim)
        x /= np.linalg.norm(x)
        E0, psi, n, a, b = S.lanczos_gs(start=x, accur=accur)
        pa, pb, pe = _plain(S.hv, x, accur, 1000)
        psi = psi.to_host()
        print(name, S.dim, n, len(pa), E0, flush=True)
        # the last steps of a small space follow a vanishing beta, where the stopping test
        # sits at round-off: one step either way
        assert abs(n - len(pa)) <= 1
        assert abs(E0 - pe) <= 1e-11 * max(1.0, abs(pe))
        k = max(1, min(n, len(pa)) // 2)  # before orthogonality is lost
        np.testing.assert_allclose(a[:k], pa[:k], rtol=0, atol=1e-9 * max(1.0, np.abs(pa).max()))
        # |H psi - E0 psi| = |beta e_last| <= accur and the rounding of psi
        assert np.linalg.norm(S.hv(psi) - E0 * psi) <= 1e-9 * max(1.0, abs(E0))
        assert abs(np.linalg.norm(psi) - 1.0) <= 1e-9
        S.close()


@pytest.mark.parametrize("size", [(2, 4), (3, 3)])
def test_iteration_limit(gpu_lib, size):
    from pyqcm_amd.sector import Sector
    m, v = TM.square(*size, tp=-0.3)
    L = m.L
    S = Sector(L, L // 2, L // 2, m.flat(v))
    x = np.random.default_rng(1).standard_normal(S.dim)
    x /= np.linalg.norm(x)
    E0, _, n, a, b = S.lanczos_gs(start=x)
    E1, _, n1, a1, b1 = S.lanczos_gs(start=x, max_iter=n)  # just enough
    assert (E0, n) == (E1, n1)
    np.testing.assert_array_equal(a, a1)
    for limit in (0, 1, 7, 8, 9, 15, 16, 17, n - 1):
        with pytest.raises(gpu_lib.QEDError, match="exceeded %d iterations" % limit):
            S.lanczos_gs(start=x, max_iter=limit)
    S.close()


def test_largest_iteration_limit(gpu_lib):
    """No limit to speak of (INT_MAX): the same run as with the default one."""
    from pyqcm_amd._lib import DeviceArray
    from pyqcm_amd.sector import Sector
    m, v = TM.square(2, 4, tp=-0.3)
    S = Sector(8, 4, 4, m.flat(v))
    x = np.random.default_rng(2).standard_normal(S.dim)
    x /= np.linalg.norm(x)
    E0, psi, n, _, _ = S.lanczos_gs(start=x)
    y, E1, n1 = DeviceArray.from_host(x), np.zeros(1), np.zeros(1, np.int32)
    gpu_lib.call("qed_lanczos_gs", S.h, 1e-12, 2**31 - 1, y.ptr, gpu_lib.dp(E1), gpu_lib.ip(n1), None, None)
    assert (E1[0], n1[0]) == (E0, n)
    np.testing.assert_array_equal(y.to_host(), psi.to_host())


def test_vector_aligned_to_eight_bytes(gpu_lib):
    """A start vector behind one double of another buffer, on the two-column kernel of long
    rows: the same numbers as from an aligned one, and nothing written around it."""
    from pyqcm_amd._lib import DeviceArray
    from pyqcm_amd.sector import Sector
    m, v = TM.square(4, 4, tp=-0.3)
    S = Sector(16, 8, 1, m.flat(v))
    x = np.random.default_rng(6).standard_normal(S.dim)
    x /= np.linalg.norm(x)
    out = []
    for shift in (0, 1):
        buf = DeviceArray.from_host(np.concatenate([np.full(shift, 7.0), x, [9.0]]))
        E0, nit = np.zeros(1), np.zeros(1, np.int32)
        gpu_lib.call("qed_lanczos_gs", S.h, 1e-12, 400, buf.offset(shift), gpu_lib.dp(E0), gpu_lib.ip(nit), None, None)
        h = buf.to_host()
        assert h[-1] == 9.0 and (shift == 0 or h[0] == 7.0)
        out.append((float(E0[0]), int(nit[0]), h[shift:-1]))
    assert out[0][:2] == out[1][:2]
    np.testing.assert_array_equal(out[0][2], out[1][2])


def test_more_long_rows_than_folded_parts(gpu_lib):
    """19 sites, 5 up and 8 down: 75,582 rows of 11,628 (more than 2^16 parts of a scalar
    product) take the kernel of long rows. A step's alpha and beta against the product and dot
    products of the plain recurrence, and less time than that of its separate passes."""
    from pyqcm_amd._lib import DeviceArray
    from pyqcm_amd.sector import Sector
    m, v = TM.chain(19, U=4.0, mu=2.0)
    S = Sector(19, 5, 8, m.flat(v))
    assert S.dd > 1 << 16 and S.du >= 4096 and S.du % 2 == 0
    x = DeviceArray(S.dim)
    gpu_lib.call("qed_start_vector", S.h, 1, x.ptr)
    ms = np.zeros(2)
    gpu_lib.call("qed_lanczos_steps_timed", S.h, x.ptr, 3, gpu_lib.dp(ms))
    assert ms[0] < ms[1]
    h = x.to_host()
    w = S.hv(h)
    a0 = float(h @ w)
    w -= a0 * h
    b0 = float(np.linalg.norm(w))
    E0, nit = np.zeros(1), np.zeros(1, np.int32)
    alpha, beta = np.zeros(2), np.zeros(2)
    # any first Ritz value passes this limit: one step
    gpu_lib.call("qed_lanczos_gs", S.h, 1e6, 1, x.ptr, gpu_lib.dp(E0), gpu_lib.ip(nit), gpu_lib.dp(alpha), gpu_lib.dp(beta))
    assert nit[0] == 1
    np.testing.assert_allclose([alpha[0], beta[0]], [a0, b0], rtol=1e-11)
    x.free()
    S.close()
