"""Which kernels a call runs, as the handle reports it, and the results of either
choice against the oracle: whole-recursion or step kernels for small lattices."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import fermi_coeffs, rel_err

pytestmark = pytest.mark.gpu

FP64_TOL = 1e-10


def _engine(dtype="cx_double", prec="fp64"):
    from fastkpm_amd import HipEngine
    return HipEngine(dtype, prec)


def _set_up(oracle, H, S, seed=1, real=False, prec="fp64", dense=True):
    """Engine and oracle with H, scaled by its row sums, and S random columns
    (dense, or one nonzero per orbital row)."""
    from fastkpm_amd import EnergyScale
    rng = np.random.default_rng(seed)
    n, b = H.n_rows * H.b_len, H.b_len
    R = rng.standard_normal((n, S)) + (0 if real else 1j) * rng.standard_normal((n, S))
    if not dense:
        keep = np.zeros((n, S))
        keep[np.arange(n), rng.integers(0, S, n)] = 1.0
        R = R * keep
    absrow = np.zeros((H.n_rows, b))
    np.add.at(absrow, H.row_idx, np.abs(H.val.reshape(-1, b, b)).sum(axis=1))
    bound = float(absrow.max())
    eng = _engine("double" if real else "cx_double", prec)
    eng.set_R(R)
    eng.set_H(H, EnergyScale(-bound, bound))
    orc = oracle.Engine()
    orc.set_H(H, -bound, bound)
    orc.set_R(R)
    return eng, orc, bound


@pytest.mark.parametrize("whole", [True, False])
def test_timing_counts_the_launches_of_either_path(oracle, whole):
    """fkpm_get_timing: one launch per recursion (and one for the table sums) with
    the whole-recursion kernels, one per Chebyshev step with the step kernels."""
    from fastkpm_amd import lattice
    eng, _, bound = _set_up(oracle, lattice.lattice((8, 8), b=2, seed=3, J=1.0), 4)
    if not whole:
        eng.set_store_alpha(2)  # names the step kernels' table
    eng.set_timing(True)
    M = 40
    c = fermi_coeffs(oracle, M, -bound, bound)
    D = lattice.lattice((8, 8), b=2, seed=3, J=1.0)
    eng.moments(M)
    assert eng.whole_recursion() is whole
    assert eng.alpha_table() is (not whole)
    eng.autodiff_matrix(c, D)
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "table"
    eng.set_stoch_method("clenshaw")
    t = eng.timing()
    eng.stoch_matrix(c, D)
    assert t["moments_launches"] == (1 if whole else M // 2)
    assert t["autodiff_launches"] == (1 if whole else M // 2 - 1)
    assert t["stoch_launches"] == (2 if whole else M // 2 + 1)
    assert eng.timing()["stoch_launches"] == (1 if whole else M - 1)
    eng.moments(2)
    eng.autodiff_matrix(c[:2], D)
    assert eng.timing()["moments_launches"] == 1 and eng.timing()["autodiff_launches"] == 0
    eng.close()


def _pattern(nb, b, reach=0, hub=0, real=False, seed=5):
    """Random Hermitian blocks on a periodic chain of nb sites: neighbours up to
    `reach` away and, for site 0, `hub` more (the rows then have uneven lengths)."""
    from fastkpm_amd import lattice
    rng = np.random.default_rng(seed)
    i = np.arange(nb)
    pairs = [np.stack([i, (i + d) % nb]) for d in range(1, reach + 1)]
    if hub:
        pairs.append(np.stack([np.zeros(hub, dtype=int),
                               np.sort(rng.choice(np.arange(reach + 1, nb - reach), hub, False))]))
    r, c = np.concatenate(pairs, axis=1)
    T = rng.standard_normal((len(r), b, b)) + (0 if real else 1j) * rng.standard_normal((len(r), b, b))
    X = rng.standard_normal((nb, b, b)) + (0 if real else 1j) * rng.standard_normal((nb, b, b))
    X = X + np.conj(X.transpose(0, 2, 1))
    return lattice.coo_to_bsr(nb, b, np.concatenate([i, r, c]), np.concatenate([i, c, r]),
                              np.concatenate([X, T, np.conj(T.transpose(0, 2, 1))]),
                              np.float64 if real else np.complex128)


def _check_all(oracle, eng, orc, H, M, bound, tol=FP64_TOL):
    """moments, autodiff_matrix and stoch_matrix (from the kept vectors, and by the
    recurrence) against the oracle."""
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.05)
    D = H.like(eng.np_dtype)
    assert rel_err(eng.moments(M), orc.moments(M)) < tol
    eng.autodiff_matrix(c, D)
    assert rel_err(D.val, orc.autodiff_matrix(c, H)) < tol
    s = orc.stoch_matrix(c, H)
    eng.stoch_matrix(c, D)
    assert rel_err(D.val, s) < tol
    eng.set_stoch_method("clenshaw")
    eng.stoch_matrix(c, D)
    assert rel_err(D.val, s) < tol
    eng.set_stoch_method("auto")


# (rows, block size, reach, hub bonds, real, whole recursion): either side of the
# loads a thread may stream, rows padded to a hub's length among them
@pytest.mark.parametrize("nb,b,reach,hub,real,whole", [
    (2000, 1, 9, 0, False, True), (2000, 1, 2, 16, False, False),
    (3000, 1, 4, 0, False, True), (3000, 1, 6, 0, False, False), (3000, 1, 2, 10, False, False),
    (3000, 1, 13, 0, True, False), (1000, 1, 2, 40, False, True),
    (1500, 2, 3, 0, False, True), (1500, 2, 4, 0, False, False), (1000, 2, 2, 12, False, True),
    (1100, 2, 2, 10, False, False), (500, 4, 3, 0, False, True), (600, 4, 2, 0, False, False)])
def test_rows_too_long_for_the_whole_recursion(oracle, nb, b, reach, hub, real, whole):
    H = _pattern(nb, b, reach, hub, real)
    eng, orc, bound = _set_up(oracle, H, 3, real=real)
    _check_all(oracle, eng, orc, H, 12, bound)
    eng.moments(2)
    assert eng.whole_recursion() is whole
    eng.close()


# (lattice, block size, columns, real, M, backward recursion as one launch): either
# side of the streamed blocks and the order at which autodiff_matrix goes to the step
# kernels
@pytest.mark.parametrize("shape,b,S,real,M,whole", [
    ((50, 50), 1, 3, False, 24, True), ((57, 57), 1, 3, False, 24, False),
    ((57, 57), 1, 3, False, 22, True), ((64, 64), 1, 1, False, 24, False),
    ((64, 64), 1, 33, False, 26, False), ((14, 14, 14), 1, 17, False, 30, False),
    ((64, 64), 1, 5, True, 24, True), ((40, 40), 2, 3, False, 96, True),
    ((11, 11, 11), 2, 5, False, 96, True), ((12, 12, 12), 2, 31, False, 96, False),
    ((12, 12, 12), 2, 3, False, 94, True), ((12, 12, 12), 2, 2, False, 2, True)])
@pytest.mark.parametrize("own_pattern", [True, False])
def test_backward_recursion_of_streamed_lattices(oracle, shape, b, S, real, M, whole, own_pattern):
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=b, seed=7, W=1.0, J=0.0 if b == 1 else 1.0,
                        dtype=np.float64 if real else np.complex128)
    eng, orc, bound = _set_up(oracle, H, S, real=real)
    eng.set_timing(True)
    nb = H.n_rows
    Dp = H if own_pattern else lattice.coo_to_bsr(nb, b, range(nb), range(nb), np.zeros((nb, b, b)))
    D = Dp.like(eng.np_dtype)
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.05)
    mu_o = orc.moments(M)
    d_o = orc.autodiff_matrix(c, Dp)
    for _ in range(3):  # the step loop is captured, then replayed
        assert rel_err(eng.moments(M), mu_o) < FP64_TOL
        assert eng.whole_recursion()
        eng.autodiff_matrix(c, D)
        assert eng.timing()["autodiff_launches"] == (0 if M == 2 else 1 if whole else M // 2 - 1)
        assert rel_err(D.val, d_o) < FP64_TOL
    # the resident table is still whole
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "table"
    assert rel_err(D.val, orc.stoch_matrix(c, Dp)) < FP64_TOL
    eng.close()


# (lattice, block size, columns, precision, one launch): either side of the streamed
# blocks, the vector size and the order at which the Clenshaw recurrence goes to the
# step kernels
@pytest.mark.parametrize("shape,b,S,prec,whole", [
    ((64, 64), 1, 3, "fp64", True), ((13, 13, 13), 1, 3, "fp64", False),
    ((13, 13, 13), 1, 64, "fp64", True), ((45, 42), 2, 5, "fp64", True),
    ((12, 12, 12), 2, 5, "fp64", False), ((12, 12, 12), 2, 5, "fp32", True),
    ((8, 8, 8), 4, 2, "fp64", True)])
@pytest.mark.parametrize("dense", [True, False])
def test_clenshaw_of_streamed_lattices(oracle, shape, b, S, prec, whole, dense):
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=b, seed=9, W=1.0, J=1.0 if b == 2 else 0.0, orbital_blocks=b > 2)
    eng, orc, bound = _set_up(oracle, H, S, prec=prec, dense=dense)
    eng.set_timing(True)
    M = 17
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.05, kind=1)
    D = H.like()
    # FP32: M recursion steps of 16 roundings each
    tol = FP64_TOL if prec == "fp64" else M * 16 * 2.0 ** -24
    for m in (M, 15, 2):
        s = orc.stoch_matrix(c[:m], H)
        for _ in range(3):
            eng.stoch_matrix(c[:m], D)
            assert eng.stoch_method() == "clenshaw"
            assert eng.timing()["stoch_launches"] == (1 if whole or m < 16 else m - 1)
            assert rel_err(D.val, s) < tol
    assert eng.state()["r_compact"] is (not dense)
    # a table of the same R and H is used by the whole-recursion kernels on either side
    eng.moments(M + 1)
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "table" and eng.timing()["stoch_launches"] == 2
    assert rel_err(D.val, orc.stoch_matrix(c, H)) < tol
    eng.close()


def test_moments_alone_holds_one_table(oracle):
    """The table of backward vectors is autodiff_matrix's: moments allocates only the
    forward one (M/2 + 1 vectors), autodiff_matrix as much again."""
    import ctypes
    import gc
    from fastkpm_amd import _capi, lattice

    def free():  # of the runtime that the library itself is linked to
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert _capi.lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    H = lattice.lattice((16, 16), b=2, seed=3, J=1.0)
    S, M = 256, 512
    eng, _, bound = _set_up(oracle, H, S)
    table = (M // 2 + 1) * H.n_rows * 2 * S * 16  # 539 MB
    eng.moments(2)
    gc.collect()  # engines of earlier tests give their memory back now, not below
    used = [free()]
    eng.moments(M)
    assert eng.whole_recursion()
    used.append(free())
    eng.autodiff_matrix(fermi_coeffs(oracle, M, -bound, bound), H.like())
    used.append(free())
    assert 0.9 * table < used[0] - used[1] < 1.5 * table
    assert 0.9 * table < used[1] - used[2] < 1.5 * table
    eng.close()


def test_large_D_into_pinned_memory():
    """A D of 57 MB into pinned and into pageable memory: the same bits, and the pinned
    copy (one transfer at the link's rate, 0.65 of the time) not through the staging
    ring of the pageable one (the same time)."""
    import ctypes
    import time
    from fastkpm_amd import EnergyScale, _capi, lattice
    H = lattice.lattice((20, 20, 20), b=8, seed=3, orbital_blocks=True)
    eng = _engine()
    eng.set_R(np.ones((H.n_rows * 8, 1), dtype=np.complex128))
    eng.set_H(H, EnergyScale(-60.0, 60.0))
    D = H.like()
    eng.stoch_matrix([0.5, 0.25, 0.125], D)
    want = D.val.copy()

    def best():
        t = []
        for _ in range(20):
            t0 = time.perf_counter()
            eng.get_D(D)
            t.append(time.perf_counter() - t0)
        return min(t)

    t_pageable = best()
    p = ctypes.c_void_p()
    assert _capi.lib().hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(want.nbytes), 0) == 0
    D.val = np.frombuffer((ctypes.c_char * want.nbytes).from_address(p.value), dtype=np.complex128)
    D.val[:] = 0
    eng.get_D(D)
    assert np.array_equal(D.val, want)
    t_pinned = best()
    D.val = None
    eng.close()
    _capi.lib().hipHostFree(p)
    assert t_pinned < 0.95 * t_pageable, (t_pinned, t_pageable)


@pytest.mark.parametrize("shape,b,prec", [((48, 45), 2, "fp64"), ((70, 61), 1, "fp32"),
                                          ((6, 6, 6), 8, "fp64")])
def test_moments_in_a_row_keep_no_table(oracle, shape, b, prec):
    """From the third moments on that nothing followed the ring is used (not with the
    matrix-core steps): the same bits, and autodiff_matrix and stoch_matrix as before;
    either of them brings the table back."""
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=b, seed=5, W=1.0, J=1.0 if b == 2 else 0.0, orbital_blocks=b > 2)
    eng, orc, bound = _set_up(oracle, H, 5, prec=prec)
    M = 20
    tol = FP64_TOL if prec == "fp64" else M * 16 * 2.0 ** -24
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.05)
    D = H.like()
    mu_o = orc.moments(M)
    d_o, s_o = orc.autodiff_matrix(c, H), orc.stoch_matrix(c, H)
    for follow in ("autodiff_matrix", "stoch_matrix"):
        mu = [eng.moments(M)]
        for kept in (True, False, False):
            mu.append(eng.moments(M))
            assert eng.alpha_table() is (kept or b == 8)
            assert np.array_equal(mu[-1], mu[0])
        assert rel_err(mu[0], mu_o) < tol
        getattr(eng, follow)(c, D)
        assert rel_err(D.val, d_o if follow == "autodiff_matrix" else s_o) < tol
        for name, want in (("autodiff_matrix", d_o), ("stoch_matrix", s_o)):
            assert np.array_equal(eng.moments(M), mu[0]) and eng.alpha_table()
            getattr(eng, name)(c, D)
            assert rel_err(D.val, want) < tol
        assert eng.stoch_method() == "table"
    eng.set_store_alpha(2)
    for _ in range(4):
        eng.moments(M)
        assert eng.alpha_table()
    eng.close()
