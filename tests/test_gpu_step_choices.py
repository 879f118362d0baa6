"""The step kernels on lattices past the whole-recursion kernels: the untuned choice of
each kind by size, the tuned ones, and a cut-short table at high order in FP32."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import fermi_coeffs, rel_err
from test_gpu_dispatch import FP64_TOL, _check_all, _engine, _pattern, _set_up

pytestmark = pytest.mark.gpu


def _tol(prec, M):
    return FP64_TOL if prec == "fp64" else M * 16 * 2.0 ** -24


# (lattice, block size, columns, precision, lanes x packets of the forward step and of
# the backward step reading the table): two packets a lane below 64 and four while the
# vectors stay in the last-level cache, from 256 workgroups on
@pytest.mark.parametrize("shape,b,S,prec,fwd,bwd", [
    ((70, 61), 2, 31, "fp64", (16, 2), (16, 2)), ((48, 45), 2, 31, "fp64", (32, 1), (32, 1)),
    ((96, 90), 2, 31, "fp64", (16, 2), (8, 4)), ((96, 90), 2, 16, "fp64", (8, 2), (8, 2)),
    ((70, 61), 2, 16, "fp64", (16, 1), (16, 1)), ((70, 61), 2, 64, "fp64", (64, 1), (16, 4)),
    ((48, 45), 2, 64, "fp64", (64, 1), (64, 1)), ((70, 61), 2, 62, "fp32", (16, 2), (16, 2)),
    ((96, 90), 2, 31, "fp32", (8, 2), (8, 2)), ((96, 90), 2, 62, "fp32", (16, 2), (8, 4)),
    ((64, 64), 4, 31, "fp64", (16, 2), (16, 2)), ((48, 45), 4, 31, "fp64", (32, 1), (32, 1)),
    ((64, 64), 4, 62, "fp32", (16, 2), (16, 2)), ((70, 61), 1, 32, "fp64", (16, 2), (16, 2)),
    ((70, 61), 1, 64, "fp64", (64, 1), (16, 4)), ((70, 61), 1, 128, "fp32", (64, 1), (16, 4))])
def test_untuned_geometry(oracle, shape, b, S, prec, fwd, bwd):
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=b, seed=3, W=1.0, J=1.0 if b == 2 else 0.0, orbital_blocks=b > 2)
    eng, orc, bound = _set_up(oracle, H, S, prec=prec)
    M = 8
    _check_all(oracle, eng, orc, H, M, bound, _tol(prec, M))
    for kind, want in ((0, fwd), (4, fwd), (5, bwd)):
        c = eng.kernel_config(kind)
        assert (c["lanes"], c["kq"]) == want and c["sweep"] == 0 and not c["nt"], (kind, c)
    eng.close()


@pytest.mark.parametrize("shape,b,S,sweep,order", [((200, 200), 2, 64, 0, False),
                                                   ((200, 200), 2, 128, 2, False),
                                                   ((40, 40, 40), 2, 128, 0, True)])
def test_untuned_sweep_by_cache_and_lattice(shape, b, S, sweep, order):
    """Per XCD while three vectors stay in 256 MB, one front past that, the lattice row
    order (per XCD again) for 3-D lattices with 4 KiB a block row."""
    from fastkpm_amd import EnergyScale, lattice
    H = lattice.lattice(shape, b=b, seed=3, J=1.0)
    n = H.n_rows * b
    R = np.zeros((n, S), dtype=np.complex128, order="F")
    R[np.arange(n), np.arange(n) % S] = 1.0
    eng = _engine()
    eng.set_R(R)
    eng.set_H(H, EnergyScale(-8.0, 8.0))
    assert abs(eng.moments(4)[0] - n) < 1e-9 * n
    c = eng.kernel_config(0)
    assert c["sweep"] == sweep and bool(c["nt"] & 8) is order, c
    eng.close()


@pytest.mark.parametrize("how", ["call", "environment"])
@pytest.mark.parametrize("prec,store", [("fp64", 1), ("fp32", 1), ("fp64", 2), ("fp32", 2)])
def test_tuned_step_kernels(oracle, monkeypatch, prec, store, how):
    """The tuned geometries, on a lattice whose calls run them."""
    from fastkpm_amd import lattice
    if how == "environment":
        monkeypatch.setenv("FKPM_AUTOTUNE", "1")
    H = lattice.lattice((48, 45), b=2, seed=4, J=2.0)
    # a shape of its own for each case, so that no other case has tuned it
    S = 5 + 2 * store + (prec == "fp32") + 8 * (how == "call")
    eng, orc, bound = _set_up(oracle, H, S, prec=prec)
    eng.set_store_alpha(store)
    if how == "call":
        eng.autotune()
    M = 24
    eng.set_timing(True)
    eng.moments(M)
    assert eng.state()["tuned"] and eng.alpha_table() and not eng.whole_recursion()
    assert eng.timing()["moments_launches"] == M // 2
    _check_all(oracle, eng, orc, H, M, bound, _tol(prec, M))
    assert eng.timing()["autodiff_launches"] == M // 2 - 1
    eng.close()


@pytest.mark.parametrize("b,S", [(2, 9), (8, 9)])
@pytest.mark.parametrize("M", [160, 501])
def test_cut_table_at_high_order_fp32(oracle, monkeypatch, b, S, M):
    """stoch_matrix from a third of the forward vectors in FP32: its two recurrences of
    ceil(M/3) steps on sums of weight up to 2, doubled, stay within four times the error
    of the Clenshaw recurrence (and the output's rounding)."""
    from fastkpm_amd import lattice
    H = lattice.lattice((4, 3, 3), b=b, orbital_blocks=b > 2, W=1.0, J=1.0 if b == 2 else 0.0, seed=S)
    eng, orc, bound = _set_up(oracle, H, S, prec="fp32")
    eng.set_store_alpha(2)
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.02, kind=1)
    want = orc.stoch_matrix(c, H)
    D = H.like()
    eng.moments(2)  # the padded width
    vb = H.n_rows * b * eng.config()["s_padded"] * 8
    monkeypatch.setenv("FKPM_ALPHA_TABLE_BYTES", str(-(-(M + M % 2) // 3) * vb))
    eng.moments(M + M % 2)
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "table"
    err = rel_err(D.val, want)
    eng.set_stoch_method("clenshaw")
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "clenshaw"
    assert err < 4 * rel_err(D.val, want) + 2.0 ** -22
    eng.close()


@pytest.mark.parametrize("prec,S", [("fp64", 127), ("fp32", 253)])
@pytest.mark.parametrize("shape", [(64, 32), (33, 63)])
def test_eight_row_blocks_on_a_wave(oracle, shape, prec, S):
    """The forward step's two forms: 2048 block rows and 2079, a ragged column tile."""
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=8, seed=5, orbital_blocks=True)
    H.val = np.ascontiguousarray(H.val.real)
    eng, orc, bound = _set_up(oracle, H, S, real=True, prec=prec, dense=False)
    M = 8
    _check_all(oracle, eng, orc, H, M, bound, _tol(prec, M))
    c = eng.kernel_config(0)
    assert (c["lanes"], c["kq"]) == (64, 1), c
    eng.close()


@pytest.mark.parametrize("own_pattern", [True, False])
@pytest.mark.parametrize("prec,S", [("fp64", 127), ("fp32", 253)])
@pytest.mark.parametrize("shape", [(4, 4), (32, 32), (25, 41)])
def test_backward_of_eight_row_blocks_on_a_wave(oracle, shape, prec, S, own_pattern):
    """Vectors computed anew beside a kept table up to 1024 block rows, read from 1025
    on; the table still serves a stoch_matrix that follows."""
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=8, seed=5, orbital_blocks=True)
    H.val = np.ascontiguousarray(H.val.real)
    eng, orc, bound = _set_up(oracle, H, S, real=True, prec=prec, dense=False)
    nb, M = H.n_rows, 10
    Dp = H if own_pattern else lattice.coo_to_bsr(nb, 8, range(nb), range(nb),
                                                  np.zeros((nb, 8, 8)))
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.05)
    mu = orc.moments(M)
    want, xi = orc.autodiff_matrix(c, Dp), orc.stoch_matrix(c, Dp)
    for store in (1, 2, 0):  # read at once where it is forced, no table at all
        eng.set_store_alpha(store)
        assert rel_err(eng.moments(M), mu) < _tol(prec, M)
        D = Dp.like(eng.np_dtype)
        eng.autodiff_matrix(c, D)
        assert rel_err(D.val, want) < _tol(prec, M), store
        assert eng.kernel_config(2)["lanes"] == 64
        eng.stoch_matrix(c, D)
        assert rel_err(D.val, xi) < _tol(prec, M), store
    eng.close()


# columns and passes of the forward method's step: the passes of a row side by side up to
# 128 workgroups a sweep, one after another from there on
@pytest.mark.parametrize("prec,S,passes", [("fp64", 33, 3), ("fp64", 129, 9), ("fp32", 129, 5)])
@pytest.mark.parametrize("shape,apart", [((3, 3), True), ((45, 45), True), ((46, 45), False)])
@pytest.mark.parametrize("sliced", [False, True])
def test_forward_method_column_passes(oracle, shape, apart, prec, S, passes, sliced):
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=8, seed=5, orbital_blocks=True)
    eng, orc, bound = _set_up(oracle, H, S, prec=prec, dense=False)
    eng.set_stoch_method("forward")
    if sliced:
        eng.set_slice(1)
    M = 8
    c = fermi_coeffs(oracle, M, -bound, bound, kT=0.05, kind=1)
    D = H.like(eng.np_dtype)
    want = orc.stoch_matrix(c, H)
    for _ in range(3):  # the step loop is captured, then replayed
        eng.stoch_matrix(c, D)
        assert rel_err(D.val, want) < _tol(prec, M)
    k = eng.kernel_config(1)
    ne = 1 if prec == "fp64" else 2
    assert eng.config()["s_padded"] == passes * k["lanes"] * k["kq"] * ne
    assert (k["n_wg"] <= 128) is apart
    eng.close()


def _bonds(nb, b, pairs, real=False):
    """A chain of rows of five blocks and the bonds `pairs` besides."""
    from fastkpm_amd import lattice
    H = _pattern(nb, b, 2, 0, real)
    r, c = np.array(pairs, dtype=int).reshape(-1, 2).T
    T = np.random.default_rng(3).standard_normal((len(r), b, b))
    blocks = np.concatenate([H.val.reshape(-1, b, b).transpose(0, 2, 1), T, T.transpose(0, 2, 1)])
    return lattice.coo_to_bsr(nb, b, np.concatenate([H.row_idx, r, c]),
                              np.concatenate([H.col_idx, c, r]), blocks, H.val.dtype)


# (rows, block size, columns, precision, real, blocks more in one row, lanes x packets of
# the forward step): one packet a lane where the long row's chain outlasts the others
@pytest.mark.parametrize("nb,b,S,prec,real,hub,want", [
    (9000, 2, 11, "fp64", False, 20, (16, 1)), (9000, 2, 11, "fp64", False, 0, (8, 2)),
    (9000, 2, 11, "fp64", False, 5, (8, 2)), (25000, 2, 11, "fp64", False, 20, (8, 2)),
    (9000, 1, 11, "fp64", False, 9, (16, 1)), (9000, 2, 24, "fp32", False, 8, (16, 1)),
    (9000, 4, 24, "fp64", True, 20, (16, 1)), (9000, 4, 24, "fp32", False, 20, (16, 1))])
def test_one_long_row(oracle, nb, b, S, prec, real, hub, want):
    """... and the choice follows a pattern of as many rows and blocks."""
    from fastkpm_amd import EnergyScale
    long = [(0, 1000 + 7 * k) for k in range(hub)]
    even = [(20 * k, 3000 + 20 * k) for k in range(hub)]
    M = 8
    H = _bonds(nb, b, long, real)
    eng, orc, bound = _set_up(oracle, H, S, real=real, prec=prec, dense=False)
    for pairs, geo in ((long, want), (even, (8, 2)), (long, want)):
        H = _bonds(nb, b, pairs, real)
        eng.set_H(H, EnergyScale(-bound, bound))
        orc.set_H(H, -bound, bound)
        _check_all(oracle, eng, orc, H, M, bound, _tol(prec, M))
        for kind in (0, 4):
            c = eng.kernel_config(kind)
            assert (c["lanes"], c["kq"]) == geo, (pairs[:1], kind, c)
    eng.close()
