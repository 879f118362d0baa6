"""The whole-recursion kernels of small lattices (kpm_resident.h) against the
oracle and against the step kernels, at the edges of their ranges: workgroups
of 64 to 512 threads, every count of block rows per thread, rows with more
blocks than the registers keep, rows of uneven length, one column and odd
column counts, M from 2, a D pattern other than H's, both stoch_matrix methods.

Tolerances (norm-wise): FP64 1e-10.  FP32 storage: at most about 16 roundings
of 2^-24 per element and step over M/2 steps, M * 2^-24 * 16; against the step
kernels the vectors are the same operations, so the FP64 moment sums differ by
their order only (1e-12), D by the FP32 partial sums of the step kernels.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24


def _random_H(nb, b, bonds, real, seed):
    """Hermitian BSR matrix with the diagonal: on small nb random bonds (`bonds`
    per row on average, uneven rows), else each bond i - i + d (mod nb) of
    `bonds` distances with probability 0.9."""
    from fastkpm_amd import lattice
    rng = np.random.default_rng(seed)
    if nb < 200:
        n = int(nb * bonds / 2)
        i = rng.integers(0, nb, n)
        j = np.where(rng.random(n) < 0.05, 0, rng.integers(0, nb, n))
    else:
        d = np.array([1, 7, 32, 90, 3, 11, 50, 71])[:bonds]
        i = np.repeat(np.arange(nb), len(d))
        j = (i + np.tile(d, nb)) % nb
        some = rng.random(len(i)) < 0.9
        i, j = i[some], j[some]
    keep = i != j
    i, j = i[keep], j[keep]
    T = rng.standard_normal((len(i), b, b)) + (0 if real else 1j) * rng.standard_normal((len(i), b, b))
    on = rng.standard_normal((nb, b, b)) + (0 if real else 1j) * rng.standard_normal((nb, b, b))
    H = lattice.coo_to_bsr(nb, b, np.concatenate([np.arange(nb), i, j]),
                           np.concatenate([np.arange(nb), j, i]),
                           np.concatenate([on + np.conj(on.transpose(0, 2, 1)), T,
                                           np.conj(T.transpose(0, 2, 1))]))
    if real:
        H.val = H.val.real.copy()
    rows = np.zeros(nb * b)
    np.add.at(rows.reshape(nb, b), H.row_idx, np.abs(H.val.reshape(-1, b, b)).sum(axis=1))
    return H, float(rows.max()) * 1.01


# nb, b, bonds per row, real, S, M
CASES = [
    (1, 1, 0, False, 1, 6), (3, 2, 2, False, 5, 2), (64, 1, 4, True, 7, 4), (65, 2, 4, False, 3, 18),
    (511, 1, 8, False, 2, 12), (512, 2, 5, False, 4, 10), (513, 1, 2, False, 3, 10),
    (512, 4, 3, True, 3, 8), (513, 2, 2, True, 3, 10), (1024, 1, 2, False, 16, 30),
    (1025, 2, 3, False, 2, 8), (1024, 4, 1, False, 2, 6), (2048, 2, 2, False, 2, 8),
    (4096, 1, 3, False, 1, 8), (4096, 1, 2, True, 5, 8), (2047, 1, 6, True, 9, 14),
]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nb,b,bonds,real,S,M", CASES)
def test_resident_matches_oracle_and_step_kernels(oracle, nb, b, bonds, real, S, M, prec):
    from fastkpm_amd import EnergyScale, HipEngine, lattice
    H, bound = _random_H(nb, b, bonds, real, seed=nb + b)
    rng = np.random.default_rng(7)
    R = rng.standard_normal((nb * b, S)) + (0 if real else 1j) * rng.standard_normal((nb * b, S))
    lo, hi = -bound, bound * 1.03
    es = EnergyScale(lo, hi)
    c = rng.standard_normal(M) / (1.0 + np.arange(M))
    Dd = lattice.coo_to_bsr(nb, b, np.arange(nb), np.arange(nb), np.zeros((nb, b, b)))
    if real:
        Dd.val = Dd.val.real.copy()
    orc = oracle.Engine()
    orc.set_H(H, lo, hi)
    orc.set_R(R)
    mu_o = orc.moments(M)
    ad_o = orc.autodiff_matrix(c, H.like())
    orc.moments(M)
    adf_o = orc.autodiff_matrix(c, Dd)
    st_o = orc.stoch_matrix(c, H.like())
    got = {}
    for steps in (False, True):
        eng = HipEngine("double" if real else "cx_double", prec)
        if steps:
            eng.set_sweep(2)  # a forced sweep asks for the step kernels
        eng.set_R(R)
        eng.set_H(H, es)
        D = H.like()
        out = [eng.moments(M)]
        eng.autodiff_matrix(c, D)
        out.append(D.val.copy())
        eng.moments(M)
        eng.autodiff_matrix(c, Dd)
        out.append(Dd.val.copy())
        eng.stoch_matrix(c, D)  # from the table the resident kernels kept
        if not steps:
            assert eng.stoch_method() == "table"
        out.append(D.val.copy())
        eng.set_stoch_method("clenshaw")
        eng.stoch_matrix(c, D)
        out.append(D.val.copy())
        got[steps] = out
        eng.close()
    tol = 1e-10 if prec == "fp64" else max(M, 8) * U32 * 16
    for a, o in zip(got[False], (mu_o, ad_o, adf_o, st_o, st_o)):
        assert rel_err(a, o) < tol
    assert rel_err(got[False][0], got[True][0]) < 1e-12
    for a, o in zip(got[False][1:], got[True][1:]):
        assert rel_err(a, o) < tol


def test_resident_new_H_on_one_handle(oracle):
    """A second H of another size, then the first again, on one handle: the
    packed H, the tables and the stale forward vectors are replaced."""
    from fastkpm_amd import EnergyScale, HipEngine
    eng = HipEngine("cx_double", "fp64")
    M = 12
    c = 1.0 / (1.0 + np.arange(M))
    for k, (nb, b) in enumerate([(40, 2), (600, 2), (40, 2), (80, 1)]):
        H, bound = _random_H(nb, b, 4, False, seed=nb)
        rng = np.random.default_rng(k)
        R = rng.standard_normal((nb * b, 3 + k)) + 1j * rng.standard_normal((nb * b, 3 + k))
        eng.set_R(R)
        eng.set_H(H, EnergyScale(-bound, bound))
        orc = oracle.Engine()
        orc.set_H(H, -bound, bound)
        orc.set_R(R)
        D = H.like()
        eng.stoch_matrix(c, D)
        assert eng.stoch_method() == "clenshaw"  # no forward vectors of this H
        assert rel_err(D.val, orc.stoch_matrix(c, D)) < 1e-10
        assert rel_err(eng.moments(M), orc.moments(M)) < 1e-10
        eng.autodiff_matrix(c, D)
        assert rel_err(D.val, orc.autodiff_matrix(c, D)) < 1e-10
    eng.close()


def test_resident_table_over_budget_runs_the_step_kernels(oracle, monkeypatch):
    from fastkpm_amd import EnergyScale, HipEngine
    monkeypatch.setenv("FKPM_ALPHA_TABLE_BYTES", "1000")
    H, bound = _random_H(100, 2, 4, False, seed=5)
    rng = np.random.default_rng(1)
    R = rng.standard_normal((200, 4)) + 1j * rng.standard_normal((200, 4))
    eng = HipEngine("cx_double", "fp64")
    eng.set_R(R)
    eng.set_H(H, EnergyScale(-bound, bound))
    orc = oracle.Engine()
    orc.set_H(H, -bound, bound)
    orc.set_R(R)
    M = 20
    c = 1.0 / (1.0 + np.arange(M))
    assert rel_err(eng.moments(M), orc.moments(M)) < 1e-10
    D = H.like()
    eng.autodiff_matrix(c, D)
    assert rel_err(D.val, orc.autodiff_matrix(c, D)) < 1e-10
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "clenshaw"
    assert rel_err(D.val, orc.stoch_matrix(c, D)) < 1e-10
    eng.close()
