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
