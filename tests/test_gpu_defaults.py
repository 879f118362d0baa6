"""The untuned choices of the step kernels against the oracle (FP64, 1e-10): the
per-XCD sweep and two-packet geometries of lattices past the whole-recursion
kernels, the padded widths of the matrix-core kernels, and the fused 4x4 outer
product reduced in one reduce-scatter on every compiled lane count."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu


def _run(oracle, H, S, M=8, prec="fp64", before=None, real=False):
    from fastkpm_amd import EnergyScale, HipEngine
    rng = np.random.default_rng(S)
    n = H.n_rows * H.b_len
    R = rng.standard_normal((n, S)) + (0 if real else 1j) * rng.standard_normal((n, S))
    b = H.b_len
    absrow = np.zeros((H.n_rows, b))
    np.add.at(absrow, H.row_idx, np.abs(H.val.reshape(-1, b, b)).sum(axis=1))
    bound = float(absrow.max())
    eng = HipEngine("double" if real else "cx_double", prec)
    if before:
        before(eng)
    eng.set_R(R)
    eng.set_H(H, EnergyScale(-bound, bound))
    orc = oracle.Engine()
    orc.set_H(H, -bound, bound)
    orc.set_R(R)
    c = 1.0 / (1.0 + np.arange(M))
    tol = 1e-10 if prec == "fp64" else M * 16 * 2.0 ** -24
    D = H.like()
    assert rel_err(eng.moments(M), orc.moments(M)) < tol
    eng.autodiff_matrix(c, D)
    assert rel_err(D.val, orc.autodiff_matrix(c, D)) < tol
    eng.stoch_matrix(c, D)
    assert rel_err(D.val, orc.stoch_matrix(c, D)) < tol
    return eng


# N past the whole-recursion kernels; S at and beside the compiled widths
@pytest.mark.parametrize("shape,b,S,real", [((70, 61), 1, 8, False), ((70, 61), 1, 17, True),
                                            ((17, 16, 16), 1, 33, False), ((48, 45), 2, 16, False),
                                            ((48, 45), 2, 31, False), ((48, 45), 2, 64, False),
                                            ((13, 13, 14), 2, 65, False)])
def test_default_sweep_and_geometry(oracle, shape, b, S, real):
    from fastkpm_amd import lattice
    H = lattice.lattice(shape, b=b, W=1.0, J=0.0 if b == 1 else 1.0, seed=3,
                        dtype=np.float64 if real else np.complex128)
    eng = _run(oracle, H, S, real=real)
    c = eng.kernel_config(0)
    assert c["sweep"] in (0, 2)
    eng.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("S", [1, 16, 17, 33, 48, 80, 144])
def test_matrix_core_padded_width(oracle, S, prec):
    """144 columns take 144 (FP64) or 160 (FP32, pairs of tiles), not 192."""
    from fastkpm_amd import lattice
    H = lattice.lattice((4, 3, 3), b=8, orbital_blocks=True, seed=S)
    eng = _run(oracle, H, S, prec=prec)
    tile = 16 if prec == "fp64" or S <= 16 else 32
    assert eng.config()["s_padded"] == -(-S // tile) * tile
    assert eng.kernel_config(0)["mfma"]
    eng.close()


@pytest.mark.parametrize("lanes,kq", [(4, 1), (4, 2), (8, 2), (16, 1), (16, 2), (32, 1), (32, 2),
                                      (64, 1), (64, 2)])
@pytest.mark.parametrize("store", [0, 2])
def test_fused_4x4_outer_product(oracle, lanes, kq, store):
    from fastkpm_amd import lattice
    H = lattice.lattice((5, 4), b=4, orbital_blocks=True, seed=2)

    def force(eng):
        eng.set_geometry(lanes, kq, 0)
        eng.set_store_alpha(store)
    _run(oracle, H, 11, before=force).close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("rows", [7, 8, "long"])
@pytest.mark.parametrize("S", [3, 16, 40, 64])
def test_matrix_core_backward_step_from_the_table(oracle, rows, S, prec):
    """8x8 blocks with the forward vectors kept: row-resident steps on 7 and 8
    block slots and the general step on longer rows, one and two column tiles,
    D on H's pattern and on the diagonal, stoch_matrix from the table."""
    from fastkpm_amd import EnergyScale, HipEngine, lattice
    from helpers import with_partner_bonds
    from test_gpu_resident import _random_H
    if rows == "long":
        H, bound = _random_H(40, 8, 9, False, seed=S)
        assert np.diff(H.row_ptr).max() > 8
    else:
        H = lattice.lattice((4, 3, 3), b=8, orbital_blocks=True, seed=S)
        if rows == 8:
            H = with_partner_bonds(H, (4, 3, 3), seed=S)
        bound = float(np.abs(np.linalg.eigvalsh(H.to_dense())).max()) * 1.01
        assert np.diff(H.row_ptr).max() == rows
    rng = np.random.default_rng(S)
    R = rng.standard_normal((H.n_rows * 8, S)) + 1j * rng.standard_normal((H.n_rows * 8, S))
    nb = H.n_rows
    Dd = lattice.coo_to_bsr(nb, 8, np.arange(nb), np.arange(nb), np.zeros((nb, 8, 8)))
    M = 14
    c = 1.0 / (1.0 + np.arange(M))
    eng = HipEngine("cx_double", prec)
    eng.set_store_alpha(2)
    eng.set_R(R)
    eng.set_H(H, EnergyScale(-bound, bound))
    orc = oracle.Engine()
    orc.set_H(H, -bound, bound)
    orc.set_R(R)
    tol = 1e-10 if prec == "fp64" else M * 16 * 2.0 ** -24
    for D in (H.like(), Dd):
        assert rel_err(eng.moments(M), orc.moments(M)) < tol
        assert eng.alpha_table() and eng.kernel_config(5)["mfma"]
        eng.autodiff_matrix(c, D)
        assert rel_err(D.val, orc.autodiff_matrix(c, D)) < tol
    eng.stoch_matrix(c, D)
    assert eng.stoch_method() == "table"
    assert rel_err(D.val, orc.stoch_matrix(c, D)) < tol
    eng.close()


@pytest.mark.parametrize("shapes", [((20, 18), (20, 18)), ((20, 18), (18, 20)),
                                    ((20, 18), (70, 70)), ((70, 70), (20, 18))])
def test_set_H_arrays_are_free_on_return(oracle, shapes):
    """H values below and above the staged size, on a held and on a new
    pattern: the caller's arrays may change as soon as set_H returns."""
    from fastkpm_amd import EnergyScale, HipEngine, lattice
    eng = HipEngine("cx_double", "fp64")
    for k, shape in enumerate(shapes * 2):
        H = lattice.lattice(shape, b=2, J=1.0 + k, seed=k)
        rng = np.random.default_rng(k)
        R = rng.standard_normal((H.n_rows * 2, 3)) + 1j * rng.standard_normal((H.n_rows * 2, 3))
        orc = oracle.Engine()
        orc.set_H(H, -12.0, 12.0)
        orc.set_R(R)
        want = orc.moments(12)
        if k % 2:  # values that must not survive
            eng.set_H(lattice.lattice(shape, b=2, J=9.0, seed=77), EnergyScale(-20.0, 20.0))
        eng.set_R(R)
        eng.set_H(H, EnergyScale(-12.0, 12.0))
        H.val[:] = 1e30
        assert rel_err(eng.moments(12), want) < 1e-10
    eng.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("S", [1, 16, 17, 48, 130])
def test_matrix_core_outer_product(oracle, S, prec):
    """stoch_matrix of 8x8 blocks on a D pattern of its own: rows of 0 to 9 blocks
    (groups of four and their remainders), one column to several passes."""
    from fastkpm_amd import EnergyScale, HipEngine, lattice
    H = lattice.lattice((4, 3, 3), b=8, orbital_blocks=True, seed=S)
    nb = H.n_rows
    rng = np.random.default_rng(S)
    rows = np.repeat(np.arange(nb), np.arange(nb) % 10)
    cols = np.concatenate([rng.choice(nb, k % 10, replace=False) for k in range(nb)])
    D = lattice.coo_to_bsr(nb, 8, rows, cols, np.zeros((len(rows), 8, 8)))
    R = rng.standard_normal((nb * 8, S)) + 1j * rng.standard_normal((nb * 8, S))
    M = 6
    c = 1.0 / (1.0 + np.arange(M))
    bound = float(np.abs(np.linalg.eigvalsh(H.to_dense())).max()) * 1.01
    eng = HipEngine("cx_double", prec)
    eng.set_R(R)
    eng.set_H(H, EnergyScale(-bound, bound))
    orc = oracle.Engine()
    orc.set_H(H, -bound, bound)
    orc.set_R(R)
    eng.stoch_matrix(c, D)
    want = orc.stoch_matrix(c, D)
    assert rel_err(D.val, want) < (1e-10 if prec == "fp64" else M * 16 * 2.0 ** -24)
    eng.close()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("b,S", [(1, 5), (2, 17), (4, 6), (8, 20)])
@pytest.mark.parametrize("M", [14, 16, 18])
def test_first_forward_vectors_kept(oracle, monkeypatch, M, b, S, prec):
    """A table too small for every forward vector keeps the first ones from a
    third of the orders on: autodiff_matrix recomputes down to them and reads
    the rest (D on H's pattern and on the diagonal), stoch_matrix starts from
    them up to the order they were kept for."""
    from fastkpm_amd import EnergyScale, HipEngine, lattice
    H = lattice.lattice((4, 3, 3), b=b, orbital_blocks=b > 2, W=1.0, J=1.0 if b == 2 else 0.0,
                        seed=S)
    bound = float(np.abs(np.linalg.eigvalsh(H.to_dense())).max()) * 1.01
    nb = H.n_rows
    rng = np.random.default_rng(S)
    R = rng.standard_normal((nb * b, S)) + 1j * rng.standard_normal((nb * b, S))
    Dd = lattice.coo_to_bsr(nb, b, np.arange(nb), np.arange(nb), np.zeros((nb, b, b)))
    c = 1.0 / (1.0 + np.arange(M + 2))
    orc = oracle.Engine()
    orc.set_H(H, -bound, bound)
    orc.set_R(R)
    tol = 1e-10 if prec == "fp64" else M * 16 * 2.0 ** -24
    least = -(-M // 3)
    for slots in (least - 1, least, least + 1, M // 2 - 1):
        eng = HipEngine("cx_double", prec)
        eng.set_store_alpha(2)
        eng.set_R(R)
        eng.set_H(H, EnergyScale(-bound, bound))
        eng.moments(2)  # the padded width
        vb = nb * b * eng.config()["s_padded"] * (16 if prec == "fp64" else 8)
        monkeypatch.setenv("FKPM_ALPHA_TABLE_BYTES", str(slots * vb))
        for D in (H.like(), Dd):
            assert rel_err(eng.moments(M), orc.moments(M)) < tol
            assert eng.alpha_table() == (slots >= least)
            eng.autodiff_matrix(c[:M], D)
            assert rel_err(D.val, orc.autodiff_matrix(c[:M], D)) < tol
        for m in (M, M - 1, M - 2, 3, M + 2):
            eng.stoch_matrix(c[:m], D)
            kept = slots >= least and m <= M or m <= 2 * slots and slots >= least
            assert eng.stoch_method() == ("table" if kept else "clenshaw"), (slots, m)
            assert rel_err(D.val, orc.stoch_matrix(c[:m], D)) < tol
        monkeypatch.delenv("FKPM_ALPHA_TABLE_BYTES")
        eng.close()
