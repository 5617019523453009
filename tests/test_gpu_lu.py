"""Numeric LU on the GPU at the edges of the panel kernels' ranges: a mesh
analysed with a leaf size above its unknowns is one dense front (s = the
number of unknowns), so the panel sees s, s - 32, ... pivot candidates on its
way down, and smaller leaves give fronts of many sizes.  The matrices are
random with rows scaled so that partial pivoting interchanges rows throughout
(a factorisation that loses an interchange or a panel column is wrong by
O(1)).  The solution is checked by the
row-wise backward error: 1e-11 for one front (n eps = 8e-13 at 3,600 rows, times
10), 1e-8 for trees (pivots restricted to a front's own rows: no bound on the
growth of a random matrix, but a lost interchange still shows as O(1))."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh_file(tmp_path, ntri):
    from emustack_amd import mesher
    p = os.path.join(str(tmp_path), 'cell_%d.mail' % ntri)
    mesher.write_mail(p, mesher.ellipse_cell_ntri(500.0, 500.0, 120.0, 120.0, ntri, seed=2))
    return p


def _grating(ctx, nel, leaf):
    from emustack_amd import _lib
    x = np.linspace(0.0, 1.0, 2 * nel + 1)
    i = np.arange(nel)
    tn = np.stack((2 * i + 1, 2 * i + 3, 2 * i + 2), axis=1)
    return _lib.MeshHandle1D(x, tn, np.where(i < nel // 3, 2, 1), ctx, leaf_size=leaf)


def _check(ctx, mh, seed, nb=2, tol=1e-11):
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    from emustack_amd import _lib
    rp, ci = np.zeros(mh.neq + 1, np.int64), np.zeros(mh.nnz, np.int32)
    _lib.check(_lib.lib().emu_mesh_arrays(mh.h, _lib.ptr(rp, _lib.c_i64p), _lib.ptr(ci, _lib.c_i32p), None, None,
                                          None))
    vals = rng.standard_normal((nb, mh.nnz)) + 1j * rng.standard_normal((nb, mh.nnz))
    rows = np.repeat(np.arange(mh.neq), np.diff(rp))
    vals *= np.exp(rng.uniform(-3.0, 3.0, mh.neq))[rows]
    b = rng.standard_normal((nb, 2, mh.neq)) + 1j * rng.standard_normal((nb, 2, mh.neq))
    x, npert = ctx.lu_solve(mh, vals, b)
    assert npert == 0
    for k in range(nb):
        A = sp.csr_matrix((vals[k], ci, rp), shape=(mh.neq, mh.neq))
        # backward error row by row: |A x - b| against |A| |x| + |b|
        res = np.abs(A @ x[k].T - b[k].T)
        scale = (abs(A) @ np.abs(x[k].T)).max() + np.abs(b[k]).max()
        assert res.max() <= tol * scale, (mh.neq, k, res.max() / scale)


@pytest.mark.parametrize('nel', [3, 4, 8, 9, 16, 17, 33, 64, 65, 129])
def test_dense_front_of_a_grating(gpu_ctx, nel):
    """One front of 8 nel unknowns: from below one panel to past 1,024 rows."""
    _check(gpu_ctx, _grating(gpu_ctx, nel, 100000), nel)


@pytest.mark.parametrize('ntri,leaf', [(100, 100000), (180, 100000), (300, 100000), (300, 40), (300, 97),
                                       (500, 200), (500, 1)])
def test_fronts_of_a_cell(gpu_ctx, tmp_path, ntri, leaf):
    """Single dense fronts up to 3,600 rows and trees of many front sizes."""
    from emustack_amd import _lib
    _check(gpu_ctx, _lib.MeshHandle(_mesh_file(tmp_path, ntri), gpu_ctx, leaf_size=leaf), ntri,
           tol=1e-11 if leaf == 100000 else 1e-8)


@pytest.mark.parametrize('nel', [257, 513])
def test_dense_front_beyond_two_and_four_thousand_rows(gpu_ctx, nel):
    """2,056 unknowns: just into the panels of 2,049 to 4,096 candidates.  4,104:
    the first panel step in memory, the second takes over in registers (n eps
    times 10 = 9e-12)."""
    _check(gpu_ctx, _grating(gpu_ctx, nel, 100000), nel, nb=1)


def test_zero_pivot_is_replaced_and_counted(gpu_ctx):
    """An all-zero matrix: every pivot is replaced and counted, nothing hangs."""
    mh = _grating(gpu_ctx, 9, 100000)
    _, npert = gpu_ctx.lu_solve(mh, np.zeros((1, mh.nnz), complex), np.zeros((1, 1, mh.neq), complex))
    assert npert == mh.neq
