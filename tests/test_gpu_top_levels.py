"""Solves of trees whose top levels go through one launch (small fronts, up to
8 right-hand sides) against the level-by-level launches that more right-hand
sides take: gratings and cells of one to many levels, leaves of one to 96
unknowns, so that the fused part is none, some, 16 (its limit) or all levels,
with fronts of one tile and more."""
import numpy as np
import pytest

from test_gpu_lu import _grating, _mesh_file

pytestmark = pytest.mark.gpu


def _compare(ctx, mh, seed):
    from emustack_amd import _lib
    rng = np.random.default_rng(seed)
    rp, ci = np.zeros(mh.neq + 1, np.int64), np.zeros(mh.nnz, np.int32)
    _lib.check(_lib.lib().emu_mesh_arrays(mh.h, _lib.ptr(rp, _lib.c_i64p), _lib.ptr(ci, _lib.c_i32p), None, None,
                                          None))
    nb = 3
    rows = np.repeat(np.arange(mh.neq), np.diff(rp))
    vals = rng.standard_normal((nb, mh.nnz)) + 1j * rng.standard_normal((nb, mh.nnz))
    vals[:, ci == rows] += 4.0 * np.diff(rp).max()  # diagonally dominant: condition number below 10
    b = rng.standard_normal((nb, 9, mh.neq)) + 1j * rng.standard_normal((nb, 9, mh.neq))
    many, npert = ctx.lu_solve(mh, vals, b)
    assert npert == 0
    for nrhs in (1, 3, 8):
        x, _ = ctx.lu_solve(mh, vals, b[:, :nrhs])
        # sums of at most a few hundred terms in another order, condition number 10
        assert np.abs(x - many[:, :nrhs]).max() <= 1e-12 * np.abs(many).max(), nrhs


@pytest.mark.parametrize('nel,leaf', [(3, 1), (9, 1), (64, 1), (64, 24), (300, 1), (300, 24), (300, 96), (300, 100000)])
def test_gratings(gpu_ctx, nel, leaf):
    _compare(gpu_ctx, _grating(gpu_ctx, nel, leaf), nel + leaf)


@pytest.mark.parametrize('ntri,leaf', [(40, 1), (100, 24), (300, 96)])
def test_cells(gpu_ctx, tmp_path, ntri, leaf):
    from emustack_amd import _lib
    _compare(gpu_ctx, _lib.MeshHandle(_mesh_file(tmp_path, ntri), gpu_ctx, leaf_size=leaf), ntri + leaf)
