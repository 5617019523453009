"""The Gram-Schmidt steps of the Krylov expansion at the sizes where their
kernels change: one vector or a block, few or many row pieces (several lights
push a call over the limit of the small-batch kernels), subspaces beyond 256
columns (the staging of the coefficients), the default block.  The eigenpairs
do not depend on any of it."""
import numpy as np
import pytest

from test_gpu_parity import _params, mesh600  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def reference(gpu_ctx, mesh600, mats):  # noqa: F811
    mh, _ = mesh600
    p = _params(700.0, 600., mats('Si_c', 700.0), 20, 40)
    return p, gpu_ctx.calc_modes_batch(mh, [p[0]], 40, 1, [p[2]], [p[3]], [p[4]], 5, block=8)


@pytest.mark.parametrize('block,ncv,lights', [(1, 0, 1), (1, 290, 1), (1, 0, 24), (2, 290, 1), (2, 0, 24),
                                              (4, 290, 1), (4, 0, 24), (0, 0, 1), (0, 290, 3), (8, 0, 24)])
def test_gram_schmidt_sizes(gpu_ctx, mesh600, reference, block, ncv, lights):  # noqa: F811
    mh, _ = mesh600
    p, (bref, Jref, Jdref, _) = reference
    rep = lambda x: [x] * lights
    beta, J, Jd, _ = gpu_ctx.calc_modes_batch(mh, rep(p[0]), 40, 1, rep(p[2]), rep(p[3]), rep(p[4]), 5, block=block,
                                              ncv=ncv)
    Pref = Jref[0] @ Jdref[0]
    for b in (0, lights - 1):
        # both are converged to 1e-12 or better; the bounds of the comparison with the oracle
        np.testing.assert_allclose(beta[b], bref[0], rtol=1e-9, atol=1e-9 * np.abs(bref[0]).max())
        assert np.abs(J[b] @ Jd[b] - Pref).max() <= 1e-8 * np.abs(Pref).max()
