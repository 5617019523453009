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


@pytest.fixture(scope='module')
def spectrum(gpu_ctx, mesh600):  # noqa: F811
    """24 lights, each with its own wavelength, angle and index, solved alone."""
    mh, _ = mesh600
    ps = [_params(480.0 + 17.0 * i, 600., 2.2 + 0.06 * i + 0.01j, 5.0 + 1.3 * i, 31.0) for i in range(24)]
    return ps, [gpu_ctx.calc_modes_batch(mh, [p[0]], 40, 1, [p[2]], [p[3]], [p[4]], 5, block=8) for p in ps]


@pytest.mark.parametrize('block,lights', [(1, 5), (1, 24), (2, 7), (4, 7), (4, 24), (8, 24), (0, 7)])
def test_lights_of_a_batch_are_their_own(gpu_ctx, mesh600, spectrum, block, lights):  # noqa: F811
    """Every light of a batch against itself alone: the instances differ, so
    data read across them shows, and they converge after different numbers of
    restarts, so the active ones move to other slots on the way."""
    mh, _ = mesh600
    ps, alone = spectrum
    pick = [23 - i for i in range(lights)]
    col = lambda k: [ps[i][k] for i in pick]
    beta, J, Jd, _ = gpu_ctx.calc_modes_batch(mh, col(0), 40, 1, col(2), col(3), col(4), 5, block=block)
    for b, i in enumerate(pick):
        bref, Jref, Jdref, _ = alone[i]
        # the bounds of test_gram_schmidt_sizes, for the same reason
        np.testing.assert_allclose(beta[b], bref[0], rtol=1e-9, atol=1e-9 * np.abs(bref[0]).max())
        Pref = Jref[0] @ Jdref[0]
        assert np.abs(J[b] @ Jd[b] - Pref).max() <= 1e-8 * np.abs(Pref).max()
