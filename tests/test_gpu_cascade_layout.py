"""Mode overlaps handed to the cascade row-major, column-major or strided: the
device turns row-major ones through 32 x 32 tiles, and batches of 1 MB and more
are uploaded beside the kernels.  Every layout of the same numbers has to give
the same bits, and every point of a batch the result it has alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(nb, P, m):
    rng = np.random.default_rng(100 * P + m)
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    d = 2 * P
    Z = [1 + 0.1 * c(nb, d), None, 1.5 + 0.1 * c(nb, d)]
    kz = [c(nb, d), 1 + 0.1 * c(nb, m), c(nb, d)]
    J = [None, c(nb, d, m) / np.sqrt(d), None]
    Jd = [None, c(nb, m, d) / np.sqrt(d), None]
    heights = 0.1 + rng.random((nb, 3))
    return [[0, 1, 0], kz, Z, J, Jd, heights, 1 + 0.1 * c(nb, d), c(nb, d), np.full((nb, 3), min(P, 2))]


def _layout(a, how):
    if a is None or how == 'C':
        return a
    if how == 'F':
        return np.ascontiguousarray(a.transpose(0, 2, 1)).transpose(0, 2, 1)
    wide = np.zeros((a.shape[0], a.shape[1], 2 * a.shape[2]), complex)  # every other column
    wide[:, :, ::2] = a
    return wide[:, :, ::2]


@pytest.mark.parametrize('nb,P,m', [(1, 1, 1), (3, 1, 33), (3, 15, 31), (3, 16, 32), (2, 17, 33), (2, 33, 64),
                                    (70, 16, 33)])
def test_layouts(gpu_ctx, nb, P, m):
    args = _inputs(nb, P, m)
    ref = gpu_ctx.star_cascade(*args, want_nets=True)
    for jl, jdl in (('F', 'F'), ('C', 'F'), ('F', 'C'), ('S', 'S')):
        other = list(args)
        other[3] = [_layout(x, jl) for x in args[3]]
        other[4] = [_layout(x, jdl) for x in args[4]]
        for x, y in zip(ref, gpu_ctx.star_cascade(*other, want_nets=True)):
            assert np.array_equal(x, y)
    if nb > 8:
        for b in (0, nb // 2, nb - 1):
            one = [args[0]] + [[None if x is None else x[b:b + 1] for x in v] for v in args[1:5]] + \
                  [v[b:b + 1] for v in args[5:]]
            for x, y in zip(ref, gpu_ctx.star_cascade(*one, want_nets=True)):
                # the same kernels on the same numbers, but tiles may differ with the batch: rounding
                # of sums of 33 products through three solves of random (condition ~ 1e3) matrices
                assert np.abs(x[b] - y[0]).max() <= 1e-9 * max(1.0, np.abs(x[b]).max())


@pytest.mark.parametrize('nb,P,m', [(1, 1, 1), (2, 8, 17), (2, 33, 64), (3, 10, 130), (2, 70, 200)])
def test_flux_products(gpu_ctx, nb, P, m):
    """r and the last t are those of the nets applied to the incident
    amplitudes (products of 2 to 200 columns on the device)."""
    args = _inputs(nb, P, m)
    a, r, t, R, T = gpu_ctx.star_cascade(*args, want_nets=True)
    n = args[8][0, 0]
    prop = np.arange(2 * P) % P < n
    for b in range(nb):
        v = args[7][b]
        down = np.sum(np.abs(v[prop]) ** 2)
        # one product in another order: 140 roundings of its terms
        assert abs(r[b] - np.sum(np.abs((R[b] @ v)[prop]) ** 2) / down) <= 1e-12 * max(1, r[b])
        # three products one after the other against the product of the matrices (condition ~ 1e3)
        assert abs(t[b, -1] - np.sum(np.abs((T[b] @ v)[prop]) ** 2) / down) <= 1e-9 * max(1, t[b, -1])
