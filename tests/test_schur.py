"""Schur form of the projected matrices on the host (schur.cpp): backward
error, unitarity and the order of the eigenvalues against LAPACK's zgees, at
the sizes where the code changes path: blocks that the small solver finishes
(26), bulges per train (80, 160, 320), the reduction (192), remainders of the
strips of eight; and the shapes the eigensolver makes (a triangular part, a
spike, a band below the diagonal)."""
import ctypes
import os
import re

import numpy as np
import pytest
import scipy.linalg as sl

from emustack_amd import _lib

EPS = np.finfo(float).eps


def _schur(a, sel):
    n = len(a)
    a = np.array(a, np.complex128, order='F')
    t, q = np.zeros((n, n), np.complex128, order='F'), np.zeros((n, n), np.complex128, order='F')
    dp = lambda x: x.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    sel = np.ascontiguousarray(sel, np.int32)
    _lib.check(_lib.lib().emu_schur(n, dp(a), sel.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)), dp(t), dp(q)))
    return t, q


def _matrix(kind, n):
    rng = np.random.default_rng(n)
    g = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    if kind == 'dense':
        return g
    if kind == 'krylov':  # locked and kept triangular part, spike rows, band of four below the diagonal
        k = n // 2
        a = np.triu(g, -4) * np.exp(-4 * np.arange(n) / n)[:, None]
        a[:k, :k] = np.triu(a[:k, :k])
        a[k:k + 4, :k] = g[k:k + 4, :k] * 1e-3
        return a
    if kind == 'split':  # decoupled blocks, one of them zero, and equal eigenvalues
        a = np.zeros((n, n), complex)
        k = n // 3
        a[:k, :k] = g[:k, :k]
        a[2 * k:, 2 * k:] = np.triu(g[2 * k:, 2 * k:], 1) + np.eye(n - 2 * k)
        return a
    if kind == 'ones':  # rank one: the reduction leaves entries down to the smallest numbers
        return np.ones((n, n))
    if kind == 'steep':  # columns of 1e-160 and less on the way
        return g * 10.0 ** -np.linspace(0, 300, n)[:, None]
    if kind == 'huge':
        return g * 1e150
    return g * 1e-120  # tiny


@pytest.mark.parametrize('kind,n', [(k, n) for k in ('dense', 'krylov', 'split')
                                    for n in (1, 2, 3, 9, 25, 26, 27, 28, 33, 65, 79, 80, 104, 159, 161, 191, 193,
                                              319, 321, 504)] + [('huge', 40), ('tiny', 40), ('steep', 40), ('steep', 90), ('ones', 30), ('ones', 90), ('ones', 193),
                                                                         ('ones', 300)])
def test_schur_form(kind, n):
    a = _matrix(kind, n)
    rng = np.random.default_rng(n + 1)
    sel = (rng.random(n) < 0.6).astype(np.int32)
    t, q = _schur(a, sel)
    none = _schur(a, np.zeros(n, np.int32))[0]
    # an entry meets about 3 n rotations or reflections, each of which adds
    # at most four roundings of its size, of either sign
    tol = 4 * EPS * (1 + np.sqrt(3 * n))
    scale = np.abs(a).max()
    assert np.array_equal(t, np.triu(t))
    assert np.linalg.norm(q @ (t / scale) @ q.conj().T - a / scale) <= tol * np.linalg.norm(a / scale)
    assert np.linalg.norm(q.conj().T @ q - np.eye(n)) <= tol * np.sqrt(n)
    # the selected eigenvalues first, both groups in their order (the moves round)
    w = np.diag(none)
    want = np.concatenate((w[sel != 0], w[sel == 0]))
    assert np.abs(np.diag(t) - want).max() <= tol * np.linalg.norm(a / scale) * scale
    if kind == 'dense':
        ref = np.diag(sl.schur(a, output='complex')[0])
        near = np.abs(ref[:, None] - np.diag(t)[None, :])
        # a random dense matrix: condition numbers of its eigenvalues up to a few n
        assert near.min(axis=1).max() <= 10 * n * tol * np.linalg.norm(a)


@pytest.mark.parametrize('value', [256, -65536, 1 << 30])
def test_any_nonzero_selects(value):
    """A row is selected by any value but zero, also one whose lowest byte is zero."""
    a = _matrix('dense', 40)
    sel = (np.arange(40) % 3 == 1).astype(np.int32)
    t, q = _schur(a, sel)
    t2, q2 = _schur(a, sel * value)
    assert np.array_equal(t, t2) and np.array_equal(q, q2)


def test_every_instruction_set_in_use_is_asked_for():
    """The code is compiled for a list of CPU features; schur_available has to
    ask for each of them (a virtual machine can mask any one)."""
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), '..', 'emustack_amd', 'csrc', 'schur.cpp')
    with open(src) as f:
        text = f.read()
    used = re.search(r'target\("([^"]*)"\)', text).group(1).split(',')
    asked = re.findall(r'__builtin_cpu_supports\("([^"]*)"\)', text)
    assert sorted(used) == sorted(asked)
