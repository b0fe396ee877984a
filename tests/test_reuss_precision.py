"""The unpivoted Reuss solve (sfg_wave.hip, compiled for the CPU) against the
same system solved in extended precision, over grains up to a thousand times
softer in one direction than in another and over coefficients no grain gives."""
import ctypes
import itertools
import os
import subprocess
import tempfile

import numpy as np
import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "specfab_amd", "csrc")
MANDEL = [(0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1)]


def reuss_lib():
    out = os.path.join(tempfile.gettempdir(), "sfg_emul_reuss_%d.so" % os.getpid())
    if not os.path.exists(os.path.join(CSRC, "generated", "sfg_l4maps.h")):
        pytest.skip("generated tables not present (run the build)")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-DSFG_HOST_EMUL", "-w", "-I", CSRC, "-x", "c++",
                           os.path.join(ROOT, "tests", "emul_reuss.cpp"), os.path.join(CSRC, "sfg_wave_host.cpp"),
                           os.path.join(CSRC, "sfg_basis.cpp"), "-o", out])
    return ctypes.CDLL(out)


def coefficients(lam, mu, El, Em, Eg):
    """The compliance's five coefficients of a transversely isotropic grain
    (elas_fwdparams, src/elasticities.f90)."""
    gam = lam + 2 * mu
    xi = 2 * Eg * gam * (lam + mu) - 2 * (El * lam) ** 2
    return [((El * lam) ** 2 - Eg * gam * lam) / (2 * mu * xi), 1 / (2 * mu),
            (Eg * gam * lam - El * lam * (El * lam + 2 * mu)) / (2 * mu * xi),
            (4 * mu * lam * (1 + El) + 4 * mu * mu + Eg * gam * gam - El * El * lam * lam) / (2 * mu * xi) - 1 / (Em * mu),
            (1 - Em) / (2 * Em * mu)]


def moments(c, w):
    """Mandel a2 and the 15 sorted a4 entries of axes c (N, 3), weights w."""
    a2 = np.einsum("n,ni,nj->ij", w, c, c)
    r = np.array([1, 1, 1, np.sqrt(2), np.sqrt(2), np.sqrt(2)])
    a2v = np.array([a2[i, j] for i, j in MANDEL]) * r
    u = [np.sum(w * np.prod([c[:, k] for k in q], axis=0)) for q in itertools.combinations_with_replacement(range(3), 4)]
    return a2v, np.array(u)


def system(a2v, u, k):
    """The 6 x 6 Mandel compliance, in extended precision."""
    ld = np.longdouble
    r2 = np.sqrt(ld(2))
    a2v, u, k = (np.asarray(x, ld) for x in (a2v, u, k))
    r = np.array([1, 1, 1, r2, r2, r2], ld)
    idx = {q: n for n, q in enumerate(itertools.combinations_with_replacement(range(3), 4))}
    a4 = np.array([[r[I] * r[J] * u[idx[tuple(sorted(MANDEL[I] + MANDEL[J]))]] for J in range(6)] for I in range(6)])
    m = np.zeros((3, 3), ld)
    for I, (i, j) in enumerate(MANDEL):
        m[i, j] = m[j, i] = a2v[I] / r[I]
    # {a2, .}: the Mandel matrix of S -> a2 S + S a2
    L = np.zeros((6, 6), ld)
    for J, (i, j) in enumerate(MANDEL):
        S = np.zeros((3, 3), ld)
        S[i, j] = S[j, i] = 1 if i == j else 1 / r2
        T = m @ S + S @ m
        L[:, J] = [T[p, q] * r[I] for I, (p, q) in enumerate(MANDEL)]
    one = np.array([1, 1, 1, 0, 0, 0], ld)
    return (k[0] * np.outer(one, one) + k[1] * np.eye(6, dtype=ld) + k[2] * (np.outer(one, a2v) + np.outer(a2v, one)) +
            k[3] * a4 + k[4] * L)


def solve(A, B):
    """Gaussian elimination with partial pivoting in the type of A."""
    A, B = A.copy(), B.copy()
    for c in range(6):
        p = c + int(np.argmax(np.abs(A[c:, c])))
        A[[c, p]], B[[c, p]] = A[[p, c]], B[[p, c]]
        for r in range(c + 1, 6):
            f = A[r, c] / A[c, c]
            A[r] -= f * A[c]
            B[r] -= f * B[c]
    for r in range(5, -1, -1):
        B[r] = (B[r] - A[r, r + 1:] @ B[r + 1:]) / A[r, r]
    return B


@pytest.mark.parametrize("family", ["grains", "coefficients"])
def test_unpivoted_reuss_as_accurate_as_the_pivoted(family):
    """In every decade of the compliance's condition the largest error is that
    of the pivoted solve: both are backward stable for a positive definite
    matrix, so both are bound by the rounding of its entries times the
    condition (a factor of four for the largest of a few tens of samples)."""
    rng = np.random.default_rng(7)
    ld = np.longdouble
    ex = lambda d: 10.0 ** rng.uniform(-d, d)
    N, cases = 600, []
    for n in range(N):
        # single maxima, girdles and axes along the coordinates
        spread = rng.choice([0.0, 1e-3, 0.02, 0.1, 1.0])
        c = rng.normal(size=(20, 3)) * spread + (np.eye(3)[n % 3] if n % 4 == 0 else rng.normal(size=3))
        c = c * [1, 1, 0.01] if n % 5 == 0 else c
        c /= np.linalg.norm(c, axis=1)[:, None]
        w = rng.uniform(0.5, 1, 20)
        if family == "grains":
            k = coefficients(ex(2), 1.0, ex(1), ex(3), ex(3))
        else:
            k = [ex(2) * rng.integers(2), ex(3), rng.normal() * rng.integers(2), ex(3) * rng.integers(2), ex(3) * rng.integers(2)]
        cases.append(moments(c, w / w.sum()) + (np.array(k, float),))
    a2v, u, k = (np.ascontiguousarray([c[i] for c in cases]) for i in range(3))
    Qs, Ql, ok = np.zeros((N, 3, 3)), np.zeros((N, 3, 3)), np.zeros(N, np.int32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    reuss_lib().emul_reuss(ctypes.c_int64(N), ptr(a2v), ptr(u), ptr(k), ptr(Qs), ptr(ok), ptr(Ql))
    r2 = np.sqrt(ld(2))
    rhs = np.zeros((6, 3), ld)
    rhs[4, 0] = rhs[3, 1] = 1 / r2
    rhs[2, 2] = 1
    rows = []
    for i in np.flatnonzero(ok):
        A = system(a2v[i], u[i], k[i])
        x = solve(A, rhs)
        Q = np.array([x[4] / r2, x[3] / r2, x[2]])
        rows.append([np.linalg.cond(A.astype(float))] + [float(np.abs(q - Q).max() / np.abs(Q).max()) for q in (Qs[i], Ql[i])])
    cond, es, el = np.array(rows).T
    assert len(cond) > N / 2 and cond.max() > 1e4
    for d in range(7):
        m = (cond >= 10.0 ** d) & (cond < 10.0 ** (d + 1))
        if m.sum() >= 10:
            print("%s, condition 1e%d: %d, error %.1e (pivoted %.1e)" % (family, d, m.sum(), es[m].max(), el[m].max()))
            assert es[m].max() < 4 * el[m].max() + 1e-15
