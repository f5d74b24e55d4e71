"""Eigenpairs of Dirichlet mass and stiffness pairs, diagonalised one parity at a
time (la/tpmatrix.py axis_eig), against the fast-diagonalisation solve refined in
extended precision."""

import time

import numpy as np
import pytest
import torch

from jaxfun_amd.la import tpmatrix as T


def _pair(family, N):
    n, k = N - 2, np.arange(N)
    S = np.eye(n, N) - np.eye(n, N, 2)
    if family == "legendre":
        return S @ np.diag(2.0 / (2 * k + 1)) @ S.T, -np.diag(4.0 * np.arange(n) + 6.0)
    h = np.full(N, np.pi / 2)
    h[0] = np.pi
    off = k[None, :] - k[:, None]
    A = np.where((off >= 2) & (off % 2 == 0), k[None, :] * (k[None, :]**2 - k[:, None]**2) * np.pi / 2, 0.0)
    return S @ np.diag(h) @ S.T, S @ A @ S.T


def _solve_error(eig, M, K, F):
    lam, V, W = eig
    D = lam[:, None] + lam[None, :]

    def once(R):
        return V @ ((W @ R @ W.T) / D) @ V.T

    X = once(F)
    Y, Ml, Kl = (a.astype(np.longdouble) for a in (X, M, K))
    for _ in range(3):
        Y = Y + once((F - (Kl @ Y @ Ml.T + Ml @ Y @ Kl.T)).astype(np.float64))
    return float(np.linalg.norm(X - Y) / np.linalg.norm(Y))


@pytest.mark.parametrize("family", ["legendre", "chebyshev"])
@pytest.mark.parametrize("N", [5, 6, 16, 33, 50, 64, 65, 100, 128])
def test_parity_blocks(family, N):
    M, K = _pair(family, N)
    n = N - 2
    lam, V, W = T.axis_eig(K, M)
    assert np.all(np.diff(lam) >= 0)
    order = T._parity_order(V, W)
    assert order is not None
    Vp, Wp = V[:, order], W[order]
    odd = np.add.outer(np.arange(n), np.arange(n)) % 2 == 1
    assert not Vp[odd].any() and not Wp[odd].any()
    f = np.random.default_rng(N).standard_normal((n, n)) * np.outer((1.0 + np.arange(n))**-2, (1.0 + np.arange(n))**-2)
    err, whole = _solve_error((lam, V, W), M, K, f), _solve_error(T._axis_eig(K, M), M, K, f)
    assert err <= 1.2 * whole + 4e-16  # no further off than the pair diagonalised as a whole


def _degenerate_pairs():
    n, rng = 12, np.random.default_rng(3)
    k2 = np.fft.fftfreq(20, 1.0 / 20)**2
    M, K = _pair("legendre", 16)
    close = np.diag(np.repeat(np.arange(1.0, n // 4 + 1), 4)) + 1e-13 * np.diag(rng.standard_normal(n))
    return {"identity": (np.eye(n), np.eye(n)),
            "chebyshev mass": (np.diag(np.where(np.arange(n) == 0, np.pi, np.pi / 2)), np.eye(n)),
            "fourier": (2 * np.pi * np.diag(k2), 2 * np.pi * np.eye(20)),
            "fourier mass": (2 * np.pi * np.eye(20), np.eye(20)),
            "mass against itself": (M, M),
            "multiples on blocks": (np.kron(np.eye(2), K), np.kron(np.eye(2), M)),
            "nearly equal": (close, np.eye(n))}


@pytest.mark.parametrize("name", list(_degenerate_pairs()))
def test_repeated_eigenvalues(name):
    """Pairs with equal and nearly equal eigenvalues within one parity: finite
    vectors that diagonalise the pair, to the rounding of n-term FP64 sums."""
    A, B = _degenerate_pairs()[name]
    lam, V, W = T.axis_eig(A, B)
    assert np.isfinite(lam).all() and np.isfinite(V).all() and np.isfinite(W).all()
    tol = 8 * len(lam) * np.finfo(float).eps
    cond = np.linalg.norm(W) * np.linalg.norm(B @ V)
    assert np.linalg.norm(W @ B @ V - np.eye(len(lam))) <= tol * cond
    assert np.linalg.norm(W @ A @ V - np.diag(lam)) <= tol * cond * np.abs(lam).max()
    ref = np.sort(T._axis_eig(A, B)[0])
    np.testing.assert_allclose(lam, ref, rtol=tol * np.linalg.cond(B), atol=tol * np.abs(ref).max())


def test_pairs_without_parity_are_left_whole():
    rng = np.random.default_rng(0)
    A = rng.standard_normal((7, 7))
    A = A + A.T
    lam, V, W = T.axis_eig(A, np.eye(7))
    ref = T._axis_eig(A, np.eye(7))
    assert all(np.array_equal(a, b) for a, b in zip((lam, V, W), ref))
    assert T._parity_order(V, W) is None


@pytest.mark.parametrize("family", ["legendre", "chebyshev"])
def test_host_factors_follow_one_order(family, monkeypatch):
    """eigvecs_host, lefts_host and D_host together solve the problem, as the
    operators built from them do."""
    monkeypatch.setattr(T.K, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(T.K, "prepare_fragments", lambda ops: None)
    (M0, K0), (M1, K1) = _pair(family, 11), _pair(family, 16)
    fd = T.tpmats_lu_factor([T.TPMatrix([T.Matrix(K0), T.Matrix(M1)]), T.TPMatrix([T.Matrix(M0), T.Matrix(K1)])])
    F = np.random.default_rng(5).standard_normal(fd.shape)
    (W0, W1), (V0, V1) = fd.lefts_host, fd.eigvecs_host
    X = V0 @ ((W0 @ F @ W1.T) / fd.D_host) @ V1.T
    assert np.linalg.norm(K0 @ X @ M1.T + M0 @ X @ K1.T - F) <= 1e-12 * np.linalg.norm(F)
    for host, ops in ((fd.eigvecs_host, fd.V), (fd.lefts_host, fd.W)):
        assert all(np.array_equal(h, o.A64.numpy()) for h, o in zip(host, ops))


@pytest.mark.parametrize("n,spread", [(1, 0), (2, 3), (33, 6), (200, 2), (257, 0)])
def test_sliced_product(n, spread):
    """Products of slices against the extended product, entries of unequal sizes and
    a zero row and column among them."""
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, n)).astype(np.longdouble) * 10.0**rng.uniform(-spread, spread, (n, n))
    X = X + X * np.longdouble(2.0)**-60
    Y = rng.standard_normal((n, n)) * 10.0**rng.uniform(-spread, spread, (n, n))
    if n > 2:
        X[1], Y[:, 2] = 0.0, 0.0
    got = sum(t.astype(np.longdouble) for t in T._sliced_product(X, Y))
    bound = np.abs(X).max(1)[:, None] * np.abs(Y).max(0) * n
    assert np.all(np.abs(got - X @ Y.astype(np.longdouble)) <= 2.0**-60 * bound)


def test_diagonalisation_time():
    """The correction's extended arithmetic stays on the order of the eigenvalue
    solve (twice it at this size; 7 times with extended matrix products)."""
    M, K = _pair("legendre", 1200)

    def seconds(f):
        t = time.perf_counter()
        f()
        return time.perf_counter() - t

    T.axis_eig(K[:64, :64], M[:64, :64])
    assert any(seconds(lambda: T.axis_eig(K, M)) < 4 * seconds(lambda: T._axis_eig(K, M)) for _ in range(3))


def test_structure_is_looked_for_where_it_is_used(monkeypatch):
    """A matrix finds its structure for its operator up to the sizes that kernels
    take, 1024 x 512, and never beyond."""
    looked = []
    structure = T.K.host_structure
    monkeypatch.setattr(T.K, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(T.K, "host_structure", lambda A: looked.append(A.shape) or structure(A))
    for shape, taken in (((6, 6), True), ((1024, 512), True), ((1025, 512), False), ((40, 513), False)):
        op = T.Matrix(np.eye(*shape)).operator()
        assert op.parity == (T.K.mixes_parity(1, 0, 0) if taken else None)
        assert (shape in looked) == taken
