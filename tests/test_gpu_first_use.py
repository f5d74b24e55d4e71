"""First uses: what building an operator or a single product prepares, counted by
the library's entry points, and the results against the host."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def calls(monkeypatch):
    """Names of the library's entry points in the order they are called."""
    from jaxfun_amd import _lib

    names, call = [], _lib.call

    def record(name, *args):
        names.append(name)
        return call(name, *args)

    monkeypatch.setattr(_lib, "call", record)
    return names


def _prepared(names):
    return sum(n.startswith("jfx_par_prepare") for n in names)


def _dirichlet(family, N):
    from jaxfun_amd import Chebyshev, FunctionSpace, Legendre

    return FunctionSpace(N, Legendre if family == "legendre" else Chebyshev, {"left": {"D": 0}, "right": {"D": 0}})


def test_building_operators_prepares_nothing(dev, calls):
    from jaxfun_amd import TestFunction, TrialFunction, inner
    from jaxfun_amd.galerkin.inner import test_operator as weighted_test

    D = _dirichlet("chebyshev", 23)
    x = D.system.base_scalars()[0]
    v, u = TestFunction(D), TrialFunction(D)
    D.backward_operator(30)
    D.backward_operator(30, 1)
    D.scalar_product_operator()
    D.forward_operator()
    weighted_test(D, 1, 27)
    inner((1 + x**2) * v * u, sparse=False)
    assert "jfx_vandermonde_f64" in calls and _prepared(calls) == 0


def test_products_from_the_right_prepare_once(dev, calls):
    from jaxfun_amd.la import DiaMatrix

    rng = np.random.default_rng(0)
    H = np.diag(rng.standard_normal(40)) + np.diag(rng.standard_normal(38), 2)
    A = DiaMatrix.from_dense(H)
    for i in range(3):
        X = rng.standard_normal((5, 40))
        y = (X @ A).cpu().numpy()
        assert np.abs(y - X @ H).max() <= 1e-13
        assert _prepared(calls) <= 1


@pytest.mark.parametrize("M,Kd,P,Q", [(7, 5, 3, 2), (64, 64, 1, 2), (64, 64, 1024, 2), (1, 50, 4, 33), (40, 20, 64, 20),
                                      (600, 9, 20000, 1), (513, 30, 2, 8300)])
def test_single_products(dev, M, Kd, P, Q):
    """Either side of the rule that cuts fragments for one product, and sizes they
    do not take: each entry a sum of K products."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(M + Q)
    A, X = rng.standard_normal((M, Kd)), rng.standard_normal((P, Kd, Q))
    op = K.AxisOperator(torch.tensor(A, device="cuda"), once=True)
    for _ in range(2):
        y = K.apply_along(op, torch.tensor(X, device="cuda"), 1).cpu().numpy()
        bound = np.einsum("mk,pkq->pmq", np.abs(A), np.abs(X))
        assert np.all(np.abs(y - np.einsum("mk,pkq->pmq", A, X)) <= 2 * (Kd + 4) * 2.0**-53 * bound)
    assert op._prep.get("par_f64") is None


def test_evaluations_prepare_nothing_after_the_first(dev, calls):
    import torch

    from jaxfun_amd import Fourier, TensorProduct

    rng = np.random.default_rng(1)
    F, D = Fourier(10), _dirichlet("legendre", 14)
    T = TensorProduct(F, D)
    c = torch.tensor(rng.standard_normal((10, 12)) + 1j * rng.standard_normal((10, 12)), device="cuda")
    pts = [rng.uniform(0.1, 6.0, 9), rng.uniform(-0.9, 0.9, 9)]
    ref = None
    for i in range(3):
        del calls[:]
        e = [T.evaluate(pts, c), F.evaluate(pts[0], c[:, 0].contiguous()), F.derivative_coeffs(c[:, 0].contiguous(), 2),
             D.evaluate(pts[1], c[0].real.contiguous())]
        e = [t.cpu().numpy() for t in e]
        assert i == 0 or _prepared(calls) == 0
        assert ref is None or all(np.array_equal(a, b) for a, b in zip(e, ref))
        ref = e
    m = F.wavenumbers()
    V = np.polynomial.legendre.legvander(pts[1], 13)
    phi = D.stencil_matrix() @ V.T
    E = np.exp(1j * np.outer(pts[0], m))
    ch = c.cpu().numpy()
    assert np.abs(ref[0] - np.einsum("pk,kl,lp->p", E, ch, phi)).max() <= 1e-12
    assert np.abs(ref[1] - E @ ch[:, 0]).max() <= 1e-12
    assert np.abs(ref[2] - (1j * m)**2 * ch[:, 0]).max() <= 1e-12
    assert np.abs(ref[3] - ch[0].real @ phi).max() <= 1e-12


def test_one_preparation_for_a_pass(dev, calls):
    """All operators of a transform, a solve or a nonlinear term in one launch."""
    import torch

    from jaxfun_amd import Div, Fourier, Grad, TensorProduct, TestFunction, TrialFunction, inner

    T = TensorProduct(_dirichlet("chebyshev", 20), _dirichlet("legendre", 31), _dirichlet("chebyshev", 26))
    c = torch.randn(18, 29, 24, dtype=torch.float64, device="cuda")
    u = T.backward(c)
    assert _prepared(calls) == 1
    assert torch.linalg.norm(T.forward(u) - c) <= 1e-11 * torch.linalg.norm(c)
    assert _prepared(calls) == 2
    T.forward(T.backward(c))
    assert _prepared(calls) == 2
    del calls[:]
    T = TensorProduct(Fourier(12), _dirichlet("legendre", 33))
    T.backward(torch.randn(3, 12, 31, dtype=torch.complex128, device="cuda"))
    assert _prepared(calls) == 1
    T = TensorProduct(_dirichlet("legendre", 20), _dirichlet("chebyshev", 31))
    v, u = TestFunction(T), TrialFunction(T)
    A = inner(v * Div(Grad(u)), sparse=True)
    del calls[:]
    f = A.fd_factor()
    assert _prepared(calls) == 1
    f.solve(torch.ones(18, 29, dtype=torch.float64, device="cuda"))
    assert _prepared(calls) == 1


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_operators_cut_together_as_alone(dev, prec):
    """More operators than one launch takes, of every structure and unequal sizes:
    the same fragments bit for bit; sizes that are not taken are left out."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(7)
    structures = [None, K.evaluates_parity(), K.evaluates_parity(-1), K.projects_parity(), K.mixes_parity(),
                  K.mixes_parity(-1, 1, 3)]
    sizes = [(1, 1), (17, 33), (128, 126), (5, 512), (512, 5), (2000, 3)]
    ops = [(torch.tensor(rng.standard_normal(s), device="cuda"), p) for p in structures for s in sizes]
    together, alone = ([K.AxisOperator(A, p) for A, p in ops] for _ in range(2))
    K.prepare_fragments(together + together[:3], prec)
    for a, b in zip(together, alone):
        assert K.PAR_KEYS[prec] in a._prep
        fa, fb = a.fragments(prec), b.fragments(prec)
        assert (fa is None) == (fb is None) == (a.M == 2000)
        assert fa is None or (fa[1:] == fb[1:] and torch.equal(fa[0], fb[0]))


@pytest.mark.parametrize("side", ["built", "used", "foreign"])
def test_operators_built_on_another_stream(dev, side):
    """An operator whose matrix is still being computed on its own stream when a
    product on another stream cuts it: the kept fragments are the finished matrix's."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(9)
    A, X = rng.standard_normal((40, 40)), rng.standard_normal((3, 40, 24))
    A *= np.add.outer(np.arange(40), np.arange(40)) % 2 == 0
    src, x = torch.tensor(A, device="cuda"), torch.tensor(X, device="cuda")
    dst, big = torch.zeros_like(src), torch.full((4096, 4096), 1e-4, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    build, use = (torch.cuda.current_stream(), other) if side == "used" else (other, torch.cuda.current_stream())
    if side == "foreign":
        build = torch.cuda.ExternalStream(other.cuda_stream)
    with torch.cuda.stream(build):
        for _ in range(8):  # some 15 ms ahead of the matrix
            big = big @ big
        dst.copy_(src)
        op = K.AxisOperator(dst, K.mixes_parity())
    with torch.cuda.stream(use):
        first = K.apply_along(op, x, 1)
    torch.cuda.synchronize()
    second = K.apply_along(op, x, 1)
    ref = np.einsum("mk,pkq->pmq", A, X)
    for y in (first, second):
        assert np.abs(y.cpu().numpy() - ref).max() <= 1e-13 * np.abs(ref).max()
