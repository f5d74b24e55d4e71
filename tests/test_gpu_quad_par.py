"""The fused quadratic term (csrc/quad_par.hip) against host FP64.

Its sums are those of the products written out, in another order: relative to the
largest entry the error is a few eps times the contracted sizes."""

import numpy as np
import pytest
import sympy as sp

from test_gpu_contract_par import _structured

pytestmark = pytest.mark.gpu


# 4, 8 and 12 waves; odd meshes (a middle point), one strip and many, unequal axes
SIZES = [(1, 2, 1, 2), (3, 6, 5, 9), (16, 32, 17, 33), (30, 48, 22, 31), (31, 49, 62, 96), (62, 96, 33, 128),
         (79, 122, 96, 150), (126, 192, 126, 192), (128, 191, 100, 97), (15, 24, 126, 192)]


@pytest.mark.parametrize("n0,Q0,n1,Q1", SIZES)
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_quadratic_term(dev, n0, Q0, n1, Q1, dtype):
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(n0 * Q1)
    mats = [_structured(rng, Q0, n0, 1, 1), _structured(rng, Q0, n0, 1, -1), _structured(rng, Q1, n1, 1, 1),
            _structured(rng, Q1, n1, 1, -1), _structured(rng, n0, Q0, 2, 1), _structured(rng, n1, Q1, 2, 1)]
    pars = [(1, 1, -1, -1), (1, -1, -1, -1)] * 2 + [(2, 1, -1, -1)] * 2
    ops = [K.AxisOperator(torch.tensor(m, device=dev), p) for m, p in zip(mats, pars)]
    assert K.quad_ok(*ops)
    B0, D0, B1, D1, S0, S1 = mats
    U = rng.standard_normal((3, n0, n1)).astype(dtype)
    for c in ((0, -1, -2, 0, 0, 0), (0.3, 0, 0.7, -1, -0.5, 2.0)):
        y = K.quadratic_term(*ops, c, torch.tensor(U, device=dev)).cpu().numpy()
        assert y.dtype == dtype
        Ud = U.astype(np.float64)
        u, ux, uy = B0 @ Ud @ B1.T, D0 @ Ud @ B1.T, B0 @ Ud @ D1.T
        w = c[0] * u * u + c[1] * u * ux + c[2] * u * uy + c[3] * ux * ux + c[4] * ux * uy + c[5] * uy * uy
        ref = S0 @ w @ S1.T
        a, ax, ay = (np.abs(p) @ np.abs(Ud) @ np.abs(q).T for p, q in ((B0, B1), (D0, B1), (B0, D1)))
        aw = (abs(c[0]) * a * a + abs(c[1]) * a * ax + abs(c[2]) * a * ay + abs(c[3]) * ax * ax + abs(c[4]) * ax * ay +
              abs(c[5]) * ay * ay)
        bound = np.abs(S0) @ aw @ np.abs(S1).T
        eps = 2.0**-53 * (2 * (n0 + n1) + Q0 + Q1 + 20)
        assert np.all(np.abs(y - ref) <= eps * bound + (2.0**-23 * np.abs(ref) if dtype == "float32" else 0) + 1e-300)


def test_sizes_that_are_not_taken(dev):
    from jaxfun_amd import _lib

    ok = _lib.load().jfx_quad_par_ok
    assert ok(126, 192, 126, 192) == 1 and ok(128, 192, 128, 192) == 1
    assert ok(158, 240, 158, 240) == 0 and ok(126, 256, 126, 256) == 0 and ok(0, 4, 4, 4) == 0


@pytest.mark.parametrize("family", ["legendre", "chebyshev"])
@pytest.mark.parametrize("N0,N1,batch", [(20, 25, 3), (128, 90, 100), (128, 128, 2)])
@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_step_is_the_same_with_and_without(dev, family, N0, N1, batch, precision):
    """The integrator's nonlinear term, fused and by separate launches."""
    import torch

    from jaxfun_amd import Chebyshev, Div, FunctionSpace, Grad, Legendre, TensorProduct, TestFunction, TrialFunction
    from jaxfun_amd.galerkin.arguments import t
    from jaxfun_amd.integrators import ARS443, IMEXRungeKutta

    fam = {"legendre": Legendre, "chebyshev": Chebyshev}[family]
    T = TensorProduct(*[FunctionSpace(n, fam, {"left": {"D": 0}, "right": {"D": 0}}) for n in (N0, N1)])
    v, u = TestFunction(T), TrialFunction(T, transient=True)
    x, y = T.system.base_scalars()
    weak = v * (u.diff(t) + u * (u.diff(x) + 2 * u.diff(y)) - 0.5 * u.diff(x) * u.diff(y) - 1e-2 * Div(Grad(u)))
    it = IMEXRungeKutta(weak, tableau=ARS443, initial=sp.S.Zero, precision=precision)
    assert it._quad_operators() is not None
    rng = np.random.default_rng(0)
    k0, k1 = np.arange(N0 - 2)[:, None], np.arange(N1 - 2)[None, :]
    U = torch.tensor(rng.standard_normal((batch, N0 - 2, N1 - 2)) / ((1 + k0) * (1 + k1))**2, device=dev).to(it.dt_io)
    out = []
    for pays in (True, False):
        it._quad_pays = lambda n, p=pays: p
        out.append(it.nonlinear_rhs_scalar_product(U).double())
    tol = 1e-13 if precision == "f64" else 2e-6
    assert float((out[0] - out[1]).norm() / out[1].norm()) < tol


@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_the_other_data_type_is_refused(dev, precision):
    """Fused and separate alike."""
    import torch

    from jaxfun_amd import Div, FunctionSpace, Grad, Legendre, TensorProduct, TestFunction, TrialFunction
    from jaxfun_amd.galerkin.arguments import t
    from jaxfun_amd.integrators import ARS443, IMEXRungeKutta

    D = FunctionSpace(12, Legendre, {"left": {"D": 0}, "right": {"D": 0}})
    T = TensorProduct(D, D)
    v, u = TestFunction(T), TrialFunction(T, transient=True)
    x, y = T.system.base_scalars()
    weak = v * (u.diff(t) + u * (u.diff(x) + u.diff(y)) - 1e-2 * Div(Grad(u)))
    it = IMEXRungeKutta(weak, tableau=ARS443, initial=sp.S.Zero, precision=precision)
    assert it._quad_operators() is not None
    other = torch.float32 if it.dt_io == torch.float64 else torch.float64
    for pays in (True, False):
        it._quad_pays = lambda n, p=pays: p
        with pytest.raises(TypeError):
            it.nonlinear_rhs_scalar_product(torch.zeros((2, 10, 10), dtype=other, device=dev))
        it.nonlinear_rhs_scalar_product(torch.zeros((2, 10, 10), dtype=it.dt_io, device=dev))
