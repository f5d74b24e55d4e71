"""Contractions by operators with decoupled even and odd parts
(csrc/contract_par.hip) against dense FP64 products on the host.

Every result is a sum of at most K products plus one fold of the input and one
of the halves, so |error| <= (K + 4) eps sum_k |A[m, k]| |X[k]| entry by entry.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = {"f64": 2.0**-53, "f32": 2.0**-24}


def _structured(rng, M, K, mode, sgn, p=-1, q=-1):
    A = rng.standard_normal((M, K))
    m, k = np.arange(M)[:, None], np.arange(K)[None, :]
    if mode == 1:
        A = 0.5 * (A + sgn * (1 - 2 * (k % 2)) * A[::-1])
    elif mode == 2:
        A = 0.5 * (A + sgn * (1 - 2 * (m % 2)) * A[:, ::-1])
    elif mode == 3:
        A = A * ((m + k) % 2 == (0 if sgn > 0 else 1))
        if p >= 0:
            A = A * ((k - m >= -p) & (k - m <= q))
    return A


def _check(op, A, X, axis, prec):
    import torch

    from jaxfun_amd import kernels as K

    x = torch.tensor(X, device="cuda", dtype=K.io_dtype(prec))
    y = K.apply_along(op, x, axis, prec).cpu().numpy().astype(np.float64)
    xh = np.moveaxis(x.cpu().numpy().astype(np.float64), axis, -1)
    ref = np.moveaxis(xh @ A.T, -1, axis)
    bound = np.moveaxis(np.abs(xh) @ np.abs(A).T, -1, axis)
    # FP32 operators carry one more rounding of their entries
    assert np.all(np.abs(y - ref) <= (A.shape[1] + 5) * 2 * EPS[prec] * bound + 1e-300)


# edges of the 16-row blocks, the 32-column tiles and the k-steps; one past them; the largest sizes
SIZES = [(1, 1), (2, 3), (5, 4), (16, 16), (17, 33), (31, 32), (33, 31), (64, 62), (128, 128), (127, 126), (126, 193),
         (192, 126), (300, 40), (40, 300), (512, 5), (5, 512)]
LAYOUTS = [((1,), ()), ((70,), ()), ((2,), (37,)), ((3,), (64,)), ((1,), (1, 129)), ((5,), (2,))]


@pytest.mark.parametrize("mode,sgn,p,q", [(1, 1, -1, -1), (1, -1, -1, -1), (2, 1, -1, -1), (2, -1, -1, -1),
                                          (3, 1, -1, -1), (3, -1, -1, -1), (3, 1, 2, 2), (3, -1, 1, 5), (3, 1, 0, 400),
                                          (0, 1, -1, -1)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_structured_contraction(dev, mode, sgn, p, q, prec):
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(mode * 10 + sgn)
    for M, Kd in SIZES:
        A = _structured(rng, M, Kd, mode, sgn, p, q)
        op = K.AxisOperator(torch.tensor(A, device=dev), None if mode == 0 else (mode, sgn, p, q))
        for lead, trail in LAYOUTS:
            _check(op, A, rng.standard_normal(lead + (Kd,) + trail), len(lead), prec)


def test_unaligned_views_and_large_results(dev):
    """Inputs one element off 16-byte alignment take the element loads; whole-line
    results above 64 MiB are stored past the L2."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(5)
    A = _structured(rng, 64, 62, 1, 1)
    op = K.AxisOperator(torch.tensor(A, device=dev), K.evaluates_parity())
    for shape, axis in (((9, 62), 1), ((62, 10), 0)):
        n = int(np.prod(shape))
        base = torch.tensor(rng.standard_normal(n + 1), device=dev)
        x = base[1:].view(shape)
        y = K.apply_along(op, x, axis)
        torch.testing.assert_close(y, K.apply_along(op, x.clone(), axis), rtol=0, atol=0)
    for shape, axis in (((64 * 2100, 62), 1), ((2100, 62, 64), 1)):
        X = rng.standard_normal(shape)
        _check(op, A, X, axis, "f64")
        opt = op.t()
        X = rng.standard_normal(tuple(64 if s == 62 else s for s in shape[:axis + 1]) + shape[axis + 1:])
        _check(opt, A.T, X, axis, "f64")


def test_space_operators_match_their_dense_matrices(dev):
    """The structures that spaces and matrices declare hold: every operator gives
    what its dense matrix gives, to rounding of the mesh symmetry."""
    import torch

    from jaxfun_amd import Chebyshev, FunctionSpace, Legendre, TestFunction, TrialFunction, Ultraspherical, inner
    from jaxfun_amd import kernels as K
    from jaxfun_amd.galerkin.inner import test_operator as weighted

    rng = np.random.default_rng(3)
    D, N, R = {"left": {"D": 0}, "right": {"D": 0}}, {"left": {"N": 0}, "right": {"N": 0}}, \
        {"left": {"D": 0}, "right": {"N": 0}}
    ops = []
    for fam in (Legendre, Chebyshev, Ultraspherical):
        kw = {"lambda_": 1} if fam is Ultraspherical else {}
        spaces = [fam(21, **kw), FunctionSpace(20, fam, bcs=D, **kw), FunctionSpace(21, fam, bcs=R, domain=(0, 3), **kw)]
        if fam is not Chebyshev:
            spaces.append(FunctionSpace(20, fam, bcs=N, **kw))
        for V in spaces:
            ops += [V.backward_operator(33, k) for k in (0, 1, 2)] + [V.scalar_product_operator(), V.forward_operator(31)]
            ops += [weighted(V, i, 24) for i in (0, 1)]
            if V.is_orthogonal:
                continue
            assert V.has_parity() == (V.bcs != R)
            v, u = TestFunction(V), TrialFunction(V)
            ops += [inner(v * u).operator(), inner(v * u.diff(V.system.base_scalars()[0], 2)).operator()]
    assert sum(op.parity is not None for op in ops) > len(ops) // 2
    for op in ops:
        A = op.A64.cpu().numpy()
        X = rng.standard_normal((op.K, 7))
        y = K.apply_along(op, torch.tensor(X, device=dev), 0).cpu().numpy()
        # entries of mirrored rows differ by rounding of the nodes, amplified by up to K^2 per derivative
        assert np.abs(y - A @ X).max() <= 1e-12 * np.abs(A).max() * op.K


def test_first_use_inside_a_capture(dev):
    """An operator whose fragments are not prepared yet can be captured, and is
    prepared by a later eager use."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(8)
    A = _structured(rng, 48, 40, 2, 1)
    op = K.AxisOperator(torch.tensor(A, device=dev), K.projects_parity())
    x = torch.tensor(rng.standard_normal((40, 64)), device=dev)
    y = torch.zeros(48, 64, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        K.apply_along(op, x, 0, out=y)
    for _ in range(3):
        x.copy_(torch.tensor(rng.standard_normal((40, 64)), device=dev))
        g.replay()
        torch.cuda.synchronize()
        ref = A @ x.cpu().numpy()
        assert np.abs(y.cpu().numpy() - ref).max() < 1e-12 * np.abs(ref).max()
        eager = K.apply_along(op, x, 0).cpu().numpy()
        assert np.abs(eager - ref).max() < 1e-12 * np.abs(ref).max()


def test_prepared_on_another_stream():
    """An operator first used on a busy stream is ready for one that does not wait for it."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(5)
    A = _structured(rng, 96, 64, 1, 1)
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.ones((4096, 4096), device="cuda")
    x = torch.tensor(rng.standard_normal((7, 64)), device="cuda")
    op = K.AxisOperator(torch.tensor(A, device="cuda"), (1, 1, -1, -1))
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        for _ in range(20):
            big = big @ big * 2.0**-12
        K.apply_along(op, x, 1, "f64")
    with torch.cuda.stream(other):
        y = K.apply_along(op, x, 1, "f64")
    torch.cuda.synchronize()
    bound = np.abs(x.cpu().numpy()) @ np.abs(A).T
    assert np.all(np.abs(y.cpu().numpy() - x.cpu().numpy() @ A.T) <= 68 * EPS["f64"] * bound)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("M,Kd,pre,post", [(33, 160, (2,), (37,)), (33, 161, (2,), (37,)), (65, 176, (3,), (18,)),
                                           (17, 192, (1,), (70,)), (40, 193, (2,), (5,)), (512, 5, (821,), (10,)),
                                           (321, 161, (1639,), (10,)), (300, 256, (1,), (33,)), (9, 400, (2,), (15,))])
def test_dense_operators_in_ragged_layouts(dev, prec, M, Kd, pre, post):
    """Around the K at which a workgroup takes 16 columns instead of 32, and the
    ends of the ranges that go by fragments."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(M + Kd)
    A = rng.standard_normal((M, Kd))
    op = K.AxisOperator(torch.tensor(A, device="cuda"))
    _check(op, A, rng.standard_normal(pre + (Kd,) + post), len(pre), prec)
    assert (op._prep.get(K.PAR_KEYS[prec]) is not None) == K._use_fragments(op, int(np.prod(pre)), int(np.prod(post)), prec)
