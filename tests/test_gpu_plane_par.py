"""Fused two-axis slab kernels for operators with decoupled even and odd parts
(csrc/plane_par.hip) against dense FP64 products on the host.

Entry by entry |error| <= (K0 + K1 + c) eps (|A0| |X| |A1|^T) per pass: K products
and the folds of each axis, and a few roundings of the epilogue."""

import numpy as np
import pytest

from test_gpu_contract_par import _structured

pytestmark = pytest.mark.gpu

EPS = 2.0**-53
# edges of the 16-row blocks, of the 4-, 8- and 16-wave kernels, and the largest slab
SIZES = [(1, 1), (2, 3), (5, 4), (16, 16), (17, 33), (33, 31), (64, 62), (48, 50), (100, 97), (81, 128), (128, 128)]


@pytest.mark.parametrize("mode,s0,s1", [(1, 1, 1), (1, -1, 1), (1, 1, -1), (2, 1, 1), (2, -1, 1), (2, 1, -1),
                                        (3, 1, 1), (3, -1, 1), (3, 1, -1)])
def test_plane(dev, mode, s0, s1):
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(17 * mode + 3 * s0 + s1)
    for i, (M0, K0) in enumerate(SIZES):
        for j, (M1, K1) in enumerate(SIZES):
            if (i + j) % 2 and i != j + 1:
                continue
            band = ((-1, -1), (2, 2), (0, 9))[(i + 2 * j) % 3] if mode == 3 else (-1, -1)
            A0, A1 = _structured(rng, M0, K0, mode, s0, *band), _structured(rng, M1, K1, mode, s1, *band)
            op0 = K.AxisOperator(torch.tensor(A0, device=dev), (mode, s0, *band))
            op1 = K.AxisOperator(torch.tensor(A1, device=dev), (mode, s1, *band))
            X, E, Y0 = rng.standard_normal((3, K0, K1)), rng.uniform(0.5, 2, (M0, M1)), rng.standard_normal((3, M0, M1))
            epi = (None, "div", "mul")[(i + j) % 3]
            alpha, acc = (1.0, False) if i % 2 else (-0.3, True)
            y = K.plane(op0, op1, torch.tensor(X, device=dev), "f64",
                        epi=None if epi is None else (epi, torch.tensor(E, device=dev)), alpha=alpha,
                        out=torch.tensor(Y0, device=dev) if acc else None, accumulate=acc).cpu().numpy()
            f = {None: np.ones_like(E), "div": 1 / E, "mul": E}[epi]
            ref = alpha * (A0 @ X @ A1.T) * f + (Y0 if acc else 0)
            bound = abs(alpha) * (np.abs(A0) @ np.abs(X) @ np.abs(A1).T) * f + (np.abs(Y0) if acc else 0)
            assert np.all(np.abs(y - ref) <= (K0 + K1 + 10) * 2 * EPS * bound + 1e-300), (M0, K0, M1, K1, epi, acc)


def test_many_slabs(dev):
    """More than three slabs per CU above 32 x 32 take the four-wave kernels: the same
    values as a batch that does not, up to the order of sums."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(2)
    for n, N in ((62, 64), (33, 40), (30, 32)):
        A, W = _structured(rng, N, n, 1, 1), _structured(rng, n, n, 3, 1)
        op, w = K.AxisOperator(torch.tensor(A, device=dev), K.evaluates_parity()), \
            K.AxisOperator(torch.tensor(W, device=dev), K.mixes_parity())
        X = torch.tensor(rng.standard_normal((800, n, n)), device=dev)
        E = torch.tensor(rng.uniform(0.5, 2, (n, n)), device=dev)
        for f in (lambda x: K.plane(op, op, x), lambda x: K.plane_fd(w, w, w, w, x, E)):
            many, few = f(X), f(X[:700].contiguous())
            scale = float(few.abs().max())
            assert float((many[:700] - few).abs().max()) <= 1e-13 * n * scale
            assert float((f(X[700:].contiguous()) - many[700:]).abs().max()) <= 1e-13 * n * scale


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("M0,K0,M1,K1", [(128, 128, 127, 126), (100, 118, 128, 120), (97, 101, 99, 110)])
def test_streamed_slabs(dev, mode, M0, K0, M1, K1):
    """More than one slab per CU, each filling its LDS: the persistent kernel."""
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(M0 + mode)
    A0, A1 = _structured(rng, M0, K0, mode, 1), _structured(rng, M1, K1, mode, 1)
    op0, op1 = (K.AxisOperator(torch.tensor(a, device=dev), (mode, 1, -1, -1)) for a in (A0, A1))
    for B in (257, 600):
        X = torch.tensor(rng.standard_normal((B, K0, K1)), device=dev)
        y = K.plane(op0, op1, X, alpha=0.5)
        for b in (0, 1, 255, 256, B - 1):
            x = X[b].cpu().numpy()
            bound = 0.5 * np.abs(A0) @ np.abs(x) @ np.abs(A1).T
            assert np.all(np.abs(y[b].cpu().numpy() - 0.5 * A0 @ x @ A1.T) <= (K0 + K1 + 10) * 2 * EPS * bound + 1e-300)


@pytest.mark.parametrize("n0,n1", [(1, 1), (2, 5), (16, 16), (31, 33), (62, 62), (64, 64), (97, 40), (62, 126), (128, 128)])
def test_plane_fd(dev, n0, n1):
    import torch

    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(n0 + n1)
    A = [_structured(rng, n, n, 3, 1) for n in (n0, n1, n0, n1)]
    ops = [K.AxisOperator(torch.tensor(a, device=dev), K.mixes_parity()) for a in A]
    X, E = rng.standard_normal((3, n0, n1)), rng.uniform(0.5, 2, (n0, n1))
    y = K.plane_fd(*ops, torch.tensor(X, device=dev), torch.tensor(E, device=dev)).cpu().numpy()
    ref = A[2] @ ((A[0] @ X @ A[1].T) / E) @ A[3].T
    bound = np.abs(A[2]) @ ((np.abs(A[0]) @ np.abs(X) @ np.abs(A[1]).T) / E) @ np.abs(A[3]).T
    assert np.all(np.abs(y - ref) <= (2 * (n0 + n1) + 10) * 2 * EPS * bound)
