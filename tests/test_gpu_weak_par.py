"""The fused variable-coefficient operator, the PCG steps and the per-slab factors
(csrc/weak_par.hip, csrc/mlp_pcg.hip, csrc/plane_par.hip) against host FP64."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,batch", [(5, 1), (17, 3), (18, 2), (33, 5), (64, 9), (66, 2), (97, 2), (128, 3), (131, 1)])
def test_operator_and_preconditioners(dev, N, batch):
    """N 5..128 run fused (4, 8 and 16 waves), 131 by separate contractions."""
    import torch

    from jaxfun_amd.learned import VarCoeffPoisson2D

    op = VarCoeffPoisson2D(N, 4)
    rng = np.random.default_rng(N)
    n = N - 2
    k, U = rng.uniform(0.5, 2.0, (batch, N, N)), rng.standard_normal((batch, n, n))
    B, D, TB, TD, F = (o.A64.cpu().numpy() for o in (op.B, op.Dx, op.TB, op.TD, op.F))

    def both(a0, a1, x):
        return a0 @ x @ a1.T

    kd, Ud = torch.tensor(k, device=dev), torch.tensor(U, device=dev)
    ref = both(TD, TB, k * both(D, B, U)) + both(TB, TD, k * both(B, D, U))
    y = op.apply(kd, Ud).cpu().numpy()
    # the mesh's mirror symmetry holds to rounding, amplified in D by up to N^2
    assert np.linalg.norm(y - ref) <= 1e-13 * N * np.linalg.norm(ref)
    one = op.apply(kd[:1].contiguous(), Ud).cpu().numpy()  # one field for every system
    ref1 = both(TD, TB, k[:1] * both(D, B, U)) + both(TB, TD, k[:1] * both(B, D, U))
    assert np.linalg.norm(one - ref1) <= 1e-13 * N * np.linalg.norm(ref1)
    # plain: L^-1 / kbar; scaled: F s B L^-1 (F s B)^T
    L = op.L.solve(Ud)
    kbar = op.kbar(kd)
    torch.testing.assert_close(op.plain_precond(kbar)(Ud), L / kbar[:, None, None], rtol=1e-13, atol=1e-14 * float(L.abs().max()))
    P = op.scaled_precond(kd)(Ud).cpu().numpy()
    c = both(B.T, B.T, k * both(F.T, F.T, U))
    ref = both(F, F, k * both(B, B, op.L.solve(torch.tensor(c, device=dev)).cpu().numpy()))
    assert np.linalg.norm(P - ref) <= 1e-12 * N * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [1, 63, 512, 513, 3844])
def test_pcg_steps(dev, n):
    """One step and one direction against the formulas, with systems that are
    stopped (unchanged), that stop here, that go on and that break down."""
    import torch

    from jaxfun_amd import _lib
    from jaxfun_amd import kernels as K

    rng = np.random.default_rng(n)
    Bt = 5
    x, r, p, q, z = rng.standard_normal((5, Bt, n))
    p, q = np.abs(p) + 0.1, np.abs(q) + 0.1
    q[4, -1] = np.nan
    rz, bb = rng.uniform(0.5, 1, Bt), np.array([1.0, 1e30, 1e-30, 1.0, 1.0])
    act, it = np.array([0, 1, 1, 1, 1], np.int32), np.array([7, 2, 2, 2, 2], np.int32)
    T = lambda a: torch.tensor(a, device=dev)  # noqa: E731
    xd, rd, pd, qd, zd, rzd, bbd, ad, itd = (T(a) for a in (x, r, p, q, z, rz, bb, act, it))
    left = torch.zeros(1, dtype=torch.int32, device=dev)
    host = torch.full((1,), -7, dtype=torch.int32).pin_memory()
    _lib.call("jfx_pcg_step", K._p(xd), K._p(rd), K._p(pd), K._p(qd), K._p(rzd), K._p(bbd), 1e-20, K._p(ad), K._p(itd),
              K._p(left), host.data_ptr(), Bt, n, K._s())
    torch.cuda.synchronize()
    a = rz / np.sum(p * q, axis=1)
    x1, r1 = x + a[:, None] * p, r - a[:, None] * q
    x1[0], r1[0] = x[0], r[0]
    eps = 1e-15 * n + 1e-14
    np.testing.assert_allclose(xd.cpu().numpy()[:4], x1[:4], rtol=eps, atol=eps)
    np.testing.assert_allclose(rd.cpu().numpy()[:4], r1[:4], rtol=eps, atol=eps)
    assert ad.cpu().tolist() == [0, 0, 1, 1, 0] and itd.cpu().tolist() == [7, 3, 3, 3, -1] and int(left) == (Bt << 16) + 2
    assert int(host[0]) == 2
    rnow, p0 = rd.cpu().numpy(), pd.clone()
    _lib.call("jfx_pcg_direction", K._p(pd), K._p(zd), K._p(rd), K._p(rzd), K._p(ad), Bt, n, K._s())
    s = np.sum(rnow * z, axis=1)
    for b in range(Bt):
        if b in (2, 3):
            np.testing.assert_allclose(float(rzd[b]), s[b], rtol=1e-12, atol=1e-13 * n)
            np.testing.assert_allclose(pd[b].cpu().numpy(), z[b] + s[b] / rz[b] * p[b], rtol=1e-11, atol=1e-11 * n)
        else:
            assert torch.equal(pd[b], p0[b]) and float(rzd[b]) == rz[b]


def test_pcg_stops_and_counts(dev):
    """Iteration counts, early stops, snapshots and the iteration limit are those of
    the recurrence on the host."""
    import torch

    from jaxfun_amd.learned import pcg

    rng = np.random.default_rng(1)
    Bt, n = 6, 40
    lam = 10.0**rng.uniform(0, 2, (Bt, 1, n))
    lam[2] = 3.0  # one iteration
    b = rng.standard_normal((Bt, 1, n))
    b[5] = 0.0  # converged from the start
    ld, bd = torch.tensor(lam, device=dev), torch.tensor(b, device=dev)

    def host(limit):
        x, its = np.zeros_like(b), np.zeros(Bt, int)
        for s in range(Bt):
            r, xs = b[s].copy(), np.zeros_like(b[s])
            p, rz = r.copy(), float(np.sum(r * r))
            while its[s] < limit and np.sum(r * r) > 1e-20 * np.sum(b[s]**2):
                q = lam[s] * p
                a = rz / np.sum(p * q)
                xs, r, its[s] = xs + a * p, r - a * q, its[s] + 1
                s2 = np.sum(r * r)
                p, rz = r + s2 / rz * p, s2
            x[s] = xs
        return x, its

    for limit, every in ((2000, 1), (2000, 4), (3, 1), (1, 1)):
        snaps = {}
        x, it = pcg(lambda U: ld * U, bd, lambda R: R, rtol=1e-10, maxiter=limit, check_every=every, snapshots=(1, 2, 1500),
                    snap_out=snaps)
        xr, itr = host(limit)
        assert np.all(np.abs(it.cpu().numpy() - itr) <= (0 if limit < 9 else 2)) and int(it[2]) == 1 and int(it[5]) == 0
        np.testing.assert_allclose(x.cpu().numpy(), xr, rtol=1e-8, atol=1e-8)
        assert sorted(snaps) == [k for k in (1, 2) if k <= limit]


@pytest.mark.parametrize("N", [20, 97])
def test_first_use_inside_a_capture(dev, N):
    """The scaled preconditioner whose operators are used for the first time inside
    a graph capture (its solve before): every replay against the eager result."""
    import torch

    from jaxfun_amd import kernels as K
    from jaxfun_amd.learned import VarCoeffPoisson2D

    op, eager = VarCoeffPoisson2D(N, 4), VarCoeffPoisson2D(N, 4)
    rng = np.random.default_rng(N)
    batch = 130  # both ends of the slab kernel's rule take it
    s = torch.tensor(rng.uniform(0.5, 2.0, (batch, N, N)), device=dev)
    R = torch.tensor(rng.standard_normal((batch, N - 2, N - 2)), device=dev)
    op.L.solve(R)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        z = op.scaled_precond(s)(R)
    for _ in range(3):
        R.copy_(torch.tensor(rng.standard_normal(R.shape), device=dev))
        g.replay()
        ref = eager.scaled_precond(s)(R)
        torch.cuda.synchronize()
        assert torch.linalg.norm(z - ref) <= 1e-13 * N * torch.linalg.norm(ref)
    assert torch.equal(op.scaled_precond(s)(R), ref)  # prepared at the next use outside
    # with a scale and added to an output, as the fused kernel does it
    a, b = K.AxisOperator(op.B.A64, op.B.parity), K.AxisOperator(op.B.A64, op.B.parity)
    out, want = torch.ones_like(s), torch.ones_like(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        K.plane(a, b, R, "f64", ("mul_each", s), 0.5, out, True)
    g.replay()
    K.plane(op.B, op.B, R, "f64", ("mul_each", s), 0.5, want, True)
    torch.testing.assert_close(out, want, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("where", ["apply", "precond"])
def test_pcg_leaves_no_queued_store_behind(dev, where):
    """A callback that raises: the steps queued so far, which store to a pinned
    buffer of the call, are finished when the exception comes out."""
    import torch

    from jaxfun_amd.learned import pcg

    b = torch.tensor(np.random.default_rng(2).standard_normal((3, 1, 20)), device=dev)
    lam = torch.linspace(1.0, 50.0, 20, dtype=torch.float64, device=dev)
    big = torch.full((4096, 4096), 1e-4, dtype=torch.float64, device=dev)
    count = {"apply": 0, "precond": 0}

    def step(name, y):
        count[name] += 1
        if name == where and count[name] == 4:
            raise RuntimeError("stop here")
        if name == "apply":
            for _ in range(4):  # some 8 ms of queued work ahead of the step
                torch.mm(big, big)
        return y

    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="stop here"):
        pcg(lambda U: step("apply", lam * U), b, lambda R: step("precond", R.clone()), rtol=1e-14)
    assert torch.cuda.current_stream().query()
