"""Thin torch-tensor wrappers around the libjfx C ABI.

Every function here launches a hand-written HIP kernel from ``libjfx.so`` on
the current torch stream; torch provides only device memory and the stream.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from . import _lib

PRECISIONS = ("f64", "f32", "bf16x3", "bf16x6", "ozaki3", "ozaki4", "ozaki5", "i8x5", "i8x6", "i8x7")
FAMILY = {"legendre": 0, "chebyshev": 1}


def device() -> torch.device:
    if not torch.cuda.is_available():
        raise RuntimeError("jaxfun_amd needs a ROCm GPU (gfx950); none is visible")
    _lib.load()
    return torch.device("cuda", torch.cuda.current_device())


def _p(t: torch.Tensor | None):
    """Device address for a pointer argument (None: null)."""
    return None if t is None else t.data_ptr()


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _s():
    """The current stream of the current device, as an address.  The raw query
    builds no Stream object (0.3 against 2 us per launch)."""
    if _raw_stream is not None:
        return _raw_stream(torch.cuda.current_device())
    return torch.cuda.current_stream().cuda_stream


_stream_of = getattr(torch._C, "_cuda_getCurrentStream", None)


def _stream_id() -> tuple:
    """(stream id, device index, device type) of the current stream, from which
    PyTorch's own streams can be named again later."""
    if _stream_of is not None:
        return _stream_of(torch.cuda.current_device())
    s = torch.cuda.current_stream()
    return s.stream_id, s.device_index, s.device_type


def _wait_for(stream: tuple) -> None:
    """The current stream's next work follows what ``stream`` (:func:`_stream_id`)
    has been given so far.  Stream 0 and odd ids are PyTorch's streams, which it
    never destroys; others are foreign handles that may be gone by now: the device."""
    sid, index, kind = stream
    if sid == 0 or sid & 1:
        torch.cuda.current_stream().wait_stream(torch.cuda.Stream(stream_id=sid, device_index=index, device_type=kind))
    else:
        torch.cuda.synchronize()


def _req(t: torch.Tensor, dtype: torch.dtype, name: str) -> None:
    if isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == dtype and t.is_contiguous():
        return
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise TypeError(f"{name} must be a CUDA/HIP torch tensor")
    if t.dtype != dtype:
        raise TypeError(f"{name} must be {dtype}, got {t.dtype}")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


# ---------------------------------------------------------------- basis


def gauss_nodes(family: str, N: int) -> tuple[torch.Tensor, torch.Tensor]:
    dev = device()
    x = torch.empty(N, dtype=torch.float64, device=dev)
    w = torch.empty(N, dtype=torch.float64, device=dev)
    _lib.call("jfx_gauss_nodes", FAMILY[family], N, _p(x), _p(w), _s())
    return x, w


def vandermonde(family: str, x: torch.Tensor, N: int, k: int = 0, scale: float = 1.0) -> torch.Tensor:
    _req(x, torch.float64, "x")
    V = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device)
    _lib.call("jfx_vandermonde_f64", FAMILY[family], _p(x), x.shape[0], N, k, float(scale), _p(V), _s())
    return V


def vandermonde_rec(rec: torch.Tensor, x: torch.Tensor, N: int, k: int = 0, scale: float = 1.0) -> torch.Tensor:
    """(Q, N) Vandermonde of the basis with recurrence table ``rec`` (3, N)."""
    _req(x, torch.float64, "x")
    _req(rec, torch.float64, "rec")
    if rec.numel() != 3 * N:
        raise ValueError(f"vandermonde_rec: recurrence table has {rec.numel()} entries, need {3 * N}")
    V = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device)
    _lib.call("jfx_vandermonde_rec_f64", _p(x), x.shape[0], N, k, _p(rec), float(scale), _p(V), _s())
    return V


def scale_transpose(V: torch.Tensor, rowscale: torch.Tensor | None = None,
                    colscale: torch.Tensor | None = None, s: float = 1.0) -> torch.Tensor:
    """``out[c, r] = V[r, c] * rowscale[r] * colscale[c] * s``."""
    _req(V, torch.float64, "V")
    R, C = V.shape
    out = torch.empty((C, R), dtype=torch.float64, device=V.device)
    _lib.call("jfx_scale_transpose", _p(V), R, C, _p(rowscale), _p(colscale), float(s), _p(out), _s())
    return out


# ---------------------------------------------------------------- casts / elementwise


def cast(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    if x.dtype == dtype:
        return x
    x = x.contiguous()
    y = torch.empty(x.shape, dtype=dtype, device=x.device)
    if x.dtype == torch.float64 and dtype == torch.float32:
        _lib.call("jfx_cast", 0, _p(x), _p(y), x.numel(), _s())
    elif x.dtype == torch.float32 and dtype == torch.float64:
        _lib.call("jfx_cast", 1, _p(x), _p(y), x.numel(), _s())
    else:
        raise TypeError(f"unsupported cast {x.dtype} -> {dtype}")
    return y


def lincomb(terms, out: torch.Tensor | None = None, accumulate: bool = False) -> torch.Tensor:
    """``out (+)= sum c_j x_j`` for up to 8 same-shape tensors in one pass
    (real coefficients; complex tensors through their real views)."""
    terms = [(float(c), x) for c, x in terms]
    if any(x.is_complex() for _, x in terms) or (out is not None and out.is_complex()):
        terms = [(c, x if x.is_complex() else to_complex(x.contiguous())) for c, x in terms]
        ref = out if out is not None else terms[0][1]
        res = torch.empty_like(ref) if out is None else out
        lincomb([(c, torch.view_as_real(x)) for c, x in terms], torch.view_as_real(res), accumulate)
        return res
    if not terms and out is None:
        raise ValueError("lincomb needs at least one term or an output")
    ref = out if out is not None else terms[0][1]
    if out is None:
        out = torch.empty_like(ref)
    dt = {torch.float64: 0, torch.float32: 1}[out.dtype]
    for chunk_start in range(0, max(1, len(terms)), 8):
        chunk = terms[chunk_start:chunk_start + 8]
        for _, x in chunk:
            _req(x, out.dtype, "lincomb input")
            if x.shape != out.shape:
                raise ValueError("lincomb: shape mismatch")
        ptrs = (ctypes.c_void_p * 8)(*[x.data_ptr() for _, x in chunk])
        cs = (ctypes.c_double * 8)(*[c for c, _ in chunk])
        acc = 1 if (accumulate or chunk_start > 0) else 0
        _lib.call("jfx_lincomb", dt, len(chunk), ptrs, cs, _p(out), out.numel(), acc, _s())
    return out


def sum_products(terms, out: torch.Tensor | None = None) -> torch.Tensor:
    """``out = sum_t c_t * a_t * b_t`` pointwise for up to 4 (c, a, b) terms."""
    terms = [(float(c), a, b) for c, a, b in terms]
    if not 1 <= len(terms) <= 4:
        raise ValueError("sum_products takes 1 to 4 terms")
    ref = terms[0][1]
    out = torch.empty_like(ref) if out is None else out
    _req(out, out.dtype, "out")
    for _, a, b in terms:
        _req(a, out.dtype, "a")
        _req(b, out.dtype, "b")
        if a.shape != out.shape or b.shape != out.shape:
            raise ValueError(f"sum_products: shapes {tuple(a.shape)}, {tuple(b.shape)} do not match "
                             f"the output {tuple(out.shape)}")
    A = (ctypes.c_void_p * 4)(*[a.data_ptr() for _, a, _ in terms])
    B = (ctypes.c_void_p * 4)(*[b.data_ptr() for _, _, b in terms])
    C = (ctypes.c_double * 4)(*[c for c, _, _ in terms])
    dt = {torch.float64: 0, torch.float32: 1}[out.dtype]
    _lib.call("jfx_sum_products", dt, len(terms), A, B, C, _p(out), out.numel(), _s())
    return out


def mul_bcast(X: torch.Tensor, C: torch.Tensor) -> torch.Tensor:
    """``Y[b, ...] = X[b, ...] * C[...]`` (FP64, C broadcast over leading dims):
    the pointwise coefficient product of a non-separable form on the mesh."""
    _req(X, torch.float64, "X")
    _req(C, torch.float64, "C")
    if C.numel() == 0 or X.numel() % C.numel() != 0:
        raise ValueError(f"mul_bcast: {X.numel()} entries are not a whole number of {C.numel()}-entry blocks")
    Y = torch.empty_like(X)
    _lib.call("jfx_mul_bcast_f64", _p(X), _p(C), _p(Y), X.numel(), C.numel(), _s())
    return Y


def div_bcast(X: torch.Tensor, D: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """``out[b, ...] = X[b, ...] / D[...]`` with D broadcast over leading dims."""
    _req(X, X.dtype, "X")
    _req(D, X.dtype, "D")
    out = torch.empty_like(X) if out is None else out
    name = "jfx_div_bcast_f64" if X.dtype == torch.float64 else "jfx_div_bcast_f32"
    _lib.call(name, _p(X), _p(D), _p(out), X.numel(), D.numel(), _s())
    return out


def add_bcast(X: torch.Tensor, D: torch.Tensor, alpha: float = 1.0,
              out: torch.Tensor | None = None) -> torch.Tensor:
    """``out[b, ...] = X[b, ...] + alpha * D[...]`` (FP64, real or complex) with D
    broadcast over leading dims; a real X with a complex D gives a complex result."""
    if X.is_complex() or D.is_complex():
        if not X.is_complex():
            X = to_complex(X)
        if not D.is_complex():
            D = to_complex(D)
        out = torch.empty_like(X) if out is None else out
        add_bcast(torch.view_as_real(X), torch.view_as_real(D), alpha, torch.view_as_real(out))
        return out
    _req(X, torch.float64, "X")
    _req(D, torch.float64, "D")
    if tuple(X.shape[X.ndim - D.ndim:]) != tuple(D.shape):
        raise ValueError(f"add_bcast: trailing shape {tuple(X.shape)} does not end with {tuple(D.shape)}")
    out = torch.empty_like(X) if out is None else out
    if X.numel() == 0:
        return out
    _lib.call("jfx_axpy_bcast_f64", _p(X), _p(D), float(alpha), _p(out), X.numel(), D.numel(), _s())
    return out


def cmul_bcast(X: torch.Tensor, D: torch.Tensor) -> torch.Tensor:
    """``Y[b, ...] = X[b, ...] * D[...]`` (complex128) with D broadcast over leading dims."""
    if not X.is_complex():
        X = to_complex(X.contiguous())
    _req(X, torch.complex128, "X")
    _req(D, torch.complex128, "D")
    Y = torch.empty_like(X)
    _lib.call("jfx_cmul_bcast", _p(X), _p(D), _p(Y), X.numel(), D.numel(), _s())
    return Y


def to_complex(X: torch.Tensor) -> torch.Tensor:
    """Real FP64 array as complex128 (imaginary part zero) through the
    complex-combine kernel's real-input form."""
    _req(X, torch.float64, "X")
    Y = torch.empty(X.shape, dtype=torch.complex128, device=X.device)
    n = X.numel()
    if n:
        Z = torch.cat([X.reshape(1, 1, n), torch.zeros_like(X).reshape(1, 1, n)], 1)
        _lib.call("jfx_cplx_combine", _p(Z), _p(Y), 1, 1, n, 1, _s())
    return Y


# ---------------------------------------------------------------- banded LU


def band_lu_factor(band: torch.Tensor, p: int, q: int) -> torch.Tensor:
    """Factor a (n, p+q+1) by-row band matrix without pivoting.

    Raises ValueError on a zero or non-finite pivot, like
    ``DiaMatrix.lu_factor`` (la/diamatrix.py:461-471).
    """
    _req(band, torch.float64, "band")
    n = band.shape[0]
    lu = torch.empty_like(band)
    st = torch.zeros(1, dtype=torch.int32, device=band.device)
    _lib.call("jfx_band_lu_factor", _p(band), n, p, q, _p(lu), _p(st), _s())
    s = int(st.item())
    if s != 0:
        raise ValueError(f"Zero or non-finite pivot at row {s - 1} in banded LU factorization")
    return lu


def band_lu_factor_batched(band: torch.Tensor, p: int, q: int) -> torch.Tensor:
    """Factor nsys band matrices (nsys, n, p+q+1) without pivoting, one lane
    each (real FP64 or complex128)."""
    nsys, n = band.shape[0], band.shape[1]
    lu = torch.empty_like(band)
    st = torch.zeros(1, dtype=torch.int32, device=band.device)
    if band.is_complex():
        _req(band, torch.complex128, "band")
        _lib.call("jfx_band_lu_factor_batched_z", _p(band), nsys, n, p, q, _p(lu), _p(st), _s())
    else:
        _req(band, torch.float64, "band")
        _lib.call("jfx_band_lu_factor_batched", _p(band), nsys, n, p, q, _p(lu), _p(st), _s())
    s = int(st.item())
    if s != 0:
        raise ValueError(f"Zero or non-finite pivot at row {s - 1} in a batched banded LU factorization")
    return lu


BAND_SOLVE_METHODS = {"auto": 0, "lanes": 1, "wave": 2, "grid": 3}


def band_lu_solve_batched(lu: torch.Tensor, p: int, q: int, X: torch.Tensor, axis: int,
                          method: str = "auto") -> torch.Tensor:
    """Solve in place along ``axis`` of X; the systems run over the other axes
    in C order (one factor per line, the re/im pair of complex X sharing one).
    ``method`` as for ``band_lu_solve`` (real factors; complex factors use
    one lane per line)."""
    if method not in BAND_SOLVE_METHODS:
        raise ValueError(f"band solve: method must be one of {sorted(BAND_SOLVE_METHODS)}, got {method!r}")
    nsys, n = lu.shape[0], lu.shape[1]
    axis = axis % X.ndim
    if X.shape[axis] != n:
        raise ValueError(f"band solve: axis {axis} has length {X.shape[axis]}, matrices are {n}")
    if (X.numel() // n) % nsys:
        raise ValueError(f"band solve: {X.numel() // n} lines is not a multiple of {nsys} systems")
    if lu.is_complex():
        if not X.is_complex():
            raise TypeError("complex factors need a complex right-hand side")
        _req(X, torch.complex128, "X")
        P = math.prod(X.shape[:axis])
        Q = math.prod(X.shape[axis + 1:])
        _lib.call("jfx_band_lu_solve_batched_z", _p(lu), nsys, n, p, q, _p(X), P, Q, _s())
        return X
    qdiv = 1
    Xr = X
    if X.is_complex():
        _req(X, torch.complex128, "X")
        Xr = torch.view_as_real(X)
        qdiv = 2
    _req(Xr, torch.float64, "X")
    P = math.prod(X.shape[:axis])
    Q = math.prod(X.shape[axis + 1:]) * qdiv
    if method == "wave" and max(p, q) > 4:
        raise ValueError(f"band solve: the wavefront solve takes bandwidths <= 4, got p={p}, q={q}")
    _lib.call("jfx_band_lu_solve_batched_mode", _p(lu), nsys, n, p, q, _p(Xr), P, Q, qdiv, BAND_SOLVE_METHODS[method],
              _s())
    return X


def band_lu_solve(lu: torch.Tensor, p: int, q: int, X: torch.Tensor, axis: int, method: str = "auto") -> torch.Tensor:
    """Solve in place along ``axis`` of X with a factored band matrix (a complex
    X is solved through its real view: the same real factor for re and im).

    ``method``: "lanes" runs one lane per line (a sequential sweep), "wave"
    one wavefront per line (rows split over the 64 lanes, p, q <= 4), "grid"
    each line's rows over several workgroups that hand the boundary window on
    (few lines of at least 8192 rows, p, q <= 4), "auto" the grid solve where
    it applies, else the wavefront solve for few long lines and the per-lane
    sweep otherwise."""
    if method not in BAND_SOLVE_METHODS:
        raise ValueError(f"band solve: method must be one of {sorted(BAND_SOLVE_METHODS)}, got {method!r}")
    if X.is_complex():
        _req(X, torch.complex128, "X")
        band_lu_solve(lu, p, q, torch.view_as_real(X), axis % X.ndim, method)
        return X
    _req(X, torch.float64, "X")
    n = lu.shape[0]
    if X.shape[axis] != n:
        raise ValueError(f"band solve: axis {axis} has length {X.shape[axis]}, matrix is {n}")
    if method == "wave" and max(p, q) > 4:
        raise ValueError(f"band solve: the wavefront solve takes bandwidths <= 4, got p={p}, q={q}")
    P = math.prod(X.shape[:axis])
    Q = math.prod(X.shape[axis + 1:])
    if method in ("auto", "grid"):
        nbytes = _lib.load().jfx_band_lu_solve_grid_work_bytes(n, p, q, P, Q)
        if nbytes > 0:
            work = torch.empty(nbytes, dtype=torch.uint8, device=X.device)
            _lib.call("jfx_band_lu_solve_grid", _p(lu), n, p, q, _p(X), P, Q, _p(work), nbytes, _s())
            return X
        if method == "grid":
            raise ValueError(f"band solve: the grid solve takes few lines of >= 8192 rows and p, q <= 4 "
                             f"(n={n}, lines={P * Q}, p={p}, q={q})")
    _lib.call("jfx_band_lu_solve_mode", _p(lu), n, p, q, _p(X), P, Q, BAND_SOLVE_METHODS[method], _s())
    return X


# ---------------------------------------------------------------- dense LU

def dense_lu_factor(A: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """LU with partial pivoting of a square FP64 or complex128 matrix (row
    pivoting on the largest |re| + |im|), blocked over 32-column panels
    (16 complex).  Returns (LU, perm): L unit lower and U in one array, and
    row i of P A = row perm[i] of A.  Raises ValueError on a zero pivot, as
    Matrix.lu_factor does (la/matrix.py:137-167)."""
    if A.ndim != 2 or A.shape[0] != A.shape[1]:
        raise ValueError(f"dense LU needs a square matrix, got shape {tuple(A.shape)}")
    cplx = A.is_complex()
    _req(A, torch.complex128 if cplx else torch.float64, "A")
    n = A.shape[0]
    LU = A.contiguous().clone()
    ipiv = torch.empty(n, dtype=torch.int32, device=A.device)
    perm = torch.empty(n, dtype=torch.int32, device=A.device)
    st = torch.zeros(1, dtype=torch.int32, device=A.device)
    work = torch.empty(n * 32, dtype=torch.float64, device=A.device)  # a column-major copy of one panel
    _lib.call("jfx_dense_lu_factor", int(cplx), _p(LU), n, _p(ipiv), _p(perm), _p(st), _p(work), _s())
    s = int(st.item())
    if s != 0:
        raise ValueError(f"Matrix is singular: zero pivot in LU factorisation (column {s - 1})")
    return LU, perm


def _dense_solve_work(n: int, nrhs: int, like: torch.Tensor) -> torch.Tensor:
    """Work buffer of ``jfx_dense_lu_solve``: n x nrhs values, then
    2 ceil(n / 64) ints of block flags."""
    elt = like.element_size()
    extra = (2 * ((n + 63) // 64) * 4 + elt - 1) // elt
    return torch.empty(n * nrhs + extra, dtype=like.dtype, device=like.device)


def dense_lu_solve(LU: torch.Tensor, perm: torch.Tensor, B: torch.Tensor) -> torch.Tensor:
    """X = A^-1 B for B of shape (n,) or (n, nrhs), with (LU, perm) from
    ``dense_lu_factor``.  A complex B with a real factor is solved as its
    real and imaginary parts; a real B with a complex factor is promoted."""
    n = LU.shape[0]
    if B.shape[0] != n:
        raise ValueError(f"dense LU solve: B has {B.shape[0]} rows, the matrix is {n} x {n}")
    vec = B.ndim == 1
    B2 = B.reshape(n, -1)
    if LU.is_complex():
        B2 = (B2 if B2.is_complex() else to_complex(B2.contiguous())).contiguous()
        _req(B2, torch.complex128, "B")
        X = torch.empty_like(B2)
        W = _dense_solve_work(n, B2.shape[1], B2)
        _lib.call("jfx_dense_lu_solve", 1, _p(LU), n, _p(perm), _p(B2), _p(X), B2.shape[1], _p(W), _s())
    elif B2.is_complex():
        B2 = B2.contiguous()
        _req(B2, torch.complex128, "B")
        Br = torch.view_as_real(B2).reshape(n, -1)  # (n, 2 nrhs): re, im interleaved
        Xr = torch.empty_like(Br)
        W = _dense_solve_work(n, Br.shape[1], Br)
        _lib.call("jfx_dense_lu_solve", 0, _p(LU), n, _p(perm), _p(Br), _p(Xr), Br.shape[1], _p(W), _s())
        X = torch.view_as_complex(Xr.reshape(n, -1, 2))
    else:
        B2 = B2.contiguous()
        _req(B2, torch.float64, "B")
        X = torch.empty_like(B2)
        W = _dense_solve_work(n, B2.shape[1], B2)
        _lib.call("jfx_dense_lu_solve", 0, _p(LU), n, _p(perm), _p(B2), _p(X), B2.shape[1], _p(W), _s())
    return X.reshape(n) if vec else X


# ---------------------------------------------------------------- per-axis contraction


PAR_KEYS = {"f64": "par_f64", "f32": "par_f32"}
PAR_DENSE, PAR_EVAL, PAR_PROJ, PAR_MIX = range(4)  # operator structures of csrc/contract_par.hip


def evaluates_parity(sgn: int = 1) -> tuple:
    """Structure of a (mesh x modes) operator on a symmetric mesh:
    A[M-1-m, k] = sgn (-1)^k A[m, k]."""
    return (PAR_EVAL, sgn, -1, -1)


def projects_parity(sgn: int = 1) -> tuple:
    """Structure of a (modes x mesh) operator: A[m, K-1-k] = sgn (-1)^m A[m, k]."""
    return (PAR_PROJ, sgn, -1, -1)


def mixes_parity(sgn: int = 1, p: int = -1, q: int = -1) -> tuple:
    """Structure of a (modes x modes) operator that couples equal (sgn = 1) or
    opposite (sgn = -1) parities only, with ``p`` lower and ``q`` upper bands
    (-1: all)."""
    return (PAR_MIX, sgn, p, q)


def host_structure(A: np.ndarray) -> tuple | None:
    """:func:`mixes_parity` of a host matrix whose entries vanish exactly on
    every second diagonal, else None."""
    if np.iscomplexobj(A) or A.ndim != 2 or 0 in A.shape or not np.all(np.isfinite(A)):
        return None
    r, c = np.nonzero(A)
    if r.size == 0:
        return None
    d = c - r
    odd = (d & 1).astype(bool)
    if odd.any() and not odd.all():
        return None
    return mixes_parity(-1 if odd.any() else 1, max(0, int(-d.min())), max(0, int(d.max())))


def fragment_values(M: int, K: int, mode: int) -> int:
    """Values of an (M x K) operator's fragments, 0 for sizes that are not taken."""
    return _lib.load().jfx_par_frag_elems(M, K, mode)


class AxisOperator:
    """A constant (M x K) matrix applied along one axis, prepared per precision.

    ``parity``: its structure (:func:`evaluates_parity`, :func:`projects_parity`,
    :func:`mixes_parity`), which FP64 and FP32 contractions use to halve their
    products; the caller vouches for it up to rounding.  ``once``: for a single
    product, nothing is prepared for later ones.

    ``f64`` uses the FP64 matrix; ``f32`` an FP32 copy; ``bf16x3``/``bf16x6``
    2/3 bf16 float slices; ``ozakiS`` S fixed-point digit slices with
    power-of-two row scales; ``i8xS`` S balanced int8 digit slices with
    power-of-two row scales (FP64 data, int8 MFMA, exact integer sums).  Preparations are cached on the object, like the
    reference caches factorizations on its matrix objects.
    """

    def __init__(self, A: torch.Tensor, parity: tuple | None = None, once: bool = False):
        if A.dtype != torch.float64:
            A = A.to(torch.float64)
        self.A64 = A.contiguous()
        self.M, self.K = self.A64.shape
        self.parity = parity
        self.once = once
        self._made_on = _stream_id() if self.A64.is_cuda else None  # the stream that A64 is ordered on
        self._prep: dict[str, tuple] = {}

    def t(self) -> "AxisOperator":
        """The transposed operator, its structure transposed with it."""
        par = self.parity
        if par is not None:
            mode, sgn, p, q = par
            par = ({PAR_EVAL: PAR_PROJ, PAR_PROJ: PAR_EVAL, PAR_MIX: PAR_MIX}[mode], sgn, q, p)
        return AxisOperator(self.A64.t().contiguous(), par)

    def fragments(self, prec: str, peers=()):
        """MFMA fragments of ``csrc/contract_par.hip`` and their structure
        ``(fragments, mode, sgn, p, q)`` for ``prec`` f64 or f32, or None where
        the sizes are not taken.  A first use inside a graph capture gives None
        too: the capture would record the preparation instead of running it.
        Those of a ``once`` operator serve the current stream's next product and
        are not kept, so nothing waits for them.  ``peers``: operators of the same
        pass, prepared with this one if they have a structure."""
        key = PAR_KEYS[prec]
        fr = self._prep.get(key, 0)
        if fr != 0:
            return fr
        if not self.once:
            prepare_fragments((self, *(o for o in peers if type(o) is AxisOperator and o.parity is not None)), prec)
            return self._prep.get(key)
        mode, sgn, p, q = self.parity or (PAR_DENSE, 1, -1, -1)
        n = fragment_values(self.M, self.K, mode)
        if n == 0:
            return None
        f = torch.empty(n, dtype=io_dtype(prec), device=self.A64.device)
        _lib.call("jfx_par_prepare", 0 if prec == "f64" else 1, _p(self.A64), self.M, self.K, mode, sgn, _p(f), _s())
        return f, mode, sgn, p, q

    def _padded(self):
        """Zero-pad K to a multiple of 32 (the slice row stride the kernels read)."""
        Kp = (self.K + 31) // 32 * 32
        if Kp == self.K:
            return self.A64, Kp
        Ap = torch.zeros((self.M, Kp), dtype=torch.float64, device=self.A64.device)
        Ap[:, :self.K] = self.A64
        return Ap, Kp

    def prepared(self, prec: str):
        if prec in self._prep:
            return self._prep[prec]
        A = self.A64
        if prec == "f64":
            r = (A,)
        elif prec == "f32":
            r = (cast(A, torch.float32),)
        elif prec in ("bf16x3", "bf16x6"):
            S = 2 if prec == "bf16x3" else 3
            Ap, Kp = self._padded()
            sl = torch.empty((S, self.M, Kp), dtype=torch.int16, device=A.device)
            _lib.call("jfx_split_matrix", _p(Ap), self.M, Kp, 0, S, _p(sl), _p(None), _s())
            r = (sl, S)
        elif prec.startswith("ozaki"):
            S = int(prec[5:])
            Ap, Kp = self._padded()
            sl = torch.empty((S, self.M, Kp), dtype=torch.int16, device=A.device)
            rs = torch.empty(self.M, dtype=torch.float64, device=A.device)
            _lib.call("jfx_split_matrix", _p(Ap), self.M, Kp, 1, S, _p(sl), _p(rs), _s())
            r = (sl, rs, S)
        elif prec.startswith("i8x") and prec in PRECISIONS:
            S = int(prec[3:])
            Kp = (self.K + 63) // 64 * 64
            sl = torch.empty((S, self.M, Kp), dtype=torch.int8, device=A.device)
            ex = torch.empty(self.M, dtype=torch.int32, device=A.device)
            _lib.call("jfx_split_matrix_i8", _p(A), self.M, self.K, S, _p(sl), _p(ex), _s())
            r = (sl, ex, S)
        else:
            raise ValueError(f"unknown precision {prec!r}; expected one of {PRECISIONS}")
        self._prep[prec] = r
        return r


def prepare_fragments(ops, prec: str = "f64") -> None:
    """Cut the fragments of every operator in ``ops`` that has none yet, in one
    launch with one wait (20 us for one operator, 28 for four; most of it is the
    wait).  Inside a graph capture this does nothing, see
    :meth:`AxisOperator.fragments`."""
    key = PAR_KEYS[prec]
    todo = []
    for op in ops:
        if type(op) is AxisOperator and not op.once and key not in op._prep and all(op is not o for o, _, _ in todo):
            par = op.parity or (PAR_DENSE, 1, -1, -1)
            n = fragment_values(op.M, op.K, par[0])
            if n == 0:
                op._prep[key] = None
            else:
                todo.append((op, par, n))
    if not todo or torch.cuda.is_current_stream_capturing():
        return
    # what is kept must not be cut from a matrix that another stream is still computing
    for stream in {op._made_on for op, _, _ in todo} - {_stream_id()}:
        _wait_for(stream)
    n = len(todo)
    frags = [torch.empty(m, dtype=io_dtype(prec), device=op.A64.device) for op, _, m in todo]
    A = (ctypes.c_void_p * n)(*[op.A64.data_ptr() for op, _, _ in todo])
    F = (ctypes.c_void_p * n)(*[f.data_ptr() for f in frags])
    shape = (ctypes.c_int * (4 * n))(*[v for op, par, _ in todo for v in (op.M, op.K, par[0], par[1])])
    # complete before they are published: the next use may be on another stream
    _lib.call("jfx_par_prepare_many", 0 if prec == "f64" else 1, n, A, shape, F, 1, _s())
    for (op, par, _), f in zip(todo, frags):
        op._prep[key] = (f, *par)


def io_dtype(prec: str) -> torch.dtype:
    return torch.float32 if prec in ("f32", "bf16x3", "bf16x6") else torch.float64


class ComplexAxisOperator:
    """A constant complex (M x K) matrix applied along one axis (FP64).

    Kept as the stacked real (2M x K) operator [Re A; Im A]: one real MFMA
    contraction over the real view of X, then ``jfx_cplx_combine`` forms
    ``Re + i Im`` of the result.
    """

    is_complex = True

    def __init__(self, A: torch.Tensor, once: bool = False):
        A = A.to(torch.complex128)
        self.M, self.K = A.shape
        self.A = A.contiguous()
        self.stacked = AxisOperator(torch.cat([A.real, A.imag], 0).contiguous(), once=once)

    def prepared(self, prec: str):
        if prec != "f64":
            raise ValueError("complex operators are applied in f64 only")
        return self.stacked.prepared(prec)


def _apply_complex(op: ComplexAxisOperator, X: torch.Tensor, axis: int, peers=()) -> torch.Tensor:
    axis = axis % X.ndim
    if X.shape[axis] != op.K:
        raise ValueError(f"apply_along: axis {axis} has length {X.shape[axis]}, operator expects {op.K}")
    P = math.prod(X.shape[:axis])
    Q = math.prod(X.shape[axis + 1:])
    shape = list(X.shape)
    shape[axis] = op.M
    Y = torch.empty(shape, dtype=torch.complex128, device=X.device)
    if X.is_complex():
        _req(X, torch.complex128, "X")
        Z = apply_along(op.stacked, torch.view_as_real(X).reshape(P, op.K, 2 * Q), 1, peers=peers)
        _lib.call("jfx_cplx_combine", _p(Z), _p(Y), P, op.M, Q, 0, _s())
    else:
        _req(X, torch.float64, "X")
        Z = apply_along(op.stacked, X.reshape(P, op.K, Q), 1, peers=peers)
        _lib.call("jfx_cplx_combine", _p(Z), _p(Y), P, op.M, Q, 1, _s())
    return Y


def _use_fragments(op: AxisOperator, P: int, Q: int, prec: str) -> bool:
    """Whether FP64/FP32 contractions of ``op`` run from MFMA fragments.

    Operators with a structure: always.  Others: in layouts that the kernels for the
    plain matrix read badly, where (us, plain / fragments) the fragments are the
    faster ones.  A workgroup takes all rows of its columns, so many rows want many
    columns; K beyond ``kmax`` leaves room for 16 columns and little overlap, which
    few columns do not mind.  FP64, 65536 columns: 128 x 192 142 / 138, 200 x 200 213 /
    210, 224 x 222 243 / 340, 100 x 400 284 / 394, 512 x 100 295 / 193; 4096 columns: 224
    x 222 47 / 41, 100 x 400 76 / 44, 512 x 100 27 / 48, 512 x 256 58 / 103.  FP32, 65536:
    256 x 254 150 / 143, 300 x 298 213 / 250, 100 x 400 122 / 189, 512 x 256 300 / 261;
    4096: 100 x 400 59 / 27, 400 x 200 35 / 41.

    For a single product they have to be cut first, which pays from 32 columns a row
    on: 64 x 64 on 2048 columns 14.3 / 10.1; 256 x 64 on 2048 16.3 / 22.2, on 32768
    50.7 / 38.9; 512 x 128 on 2048 28.7 / 63.7, on 32768 149 / 108; 1 x 50 on 1000 11.7 /
    9.7, on 1e6 634 / 116."""
    if op.parity is None:
        if Q == 1 or Q % 64 == 0:
            return False
        kmax, few = (208, 8192) if prec == "f64" else (256, 16384)
        if op.M <= 320:
            if op.K > kmax and P * Q > min(2 * few, 320 * few // op.M):
                return False
        elif op.K > kmax or P * Q <= few:
            return False
    return not op.once or P * Q >= 32 * op.M


def apply_along(op: AxisOperator, X: torch.Tensor, axis: int, prec: str = "f64",
                out: torch.Tensor | None = None, peers=()) -> torch.Tensor:
    """``Y = A`` applied along ``axis`` of X: Y[p, m, q] = sum_k A[m, k] X[p, k, q].

    A complex X (FP64 only) is contracted through its real view (the re/im
    pair rides along the trailing axis); a :class:`ComplexAxisOperator`
    gives a complex result.  ``peers``: see :meth:`AxisOperator.fragments`.
    """
    if getattr(op, "is_complex", False):
        if prec != "f64" or out is not None:
            raise ValueError("complex operators are applied in f64 without an out= tensor")
        return _apply_complex(op, X, axis, peers)
    if X.is_complex():
        if prec != "f64":
            raise ValueError("complex arrays are transformed in f64 only")
        _req(X, torch.complex128, "X")
        axis = axis % X.ndim
        shape = list(X.shape)
        shape[axis] = op.M
        Y = torch.empty(shape, dtype=torch.complex128, device=X.device) if out is None else out
        apply_along(op, torch.view_as_real(X), axis, "f64", out=torch.view_as_real(Y), peers=peers)
        return Y
    dt = io_dtype(prec)
    _req(X, dt, "X")
    shape = list(X.shape)
    axis = axis % len(shape)
    K = shape[axis]
    if K != op.K:
        raise ValueError(f"apply_along: axis {axis} has length {K}, operator expects {op.K}")
    P = Q = 1
    for n in shape[:axis]:
        P *= n
    for n in shape[axis + 1:]:
        Q *= n
    shape[axis] = op.M
    Y = torch.empty(shape, dtype=dt, device=X.device) if out is None else out
    if out is not None:
        _req(out, dt, "out")
        if list(out.shape) != shape:
            raise ValueError("apply_along: bad out shape")
    if prec in ("f64", "f32") and P * Q > 0 and _use_fragments(op, P, Q, prec):
        fr = op.fragments(prec, peers)
        if fr is not None:
            _lib.call("jfx_contract_par", 0 if prec == "f64" else 1, _p(fr[0]), op.M, K, fr[1], fr[2], fr[3], fr[4],
                      _p(X), _p(Y), P, Q, _s())
            return Y
    prep = op.prepared(prec)
    if prec == "f64":
        _lib.call("jfx_contract_f64", _p(prep[0]), op.M, K, _p(X), _p(Y), P, Q, _s())
    elif prec == "f32":
        _lib.call("jfx_contract_f32", _p(prep[0]), op.M, K, _p(X), _p(Y), P, Q, _s())
    elif prec in ("bf16x3", "bf16x6"):
        _lib.call("jfx_contract_bf16x", _p(prep[0]), prep[1], op.M, K, _p(X), _p(Y), P, Q, _s())
    elif prec.startswith("i8x"):
        if op.M > 128 or K > 128 or not (Q == 1 or Q % 64 == 0) or (Q == 1 and K % 2):
            raise ValueError(f"precision {prec}: needs M, K <= 128 and a trailing size of 1 (K even) or a "
                             f"multiple of 64; got M={op.M}, K={K}, trailing size {Q}")
        _lib.call("jfx_contract_i8", _p(prep[0]), _p(prep[1]), prep[2], op.M, K, _p(X), _p(Y), P, Q, _s())
    else:
        _lib.call("jfx_contract_ozaki", _p(prep[0]), _p(prep[1]), prep[2], op.M, K, _p(X), _p(Y), P, Q,
                  _s())
    return Y


def weak_laplacian(B: AxisOperator, D: AxisOperator, TB: AxisOperator, TD: AxisOperator, k: torch.Tensor,
                   U: torch.Tensor) -> torch.Tensor | None:
    """``TD (k * (D U B^T)) TB^T + TB (k * (B U D^T)) TD^T`` per slab of U (FP64) in one
    launch (csrc/weak_par.hip), or None where its operators do not fit: B, D
    evaluate a parity basis and its derivative, TB, TD project, all up to 128."""
    n, Q = B.K, B.M
    if max(n, Q) > 128 or any(o.parity is None or o.parity[0] != md or (o.M, o.K) != sz for o, md, sz in (
            (B, PAR_EVAL, (Q, n)), (D, PAR_EVAL, (Q, n)), (TB, PAR_PROJ, (n, Q)), (TD, PAR_PROJ, (n, Q)))):
        return None
    fr = _kept_fragments((B, D, TB, TD))
    if fr is None:
        return None
    _req(U, torch.float64, "U")
    _req(k, torch.float64, "k")
    nb = math.prod(U.shape[:-2])
    if tuple(U.shape[-2:]) != (n, n) or tuple(k.shape) != tuple(U.shape[:-2]) + (Q, Q):
        raise ValueError(f"weak_laplacian: U {tuple(U.shape)} and k {tuple(k.shape)} do not fit n = {n}, Q = {Q}")
    Y = torch.empty_like(U)
    _lib.call("jfx_weak_par", _p(fr[0][0]), fr[0][2], _p(fr[1][0]), fr[1][2], _p(fr[2][0]), fr[2][2], _p(fr[3][0]),
              fr[3][2], n, Q, _p(U), _p(k), _p(Y), nb, _s())
    return Y


def quad_ok(B0, D0, B1, D1, S0, S1) -> bool:
    """Whether the fused quadratic term (csrc/quad_par.hip) takes these operators:
    B, D evaluate a parity basis and its derivative, S projects, per axis."""
    ops = (B0, D0, B1, D1, S0, S1)
    if any(type(o) is not AxisOperator or o.parity is None for o in ops):
        return False
    n0, Q0, n1, Q1 = B0.K, B0.M, B1.K, B1.M
    if any((o.M, o.K, o.parity[0]) != want for o, want in zip(ops, (
            (Q0, n0, PAR_EVAL), (Q0, n0, PAR_EVAL), (Q1, n1, PAR_EVAL), (Q1, n1, PAR_EVAL), (n0, Q0, PAR_PROJ),
            (n1, Q1, PAR_PROJ)))) or S0.parity[1] != 1:
        return False
    if _lib.load().jfx_quad_par_ok(n0, Q0, n1, Q1) != 1:
        return False
    prepare_fragments(ops)
    return all(o.fragments("f64") is not None for o in ops)


def quadratic_term(B0, D0, B1, D1, S0, S1, coefficients, U: torch.Tensor) -> torch.Tensor:
    """``S0 w S1^T`` over the last two axes of U (FP64 or FP32, FP64 arithmetic) with
    w = c0 u u + c1 u u_x + c2 u u_y + c3 u_x u_x + c4 u_x u_y + c5 u_y u_y on the mesh
    (operators as :func:`quad_ok` takes them)."""
    _req(U, torch.float32 if U.dtype == torch.float32 else torch.float64, "U")
    if tuple(U.shape[-2:]) != (B0.K, B1.K):
        raise ValueError(f"quadratic_term: U {tuple(U.shape)} does not end with {(B0.K, B1.K)}")
    fr = [o.fragments("f64") for o in (B0, D0, B1, D1, S0, S1)]
    F = (ctypes.c_void_p * 6)(*[f[0].data_ptr() for f in fr])
    sgn = (ctypes.c_int * 6)(*[f[2] for f in fr])
    c = (ctypes.c_double * 6)(*[float(v) for v in coefficients])
    Y = torch.empty_like(U)
    _lib.call("jfx_quad_par", 0 if U.dtype == torch.float64 else 1, F, sgn, c, B0.K, B0.M, B1.K, B1.M, _p(U), _p(Y),
              math.prod(U.shape[:-2]), _s())
    return Y


PLANE_PRECISIONS = ("f64", "bf16x6", "i8x5", "i8x6")


_NUM_CUS = None


def num_cus() -> int:
    """Compute units of the current device (cached)."""
    global _NUM_CUS
    if _NUM_CUS is None:
        _NUM_CUS = torch.cuda.get_device_properties(device()).multi_processor_count
    return _NUM_CUS


def plane_ok(op0: AxisOperator, op1: AxisOperator, prec: str) -> bool:
    if getattr(op0, "is_complex", False) or getattr(op1, "is_complex", False):
        return False
    if prec.startswith("i8x") and op1.K % 2:
        return False  # the int8 plane kernel reads rows in 16-byte pairs
    return prec in PLANE_PRECISIONS and max(op0.M, op0.K, op1.M, op1.K) <= 128


def _kept_fragments(ops):
    """FP64 fragments of every operator, cut together on first use; None if one has none."""
    fr = [o._prep.get("par_f64") for o in ops]
    if None in fr:
        prepare_fragments(ops)
        fr = [o._prep.get("par_f64") for o in ops]
    return None if None in fr else fr


def _slab_fragments(ops):
    """FP64 fragments of structured operators for the fused slab kernels
    (csrc/plane_par.hip): one structure, at most 128 rows and columns; else None."""
    for o in ops:
        if type(o) is not AxisOperator or o.parity is None or o.M > 128 or o.K > 128 or \
                o.parity[0] != ops[0].parity[0]:
            return None
    return _kept_fragments(ops)


def slab_pays(op0, op1, nslabs: int) -> bool | None:
    """Whether ``nslabs`` slabs run faster through the fused FP64 slab kernel than
    axis by axis; None where that kernel does not take the operators.  A slab is
    one workgroup's work: up to 64 x 128 values always (us, slab / per axis: one of 64
    x 64 10.2 / 14.9, 256 12.0 / 16.5; one of 128 x 64 14.1 / 16.5, one of 128 x 20
    10.2 / 16.1, 100 of 80 x 80 16.8 / 16.8), larger ones when they occupy half the CUs
    (96 x 96: 16 slabs 18.4 / 16.3, 128 20.0 / 23.3; 128 x 128: 16 27 / 17, 128 29 / 34,
    256 33 / 44)."""
    if any(type(o) is not AxisOperator or o.parity is None or max(o.M, o.K) > 128 for o in (op0, op1)) or \
            op0.parity[0] != op1.parity[0]:
        return None
    return max(op0.M, op0.K) * max(op1.M, op1.K) <= 64 * 128 or 2 * nslabs >= num_cus()


def plane_fd_par_ok(ops) -> bool:
    """The fused FP64 solve of operators that couple equal parities applies
    (W0, W1, V0, V1 square, up to 128, the two axes of any sizes)."""
    return all(type(o) is AxisOperator and o.parity == (PAR_MIX, 1, -1, -1) and o.M == o.K <= 128 for o in ops) and \
        ops[0].M == ops[2].M and ops[1].M == ops[3].M


def plane_fd_ok(ops, prec: str) -> bool:
    """The fused 2D solve applies: four real n x n operators, n <= 64 (FP64) or 128 (bf16x6)."""
    if prec not in ("f64", "bf16x6"):
        return False
    if any(type(o) is not AxisOperator for o in ops):
        return False
    n = ops[0].M
    if any(o.M != n or o.K != n for o in ops):
        return False
    return n <= (64 if prec == "f64" else 128)


def plane_fd(W0: AxisOperator, W1: AxisOperator, V0: AxisOperator, V1: AxisOperator, X: torch.Tensor,
             E: torch.Tensor, prec: str = "f64", scale: torch.Tensor | None = None) -> torch.Tensor:
    """``Y[b] = V0 ((W0 X[b] W1^T) / E) V1^T`` over the last two axes in one kernel,
    times ``scale[b]`` if given (FP64 operators that couple equal parities)."""
    dt = io_dtype(prec)
    _req(X, dt, "X")
    _req(E, dt, "E")
    if prec == "f64" and plane_fd_par_ok([W0, W1, V0, V1]):
        fr = _slab_fragments([W0, W1, V0, V1])
        if fr is not None:
            shape = (W0.M, W1.M)
            if tuple(X.shape[-2:]) != shape or tuple(E.shape) != shape:
                raise ValueError("plane_fd: operators, array or divisor do not fit the fused solve")
            Y = torch.empty_like(X)
            B = math.prod(X.shape[:-2])
            if scale is not None:
                _req(scale, torch.float64, "scale")
                if scale.numel() != B:
                    raise ValueError(f"plane_fd: {scale.numel()} scales for {B} slabs")
            _lib.call("jfx_plane_fd_par", _p(fr[0][0]), _p(fr[1][0]), _p(fr[2][0]), _p(fr[3][0]), _p(X), _p(Y), _p(E),
                      _p(scale), B, W0.M, W1.M, _s())
            return Y
    if scale is not None:
        raise ValueError("plane_fd: scale needs FP64 operators that couple equal parities")
    n = W0.M
    if not plane_fd_ok([W0, W1, V0, V1], prec) or tuple(X.shape[-2:]) != (n, n) or tuple(E.shape) != (n, n):
        raise ValueError("plane_fd: operators, array or divisor do not fit the fused solve")
    B = math.prod(X.shape[:-2])
    Y = torch.empty_like(X)
    if prec == "f64":
        _lib.call("jfx_plane_fd", 0, _p(W0.A64), _p(W1.A64), _p(V0.A64), _p(V1.A64), _p(None), _p(None), _p(None),
                  _p(None), _p(X), _p(Y), _p(E), B, n, _s())
    else:
        s = [o.prepared("bf16x6")[0] for o in (W0, W1, V0, V1)]
        _lib.call("jfx_plane_fd", 1, _p(None), _p(None), _p(None), _p(None), _p(s[0]), _p(s[1]), _p(s[2]), _p(s[3]),
                  _p(X), _p(Y), _p(E), B, n, _s())
    return Y


def plane(op0: AxisOperator, op1: AxisOperator, X: torch.Tensor, prec: str = "f64",
          epi: tuple | None = None, alpha: float = 1.0, out: torch.Tensor | None = None,
          accumulate: bool = False) -> torch.Tensor:
    """``Y[b] = alpha A0 X[b] A1^T`` over the last two axes of X in one kernel
    (optionally ``/ E`` or ``* E`` with ``epi=("div"|"mul", E)``, or ``* E[b]`` with
    ``epi=("mul_each", E)``); with ``accumulate`` the result is added to ``out``."""
    dt = io_dtype(prec)
    _req(X, dt, "X")
    if X.shape[-2] != op0.K or X.shape[-1] != op1.K:
        raise ValueError("plane: operator/array shape mismatch")
    B = math.prod(X.shape[:-2])
    shape = X.shape[:-2] + (op0.M, op1.M)
    if out is None:
        if accumulate:
            raise ValueError("plane: accumulate needs out=")
        Y = torch.empty(shape, dtype=dt, device=X.device)
    else:
        _req(out, dt, "out")
        if tuple(out.shape) != tuple(shape):
            raise ValueError("plane: bad out shape")
        if out.data_ptr() == X.data_ptr():
            raise ValueError("plane: out must not alias X")
        Y = out
    mode, E = 0, None
    if epi is not None:
        mode = {"div": 1, "mul": 2, "mul_each": 3}[epi[0]]
        E = epi[1]
        _req(E, dt, "E")
        if tuple(E.shape) != (tuple(shape) if mode == 3 else (op0.M, op1.M)):
            raise ValueError("plane: epilogue shape mismatch")
        if mode == 3 and (prec != "f64" or slab_pays(op0, op1, B) is None):
            raise ValueError("plane: a factor per slab needs FP64 operators with decoupled parities")
    acc = 1 if accumulate else 0
    if prec.startswith("i8x"):
        if mode or accumulate or alpha != 1.0:
            raise ValueError("plane: the int8 path has no epilogue, scale or accumulation")
        if not plane_ok(op0, op1, prec):
            raise ValueError(f"plane: precision {prec} needs dims <= 128 and an even last axis")
        p0, p1 = op0.prepared(prec), op1.prepared(prec)
        _lib.call("jfx_plane_i8", _p(p0[0]), _p(p0[1]), _p(p1[0]), _p(p1[1]), p0[2], _p(X), _p(Y), B, op0.M, op0.K,
                  op1.M, op1.K, _s())
        return Y
    if prec == "f64":
        fr = _slab_fragments((op0, op1))
        if fr is not None:
            (f0, md, s0, p0, q0), (f1, _, s1, p1, q1) = fr
            _lib.call("jfx_plane_par", md, _p(f0), op0.M, op0.K, s0, p0, q0, _p(f1), op1.M, op1.K, s1, p1, q1, _p(X),
                      _p(Y), _p(E), mode, float(alpha), acc, B, _s())
            return Y
        if mode == 3:  # unprepared operators inside a graph capture
            return lincomb([(1.0, mul_bcast(plane(op0, op1, X, prec, alpha=alpha), E))], Y, accumulate)
        _lib.call("jfx_plane_contract", 0, _p(op0.A64), _p(op1.A64), _p(None), _p(None), _p(X), _p(Y), _p(E),
                  mode, float(alpha), acc, B, op0.M, op0.K, op1.M, op1.K, _s())
    else:
        s0, s1 = op0.prepared("bf16x6")[0], op1.prepared("bf16x6")[0]
        _lib.call("jfx_plane_contract", 1, _p(None), _p(None), _p(s0), _p(s1), _p(X), _p(Y), _p(E),
                  mode, float(alpha), acc, B, op0.M, op0.K, op1.M, op1.K, _s())
    return Y
