// Quadratic nonlinear term of 2D Galerkin time stepping in one launch:
//     Y[b] = S0 w S1^T,   w = sum of c_fg f g over products of f, g in {u, u_x, u_y},
//     u = B0 U[b] B1^T,   u_x = D0 U[b] B1^T,   u_y = B0 U[b] D1^T
// with B, D (Q x n) a parity basis and its first derivative on a padded Gauss mesh
// and S (n x Q) the weighted projection, per axis (structures and fragments:
// contract_par.hip).  FP64 arithmetic; U and Y in FP64 or FP32.
//
// Axis by axis this is five evaluations, a pointwise pass and two projections that
// move about 1 GB through HBM for 256 problems of 126 x 126 on 192 x 192 meshes.
// Here one workgroup takes a problem and walks strips of 16 mesh points along axis
// 1 together with their 16 mirror images; the mesh fields never leave the CU:
//   1  T = U B1^T, T' = U D1^T on the strip (32 columns)         registers -> LDS
//   2  u, u_x, u_y on 16 mesh points of axis 0 and their mirror images, the
//      products, and their sums and differences under the mirror registers -> LDS
//   3  s = S0 w, 32 columns                                       registers -> LDS
//   4  Y += s S1^T, accumulated in registers over the strips
// U comes from L2 in every strip.  What bounds it: FP64 products (the strip's four
// steps are 584 MFMAs per SIMD, 93 us for that problem) with four barriers a strip;
// measured 173 us for 256 problems, axis by axis 328 us (FP32 in and out, with
// bf16x6 contractions axis by axis: 163 against 181 us).
#include "par_blocks.h"

namespace jfx {

struct QuadOp {
  const double* f;      // fragments [part][rb][s][64]
  int M, K, S, nrb, sgn;
};
bool par_shape(int M, int K, int mode, int& S, int& nrb);

struct QuadMap {
  QuadOp b0, d0, b1, d1, s0, s1;
  double c[6];  // u u, u u_x, u u_y, u_x u_x, u_x u_y, u_y u_y
};

constexpr int QLT = 40;  // LDS row strides: T and w are read 16 columns wide (8 mod 16) ...
constexpr int QLS = 34;  // ... s 16 rows deep (2 mod 4)
constexpr int QOUT = 3;  // 16 x 16 blocks of Y (both parities) per wave

__host__ __device__ constexpr int quad_pad(int n) { return (n + 15) & ~15; }
static size_t quad_lds(const QuadMap& m) {
  return ((size_t)2 * quad_pad(m.b0.K) + 2 * 16 * m.b0.nrb) * QLT * sizeof(double);
}

template <typename TIO, int NW>
__global__ __launch_bounds__(64 * NW) void quad_par_kernel(const TIO* __restrict__ U, TIO* __restrict__ Y, QuadMap qm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int n0 = qm.b0.K, n1 = qm.b1.K, R0 = quad_pad(n0), nxb = qm.b0.nrb, nst = qm.b1.nrb;
  double* T = reinterpret_cast<double*>(smem);
  double* T2 = T + R0 * QLT;
  double* W = T2 + R0 * QLT;            // w summed over the mirror image ...
  double* W2 = W + 16 * nxb * QLT;      // ... and the difference
  double* s = T;                        // after step 2 (R0 * QLS <= R0 * QLT)
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long b = blockIdx.x;
  const TIO* Ub = U + b * n0 * n1;
  const int nmc = qm.s1.nrb, nout = (R0 >> 4) * nmc;
  v4d out[QOUT][2];
#pragma unroll
  for (int t = 0; t < QOUT; ++t) out[t][0] = out[t][1] = v4d{0, 0, 0, 0};
  const double sB1 = qm.b1.sgn, sD1 = qm.d1.sgn, sB0 = qm.b0.sgn, sD0 = qm.d0.sgn;
  const double c0 = qm.c[0], c1 = qm.c[1], c2 = qm.c[2], c3 = qm.c[3], c4 = qm.c[4], c5 = qm.c[5];

#pragma unroll 1
  for (int st = 0; st < nst; ++st) {
    // (lane indices are taken anew in every step, see own_lane)
    // ---- 1: T, T' on the strip; rows past n0 are copies of the last (operators past K are zero)
#pragma unroll 1
    for (int rb = w; rb < (R0 >> 4); rb += NW) {
      const int lane = own_lane(), kk = lane >> 4, cl = lane & 15;
      const int S = qm.b1.S, i = 16 * rb + cl;
      const TIO* row = Ub + (i < n0 ? i : n0 - 1) * n1;
      const double* pb = qm.b1.f + (st * S) * 64 + lane;
      const double* pd = qm.d1.f + (st * S) * 64 + lane;
      const int po = nst * S * 64;  // odd part
      v4d be = {0, 0, 0, 0}, bo = be, de = be, dq = be;
      double x[2][2], f[2][4], xn[2][2], fn[2][4];
      auto ld = [&](int s0, double(&xv)[2][2], double(&fv)[2][4]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int k = 8 * (s0 + u) + 2 * kk;
          xv[u][0] = row[k < n1 ? k : n1 - 1];
          xv[u][1] = row[k + 1 < n1 ? k + 1 : n1 - 1];
          fv[u][0] = pb[(s0 + u) * 64];
          fv[u][1] = pb[po + (s0 + u) * 64];
          fv[u][2] = pd[(s0 + u) * 64];
          fv[u][3] = pd[po + (s0 + u) * 64];
        }
      };
      ld(0, x, f);
#pragma unroll 1
      for (int s0 = 0; s0 < S; s0 += 2) {
        ld(s0 + 2 < S ? s0 + 2 : s0, xn, fn);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          be = mfma_f64(x[u][0], f[u][0], be);
          bo = mfma_f64(x[u][1], f[u][1], bo);
          de = mfma_f64(x[u][0], f[u][2], de);
          dq = mfma_f64(x[u][1], f[u][3], dq);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          x[u][0] = xn[u][0];
          x[u][1] = xn[u][1];
#pragma unroll
          for (int h = 0; h < 4; ++h) f[u][h] = fn[u][h];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = (16 * rb + mfma16_row_f64(lane, r)) * QLT + cl;
        T[o] = be[r] + bo[r];
        T[o + 16] = sB1 * (be[r] - bo[r]);
        T2[o] = de[r] + dq[r];
        T2[o + 16] = sD1 * (de[r] - dq[r]);
      }
    }
    __syncthreads();
    // ---- 2: the fields and w on 16 points of axis 0 and their mirror images
#pragma unroll 1
    for (int it = w; it < 2 * nxb; it += NW) {
      const int lane = own_lane(), kk = lane >> 4, cl = lane & 15;
      const int c = 16 * (it & 1) + cl, xb = it >> 1, S = qm.b0.S;
      const double* pb = qm.b0.f + (xb * S) * 64 + lane;
      const double* pd = qm.d0.f + (xb * S) * 64 + lane;
      const int po = nxb * S * 64;
      v4d ue = {0, 0, 0, 0}, uo = ue, xe = ue, xo = ue, ye = ue, yo = ue;
      double f[4], fn[4];
      auto ld = [&](int s0, double(&fv)[4]) {
        fv[0] = pb[s0 * 64];
        fv[1] = pb[po + s0 * 64];
        fv[2] = pd[s0 * 64];
        fv[3] = pd[po + s0 * 64];
      };
      ld(0, f);
      const double *t1 = T + 2 * kk * QLT + c, *t2 = T2 + 2 * kk * QLT + c;
#pragma unroll 2
      for (int s0 = 0; s0 < S; ++s0) {
        ld(s0 + 1 < S ? s0 + 1 : s0, fn);
        const double te = t1[0], to = t1[QLT], ge = t2[0], go = t2[QLT];
        t1 += 8 * QLT;
        t2 += 8 * QLT;
        ue = mfma_f64(f[0], te, ue);
        uo = mfma_f64(f[1], to, uo);
        xe = mfma_f64(f[2], te, xe);
        xo = mfma_f64(f[3], to, xo);
        ye = mfma_f64(f[0], ge, ye);
        yo = mfma_f64(f[1], go, yo);
#pragma unroll
        for (int h = 0; h < 4; ++h) f[h] = fn[h];
      }
      auto quad = [&](double u, double ux, double uy) {
        return u * (c0 * u + (c1 * ux + c2 * uy)) + (ux * (c3 * ux + c4 * uy) + c5 * (uy * uy));
      };
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double wp = quad(ue[r] + uo[r], xe[r] + xo[r], ye[r] + yo[r]);
        const double wm = quad(sB0 * (ue[r] - uo[r]), sD0 * (xe[r] - xo[r]), sB0 * (ye[r] - yo[r]));
        const int o = (16 * xb + mfma16_row_f64(lane, r)) * QLT + c;
        W[o] = wp + wm;
        W2[o] = wp - wm;
      }
    }
    __syncthreads();
    // ---- 3: s = S0 w
#pragma unroll 1
    for (int it = w; it < 2 * qm.s0.nrb; it += NW) {
      const int lane = own_lane(), kk = lane >> 4, cl = lane & 15;
      const int c = 16 * (it & 1) + cl, mb = it >> 1, S = qm.s0.S;
      const double* p = qm.s0.f + (mb * S) * 64 + lane;
      const int po = qm.s0.nrb * S * 64;
      v4d e = {0, 0, 0, 0}, o = e;
      double f[2][2], fn[2][2];
      auto ld = [&](int s0, double(&fv)[2][2]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          fv[u][0] = p[(s0 + u) * 64];
          fv[u][1] = p[po + (s0 + u) * 64];
        }
      };
      ld(0, f);
      const double *t1 = W + kk * QLT + c, *t2 = W2 + kk * QLT + c;
#pragma unroll 2
      for (int s0 = 0; s0 < S; s0 += 2) {
        ld(s0 + 2 < S ? s0 + 2 : s0, fn);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          e = mfma_f64(f[u][0], t1[4 * u * QLT], e);
          o = mfma_f64(f[u][1], t2[4 * u * QLT], o);
        }
        t1 += 8 * QLT;
        t2 += 8 * QLT;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f[u][0] = fn[u][0];
          f[u][1] = fn[u][1];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 2 * (16 * mb + mfma16_row_f64(lane, r));
        if (m < R0) {
          s[m * QLS + c] = e[r];
          s[(m + 1) * QLS + c] = o[r];
        }
      }
    }
    // ---- 4: Y += s S1^T on the strip; the first block's fragments are on their
    // way before the barrier, the next block's while one multiplies
    const int lane = own_lane(), kk = lane >> 4, cl = lane & 15;
    double f[2][4][2];
    auto ldf = [&](int t) {
      const int it = w + NW * t < nout ? w + NW * t : 0, mc = it % nmc, S = qm.s1.S;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ks = 4 * st + q < S ? 4 * st + q : S - 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) f[t & 1][q][h] = qm.s1.f[((h * nmc + mc) * S + ks) * 64 + lane];
      }
    };
    ldf(0);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < QOUT; ++t) {
      const int it = w + NW * t;
      if (t + 1 < QOUT) ldf(t + 1);
      if (it < nout) {
        const double* row = s + (16 * (it / nmc) + cl) * QLS + kk;
        const double sg = qm.s1.sgn;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (4 * st + q < qm.s1.S) {
            const double x = row[4 * q], y = sg * row[4 * q + 16];
            out[t][0] = mfma_f64(x + y, f[t & 1][q][0], out[t][0]);
            out[t][1] = mfma_f64(x - y, f[t & 1][q][1], out[t][1]);
          }
      }
    }
    __syncthreads();
  }
  const int lane = own_lane(), cl = lane & 15;
  TIO* Yb = Y + b * n0 * n1;
#pragma unroll
  for (int t = 0; t < QOUT; ++t) {
    const int it = w + NW * t;
    if (it >= nout) break;
    const int m = 2 * (16 * (it % nmc) + cl);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * (it / nmc) + mfma16_row_f64(lane, r);
      if (i < n0) {
        if (m < n1) Yb[i * n1 + m] = (TIO)out[t][0][r];
        if (m + 1 < n1) Yb[i * n1 + m + 1] = (TIO)out[t][1][r];
      }
    }
  }
}

static bool quad_op(const double* f, int M, int K, int mode, int sgn, QuadOp& o) {
  o.f = f;
  o.M = M;
  o.K = K;
  o.sgn = sgn;
  return f && (sgn == 1 || sgn == -1) && par_shape(M, K, mode, o.S, o.nrb);
}

// waves of the kernel for these sizes (0: not taken): step 2 wants two per 16 half
// points of axis 0, step 4 at most QOUT blocks of Y each, and the strip's arrays
// must fit the LDS
static int quad_waves(const QuadMap& m) {
  const int it2 = 2 * m.b0.nrb, nout = (quad_pad(m.b0.K) >> 4) * m.s1.nrb;
  if (quad_lds(m) > 160 * 1024) return 0;
  for (int nw = 4; nw <= 12; nw += 4)
    if (nw >= it2 && QOUT * nw >= nout) return nw;
  return 0;
}

template <typename TIO, int NW>
static int launch_quad(const TIO* U, TIO* Y, const QuadMap& qm, long long B, hipStream_t st) {
  const size_t shm = quad_lds(qm);
  if (shm > 64 * 1024)
    JFX_CHECK_HIP(hipFuncSetAttribute((const void*)quad_par_kernel<TIO, NW>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
  hipLaunchKernelGGL((quad_par_kernel<TIO, NW>), dim3((unsigned)B), dim3(64 * NW), shm, st, U, Y, qm);
  JFX_LAUNCH_CHECK();
  return JFX_OK;
}

template <typename TIO>
static int launch_quad_t(const TIO* U, TIO* Y, const QuadMap& qm, long long B, hipStream_t st) {
  switch (quad_waves(qm)) {
    case 4: return launch_quad<TIO, 4>(U, Y, qm, B, st);
    case 8: return launch_quad<TIO, 8>(U, Y, qm, B, st);
    case 12: return launch_quad<TIO, 12>(U, Y, qm, B, st);
  }
  return set_error("quad_par: sizes not taken"), JFX_ESHAPE;
}

static bool quad_map(const double* const* F, const int* sgn, const double* c, int n0, int Q0, int n1, int Q1,
                     QuadMap& qm) {
  for (int i = 0; i < 6; ++i) qm.c[i] = c ? c[i] : 0.0;
  return n0 > 0 && n1 > 0 && quad_op(F[0], Q0, n0, 1, sgn[0], qm.b0) && quad_op(F[1], Q0, n0, 1, sgn[1], qm.d0) &&
         quad_op(F[2], Q1, n1, 1, sgn[2], qm.b1) && quad_op(F[3], Q1, n1, 1, sgn[3], qm.d1) &&
         quad_op(F[4], n0, Q0, 2, sgn[4], qm.s0) && quad_op(F[5], n1, Q1, 2, sgn[5], qm.s1) && sgn[4] == 1;
}

}  // namespace jfx

using namespace jfx;

extern "C" {

int jfx_quad_par_ok(int n0, int Q0, int n1, int Q1) {
  const double one = 0.0;
  const double* F[6] = {&one, &one, &one, &one, &one, &one};
  const int sgn[6] = {1, -1, 1, -1, 1, 1};
  QuadMap qm;
  return quad_map(F, sgn, nullptr, n0, Q0, n1, Q1, qm) && quad_waves(qm) > 0 ? 1 : 0;
}

int jfx_quad_par(int dtype, const double* const* F, const int* sgn, const double* c, int n0, int Q0, int n1, int Q1,
                 const void* U, void* Y, long long B, hipStream_t stream) {
  if (!F || !sgn || !c || !U || !Y) return set_error("quad_par: null pointer"), JFX_EARG;
  QuadMap qm;
  if (!quad_map(F, sgn, c, n0, Q0, n1, Q1, qm) || !quad_waves(qm) || B < 0 || B > 0x7fffffffLL)
    return set_error("quad_par: n = (%d, %d), Q = (%d, %d), %lld problems", n0, n1, Q0, Q1, B), JFX_ESHAPE;
  if (B == 0) return JFX_OK;
  if (dtype == 0) return launch_quad_t<double>((const double*)U, (double*)Y, qm, B, stream);
  if (dtype == 1) return launch_quad_t<float>((const float*)U, (float*)Y, qm, B, stream);
  return set_error("quad_par: dtype must be 0 or 1"), JFX_EARG;
}

}  // extern "C"
