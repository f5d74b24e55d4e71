// Building blocks of the fused 2D FP64 kernels for operators with decoupled
// even and odd parts (structures and fragments: contract_par.hip).
//
// One workgroup of NW waves holds a slab in LDS and applies one operator along
// each axis:  T = X A1^T (rows x M1),  Y = A0 T (M0 x M1).
//   phase A  a wave owns 16 rows of X and two half column blocks of T, even and
//            odd part (4 accumulators): all of T sits in the workgroup's
//            registers, so T overwrites X in LDS
//   phase B  a wave owns a half row block of Y and two column blocks
// Rows of X are 16-byte pairs (even k, odd k) for EVAL and MIX; LDX = 2 (mod 16)
// puts 16 rows on distinct banks.  T is read in rows 2 apart, 16 columns wide;
// LDT = 8 (mod 16) does the same there.  Rows past the slab and columns past K1
// are zero in LDS, as the operators' fragments are.
#pragma once
#include "jfx_common.h"

namespace jfx {

enum { MODE_DENSE = 0, MODE_EVAL = 1, MODE_PROJ = 2, MODE_MIX = 3 };

constexpr int SLAB_MAX = 128;  // largest slab dimension

// One operator's fragments: [part][rb][s][64]; lo / hi: k-steps (even) of each
// half row block, both parts.
struct ParOp {
  const double* f;
  int M, K, S, nrb, sgn;
  signed char lo[4], hi[4];
};

__host__ __device__ constexpr int slab_pad(int n) { return (n + 15) & ~15; }
__host__ __device__ constexpr int slab_ldx(int n) { return slab_pad(n) + 2; }
__host__ __device__ constexpr int slab_ldt(int n) { return slab_pad(n) + 8; }

// LDS values of a pass over a (K0 x K1) slab by operators (M0 x K0), (M1 x K1)
__host__ __device__ inline int slab_lds(int K0, int K1, int M1) {
  const int lx = slab_ldx(K1), lt = slab_ldt(M1);
  return slab_pad(K0) * (lx > lt ? lx : lt);
}

typedef double d2 __attribute__((ext_vector_type(2)));

// Zeros around a (K0 x K1) slab in LDS, rows and columns up to multiples of 16.
template <int NT>
__device__ __forceinline__ void slab_zero_pad(int K0, int K1, double* Xs) {
  const int LDX = slab_ldx(K1), R = slab_pad(K0), C = slab_pad(K1), tid = threadIdx.x;
  const int nz = C - K1;
  if (nz)
    for (int e = tid; e < K0 * nz; e += NT) {
      const int i = e / nz;
      Xs[i * LDX + K1 + (e - i * nz)] = 0.0;
    }
  for (int e = tid; e < (R - K0) * C; e += NT) {
    const int i = e / C;
    Xs[(K0 + i) * LDX + (e - i * C)] = 0.0;
  }
}

// X (K0 x K1, contiguous) into LDS, rows LDX apart, zero padded to 16s.
template <int NT>
__device__ __forceinline__ void slab_stage(const double* __restrict__ X, int K0, int K1, double* Xs) {
  const int LDX = slab_ldx(K1), tid = threadIdx.x;
  constexpr int U = 8;
  if (K1 % 2 == 0 && ((uintptr_t)X & 15) == 0) {
    const unsigned kh = K1 / 2;
    const int n2 = K0 * (int)kh;
    for (int eb = tid; eb < n2; eb += NT * U) {
      d2 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = eb + NT * u;
        v[u] = e < n2 ? *(const d2*)(X + 2 * e) : d2{0, 0};
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const unsigned e = eb + NT * u, i = e / kh, k = e - i * kh;
        if ((int)e < n2) *(d2*)&Xs[i * LDX + 2 * k] = v[u];
      }
    }
  } else {
    const int n1 = K0 * K1;
    for (int eb = tid; eb < n1; eb += NT * U) {
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = eb + NT * u;
        v[u] = e < n1 ? X[e] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const unsigned e = eb + NT * u, i = e / (unsigned)K1, k = e - i * (unsigned)K1;
        if ((int)e < n1) Xs[i * LDX + k] = v[u];
      }
    }
  }
  slab_zero_pad<NT>(K0, K1, Xs);
}

// even and odd operand of k-step s from a row of X (element stride 1)
template <int MODE>
__device__ __forceinline__ void row_operands(const double* row, int s, int kk, int K, double sg, double& e, double& o) {
  if constexpr (MODE == MODE_PROJ) {
    const int k = 4 * s + kk, kr = K - 1 - k;
    const double x = row[k], y = sg * row[kr < 0 ? K : kr];
    e = x + y;
    o = x - y;
  } else {
    const d2 v = *(const d2*)&row[8 * s + 2 * kk];
    e = v[0];
    o = v[1];
  }
}
template <int MODE>
__device__ __forceinline__ void col_operands(const double* T, int LDT, int c, int s, int kk, int K, double sg,
                                             double& e, double& o) {
  if constexpr (MODE == MODE_PROJ) {
    const int k = 4 * s + kk, kr = K - 1 - k;
    const double x = T[k * LDT + c], y = sg * T[(kr < 0 ? K : kr) * LDT + c];
    e = x + y;
    o = x - y;
  } else {
    const int k = 8 * s + 2 * kk;
    e = T[k * LDT + c];
    o = T[(k + 1) * LDT + c];
  }
}

typedef v4d Acc4[2][2];  // [part][block]

__device__ __forceinline__ void acc_zero(Acc4& a) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 2; ++j) a[h][j] = v4d{0, 0, 0, 0};
}

// Waves of phase A: (row block, pair of half column blocks); -1: idle.
struct WaveA {
  int rb, cb[2];
  bool on, on1;
};
__device__ __forceinline__ WaveA wave_a(int w, int K0, const ParOp& o) {
  const int ncg = (o.nrb + 1) >> 1, nrow = slab_pad(K0) >> 4;
  WaveA a;
  a.rb = w / ncg;
  const int cg = w - a.rb * ncg;
  a.on = a.rb < nrow;
  a.cb[0] = 2 * cg;
  a.on1 = 2 * cg + 1 < o.nrb;
  a.cb[1] = a.on1 ? 2 * cg + 1 : 2 * cg;  // a copy whose results are not stored
  return a;
}

template <int MODE>
__device__ __forceinline__ void phase_a(const double* Xs, int LDX, const ParOp& o, const WaveA& wa, Acc4& acc) {
  const int lane = threadIdx.x & 63, kk = lane >> 4, cl = lane & 15;
  const double* row = Xs + (16 * wa.rb + cl) * LDX;
  const double sg = o.sgn;
  int lo = o.lo[wa.cb[0]], hi = o.hi[wa.cb[0]];
  lo = o.lo[wa.cb[1]] < lo ? o.lo[wa.cb[1]] : lo;
  hi = o.hi[wa.cb[1]] > hi ? o.hi[wa.cb[1]] : hi;
  const double* p[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 2; ++j) p[h][j] = o.f + ((h * o.nrb + wa.cb[j]) * o.S) * 64 + lane;
  double a[2][2][2], n[2][2][2];  // [step][part][block]
  auto ld = [&](int s, double(&d)[2][2][2]) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) d[u][h][j] = p[h][j][(s + u) * 64];
  };
  if (lo < hi) ld(lo, a);
  for (int s = lo; s < hi; s += 2) {
    if (s + 2 < hi) ld(s + 2, n);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      double e, d;
      row_operands<MODE>(row, s + u, kk, o.K, sg, e, d);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        acc[0][j] = mfma_f64(e, a[u][0][j], acc[0][j]);
        acc[1][j] = mfma_f64(d, a[u][1][j], acc[1][j]);
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) a[u][h][j] = n[u][h][j];
  }
}

// T (rows 16 rb.., M1 columns) into LDS, rows LDT apart
template <int MODE>
__device__ __forceinline__ void store_t(double* T, int LDT, const ParOp& o, const WaveA& wa, const Acc4& acc) {
  const int lane = threadIdx.x & 63, cl = lane & 15;
  const double sg = o.sgn;
  const int M = o.M, Mh = (M + 1) >> 1;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (j == 1 && !wa.on1) break;
    const int m = 16 * wa.cb[j] + cl;
    if (m >= Mh) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double* d = T + (16 * wa.rb + mfma16_row_f64(lane, r)) * LDT;
      const double e = acc[0][j][r], q = acc[1][j][r];
      if constexpr (MODE == MODE_EVAL) {
        d[m] = e + q;
        d[M - 1 - m] = M - 1 - m == m ? e + q : sg * (e - q);
      } else {
        const bool sw = MODE == MODE_MIX && o.sgn < 0;
        *(d2*)&d[2 * m] = sw ? d2{q, e} : d2{e, q};  // column M (odd M) is padding
      }
    }
  }
}

// Items of phase B: (half row block of A0, pair of column blocks of T)
__device__ __forceinline__ int items_b(const ParOp& o, int M1) {
  return o.nrb * (((slab_pad(M1) >> 4) + 1) >> 1);
}
struct ItemB {
  int rb, c[2];
  bool on1;
};
__device__ __forceinline__ ItemB item_b(int it, const ParOp& o, int M1) {
  const int ncb = slab_pad(M1) >> 4, ncg = (ncb + 1) >> 1;
  ItemB b;
  b.rb = it / ncg;
  const int cg = it - b.rb * ncg;
  b.c[0] = 32 * cg;
  b.on1 = 2 * cg + 1 < ncb;
  b.c[1] = b.on1 ? 32 * cg + 16 : 32 * cg;
  return b;
}

template <int MODE>
__device__ __forceinline__ void phase_b(const double* T, int LDT, const ParOp& o, const ItemB& b, Acc4& acc) {
  const int lane = threadIdx.x & 63, kk = lane >> 4, cl = lane & 15;
  const double sg = o.sgn;
  const int lo = o.lo[b.rb], hi = o.hi[b.rb];
  const double* p0 = o.f + (b.rb * o.S) * 64 + lane;
  const double* p1 = p0 + o.nrb * o.S * 64;
  double a[2][2], n[2][2];  // [step][part]
  auto ld = [&](int s, double(&d)[2][2]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      d[u][0] = p0[(s + u) * 64];
      d[u][1] = p1[(s + u) * 64];
    }
  };
  if (lo < hi) ld(lo, a);
  for (int s = lo; s < hi; s += 2) {
    if (s + 2 < hi) ld(s + 2, n);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        double e, d;
        col_operands<MODE>(T, LDT, b.c[j] + cl, s + u, kk, o.K, sg, e, d);
        acc[0][j] = mfma_f64(a[u][0], e, acc[0][j]);
        acc[1][j] = mfma_f64(a[u][1], d, acc[1][j]);
      }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      a[u][0] = n[u][0];
      a[u][1] = n[u][1];
    }
  }
}

// f(m, c, value) for every element of the item inside (M x M1)
template <int MODE, typename F>
__device__ __forceinline__ void each_b(const ParOp& o, const ItemB& b, int M1, const Acc4& acc, F&& f) {
  const int lane = threadIdx.x & 63, cl = lane & 15;
  const double sg = o.sgn;
  const int M = o.M, Mh = (M + 1) >> 1;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (j == 1 && !b.on1) break;
    const int c = b.c[j] + cl;
    if (c >= M1) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * b.rb + mfma16_row_f64(lane, r);
      if (m >= Mh) continue;
      const double e = acc[0][j][r], q = acc[1][j][r];
      if constexpr (MODE == MODE_EVAL) {
        f(m, c, e + q);
        if (M - 1 - m != m) f(M - 1 - m, c, sg * (e - q));
      } else {
        const bool sw = MODE == MODE_MIX && o.sgn < 0;
        f(2 * m, c, sw ? q : e);
        if (2 * m + 1 < M) f(2 * m + 1, c, sw ? e : q);
      }
    }
  }
}

}  // namespace jfx
