// Building blocks of the fused 2D FP64 kernels for operators with decoupled
// even and odd parts (structures and fragments: contract_par.hip).
//
// One workgroup of NW waves holds a slab in LDS and applies one operator along
// each axis:  T = X A1^T (rows x M1),  Y = A0 T (M0 x M1).
//   phase A  a wave owns JW 16-row blocks of X and a half column block of T, even and
//            odd part: all of T sits in the workgroup's registers, so T overwrites X
//   phase B  a wave owns a half row block of Y and JW column blocks
// Up to 64 x 64 (JW = 1) a wave loads all its fragments of a phase before the
// barrier in front of it: with one slab per CU a phase is as long as its loads
// take, and an L2 round trip per k-step was most of it.  Larger slabs (JW = 2, 16
// waves) have no registers for that and load two k-steps ahead.
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

// Thread and lane index as opaque values: addresses computed from them are not
// shared between phases, which would hold hundreds of them in registers.
__device__ __forceinline__ int own_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}
__device__ __forceinline__ int own_lane() { return own_tid() & 63; }

// Zeros around a (K0 x K1) slab in LDS, rows and columns up to multiples of 16.
template <int NT>
__device__ __forceinline__ void slab_zero_pad(int K0, int K1, double* Xs) {
  const int LDX = slab_ldx(K1), R = slab_pad(K0), C = slab_pad(K1);
  const int tid = own_tid();
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
  const int LDX = slab_ldx(K1);
  const int tid = own_tid();
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

// The same in two halves: the loads of a slab into registers (at most 8 pairs a
// thread: 16384 values for 1024 threads; K1 even, X 16-byte aligned), and later
// the stores into LDS.
template <int NT>
__device__ __forceinline__ void slab_load8(const double* __restrict__ X, int K0, int K1, d2 (&v)[8]) {
  const int tid = own_tid(), n2 = K0 * (K1 / 2);
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int e = tid + NT * u;
    v[u] = *(const d2*)(X + 2 * (e < n2 ? e : n2 - 1));  // unconditional: v is not live through branches
  }
}
template <int NT>
__device__ __forceinline__ void slab_put8(const d2 (&v)[8], int K0, int K1, double* Xs) {
  const int tid = own_tid(), n2 = K0 * (K1 / 2), LDX = slab_ldx(K1);
  const unsigned kh = K1 / 2;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const unsigned e = tid + NT * u, i = e / kh, k = e - i * kh;
    if ((int)e < n2) *(d2*)&Xs[i * LDX + 2 * k] = v[u];
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

template <int JW>
struct Acc {
  v4d v[2][JW];  // [part][block]
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < JW; ++j) v[h][j] = v4d{0, 0, 0, 0};
  }
};

// Fragments of NB blocks of one operator, both parts: every k-step up to SMAX
// (slabs up to 64: 8), or with SMAX = 2 the step pair in use.
template <int NB, int SMAX>
struct Frag {
  const double* p[2][NB];
  int lo, hi, S;
  double v[SMAX][2][NB];

  // unconditional (steps past the last are clamped), so that no earlier value of
  // v stays live through a branch
  __device__ __forceinline__ void load(int s0) {
#pragma unroll
    for (int u = 0; u < SMAX; ++u) {
      const int s = SMAX == 2 || s0 + u < S ? s0 + u : S - 1;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < NB; ++j) v[u][h][j] = p[h][j][s * 64];
    }
  }
  // blocks rb[] of o; the first loads are issued here, ahead of the barrier
  __device__ __forceinline__ void init(const ParOp& o, const int (&rb)[NB]) {
    const int lane = own_lane();
    lo = o.lo[rb[0]];
    hi = o.hi[rb[0]];
    S = o.S;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      lo = o.lo[rb[j]] < lo ? o.lo[rb[j]] : lo;
      hi = o.hi[rb[j]] > hi ? o.hi[rb[j]] : hi;
#pragma unroll
      for (int h = 0; h < 2; ++h) p[h][j] = o.f + ((h * o.nrb + rb[j]) * o.S) * 64 + lane;
    }
    load(SMAX == 2 ? lo : 0);  // lo < S, also of an empty range
  }
  // f(k-step, fragments of that step) over the steps that are not zero
  template <typename F>
  __device__ __forceinline__ void each(F&& f) {
    if constexpr (SMAX == 2) {
      for (int s = lo; s < hi; s += 2) {
        Frag n = *this;
        n.load(s + 2 < hi ? s + 2 : s);
        f(s, v[0]);
        f(s + 1, v[1]);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < NB; ++j) v[u][h][j] = n.v[u][h][j];
      }
    } else {
#pragma unroll
      for (int s = 0; s < SMAX; ++s)
        if (s >= lo && s < hi) f(s, v[s]);
    }
  }
};
template <int JW>
constexpr int frag_steps() { return JW == 1 ? 8 : 2; }

// A wave's share of phase A: a half column block and JW row blocks, which share
// the operator's fragments (the other way round, JW column blocks of one row block,
// the fragments of a 128 x 128 pass are 512 KB from L2 instead of 256: 250 against
// 238 us for 2048 slabs).
template <int JW>
struct WaveA {
  int cb, rb[JW];
  bool on, ok[JW];
  Frag<1, frag_steps<JW>()> f;

  __device__ __forceinline__ void init(int w, int K0, const ParOp& o) {
    const int nrow = slab_pad(K0) >> 4, rg = w / o.nrb;
    cb = w - rg * o.nrb;
    on = JW * rg < nrow;
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      ok[j] = JW * rg + j < nrow;
      rb[j] = ok[j] ? JW * rg + j : 0;  // a copy whose results are not stored
    }
  }
  __device__ __forceinline__ void prefetch(const ParOp& o) {
    const int c[1] = {cb};
    f.init(o, c);
  }
};

template <int MODE, int JW>
__device__ __forceinline__ void phase_a(const double* Xs, int LDX, const ParOp& o, WaveA<JW>& wa, Acc<JW>& acc) {
  const int lane = own_lane(), kk = lane >> 4, cl = lane & 15;
  const double sg = o.sgn;
  const int K = o.K;
  wa.f.each([&](int s, const double(&a)[2][1]) {
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      double e, d;
      row_operands<MODE>(Xs + (16 * wa.rb[j] + cl) * LDX, s, kk, K, sg, e, d);
      acc.v[0][j] = mfma_f64(e, a[0][0], acc.v[0][j]);
      acc.v[1][j] = mfma_f64(d, a[1][0], acc.v[1][j]);
    }
  });
}

// T (rows 16 rb.., M1 columns) into LDS, rows LDT apart
template <int MODE, int JW>
__device__ __forceinline__ void store_t(double* T, int LDT, const ParOp& o, const WaveA<JW>& wa, const Acc<JW>& acc) {
  const int lane = own_lane(), cl = lane & 15;
  const double sg = o.sgn;
  const int M = o.M, Mh = (M + 1) >> 1;
  const int m = 16 * wa.cb + cl;
  if (m >= Mh) return;
#pragma unroll
  for (int j = 0; j < JW; ++j) {
    if (!wa.ok[j]) break;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double* d = T + (16 * wa.rb[j] + mfma16_row_f64(lane, r)) * LDT;
      const double e = acc.v[0][j][r], q = acc.v[1][j][r];
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

// A wave's share of phase B: a half row block of A0 and JW column blocks of T.
template <int JW>
__host__ __device__ __forceinline__ int items_b(const ParOp& o, int M1) {
  return o.nrb * (((slab_pad(M1) >> 4) + JW - 1) / JW);
}
template <int JW>
struct ItemB {
  int rb, c[JW];
  bool on, ok[JW];
  Frag<1, frag_steps<JW>()> f;

  __device__ __forceinline__ void init(int it, const ParOp& o, int M1) {
    const int ncb = slab_pad(M1) >> 4, ncg = (ncb + JW - 1) / JW;
    rb = it / ncg;
    const int cg = it - rb * ncg;
    on = rb < o.nrb;
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      ok[j] = JW * cg + j < ncb;
      c[j] = 16 * (ok[j] ? JW * cg + j : JW * cg);
    }
  }
  __device__ __forceinline__ void prefetch(const ParOp& o) {
    const int r[1] = {on ? rb : 0};
    f.init(o, r);
  }
};

template <int MODE, int JW>
__device__ __forceinline__ void phase_b(const double* T, int LDT, const ParOp& o, ItemB<JW>& b, Acc<JW>& acc) {
  const int lane = own_lane(), kk = lane >> 4, cl = lane & 15;
  const double sg = o.sgn;
  const int K = o.K;
  b.f.each([&](int s, const double(&a)[2][1]) {
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      double e, d;
      col_operands<MODE>(T, LDT, b.c[j] + cl, s, kk, K, sg, e, d);
      acc.v[0][j] = mfma_f64(a[0][0], e, acc.v[0][j]);
      acc.v[1][j] = mfma_f64(a[1][0], d, acc.v[1][j]);
    }
  });
}

// waves that cover phase A of (K0 rows) x o1 and phase B of o0
template <int JW>
inline int slab_items(int K0, const ParOp& o0, const ParOp& o1) {
  const int a = (slab_pad(K0) / 16 + JW - 1) / JW * o1.nrb, b = items_b<JW>(o0, o1.M);
  return a > b ? a : b;
}

// f(m, c, value) for every element of the item inside (M x M1)
template <int MODE, int JW, typename F>
__device__ __forceinline__ void each_b(const ParOp& o, const ItemB<JW>& b, int M1, const Acc<JW>& acc, F&& f) {
  const int lane = own_lane(), cl = lane & 15;
  const double sg = o.sgn;
  const int M = o.M, Mh = (M + 1) >> 1;
#pragma unroll
  for (int j = 0; j < JW; ++j) {
    if (!b.ok[j]) break;
    const int c = b.c[j] + cl;
    if (c >= M1) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * b.rb + mfma16_row_f64(lane, r);
      if (m >= Mh) continue;
      const double e = acc.v[0][j][r], q = acc.v[1][j][r];
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
