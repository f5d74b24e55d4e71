// Per-axis contraction of FP64 / FP32 arrays by operators whose even and odd
// parts decouple:
//     Y[p, m, q] = sum_k A[m, k] X[p, k, q],   X viewed as (P, K, Q), any Q.
//
// Bases on a symmetric interval have definite parity, psi_k(-x) =
// (-1)^k psi_k(x), and Gauss meshes are symmetric, so the operators of this
// package come in three structured forms, each two half-size products:
//   MODE_EVAL  (series -> mesh)   A[M-1-m, k] = sgn (-1)^k A[m, k]:
//              e = A_e x_even, o = A_o x_odd; y[m] = e + o, y[M-1-m] = sgn (e - o)
//   MODE_PROJ  (mesh -> modes)    A[m, K-1-k] = sgn (-1)^m A[m, k]:
//              y_even = A_e (x[k] + sgn x[K-1-k]), y_odd = A_o (x[k] - sgn x[K-1-k])
//   MODE_MIX   (modes -> modes)   A[m, k] = 0 unless m + k is even (sgn = +1)
//              or odd (sgn = -1): mass, stiffness and sorted eigenvector
//              matrices
//   MODE_DENSE (no structure)     one full-size product
//
// What bounds it: FP64 MFMA and vector FMA run at the same 78.6 TFLOP/s, so a
// dense 128 x 128 contraction (16 flop per byte moved) sits above the ridge at
// ~10 flop/B; halving the products puts it below, at the HBM time.
//
// One workgroup of four waves owns TN = 16 NB columns with all K rows in LDS
// (about 40 KB at K = 128, so three or four workgroups share a CU and one's
// loads and stores overlap another's products).  A wave takes one 16-row block
// of the halves and all NB column blocks, even and odd part together (so the
// sums e +- o and x[k] +- x[K-1-k] stay in registers).  The operator is read as
// MFMA fragments (512 contiguous bytes per wave load) that stay in L2; the next
// two k-steps' fragments are loaded before the current ones multiply.
//   Q > 1   LDS tile Bs[k][c]; a 16x16 result block has rows m and columns c.
//   Q == 1  LDS tile Xs[c][k]; the operands swap roles, so that result blocks
//           have rows c and columns m and stores run along the contiguous axis.
// A wave reads 4 rows times 16 columns of the tile; strides: lds_stride_cols(),
// lds_stride_rows().
// `band`: operators with A[m, k] = 0 outside -bp <= k - m <= bq skip the k-steps
// a row block does not touch (mass matrices: 5 of 16; triangular stiffness: half).
#include "par_blocks.h"

namespace jfx {

constexpr int PAR_MAXRB = 32;   // 16-row blocks of a part (M <= 1024 structured, 512 dense)
constexpr int PAR_MAXK = 512;
constexpr int PAR_NT = 256;     // threads

struct ParMap {
  long long P, Q, ncols;
  int M, K, Mh, Kh, S, nrb, sgn;
  int vec;  // 16-byte loads: pairs of columns (Q even) or of k (Q == 1, K even)
  int nt;   // results bypass L2 (whole lines of a large array)
  int ovec; // Q == 1: pairs of outputs are 16-byte aligned
  short lo[2][PAR_MAXRB], hi[2][PAR_MAXRB];  // k-steps (even counts) of each part's row block
};

// Elements between LDS rows.  Q > 1: EVAL and MIX read rows 2 apart, and 2 * stride
// = 16 (mod 32 doubles, for FP32 mod 64 words) puts their 16 columns on distinct
// banks.  DENSE and PROJ read neighbouring rows, stride = 8 or 24 apart, which share
// half their banks.  Q == 1: rows c, stride twice (FP32: four times) an odd number.
template <int NB>
__host__ __device__ constexpr int lds_stride_cols() {
  return 16 * NB + 8;
}
__host__ __device__ inline int lds_stride_rows(int kz, int elt) {
  const int u = elt == 8 ? 2 : 4;
  int n = (kz + u - 1) / u;
  return u * (n | 1);
}

template <typename T>
struct ParT;
template <>
struct ParT<double> {
  typedef v4d V;
  typedef double2 T2;
  static __device__ __forceinline__ V mfma(double a, double b, V c) { return mfma_f64(a, b, c); }
  static __device__ __forceinline__ int row(int lane, int r) { return mfma16_row_f64(lane, r); }
};
template <>
struct ParT<float> {
  typedef v4f V;
  typedef float2 T2;
  static __device__ __forceinline__ V mfma(float a, float b, V c) { return mfma_f32(a, b, c); }
  static __device__ __forceinline__ int row(int lane, int r) { return mfma16_row_f32(lane, r); }
};

// rows kept in LDS: K, zero rows up to what the k-steps read, and for PROJ a
// zero row K where the mirror index of a padded k-step would be negative
__host__ __device__ inline int par_kz(int mode, int K, int S) {
  const int reach = (mode == MODE_EVAL || mode == MODE_MIX) ? 8 * S : 4 * S;
  const int need = mode == MODE_PROJ && 4 * S > K ? K + 1 : K;
  return reach > need ? reach : need;
}

// column -> (p, q), in 32 bits where the column count allows
__device__ __forceinline__ void col_split(long long c, long long Q, bool small, long long& p, long long& q) {
  if (small) {
    const unsigned a = (unsigned)c / (unsigned)Q;
    p = a;
    q = (unsigned)c - a * (unsigned)Q;
  } else {
    p = c / Q;
    q = c - p * Q;
  }
}

template <typename T, int MODE, bool QONE, int NB, int JB, bool NTS>
__global__ __launch_bounds__(PAR_NT) void contract_par_kernel(const T* __restrict__ Af, const T* __restrict__ X,
                                                              T* __restrict__ Y, ParMap pm) {
  typedef typename ParT<T>::V V;
  typedef typename ParT<T>::T2 T2;
  constexpr int TN = 16 * NB;
  constexpr int LDC = lds_stride_cols<NB>();
  constexpr bool PARIN = MODE == MODE_EVAL || MODE == MODE_MIX;
  constexpr int NPART = MODE == MODE_DENSE ? 1 : 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T* Bs = reinterpret_cast<T*>(smem);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = pm.M, K = pm.K, S = pm.S, nrb = pm.nrb;
  const long long Q = pm.Q, c0 = (long long)blockIdx.x * TN;
  const int ncol = pm.ncols - c0 < TN ? (int)(pm.ncols - c0) : TN;
  const int kz = par_kz(MODE, K, S);
  const bool small = pm.ncols <= 0x7fffffffLL;
  const int LDR = QONE ? lds_stride_rows(kz, sizeof(T)) : 0;

  // ---- stage the tile
  if constexpr (QONE) {
    const T* src = X + c0 * K;
    constexpr int U = 8;
    if (pm.vec) {
      const int n2 = ncol * (K / 2);
      const unsigned kh = K / 2;
      for (int eb = tid; eb < n2; eb += PAR_NT * U) {
        T2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int e = eb + PAR_NT * u;
          v[u] = e < n2 ? *(const T2*)(src + 2 * e) : T2{T(0), T(0)};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const unsigned e = eb + PAR_NT * u, c = e / kh, k = e - c * kh;
          if ((int)e < n2) *(T2*)&Bs[c * LDR + 2 * k] = v[u];
        }
      }
    } else {
      const int n1 = ncol * K;
      for (int eb = tid; eb < n1; eb += PAR_NT * U) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int e = eb + PAR_NT * u;
          v[u] = e < n1 ? src[e] : T(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const unsigned e = eb + PAR_NT * u, c = e / (unsigned)K, k = e - c * (unsigned)K;
          if ((int)e < n1) Bs[c * LDR + k] = v[u];
        }
      }
    }
    // zero the k past K of every column, and columns past the last
    const int nz = kz - K;
    for (int e = tid; e < TN * nz; e += PAR_NT) {
      const int c = e / nz;
      Bs[c * LDR + K + (e - c * nz)] = T(0);
    }
    if (ncol < TN)
      for (int e = tid; e < (TN - ncol) * K; e += PAR_NT) {
        const int c = e / K;
        Bs[(ncol + c) * LDR + (e - c * K)] = T(0);
      }
  } else {
    // this thread's column(s): one 64-bit division each
    if (pm.vec) {
      constexpr int TPR = TN / 2, RP = PAR_NT / TPR;
      const int cc = 2 * (tid % TPR), k0 = tid / TPR;
      const long long c = c0 + cc;
      const bool ok = c < pm.ncols;  // pairs never straddle: Q and ncols are even
      long long p, q;
      col_split(ok ? c : 0, Q, small, p, q);
      const T* src = X + p * K * Q + q;
      constexpr int U = 8;
      for (int kb = k0; kb < K; kb += RP * U) {
        T2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = kb + RP * u;
          v[u] = (ok && k < K) ? *(const T2*)(src + (long long)k * Q) : T2{T(0), T(0)};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = kb + RP * u;
          if (k < K) *(T2*)&Bs[k * LDC + cc] = v[u];
        }
      }
    } else {
      constexpr int RP = PAR_NT / TN;
      const int cc = tid % TN, k0 = tid / TN;
      const long long c = c0 + cc;
      const bool ok = c < pm.ncols;
      long long p, q;
      col_split(ok ? c : 0, Q, small, p, q);
      const T* src = X + p * K * Q + q;
      constexpr int U = 8;
      for (int kb = k0; kb < K; kb += RP * U) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = kb + RP * u;
          v[u] = (ok && k < K) ? src[(long long)k * Q] : T(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = kb + RP * u;
          if (k < K) Bs[k * LDC + cc] = v[u];
        }
      }
    }
    for (int e = tid; e < (kz - K) * TN; e += PAR_NT) Bs[(K + e / TN) * LDC + e % TN] = T(0);
  }
  __syncthreads();

  // ---- products: items of one row block and JB column blocks, dealt to the waves
  constexpr int NCG = NB / JB;
  const int nitem = nrb * NCG;
  const int kk = lane >> 4, cl = lane & 15;
  const T sg = T(pm.sgn);
  // rotated by workgroup: where the items do not divide by four, the extra ones
  // of a CU's workgroups fall on different SIMDs
  for (int it = (w + blockIdx.x) & 3; it < nitem; it += 4) {
    const int rb = it / NCG, j0 = (it - rb * NCG) * JB;
    V acc[NPART][JB];
#pragma unroll
    for (int h = 0; h < NPART; ++h)
#pragma unroll
      for (int j = 0; j < JB; ++j) acc[h][j] = V{0, 0, 0, 0};
    int lo = pm.lo[0][rb], hi = pm.hi[0][rb];
    if constexpr (NPART == 2) {
      lo = pm.lo[1][rb] < lo ? pm.lo[1][rb] : lo;
      hi = pm.hi[1][rb] > hi ? pm.hi[1][rb] : hi;
    }
    const T* a0 = Af + ((long long)rb * S) * 64 + lane;
    const T* a1 = a0 + (long long)nrb * S * 64;
    T ae[2], ao[2], an[2], bn[2];
    auto aload = [&](int s, T(&e)[2], T(&o)[2]) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        e[u] = a0[(s + u) * 64];
        if constexpr (NPART == 2) o[u] = a1[(s + u) * 64];
      }
    };
    if (lo < hi) aload(lo, ae, ao);
    for (int s = lo; s < hi; s += 2) {
      if (s + 2 < hi) aload(s + 2, an, bn);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < JB; ++j) {
          const int c = 16 * (j0 + j) + cl;
          T be, bo = T(0);
          if constexpr (QONE) {
            if constexpr (PARIN) {
              const T2 b = *(const T2*)&Bs[c * LDR + 8 * (s + u) + 2 * kk];
              be = b.x;
              bo = b.y;
            } else {
              const int k = 4 * (s + u) + kk;
              be = Bs[c * LDR + k];
              if constexpr (MODE == MODE_PROJ) {
                const int kr = K - 1 - k;
                const T x = be, y = sg * Bs[c * LDR + (kr < 0 ? K : kr)];
                be = x + y;
                bo = x - y;
              }
            }
            acc[0][j] = ParT<T>::mfma(be, ae[u], acc[0][j]);
            if constexpr (NPART == 2) acc[1][j] = ParT<T>::mfma(bo, ao[u], acc[1][j]);
          } else {
            if constexpr (PARIN) {
              const int k = 8 * (s + u) + 2 * kk;
              be = Bs[k * LDC + c];
              bo = Bs[(k + 1) * LDC + c];
            } else {
              const int k = 4 * (s + u) + kk;
              be = Bs[k * LDC + c];
              if constexpr (MODE == MODE_PROJ) {
                const int kr = K - 1 - k;
                const T x = be, y = sg * Bs[(kr < 0 ? K : kr) * LDC + c];
                be = x + y;
                bo = x - y;
              }
            }
            acc[0][j] = ParT<T>::mfma(ae[u], be, acc[0][j]);
            if constexpr (NPART == 2) acc[1][j] = ParT<T>::mfma(ao[u], bo, acc[1][j]);
          }
        }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        ae[u] = an[u];
        if constexpr (NPART == 2) ao[u] = bn[u];
      }
    }
    // ---- results
    auto put = [&](T& d, T v) {
      if constexpr (NTS)
        __builtin_nontemporal_store(v, &d);
      else
        d = v;
    };
    T* ycol[JB];
    if constexpr (!QONE) {
#pragma unroll
      for (int j = 0; j < JB; ++j) {
        const long long c = c0 + 16 * (j0 + j) + cl;
        long long p, q;
        col_split(c < pm.ncols ? c : 0, Q, small, p, q);
        ycol[j] = Y + p * M * Q + q;
      }
    }
#pragma unroll
    for (int j = 0; j < JB; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = ParT<T>::row(lane, r);
        const int c = 16 * (j0 + j) + (QONE ? rr : cl);
        const int m = 16 * rb + (QONE ? cl : rr);
        if (c >= ncol || m >= pm.Mh) continue;
        T* dst;
        long long st;
        if constexpr (QONE) {
          dst = Y + (c0 + c) * M;
          st = 1;
        } else {
          dst = ycol[j];
          st = Q;
        }
        const T e = acc[0][j][r];
        if constexpr (MODE == MODE_DENSE) {
          put(dst[m * st], e);
        } else if constexpr (MODE == MODE_EVAL) {
          const T o = acc[1][j][r];
          put(dst[m * st], e + o);
          if (M - 1 - m != m) put(dst[(long long)(M - 1 - m) * st], sg * (e - o));
        } else {
          // part 0 goes to the rows of parity 0 (MIX with sgn < 0: parity 1)
          const T o = acc[1][j][r];
          const bool sw = MODE == MODE_MIX && pm.sgn < 0;
          const T y0 = sw ? o : e, y1 = sw ? e : o;
          if (QONE && pm.ovec) {
            typedef T tv2 __attribute__((ext_vector_type(2)));
            const tv2 y = {y0, y1};
            if constexpr (NTS)
              __builtin_nontemporal_store(y, (tv2*)(dst + 2 * m));
            else
              *(tv2*)(dst + 2 * m) = y;
          } else {
            if (2 * m < M) put(dst[(long long)(2 * m) * st], y0);
            if (2 * m + 1 < M) put(dst[(long long)(2 * m + 1) * st], y1);
          }
        }
      }
    }
  }
}

// Fragment of part h, row block rb, k-step s, lane l: the operator entry of
// half-row 16 rb + (l & 15) and half-column 4 s + (l >> 4), zero outside.
// Mirror images are averaged, so that the halves carry the rounding of both.
// One operator per blockIdx.y.
struct ParJob {
  const double* A;
  void* out;
  int M, K, mode, sgn, nrb, S, nparts;
};
constexpr int PAR_JOBS = 16;
struct ParJobs {
  ParJob j[PAR_JOBS];
};

template <typename T>
__global__ void par_prepare_kernel(ParJobs jobs) {
  const ParJob& J = jobs.j[blockIdx.y];
  const double* __restrict__ A = J.A;
  T* __restrict__ out = (T*)J.out;
  const int M = J.M, K = J.K, mode = J.mode, sgn = J.sgn, nrb = J.nrb, S = J.S;
  const long long total = (long long)J.nparts * nrb * S * 64;
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (long long)gridDim.x * blockDim.x) {
    const int l = e & 63;
    const int s = (e >> 6) % S, rb = ((e >> 6) / S) % nrb, h = (int)((e >> 6) / S / nrb);
    const int m = 16 * rb + (l & 15), k = 4 * s + (l >> 4);
    double v = 0.0;
    if (mode == MODE_DENSE) {
      if (m < M && k < K) v = A[(long long)m * K + k];
    } else if (mode == MODE_EVAL) {
      const int kc = 2 * k + h, mr = M - 1 - m;
      if (m <= mr && kc < K) {
        const double f = (h ? -1.0 : 1.0) * sgn;
        v = 0.5 * (A[(long long)m * K + kc] + f * A[(long long)mr * K + kc]);
      }
    } else if (mode == MODE_PROJ) {
      const int mr = 2 * m + h, kr = K - 1 - k;
      if (mr < M && k <= kr) {
        v = 0.5 * (A[(long long)mr * K + k] + (h ? -1.0 : 1.0) * sgn * A[(long long)mr * K + kr]);
        if (k == kr) v *= 0.5;  // the sum x[k] + x[K-1-k] counts the middle point twice
      }
    } else {
      const int mr = 2 * m + (sgn < 0 ? 1 - h : h), kc = 2 * k + h;
      if (mr < M && kc < K) v = A[(long long)mr * K + kc];
    }
    out[e] = (T)v;
  }
}

struct ParDims {
  int Mh, Kh, S, nrb, nparts;
};
static bool par_dims(int M, int K, int mode, ParDims& d) {
  if (M <= 0 || K <= 0 || mode < MODE_DENSE || mode > MODE_MIX) return false;
  d.nparts = mode == MODE_DENSE ? 1 : 2;
  d.Mh = mode == MODE_DENSE ? M : (M + 1) / 2;
  d.Kh = mode == MODE_DENSE ? K : (K + 1) / 2;
  d.S = 2 * ((d.Kh + 7) / 8);
  d.nrb = (d.Mh + 15) / 16;
  return d.nrb <= PAR_MAXRB && K <= PAR_MAXK;
}

// k-steps [lo, hi) (even numbers) in which row block rb of part h is not zero
static void par_range(const ParDims& d, int mode, int sgn, int bp, int bq, int h, int rb, short& lo, short& hi) {
  int k0 = 0, k1 = d.Kh - 1;
  if (mode == MODE_MIX && bp >= 0 && bq >= 0) {
    // rows 2 m + r, columns 2 k + h: -bp <= 2 (k - m) + h - r <= bq
    const int r = sgn < 0 ? 1 - h : h, m0 = 16 * rb, m1 = m0 + 15 < d.Mh - 1 ? m0 + 15 : d.Mh - 1;
    k0 = m0 + (r - h - bp >= 0 ? (r - h - bp + 1) / 2 : -((bp + h - r) / 2));
    k1 = m1 + (r - h + bq >= 0 ? (r - h + bq) / 2 : -((h - r - bq + 1) / 2));
    if (k0 < 0) k0 = 0;
    if (k1 > d.Kh - 1) k1 = d.Kh - 1;
  }
  lo = (short)(k0 <= k1 ? 2 * (k0 / 8) : 0);
  hi = (short)(k0 <= k1 ? 2 * (k1 / 8 + 1) : 0);
}

// Descriptor of a structured operator for the slab kernels (at most 128 rows:
// four half row blocks); k-step ranges cover both parts.
bool par_op(const double* frag, int M, int K, int mode, int sgn, int bp, int bq, ParOp& o) {
  ParDims d;
  if (!par_dims(M, K, mode, d) || d.nrb > 4 || K > SLAB_MAX || (sgn != 1 && sgn != -1)) return false;
  o.f = frag;
  o.M = M;
  o.K = K;
  o.S = d.S;
  o.nrb = d.nrb;
  o.sgn = sgn;
  for (int rb = 0; rb < 4; ++rb) o.lo[rb] = o.hi[rb] = 0;
  for (int rb = 0; rb < d.nrb; ++rb) {
    short lo[2], hi[2];
    for (int h = 0; h < 2; ++h) par_range(d, mode, sgn, bp, bq, h, rb, lo[h], hi[h]);
    if (lo[0] >= hi[0]) lo[0] = lo[1], hi[0] = hi[1];
    if (lo[1] >= hi[1]) lo[1] = lo[0], hi[1] = hi[0];
    o.lo[rb] = (signed char)(lo[0] < lo[1] ? lo[0] : lo[1]);
    o.hi[rb] = (signed char)(hi[0] > hi[1] ? hi[0] : hi[1]);
  }
  return true;
}

// k-steps and row blocks per part of an operator's fragments
bool par_shape(int M, int K, int mode, int& S, int& nrb) {
  ParDims d;
  if (!par_dims(M, K, mode, d)) return false;
  S = d.S;
  nrb = d.nrb;
  return true;
}

template <typename T, int MODE, bool QONE, int NB, int JB>
static int launch_par3(const T* Af, const T* X, T* Y, const ParMap& pm, hipStream_t st) {
  const int kz = par_kz(MODE, pm.K, pm.S);
  const size_t rows = QONE ? (size_t)16 * NB * lds_stride_rows(kz, sizeof(T))
                           : (size_t)kz * lds_stride_cols<NB>();
  const size_t shm = (rows * sizeof(T) + 15) & ~(size_t)15;
  auto kern = pm.nt ? contract_par_kernel<T, MODE, QONE, NB, JB, true> : contract_par_kernel<T, MODE, QONE, NB, JB, false>;
  if (shm > 64 * 1024) JFX_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
  const long long ntile = (pm.ncols + 16 * NB - 1) / (16 * NB);
  if (ntile > 0x7fffffffLL) return set_error("contract_par: grid too large"), JFX_ESHAPE;
  hipLaunchKernelGGL(kern, dim3((unsigned)ntile), dim3(PAR_NT), shm, st, Af, X, Y, pm);
  JFX_LAUNCH_CHECK();
  return JFX_OK;
}

template <typename T, int MODE>
static int launch_par2(const T* Af, const T* X, T* Y, const ParMap& pm, hipStream_t st) {
  // 32 columns per workgroup while at least two workgroups fit a CU's LDS.  A
  // wave takes both column blocks of a row block, so that the operator is read
  // once for both, unless that leaves waves idle.  (Single column blocks also
  // where five or six row blocks would come out more even: slower, 274 against
  // 257 us at M = 160, K = 158, 256000 columns.)  Dense FP64 operators keep all K rows
  // of a full-size product: 16 columns beyond K = 160 (128 x 192 on 2^20 columns 2072
  // -> 1628 us, plain matrix 1770; 192 x 192 2910 -> 2308).
  const bool two = pm.K <= (sizeof(T) == 8 ? (MODE == MODE_DENSE ? 160 : 192) : 384), thin = pm.nrb <= 2;
  if (pm.Q == 1)
    return !two   ? launch_par3<T, MODE, true, 1, 1>(Af, X, Y, pm, st)
           : thin ? launch_par3<T, MODE, true, 2, 1>(Af, X, Y, pm, st)
                  : launch_par3<T, MODE, true, 2, 2>(Af, X, Y, pm, st);
  return !two   ? launch_par3<T, MODE, false, 1, 1>(Af, X, Y, pm, st)
         : thin ? launch_par3<T, MODE, false, 2, 1>(Af, X, Y, pm, st)
                : launch_par3<T, MODE, false, 2, 2>(Af, X, Y, pm, st);
}

template <typename T>
static int launch_par(const T* Af, int M, int K, int mode, int sgn, int bp, int bq, const T* X, T* Y, long long P,
                      long long Q, hipStream_t st) {
  ParDims d;
  if (!par_dims(M, K, mode, d) || P < 0 || Q <= 0 || (sgn != 1 && sgn != -1))
    return set_error("contract_par: bad sizes M=%d K=%d mode=%d P=%lld Q=%lld", M, K, mode, P, Q), JFX_ESHAPE;
  ParMap pm;
  pm.P = P;
  pm.Q = Q;
  pm.ncols = P * Q;
  if (pm.ncols == 0) return JFX_OK;
  pm.M = M;
  pm.K = K;
  pm.Mh = d.Mh;
  pm.Kh = d.Kh;
  pm.S = d.S;
  pm.nrb = d.nrb;
  pm.sgn = sgn;
  const uintptr_t al = 2 * sizeof(T) - 1;
  pm.vec = ((Q == 1 ? K : Q) % 2 == 0 && ((uintptr_t)X & al) == 0) ? 1 : 0;
  pm.ovec = (M % 2 == 0 && ((uintptr_t)Y & al) == 0) ? 1 : 0;
  // 128-byte runs of a result block are whole cache lines and the array is far
  // larger than the L2s: nontemporal stores (M = K = 128, 16 x 128^3 values:
  // 170, 155, 143 -> 145, 131, 118 us along the three axes).  Partial lines
  // need L2 to merge them (Q = 126: 25 us, nontemporal 34 us).
  const long long run = Q == 1 ? M : Q;
  pm.nt = run % (128 / (int)sizeof(T)) == 0 && ((uintptr_t)Y & 127) == 0 &&
          pm.ncols * M * (long long)sizeof(T) >= (64LL << 20);
  for (int h = 0; h < 2; ++h)
    for (int rb = 0; rb < d.nrb; ++rb) par_range(d, mode, sgn, bp, bq, h, rb, pm.lo[h][rb], pm.hi[h][rb]);
  switch (mode) {
    case MODE_DENSE: return launch_par2<T, MODE_DENSE>(Af, X, Y, pm, st);
    case MODE_EVAL: return launch_par2<T, MODE_EVAL>(Af, X, Y, pm, st);
    case MODE_PROJ: return launch_par2<T, MODE_PROJ>(Af, X, Y, pm, st);
    default: return launch_par2<T, MODE_MIX>(Af, X, Y, pm, st);
  }
}

}  // namespace jfx

using namespace jfx;

extern "C" {

long long jfx_par_frag_elems(int M, int K, int mode) {
  ParDims d;
  if (!par_dims(M, K, mode, d)) return 0;
  return (long long)d.nparts * d.nrb * d.S * 64;
}

int jfx_par_prepare_many(int dtype, int n, const double* const* A, const int* shape, void* const* frag, int wait,
                         hipStream_t stream) {
  if (n < 0 || (n && (!A || !shape || !frag))) return set_error("par_prepare: null pointer"), JFX_EARG;
  if (dtype != 0 && dtype != 1) return set_error("par_prepare: dtype must be 0 or 1"), JFX_ESHAPE;
  for (int i = 0; i < n; ++i) {
    const int* s = shape + 4 * i;
    ParDims d;
    if (!A[i] || !frag[i]) return set_error("par_prepare: null pointer"), JFX_EARG;
    if (!par_dims(s[0], s[1], s[2], d) || (s[3] != 1 && s[3] != -1))
      return set_error("par_prepare: bad arguments M=%d K=%d mode=%d", s[0], s[1], s[2]), JFX_ESHAPE;
  }
  for (int i0 = 0; i0 < n; i0 += PAR_JOBS) {
    const int nj = n - i0 < PAR_JOBS ? n - i0 : PAR_JOBS;
    ParJobs jobs = {};
    long long most = 0;
    for (int i = 0; i < nj; ++i) {
      const int* s = shape + 4 * (i0 + i);
      ParDims d;
      par_dims(s[0], s[1], s[2], d);
      jobs.j[i] = ParJob{A[i0 + i], frag[i0 + i], s[0], s[1], s[2], s[3], d.nrb, d.S, d.nparts};
      const long long e = (long long)d.nparts * d.nrb * d.S * 64;
      most = e > most ? e : most;
    }
    const dim3 grid((unsigned)((most + 255) / 256 < 1024 ? (most + 255) / 256 : 1024), (unsigned)nj);
    if (dtype == 0)
      hipLaunchKernelGGL(par_prepare_kernel<double>, grid, dim3(256), 0, stream, jobs);
    else
      hipLaunchKernelGGL(par_prepare_kernel<float>, grid, dim3(256), 0, stream, jobs);
    JFX_LAUNCH_CHECK();
  }
  if (wait) JFX_CHECK_HIP(hipStreamSynchronize(stream));
  return JFX_OK;
}

int jfx_par_prepare(int dtype, const double* A, int M, int K, int mode, int sgn, void* frag, hipStream_t stream) {
  const int shape[4] = {M, K, mode, sgn};
  return jfx_par_prepare_many(dtype, 1, &A, shape, &frag, 0, stream);
}

int jfx_contract_par(int dtype, const void* frag, int M, int K, int mode, int sgn, int bp, int bq, const void* X,
                     void* Y, long long P, long long Q, hipStream_t stream) {
  if (!frag || !X || !Y) return set_error("contract_par: null pointer"), JFX_EARG;
  if (dtype == 0)
    return launch_par<double>((const double*)frag, M, K, mode, sgn, bp, bq, (const double*)X, (double*)Y, P, Q, stream);
  if (dtype == 1)
    return launch_par<float>((const float*)frag, M, K, mode, sgn, bp, bq, (const float*)X, (float*)Y, P, Q, stream);
  return set_error("contract_par: dtype must be 0 or 1"), JFX_EARG;
}

}  // extern "C"
