// Fused two-axis FP64 contractions of 2D slabs by operators with decoupled even
// and odd parts (contract_par.hip):
//     Y[b] = alpha A0 X[b] A1^T,  optionally / E, * E or * E[b],  optionally + Y[b]
// and the fast-diagonalisation solve  Y[b] = scale[b] V0 ((W0 X[b] W1^T) / E) V1^T.
//
// A slab is read once and written once; the intermediate stays in LDS
// (par_blocks.h).  One workgroup per slab: up to 8 waves for 64 x 64 (37 KB of
// LDS), 16 for larger slabs (139 KB at 128 x 128, one workgroup per CU).
#include "par_blocks.h"

namespace jfx {

struct SlabMap {
  ParOp o0, o1;  // axis 0 (M0 x K0), axis 1 (M1 x K1)
  const double* E;
  int epi;  // 0 none, 1 divide by E, 2 multiply by E, 3 multiply by E[b]
  int accum;
  double alpha;
};

template <int MODE, int NW, int JW>
__global__ __launch_bounds__(64 * NW) void plane_par_kernel(const double* __restrict__ X, double* __restrict__ Y,
                                                            SlabMap sm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  double* S = reinterpret_cast<double*>(smem);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K0 = sm.o0.K, K1 = sm.o1.K, M0 = sm.o0.M, M1 = sm.o1.M;
  const long long b = blockIdx.x;
  WaveA<JW> wa;
  ItemB<JW> ib;
  Acc<JW> acc;
  wa.init(w, K0, sm.o1);
  ib.init(w, sm.o0, M1);
  wa.prefetch(sm.o1);
  slab_stage<64 * NW>(X + b * K0 * K1, K0, K1, S);
  __syncthreads();
  acc.zero();
  if (wa.on) phase_a<MODE>(S, slab_ldx(K1), sm.o1, wa, acc);
  ib.prefetch(sm.o0);
  __syncthreads();
  const int LDT = slab_ldt(M1);
  if (wa.on) store_t<MODE>(S, LDT, sm.o1, wa, acc);
  __syncthreads();
  if (!ib.on) return;
  acc.zero();
  phase_b<MODE>(S, LDT, sm.o0, ib, acc);
  double* Yb = Y + b * M0 * M1;
  const double* E = sm.epi == 3 ? sm.E + b * M0 * M1 : sm.E;
  each_b<MODE>(sm.o0, ib, M1, acc, [&](int m, int c, double v) {
    const int i = m * M1 + c;
    v *= sm.alpha;
    if (sm.epi == 1)
      v /= E[i];
    else if (sm.epi)
      v *= E[i];
    if (sm.accum) v += Yb[i];
    Yb[i] = v;
  });
}

// Slabs of which one fills a CU's LDS, several per CU: a persistent workgroup loads
// the next slab into registers while it multiplies the current one.  2048 slabs of
// 128 x 128: 253 us one slab per workgroup, 238 us here (reading and writing take
// 101 us, the FP64 products 119 us; 16 waves in step leave the matrix units idle
// around the barriers: LDS stores of X and T and the stores of Y are 40% of a
// slab's 28 us).  Where two workgroups fit, they overlap by themselves: 512 slabs
// of 96 x 94 36 us, persistent 41 us.
template <int MODE>
__global__ __launch_bounds__(1024) void plane_par_stream_kernel(const double* __restrict__ X, double* __restrict__ Y,
                                                                SlabMap sm, long long B) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  double* S = reinterpret_cast<double*>(smem);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K0 = sm.o0.K, K1 = sm.o1.K, M0 = sm.o0.M, M1 = sm.o1.M, LDT = slab_ldt(M1);
  WaveA<2> wa;
  ItemB<2> ib;
  Acc<2> acc;
  wa.init(w, K0, sm.o1);
  ib.init(w, sm.o0, M1);
  d2 v[8];
  slab_load8<1024>(X + blockIdx.x * (long long)K0 * K1, K0, K1, v);
#pragma unroll 1
  for (long long b = blockIdx.x; b < B; b += gridDim.x) {
    wa.prefetch(sm.o1);
    slab_put8<1024>(v, K0, K1, S);
    __syncthreads();
    const long long bn = b + gridDim.x;
    slab_load8<1024>(X + (bn < B ? bn : b) * K0 * K1, K0, K1, v);
    acc.zero();
    if (wa.on) phase_a<MODE>(S, slab_ldx(K1), sm.o1, wa, acc);
    ib.prefetch(sm.o0);
    __syncthreads();
    if (wa.on) store_t<MODE>(S, LDT, sm.o1, wa, acc);
    __syncthreads();
    acc.zero();
    if (ib.on) {
      phase_b<MODE>(S, LDT, sm.o0, ib, acc);
      double* Yb = Y + b * M0 * M1;
      each_b<MODE>(sm.o0, ib, M1, acc, [&](int m, int c, double y) { Yb[m * M1 + c] = y * sm.alpha; });
    }
    __syncthreads();  // T is free for the next slab
  }
}

struct FdMap {
  ParOp w0, w1, v0, v1;
  const double *E, *scale;  // scale: one factor per slab, or null
};

template <int NW, int JW>
__global__ __launch_bounds__(64 * NW) void plane_fd_par_kernel(const double* __restrict__ X, double* __restrict__ Y,
                                                               FdMap fm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  double* S = reinterpret_cast<double*>(smem);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = fm.w0.K, n1 = fm.w1.K;
  const long long b = blockIdx.x;
  const int LDX = slab_ldx(n1), LDT = slab_ldt(n1);
  WaveA<JW> wa;
  ItemB<JW> ib;
  Acc<JW> acc;
  wa.init(w, n0, fm.w1);
  ib.init(w, fm.w0, n1);
  wa.prefetch(fm.w1);
  slab_stage<64 * NW>(X + b * n0 * n1, n0, n1, S);
  __syncthreads();
  acc.zero();
  if (wa.on) phase_a<MODE_MIX>(S, LDX, fm.w1, wa, acc);
  ib.prefetch(fm.w0);
  __syncthreads();
  if (wa.on) store_t<MODE_MIX>(S, LDT, fm.w1, wa, acc);
  __syncthreads();
  acc.zero();
  if (ib.on) phase_b<MODE_MIX>(S, LDT, fm.w0, ib, acc);
  wa.prefetch(fm.v1);
  __syncthreads();
  // G / E back into LDS as the second pass's input, zero padded like a staged slab
  if (ib.on)
    each_b<MODE_MIX>(fm.w0, ib, n1, acc, [&](int m, int c, double v) { S[m * LDX + c] = v / fm.E[m * n1 + c]; });
  slab_zero_pad<64 * NW>(n0, n1, S);
  __syncthreads();
  acc.zero();
  if (wa.on) phase_a<MODE_MIX>(S, LDX, fm.v1, wa, acc);
  ib.prefetch(fm.v0);
  __syncthreads();
  if (wa.on) store_t<MODE_MIX>(S, LDT, fm.v1, wa, acc);
  __syncthreads();
  if (!ib.on) return;
  acc.zero();
  phase_b<MODE_MIX>(S, LDT, fm.v0, ib, acc);
  double* Yb = Y + b * n0 * n1;
  const double f = fm.scale ? fm.scale[b] : 1.0;
  each_b<MODE_MIX>(fm.v0, ib, n1, acc, [&](int m, int c, double v) { Yb[m * n1 + c] = v * f; });
}

bool par_op(const double* frag, int M, int K, int mode, int sgn, int bp, int bq, ParOp& o);

// More than three slabs per CU of more than 32 rows: four waves with two blocks
// each (six workgroups a CU overlap each other, and a wave's operator fragments
// serve two blocks).  Fewer slabs, and slabs up to 32 x 32 whose workgroup is four
// waves anyway: one block a wave, fragments loaded ahead.  us, two blocks / one:
// 62 x 62 -> 64 x 64: 256 slabs 11.5 / 9.5, 768 20.7 / 20.8, 4096 75.7 / 81.7;
// 48 x 48 solves: 256 15.6 / 11.1, 768 25.2 / 25.2, 4096 102 / 112;
// 30 x 30 solves: 256 12.0 / 8.4, 4096 59.7 / 33.5.
static bool slab_many(long long B, int items) { return items > 4 && B > 3 * 256; }
static bool slab_small(const ParOp& o) { return o.M <= 64 && o.K <= 64; }

template <typename K>
static int slab_shm(K kern, size_t shm) {
  if (shm > 64 * 1024)
    JFX_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
  return JFX_OK;
}

template <int MODE, int NW, int JW>
static int launch_plane(const double* X, double* Y, const SlabMap& sm, long long B, hipStream_t st) {
  const size_t shm = (size_t)slab_lds(sm.o0.K, sm.o1.K, sm.o1.M) * sizeof(double);
  const int rc = slab_shm(plane_par_kernel<MODE, NW, JW>, shm);
  if (rc) return rc;
  hipLaunchKernelGGL((plane_par_kernel<MODE, NW, JW>), dim3((unsigned)B), dim3(64 * NW), shm, st, X, Y, sm);
  JFX_LAUNCH_CHECK();
  return JFX_OK;
}

template <int MODE>
static int launch_plane_w(const double* X, double* Y, const SlabMap& sm, long long B, hipStream_t st) {
  if (slab_small(sm.o0) && slab_small(sm.o1)) {
    const int n = slab_items<1>(sm.o0.K, sm.o0, sm.o1);
    if (slab_many(B, n)) return launch_plane<MODE, 4, 2>(X, Y, sm, B, st);
    if (n <= 2) return launch_plane<MODE, 2, 1>(X, Y, sm, B, st);
    if (n <= 4) return launch_plane<MODE, 4, 1>(X, Y, sm, B, st);
    if (n <= 6) return launch_plane<MODE, 6, 1>(X, Y, sm, B, st);
    return launch_plane<MODE, 8, 1>(X, Y, sm, B, st);
  }
  const int n = slab_items<2>(sm.o0.K, sm.o0, sm.o1);
  const size_t shm = (size_t)slab_lds(sm.o0.K, sm.o1.K, sm.o1.M) * sizeof(double);
  if (n > 8 && B > 256 && shm > 80 * 1024 && !sm.epi && !sm.accum && sm.o1.K % 2 == 0 && ((uintptr_t)X & 15) == 0) {
    const int rc = slab_shm(plane_par_stream_kernel<MODE>, shm);
    if (rc) return rc;
    hipLaunchKernelGGL(plane_par_stream_kernel<MODE>, dim3(256), dim3(1024), shm, st, X, Y, sm, B);
    JFX_LAUNCH_CHECK();
    return JFX_OK;
  }
  return n <= 8 ? launch_plane<MODE, 8, 2>(X, Y, sm, B, st) : launch_plane<MODE, 16, 2>(X, Y, sm, B, st);
}

template <int NW, int JW>
static int launch_fd(const double* X, double* Y, const FdMap& fm, long long B, hipStream_t st) {
  const size_t shm = (size_t)slab_lds(fm.w0.K, fm.w1.K, fm.w1.M) * sizeof(double);
  const int rc = slab_shm(plane_fd_par_kernel<NW, JW>, shm);
  if (rc) return rc;
  hipLaunchKernelGGL((plane_fd_par_kernel<NW, JW>), dim3((unsigned)B), dim3(64 * NW), shm, st, X, Y, fm);
  JFX_LAUNCH_CHECK();
  return JFX_OK;
}

}  // namespace jfx

using namespace jfx;

extern "C" {

int jfx_plane_par(int mode, const double* F0, int M0, int K0, int sgn0, int bp0, int bq0, const double* F1, int M1,
                  int K1, int sgn1, int bp1, int bq1, const double* X, double* Y, const double* E, int epi,
                  double alpha, int accum, long long B, hipStream_t stream) {
  if (!F0 || !F1 || !X || !Y || (epi && !E)) return set_error("plane_par: null pointer"), JFX_EARG;
  if (epi < 0 || epi > 3) return set_error("plane_par: epi must be 0..3"), JFX_EARG;
  SlabMap sm;
  if (mode < MODE_EVAL || mode > MODE_MIX || !par_op(F0, M0, K0, mode, sgn0, bp0, bq0, sm.o0) ||
      !par_op(F1, M1, K1, mode, sgn1, bp1, bq1, sm.o1) || M0 > SLAB_MAX || K0 > SLAB_MAX || M1 > SLAB_MAX ||
      K1 > SLAB_MAX || B < 0 || B > 0x7fffffffLL)
    return set_error("plane_par: sizes (%d x %d), (%d x %d), %lld slabs, mode %d", M0, K0, M1, K1, B, mode), JFX_ESHAPE;
  if (B == 0) return JFX_OK;
  sm.E = E;
  sm.epi = epi;
  sm.alpha = alpha;
  sm.accum = accum;
  switch (mode) {
    case MODE_EVAL: return launch_plane_w<MODE_EVAL>(X, Y, sm, B, stream);
    case MODE_PROJ: return launch_plane_w<MODE_PROJ>(X, Y, sm, B, stream);
    default: return launch_plane_w<MODE_MIX>(X, Y, sm, B, stream);
  }
}

int jfx_plane_fd_par(const double* W0, const double* W1, const double* V0, const double* V1, const double* X,
                     double* Y, const double* E, const double* scale, long long B, int n0, int n1,
                     hipStream_t stream) {
  if (!W0 || !W1 || !V0 || !V1 || !X || !Y || !E) return set_error("plane_fd_par: null pointer"), JFX_EARG;
  FdMap fm;
  if (!par_op(W0, n0, n0, MODE_MIX, 1, -1, -1, fm.w0) || !par_op(W1, n1, n1, MODE_MIX, 1, -1, -1, fm.w1) ||
      !par_op(V0, n0, n0, MODE_MIX, 1, -1, -1, fm.v0) || !par_op(V1, n1, n1, MODE_MIX, 1, -1, -1, fm.v1) ||
      n0 > SLAB_MAX || n1 > SLAB_MAX || B < 0 || B > 0x7fffffffLL)
    return set_error("plane_fd_par: %lld slabs of %d x %d", B, n0, n1), JFX_ESHAPE;
  if (B == 0) return JFX_OK;
  fm.E = E;
  fm.scale = scale;
  if (slab_small(fm.w0) && slab_small(fm.w1)) {
    const int n = slab_items<1>(n0, fm.w0, fm.w1);
    if (slab_many(B, n)) return launch_fd<4, 2>(X, Y, fm, B, stream);
    if (n <= 2) return launch_fd<2, 1>(X, Y, fm, B, stream);
    if (n <= 4) return launch_fd<4, 1>(X, Y, fm, B, stream);
    if (n <= 6) return launch_fd<6, 1>(X, Y, fm, B, stream);
    return launch_fd<8, 1>(X, Y, fm, B, stream);
  }
  return slab_items<2>(n0, fm.w0, fm.w1) <= 8 ? launch_fd<8, 2>(X, Y, fm, B, stream)
                                              : launch_fd<16, 2>(X, Y, fm, B, stream);
}

}  // extern "C"
