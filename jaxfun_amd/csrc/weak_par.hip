// Variable-coefficient Laplacian of 2D slabs in weak form, FP64:
//     Y[b] = TD (k[b] * (D U B^T)) TB^T + TB (k[b] * (B U D^T)) TD^T
// with B, D (Q x n) a parity basis and its derivative on a symmetric mesh and TB,
// TD (n x Q) their weighted transposes: the operator of -div(k grad u), eight
// contractions, two products and a sum, in one launch.
//
// One workgroup per slab keeps everything between U and Y on chip: each half of
// the sum is an evaluation pass into registers, a product with k on the way back
// into LDS and a projection pass whose results add up in registers over the
// halves (par_blocks.h).  U is staged again for the second half (from L2), so
// that one LDS buffer serves every pass: 37 KB at 64 x 64, four workgroups per
// CU.  256 slabs of 62 x 62 on a 64 x 64 mesh: 8 contractions, 2 products and a
// sum in separate launches 115 us, here 30 us; the FP64 products alone take 7 us,
// so latency bounds it (eight phases with barriers between them per slab).
#include "par_blocks.h"

namespace jfx {

struct WeakMap {
  ParOp b, d, tb, td;
};

template <int NW, int JW>
__global__ __launch_bounds__(64 * NW) void weak_par_kernel(const double* __restrict__ U, const double* __restrict__ kq,
                                                           double* __restrict__ Y, WeakMap wm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  double* S = reinterpret_cast<double*>(smem);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = wm.b.K, Q = wm.b.M;
  const long long b = blockIdx.x;
  const double* kb = kq + b * Q * Q;
  const int LXn = slab_ldx(n), LXq = slab_ldx(Q), LTn = slab_ldt(n), LTq = slab_ldt(Q);
  Acc<JW> acc, sum;
  sum.zero();
  WaveA<JW> we, wp;
  ItemB<JW> ie, ip;
  we.init(w, n, wm.b);
  wp.init(w, Q, wm.tb);
  ie.init(w, wm.b, Q);
  ip.init(w, wm.tb, n);
  we.prefetch(wm.b);
#pragma unroll 1
  for (int t = 0; t < 2; ++t) {
    const ParOp &e0 = t ? wm.b : wm.d, &e1 = t ? wm.d : wm.b, &p0 = t ? wm.tb : wm.td, &p1 = t ? wm.td : wm.tb;
    // opaque copies: without them the loads and addresses that both halves share
    // are hoisted out of the loop and held in 150 registers
    const double *Ut = U + b * n * n, *kt = kb;
    asm volatile("" : "+s"(Ut), "+s"(kt));
    slab_stage<64 * NW>(Ut, n, n, S);
    __syncthreads();
    acc.zero();
    if (we.on) phase_a<MODE_EVAL>(S, LXn, e1, we, acc);
    ie.prefetch(e0);
    __syncthreads();
    if (we.on) store_t<MODE_EVAL>(S, LTq, e1, we, acc);
    __syncthreads();
    acc.zero();
    if (ie.on) phase_b<MODE_EVAL>(S, LTq, e0, ie, acc);
    wp.prefetch(p1);
    __syncthreads();
    if (ie.on) each_b<MODE_EVAL>(e0, ie, Q, acc, [&](int m, int c, double v) { S[m * LXq + c] = v * kt[m * Q + c]; });
    slab_zero_pad<64 * NW>(Q, Q, S);
    __syncthreads();
    acc.zero();
    if (wp.on) phase_a<MODE_PROJ>(S, LXq, p1, wp, acc);
    ip.prefetch(p0);
    __syncthreads();
    if (wp.on) store_t<MODE_PROJ>(S, LTn, p1, wp, acc);
    __syncthreads();
    if (ip.on) phase_b<MODE_PROJ>(S, LTn, p0, ip, sum);
    if (t == 0) {
      we.prefetch(wm.d);
      __syncthreads();
    }
  }
  if (ip.on) {
    double* Yb = Y + b * n * n;
    each_b<MODE_PROJ>(wm.tb, ip, n, sum, [&](int m, int c, double v) { Yb[m * n + c] = v; });
  }
}

bool par_op(const double* frag, int M, int K, int mode, int sgn, int bp, int bq, ParOp& o);

template <int NW, int JW>
static int launch_weak(const double* U, const double* kq, double* Y, const WeakMap& wm, long long B, hipStream_t st) {
  const int a = slab_lds(wm.b.K, wm.b.K, wm.b.M), c = slab_lds(wm.b.M, wm.b.M, wm.b.K);
  const size_t shm = (size_t)(a > c ? a : c) * sizeof(double);
  if (shm > 64 * 1024)
    JFX_CHECK_HIP(hipFuncSetAttribute((const void*)weak_par_kernel<NW, JW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)shm));
  hipLaunchKernelGGL((weak_par_kernel<NW, JW>), dim3((unsigned)B), dim3(64 * NW), shm, st, U, kq, Y, wm);
  JFX_LAUNCH_CHECK();
  return JFX_OK;
}

}  // namespace jfx

using namespace jfx;

extern "C" {

int jfx_weak_par(const double* FB, int sB, const double* FD, int sD, const double* FTB, int sTB, const double* FTD,
                 int sTD, int n, int Q, const double* U, const double* k, double* Y, long long B, hipStream_t stream) {
  if (!FB || !FD || !FTB || !FTD || !U || !k || !Y) return set_error("weak_par: null pointer"), JFX_EARG;
  WeakMap wm;
  if (!par_op(FB, Q, n, MODE_EVAL, sB, -1, -1, wm.b) || !par_op(FD, Q, n, MODE_EVAL, sD, -1, -1, wm.d) ||
      !par_op(FTB, n, Q, MODE_PROJ, sTB, -1, -1, wm.tb) || !par_op(FTD, n, Q, MODE_PROJ, sTD, -1, -1, wm.td) ||
      n > SLAB_MAX || Q > SLAB_MAX || B < 0 || B > 0x7fffffffLL)
    return set_error("weak_par: %lld slabs, n = %d, Q = %d", B, n, Q), JFX_ESHAPE;
  if (B == 0) return JFX_OK;
  if (Q <= 64 && n <= 64) {
    const int a = slab_items<1>(n, wm.b, wm.b), c = slab_items<1>(Q, wm.tb, wm.tb), m = a > c ? a : c;
    return m <= 2   ? launch_weak<2, 1>(U, k, Y, wm, B, stream)
           : m <= 4 ? launch_weak<4, 1>(U, k, Y, wm, B, stream)
                    : launch_weak<8, 1>(U, k, Y, wm, B, stream);
  }
  const int a = slab_items<2>(n, wm.b, wm.b), c = slab_items<2>(Q, wm.tb, wm.tb);
  return (a > c ? a : c) <= 8 ? launch_weak<8, 2>(U, k, Y, wm, B, stream) : launch_weak<16, 2>(U, k, Y, wm, B, stream);
}

}  // extern "C"
