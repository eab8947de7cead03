// RBF (Gaussian) kernel matrix, forward and backward, fp32, for MI355X
// (gfx950).  C-ABI declared in include/rbf.h.
//
// Reference semantics (cases/rbf/reference.py:14-20, delivery/README.md:8-12):
//   K[i,j] = exp(-gamma * sum_d (X[i,d] - Y[j,d])^2)
//   backward with upstream dK: W = dK o K,
//   dX[i] = -2 gamma * sum_j W[i,j] (X[i] - Y[j])
//   dY[j] = -2 gamma * sum_i W[i,j] (Y[j] - X[i])
//
// Design:
//  * Forward: K[i,j] = exp2(min(2 kappa x_i.y_j - kappa (|x_i|^2 + |y_j|^2), 0))
//    with kappa = gamma log2(e): at D = 64 on bf16 splits of the fp32 rows
//    (csrc/pairwise_split.h), else in 64 bits (rbf_fwd_kernel), at any D and
//    alignment.  Tiles whose distances that form would round too coarsely
//    (split_norm_max, f64_norm_max) go from the splits to 64 bits or to the
//    squared differences summed directly on SIMT tiles, from 64 bits to those.
//  * Backward: one pass over dK and K per 64 features.  Workgroups own
//    regions of W = dK o K and write raw partial contractions W . Y and
//    W^T . X and partial row and column sums of W to workspace slots, on the
//    bf16 splits or, for small shapes at D = 64, on fp32 MFMA
//    (csrc/pairwise_d64.h); rbf_bwd_reduce_kernel sums the slots and applies
//    dX = -2 gamma (rowsum(W) X - W Y), dY = -2 gamma (colsum(W) Y - W^T X).
//  * Without a workspace, or past the kernels' ranges, tiled SIMT
//    kernels run: W formed in LDS and walked in slices whose partial sums a
//    reduce kernel adds in order (unsplit when the caller passes no workspace
//    for them).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>

#include "../../../csrc/common.h"
#include "../../../csrc/pairwise_d64.h"
#include "../../../csrc/pairwise_generic.h"
#include "../../../csrc/pairwise_split.h"
#include "rbf.h"

using nl2k::f32x2;
using nl2k::f32x4;
using nl2k::pairwise::kD;

namespace {

constexpr double kLog2e = 1.4426950408889634;

// Forward policy of the SIMT tiles: the squared differences summed directly,
// as the reference kernel does.
struct RbfGenFwd {
  float gamma;
  __device__ __forceinline__ float x_in(float v, int64_t) const { return v; }
  __device__ __forceinline__ float y_in(float v, int64_t) const { return v; }
  __device__ __forceinline__ float step(float s, float x, float y) const {
    const float t = x - y;
    return fmaf(t, t, s);
  }
  __device__ __forceinline__ float out(float s) const { return expf(-gamma * s); }
};

// Backward policy: W = dK o K, raw X / Y rows, row and column sums of W.
struct RbfBwdOp {
  static constexpr bool kProduct = true, kScale = false, kSums = true;
};

// ------------------------------------------------------------------- forward
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x2_u __attribute__((ext_vector_type(2), aligned(4)));

// K = exp2(-kappa max(|x|^2 + |y|^2 - 2 x.y, 0)), the distance in 64 bits on
// v_mfma_f64_16x16x4_f64: fp32 products are exact there, and what the
// difference of norms and products loses is 2^-52 of the norms, so near rows
// keep their distance, K(x, x) = 1 and K(X, X) is symmetric.
// A workgroup of four waves takes 64 x 64 outputs, a wave 32 x 32: two blocks
// of 16 rows (operand A, X), and two of every second column (operand B, Y), so
// that a lane's outputs of a row lie side by side.  Lane (n, h) holds four
// features of a row, k + 4 h .. + 3, straight from global memory (the next 16
// features are in flight while these are multiplied), and the norms are summed
// from the same registers.
// A tile with a norm past norm_max, or one that is not finite, sums the
// squared differences directly; a wave that sees so in the first features
// skips the rest.
// Bound by the matrix instruction, which takes 120 cycles on a full chip (42
// TFLOP/s).  Against the squared differences summed in fp32 on SIMT tiles:
// 53 -> 39 us at 3000 x 2500 x 100, 20 -> 9.2 at 1000 x 1000 x 100, 39 -> 33
// at 4096^2 x 32, 104 -> 82 at 4096^2 x 128.  Error of K against 64 bits
// (2-norm) 1.4e-7 -> 3.4e-8 at D = 100.  (bf16 splits take 21 us at 3000 x 2500
// x 100, but a pair of rows 1 % apart is off by 7e-8 at gamma |x|^2 = 0.5 and
// 6e-7 at 4 there, against 2e-8 directly.)
constexpr int kFwdTile = 64;
struct RbfF64 {
  double neg_kappa;  // -gamma log2(e)
  double norm_max;
  float gamma;
};
__device__ __forceinline__ void rbf_f64_tile(nl2k::pairwise::SimtTile& simt,
                                             const float* __restrict__ X,
                                             const float* __restrict__ Y, float* __restrict__ K,
                                             int N, int M, int D, int i0, int j0,
                                             const RbfF64& op) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n = lane & 15, h = lane >> 4;
  const int ib = i0 + (wave >> 1) * 32, j = j0 + (wave & 1) * 32 + 2 * n;
  const float* src[4];  // rows ib + n, + 16 of X, rows j, j + 1 of Y
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    src[b] = X + (size_t)min(ib + 16 * b + n, N - 1) * D;
    src[2 + b] = Y + (size_t)min(j + b, M - 1) * D;
  }
  f64x4 acc[2][2];
  double nsq[4];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    nsq[a] = nsq[2 + a] = 0.;
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f64x4{0., 0., 0., 0.};
  }
  auto step = [&](const float (&x)[4]) {  // one feature of each row a lane
    double v[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      v[s] = (double)x[s];
      nsq[s] = fma(v[s], v[s], nsq[s]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[a], v[2 + b], acc[a][b], 0, 0, 0);
  };
  f32x4 nxt[4];
  auto load = [&](int k) {
#pragma unroll
    for (int s = 0; s < 4; ++s) nxt[s] = nl2k::pairwise::load4_u(src[s] + k + 4 * h);
  };
  bool direct = false;
  auto check_norms = [&] {
#pragma unroll
    for (int s = 0; s < 4; ++s) direct |= !(nsq[s] <= op.norm_max);
  };
  const int whole = D & ~15;
  if (whole > 0) load(0);
  for (int k = 0; k < whole; k += 16) {
    f32x4 cur[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) cur[s] = nxt[s];
    if (k + 16 < whole) load(k + 16);
#pragma unroll
    for (int u = 0; u < 4; ++u) step({cur[0][u], cur[1][u], cur[2][u], cur[3][u]});
    if (k == 0) {
      check_norms();
      if (__any(direct)) break;
    }
  }
  for (int k = whole; k < D; k += 4) {  // the last features, four at a time: zeros past D
    float x[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = src[s][min(k + h, D - 1)];
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = k + h < D ? x[s] : 0.f;
    step(x);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {  // over the row's four lanes
    nsq[s] += __shfl_xor(nsq[s], 16, 64);
    nsq[s] += __shfl_xor(nsq[s], 32, 64);
  }
  check_norms();
  if (__syncthreads_or(direct)) {
    nl2k::pairwise::simt_fwd_tile(simt, X, Y, K, (int64_t)N, (int64_t)M, (int64_t)D, (int64_t)i0,
                                  (int64_t)j0, RbfGenFwd{op.gamma});
    return;
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // accumulator r of lane (n, h): row 4 r + h, column n
      const double nx = __shfl(nsq[a], 4 * r + h, 64);
      const int i = ib + 16 * a + 4 * r + h;
      float o[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const double d2 = fma(-2., acc[a][b][r], nx + nsq[2 + b]);
        o[b] = exp2f((float)(op.neg_kappa * fmax(d2, 0.)));
      }
      if (i >= N) continue;
      float* p = K + (size_t)i * M + j;
      if (j + 1 < M)
        *reinterpret_cast<f32x2_u*>(p) = f32x2{o[0], o[1]};
      else if (j < M)
        p[0] = o[0];
    }
}

__global__ __launch_bounds__(256, 2) void rbf_fwd_kernel(const float* __restrict__ X,
                                                         const float* __restrict__ Y,
                                                         float* __restrict__ K, int N, int M,
                                                         int D, RbfF64 op, int n_jt) {
  __shared__ __attribute__((aligned(16))) nl2k::pairwise::SimtTile simt;
  rbf_f64_tile(simt, X, Y, K, N, M, D, (int)(blockIdx.x / n_jt) * kFwdTile,
               (int)(blockIdx.x % n_jt) * kFwdTile, op);
}

// Forward policy on the splits: the row term is -kappa |x|^2, the column term
// |y|^2, and K = exp2(min(2 kappa x.y - kappa (|x|^2 + |y|^2), 0)); the clamp
// keeps K <= 1 when the distance cancels to a tiny negative value.
struct RbfFwdOp {
  float neg_kappa;  // -gamma log2(e)
  float norm_max;
  RbfF64 f64;  // for tiles with larger norms
  static constexpr bool kScale = false, kDirect = true;
  __device__ __forceinline__ float row(float sx) const { return neg_kappa * sx; }
  __device__ __forceinline__ float col(float sy) const { return sy; }
  __device__ __forceinline__ float out(float dot, float rt, float ct) const {
    float t = fmaf(-2.f * neg_kappa, dot, fmaf(neg_kappa, ct, rt));
    t = t > 0.f ? 0.f : t;  // squared distance >= 0; NaN passes through
    return __builtin_amdgcn_exp2f(t);
  }
  // Workgroups of 128 x 128 have the registers for 64 bits (4096^2: 63-72 us, 87-99
  // with the sum on SIMT tiles, two of them a CU); in those of 64 x 64 they cost
  // the split itself (17.2 -> 18.1 us at 3000^2).
  template <int TB>
  __device__ __forceinline__ void direct(nl2k::pairwise::SimtTile& t, const float* X,
                                         const float* Y, float* K, int N, int M, int D, int i0,
                                         int j0) const {
    if constexpr (TB == 128)
      rbf_f64_tile(t, X, Y, K, N, M, D, i0, j0, f64);
    else
      nl2k::pairwise::simt_fwd_tile(t, X, Y, K, (int64_t)N, (int64_t)M, (int64_t)D, (int64_t)i0,
                                    (int64_t)j0, RbfGenFwd{f64.gamma});
  }
};

// ------------------------------------------------------------------ backward
// One side of the backward: its own rows A and their gradient, the other
// side's rows B, entry (r, o) of dK and K at r own + o other.
struct ReduceSide {
  const float *P, *S, *A, *B;
  float* out;
  int64_t rows, others;
  size_t own, other;
  int slots;
};

// out[r][:] = neg2g (sum_s S[s][r] A[r][:] - sum_s P[s][r][:]), one thread
// per V features (V = 4 when D is a multiple of 4: rows then hold whole
// groups); the slot loop is unrolled by 4 so that the loads of several slots
// are in flight together.  Split partials carry kSplitScale and are added up
// directly where they are not finite.
template <int V, bool SPLIT, typename I>
__device__ __forceinline__ void reduce_side(const ReduceSide& side, const float* __restrict__ dK,
                                            const float* __restrict__ K, int D, float neg2g,
                                            I first, I step) {
  typedef float vec __attribute__((ext_vector_type(V), aligned(4)));
  const float* __restrict__ P = side.P;
  const float* __restrict__ S = side.S;
  const int64_t rows = side.rows;
  const int slots = side.slots;
  const I per = (I)(D / V), groups = (I)(rows * per);
  const size_t stride = (size_t)rows * D;
  for (I e = first; e < groups; e += step) {
    const I r = e / per;
    const float* p = P + (size_t)e * V;
    const float* q = S + r;
    auto at = [&](int s) { return *reinterpret_cast<const vec*>(p + (size_t)s * stride); };
    vec a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    int s = 0;
    for (; s + 4 <= slots; s += 4) {
      a0 += at(s);
      a1 += at(s + 1);
      a2 += at(s + 2);
      a3 += at(s + 3);
      s0 += q[(size_t)s * rows];
      s1 += q[(size_t)(s + 1) * rows];
      s2 += q[(size_t)(s + 2) * rows];
      s3 += q[(size_t)(s + 3) * rows];
    }
    for (; s < slots; ++s) {
      a0 += at(s);
      s0 += q[(size_t)s * rows];
    }
    vec acc = (a0 + a1) + (a2 + a3);
    float sum = (s0 + s1) + (s2 + s3);
    if constexpr (SPLIT) {
      bool finite = fabsf(sum) < INFINITY;
#pragma unroll
      for (int v = 0; v < V; ++v) finite &= fabsf(acc[v]) < INFINITY;
      sum *= nl2k::pairwise::kSumUnscale;
      acc *= nl2k::pairwise::kPartialUnscale;
      if (__builtin_expect(!finite, 0))
        nl2k::pairwise::direct_sums<RbfBwdOp>(dK, K, (size_t)r * side.own, side.other,
                                              side.B + (size_t)(e - r * per) * V, nullptr,
                                              side.others, D, acc, sum);
    }
    const vec a = *reinterpret_cast<const vec*>(side.A + (size_t)e * V);
    *reinterpret_cast<vec*>(side.out + (size_t)e * V) = neg2g * (sum * a - acc);
  }
}

// Both outputs in one launch: block b < bx handles dX, the rest dY.
template <int V, bool SPLIT, typename I>
__global__ __launch_bounds__(256) void rbf_bwd_reduce_kernel(ReduceSide x, ReduceSide y,
                                                             const float* __restrict__ dK,
                                                             const float* __restrict__ K, int D,
                                                             int bx, float neg2g) {
  const int b = (int)blockIdx.x;
  if (b < bx)
    reduce_side<V, SPLIT, I>(x, dK, K, D, neg2g, (I)b * 256 + threadIdx.x, (I)bx * 256);
  else
    reduce_side<V, SPLIT, I>(y, dK, K, D, neg2g, (I)(b - bx) * 256 + threadIdx.x,
                             (I)((int)gridDim.x - bx) * 256);
}

// ------------------------------------------------------- generic (any D)
// Policies of the tiled SIMT kernels (csrc/pairwise_generic.h).
struct RbfGenBwd {
  float neg2g;
  static constexpr bool kSums = true;
  __device__ __forceinline__ float w(const float* __restrict__ dK, const float* __restrict__ K,
                                     int64_t idx) const {
    return dK[idx] * K[idx];
  }
  template <bool TRANS>
  __device__ __forceinline__ float b_in(float v, int64_t) const {
    return v;
  }
  __device__ __forceinline__ float finish(float rs, float a, float acc) const {
    return neg2g * (rs * a - acc);
  }
};

// out[r][d] = neg2g (sum_s psum[s][r] a[r][d] - sum_s pacc[s][r][d]), the
// slices added in order; block b < bx writes dX, the rest dY.
__global__ __launch_bounds__(256) void rbf_bwd_generic_reduce_kernel(
    const float* __restrict__ px, const float* __restrict__ sx, const float* __restrict__ X,
    float* __restrict__ dX, int64_t N, int64_t Sx, const float* __restrict__ py,
    const float* __restrict__ sy, const float* __restrict__ Y, float* __restrict__ dY, int64_t M,
    int64_t Sy, int64_t D, int bx, float neg2g) {
  const bool is_x = (int)blockIdx.x < bx;
  const float* __restrict__ P = is_x ? px : py;
  const float* __restrict__ Q = is_x ? sx : sy;
  const float* __restrict__ A = is_x ? X : Y;
  float* __restrict__ out = is_x ? dX : dY;
  const int64_t rows = is_x ? N : M, S = is_x ? Sx : Sy;
  const int64_t b0 = is_x ? 0 : bx, nb = is_x ? bx : (int64_t)gridDim.x - bx;
  const int64_t total = rows * D;
  for (int64_t e = ((int64_t)blockIdx.x - b0) * blockDim.x + threadIdx.x; e < total;
       e += nb * blockDim.x) {
    const int64_t r = e / D;
    float acc = 0.f, rs = 0.f;
    for (int64_t sl = 0; sl < S; ++sl) {
      acc += P[sl * total + e];
      rs += Q[sl * rows + r];
    }
    out[e] = neg2g * (rs * A[e] - acc);
  }
}

__global__ __launch_bounds__(256) void rbf_fill_zero_kernel(float* __restrict__ p,
                                                           size_t count) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < count;
       e += (size_t)gridDim.x * blockDim.x)
    p[e] = 0.f;
}

// ------------------------------------------------------------------ host side
int validate_sizes(int64_t N, int64_t M, int64_t D) {
  if (N < 0 || M < 0 || D < 1)
    return nl2k::fail(NL2K_ERR_SHAPE,
                      "rbf: sizes must satisfy N >= 0, M >= 0, D >= 1 (got N=%lld M=%lld D=%lld)",
                      (long long)N, (long long)M, (long long)D);
  const int64_t lim = INT32_MAX;
  if (N > lim || M > lim || D > lim || (D > 0 && (N > INT64_MAX / D || M > INT64_MAX / D)) ||
      (M > 0 && N > INT64_MAX / M))
    return nl2k::fail(NL2K_ERR_OVERFLOW, "rbf: sizes too large (N=%lld M=%lld D=%lld)",
                      (long long)N, (long long)M, (long long)D);
  return NL2K_SUCCESS;
}

// Workspace floats of the generic backward's slices (0 when neither side splits).
inline size_t generic_ws_floats(int64_t N, int64_t M, int64_t D) {
  if (N <= 0 || M <= 0) return 0;
  const nl2k::pairwise::GenericSplit gx = nl2k::pairwise::generic_split(N, M, D),
                                     gy = nl2k::pairwise::generic_split(M, N, D);
  if (gx.s == 1 && gy.s == 1) return 0;
  return (size_t)(gx.s * N * (D + 1) + gy.s * M * (D + 1));
}

// What rbf_backward_workspace_bytes reports, in floats: callers hold buffers
// of this size, and the split backward is cut so that its partials fit.  At
// D = 64 it is the fp32 regions' (pairwise_d64.h).
inline size_t workspace_floats(int64_t N, int64_t M, int64_t D) {
  if (N <= 0 || M <= 0) return 0;
  const nl2k::pairwise::BwdPlan p = nl2k::pairwise::plan_backward(N, M, D, true);
  if (p.fast) return p.ws_floats;
  return std::max(generic_ws_floats(N, M, D), nl2k::pairwise::split_floats(N, M, D, true));
}

// Forward route: D = 64 with 16-byte aligned X, Y on the bf16 splits, whose
// rounding there is that of the fp32 instructions (24.5 us at 4096^2; 64-bit
// distances take 51, fp32 instructions 30), everything else in 64 bits: as the
// reference sums squared differences, near rows keep their distance.
bool takes_split_forward(int64_t D, const float* X, const float* Y) {
  return D == kD && nl2k::aligned16(X) && nl2k::aligned16(Y);
}

// Largest squared row norm whose distances come from norms and products, |x|^2
// + |y|^2 - 2 x.y.  That leaves an error in the distance of about 2^-24 of |x|^2
// + |y|^2 on the splits and 2^-52 in 64 bits, whatever the distance is, and gamma
// carries it into K: a few 1e-7 at gamma |x|^2 = 4, and a quarter of K's last
// bit at gamma |x|^2 = 2^24.  A tile on the splits with a larger norm goes to 64
// bits or to the direct sum (RbfFwdOp::direct), one in 64 bits with a larger
// one, or one that is not finite, to the direct sum.
// A negative or NaN gamma always sums directly.
inline float split_norm_max(float gamma) {
  if (!(gamma >= 0.f)) return -1.f;
  return gamma <= 4e-30f ? 1e30f : 4.f / gamma;
}
inline double f64_norm_max(float gamma) {
  if (!(gamma >= 0.f)) return -1.;
  return gamma == 0.f ? 1e300 : 16777216. / gamma;
}

int launch_fill_zero(float* p, size_t count, hipStream_t stream) {
  if (count == 0) return NL2K_SUCCESS;
  const int blocks = (int)std::min<size_t>((count + 255) / 256, 4096);
  hipLaunchKernelGGL(rbf_fill_zero_kernel, dim3(blocks), dim3(256), 0, stream, p, count);
  return nl2k::check_launch("rbf fill");
}

// D == 64 and 16-byte aligned X, Y, dX and dY: the workspace is required.
// Any other call runs without one (or with a shorter one) on the generic
// kernels, their walks whole.
bool needs_workspace(int64_t N, int64_t M, int64_t D, const float* X, const float* Y,
                     const float* dX, const float* dY) {
  using nl2k::pairwise::kMaxTileDim;
  return D == kD && N <= kMaxTileDim && M <= kMaxTileDim && nl2k::aligned16(X) && nl2k::aligned16(Y) &&
         nl2k::aligned16(dX) && nl2k::aligned16(dY);
}

template <bool SPLIT, class Plan>
int reduce(const Plan& p, const float* ws, const float* X, const float* Y, const float* dK,
           const float* K, float* dX, float* dY, int64_t N, int64_t M, int64_t D, float neg2g,
           hipStream_t stream, const char* who) {
  const int64_t v = D % 4 == 0 ? 4 : 1;
  const int64_t gx = N * (D / v), gy = M * (D / v);
  const int bx = (int)std::min<int64_t>(nl2k::ceil_div(gx, (int64_t)256), 2048);
  const int by = (int)std::min<int64_t>(nl2k::ceil_div(gy, (int64_t)256), 2048);
  const bool small = std::max(gx, gy) < (int64_t(1) << 31);  // the strides fit 32 bits beside it
  auto* kernel = v == 4 ? (small ? &rbf_bwd_reduce_kernel<4, SPLIT, uint32_t>
                                 : &rbf_bwd_reduce_kernel<4, SPLIT, uint64_t>)
                        : (small ? &rbf_bwd_reduce_kernel<1, SPLIT, uint32_t>
                                 : &rbf_bwd_reduce_kernel<1, SPLIT, uint64_t>);
  const ReduceSide x = {ws + p.px, ws + p.rx, X, Y, dX, N, M, (size_t)M, 1, p.nRJ};
  const ReduceSide y = {ws + p.py, ws + p.ry, Y, X, dY, M, N, 1, (size_t)M, p.nRI};
  hipLaunchKernelGGL(kernel, dim3(bx + by), dim3(256), 0, stream, x, y, dK, K, (int)D, bx, neg2g);
  return nl2k::check_launch(who);
}

// Both backward entry points: the caller's workspace, or the scratch array
// below for rbf_backward_f32_noalloc.
int backward_impl(const float* X, const float* Y, const float* dK, const float* K, float* dX,
                  float* dY, int64_t N, int64_t M, int64_t D, float gamma, void* workspace,
                  size_t workspace_bytes, hipStream_t stream, const char* who) {
  int st = validate_sizes(N, M, D);
  if (st) return st;
  if (N == 0 && M == 0) return nl2k::succeed();
  if ((N > 0 && (!X || !dX)) || (M > 0 && (!Y || !dY)))
    return nl2k::fail(NL2K_ERR_NULL, "%s: X, Y, dX, dY must be non-null", who);
  // Empty sums: dX = 0 when M == 0, dY = 0 when N == 0.
  if (M == 0) return launch_fill_zero(dX, (size_t)(N * D), stream);
  if (N == 0) return launch_fill_zero(dY, (size_t)(M * D), stream);
  if (!dK || !K) return nl2k::fail(NL2K_ERR_NULL, "%s: dK and K must be non-null", who);

  const float neg2g = -2.f * gamma;
  const size_t floats = workspace_floats(N, M, D), need = floats * sizeof(float);
  const bool have = workspace != nullptr && workspace_bytes >= need;
  if (needs_workspace(N, M, D, X, Y, dX, dY)) {
    if (!have)
      return nl2k::fail(NL2K_ERR_WORKSPACE, "%s: workspace of %zu bytes required, got %zu", who,
                        need, workspace ? workspace_bytes : (size_t)0);
    if (!nl2k::aligned16(workspace))
      return nl2k::fail(NL2K_ERR_ALIGN, "%s: workspace must be 16-byte aligned", who);
  }
  if (have && reinterpret_cast<uintptr_t>(workspace) % 4 == 0) {
    float* ws = static_cast<float*>(workspace);
    const nl2k::pairwise::BwdPlan rp = nl2k::pairwise::plan_backward(N, M, D, true);
    if (needs_workspace(N, M, D, X, Y, dX, dY) &&
        nl2k::pairwise::takes_regions(rp, M, X, Y, dK, K)) {
      st = nl2k::pairwise::launch_bwd_regions<RbfBwdOp>(rp, X, Y, dK, K, ws, N, M, nullptr,
                                                        nullptr, stream, who);
      return st ? st : reduce<false>(rp, ws, X, Y, dK, K, dX, dY, N, M, D, neg2g, stream, who);
    }
    const nl2k::pairwise::SplitBwdPlan p =
        nl2k::pairwise::plan_split_backward(N, M, D, true, floats);
    if (p.ok) {
      st = nl2k::pairwise::launch_bwd_split<RbfBwdOp>(p, X, Y, dK, K, ws, N, M, D, nullptr,
                                                      nullptr, stream, who);
      return st ? st : reduce<true>(p, ws, X, Y, dK, K, dX, dY, N, M, D, neg2g, stream, who);
    }
  }

  // Generic kernels: the walks split into slices when the workspace holds
  // their partial sums (a shorter or no workspace runs them whole).
  using nl2k::pairwise::kGD;
  using nl2k::pairwise::kGT;
  const int64_t dp = nl2k::ceil_div(D, (int64_t)kGD);
  nl2k::pairwise::GenericSplit gx = nl2k::pairwise::generic_split(N, M, D),
                               gy = nl2k::pairwise::generic_split(M, N, D);
  const size_t gneed = generic_ws_floats(N, M, D) * sizeof(float);
  float* ws = static_cast<float*>(workspace);
  if (gneed == 0 || ws == nullptr || workspace_bytes < gneed ||
      reinterpret_cast<uintptr_t>(workspace) % 4 != 0) {
    gx = nl2k::pairwise::generic_whole(M);
    gy = nl2k::pairwise::generic_whole(N);
  }
  float* pxa = ws;
  float* pxs = gx.s > 1 ? pxa + gx.s * N * D : nullptr;
  float* pya = gx.s > 1 ? pxs + gx.s * N : ws;
  float* pys = gy.s > 1 ? pya + gy.s * M * D : nullptr;
  if (gx.s == 1) pxa = nullptr;
  if (gy.s == 1) pya = nullptr;
  hipLaunchKernelGGL((nl2k::pairwise::pair_bwd_generic_kernel<RbfGenBwd, false>),
                     dim3((unsigned)std::min<int64_t>(
                         nl2k::ceil_div(N, (int64_t)kGT) * dp * gx.s, 1 << 16)),
                     dim3(256), 0, stream, X, Y, dK, K, dX, pxa, pxs, N, M, D, gx.s, gx.chunk,
                     RbfGenBwd{neg2g});
  st = nl2k::check_launch(who);
  if (st) return st;
  hipLaunchKernelGGL((nl2k::pairwise::pair_bwd_generic_kernel<RbfGenBwd, true>),
                     dim3((unsigned)std::min<int64_t>(
                         nl2k::ceil_div(M, (int64_t)kGT) * dp * gy.s, 1 << 16)),
                     dim3(256), 0, stream, Y, X, dK, K, dY, pya, pys, N, M, D, gy.s, gy.chunk,
                     RbfGenBwd{neg2g});
  st = nl2k::check_launch(who);
  if (st || (gx.s == 1 && gy.s == 1)) return st;
  // dX and dY of the split sides in one launch (a side that did not split
  // has written its output already: zero blocks)
  const int bx = gx.s > 1 ? (int)std::min<int64_t>(nl2k::ceil_div(N * D, (int64_t)256), 2048) : 0;
  const int by = gy.s > 1 ? (int)std::min<int64_t>(nl2k::ceil_div(M * D, (int64_t)256), 2048) : 0;
  hipLaunchKernelGGL(rbf_bwd_generic_reduce_kernel, dim3((unsigned)(bx + by)), dim3(256), 0,
                     stream, pxa, pxs, X, dX, N, gx.s, pya, pys, Y, dY, M, gy.s, D, bx, neg2g);
  return nl2k::check_launch(who);
}

// ------------------------------------------------ scratch for the no-alloc entry
// rbf_backward_f32_noalloc keeps the backward's region partials here instead
// of in a caller workspace: 64 MiB per GPU, held from the first use of the
// library on that GPU until the process ends.  The name is a host-side
// stand-in; kernels get the device address that hipGetSymbolAddress returns,
// looked up once per device with that device current.
constexpr size_t kScratchBytes = size_t(64) << 20;

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::atomic<void*> scratch_ptr[kMaxDevices];

int scratch_address(void** out, const char* who) {
  int dev = -1;
  int st = nl2k::check_hip(hipGetDevice(&dev), who);
  if (st) return st;
  if (dev < 0 || dev >= kMaxDevices)
    return nl2k::fail(NL2K_ERR_HIP, "%s: device %d beyond the %d the library tracks", who, dev,
                      kMaxDevices);
  void* p = scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    st = nl2k::check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), who);
    if (st) return st;
    if (p == nullptr)
      return nl2k::fail(NL2K_ERR_HIP, "%s: hipGetSymbolAddress returned a null scratch", who);
    scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return NL2K_SUCCESS;
}

}  // namespace

extern "C" {

const char* rbf_last_error(void) { return nl2k::error_slot().text; }

int rbf_forward_f32(const float* X, const float* Y, float* K, int64_t N,
                    int64_t M, int64_t D, float gamma, hipStream_t stream) {
  int st = validate_sizes(N, M, D);
  if (st) return st;
  if (N == 0 || M == 0) return nl2k::succeed();
  if (!X || !Y || !K)
    return nl2k::fail(NL2K_ERR_NULL, "rbf_forward_f32: X, Y and K must be non-null");

  const RbfF64 op = {-gamma * kLog2e, f64_norm_max(gamma), gamma};
  if (takes_split_forward(D, X, Y)) {
    const nl2k::pairwise::SplitFwdPlan fp = nl2k::pairwise::plan_split_forward(N, M, D);
    if (fp.n_jt > 0)
      return nl2k::pairwise::launch_fwd_split(
          fp, X, Y, K, N, M, D, RbfFwdOp{(float)op.neg_kappa, split_norm_max(gamma), op}, nullptr,
          nullptr, stream, "rbf_forward_f32");
  }
  const int64_t n_jt = nl2k::ceil_div(M, (int64_t)kFwdTile);
  const int64_t n_tiles = nl2k::ceil_div(N, (int64_t)kFwdTile) * n_jt;
  if (std::max(std::max(N, M), D) <= INT32_MAX - 1024 && n_tiles <= nl2k::max_blocks(256)) {
    hipLaunchKernelGGL(rbf_fwd_kernel, dim3((unsigned)n_tiles), dim3(256), 0, stream, X, Y, K,
                       (int)N, (int)M, (int)D, op, (int)n_jt);
    return nl2k::check_launch("rbf_forward_f32");
  }
  const int64_t ntiles = nl2k::ceil_div(N, (int64_t)nl2k::pairwise::kGT) *
                         nl2k::ceil_div(M, (int64_t)nl2k::pairwise::kGT);
  hipLaunchKernelGGL(nl2k::pairwise::pair_fwd_generic_kernel<RbfGenFwd>,
                     dim3((unsigned)std::min<int64_t>(ntiles, 1 << 16)), dim3(256), 0, stream, X,
                     Y, K, N, M, D, RbfGenFwd{gamma});
  return nl2k::check_launch("rbf_forward_f32 (generic)");
}

size_t rbf_backward_workspace_bytes(int64_t N, int64_t M, int64_t D) {
  if (validate_sizes(N, M, D)) return 0;
  return workspace_floats(N, M, D) * sizeof(float);
}

int rbf_backward_f32(const float* X, const float* Y, const float* dK,
                     const float* K, float* dX, float* dY, int64_t N,
                     int64_t M, int64_t D, float gamma, void* workspace,
                     size_t workspace_bytes, hipStream_t stream) {
  return backward_impl(X, Y, dK, K, dX, dY, N, M, D, gamma, workspace, workspace_bytes, stream,
                       "rbf_backward_f32");
}

size_t rbf_backward_noalloc_max_bytes(void) { return kScratchBytes; }

int rbf_backward_f32_noalloc(const float* X, const float* Y, const float* dK, const float* K,
                             float* dX, float* dY, int64_t N, int64_t M, int64_t D, float gamma,
                             hipStream_t stream) {
  const char* who = "rbf_backward_f32_noalloc";
  int st = validate_sizes(N, M, D);
  if (st) return st;
  // Only calls that require a workspace use scratch; the others run whatever
  // their size, on the generic kernels.
  const size_t need = needs_workspace(N, M, D, X, Y, dX, dY)
                          ? workspace_floats(N, M, D) * sizeof(float)
                          : 0;
  if (need > kScratchBytes)
    return nl2k::fail(NL2K_ERR_WORKSPACE,
                      "%s: N=%lld M=%lld D=%lld needs %zu bytes of scratch; the library's static "
                      "scratch holds %zu (use rbf_backward_f32 with a workspace)",
                      who, (long long)N, (long long)M, (long long)D, need, kScratchBytes);
  void* ws = nullptr;
  if (need > 0 && N > 0 && M > 0) {
    st = scratch_address(&ws, who);
    if (st) return st;
  }
  return backward_impl(X, Y, dK, K, dX, dY, N, M, D, gamma, ws, kScratchBytes, stream, who);
}

}  // extern "C"
