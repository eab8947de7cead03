// Pairwise cosine similarity, forward and backward, fp32, for MI355X
// (gfx950).  C-ABI declared in include/cosine_sim.h.
//
// Reference semantics (cases/cosine_sim/reference.py:13-20): with
// s_a = 1 / (|a| + eps) and ah = s_a a (the same for B),
//   S[i,j] = ah_i . bh_j
// and, by autograd of that expression, for upstream dS:
//   dah_i = sum_j dS[i,j] bh_j
//   dA_i  = s_a dah_i - (ah_i . dah_i) / |a_i| ah_i     (0 for the second
//           term when |a_i| = 0, as torch's norm backward gives)
// and symmetrically for dB with dS^T.  (The reference's CUDA kernel,
// cosine_sim.cu:63-102, uses s_a in place of 1/|a| in the second term; the
// two agree to within eps / |a|.)
//
// Design:
//  * Forward: on bf16 splits of the fp32 rows (csrc/pairwise_split.h), at any
//    D and alignment.  A tile's rows are read once for their norms and again,
//    from L2, to be scaled by their inverse norms, split and multiplied, so
//    the epilogue is a plain store of the accumulators.  The same launch
//    writes inv_a / inv_b for the backward.
//  * Backward: one pass over dS (W = dS, no product) per 64 features, both
//    contractions dS . bh and dS^T . ah as region partials (the staged X / Y
//    rows scaled by inv_a / inv_b), on the bf16 splits or, for small shapes
//    at D = 64, on fp32 MFMA (csrc/pairwise_d64.h); cos_bwd_reduce_kernel sums
//    the partials and applies the projection.
//  * Past those kernels' ranges the tiled SIMT kernels of
//    csrc/pairwise_generic.h run (rows scaled by their inverse norms as they
//    are staged), the backward's walks in slices whose partial rows the
//    same reduce adds in order.
#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../../csrc/common.h"
#include "../../../csrc/pairwise_d64.h"
#include "../../../csrc/pairwise_generic.h"
#include "../../../csrc/pairwise_split.h"
#include "cosine_sim.h"

namespace {

__device__ __forceinline__ float inv_norm(float sumsq, float eps) {
  return 1.f / (sqrtf(sumsq) + eps);
}

// Forward policy: rows scaled by their inverse norms before the contraction,
// the inverse norms written out.
struct CosFwdOp {
  float eps;
  static constexpr bool kScale = true, kDirect = false;
  __device__ __forceinline__ float inv(float nsq) const { return inv_norm(nsq, eps); }
};

// Backward policy: W = dS, X / Y rows scaled by inv_a / inv_b, no sums.
struct CosBwdOp {
  static constexpr bool kProduct = false, kScale = true, kSums = false;
};

// One row: acc = sum of its partial rows, in slot order, then
//   out = s acc - (ah . acc) / |a| ah,  ah = s a,
// by L lanes of V features each (the sums over the row's lanes leave every
// lane the same bits).  The first kKeep groups of a lane stay in registers
// between the two passes; wider rows add their partials up again.
// Split partials carry kSplitScale and are added up directly where they are
// not finite.
constexpr int kKeep = 4;

template <int V, int L, bool SPLIT>
__device__ __forceinline__ void project_row(
    const float* __restrict__ P, const float* __restrict__ A, const float* __restrict__ inv,
    float* __restrict__ out, int64_t rows, int64_t r, int D, int slots, int lane,
    const float* __restrict__ dS, size_t own, size_t other,  // entry (r, o): r own + o other
    const float* __restrict__ B, const float* __restrict__ inv_b, int64_t others) {
  typedef float vec __attribute__((ext_vector_type(V), aligned(4)));
  const int per = D / V;
  const int64_t stride = rows * (int64_t)D;
  const float* p = P + r * D;
  const float* a = A + r * D;
  const float sc = inv[r];
  auto partial = [&](int e) {
    auto at = [&](int s) { return *reinterpret_cast<const vec*>(p + s * stride + (int64_t)e * V); };
    vec a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    int s = 0;
    for (; s + 4 <= slots; s += 4) {
      a0 += at(s);
      a1 += at(s + 1);
      a2 += at(s + 2);
      a3 += at(s + 3);
    }
    for (; s < slots; ++s) a0 += at(s);
    const vec acc = (a0 + a1) + (a2 + a3);
    return SPLIT ? acc * nl2k::pairwise::kPartialUnscale : acc;
  };
  float dot = 0.f, nn = 0.f;
  vec keep[kKeep], row[kKeep];
  auto add = [&](const vec& acc, const vec& av) {
    const vec ah = av * sc;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      dot = fmaf(ah[v], acc[v], dot);
      nn = fmaf(av[v], av[v], nn);
    }
  };
#pragma unroll
  for (int k = 0; k < kKeep; ++k) {
    const int e = lane + L * k;
    if (e < per) {
      keep[k] = partial(e);
      row[k] = *reinterpret_cast<const vec*>(a + (int64_t)e * V);
      add(keep[k], row[k]);
    }
  }
  for (int e = lane + L * kKeep; e < per; e += L)
    add(partial(e), *reinterpret_cast<const vec*>(a + (int64_t)e * V));
  auto over_row = [&] {
#pragma unroll
    for (int off = 1; off < L; off <<= 1) {
      dot += __shfl_xor(dot, off, 64);
      nn += __shfl_xor(nn, off, 64);
    }
  };
  over_row();
  auto store = [&](int e, const vec& acc, const vec& av, float coef) {
    *reinterpret_cast<vec*>(out + r * D + (int64_t)e * V) = sc * acc - coef * (av * sc);
  };
  // a partial that is not finite, or a dot that overflowed
  if (SPLIT && __builtin_expect(!(fabsf(dot) < INFINITY), 0)) {
    dot = nn = 0.f;
#pragma unroll 1
    for (int e = lane; e < per; e += L) {
      vec acc;
      float sum;
      nl2k::pairwise::direct_sums<CosBwdOp>(dS, nullptr, (size_t)r * own, other,
                                            B + (int64_t)e * V, inv_b, others, D, acc, sum);
      *reinterpret_cast<vec*>(out + r * D + (int64_t)e * V) = acc;  // read back below
      add(acc, *reinterpret_cast<const vec*>(a + (int64_t)e * V));
    }
    over_row();
    const float nrm = sqrtf(nn), coef = nrm > 0.f ? dot / nrm : 0.f;
#pragma unroll 1
    for (int e = lane; e < per; e += L)
      store(e, *reinterpret_cast<const vec*>(out + r * D + (int64_t)e * V),
            *reinterpret_cast<const vec*>(a + (int64_t)e * V), coef);
    return;
  }
  const float nrm = sqrtf(nn);
  const float coef = nrm > 0.f ? dot / nrm : 0.f;
#pragma unroll
  for (int k = 0; k < kKeep; ++k)
    if (lane + L * k < per) store(lane + L * k, keep[k], row[k], coef);
  for (int e = lane + L * kKeep; e < per; e += L)
    store(e, partial(e), *reinterpret_cast<const vec*>(a + (int64_t)e * V), coef);
}

// Both outputs in one launch: block b < bx handles dA, the rest dB.  A row's
// lanes stay together: every lane of a group has the same row.
template <int V, int L, bool SPLIT>
__global__ __launch_bounds__(256) void cos_bwd_reduce_kernel(
    const float* __restrict__ Px, const float* __restrict__ A,
    const float* __restrict__ inv_a, float* __restrict__ dA, int64_t N, int sx,
    const float* __restrict__ Py, const float* __restrict__ B,
    const float* __restrict__ inv_b, float* __restrict__ dB, int64_t M, int sy,
    const float* __restrict__ dS, int D, int bx) {
  constexpr int kRows = 256 / L;
  const int b = (int)blockIdx.x;
  const int lane = threadIdx.x % L, g = threadIdx.x / L;
  if (b < bx) {
    for (int64_t r = (int64_t)b * kRows + g; r < N; r += (int64_t)bx * kRows)
      project_row<V, L, SPLIT>(Px, A, inv_a, dA, N, r, D, sx, lane, dS, (size_t)M, 1, B, inv_b, M);
  } else {
    const int64_t nb = (int)gridDim.x - bx;
    for (int64_t r = (int64_t)(b - bx) * kRows + g; r < M; r += nb * kRows)
      project_row<V, L, SPLIT>(Py, B, inv_b, dB, M, r, D, sy, lane, dS, 1, (size_t)M, A, inv_a, N);
  }
}

// ------------------------------------------------------- generic (any D)
// inv[r] = 1 / (|V_r| + eps), one wave per row.
__global__ __launch_bounds__(256) void cos_norm_kernel(const float* __restrict__ V,
                                                       float* __restrict__ inv, int64_t rows,
                                                       int64_t D, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x / 64);
  for (int64_t r = (int64_t)blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6); r < rows;
       r += waves) {
    float ss = 0.f;
    for (int64_t d = lane; d < D; d += 64) ss = fmaf(V[r * D + d], V[r * D + d], ss);
    ss = nl2k::wave_sum(ss);
    if (lane == 0) inv[r] = inv_norm(ss, eps);
  }
}

// Policies of the tiled SIMT kernels (csrc/pairwise_generic.h).
// Forward: S = sum_d (a_d inv_a) (b_d inv_b), rows scaled as they are staged.
struct CosGenFwd {
  const float* __restrict__ inv_a;
  const float* __restrict__ inv_b;
  __device__ __forceinline__ float x_in(float v, int64_t i) const { return v * inv_a[i]; }
  __device__ __forceinline__ float y_in(float v, int64_t j) const { return v * inv_b[j]; }
  __device__ __forceinline__ float step(float s, float x, float y) const { return fmaf(x, y, s); }
  __device__ __forceinline__ float out(float s) const { return s; }
};
// Backward: dvh[r][d] = sum_o W[r, o] inv_o[o] O[o][d], W = dS (dS^T for the
// B side); the walked rows are scaled by their inverse norms as staged.
struct CosGenBwd {
  const float* __restrict__ inv_a;
  const float* __restrict__ inv_b;
  static constexpr bool kSums = false;
  __device__ __forceinline__ float w(const float* __restrict__ dS, const float*,
                                     int64_t idx) const {
    return dS[idx];
  }
  template <bool TRANS>
  __device__ __forceinline__ float b_in(float v, int64_t o) const {
    return v * (TRANS ? inv_a[o] : inv_b[o]);
  }
  __device__ __forceinline__ float finish(float, float, float acc) const { return acc; }
};

// Floats of the generic backward's partial rows: S slices a side when
// `sliced`, one otherwise.
inline size_t generic_ws_floats(int64_t N, int64_t M, int64_t D, bool sliced) {
  const int64_t sx = sliced ? nl2k::pairwise::generic_split(N, M, D).s : 1;
  const int64_t sy = sliced ? nl2k::pairwise::generic_split(M, N, D).s : 1;
  return (size_t)(sx * N * D + sy * M * D);
}

__global__ __launch_bounds__(256) void cos_fill_zero_kernel(float* __restrict__ p, size_t count) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < count;
       e += (size_t)gridDim.x * blockDim.x)
    p[e] = 0.f;
}

// ----------------------------------------------------------------- host side
int validate_sizes(int64_t N, int64_t M, int64_t D, const char* who) {
  if (N < 0 || M < 0 || D < 1)
    return nl2k::fail(NL2K_ERR_SHAPE,
                      "%s: sizes must satisfy N >= 0, M >= 0, D >= 1 (got N=%lld M=%lld D=%lld)",
                      who, (long long)N, (long long)M, (long long)D);
  const int64_t lim = INT32_MAX;
  if (N > lim || M > lim || D > lim || N > INT64_MAX / D || M > INT64_MAX / D ||
      (M > 0 && N > INT64_MAX / M))
    return nl2k::fail(NL2K_ERR_OVERFLOW, "%s: sizes too large (N=%lld M=%lld D=%lld)", who,
                      (long long)N, (long long)M, (long long)D);
  return NL2K_SUCCESS;
}

int grid_for(int64_t work, int64_t per_block, int cap) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(nl2k::ceil_div(work, per_block), cap));
}

int launch_norms(const float* V, float* inv, int64_t rows, int64_t D, float eps,
                 hipStream_t stream) {
  if (rows == 0) return NL2K_SUCCESS;
  hipLaunchKernelGGL(cos_norm_kernel, dim3(grid_for(rows, 4, 1 << 16)), dim3(256), 0, stream, V,
                     inv, rows, D, eps);
  return nl2k::check_launch("cosine_sim norms");
}

int fill_zero(float* p, size_t count, hipStream_t stream) {
  if (count == 0) return NL2K_SUCCESS;
  hipLaunchKernelGGL(cos_fill_zero_kernel, dim3(grid_for((int64_t)count, 256, 4096)), dim3(256),
                     0, stream, p, count);
  return nl2k::check_launch("cosine_sim fill");
}

// Sums the partial rows (sx of each row of A, sy of B) into dA and dB.
template <bool SPLIT>
int reduce(const float* px, const float* py, int64_t sx, int64_t sy, const float* A,
           const float* B, const float* inv_a, const float* inv_b, const float* dS, float* dA,
           float* dB, int64_t N, int64_t M, int64_t D, hipStream_t stream, const char* who) {
  const bool vec = D % 4 == 0;
  const bool wide = D > (vec ? 64 : 16);  // a wave per row, else 16 lanes
  auto* kernel =
      vec ? (wide ? &cos_bwd_reduce_kernel<4, 64, SPLIT> : &cos_bwd_reduce_kernel<4, 16, SPLIT>)
          : (wide ? &cos_bwd_reduce_kernel<1, 64, SPLIT> : &cos_bwd_reduce_kernel<1, 16, SPLIT>);
  const int bx = grid_for(N, wide ? 4 : 16, 2048), by = grid_for(M, wide ? 4 : 16, 2048);
  hipLaunchKernelGGL(kernel, dim3(bx + by), dim3(256), 0, stream, px, A, inv_a, dA, N, (int)sx,
                     py, B, inv_b, dB, M, (int)sy, dS, (int)D, bx);
  return nl2k::check_launch(who);
}

// What cosine_sim_backward_workspace_bytes reports, in floats: callers hold
// buffers of this size, and the split backward is cut so that its partials
// fit.  At D = 64 it is the fp32 regions' (pairwise_d64.h) or one partial row
// for each row, else what the generic kernels' slices or the split backward
// use.
size_t workspace_floats(int64_t N, int64_t M, int64_t D) {
  if (N == 0 || M == 0) return 0;
  const nl2k::pairwise::BwdPlan p = nl2k::pairwise::plan_backward(N, M, D, false);
  if (p.fast) return std::max(p.ws_floats, generic_ws_floats(N, M, D, false));
  return std::max(generic_ws_floats(N, M, D, true),
                  nl2k::pairwise::split_floats(N, M, D, false));
}

// What a call needs at least: all of that at D = 64, else one partial row for
// each row.
size_t least_floats(int64_t N, int64_t M, int64_t D) {
  return D == nl2k::pairwise::kD ? workspace_floats(N, M, D)
                                 : generic_ws_floats(N, M, D, false);
}

}  // namespace

extern "C" {

const char* cosine_sim_last_error(void) { return nl2k::error_slot().text; }

int cosine_sim_forward_f32(const float* A, const float* B, float* S, float* inv_a,
                           float* inv_b, int64_t N, int64_t M, int64_t D, float eps,
                           hipStream_t stream) {
  const char* who = "cosine_sim_forward_f32";
  int st = validate_sizes(N, M, D, who);
  if (st) return st;
  if ((N > 0 && (!A || !inv_a)) || (M > 0 && (!B || !inv_b)) || (N > 0 && M > 0 && !S))
    return nl2k::fail(NL2K_ERR_NULL, "%s: null pointer argument", who);
  if (!(eps >= 0.f))
    return nl2k::fail(NL2K_ERR_VALUE, "%s: eps must be >= 0 (got %g)", who, (double)eps);
  if (N == 0 || M == 0) {  // no S; the inverse norms are still defined
    st = launch_norms(A, inv_a, N, D, eps, stream);
    if (st) return st;
    return launch_norms(B, inv_b, M, D, eps, stream);
  }
  const nl2k::pairwise::SplitFwdPlan fp = nl2k::pairwise::plan_split_forward(N, M, D);
  if (fp.n_jt > 0)
    return nl2k::pairwise::launch_fwd_split(fp, A, B, S, N, M, D, CosFwdOp{eps}, inv_a, inv_b,
                                            stream, who);
  st = launch_norms(A, inv_a, N, D, eps, stream);
  if (st) return st;
  st = launch_norms(B, inv_b, M, D, eps, stream);
  if (st) return st;
  const int64_t ntiles = nl2k::ceil_div(N, (int64_t)nl2k::pairwise::kGT) *
                         nl2k::ceil_div(M, (int64_t)nl2k::pairwise::kGT);
  hipLaunchKernelGGL(nl2k::pairwise::pair_fwd_generic_kernel<CosGenFwd>,
                     dim3((unsigned)std::min<int64_t>(ntiles, 1 << 16)), dim3(256), 0, stream, A,
                     B, S, N, M, D, CosGenFwd{inv_a, inv_b});
  return nl2k::check_launch("cosine_sim_forward_f32 (generic)");
}

size_t cosine_sim_backward_workspace_bytes(int64_t N, int64_t M, int64_t D) {
  if (validate_sizes(N, M, D, "cosine_sim_backward_workspace_bytes")) return 0;
  return workspace_floats(N, M, D) * sizeof(float);
}

int cosine_sim_backward_f32(const float* A, const float* B, const float* inv_a,
                            const float* inv_b, const float* dS, float* dA, float* dB,
                            int64_t N, int64_t M, int64_t D, void* workspace,
                            size_t workspace_bytes, hipStream_t stream) {
  const char* who = "cosine_sim_backward_f32";
  int st = validate_sizes(N, M, D, who);
  if (st) return st;
  if (N == 0 && M == 0) return nl2k::succeed();
  if ((N > 0 && (!A || !inv_a || !dA)) || (M > 0 && (!B || !inv_b || !dB)))
    return nl2k::fail(NL2K_ERR_NULL, "%s: null pointer argument", who);
  // Empty sums: dA = 0 when M == 0, dB = 0 when N == 0.
  if (M == 0) return fill_zero(dA, (size_t)(N * D), stream);
  if (N == 0) return fill_zero(dB, (size_t)(M * D), stream);
  if (!dS) return nl2k::fail(NL2K_ERR_NULL, "%s: dS must be non-null", who);
  const size_t floats = workspace_floats(N, M, D), need = least_floats(N, M, D) * sizeof(float);
  if (workspace == nullptr || workspace_bytes < need)
    return nl2k::fail(NL2K_ERR_WORKSPACE, "%s: workspace of %zu bytes required, got %zu", who,
                      need, workspace ? workspace_bytes : (size_t)0);
  if (!nl2k::aligned16(workspace))
    return nl2k::fail(NL2K_ERR_ALIGN, "%s: workspace must be 16-byte aligned", who);
  float* ws = static_cast<float*>(workspace);

  const nl2k::pairwise::BwdPlan rp = nl2k::pairwise::plan_backward(N, M, D, false);
  if (nl2k::pairwise::takes_regions(rp, M, A, B, dS, dS)) {
    st = nl2k::pairwise::launch_bwd_regions<CosBwdOp>(rp, A, B, dS, nullptr, ws, N, M, inv_a,
                                                      inv_b, stream, who);
    return st ? st : reduce<false>(ws + rp.px, ws + rp.py, rp.nRJ, rp.nRI, A, B, inv_a, inv_b, dS,
                                   dA, dB, N, M, D, stream, who);
  }
  const nl2k::pairwise::SplitBwdPlan p =
      nl2k::pairwise::plan_split_backward(N, M, D, false,
                                          std::min(floats, workspace_bytes / sizeof(float)));
  if (p.ok) {
    st = nl2k::pairwise::launch_bwd_split<CosBwdOp>(p, A, B, dS, nullptr, ws, N, M, D, inv_a,
                                                    inv_b, stream, who);
    return st ? st : reduce<true>(ws + p.px, ws + p.py, p.nRJ, p.nRI, A, B, inv_a, inv_b, dS, dA,
                                  dB, N, M, D, stream, who);
  }

  // generic kernels: the walks in slices when the workspace holds their
  // partial rows, else whole (the entry check above guarantees that much)
  using nl2k::pairwise::kGT;
  nl2k::pairwise::GenericSplit gx = nl2k::pairwise::generic_split(N, M, D),
                               gy = nl2k::pairwise::generic_split(M, N, D);
  if (workspace_bytes < generic_ws_floats(N, M, D, true) * sizeof(float)) {
    gx = nl2k::pairwise::generic_whole(M);
    gy = nl2k::pairwise::generic_whole(N);
  }
  float* dah = ws;                               // [Sx][N][D]
  float* dbh = ws + (size_t)(gx.s * N * D);      // [Sy][M][D]
  const int64_t dp = nl2k::ceil_div(D, (int64_t)nl2k::pairwise::kGD);
  const CosGenBwd op{inv_a, inv_b};
  hipLaunchKernelGGL((nl2k::pairwise::pair_bwd_generic_kernel<CosGenBwd, false>),
                     dim3((unsigned)std::min<int64_t>(nl2k::ceil_div(N, (int64_t)kGT) * dp * gx.s,
                                                      1 << 16)),
                     dim3(256), 0, stream, A, B, dS, nullptr, nullptr, dah, nullptr, N, M, D, gx.s,
                     gx.chunk, op);
  st = nl2k::check_launch("cosine_sim_backward_f32 (generic dA)");
  if (st) return st;
  hipLaunchKernelGGL((nl2k::pairwise::pair_bwd_generic_kernel<CosGenBwd, true>),
                     dim3((unsigned)std::min<int64_t>(nl2k::ceil_div(M, (int64_t)kGT) * dp * gy.s,
                                                      1 << 16)),
                     dim3(256), 0, stream, B, A, dS, nullptr, nullptr, dbh, nullptr, N, M, D, gy.s,
                     gy.chunk, op);
  st = nl2k::check_launch("cosine_sim_backward_f32 (generic dB)");
  if (st) return st;
  return reduce<false>(dah, dbh, gx.s, gy.s, A, B, inv_a, inv_b, dS, dA, dB, N, M, D, stream,
                       "cosine_sim_backward_f32 (generic reduce)");
}

}  // extern "C"
