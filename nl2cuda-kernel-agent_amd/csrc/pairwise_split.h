// Pairwise row-by-row contractions in fp32 at any feature width on the bf16
// matrix instructions (gfx950): the kernels behind the RBF and
// cosine-similarity cases.
//
// Every fp32 operand is split exactly into three bf16 terms, x = h + m + l
// (each term the rounded remainder of the ones before it: 3 x 8 significant
// bits hold fp32's 24), and a product is the sum of the six term products
// that matter, hh + hm + mh + hl + lh + mm, each exact in the fp32
// accumulator's input; what is left out (ml, lm, ll) is below 2^-25 of
// |x y|.  v_mfma_f32_16x16x32_bf16 does 16 times the work of
// v_mfma_f32_16x16x4_f32 in half its cycles, so six of them for one take 2.7
// times less matrix time than fp32 instructions, and they add a contraction
// of 32 at a time, so fewer roundings reach the accumulator (errors against
// 64 bits at each kernel).
//
//  * pair_fwd_split_kernel<Op, TB>: out[i, j] = Op::out(x_i . y_j, row term,
//    column term) on TB x TB tiles.
//  * pair_bwd_split_kernel<Op>: for W = dK o K (Op::kProduct, else W = dK)
//    raw partials of W . Y, W^T . X and (Op::kSums) the row and column sums
//    of W, from one pass over the [N, M] inputs per 64 features.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "common.h"
#include "pairwise_generic.h"

namespace nl2k {
namespace pairwise {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// 16 bytes at any 4-byte boundary: rows of D or M floats start anywhere when
// D or M is no multiple of 4 (dword alignment is all the hardware needs).
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ f32x4 load4_u(const float* p) {
  return *reinterpret_cast<const f32x4_u*>(p);
}
__device__ __forceinline__ void store4_u(float* p, f32x4 v) {
  *reinterpret_cast<f32x4_u*>(p) = v;
}

// The bf16 terms of a and b, packed (a in the low half).
struct Terms2 {
  uint32_t t[3];
};
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ Terms2 split2(float a, float b) {
  Terms2 s;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    s.t[p] = bf16_pair(a, b);
    a -= __builtin_bit_cast(float, s.t[p] << 16);
    b -= __builtin_bit_cast(float, s.t[p] & 0xffff0000u);
  }
  return s;
}

// Eight consecutive contraction values of one operand row, per term.
struct Frag3 {
  u32x4 t[3];
};
__device__ __forceinline__ Frag3 split8(const float (&v)[8]) {
  Frag3 f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const Terms2 s = split2(v[2 * u], v[2 * u + 1]);
#pragma unroll
    for (int p = 0; p < 3; ++p) f.t[p][u] = s.t[p];
  }
  return f;
}

// acc[m][n] += sum_k A[m][k] B[k][n], k of 32: lane l supplies row (column)
// l % 16 at k = 8 (l / 16) .. + 7; acc element [4 (l / 16) + r][l % 16] is
// register r of lane l.
__device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

// The six term products, the smallest first: (term of A, term of B).
constexpr int kProducts = 6;
__device__ constexpr int kTermA[kProducts] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kTermB[kProducts] = {0, 2, 1, 0, 1, 0};

// ------------------------------------------------------------------ forward
// Op interface:
//   static constexpr bool kScale    rows are scaled by Op::inv(|row|^2) before
//                                   the contraction, and the scales written
//                                   to rowv [N] / colv [M]
//   static constexpr bool kDirect   a tile one of whose rows has a squared
//                                   norm past Op::norm_max is left to
//                                   Op::direct<TB>, 64 x 64 outputs at a time
//   float inv(float nsq)
//   float row(float nsq) / col(float nsq)     epilogue terms
//   float out(float dot, float rt, float ct)  the output entry
//
// A workgroup of four waves computes a TB x TB tile, 32 features at a time:
// each thread loads 8 features of a row of X and of Y (the next 32 features
// are in flight while these are multiplied), splits them and stores the terms
// in LDS in operand order (16 rows x 32 features per block, one 16-byte
// operand per lane, quarter rows 288 bytes apart so that the stores, four
// lanes of a row side by side, and the loads, 16 rows side by side, use all
// banks).  The row norms are summed from the values as they are staged.
// Operand A is Y, so a lane's four accumulators are four consecutive columns
// of a row and leave in one 16-byte store.
// Bound by vector and matrix issue together (splits and exponentials beside
// the products) and, at 64 features, by the waits of two tiles per CU; the
// stores are 5 of 27 us at 4096^2 x 64.  RBF against the fp32 MFMA kernel
// before: 31.3 -> 26.9 us at 4096^2 x 64, 103 -> 82 at 8192^2 x 64, error against
// 64 bits (2-norm) 5.7e-8 -> 5.5e-8.  (At other widths the RBF forward sums
// squared differences, or forms them in 64 bits: cases/rbf.)
constexpr int kQuarter = 288;
constexpr int kBlock = 4 * kQuarter;

template <int TB>
struct FwdLds {
  static constexpr int kNB = TB / 16;
  union {
    unsigned char planes[2][3][kNB][kBlock];  // [X or Y][term][16 rows]
    SimtTile simt;
  };
  float norm[2][TB];
};

template <class Op, int TB>
__global__ __launch_bounds__(256, TB == 128 ? 2 : 4) void pair_fwd_split_kernel(
    const float* __restrict__ X, const float* __restrict__ Y, float* __restrict__ out, int N,
    int M, int D, Op op, int n_jt, float* __restrict__ rowv, float* __restrict__ colv) {
  __shared__ __attribute__((aligned(16))) FwdLds<TB> lds;
  constexpr int kItems = TB / 64;  // rows per thread and side
  constexpr int kWB = TB / 32;     // 16-row blocks per wave and side
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, h = lane >> 4;
  const int srow = tid >> 2, sh = tid & 3;  // staging: row and quarter
  const int wi = (wave >> 1) * kWB, wj = (wave & 1) * kWB;

  const int i0 = (int)(blockIdx.x / n_jt) * TB, j0 = (int)(blockIdx.x % n_jt) * TB;
  const float* src[2][kItems];
#pragma unroll
  for (int s = 0; s < kItems; ++s) {
    src[0][s] = X + (size_t)min(i0 + srow + 64 * s, N - 1) * D;
    src[1][s] = Y + (size_t)min(j0 + srow + 64 * s, M - 1) * D;
  }
  float v[2][kItems][8];
  auto load = [&](int k0) {
    const int k = k0 + 8 * sh;
    if (k0 + 32 <= D) {
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int s = 0; s < kItems; ++s) {
          const f32x4 a = load4_u(src[e][s] + k), b = load4_u(src[e][s] + k + 4);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            v[e][s][u] = a[u];
            v[e][s][4 + u] = b[u];
          }
        }
    } else {  // the last features: zeros past D
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int s = 0; s < kItems; ++s)
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const float x = src[e][s][min(k + u, D - 1)];
            v[e][s][u] = k + u < D ? x : 0.f;
          }
    }
  };
  float nsq[2][kItems];
  auto add_norms = [&] {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int s = 0; s < kItems; ++s) {
        float p = 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) p = fmaf(v[e][s][u], v[e][s][u], p);
        nsq[e][s] += p;
      }
  };
  auto row_norms = [&] {  // over the row's four lanes
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int s = 0; s < kItems; ++s) {
        nsq[e][s] += __shfl_xor(nsq[e][s], 1, 64);
        nsq[e][s] += __shfl_xor(nsq[e][s], 2, 64);
      }
  };
#pragma unroll
  for (int e = 0; e < 2; ++e)
#pragma unroll
    for (int s = 0; s < kItems; ++s) nsq[e][s] = 0.f;

  float scale[2][kItems];
  if constexpr (Op::kScale) {
    // The norms first: the rows are read twice, the second time from L2.
    for (int k0 = 0; k0 < D; k0 += 32) {
      load(k0);
      add_norms();
    }
    row_norms();
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int s = 0; s < kItems; ++s) {
        scale[e][s] = op.inv(nsq[e][s]);
        const int r = srow + 64 * s;
        if (sh == 0 && e == 0 && j0 == 0 && i0 + r < N) rowv[i0 + r] = scale[e][s];
        if (sh == 0 && e == 1 && i0 == 0 && j0 + r < M) colv[j0 + r] = scale[e][s];
      }
  }

  f32x4 acc[kWB][kWB];
#pragma unroll
  for (int a = 0; a < kWB; ++a)
#pragma unroll
    for (int b = 0; b < kWB; ++b) acc[a][b] = zero4();

  // Whether one of the tile's rows, as far as it has been summed, has too
  // large a norm: the tile is then left to Op::direct.
  auto too_large = [&] {
    bool big = false;
    if constexpr (Op::kDirect) {
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int s = 0; s < kItems; ++s) big |= !(nsq[e][s] <= op.norm_max);
    }
    return big;
  };
  auto direct_tile = [&] {
    if constexpr (Op::kDirect) {
      for (int a = 0; a < TB; a += kGT)
        for (int b = 0; b < TB; b += kGT)
          if (i0 + a < N && j0 + b < M)
            op.template direct<TB>(lds.simt, X, Y, out, N, M, D, i0 + a, j0 + b);
    }
  };
  bool direct = false;  // workgroup-uniform

  load(0);
  for (int k0 = 0; k0 < D; k0 += 32) {
    if constexpr (!Op::kScale) add_norms();
    if constexpr (Op::kDirect) {
      // after the first features: rows far past the bound show here already
      if (k0 == 0) {
        direct = __syncthreads_or(too_large());
        if (direct) break;
      } else {
        __syncthreads();
      }
    } else {
      __syncthreads();  // the last chunk has been read
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int s = 0; s < kItems; ++s) {
        if constexpr (Op::kScale) {
#pragma unroll
          for (int u = 0; u < 8; ++u) v[e][s][u] *= scale[e][s];
        }
        const Frag3 f = split8(v[e][s]);
        const int r = srow + 64 * s;
#pragma unroll
        for (int p = 0; p < 3; ++p)
          *reinterpret_cast<u32x4*>(
              &lds.planes[e][p][r >> 4][sh * kQuarter + (r & 15) * 16]) = f.t[p];
      }
    __syncthreads();
    if (k0 + 32 < D) load(k0 + 32);
    const int off = h * kQuarter + n * 16;
    u32x4 xf[kWB][3];
#pragma unroll
    for (int a = 0; a < kWB; ++a)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        xf[a][p] = *reinterpret_cast<const u32x4*>(&lds.planes[0][p][wi + a][off]);
#pragma unroll
    for (int b = 0; b < kWB; ++b) {
      u32x4 yf[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        yf[p] = *reinterpret_cast<const u32x4*>(&lds.planes[1][p][wj + b][off]);
#pragma unroll
      for (int t = 0; t < kProducts; ++t)
#pragma unroll
        for (int a = 0; a < kWB; ++a)
          acc[a][b] = mfma32(yf[kTermA[t]], xf[a][kTermB[t]], acc[a][b]);
    }
  }

  float rt[kWB];
  f32x4 ct[kWB];
  if constexpr (!Op::kScale) {
    row_norms();
    if constexpr (Op::kDirect) {
      if (__syncthreads_or(direct || too_large())) {
        direct_tile();
        return;
      }
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int s = 0; s < kItems; ++s)
        if (sh == 0) lds.norm[e][srow + 64 * s] = e == 0 ? op.row(nsq[e][s]) : op.col(nsq[e][s]);
    __syncthreads();
#pragma unroll
    for (int a = 0; a < kWB; ++a) rt[a] = lds.norm[0][(wi + a) * 16 + n];
#pragma unroll
    for (int b = 0; b < kWB; ++b)
      ct[b] = *reinterpret_cast<const f32x4*>(&lds.norm[1][(wj + b) * 16 + 4 * h]);
  }
#pragma unroll
  for (int a = 0; a < kWB; ++a) {
    const int i = i0 + (wi + a) * 16 + n;
    if (i >= N) continue;
    float* row = out + (size_t)i * M;
#pragma unroll
    for (int b = 0; b < kWB; ++b) {
      const int j = j0 + (wj + b) * 16 + 4 * h;
      f32x4 o = acc[a][b];
      if constexpr (!Op::kScale) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = op.out(o[r], rt[a], ct[b][r]);
      }
      if (j + 3 < M) {
        store4_u(row + j, o);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (j + r < M) row[j + r] = o[r];
      }
    }
  }
}

// n_jt = 0: the shape is out of range.
struct SplitFwdPlan {
  int tb = 0, n_jt = 0;
  int64_t n_tiles = 0;
};

inline SplitFwdPlan plan_split_forward(int64_t N, int64_t M, int64_t D) {
  SplitFwdPlan p;
  constexpr int64_t lim = INT32_MAX - 1024;
  if (N > lim || M > lim || D > lim) return p;
  // Tiles of 128 x 128 (two workgroups per CU, half the LDS reads per product)
  // or of 64 x 64 (four, finer rounds): the lower of the two times, in us, that
  // rounds of 512 and 1024 workgroups measured, c chunks of 32 features each:
  // 6 + 3 c (0.65 of it when half the round or less is filled) and 2.3 + 1.85
  // c.  With 64 and with 128: 16.1 and 20.9 us at 3000^2 x 64, 9.3 and 10.9
  // at 2048^2 x 64, 28.1 and 26.7 at 4096^2 x 64, 97 and 84 at 8192^2 x 64,
  // 43.6 and 39.4 at 4096^2 x 128, 20.6 and 23.5 at 2048^2 x 256.
  const double c = (double)ceil_div(D, (int64_t)32);
  const double t128 = (double)(ceil_div(N, (int64_t)128) * ceil_div(M, (int64_t)128));
  const double t64 = (double)(ceil_div(N, (int64_t)64) * ceil_div(M, (int64_t)64));
  const double full = std::floor(t128 / 512), rest = t128 - 512 * full;
  const double cost128 = (6.0 + 3.0 * c) * (full + (rest == 0 ? 0.0 : rest <= 256 ? 0.65 : 1.0));
  const double cost64 = (2.3 + 1.85 * c) * std::max(t64 / 1024, 1.0);
  p.tb = cost128 <= 1.05 * cost64 ? 128 : 64;
  const int64_t n_jt = ceil_div(M, (int64_t)p.tb);
  p.n_tiles = ceil_div(N, (int64_t)p.tb) * n_jt;
  if (p.n_tiles <= max_blocks(256)) p.n_jt = (int)n_jt;
  return p;
}

template <class Op>
int launch_fwd_split(const SplitFwdPlan& p, const float* X, const float* Y, float* out, int64_t N,
                     int64_t M, int64_t D, Op op, float* rowv, float* colv, hipStream_t stream,
                     const char* who) {
  auto* kernel = p.tb == 128 ? &pair_fwd_split_kernel<Op, 128> : &pair_fwd_split_kernel<Op, 64>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)p.n_tiles), dim3(256), 0, stream, X, Y, out, (int)N,
                     (int)M, (int)D, op, p.n_jt, rowv, colv);
  return check_launch(who);
}

// ----------------------------------------------------------------- backward
// One workgroup of eight waves (two a SIMD: one's loads, splits and LDS
// traffic run beside the other's matrix instructions) per region of RI rows x
// (SJ strips of 256 columns) and per 64 features.  Along a strip the
// workgroup walks its rows 32 at a time:
//  * Wave w holds W[32 rows][its 32 columns]: lane (c, h) loads columns 2c,
//    2c + 1 of rows 8h .. 8h + 7 (128 bytes of a row side by side), the next
//    step's while this one is multiplied.  Packed along the rows, the split
//    values are at once the operand of W^T . X (a contraction over rows),
//    whose sums over the strip's walk stay in registers: [32 columns][64
//    features] per wave.
//  * Packed along the columns they go through LDS (operand order, 16-byte
//    slots permuted so that stores and loads use all banks), from where
//    the waves read them for W . Y: wave w takes 16 features (w % 4) and half
//    of the strip's columns (w / 4), whose Y operands stay in registers for
//    the strip.  The halves are added through LDS, and the [32][64] sums over
//    the strip's columns are complete, and stored, one step later.
//  * X, 32 rows x 64 features, is loaded a step ahead, split and staged in
//    LDS along the rows.
// The LDS buffers alternate, so a step has one barrier.  Row sums come from
// products with ones (each wave an eighth of the columns, added through
// LDS), column sums from the lanes' own values.
// Bound by memory and by issue at about equal times: a step takes 4.0 us on a
// full chip (64 KB per CU, 4.2 TB/s), 3.5 with W read from L2, 2.6 alone.
// Measured with the reduce, against the fp32 kernels before (MFMA at D = 64,
// SIMT elsewhere): 58 -> 54 us at 4096^2 x 64, 204 -> 153 at 8192^2 x 64, 97
// -> 56 at 4095 x 4097 x 64, 180 -> 40 at 3000 x 2500 x 100, 346 -> 133 at
// 4096^2 x 128.  Errors of dX, dY against 64 bits 2.3e-7 -> 1.4e-7 at 4096^2
// x 64, 3.3e-7 -> 1.4e-7 at 3000 x 2500 x 100.  One wave per SIMD (four waves
// of 64 columns, 426 registers) took 54 us for the tiles alone at 4096^2
// against 47.
//
// W, X and Y are multiplied by 2^24 first, so that the third term of a split
// (2^-24 of its operand) of any normal fp32 number is a normal bf16 number:
// partial contractions come out times 2^48, partial sums of W times 2^24, and
// the reduce takes that back.  Operands past 2^104 (infinities among them)
// leave the splits' range and give partials that are not finite; the reduce
// then adds those outputs up from W and the rows themselves (direct_sums).
// With the multiplications and the test: RBF 45.6 us as without at 4096^2 x
// 64, 39.4 -> 39.7 at 3000 x 2500 x 100, cosine 40.5 -> 41.8 at 2048 x 4096 x
// 128.  Where every output has to be added up (a NaN in each row and column):
// 1.5 ms at 4096^2 x 64.
constexpr float kSplitScale = 0x1p24f;
constexpr float kSumUnscale = 0x1p-24f;      // of Rx, Ry
constexpr float kPartialUnscale = 0x1p-48f;  // of Px, Py
constexpr int kBwdThreads = 512;
constexpr int kStripCols = 256;
constexpr int kStepRows = 32;
constexpr int kFeat = 64;  // features per pass
// Byte offsets of 32 rows of W (M floats) and of X and the partials (D floats)
// stay below 2^31; rows are indexed with int up to a step past the last one, and
// columns up to a strip; a launch holds fewer than 2^32 threads.
constexpr int64_t kMaxSplitWidth = int64_t(1) << 24;  // M and D
constexpr int64_t kMaxSplitRows = INT32_MAX - (int64_t(1) << 20);

inline bool split_in_range(int64_t N, int64_t M, int64_t D) {
  return N > 0 && M > 0 && D > 0 && N <= kMaxSplitRows && M <= kMaxSplitWidth &&
         D <= kMaxSplitWidth;
}

struct BwdLds {
  unsigned char w[2][3][2][8][1024];  // [buffer][term][16 rows][32 columns]
  unsigned char x[2][3][4][1024];     // [buffer][term][16 features]
  f32x4 half[2][4][2][64];            // [buffer][16 features][16 rows][lane]
  float rs[2][8][kStepRows];          // [buffer][wave][row]
};

// A lane offset past the bound of every buffer resource used here: loads
// return zeros and stores are dropped.
constexpr uint32_t kOutside = 0xc0000000u;

// Bytes of a buffer resource over `rows` rows of `width` floats.
__device__ __forceinline__ uint32_t rsrc_bytes(int rows, int width) {
  const uint64_t b = (uint64_t)(uint32_t)rows * (uint32_t)width * 4u;
  return (uint32_t)(b < kOutside ? b : kOutside);
}

// kNarrow: M = 1, where an 8-byte load could pass the end of W.
template <class Op, bool kNarrow>
__global__ __launch_bounds__(kBwdThreads) void pair_bwd_split_kernel(
    const float* __restrict__ X, const float* __restrict__ Y, const float* __restrict__ dK,
    const float* __restrict__ K, float* __restrict__ Px, float* __restrict__ Rx,
    float* __restrict__ Py, float* __restrict__ Ry, int N, int M, int D, int RI, int SJ, int nRJ,
    int n_regions, int n_dc, const float* __restrict__ sx, const float* __restrict__ sy) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  BwdLds& lds = *reinterpret_cast<BwdLds*>(smem);
  // Workgroups go to the 8 XCDs in turn: the passes over one region's
  // features follow each other on one XCD and find the region in its L2.
  const int xcd = (int)blockIdx.x & 7, idx = (int)blockIdx.x >> 3;
  const int dc = idx % n_dc;
  const int region = idx / n_dc * 8 + xcd;
  if (region >= n_regions) return;
  const int ri = region / nRJ, rj = region % nRJ;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fb = wave & 3, kh = wave >> 2;  // W . Y: features, half of the columns
  const int c = lane & 15, h = lane >> 4;   // also (n, h) of the operands
  const int d0 = dc * kFeat;
  const int i_begin = ri * RI, i_end = i_begin + min(RI, N - i_begin);
  const uint32_t m4 = (uint32_t)M * 4u;

  // W stores: columns 32 wave + 2c, + 1 are a quarter of a 16-byte slot of
  // column group `wave`, quarter row c / 4; row r's slot is (r % 16) ^ f, f =
  // c / 4 + 4 (group % 2 ^ r % 16 / 8).
  const int wf = (c >> 2) + 4 * ((wave ^ h) & 1);
  const int w_base = (h >> 1) * 8 * 1024 + wave * 1024 + (c >> 2) * 256 + (h & 1) * 128 +
                     wf * 16 + (c & 3) * 4;
  // W loads: row n of the block, quarter h, of the groups of this half, the
  // wave's own group first (its row sums are taken from it).
  const int r_own = (h * 256 + ((c ^ (h + 4 * (c >> 3))) << 4)) ^ ((wave & 1) * 64);
  const int r_next = r_own ^ 64;
  // X staging: feature d0 + lane, rows 4 wave .. + 3.
  const uint32_t x_off = d0 + lane < D ? (uint32_t)(d0 + lane) * 4u : kOutside;
  const int x_base = (lane >> 4) * 1024 + (wave >> 1) * 256 + (lane & 15) * 16 + (wave & 1) * 8;
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  // Output rows of a step: row c of each 16, features d .. d + 3.
  const int d_out = d0 + 16 * fb + 4 * h;

  for (int s = 0; s < SJ; ++s) {
    const int j0 = (rj * SJ + s) * kStripCols;
    if (j0 >= M) break;
    const int col = j0 + 32 * wave + 2 * c;
    // An odd M's last column is read as the second of a pair.
    const bool last_col = !kNarrow && col == M - 1;
    const uint32_t w_off =
        col < M ? (uint32_t)(8 * h) * m4 + (uint32_t)(col - (last_col ? 1 : 0)) * 4u : kOutside;

    // Loads of rows 2u, 2u + 1 of a lane's eight (and of X) of the step at
    // row i; past the walk (`valid` false) they return zeros and fetch
    // nothing.
    f32x2 ld[8], lk[8];
    float lx[4], lsx[4];
    auto issue_w = [&](int i, bool valid, int u) {
      const uint32_t bytes = valid ? rsrc_bytes(i_end - i, M) : 0u;
      uint32_t off = w_off;
      asm volatile("" : "+v"(off));  // added up each time: it costs no registers
      auto load_row = [&](const float* src, f32x2& dst, int r) {
        const buffer_rsrc rs = make_rsrc(src + (size_t)i * M, bytes);
        if constexpr (kNarrow)
          dst = f32x2{buffer_load1(rs, off + (uint32_t)r * m4, 0), 0.f};
        else
          dst = buffer_load2(rs, off + (uint32_t)r * m4, 0);
      };
#pragma unroll
      for (int r = 2 * u; r < 2 * u + 2; ++r) {
        load_row(dK, ld[r], r);
        if constexpr (Op::kProduct) load_row(K, lk[r], r);
      }
    };
    auto issue_x = [&](int i, bool valid) {
      const buffer_rsrc rx = make_rsrc(X + (size_t)i * D, valid ? kOutside : 0u);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = min(4 * wave + r, N - 1 - i);  // wave-uniform
        lx[r] = buffer_load1(rx, x_off, row * D * 4);
        if constexpr (Op::kScale) lsx[r] = sx[i + row];
      }
    };

    f32x2 csum = {0.f, 0.f};
    // The split of the loaded rows 2u, 2u + 1: packed along the rows for
    // W^T . X, packed along the columns to LDS for W . Y.
    Frag3 wt[2];
    auto stage_w = [&](int buf, int u) {
      f32x2 w[2];
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        f32x2 v = ld[2 * u + o];
        v = f32x2{v[0] * kSplitScale, v[1] * kSplitScale};
        if constexpr (Op::kProduct) v = f32x2{v[0] * lk[2 * u + o][0], v[1] * lk[2 * u + o][1]};
        w[o] = f32x2{last_col ? v[1] : v[0], last_col ? 0.f : v[1]};
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const Terms2 t = split2(w[0][q], w[1][q]);
#pragma unroll
        for (int p = 0; p < 3; ++p) wt[q].t[p][u] = t.t[p];
        if constexpr (Op::kSums) csum[q] += w[0][q] + w[1][q];
      }
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        int at = w_base + buf * (int)sizeof(lds.w[0]);
        asm volatile("" : "+v"(at));
        at ^= (2 * u + o) << 4;
#pragma unroll
        for (int p = 0; p < 3; ++p)
          *reinterpret_cast<uint32_t*>(smem + at + p * 2 * 8 * 1024) =
              __builtin_amdgcn_perm(wt[1].t[p][u], wt[0].t[p][u], o ? 0x07060302u : 0x05040100u);
      }
    };
    auto stage_x = [&](int buf) {
      float xv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        xv[r] = lx[r] * (Op::kScale ? lsx[r] * kSplitScale : kSplitScale);
      }
      const Terms2 a = split2(xv[0], xv[1]), b = split2(xv[2], xv[3]);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<u32x2*>(&lds.x[buf][p][0][0] + x_base) = u32x2{a.t[p], b.t[p]};
    };

    // The walk starts at another step in each region of a row of regions:
    // workgroups side by side then read different rows, whose lines spread
    // over the memory channels also where M is a power of two.
    const int n_steps = (i_end - i_begin + kStepRows - 1) / kStepRows;
    auto next = [&](int i) { return i + kStepRows < i_end ? i + kStepRows : i_begin; };
    const int i_first = i_begin + rj % n_steps * kStepRows;
#pragma unroll
    for (int u = 0; u < 4; ++u) issue_w(i_first, true, u);
    issue_x(i_first, true);
    // Y operands: feature d0 + 16 fb + c, columns 8h .. + 7 of group
    // 4 kh + (fb + k) % 4.
    Frag3 yf[4];
    {
      const int yd = d0 + 16 * fb + c;
      const int ydc = min(yd, D - 1);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int j = min(j0 + 128 * kh + 32 * ((fb + k) & 3) + 8 * h + u, M - 1);
          v[u] = Y[(size_t)j * D + ydc] * (Op::kScale ? sy[j] * kSplitScale : kSplitScale);
          v[u] = yd < D ? v[u] : 0.f;
        }
        yf[k] = split8(v);
      }
    }

    f32x4 accY[2][4];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int db = 0; db < 4; ++db) accY[q][db] = zero4();

    // The rows of a finished step (its buffer `b`): both halves, and the
    // waves' parts of the row sums.
    auto store_rows = [&](int i, bool valid, int b, const f32x4 (&ax)[2]) {
      if (kh == 0) {
        const buffer_rsrc rp = make_rsrc(Px + ((size_t)rj * N + i) * D,
                                         valid ? rsrc_bytes(i_end - i, D) : 0u);
        uint32_t off0 = (uint32_t)(c * D + d_out) * 4u;
        asm volatile("" : "+v"(off0));
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
          const uint32_t off = off0 + (uint32_t)(16 * mb * D) * 4u;
          f32x4 o = ax[mb] + lds.half[b][fb][mb][lane];
          if (D % 4 == 0) {
            const uint32_t at = d_out < D ? off : kOutside;
            if (s > 0) o += buffer_load4(rp, at, 0);
            buffer_store4(rp, o, at, 0);
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const uint32_t at = d_out + u < D ? off + 4u * u : kOutside;
              if (s > 0) o[u] += buffer_load1(rp, at, 0);
              buffer_store1(rp, o[u], at, 0);
            }
          }
        }
      } else if (Op::kSums && wave == 4 && dc == 0) {
        const int row = i + lane;
        if (valid && lane < kStepRows && row < i_end) {
          float v = 0.f;
#pragma unroll
          for (int g = 0; g < 8; ++g) v += lds.rs[b][g][lane];
          float* p = Rx + (size_t)rj * N + row;
          *p = s > 0 ? *p + v : v;
        }
      }
    };

    int i = i_first, i_next = next(i);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      stage_w(0, u);
      issue_w(i_next, n_steps > 1, u);
    }
    stage_x(0);
    issue_x(i_next, n_steps > 1);

    // Step t multiplies while step t + 1, whose loads were issued a step ago,
    // is split and staged: vector instructions between the matrix ones (a
    // SIMD does not issue other waves' vector instructions while a matrix
    // instruction waits for the matrix unit, so they have to alternate in
    // each wave).
    int buf = 0, i_prev = i;
    f32x4 ax[2] = {zero4(), zero4()};  // the last step's sums over this half
    for (int t = 0; t < n_steps; ++t, buf ^= 1) {
      __syncthreads();
      store_rows(i_prev, t > 0, buf ^ 1, ax);

      // W^T . X: [feature][column] += X^T W.  A step's six products are
      // summed apart from the walk's sums: one rounding of those per step.
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        u32x4 xf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          xf[p] = *reinterpret_cast<const u32x4*>(&lds.x[buf][p][db][h * 256 + c * 16]);
        f32x4 t2[2] = {zero4(), zero4()};
#pragma unroll
        for (int m = 0; m < kProducts; ++m)
#pragma unroll
          for (int q = 0; q < 2; ++q)
            t2[q] = mfma32(xf[kTermA[m]], wt[q].t[kTermB[m]], t2[q]);
#pragma unroll
        for (int q = 0; q < 2; ++q) accY[q][db] += t2[q];
      }
      __builtin_amdgcn_sched_barrier(0);
      // W . Y: [feature][row] = Y^T W^T over half the strip; the small
      // products in sums of their own.
      const int i_load = next(i_next);
      f32x4 al[2], rs[2];
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) al[mb] = ax[mb] = zero4();
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const unsigned char* src = &lds.w[buf][0][0][0][0] +
                                   (4 * kh + ((fb + k) & 3)) * 1024 + ((k & 1) ? r_next : r_own);
        u32x4 wf3[2][3];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            wf3[mb][p] = *reinterpret_cast<const u32x4*>(src + (p * 2 + mb) * 8 * 1024);
#pragma unroll
        for (int m = 0; m < kProducts; ++m)
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) {
            f32x4& a = m < 3 ? al[mb] : ax[mb];
            a = mfma32(yf[k].t[kTermA[m]], wf3[mb][kTermB[m]], a);
          }
        if constexpr (Op::kSums) {
          if (k == 0) {
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) {
              rs[mb] = zero4();
#pragma unroll
              for (int p = 2; p >= 0; --p) rs[mb] = mfma32(ones, wf3[mb][p], rs[mb]);
            }
          }
        }
        stage_w(buf ^ 1, k);
        issue_w(i_load, t + 2 < n_steps, k);
#pragma unroll
        for (int g = 0; g < 12; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a matrix instruction,
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // four vector ones
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      stage_x(buf ^ 1);
      issue_x(i_load, t + 2 < n_steps);
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        ax[mb] += al[mb];
        if (kh == 1) lds.half[buf][fb][mb][lane] = ax[mb];
        if constexpr (Op::kSums) {
          if (h == 0) lds.rs[buf][wave][16 * mb + c] = rs[mb][0];
        }
      }
      i_prev = i;
      i = i_next;
      i_next = i_load;
    }
    __syncthreads();
    store_rows(i_prev, true, buf ^ 1, ax);
    if constexpr (Op::kSums) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        csum[q] += __shfl_xor(csum[q], 16, 64);
        csum[q] += __shfl_xor(csum[q], 32, 64);
      }
      if (dc == 0 && h == 0) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
          if (col + q < M) Ry[(size_t)ri * M + col + q] = csum[q];
      }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (col + q >= M) continue;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int d = d0 + 16 * db + 4 * h;
        float* p = Py + ((size_t)ri * M + col + q) * D + d;
        if (d + 3 < D) {
          store4_u(p, accY[q][db]);
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (d + u < D) p[u] = accY[q][db][u];
        }
      }
    }
    __syncthreads();  // the buffers are free for the next strip
  }
}

// An output's contraction, and the sum of its weights, added up directly (in
// 64 bits, which overflow nowhere): acc = sum_o W_o scale_o B[o][d ..], sum =
// sum_o W_o, W_o = dK[at + o step], times K there when Op::kProduct.
template <class Op, class Vec>
__device__ __forceinline__ void direct_sums(const float* __restrict__ dK,
                                            const float* __restrict__ K, size_t at, size_t step,
                                            const float* __restrict__ B,
                                            const float* __restrict__ scale, int64_t others,
                                            int64_t D, Vec& acc, float& sum) {
  constexpr int V = sizeof(Vec) / sizeof(float);
  double a[V] = {}, s = 0.;
#pragma unroll 1  // rarely taken: little code beside the callers' own
  for (int64_t o = 0; o < others; ++o) {
    float w = dK[at + o * step];
    if constexpr (Op::kProduct) w *= K[at + o * step];
    s += (double)w;
    float sc = 1.f;
    if constexpr (Op::kScale) sc = scale[o];
#pragma unroll
    for (int v = 0; v < V; ++v) a[v] += (double)w * (double)(B[o * D + v] * sc);
  }
  sum = (float)s;
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = (float)a[v];
}

// Workspace floats with which a split backward fills the chip: at most 16
// partial rows for each row of X, one per 256 columns of W, and one for each
// row of Y per region of at least 256 rows, as many as make 256 workgroups (0:
// the shape is out of range).
inline size_t split_floats(int64_t N, int64_t M, int64_t D, bool sums) {
  if (!split_in_range(N, M, D)) return 0;
  const int64_t nrj = std::min(ceil_div(M, (int64_t)kStripCols), (int64_t)16);
  const int64_t want = ceil_div((int64_t)256, nrj * ceil_div(D, (int64_t)kFeat));
  const int64_t nri = std::min(ceil_div(N, (int64_t)256), want);
  return (size_t)(nrj * N + nri * M) * (size_t)(D + (sums ? 1 : 0));
}

// How a backward is cut: regions of RI rows x SJ strips, partials
// [nRJ][N][D], [nRJ][N], [nRI][M][D], [nRI][M] in the workspace.
struct SplitBwdPlan {
  bool ok = false;
  int RI = 0, SJ = 0, nRI = 0, nRJ = 0, n_dc = 0;
  size_t px = 0, rx = 0, py = 0, ry = 0;  // workspace offsets (floats)
  size_t ws_floats = 0;
};

// The cut with the lowest modelled time among those whose partials fit
// `budget` floats (ok = false when none does, or the shape is out of range).
// One workgroup runs per CU: a launch takes ceil(workgroups / 256) rounds of
// SJ walks, each a fill and drain of about kFill steps and RI / 32 steps; the
// partials, written once and read once, move at kStepBytes per step.
inline SplitBwdPlan plan_split_backward(int64_t N, int64_t M, int64_t D, bool sums,
                                        size_t budget) {
  SplitBwdPlan best;
  if (!split_in_range(N, M, D)) return best;
  constexpr double kFill = 1.5, kStepBytes = 15e6;
  const int64_t n_dc = ceil_div(D, (int64_t)kFeat), strips = ceil_div(M, (int64_t)kStripCols);
  const int64_t steps = ceil_div(N, (int64_t)kStepRows), row = D + (sums ? 1 : 0);
  double cost = 0.0;
  // More strips per region (their partial rows read and added to, one strip
  // after the other) only while the chip is not filled.
  for (int64_t sj = 1; (int64_t)best.nRI * best.nRJ * n_dc < 192; sj = std::min(2 * sj, strips)) {
    const int64_t nrj = ceil_div(strips, sj);
    for (int64_t k = 1;; k = k < 8 ? k + 1 : k + k / 4) {
      k = std::min(k, steps);
      const int64_t nri = ceil_div(steps, k);
      const size_t floats = (size_t)(nrj * N + nri * M) * (size_t)row;
      const int64_t wgs = ceil_div(nri * nrj, (int64_t)8) * 8 * n_dc;
      if (floats <= budget && wgs <= max_blocks(kBwdThreads)) {
        const double moved = 2.0 * (double)floats + (double)((strips - nrj) * N * row);
        const double c = (double)(ceil_div(nri * nrj * n_dc, (int64_t)256) * sj) * (k + kFill) +
                         moved * sizeof(float) / kStepBytes;
        if (!best.ok || c < cost) {
          cost = c;
          best.ok = true;
          best.RI = (int)(k * kStepRows);
          best.SJ = (int)sj;
          best.nRI = (int)nri;
          best.nRJ = (int)nrj;
        }
      }
      if (k == steps) break;
    }
    if (sj == strips) break;
  }
  if (!best.ok) return best;
  best.n_dc = (int)n_dc;
  best.rx = (size_t)best.nRJ * N * D;
  best.py = best.rx + (sums ? (size_t)best.nRJ * N : 0);
  best.ry = best.py + (size_t)best.nRI * M * D;
  best.ws_floats = best.ry + (sums ? (size_t)best.nRI * M : 0);
  return best;
}

template <class Op>
int launch_bwd_split(const SplitBwdPlan& p, const float* X, const float* Y, const float* dK,
                     const float* K, float* ws, int64_t N, int64_t M, int64_t D, const float* sx,
                     const float* sy, hipStream_t stream, const char* who) {
  auto* kernel = M == 1 ? &pair_bwd_split_kernel<Op, true> : &pair_bwd_split_kernel<Op, false>;
  const int st = raise_dynamic_lds(reinterpret_cast<const void*>(kernel), (int)sizeof(BwdLds));
  if (st) return st;
  const int64_t regions = (int64_t)p.nRI * p.nRJ;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(ceil_div(regions, (int64_t)8) * 8 * p.n_dc)),
                     dim3(kBwdThreads), sizeof(BwdLds), stream, X, Y, dK, K, ws + p.px, ws + p.rx,
                     ws + p.py, ws + p.ry, (int)N, (int)M, (int)D, p.RI, p.SJ, p.nRJ,
                     (int)regions, p.n_dc, sx, sy);
  return check_launch(who);
}

}  // namespace pairwise
}  // namespace nl2k
