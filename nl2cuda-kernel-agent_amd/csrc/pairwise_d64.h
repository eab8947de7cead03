// The backward of the pairwise cases at feature width 64 on fp32 MFMA
// (v_mfma_f32_16x16x4_f32, gfx950), for the sizes where it is the faster one
// (takes_regions): for an upstream [N, M] matrix W (W = dK o K when
// Op::kProduct, else W = dK) both contractions W . Y and W^T . X in one pass
// over the [N, M] inputs, as raw partials per region (and, when Op::kSums,
// partial row / column sums of W); Op::kScale multiplies every staged X row i
// by sx[i] and Y row j by sy[j] first.  A case-specific reduce kernel sums
// the partials and applies its epilogue.
#pragma once

#include <algorithm>
#include <cstdint>

#include "common.h"

namespace nl2k {
namespace pairwise {

constexpr int kD = 64;           // feature width of the MFMA path
constexpr int kTile = 64;        // tile edge
constexpr int kLds = 68;         // padded LDS row stride (floats)
constexpr int kTileFloats = kTile * kLds;
constexpr int kTargetRegions = 256;  // one backward workgroup per CU
// The tile kernels index rows and columns with int, up to a tile or region
// past the last one; larger N or M take the callers' generic (int64) kernels.
constexpr int64_t kMaxTileDim = INT32_MAX - 1024;

// Op interface: static constexpr bool kProduct (W = dK o K, else W = dK),
// kScale (scale X rows by sx, Y rows by sy), kSums (row / column sums).
//
// ----------------------------------------------------------------- backward
// Region = RI x RJ entries of W (RJ = 64 JC), walked in 64x64 tiles, i-chunk
// outer, j-chunk inner, by a workgroup of twelve waves in three roles, one
// wave of each per SIMD (wave w on SIMD w % 4).  A role owns 16 rows and 16
// columns of every tile per wave:
//  * waves 0-3 run the (W.Y)^T contraction (rows 16 (w & 3)..: A =
//    P[i][j..j+3], B = Yt[d][j..j+3]), accumulated over the region's columns
//    and flushed per i-chunk;
//  * waves 4-7 run the (W^T.X)^T contraction (columns 16 (w & 3)..: A =
//    P[i..i+3][j], four 4-byte reads, B = Xt[d][i..i+3]), accumulated over
//    the region's rows and flushed at the end;
//  * waves 8-11 stage: they load the upstream tiles up to three tiles ahead
//    into registers, form W into the LDS tile buffer of the next tile, and
//    stage the next i-chunk's X rows, loaded one step ahead (issued first in
//    its step, so waiting for it retires only loads at least two steps old
//    apart from itself).
// LDS: Yt = the region's Y rows, transposed [d][j], staged once; Xt = X rows
// of an i-chunk, transposed [d][i], double buffered; P = W tile [i][j],
// double buffered.  Every role runs the same loop nest and passes exactly one
// workgroup barrier per tile.  Each region writes raw partial contractions
// (and partial row / column sums of W) to its workspace slot.
// Each SIMD has two waves issuing MFMAs, and one's waits on LDS, barriers or
// its partial stores are covered by the other's matrix work.  The role index
// is read through readfirstlane so the compiler sees wave-uniform branches
// and gives each role its own live ranges (at most 168 VGPRs: three waves per
// SIMD).
// kFull (N and M multiples of 64, every byte offset of dK / K below 2^31):
// no tile is ragged, so the staging waves load through buffer resources
// with the tile's offset in a scalar register and a fixed per-lane offset,
// and form W without clamps or selects.  That takes about 50 of the ~75
// vector instructions per staging step off the SIMDs the matrix waves
// issue on (vector ALU and MFMA issue share a SIMD), with identical bits.
// Otherwise every tile is loaded with clamped addresses and masked (float4
// loads: M is a multiple of 4).
template <class Op, int JC, bool kFull>
__global__ __launch_bounds__(768) void pair_bwd_d64_3r_kernel(
    const float* X, const float* __restrict__ Y,
    const float* dK, const float* Kf,
    float* __restrict__ Px, float* __restrict__ Rx, float* __restrict__ Py,
    float* __restrict__ Ry, int N, int M, int RI, int nRJ,
    const float* sx, const float* __restrict__ sy) {
  // X, sx, dK and Kf are deliberately not __restrict__: with it the compiler
  // treats their loads as invariant and sinks a prefetch past the workgroup
  // barriers to its use (for dK / K, tile t+2's, which serialises the memory
  // latency; for X, the reload before the staging loop, which leaves the
  // loop's wait counts pessimistic).
  constexpr int RJ = JC * kTile;
  constexpr int kYtLds = RJ + 4;
  __shared__ __attribute__((aligned(16))) float P[2][kTileFloats];
  __shared__ __attribute__((aligned(16))) float Xt[2][kTileFloats];
  __shared__ __attribute__((aligned(16))) float Yt[kD * kYtLds];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform role
  const int n = lane & 15;
  const int h = lane >> 4;

  const int ri = blockIdx.x / nRJ;
  const int rj = blockIdx.x - ri * nRJ;
  const int ibase = ri * RI;
  const int jbase = rj * RJ;
  const int rows = min(RI, N - ibase);
  const int cols = min(RJ, M - jbase);
  const int n_ic = (rows + kTile - 1) / kTile;
  const int n_jc = (cols + kTile - 1) / kTile;
  const int n_tiles = n_ic * n_jc;
  // Skewed walk: region (ri, rj) visits its i-chunks starting at rj mod n_ic
  // and its j-chunks starting at ri mod n_jc.  With every region on the same
  // walk, the concurrent dK / K reads of all CUs share their address bits
  // and crowd the same memory channels; a 4096^2 read in 64 x 64 tiles took
  // 16.1 us in lockstep and 13.1 us skewed (12.2 us as whole rows).  The
  // walk position, not the chunk, selects the double buffers; the column
  // accumulators are kept per walk position and mapped back at the flush.
  const int ic0 = rj % n_ic, jc0 = ri % n_jc;
  auto chunk_at = [&](int pos) { return pos + ic0 < n_ic ? pos + ic0 : pos + ic0 - n_ic; };
  auto col_at = [&](int pos) { return pos + jc0 < n_jc ? pos + jc0 : pos + jc0 - n_jc; };

  // Staging-wave state (declared for all waves; only waves 8-11 use it).
  const int ptid = tid - 512;
  // W: float4 (row (p>>4) + 16 s, cols 4 (p & 15)..), s = 0..3.
  const int srow = (ptid >> 4) & 15;
  const int scol = (ptid & 15) * 4;
  // X chunk: row p & 63 (lanes along rows), float4 columns (p>>6) + 4 s.
  const int xrow = ptid & 63;
  const int xcol = ((ptid >> 6) & 3) * 4;
  f32x4 g_dk[3][4], g_k[3][4], g_x[4];
  float g_xs;
  bool g_ok[3][4];
  // Full-tile addressing: byte offsets of row srow, column scol of a tile
  // (and of row xrow, column xcol of an X chunk) from the tile's corner.
  const uint32_t lane_off = ((uint32_t)srow * (uint32_t)M + (uint32_t)scol) * 4u;
  const uint32_t xlane_off = (uint32_t)(xrow * kD + xcol) * 4u;
  const uint32_t nm_bytes = kFull ? (uint32_t)N * (uint32_t)M * 4u : 0u;
  const buffer_rsrc rdk = make_rsrc(dK, nm_bytes);
  const buffer_rsrc rkk = make_rsrc(Kf, Op::kProduct ? nm_bytes : 0u);
  const buffer_rsrc rxx = make_rsrc(X, kFull ? (uint32_t)N * (uint32_t)kD * 4u : 0u);
  auto load_stage = [&](int t, f32x4 (&dk)[4], f32x4 (&kk)[4], bool (&ok)[4]) {
    const int pi = t / n_jc;
    const int ic = chunk_at(pi), jc = col_at(t - pi * n_jc);
    const int ib = ibase + ic * kTile;
    const int jb = jbase + jc * kTile;
    if constexpr (kFull) {
      const int toff = (ib * M + jb) * 4;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        ok[s] = true;
        dk[s] = buffer_load4(rdk, lane_off, toff + s * 64 * M);
        if constexpr (Op::kProduct) kk[s] = buffer_load4(rkk, lane_off, toff + s * 64 * M);
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int gi = ib + srow + 16 * s;
        const int gj = jb + scol;
        ok[s] = gi < N && gj < M;
        const size_t o = (size_t)min(gi, N - 1) * M + min(gj, M - 4);
        dk[s] = load4(dK + o);
        if constexpr (Op::kProduct) kk[s] = load4(Kf + o);
      }
    }
  };
  auto commit_stage = [&](int t, const f32x4 (&dk)[4], const f32x4 (&kk)[4],
                          const bool (&ok)[4]) {
    float* dst = P[t & 1];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      f32x4 w = dk[s];
      if constexpr (Op::kProduct) w = w * kk[s];
      if constexpr (!kFull) w = ok[s] ? w : zero4();
      store4(&dst[(srow + 16 * s) * kLds + scol], w);
    }
  };
  auto load_x = [&](int pos, f32x4 (&xs)[4], float& sc) {
    if constexpr (kFull && !Op::kScale) {
      const int xoff = (ibase + chunk_at(pos) * kTile) * kD * 4;
#pragma unroll
      for (int s = 0; s < 4; ++s) xs[s] = buffer_load4(rxx, xlane_off + 64 * s, xoff);
      return;
    }
    const size_t r = (size_t)min(ibase + chunk_at(pos) * kTile + xrow, N - 1);
#pragma unroll
    for (int s = 0; s < 4; ++s) xs[s] = load4(X + r * kD + xcol + 16 * s);
    if constexpr (Op::kScale) sc = sx[r];
  };
  auto commit_x = [&](int pos, const f32x4 (&xs)[4], float sc) {
    float* dst = Xt[pos & 1];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (Op::kScale)
          dst[(xcol + 16 * s + u) * kLds + xrow] = xs[s][u] * sc;
        else
          dst[(xcol + 16 * s + u) * kLds + xrow] = xs[s][u];
      }
  };
  // X chunk (walk position) published at step t: the one after tile t's
  // (clamped; at the last chunk that rewrites the chunk in use with
  // identical bits).
  auto x_chunk = [&](int t) { return min(t / n_jc + 1, n_ic - 1); };

  // Tile 0's loads go out first.  The region's Y rows are staged by waves
  // 0-7 as four 64-column chunks, transposed into Yt[d][j]: the chunk of the
  // first walk position before the first barrier, the others (loaded now,
  // behind it) right after it, before the barrier that ends step 0 (the
  // first step that needs them).  Holding the first barrier for all 64 KB
  // of Y delayed every region's first tile by about 2 us.  Thread tid < 512
  // moves float4 f = tid + 512 k of a chunk: column f % 64 (lanes along j,
  // so the transposed LDS writes hit consecutive banks), d-group f / 64.
  if (wave >= 8) {
    load_x(0, g_x, g_xs);
    load_stage(0, g_dk[0], g_k[0], g_ok[0]);
  }
  constexpr int kYc = 2;  // float4 per thread per chunk
  f32x4 yv[JC][kYc];
  float ys[JC][kYc];
  auto commit_y = [&](int pc) {
#pragma unroll
    for (int k2 = 0; k2 < kYc; ++k2) {
      const int f = tid + 512 * k2;
      const int j = col_at(pc) * kTile + (f & 63);
      const int c = (f >> 6) * 4;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (Op::kScale)
          Yt[(c + u) * kYtLds + j] = yv[pc][k2][u] * ys[pc][k2];
        else
          Yt[(c + u) * kYtLds + j] = yv[pc][k2][u];
      }
    }
  };
  if (tid < 512) {
#pragma unroll
    for (int pc = 0; pc < JC; ++pc) {
      if (pc < n_jc) {
#pragma unroll
        for (int k2 = 0; k2 < kYc; ++k2) {
          const int f = tid + 512 * k2;
          const size_t yr = (size_t)min(jbase + col_at(pc) * kTile + (f & 63), M - 1);
          yv[pc][k2] = load4(Y + yr * kD + (f >> 6) * 4);
          if constexpr (Op::kScale) ys[pc][k2] = sy[yr];
        }
      }
    }
    commit_y(0);
  }
  // Both roles pass 1 + n_tiles barriers.

  if (wave >= 8) {
    // ------------------------------------------------------ staging waves
    // Every step t runs the same straight-line sequence (no branches, so the
    // loads of later tiles stay in flight across steps): publish the X chunk
    // after tile t's (its registers were loaded last step), load the X chunk
    // for step t+1, load tile t+3 into the register stage published last
    // step, then publish W of tile t+1 from stage (t+1) % 3, loaded two steps
    // ago.  The memory counter retires in order, so the X wait, on the
    // step's oldest young load, retires nothing younger than two steps but
    // that load.  Indices are clamped: loads past the last tile fetch valid
    // data nobody uses; commits past it fill the idle P buffer.  A
    // republished X chunk rewrites the buffer the compute waves are reading
    // only with identical bits.  The three W register stages are addressed
    // statically (the loop is unrolled by three): a runtime stage index would
    // be if-converted into selects on the loaded data, forcing a wait right
    // after each load.
    // The X reload goes out before tiles 1 and 2 (the barrier keeps the
    // compiler from hoisting their loads above it): the loop then starts
    // with the same order of outstanding loads as every later pass, and the
    // wait counts at the loop head stay as tight as in the body.  Otherwise
    // the loop's first step of every three waited for the previous step's
    // tiles.
    commit_x(0, g_x, g_xs);
    load_x(x_chunk(0), g_x, g_xs);
    __builtin_amdgcn_sched_barrier(0);
    load_stage(min(1, n_tiles - 1), g_dk[1], g_k[1], g_ok[1]);
    load_stage(min(2, n_tiles - 1), g_dk[2], g_k[2], g_ok[2]);
    __builtin_amdgcn_sched_barrier(0);
    commit_stage(0, g_dk[0], g_k[0], g_ok[0]);
    __syncthreads();
    auto step = [&](int t, f32x4 (&ldk)[4], f32x4 (&lk)[4], bool (&lok)[4],
                    const f32x4 (&cdk)[4], const f32x4 (&ck)[4], const bool (&cok)[4]) {
      __builtin_amdgcn_sched_barrier(0);
      commit_x(x_chunk(t), g_x, g_xs);
      load_x(x_chunk(t + 1), g_x, g_xs);
      load_stage(min(t + 3, n_tiles - 1), ldk, lk, lok);
      commit_stage(t + 1, cdk, ck, cok);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
    };
    int t = 0;
    for (; t + 3 <= n_tiles; t += 3) {
      step(t, g_dk[0], g_k[0], g_ok[0], g_dk[1], g_k[1], g_ok[1]);
      step(t + 1, g_dk[1], g_k[1], g_ok[1], g_dk[2], g_k[2], g_ok[2]);
      step(t + 2, g_dk[2], g_k[2], g_ok[2], g_dk[0], g_k[0], g_ok[0]);
    }
    // the last n_tiles % 3 steps, on the same static stages (no padding
    // steps: each would cost a barrier round and a reload of the last tile)
    if (t < n_tiles) step(t, g_dk[0], g_k[0], g_ok[0], g_dk[1], g_k[1], g_ok[1]);
    if (t + 1 < n_tiles) step(t + 1, g_dk[1], g_k[1], g_ok[1], g_dk[2], g_k[2], g_ok[2]);
    return;
  }

  // ------------------------------------------------------- compute waves
  const int wb = wave & 3;  // 16-row block of (W.Y)^T / 16-column block of (W^T.X)^T
  __syncthreads();
#pragma unroll
  for (int pc = 1; pc < JC; ++pc)
    if (pc < n_jc) commit_y(pc);
  if (wave < 4) {
    // (W.Y)^T rows 16 wb.. of every tile, accumulated over the region's
    // columns and flushed per i-chunk (dX side).
    for (int pi = 0; pi < n_ic; ++pi) {
      const int ic = chunk_at(pi);
      f32x4 accX[4];
#pragma unroll
      for (int db = 0; db < 4; ++db) accX[db] = zero4();
      float rp = 0.f;
#pragma unroll
      for (int pj = 0; pj < JC; ++pj) {
        if (pj < n_jc) {
          const int t = pi * n_jc + pj;
          const float* Pb = P[t & 1];
          const float* Yb = Yt + col_at(pj) * kTile;
          f32x4 xa[2], xbv[2][4];
          xa[0] = load4(&Pb[(wb * 16 + n) * kLds + 4 * h]);
#pragma unroll
          for (int db = 0; db < 4; ++db) xbv[0][db] = load4(&Yb[(db * 16 + n) * kYtLds + 4 * h]);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int c = q & 1;
            if (q < 3) {
              const int k1 = 16 * (q + 1) + 4 * h;
              xa[c ^ 1] = load4(&Pb[(wb * 16 + n) * kLds + k1]);
#pragma unroll
              for (int db = 0; db < 4; ++db) xbv[c ^ 1][db] = load4(&Yb[(db * 16 + n) * kYtLds + k1]);
            }
            if constexpr (Op::kSums) rp += (xa[c][0] + xa[c][1]) + (xa[c][2] + xa[c][3]);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int db = 0; db < 4; ++db) accX[db] = mfma16x4(xa[c][u], xbv[c][db][u], accX[db]);
          }
          __syncthreads();
        }
      }
      const size_t slot = (size_t)rj * N;
      const int i_base = ibase + ic * kTile + wb * 16;
      if constexpr (Op::kSums) {
        float rs = rp;
        rs += __shfl_xor(rs, 16, 64);
        rs += __shfl_xor(rs, 32, 64);
        if (h == 0 && i_base + n < N) Rx[slot + i_base + n] = rs;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i_base + 4 * h + r;
        if (i < N) {
#pragma unroll
          for (int db = 0; db < 4; ++db) Px[(slot + i) * kD + db * 16 + n] = accX[db][r];
        }
      }
    }
    return;
  }

  // (W^T.X)^T columns 16 wb.. of every tile, accumulated over the region's
  // rows (dY side), flushed at the end.
  f32x4 accY[JC][4];
  float cp[JC];
#pragma unroll
  for (int c = 0; c < JC; ++c) {
    cp[c] = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db) accY[c][db] = zero4();
  }
  for (int pi = 0; pi < n_ic; ++pi) {
    const float* Xb = Xt[pi & 1];
#pragma unroll
    for (int jc = 0; jc < JC; ++jc) {  // walk position; column chunk col_at(jc)
      if (jc < n_jc) {
        const int t = pi * n_jc + jc;
        const float* Pb = P[t & 1];
        f32x4 yb[2][4];
        float ya[2][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) ya[0][u] = Pb[(4 * h + u) * kLds + wb * 16 + n];
#pragma unroll
        for (int db = 0; db < 4; ++db) yb[0][db] = load4(&Xb[(db * 16 + n) * kLds + 4 * h]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = q & 1;
          if (q < 3) {
            const int k1 = 16 * (q + 1) + 4 * h;
#pragma unroll
            for (int u = 0; u < 4; ++u) ya[c ^ 1][u] = Pb[(k1 + u) * kLds + wb * 16 + n];
#pragma unroll
            for (int db = 0; db < 4; ++db) yb[c ^ 1][db] = load4(&Xb[(db * 16 + n) * kLds + k1]);
          }
          if constexpr (Op::kSums) cp[jc] += (ya[c][0] + ya[c][1]) + (ya[c][2] + ya[c][3]);
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int db = 0; db < 4; ++db)
              accY[jc][db] = mfma16x4(ya[c][u], yb[c][db][u], accY[jc][db]);
        }
        __syncthreads();
      }
    }
  }
  const size_t slot = (size_t)ri * M;
#pragma unroll
  for (int jc = 0; jc < JC; ++jc) {
    if (jc < n_jc) {
      const int j_base = jbase + col_at(jc) * kTile + wb * 16;
      if constexpr (Op::kSums) {
        float cs = cp[jc];
        cs += __shfl_xor(cs, 16, 64);
        cs += __shfl_xor(cs, 32, 64);
        if (h == 0 && j_base + n < M) Ry[slot + j_base + n] = cs;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = j_base + 4 * h + r;
        if (j < M) {
#pragma unroll
          for (int db = 0; db < 4; ++db) Py[(slot + j) * kD + db * 16 + n] = accY[jc][db][r];
        }
      }
    }
  }
}

// Regions, workspace layout (floats) and, for every edge, the workspace bytes
// that callers are told: partial (W.Y) [nRJ][N][64], partial row sums
// [nRJ][N] (sums only), partial (W^T.X) [nRI][M][64], partial column sums
// [nRI][M] (sums only).
struct BwdPlan {
  bool fast = false;
  int R = 64;  // region edge (rows and columns)
  int JC = 1;  // R / 64
  int nRI = 0, nRJ = 0;
  size_t px = 0, rx = 0, py = 0, ry = 0;  // workspace offsets (floats)
  size_t ws_floats = 0;
};

inline BwdPlan plan_backward(int64_t N, int64_t M, int64_t D, bool sums) {
  BwdPlan p;
  if (D != kD || N <= 0 || M <= 0 || N > kMaxTileDim || M > kMaxTileDim) return p;
  p.fast = true;
  // The edge with the lowest modelled time, in units of one 64 x 64 tile step
  // (~2.35 us): one workgroup runs per CU at a time, so a launch takes
  // ceil(regions / 256) rounds of (R / 64)^2 steps plus about four steps of
  // fill and drain each, and the reduce moves the partial rows (written once,
  // read once) at about kStepBytes per step.  Edges above 128 are planned for
  // their workspace size alone (see takes_regions).
  constexpr double kStepBytes = 11.75e6;
  int R = 64;
  double best = 0.0;
  for (int cand : {256, 192, 128, 64}) {
    const int64_t jc = cand / kTile, nri = ceil_div(N, cand), nrj = ceil_div(M, cand);
    const int64_t rounds = ceil_div(nri * nrj, kTargetRegions);
    const double partial_bytes = (double)(nrj * N + nri * M) * (kD + 1) * sizeof(float) * 2;
    const double cost = (double)(rounds * (jc * jc + 4)) + partial_bytes / kStepBytes;
    if (cand == 256 || cost < best) {
      best = cost;
      R = cand;
    }
  }
  p.R = R;
  p.JC = R / kTile;
  p.nRI = (int)ceil_div(N, R);
  p.nRJ = (int)ceil_div(M, R);
  p.px = 0;
  p.rx = p.px + (size_t)p.nRJ * N * kD;
  p.py = p.rx + (sums ? (size_t)p.nRJ * N : 0);
  p.ry = p.py + (size_t)p.nRI * M * kD;
  p.ws_floats = p.ry + (sums ? (size_t)p.nRI * M : 0);
  return p;
}

// Which backwards run here rather than on the bf16 splits
// (pairwise_split.h): regions of at most 128 (N, M up to about 2048), rows of
// W in whole float4.  A region is then one to four tile steps, over before
// the split kernel's longer code and 256-column strips have filled (both
// kernels with their reduce: 9.0 against 16.3 us at 256 x 256, 14.8 against
// 19.9 at 1024 x 1024, 22.9 against 25.0 at 2048 x 2048); past it the split
// kernel's shorter matrix time counts (37.8 against 34.9 us at 3000 x 3000,
// 58.0 against 54.0 at 4096 x 4096, 204 against 153 at 8192 x 8192), and rows
// of other lengths, which here load element by element, are faster there at
// every size (22.4 against 19.8 us at 1001 x 999).
inline bool takes_regions(const BwdPlan& p, int64_t M, const float* X, const float* Y,
                          const float* dK, const float* K) {
  return p.fast && p.R <= 2 * kTile && M % 4 == 0 && aligned16(X) && aligned16(Y) &&
         aligned16(dK) && aligned16(K);
}

template <class Op, int JC>
void launch_regions(const BwdPlan& p, const float* X, const float* Y, const float* dK,
                    const float* K, float* ws, int N, int M, const float* sx, const float* sy,
                    hipStream_t stream) {
  // Full-tile buffer addressing when no tile is ragged and every byte offset
  // fits the resource's 32-bit range.
  const bool full = N % kTile == 0 && M % kTile == 0 &&
                    (int64_t)N * M * (int64_t)sizeof(float) < ((int64_t)1 << 31);
  auto* kernel = full ? &pair_bwd_d64_3r_kernel<Op, JC, true> : &pair_bwd_d64_3r_kernel<Op, JC, false>;
  hipLaunchKernelGGL(kernel, dim3(p.nRI * p.nRJ), dim3(768), 0, stream, X, Y, dK, K, ws + p.px,
                     ws + p.rx, ws + p.py, ws + p.ry, N, M, p.R, p.nRJ, sx, sy);
}

// Call only when takes_regions.
template <class Op>
int launch_bwd_regions(const BwdPlan& p, const float* X, const float* Y, const float* dK,
                       const float* K, float* ws, int64_t N, int64_t M, const float* sx,
                       const float* sy, hipStream_t stream, const char* who) {
  if (p.JC == 1)
    launch_regions<Op, 1>(p, X, Y, dK, K, ws, (int)N, (int)M, sx, sy, stream);
  else
    launch_regions<Op, 2>(p, X, Y, dK, K, ws, (int)N, (int)M, sx, sy, stream);
  return check_launch(who);
}

}  // namespace pairwise
}  // namespace nl2k
