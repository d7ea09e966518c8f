// The tied output head on gfx950: logits[b][o] = dot(hidden[b], embed[o])
// for B rows and V outputs, in the reference's order, so the sampler that
// follows sees the reference's logits bit for bit.
//
// crates/llm-core/src/model.rs:396-397 computes a decode step's logits as
// ops::linear_fwd(&final_normed, &weights.embed, 1, h, vocab), whose dot
// product (crates/llm-core/src/ops/linear.rs:19-32) keeps four
// accumulators over the chunks of 4 (acc[k] += a[4j+k] * b[4j+k], a
// binary32 multiply then a binary32 add, in increasing j), folds the
// remainder's products from zero, and returns ((acc0 + acc1) + (acc2 +
// acc3)) + tail. Matching those bits rules out fused multiply-adds, and so
// accumulating in the matrix cores; every product is rounded on its own and
// every accumulator takes its additions one at a time.
//
// Four kernels share this file (launch_tied_head picks one):
//
//  * tied_head_mfma_kernel: the matrix cores make the products and the
//    vector ALUs only add them, in 32 x 32 tiles per wave.
//  * tied_head_mfma16_kernel: the same in 16 x 16 tiles, for few rows or
//    few tiles.
//  * tied_head_valu_kernel: vector multiplies and adds, for short rows (h up
//    to 64), where the logits' writes and the workgroups' latency are the time.
//  * tied_head_gemv_kernel (one to four rows): one pass over embed with no
//    padding rows, bound by reading embed.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace llmhip {

struct HeadArgs {
  const float* hidden;  // [B][ldh]
  const float* embed;   // [V][lde]
  float* logits;        // [B][ldl]
  uint64_t ldh, lde, ldl;
  uint32_t B, V, h;
  uint32_t row0, row_tiles;  // the matrix-core launch's rows: row_tiles tiles from row0
  uint32_t out0, out_tiles;  // and its outputs
};

// Four floats of a row. Rows need no alignment beyond a float's: gfx950's
// 16-byte global loads take any 4-byte aligned address.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Chunk c of a row (floats 4c .. 4c+3), zeros past the row's nch chunks: a
// product 0 * 0 added to an accumulator leaves its value unchanged (an
// accumulator is never -0: it starts at +0).
__device__ __forceinline__ f4 head_chunk(const float* row, uint32_t c, uint32_t nch) {
  const bool ok = c < nch;
  const f4 v = *reinterpret_cast<const f4u*>(row + (ok ? 4u * c : 0u));
  return ok ? v : f4{0.0f, 0.0f, 0.0f, 0.0f};
}

// The remainder's fold, from zero (h % 4 products).
__device__ __forceinline__ float head_tail(const float* x, const float* w, uint32_t h) {
  float t = 0.0f;
  for (uint32_t j = h & ~3u; j < h; ++j) t = t + x[j] * w[j];
  return t;
}

// ---------------------------------------------------------------------------
// Matrix-core products. v_mfma_f32_32x32x1_2b multiplies a 32-element column
// by a 32-element row in each of two blocks and adds C. With one product per
// result and C = 0 each result is one binary32 product, rounded to nearest
// even with denormals kept: the bits of v_mul_f32 (checked over random bit
// patterns, denormal inputs and denormal products). Block 0 takes chunk 2p's
// element k and block 1 chunk 2p+1's, so one instruction makes the next two
// products of accumulator k for a 32 x 32 tile, and 32 vector adds per wave
// put them into the accumulators in the reference's order.
//
// Bound: the SIMDs' binary32 units, which binary32 matrix instructions share
// with the vector ALU (a product instruction and 32 adds take 66 + 140 cycles
// whether or not they depend on each other). A product costs half a vector
// multiply there, so a multiply-add takes 3/4 of the time of a vector
// multiply and a vector add. B = 256, V = 32000, h = 512: 190 us with vector
// multiplies (32 x 128 tiles of 4 x 4 results per thread), 164 us so, against
// 160 us for the instructions alone at the 2.2 GHz that the card holds here.
// A wave holds 32 rows x 32 outputs x 4 accumulators in 64 registers and two
// sets of products in 64 more; the next products are issued before the adds
// of the last.
//
// A workgroup of 4 waves takes 64 rows x 64 outputs, the shared dimension
// staged through LDS 32 floats at a time. A stage's global loads go out two
// stages before its products (one stage ahead: 171 us, and 1.3 times the
// time at 64 rows and fewer). Chunk q of row r is at [q][r]: a wave's reads
// are 32 consecutive float4 in each half; the odd row stride spreads the 8
// chunks that 8 threads store for one row over the banks.
// ---------------------------------------------------------------------------
constexpr uint32_t kHeadThreads = 256;
constexpr uint32_t kHeadStage = 8;  // chunks per stage
typedef float f32x32 __attribute__((ext_vector_type(32)));

__global__ __launch_bounds__(kHeadThreads, 2) void tied_head_mfma_kernel(HeadArgs a) {
  constexpr uint32_t WR = 2u, WO = 2u;  // waves by rows and by outputs
  constexpr uint32_t kRows = 32u * WR, kOuts = 32u * WO;
  __shared__ f4 xs[2][kHeadStage][kRows + 1];
  __shared__ f4 ws[2][kHeadStage][kOuts + 1];
  const uint32_t t = threadIdx.x, lane = t & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(t >> 6));
  // Workgroups go to the 8 XCDs in turn. Each XCD takes whole output tiles,
  // all their row tiles one after the other, so a tile's part of embed is
  // read into one L2 once.
  const uint32_t q = blockIdx.x >> 3;
  const uint32_t rt = q % a.row_tiles, ot = (q / a.row_tiles) * 8u + (blockIdx.x & 7u);
  if (ot >= a.out_tiles) return;
  const uint32_t r0 = a.row0 + rt * kRows, o0 = a.out0 + ot * kOuts;
  const uint32_t nch = a.h >> 2;

  // Staging: thread t loads chunk t & 7 of rows t >> 3 and 32 apart. Rows
  // past the last read the last (their results are not stored).
  const uint32_t sq = t & 7u, sr = t >> 3;
  const float* xrow[WR];
  const float* wrow[WO];
#pragma unroll
  for (int i = 0; i < WR; ++i) xrow[i] = a.hidden + (size_t)min(r0 + sr + 32u * i, a.B - 1u) * a.ldh;
#pragma unroll
  for (int i = 0; i < WO; ++i) wrow[i] = a.embed + (size_t)min(o0 + sr + 32u * i, a.V - 1u) * a.lde;
  f4 xga[WR], wga[WO], xgb[WR], wgb[WO];
  auto fetch = [&](f4 (&xg)[WR], f4 (&wg)[WO], uint32_t c0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WR; ++i) xg[i] = head_chunk(xrow[i], c0 + sq, nch);
#pragma unroll
    for (int i = 0; i < WO; ++i) wg[i] = head_chunk(wrow[i], c0 + sq, nch);
  };
  auto stage = [&](const f4 (&xg)[WR], const f4 (&wg)[WO], uint32_t buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WR; ++i) xs[buf][sq][sr + 32u * i] = xg[i];
#pragma unroll
    for (int i = 0; i < WO; ++i) ws[buf][sq][sr + 32u * i] = wg[i];
  };

  const uint32_t wr = wave % WR, wo = wave / WR, half = lane >> 5, l32 = lane & 31u;
  f4 acc[4][4];  // [accumulator k][result registers 4g .. 4g+3]
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[k][g] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // One stage's products and adds from LDS buffer buf.
  auto multiply = [&](uint32_t buf) __attribute__((always_inline)) {
    f4 xr[2], wv[2];
    auto operands = [&](int p, f4& x, f4& w) __attribute__((always_inline)) {
      x = xs[buf][2 * p + half][32u * wr + l32];
      w = ws[buf][2 * p + half][32u * wo + l32];
    };
    operands(0, xr[0], wv[0]);
    const f32x32 zero = {};
    f32x32 pr[2];
    pr[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(xr[0][0], wv[0][0], zero, 0, 0, 0);
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      const int p = m >> 2, k = m & 3;
      if (k == 0 && p < 3) operands(p + 1, xr[(p + 1) & 1], wv[(p + 1) & 1]);
      // The next products go out ahead of this step's adds.
      if (m < 15) {
        const int pn = (m + 1) >> 2, kn = (m + 1) & 3;
        pr[(m + 1) & 1] = __builtin_amdgcn_mfma_f32_32x32x1f32(xr[pn & 1][kn], wv[pn & 1][kn], zero, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      const f32x32& c = pr[m & 1];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[k][e >> 2][e & 3] = acc[k][e >> 2][e & 3] + c[16 * b + e];
      // The adds stay here (left to itself the compiler moves them behind
      // every product of the stage and spills the products).
      asm volatile("" : "+v"(acc[k][0]), "+v"(acc[k][1]), "+v"(acc[k][2]), "+v"(acc[k][3]));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Stage i's loads go out two stages before its products (chunks past the
  // row's last read as zero).
  const uint32_t ns = (nch + kHeadStage - 1u) / kHeadStage;
  if (ns != 0u) {
    fetch(xga, wga, 0u);
    fetch(xgb, wgb, kHeadStage);
    stage(xga, wga, 0u);
    __syncthreads();
  }
  for (uint32_t i = 0; i < ns; i += 2u) {
    fetch(xga, wga, (i + 2u) * kHeadStage);
    multiply(0u);
    stage(xgb, wgb, 1u);
    __syncthreads();
    fetch(xgb, wgb, (i + 3u) * kHeadStage);
    if (i + 1u < ns) multiply(1u);
    stage(xga, wga, 0u);
    __syncthreads();
  }

  // ((acc0 + acc1) + (acc2 + acc3)) + tail. Result register e of a lane is
  // row 8 (e / 4) + 4 half + e % 4, output l32 of the wave's tile.
  const uint32_t out = o0 + 32u * wo + l32;
  if (out >= a.V) return;
  const float* wo_row = a.embed + (size_t)out * a.lde;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const uint32_t row = r0 + 32u * wr + 8u * (uint32_t)(e >> 2) + 4u * half + (uint32_t)(e & 3);
    if (row >= a.B) continue;
    const float s = (acc[0][e >> 2][e & 3] + acc[1][e >> 2][e & 3]) + (acc[2][e >> 2][e & 3] + acc[3][e >> 2][e & 3]);
    a.logits[(size_t)row * a.ldl + out] = s + head_tail(a.hidden + (size_t)row * a.ldh, wo_row, a.h);
  }
}

// ---------------------------------------------------------------------------
// The same with 16 x 16 tiles per wave: v_mfma_f32_16x16x1_4b makes one
// chunk's four products (block k: accumulator k) of a tile, and 16 adds take
// them. A quarter of the registers and of a wave's work, so four times the
// waves hide the loads' latency where 32 x 32 tiles would leave SIMDs with
// one wave or none, and fewer padding rows. The staged rows are 36 floats
// apart, so the 16 rows x 4 elements that a wave reads lie in 64 different
// banks. V = 32000, h = 512: 16.3 us for 16 rows (vector multiplies: 62; 32 x
// 32 tiles: 31), 25.4 for 32 (42), 37.8 for 48 (41.5); embed's read is 13.
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int WR, int WO>
__global__ __launch_bounds__(kHeadThreads, 4) void tied_head_mfma16_kernel(HeadArgs a) {
  static_assert(WR * WO == 4, "four waves");
  constexpr uint32_t kRows = 16u * WR, kOuts = 16u * WO, kPitch = 4u * kHeadStage + 4u;
  constexpr int NX = (kRows + 31) / 32, NW = (kOuts + 31) / 32;
  __shared__ __attribute__((aligned(16))) float xs[2][kRows][kPitch];
  __shared__ __attribute__((aligned(16))) float ws[2][kOuts][kPitch];
  const uint32_t t = threadIdx.x, lane = t & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(t >> 6));
  const uint32_t q = blockIdx.x >> 3;
  const uint32_t rt = q % a.row_tiles, ot = (q / a.row_tiles) * 8u + (blockIdx.x & 7u);
  if (ot >= a.out_tiles) return;
  const uint32_t r0 = a.row0 + rt * kRows, o0 = a.out0 + ot * kOuts;
  const uint32_t nch = a.h >> 2;

  const uint32_t sq = t & 7u, sr = t >> 3;
  const float* xrow[NX];
  const float* wrow[NW];
#pragma unroll
  for (int i = 0; i < NX; ++i) xrow[i] = a.hidden + (size_t)min(r0 + (sr + 32u * i) % kRows, a.B - 1u) * a.ldh;
#pragma unroll
  for (int i = 0; i < NW; ++i) wrow[i] = a.embed + (size_t)min(o0 + (sr + 32u * i) % kOuts, a.V - 1u) * a.lde;
  f4 xga[NX], wga[NW], xgb[NX], wgb[NW];
  auto fetch = [&](f4 (&xg)[NX], f4 (&wg)[NW], uint32_t c0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NX; ++i) xg[i] = head_chunk(xrow[i], c0 + sq, nch);
#pragma unroll
    for (int i = 0; i < NW; ++i) wg[i] = head_chunk(wrow[i], c0 + sq, nch);
  };
  auto stage = [&](const f4 (&xg)[NX], const f4 (&wg)[NW], uint32_t buf) __attribute__((always_inline)) {
    // (A tile side of 16: threads 128 .. 255 store what 0 .. 127 do.)
#pragma unroll
    for (int i = 0; i < NX; ++i) *reinterpret_cast<f4*>(&xs[buf][(sr + 32u * i) % kRows][4u * sq]) = xg[i];
#pragma unroll
    for (int i = 0; i < NW; ++i) *reinterpret_cast<f4*>(&ws[buf][(sr + 32u * i) % kOuts][4u * sq]) = wg[i];
  };

  const uint32_t wr = wave % WR, wo = wave / WR, quarter = lane >> 4, l16 = lane & 15u;
  f4 acc[4];  // [accumulator k]: rows 4 quarter .. + 3 of the tile, output l16
#pragma unroll
  for (int k = 0; k < 4; ++k) acc[k] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](uint32_t buf) __attribute__((always_inline)) {
    const float* x = &xs[buf][16u * wr + l16][quarter];
    const float* w = &ws[buf][16u * wo + l16][quarter];
    float xv[kHeadStage], wv[kHeadStage];
#pragma unroll
    for (uint32_t c = 0; c < kHeadStage; ++c) {
      xv[c] = x[4u * c];
      wv[c] = w[4u * c];
    }
    const f32x16 zero = {};
    f32x16 pr[2];
    pr[0] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[0], wv[0], zero, 0, 0, 0);
#pragma unroll
    for (uint32_t c = 0; c < kHeadStage; ++c) {
      // The next products go out ahead of this step's adds.
      if (c + 1u < kHeadStage) pr[(c + 1u) & 1u] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[c + 1u], wv[c + 1u], zero, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[k][e] = acc[k][e] + pr[c & 1u][4 * k + e];
      asm volatile("" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const uint32_t ns = (nch + kHeadStage - 1u) / kHeadStage;
  if (ns != 0u) {
    fetch(xga, wga, 0u);
    fetch(xgb, wgb, kHeadStage);
    stage(xga, wga, 0u);
    __syncthreads();
  }
  for (uint32_t i = 0; i < ns; i += 2u) {
    fetch(xga, wga, (i + 2u) * kHeadStage);
    multiply(0u);
    stage(xgb, wgb, 1u);
    __syncthreads();
    fetch(xgb, wgb, (i + 3u) * kHeadStage);
    if (i + 1u < ns) multiply(1u);
    stage(xga, wga, 0u);
    __syncthreads();
  }

  const uint32_t out = o0 + 16u * wo + l16;
  if (out >= a.V) return;
  const float* wo_row = a.embed + (size_t)out * a.lde;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t row = r0 + 16u * wr + 4u * quarter + (uint32_t)e;
    if (row >= a.B) continue;
    const float s = (acc[0][e] + acc[1][e]) + (acc[2][e] + acc[3][e]);
    a.logits[(size_t)row * a.ldl + out] = s + head_tail(a.hidden + (size_t)row * a.ldh, wo_row, a.h);
  }
}

// ---------------------------------------------------------------------------
// Short rows: vector multiplies and adds. A workgroup computes 32 rows x 128
// outputs, thread (tr, to) of its 8 x 32 threads rows tr + 8i and outputs to +
// 32j, 64 accumulators in registers. The shared dimension is staged 16 floats
// at a time with no load in flight behind the products, so it loses where h is
// long; where h is short its small prologue and its writes, consecutive
// workgroups filling consecutive parts of the same rows, win. B = 256, h = 32:
// V = 32000 28.3 us with the sampler (34.5 with 32 x 32 tiles, 32.5 with 16 x
// 16), V = 65536 51.5 (65.5, 62.3); h = 16: 24.4 (34.9, 33.3).
// ---------------------------------------------------------------------------
constexpr uint32_t kValuRows = 32, kValuOuts = 128, kValuStage = 4;  // chunks per stage

__global__ __launch_bounds__(kHeadThreads) void tied_head_valu_kernel(HeadArgs a) {
  __shared__ f4 xs[kValuStage][kValuRows];
  __shared__ f4 ws[kValuStage][kValuOuts];
  const uint32_t t = threadIdx.x, tr = t >> 5, to = t & 31u;
  const uint32_t o0 = a.out0 + (blockIdx.x % a.out_tiles) * kValuOuts;
  const uint32_t r0 = a.row0 + (blockIdx.x / a.out_tiles) * kValuRows;
  const uint32_t nch = a.h >> 2;

  f4 acc[4][4];  // [row i][output j], element k: accumulator k
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // Staging: thread t loads chunk t & 3 of embed rows t >> 2 and 64 further,
  // and below 128 of hidden row t >> 2. Rows past the last read the last
  // (their results are not stored).
  const uint32_t sq = t & 3u, sr = t >> 2;
  const float* xrow = a.hidden + (size_t)min(r0 + (sr & 31u), a.B - 1u) * a.ldh;
  const float* wrow0 = a.embed + (size_t)min(o0 + sr, a.V - 1u) * a.lde;
  const float* wrow1 = a.embed + (size_t)min(o0 + 64u + sr, a.V - 1u) * a.lde;
  for (uint32_t c0 = 0; c0 < nch; c0 += kValuStage) {
    const f4 xv = head_chunk(xrow, c0 + sq, nch);
    const f4 wv0 = head_chunk(wrow0, c0 + sq, nch), wv1 = head_chunk(wrow1, c0 + sq, nch);
    __syncthreads();  // the previous stage's reads are done
    if (t < 128u) xs[sq][sr] = xv;
    ws[sq][sr] = wv0;
    ws[sq][64u + sr] = wv1;
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < kValuStage; ++c) {
      f4 x[4], w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = xs[c][tr + 8u * i];
        w[i] = ws[c][to + 32u * i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int k = 0; k < 4; ++k) acc[i][j][k] = acc[i][j][k] + x[i][k] * w[j][k];
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t row = r0 + tr + 8u * i;
    if (row >= a.B) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t out = o0 + to + 32u * j;
      if (out >= a.V) continue;
      const float s = (acc[i][j][0] + acc[i][j][1]) + (acc[i][j][2] + acc[i][j][3]);
      a.logits[(size_t)row * a.ldl + out] =
          s + head_tail(a.hidden + (size_t)row * a.ldh, a.embed + (size_t)out * a.lde, a.h);
    }
  }
}

// ---------------------------------------------------------------------------
// Few rows: one pass over embed. A wave takes 16 outputs; lanes 4i .. 4i+3
// share output i, lane j of the four holding its accumulator j for all R
// rows. They load 4 consecutive chunks of the row at a time (64 bytes, a
// float4 each) and exchange them (a 4 x 4 transpose by quad moves), so that
// lane j has element j of each, in order. The hidden rows are in LDS with
// element j of consecutive chunks contiguous. 8 loads per lane are in
// flight while the 8 before them are used.
//
// Bound: reading embed (4 V h bytes, once), up to the LDS reads of the hidden
// rows (one b128 per row for 4 chunks). V = 32000, h = 512: 12.5 us for one
// row (5.2 TB/s; 62 us with 32-row tiles), 14.2 for 2, 18.2 for 4.
// ---------------------------------------------------------------------------
constexpr uint32_t kGemvBatch = 8;        // float4 loads per lane and batch (groups of 4 chunks)
constexpr uint32_t kGemvBlockCh = 256;    // chunks of the hidden rows in LDS at a time
constexpr uint32_t kGemvWaves = 2;

template <int CTRL>
__device__ __forceinline__ float quad_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

template <int R>
__global__ __launch_bounds__(64 * kGemvWaves, 4) void tied_head_gemv_kernel(HeadArgs a) {
  constexpr uint32_t kPitch = kGemvBlockCh + 4u;  // the four elements' rows start 4 banks apart
  __shared__ __attribute__((aligned(16))) float xs[R][4][kPitch];
  constexpr int kXor1 = 0xB1, kXor2 = 0x4E;  // quad_perm [1,0,3,2] and [2,3,0,1]
  const uint32_t t = threadIdx.x, lane = t & 63u, j = lane & 3u;
  const uint32_t out = (blockIdx.x * kGemvWaves + (t >> 6)) * 16u + (lane >> 2);
  const float* wrow = a.embed + (size_t)min(out, a.V - 1u) * a.lde;
  const uint32_t nch = a.h >> 2;
  const bool odd = (j & 1u) != 0u, high = (j & 2u) != 0u;
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0f;

  // Batch i: chunks kStep i .. of the row (whole batches only).
  constexpr uint32_t kStep = 4u * kGemvBatch;
  auto fetch = [&](f4 (&w)[kGemvBatch], uint32_t i) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t g = 0; g < kGemvBatch; ++g) w[g] = *reinterpret_cast<const f4u*>(wrow + 4u * (kStep * i + 4u * g + j));
  };
  // Four chunks' products and adds; cb: the first of them within the LDS block.
  auto use4 = [&](const f4& w, uint32_t cb) __attribute__((always_inline)) {
    // Element j of the four chunks, from the four lanes (every lane moves: a
    // quad move reads the other lanes' registers).
    const float x0 = quad_move<kXor1>(w[0]), x1 = quad_move<kXor1>(w[1]);
    const float x2 = quad_move<kXor1>(w[2]), x3 = quad_move<kXor1>(w[3]);
    const float n0 = odd ? x1 : w[0], n1 = odd ? w[1] : x0;
    const float n2 = odd ? x3 : w[2], n3 = odd ? w[3] : x2;
    const float y0 = quad_move<kXor2>(n0), y1 = quad_move<kXor2>(n1);
    const float y2 = quad_move<kXor2>(n2), y3 = quad_move<kXor2>(n3);
    const f4 e = f4{high ? y2 : n0, high ? y3 : n1, high ? n2 : y0, high ? n3 : y1};
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const f4 x = *reinterpret_cast<const f4*>(&xs[r][j][cb]);
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[r] = acc[r] + x[c] * e[c];
    }
    // (Four chunks at a time: hoisting every chunk's hidden values would
    // take over 200 registers at R = 4.)
    __builtin_amdgcn_sched_barrier(0);
  };
  auto use = [&](const f4 (&w)[kGemvBatch], uint32_t i) __attribute__((always_inline)) {
    const uint32_t cb = i % (kGemvBlockCh / kStep) * kStep;
#pragma unroll
    for (uint32_t g = 0; g < kGemvBatch; ++g) use4(w[g], cb + 4u * g);
  };
  // The hidden chunks of LDS block k, zeros past the row.
  auto stage = [&](uint32_t k) __attribute__((always_inline)) {
    const uint32_t f0 = 4u * kGemvBlockCh * k, n = min(4u * kGemvBlockCh, (4u * nch - f0 + 15u) & ~15u);
    if (k != 0u) __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float* x = a.hidden + (size_t)min((uint32_t)r, a.B - 1u) * a.ldh + f0;
      for (uint32_t i = t; i < n; i += 64u * kGemvWaves) xs[r][i & 3u][i >> 2] = f0 + i < 4u * nch ? x[i] : 0.0f;
    }
    __syncthreads();
  };

  const uint32_t nb = nch / kStep;
  static_assert(kGemvBlockCh % (2u * kStep) == 0u, "a pair of batches lies in one block");
  if (nb != 0u) {
    f4 wa[kGemvBatch], wb[kGemvBatch];
    fetch(wa, 0u);
    for (uint32_t i = 0; i < nb; i += 2u) {
      if (i % (kGemvBlockCh / kStep) == 0u) stage(i / (kGemvBlockCh / kStep));
      // (The last fetches repeat the row's last batch: no branch around them.)
      fetch(wb, min(i + 1u, nb - 1u));
      use(wa, i);
      fetch(wa, min(i + 2u, nb - 1u));
      if (i + 1u < nb) use(wb, i + 1u);
    }
  }
  // The chunks past the last whole batch.
  if (nb % (kGemvBlockCh / kStep) == 0u && nb * kStep < nch) stage(nb / (kGemvBlockCh / kStep));
  for (uint32_t c = nb * kStep; c < nch; c += 4u) use4(head_chunk(wrow, c + j, nch), c % kGemvBlockCh);

#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float s01 = acc[r] + quad_move<kXor1>(acc[r]);  // lanes 0-1: acc0 + acc1, lanes 2-3: acc2 + acc3
    const float s = s01 + quad_move<kXor2>(s01);
    if ((uint32_t)r < a.B && out < a.V && j == 0u)
      a.logits[(size_t)r * a.ldl + out] = s + head_tail(a.hidden + (size_t)r * a.ldh, wrow, a.h);
  }
}

namespace {

template <int R>
hipError_t launch_gemv(const HeadArgs& a0, hipStream_t s) {
  HeadArgs a = a0;
  constexpr uint32_t kOuts = 16u * kGemvWaves;
  // (V < 2^31: at most 2^26 workgroups of 128 threads; the device takes
  // fewer than 2^32 threads a launch, so a larger V goes in slices.)
  constexpr uint32_t kMaxOuts = (1u << 20) * kOuts;
  for (uint32_t o = 0; o < a0.V; o += kMaxOuts) {
    a.embed = a0.embed + (size_t)o * a0.lde;
    a.logits = a0.logits + o;
    a.V = std::min(kMaxOuts, a0.V - o);
    hipLaunchKernelGGL(tied_head_gemv_kernel<R>, dim3((a.V + kOuts - 1u) / kOuts), dim3(64u * kGemvWaves), 0, s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Launches over slices of at most 2^10 row tiles x 2^12 output tiles.
template <class Launch>
hipError_t launch_slices(const HeadArgs& a0, uint32_t rows, uint32_t outs, Launch&& launch) {
  HeadArgs a = a0;
  constexpr uint32_t kMaxRowTiles = 1u << 10, kMaxOutTiles = 1u << 12;
  const uint32_t rts = (a.B + rows - 1u) / rows, ots = (a.V + outs - 1u) / outs;
  for (uint32_t t0 = 0; t0 < rts; t0 += kMaxRowTiles) {
    a.row0 = t0 * rows;
    a.row_tiles = std::min(kMaxRowTiles, rts - t0);
    for (uint32_t u0 = 0; u0 < ots; u0 += kMaxOutTiles) {
      a.out0 = u0 * outs;
      a.out_tiles = std::min(kMaxOutTiles, ots - u0);
      launch(a);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

// TILE x TILE results per wave, WR x WO waves.
template <int TILE, int WR, int WO>
hipError_t launch_mfma(const HeadArgs& a0, hipStream_t s) {
  return launch_slices(a0, TILE * WR, TILE * WO, [&](const HeadArgs& a) {
    const uint32_t grid = (a.out_tiles + 7u) / 8u * 8u * a.row_tiles;
    if constexpr (TILE == 16) {
      hipLaunchKernelGGL((tied_head_mfma16_kernel<WR, WO>), dim3(grid), dim3(kHeadThreads), 0, s, a);
    } else {
      static_assert(TILE == 32 && WR == 2 && WO == 2, "the 32 x 32 kernel's workgroup");
      hipLaunchKernelGGL(tied_head_mfma_kernel, dim3(grid), dim3(kHeadThreads), 0, s, a);
    }
  });
}

hipError_t launch_valu(const HeadArgs& a0, hipStream_t s) {
  return launch_slices(a0, kValuRows, kValuOuts, [&](const HeadArgs& a) {
    hipLaunchKernelGGL(tied_head_valu_kernel, dim3(a.out_tiles * a.row_tiles), dim3(kHeadThreads), 0, s, a);
  });
}

}  // namespace

hipError_t launch_tied_head(const float* hidden, uint64_t ldh, const float* embed, uint64_t lde, float* logits,
                            uint64_t ldl, uint32_t B, uint32_t V, uint32_t h, hipStream_t s) {
  if (B == 0 || V == 0) return hipSuccess;
  const HeadArgs a{hidden, embed, logits, ldh, lde, ldl, B, V, h, 0u, 0u, 0u, 0u};
  // Few rows. At 3 and 4 rows the matrix products overtake the pass over
  // embed where there are enough outputs to fill the chip with tiles (V =
  // 32000, h = 512, 4 rows: 18.2 against 16.0 us; V = 8192, h = 256: 5.3
  // against 7.1).
  if (B == 1) return launch_gemv<1>(a, s);
  if (B == 2) return launch_gemv<2>(a, s);
  if (B <= 4 && V <= 16384) return launch_gemv<4>(a, s);
  // Short rows and many results: vector multiplies. B x V, us with the sampler,
  // those and the better matrix-core kernel: h = 16 8 x 65536 24.7 / 25.4, 64 x
  // 32000 14.2 / 16.2, 512 x 32000 36.4 / 54.3; h = 48 64 x 32000 17.1 / 17.6, 256
  // x 32000 33.3 / 39.6, but 64 x 8192 13.5 / 11.8 and 32 x 100000 45.0 / 43.7; h =
  // 64 256 x 65536 71.9 / 76.4, 512 x 32000 68.5 / 68.5, 128 x 32000 25.3 / 25.6,
  // but 128 x 100000 73.0 / 70.9; h = 96 256 x 65536 94.2 / 94.8, 256 x 32000 50.4
  // / 48.2.
  const uint64_t results = (uint64_t)B * V;
  if (h <= 16u   ? B >= 8u && results >= 1u << 19
      : h <= 48u ? B >= 64u && results >= 2000000u
                 : h <= 64u && results >= 16000000u)
    return launch_valu(a, s);
  // 32 x 32 tiles need two per SIMD to hide their loads (1024 tiles, V =
  // 8192 at 128 rows, h = 256: 17.7 us against 15.0 with 16 x 16 tiles; 2048,
  // at 256 rows: 25.0 against 26.9), and pay for rows padded to 64 (V = 32000,
  // h = 512: 41.5 us against 37.8 at 48 rows, 42.7 against 44.7 at 64). Over a
  // shorter h their prologue counts, the more the more tiles there are. B x V, us
  // with the sampler, 32 x 32 and 16 x 16: h = 64 256 x 32000 41.0 / 39.1, 512 x
  // 8192 30.0 / 29.3; h = 96 256 x 8192 19.6 / 20.4, 64 x 50257 39.2 / 35.6, 512 x
  // 65536 186 / 182; h = 128 256 x 8192 21.5 / 22.3, 256 x 32000 56.0 / 56.4, 128 x
  // 50257 60.1 / 55.4, 256 x 100000 169 / 165; h = 192 256 x 32000 72.6 / 73.7, 256
  // x 65536 145 / 147.
  const uint64_t tiles = (uint64_t)((B + 31u) / 32u) * ((V + 31u) / 32u);
  const uint64_t pad64 = ((uint64_t)B + 63u) / 64u * 64u, rows16 = ((uint64_t)B + 15u) / 16u;
  const bool long_rows = h >= 160u || (h > 64u && V <= 40000u);
  if (long_rows && tiles >= 2048u && pad64 * 8u <= rows16 * 16u * 9u) return launch_mfma<32, 2, 2>(a, s);
  // Pairs of 16-row tiles share a workgroup's part of embed; an odd count
  // would pad (24 rows: 26.6 us one by one, 25.3 in a pair; 48: 37.8, 44.0).
  return rows16 % 2u ? launch_mfma<16, 1, 4>(a, s) : launch_mfma<16, 2, 2>(a, s);
}

}  // namespace llmhip
