// DSA indexer projection of the decode step: the LIM query rows and head
// weights of each token.
//
//   q[t, h, :]  = RoPE(q_c[t, :] . wq_b[h*D .. h*D+D-1, :]^T)   (first rope_dim dims)
//   w[t, h]     = hidden[t, :] . w_proj[h, :]^T  (x score_scale)
//
// Semantics: nanovllm/models/dsa_indexer_project.py:245-360
// (dsa_indexer_project_query_only): q rounded to 16 bits after the
// projection, then the interleaved-pair RoPE of
// ops/dsa_indexer_project/op_kernel/dsa_indexer_project_kernel.cpp:105-176
// (fp32 x*cos, fp32 rotated*sin, fp32 sum, round to nearest even), the
// weights rounded after the projection and again after the scale
// (_query_only_weights_proj_pure, :74-86).
//
// Design: the q projection is a skinny GEMM (tokens <= 64 per workgroup
// column, thousands of weight rows), bound by reading wq_b once from HBM.
// One launch covers both projections: workgroup x owns 16 rows of wq_b, and
// the head weights are spread over the same workgroups' waves, one wave per
// (token, head) dot product over hidden_size with coalesced 1 KiB loads and
// a fixed-order shuffle reduction (rather than 2 MFMA row tiles that would
// each walk all of hidden_size, or workgroups of their own that would not
// fit beside the q workgroups in one round).  In the q part the weight rows
// are the MFMA A
// operand (16 rows x 32 K per 16x16x32 step) and the tokens the B operand,
// so a lane's four accumulator values are four consecutive output rows of
// one token: the RoPE pairs (2i, 2i+1) meet in one thread after the
// cross-wave reduction.  K is walked in 256-wide chunks spread over the 8
// waves (a wave prefetches its next chunk's weight rows while it multiplies
// the current one).
#include <algorithm>

#include "nvdsa_common.h"
#include "nvdsa_kernels.h"

namespace nvdsa {
namespace {

constexpr int kProjWaves = 8;
constexpr int kProjThreads = kProjWaves * kWave;
constexpr int kRowTile = 16;              // weight rows (outputs) per workgroup
constexpr int kTokTiles = 4;              // 16-token MFMA column tiles per workgroup
constexpr int kTokPerGroup = 16 * kTokTiles;
constexpr int kSteps = 8;                 // MFMA steps per chunk, 32 K each
constexpr int kKChunk = 32 * kSteps;      // 256

// The interleaved-pair rotation of one (even, odd) pair, in fp32 with every
// product and the sum rounded separately (no fused multiply-add), as the
// reference kernel's Mul / Mul / Add.
__device__ inline void rope_pair(float x0, float x1, float c0, float c1, float s0, float s1, float& y0, float& y1) {
#pragma clang fp contract(off)
  y0 = x0 * c0 + (-x1) * s0;
  y1 = x1 * c1 + x0 * s1;
}

// Head weights: wave `wid` of the weight workgroups computes
// w[t, h] = round16(hidden[t] . w_proj[h]) (x score_scale, rounded again),
// t = wid / heads, h = wid % heads.  Lane l accumulates the products of K
// indices 512j + 8l .. +7 in fp32 (ascending j, then ascending element),
// then the lanes combine in a fixed butterfly.
template <typename T>
__device__ __forceinline__ void head_weight(const IndexerArgs& a, int64_t t, int64_t h, int lane) {
  const u32x4_t* x = reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.hidden) + t * a.hid) + lane;
  const u32x4_t* w = reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.w_proj) + h * a.hid) + lane;
  constexpr int kBatch = 12;  // 12 x 2 loads in flight per lane: all of hidden_size 6144 at once
  const int64_t iters = a.hid / 512;
  float acc = 0.f;
  for (int64_t j0 = 0; j0 < iters; j0 += kBatch) {
    u32x4_t xv[kBatch], wv[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t j = j0 + u < iters ? j0 + u : iters - 1;
      xv[u] = x[64 * j];
      wv[u] = w[64 * j];
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (j0 + u < iters) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc = fmaf(T::to_float(static_cast<uint16_t>(xv[u][e])), T::to_float(static_cast<uint16_t>(wv[u][e])), acc);
          acc = fmaf(T::to_float(static_cast<uint16_t>(xv[u][e] >> 16)),
                     T::to_float(static_cast<uint16_t>(wv[u][e] >> 16)), acc);
        }
      }
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, 64);
  if (lane == 0) {
    uint16_t o = T::from_float(acc);
    if (a.score_scale != 1.f) o = T::from_float(T::to_float(o) * a.score_scale);
    static_cast<uint16_t*>(a.w_out)[t * a.heads + h] = o;
  }
}

template <typename T>
__global__ __launch_bounds__(kProjThreads) void indexer_project_kernel(IndexerArgs a, int q_tiles) {
  __shared__ f32x4_t red[kProjWaves][kTokTiles][kWave];
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRowTile;
  const uint16_t* W = static_cast<const uint16_t*>(a.wq_b);
  const uint16_t* X = static_cast<const uint16_t*>(a.q_c);
  const int64_t K = a.rank;
  const int64_t tok0 = static_cast<int64_t>(blockIdx.y) * kTokPerGroup;
  const int64_t ntok = a.tokens;
  const int ntt = static_cast<int>(min<int64_t>(kTokTiles, ceil_div(ntok - tok0, 16)));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;

  f32x4_t acc[kTokTiles];
#pragma unroll
  for (int tt = 0; tt < kTokTiles; ++tt) acc[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // Step s of a chunk covers K [32s, 32s+32); lane group g takes its 8
  // values at 8g (the MFMA operand layout), so one load instruction reads 64
  // contiguous bytes of each of 16 rows.  The next chunk's weight rows are
  // loaded before the current chunk's MFMAs.
  const int64_t chunks = K / kKChunk;
  const u32x4_t* wrow = reinterpret_cast<const u32x4_t*>(W + (row0 + r) * K + g * 8);
  u32x4_t wa[kSteps];
  if (wave < chunks) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) wa[s] = wrow[(wave * kKChunk + 32 * s) / 8];
  }
  // The token group's head weights ride along while those loads are in
  // flight: dot product j of the group (token tok0 + j / heads, head
  // j % heads) belongs to wave (j / q_tiles) % 8 of workgroup j % q_tiles.
  if (a.w_proj != nullptr) {
    const int64_t dots = min<int64_t>(kTokPerGroup, ntok - tok0) * a.heads;
    for (int64_t j = static_cast<int64_t>(wave) * q_tiles + blockIdx.x; j < dots;
         j += static_cast<int64_t>(kProjWaves) * q_tiles)
      head_weight<T>(a, tok0 + j / a.heads, j % a.heads, lane);
  }
  for (int64_t c = wave; c < chunks; c += kProjWaves) {
    const int64_t k0 = c * kKChunk + g * 8;
    u32x4_t xb[kTokTiles][kSteps];
#pragma unroll
    for (int tt = 0; tt < kTokTiles; ++tt) {
      if (tt >= ntt) break;  // uniform
      const int64_t t = tok0 + tt * 16 + r;
      const bool valid = t < ntok;
      const u32x4_t* xp = reinterpret_cast<const u32x4_t*>(X + (valid ? t : ntok - 1) * K + k0);
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const u32x4_t v = xp[4 * s];
        xb[tt][s] = valid ? v : u32x4_t{0u, 0u, 0u, 0u};
      }
    }
    u32x4_t wn[kSteps];
    const int64_t cn = c + kProjWaves;
    if (cn < chunks) {
#pragma unroll
      for (int s = 0; s < kSteps; ++s) wn[s] = wrow[(cn * kKChunk + 32 * s) / 8];
    }
#pragma unroll
    for (int tt = 0; tt < kTokTiles; ++tt) {
      if (tt >= ntt) break;
#pragma unroll
      for (int s = 0; s < kSteps; ++s)
        acc[tt] = T::mfma16(__builtin_bit_cast(typename T::vec8, wa[s]), __builtin_bit_cast(typename T::vec8, xb[tt][s]),
                            acc[tt]);
    }
#pragma unroll
    for (int s = 0; s < kSteps; ++s) wa[s] = wn[s];
  }
#pragma unroll
  for (int tt = 0; tt < kTokTiles; ++tt) red[wave][tt][lane] = acc[tt];
  __syncthreads();

  // One (even, odd) output-row pair of one token per thread.  Lane l of a
  // wave held rows 4(l>>4) .. +3 of token l&15 of each 16-token tile.
  const int p = threadIdx.x & 7;      // row pair within the tile
  const int tl = threadIdx.x >> 3;    // token within the group (0..63)
  const int64_t t = tok0 + tl;
  if (t >= ntok) return;
  const int rho = 2 * p;              // even row
  const int tt = tl >> 4;
  const int src_lane = (rho >> 2) * 16 + (tl & 15);
  float v0 = 0.f, v1 = 0.f;
#pragma unroll
  for (int w = 0; w < kProjWaves; ++w) {  // fixed order: deterministic sums
    const f32x4_t x = red[w][tt][src_lane];
    v0 += x[rho & 3];
    v1 += x[(rho & 3) + 1];
  }
  const int64_t n = row0 + rho;  // output column of the even row
  uint16_t o0 = T::from_float(v0), o1 = T::from_float(v1);
  const int64_t d = n % a.head_dim;
  if (d < a.rope_dim) {
    const uint32_t c2 = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(a.cos) + t * a.cos_stride + d);
    const uint32_t s2 = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(a.sin) + t * a.cos_stride + d);
    float y0, y1;
    rope_pair(T::to_float(o0), T::to_float(o1), T::to_float(static_cast<uint16_t>(c2)),
              T::to_float(static_cast<uint16_t>(c2 >> 16)), T::to_float(static_cast<uint16_t>(s2)),
              T::to_float(static_cast<uint16_t>(s2 >> 16)), y0, y1);
    o0 = T::from_float(y0);
    o1 = T::from_float(y1);
  }
  *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(a.q_out) + t * a.heads * a.head_dim + n) =
      static_cast<uint32_t>(o0) | (static_cast<uint32_t>(o1) << 16);
}

// ---------------------------------------------------------------------------
// The q projection of many tokens (a prompt, a large batch): a tiled GEMM with
// the rotation in its epilogue.  The 64-token groups above re-read wq_b for
// every group and multiply out of registers that each MFMA waits to be
// loaded; from a few hundred tokens on the product itself is the work.
//
// A workgroup owns TOK tokens x OUT weight rows.  Both tiles go through LDS in
// K steps of 64 (128-byte rows of eight 16-byte chunks, chunk c of row r kept
// at c ^ (r & 7): the operand reads of eight consecutive rows touch all
// banks), two buffers: the next step's loads are issued before this step's
// MFMAs and stored after them, one barrier per step.  At 4096 tokens a step of
// a 256 x 256 tile takes 1.7 us (4.1k cycles, half of them MFMA): its 64 KB
// arrive at the ~16 bytes per clock that one CU pulls, whatever the order of
// loads, stores and MFMAs in it (five orders within 3%).  Wave tiles are
// TOK/WT x OUT/WO of 32x32x16 MFMAs, the weight rows as the A operand, so a
// lane holds runs of four consecutive outputs of one token (the rotation's
// pairs).  The rotated 16-bit tile is turned through LDS and stored in whole
// 16-byte chunks of a token's row (words where the output is not 16-byte
// aligned).
constexpr int kGemmK = 64;
constexpr int kGemmChunks = kGemmK / 8;

template <int TOK, int OUT, int WT, int WO>
struct GemmShape {
  static constexpr int kThreads = 64 * WT * WO;
  static constexpr int kTokW = TOK / WT, kOutW = OUT / WO;     // wave tile
  static constexpr int kTT = kTokW / 32, kOT = kOutW / 32;     // its 32x32 tiles
  static constexpr int kXLoads = TOK * kGemmChunks / kThreads;  // 16-byte chunks per thread and K step
  static constexpr int kWLoads = OUT * kGemmChunks / kThreads;
  static constexpr int kBuf = (TOK + OUT) * kGemmK;             // elements of one buffer
  static constexpr int kOutStride = OUT + 8;                    // epilogue row, elements
  static constexpr int kLds = 2 * kBuf > TOK * kOutStride ? 2 * kBuf : TOK * kOutStride;
  static_assert(TOK * kGemmChunks % kThreads == 0 && OUT * kGemmChunks % kThreads == 0 && kTokW % 32 == 0 &&
                kOutW % 32 == 0, "GEMM tiling");
};

template <typename T, int TOK, int OUT, int WT, int WO>
__global__ __launch_bounds__(64 * WT * WO) void indexer_project_gemm_kernel(IndexerArgs a, int tok_tiles,
                                                                            int out_tiles) {
  using S = GemmShape<TOK, OUT, WT, WO>;
  __shared__ __align__(16) uint16_t lds[S::kLds];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int grp = lane >> 5;
  const int wt = wave / WO, wo = wave % WO;

  // Workgroup -> tile, XCD by XCD (the dispatcher deals ids to the 8 XCDs in
  // turn): each XCD takes a contiguous run of tiles, ordered in bands of
  // kBand token tiles, so the tiles an XCD runs together share both operands
  // in its L2.
  constexpr int kBand = 4;
  const int ntiles = tok_tiles * out_tiles;
  int p = blockIdx.x;
  {
    const int base = ntiles >> 3, extra = ntiles & 7, x = p & 7;
    p = x * base + min(x, extra) + (p >> 3);
  }
  const int band = p / (kBand * out_tiles);
  const int band_rows = min(kBand, tok_tiles - band * kBand);
  const int q = p - band * kBand * out_tiles;
  const int tok0 = (band * kBand + q % band_rows) * TOK;
  const int out0 = q / band_rows * OUT;

  const int K = static_cast<int>(a.rank);
  const int ntok = static_cast<int>(a.tokens);
  // Thread's chunk of each load round: row tid / 8 (+ rounds), chunk tid % 8.
  const int lrow = tid >> 3, lch = tid & 7;
  constexpr int kRound = S::kThreads / kGemmChunks;
  const u32x4_t* xsrc[S::kXLoads];
  const u32x4_t* wsrc[S::kWLoads];
#pragma unroll
  for (int j = 0; j < S::kXLoads; ++j) {  // tokens past the last reread it (their results are not stored)
    const int t = min(tok0 + lrow + j * kRound, ntok - 1);
    xsrc[j] = reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.q_c) + static_cast<int64_t>(t) * K) + lch;
  }
#pragma unroll
  for (int j = 0; j < S::kWLoads; ++j)
    wsrc[j] = reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.wq_b) +
                                               static_cast<int64_t>(out0 + lrow + j * kRound) * K) + lch;
  const int lpos = lrow * kGemmK + ((lch ^ (lrow & 7)) * 8);  // (kRound is a multiple of 8: the same swizzle every round)
  static_assert(kRound % 8 == 0, "swizzle");

  u32x4_t xv[S::kXLoads], wv[S::kWLoads];
  auto load = [&](int step) {
#pragma unroll
    for (int j = 0; j < S::kXLoads; ++j) xv[j] = xsrc[j][step * kGemmChunks];
#pragma unroll
    for (int j = 0; j < S::kWLoads; ++j) wv[j] = wsrc[j][step * kGemmChunks];
  };
  auto store = [&](uint16_t* buf) {
#pragma unroll
    for (int j = 0; j < S::kXLoads; ++j) *reinterpret_cast<u32x4_t*>(&buf[lpos + j * kRound * kGemmK]) = xv[j];
#pragma unroll
    for (int j = 0; j < S::kWLoads; ++j)
      *reinterpret_cast<u32x4_t*>(&buf[TOK * kGemmK + lpos + j * kRound * kGemmK]) = wv[j];
  };

  f32x16_t acc[S::kOT][S::kTT];
#pragma unroll
  for (int i = 0; i < S::kOT; ++i)
#pragma unroll
    for (int j = 0; j < S::kTT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int steps = K / kGemmK;
  load(0);
  store(lds);
  load(min(1, steps - 1));
  lds_barrier();
  const int xrow = (wt * S::kTokW + l32) * kGemmK;
  const int wrow = TOK * kGemmK + (wo * S::kOutW + l32) * kGemmK;
  typename T::vec8 wf[2][S::kOT], xf[2][S::kTT];
  auto read = [&](const uint16_t* buf, int kk, int set) {
    const int ch = ((2 * kk + grp) ^ (l32 & 7)) * 8;
#pragma unroll
    for (int i = 0; i < S::kOT; ++i)
      wf[set][i] = *reinterpret_cast<const typename T::vec8*>(&buf[wrow + i * 32 * kGemmK + ch]);
#pragma unroll
    for (int j = 0; j < S::kTT; ++j)
      xf[set][j] = *reinterpret_cast<const typename T::vec8*>(&buf[xrow + j * 32 * kGemmK + ch]);
  };
  read(lds, 0, 0);
  for (int s = 0; s < steps; ++s) {
    const uint16_t* cur = lds + (s & 1) * S::kBuf;
    uint16_t* next = lds + ((s + 1) & 1) * S::kBuf;
#pragma unroll
    for (int kk = 0; kk < kGemmK / 16; ++kk) {
      if (kk + 1 < kGemmK / 16) read(cur, kk + 1, (kk + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < S::kOT; ++i)
#pragma unroll
        for (int j = 0; j < S::kTT; ++j) acc[i][j] = T::mfma32(wf[kk & 1][i], xf[kk & 1][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      if (kk == 1) {
        store(next);
        load(min(s + 2, steps - 1));  // (the last steps reload the last tile: no branch in the loop)
      }
    }
    lds_barrier();  // the next buffer is stored; this one is free (loads in flight stay in flight)
    read(next, 0, 0);
  }

  // The products rounded to 16 bits, through LDS: element e of a 32x32 tile is
  // output row 8 (e >> 2) + 4 grp + (e & 3) of token l32.
#pragma unroll
  for (int j = 0; j < S::kTT; ++j)
#pragma unroll
    for (int i = 0; i < S::kOT; ++i)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4)
        *reinterpret_cast<uint2*>(&lds[(wt * S::kTokW + j * 32 + l32) * S::kOutStride + wo * S::kOutW + i * 32 +
                                       8 * g4 + 4 * grp]) =
            make_uint2(T::pack2(acc[i][j][4 * g4], acc[i][j][4 * g4 + 1]),
                       T::pack2(acc[i][j][4 * g4 + 2], acc[i][j][4 * g4 + 3]));
  __syncthreads();
  // Then rotated and stored by 16-byte chunks (eight outputs of one token,
  // within one head).  A rolled loop: unrolled over the accumulators the
  // rotation is tens of KB of straight-line code, and fetching it cost more
  // than running it (30 us of a launch of 256 x 256 tiles).
  constexpr int kRowChunks = OUT / 8;
  const int head_dim = static_cast<int>(a.head_dim), rope = static_cast<int>(a.rope_dim);
  const int64_t row_elems = a.heads * a.head_dim;
  // Batches of kBatch chunks per thread, every cos and sin load of a batch in
  // flight together, 16 bytes each where the rows allow it (one chunk at a
  // time the loop is a chain of round trips: 7 of 76 us at 4096 tokens).
  constexpr int kIters = TOK * kRowChunks / S::kThreads;
  constexpr int kBatch = kIters < 4 ? kIters : 4;
  static_assert(TOK * kRowChunks % S::kThreads == 0 && kIters % kBatch == 0, "epilogue tiling");
  const bool out16 = (reinterpret_cast<uintptr_t>(a.q_out) & 15) == 0;  // (outputs come 4-byte aligned)
  const bool vec = (a.cos_stride & 7) == 0 && ((reinterpret_cast<uintptr_t>(a.cos) | reinterpret_cast<uintptr_t>(a.sin)) & 15) == 0;
#pragma unroll 1
  for (int c0 = 0; c0 < kIters; c0 += kBatch) {
    u32x4_t v[kBatch], cv[kBatch], sv[kBatch];
    int64_t t[kBatch];
    int d[kBatch];
    const int ch = tid % kRowChunks;  // (kThreads is a multiple of kRowChunks: the same chunk of every row)
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int r = ((c0 + i) * S::kThreads + tid) / kRowChunks;
      t[i] = tok0 + r;
      d[i] = (out0 + ch * 8) % head_dim;
      v[i] = *reinterpret_cast<const u32x4_t*>(&lds[r * S::kOutStride + ch * 8]);
      const int64_t at = min<int64_t>(t[i], ntok - 1) * a.cos_stride + d[i];
      const uint16_t* cp = static_cast<const uint16_t*>(a.cos) + at;
      const uint16_t* sp = static_cast<const uint16_t*>(a.sin) + at;
      if (vec && d[i] + 8 <= rope) {
        cv[i] = *reinterpret_cast<const u32x4_t*>(cp);
        sv[i] = *reinterpret_cast<const u32x4_t*>(sp);
      } else {
#pragma unroll
        for (int h = 0; h < 4; ++h)
          if (d[i] + 2 * h < rope) {
            cv[i][h] = reinterpret_cast<const uint32_t*>(cp)[h];
            sv[i][h] = reinterpret_cast<const uint32_t*>(sp)[h];
          }
      }
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        if (d[i] + 2 * h < rope) {
          const uint32_t x2 = v[i][h], c2 = cv[i][h], s2 = sv[i][h];
          float y0, y1;
          rope_pair(T::to_float(static_cast<uint16_t>(x2)), T::to_float(static_cast<uint16_t>(x2 >> 16)),
                    T::to_float(static_cast<uint16_t>(c2)), T::to_float(static_cast<uint16_t>(c2 >> 16)),
                    T::to_float(static_cast<uint16_t>(s2)), T::to_float(static_cast<uint16_t>(s2 >> 16)), y0, y1);
          v[i][h] = T::pack2(y0, y1);
        }
      }
      if (t[i] < ntok) {
        uint16_t* out = static_cast<uint16_t*>(a.q_out) + t[i] * row_elems + out0 + ch * 8;
        if (out16) {
          *reinterpret_cast<u32x4_t*>(out) = v[i];
        } else {
#pragma unroll
          for (int h = 0; h < 4; ++h) reinterpret_cast<uint32_t*>(out)[h] = v[i][h];
        }
      }
    }
  }
}

template <typename T, int TOK, int OUT, int WT, int WO>
void launch_gemm_shape(const IndexerArgs& a, hipStream_t stream) {
  const int tt = static_cast<int>(ceil_div(a.tokens, TOK)), ot = static_cast<int>(a.heads * a.head_dim / OUT);
  launch_kernel(kKernIdxProject, indexer_project_gemm_kernel<T, TOK, OUT, WT, WO>, dim3(static_cast<uint32_t>(tt * ot)),
                dim3(GemmShape<TOK, OUT, WT, WO>::kThreads), stream, a, tt, ot);
}

// ---------------------------------------------------------------------------
// The products of hidden_states that go with many tokens: the index key
// k = hidden . wk^T (128 wide, 16-bit) and the head weights hidden . w_proj^T
// (w_proj in fp32, or 16-bit).  Both read hidden_states, the only large
// operand, so one kernel reads it once: a workgroup owns 128 tokens x every
// column x one slice of hidden_size (split so that about one workgroup per CU
// runs), through LDS as above.  Everything runs on 32x32x16 16-bit MFMAs.  An
// fp32 head weight is cut into three bf16 parts by truncation, 8 mantissa bits
// each, which hold it exactly (an fp16 activation likewise into two), so every
// product is exact and only the fp32 sums round, as in an fp32 GEMM; sums that
// an infinity makes NaN are taken again by the finish kernel.  (On the
// fp32 MFMA, at 1/16 of the rate, the kernel takes 33 us at 4096 tokens, this
// form 28.6 us, both 2.0e-3 off fp64 in the rounded outputs.  Counters: its
// waves wait for loads or barriers 61% of their cycles and the MFMA pipes are
// busy 16% of the time; its operands arrive at 7 bytes per clock and CU, where
// the GEMM above pulls 16, so that pull is not what holds it, and which of
// the two waits does is not known.)  It replaces two library GEMMs (27 +
// 24 us), the fp32 copy of hidden_states (22 us), a layer norm, the rotation
// and six small copies and casts.  Slices leave fp32 partial sums; the finish
// kernel adds them in slice order, rounds, and does the layer norm, the
// rotation and the scale: one wave per token.
constexpr int kKwTok = 128;
constexpr int kKwThreads = 512;
constexpr int kKwDim = 128;                   // index key width
constexpr int kKwMaxSlices = 48;
constexpr int kKwParts = 3;                    // bf16 parts of a head weight

// The bf16 parts of a value, truncated: v = p0 + p1 + p2 exactly.  (Infinities
// and NaNs stay in p0.)
__device__ __forceinline__ void bf16_parts(float v, uint16_t (&p)[kKwParts]) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7f800000u) == 0x7f800000u) {
    p[0] = static_cast<uint16_t>((u >> 16) | ((u & 0x007fffffu) != 0u ? 0x40u : 0u));
    p[1] = p[2] = 0;
    return;
  }
  p[0] = static_cast<uint16_t>(u >> 16);
  const float r1 = v - __uint_as_float(u & 0xffff0000u);
  p[1] = static_cast<uint16_t>(__float_as_uint(r1) >> 16);
  const float r2 = r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
  p[2] = static_cast<uint16_t>(__float_as_uint(r2) >> 16);
}

// HT: 32-head tiles (16 heads: the upper half of the one tile is zeros).  K:
// the key columns too.
template <typename T, int HT, bool K>
__global__ __launch_bounds__(kKwThreads) void indexer_kw_kernel(IndexerKwArgs a, int slices) {
  constexpr int kRows = 32 * HT;                 // head-weight rows in LDS
  const int heads = static_cast<int>(a.heads);
  const int cols = (K ? kKwDim : 0) + heads;
  constexpr int kX = kKwTok * kGemmK, kWk = K ? kKwDim * kGemmK : 0;  // elements of one buffer
  __shared__ __align__(16) uint16_t xs[2][kX];
  __shared__ __align__(16) uint16_t wks[2][K ? kWk : 8];
  __shared__ __align__(16) uint16_t wps[2][kKwParts][kRows * kGemmK];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int slice = blockIdx.x % slices;
  const int tok0 = static_cast<int>(blockIdx.x / slices) * kKwTok;
  const int ntok = static_cast<int>(a.tokens);
  const int hid = static_cast<int>(a.hid);
  const int steps = hid / kGemmK;
  const int per = static_cast<int>(ceil_div(steps, slices));
  const int s_begin = slice * per, s_end = min(steps, s_begin + per);

  const int lrow = tid >> 3, lch = tid & 7;     // 64 rows of eight chunks per round
  constexpr int kXl = kKwTok / 64, kWl = K ? kKwDim / 64 : 0;
  const u32x4_t* xsrc[kXl];
  const u32x4_t* wsrc[kWl > 0 ? kWl : 1];
#pragma unroll
  for (int j = 0; j < kXl; ++j)
    xsrc[j] = reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.hidden) +
                                               static_cast<int64_t>(min(tok0 + lrow + 64 * j, ntok - 1)) * hid) + lch;
#pragma unroll
  for (int j = 0; j < kWl; ++j)
    wsrc[j] = reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.wk) +
                                               static_cast<int64_t>(lrow + 64 * j) * hid) + lch;
  const int lpos = lrow * kGemmK + ((lch ^ (lrow & 7)) * 8);
  // Two sets of staged loads: two K steps are in flight while one is multiplied.
  u32x4_t xv[2][kXl], wv[2][kWl > 0 ? kWl : 1], pv[2][2];
  auto load = [&](int set, int s) {
#pragma unroll
    for (int j = 0; j < kXl; ++j) xv[set][j] = xsrc[j][s * kGemmChunks];
#pragma unroll
    for (int j = 0; j < kWl; ++j) wv[set][j] = wsrc[j][s * kGemmChunks];
    // Head-weight row lrow (the kernel has at most 64), eight values.
    const int64_t at = static_cast<int64_t>(min(lrow, heads - 1)) * hid + s * kGemmK + lch * 8;
    if (a.w_fp32) {  // uniform
      const u32x4_t* p = reinterpret_cast<const u32x4_t*>(static_cast<const float*>(a.w_proj) + at);
      pv[set][0] = p[0];
      pv[set][1] = p[1];
    } else {
      pv[set][0] = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(a.w_proj) + at);
    }
  };
  auto store = [&](int set, int buf) {
#pragma unroll
    for (int j = 0; j < kXl; ++j) *reinterpret_cast<u32x4_t*>(&xs[buf][lpos + 64 * j * kGemmK]) = xv[set][j];
#pragma unroll
    for (int j = 0; j < kWl; ++j) *reinterpret_cast<u32x4_t*>(&wks[buf][lpos + 64 * j * kGemmK]) = wv[set][j];
    if (lrow < kRows) {
      u32x4_t part[kKwParts] = {};
      if (lrow < heads) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float v;
          if (a.w_fp32)
            v = __uint_as_float(pv[set][e >> 2][e & 3]);
          else
            v = T::to_float(static_cast<uint16_t>(pv[set][0][e >> 1] >> (16 * (e & 1))));
          uint16_t q[kKwParts];
          bf16_parts(v, q);
#pragma unroll
          for (int i = 0; i < kKwParts; ++i) part[i][e >> 1] |= static_cast<uint32_t>(q[i]) << (16 * (e & 1));
        }
      }
#pragma unroll
      for (int i = 0; i < kKwParts; ++i) *reinterpret_cast<u32x4_t*>(&wps[buf][i][lpos]) = part[i];
    }
  };

  // Waves 0-3: the key columns of 32 tokens each; waves 4-7: their head
  // weights (a SIMD holds one of either).
  const int l32 = lane & 31, grp = lane >> 5;
  const int wt = wave & 3;
  const bool key_wave = wave < 4;
  constexpr int kAcc = K && 4 > HT ? 4 : HT;
  f32x16_t acc[kAcc];
#pragma unroll
  for (int i = 0; i < kAcc; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  if (s_begin < s_end) {
    const int last = s_end - 1;
    load(0, s_begin);
    store(0, 0);
    load(1, min(s_begin + 1, last));
    load(0, min(s_begin + 2, last));
    lds_barrier();
    auto step = [&](int s, auto parity) {
      constexpr int cur = decltype(parity)::value;  // this step's buffer; the next one's tile is in set cur ^ 1
#pragma unroll
      for (int kk = 0; kk < kGemmK / 16; ++kk) {
        const int ch = ((2 * kk + grp) ^ (l32 & 7)) * 8;
        const u32x4_t x8 = *reinterpret_cast<const u32x4_t*>(&xs[cur][(wt * 32 + l32) * kGemmK + ch]);
        if (key_wave) {
          if constexpr (K) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              acc[i] = T::mfma32(*reinterpret_cast<const typename T::vec8*>(&wks[cur][(i * 32 + l32) * kGemmK + ch]),
                                 __builtin_bit_cast(typename T::vec8, x8), acc[i]);
          }
        } else {
          // The activations as bf16: themselves, or an fp16 value's two parts.
          constexpr int kXParts = std::is_same<T, Bf16>::value ? 1 : 2;
          u32x4_t xp[kXParts];
          if constexpr (kXParts == 1) {
            xp[0] = x8;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              uint16_t q0[kKwParts], q1[kKwParts];
              bf16_parts(T::to_float(static_cast<uint16_t>(x8[e])), q0);
              bf16_parts(T::to_float(static_cast<uint16_t>(x8[e] >> 16)), q1);
#pragma unroll
              for (int h = 0; h < kXParts; ++h) xp[h][e] = static_cast<uint32_t>(q0[h]) | (static_cast<uint32_t>(q1[h]) << 16);
            }
          }
#pragma unroll
          for (int i = 0; i < HT; ++i)
#pragma unroll
            for (int p = 0; p < kKwParts; ++p) {
              const auto wf = *reinterpret_cast<const bf16x8_t*>(&wps[cur][p][(i * 32 + l32) * kGemmK + ch]);
#pragma unroll
              for (int h = 0; h < kXParts; ++h) acc[i] = Bf16::mfma32(wf, __builtin_bit_cast(bf16x8_t, xp[h]), acc[i]);
            }
        }
      }
      store(cur ^ 1, cur ^ 1);
      load(cur ^ 1, min(s + 3, last));
      lds_barrier();
    };
    for (int s = s_begin; s < s_end; s += 2) {
      step(s, std::integral_constant<int, 0>{});
      if (s + 1 < s_end) step(s + 1, std::integral_constant<int, 1>{});
    }
  }
  // Partial sums [slice][token][column]: the key columns, then the heads.
  // (Columns from the wave's first one; heads end inside the tile at 16.)
  const int t = tok0 + wt * 32 + l32;
  if (t >= ntok || (key_wave && !K)) return;
  float* out = a.partial + (static_cast<int64_t>(slice) * ntok + t) * cols + (K && !key_wave ? kKwDim : 0);
  const int width = key_wave ? kKwDim : heads;
#pragma unroll
  for (int i = 0; i < kAcc; ++i)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int col = i * 32 + 8 * g4 + 4 * grp;
      if (col < width)
        *reinterpret_cast<float4*>(out + col) =
            make_float4(acc[i][4 * g4], acc[i][4 * g4 + 1], acc[i][4 * g4 + 2], acc[i][4 * g4 + 3]);
    }
}

// One wave per token: lane l holds key dims 2 l, 2 l + 1 (the rotation's
// pairs) and, for l < heads, head l's weight.
template <typename T, bool K>
__global__ __launch_bounds__(256) void indexer_kw_finish_kernel(IndexerKwArgs a, int slices) {
  const int lane = threadIdx.x & 63;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (t >= a.tokens) return;
  const int heads = static_cast<int>(a.heads);
  const int cols = (K ? kKwDim : 0) + heads;
  const float* p = a.partial + t * cols;
  const int64_t stride = a.tokens * cols;
  float k0 = 0.f, k1 = 0.f, w = 0.f;
#pragma unroll 4
  for (int s = 0; s < slices; ++s) {
    if constexpr (K) {
      const float2 v = *reinterpret_cast<const float2*>(p + s * stride + 2 * lane);
      k0 += v.x;
      k1 += v.y;
    }
    if (lane < heads) w += p[s * stride + (K ? kKwDim : 0) + lane];
  }
  const auto store_weight = [&](int head, float v) {
    uint16_t* out = static_cast<uint16_t*>(a.w_out) + t * heads + head;
    if (a.w_fp32) {
      *out = T::from_float(v * a.score_scale);
    } else {  // rounded after the projection and again after the scale
      uint16_t o = T::from_float(v);
      if (a.score_scale != 1.f) o = T::from_float(T::to_float(o) * a.score_scale);
      *out = o;
    }
  };
  if (lane < heads) store_weight(lane, w);
  if constexpr (K) {
    // The projection is rounded to 16 bits, then the layer norm in fp32
    // (eps 1e-6), rounded, then the rotation.
    const float x0 = T::to_float(T::from_float(k0)), x1 = T::to_float(T::from_float(k1));
    const float mean = wave_all_op(x0 + x1, AddOp{}) * (1.f / kKwDim);
    const float d0 = x0 - mean, d1 = x1 - mean;
    const float var = wave_all_op(d0 * d0 + d1 * d1, AddOp{}) * (1.f / kKwDim);
    const float rstd = 1.f / sqrtf(var + 1e-6f);
    const uint32_t gw = static_cast<const uint32_t*>(a.norm_weight)[lane];
    float y0 = d0 * rstd * T::to_float(static_cast<uint16_t>(gw));
    float y1 = d1 * rstd * T::to_float(static_cast<uint16_t>(gw >> 16));
    if (a.norm_bias != nullptr) {
      const uint32_t gb = static_cast<const uint32_t*>(a.norm_bias)[lane];
      y0 += T::to_float(static_cast<uint16_t>(gb));
      y1 += T::to_float(static_cast<uint16_t>(gb >> 16));
    }
    uint32_t o = T::pack2(y0, y1);
    if (2 * lane < a.rope_dim) {
      const uint32_t c2 = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(a.cos) + t * a.cos_stride + 2 * lane);
      const uint32_t s2 = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(a.sin) + t * a.cos_stride + 2 * lane);
      float r0, r1;
      rope_pair(T::to_float(static_cast<uint16_t>(o)), T::to_float(static_cast<uint16_t>(o >> 16)),
                T::to_float(static_cast<uint16_t>(c2)), T::to_float(static_cast<uint16_t>(c2 >> 16)),
                T::to_float(static_cast<uint16_t>(s2)), T::to_float(static_cast<uint16_t>(s2 >> 16)), r0, r1);
      o = T::pack2(r0, r1);
    }
    static_cast<uint32_t*>(a.k_out)[t * (kKwDim / 2) + lane] = o;
  }
  // An infinite operand times another's zero part is NaN where the product
  // itself is infinite: a NaN sum is taken again in whole values (a wave per
  // head; only non-finite operands or overflowing sums come here).  After the
  // stores: in front of them it cost finite inputs 4 us at 4096 tokens, here none.
  uint64_t again = __ballot(lane < heads && w != w);
  while (__builtin_expect(again != 0, 0)) {
    const int h = __ffsll(static_cast<unsigned long long>(again)) - 1;
    again &= again - 1;
    const uint16_t* x = static_cast<const uint16_t*>(a.hidden) + t * a.hid;
    const int64_t wrow = h * a.hid;
    float sum = 0.f;
#pragma unroll 1
    for (int64_t i = lane; i < a.hid; i += 64)
      sum += T::to_float(x[i]) * (a.w_fp32 ? static_cast<const float*>(a.w_proj)[wrow + i]
                                           : T::to_float(static_cast<const uint16_t*>(a.w_proj)[wrow + i]));
    sum = wave_all_op(sum, AddOp{});
    if (lane == h) store_weight(h, sum);
  }
}

// K slices of a launch: about one workgroup per CU.
int kw_slices(int64_t tokens, int64_t hid) {
  const int64_t s = std::min<int64_t>({256 / std::max<int64_t>(1, ceil_div(tokens, kKwTok)), kKwMaxSlices, hid / kGemmK});
  return static_cast<int>(std::max<int64_t>(1, s));
}

template <typename T, int HT, bool K>
hipError_t launch_kw_shape(const IndexerKwArgs& a, hipStream_t stream) {
  const int slices = kw_slices(a.tokens, a.hid);
  launch_kernel(kKernIdxKw, indexer_kw_kernel<T, HT, K>, dim3(static_cast<uint32_t>(ceil_div(a.tokens, kKwTok) * slices)),
                dim3(kKwThreads), stream, a, slices);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  launch_kernel(kKernIdxKwFinish, indexer_kw_finish_kernel<T, K>, dim3(static_cast<uint32_t>(ceil_div(a.tokens, 4))),
                dim3(256), stream, a, slices);
  return hipGetLastError();
}

template <typename T, bool K>
hipError_t launch_kw(const IndexerKwArgs& a, hipStream_t stream) {
  switch (a.heads) {
    case 16:
    case 32: return launch_kw_shape<T, 1, K>(a, stream);
    default: return launch_kw_shape<T, 2, K>(a, stream);
  }
}

// In-place RoPE of the first rope_dim dims of every [token, head] row: one
// (even, odd) pair per thread (the reference op
// dsa_indexer_query_rope_inplace, dsa_indexer_project_kernel.cpp:60-90).
template <typename T>
__global__ __launch_bounds__(256) void indexer_rope_kernel(RopeArgs a) {
  const int64_t half = a.rope_dim / 2;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.rows * half) return;
  const int64_t row = i / half;
  const int64_t d = 2 * (i - row * half);
  const int64_t t = row / a.heads;
  uint32_t* qp = reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(a.q) + row * a.head_dim + d);
  const uint32_t x2 = *qp;
  const uint32_t c2 = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(a.cos) + t * a.rope_dim + d);
  const uint32_t s2 = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(a.sin) + t * a.rope_dim + d);
  float y0, y1;
  rope_pair(T::to_float(static_cast<uint16_t>(x2)), T::to_float(static_cast<uint16_t>(x2 >> 16)),
            T::to_float(static_cast<uint16_t>(c2)), T::to_float(static_cast<uint16_t>(c2 >> 16)),
            T::to_float(static_cast<uint16_t>(s2)), T::to_float(static_cast<uint16_t>(s2 >> 16)), y0, y1);
  *qp = static_cast<uint32_t>(T::from_float(y0)) | (static_cast<uint32_t>(T::from_float(y1)) << 16);
}

template <typename T>
hipError_t launch_project(const IndexerArgs& a, hipStream_t stream) {
  const int q_tiles = static_cast<int>(a.heads * a.head_dim / kRowTile);
  if (a.w_proj == nullptr && a.tokens > kTokPerGroup) {
    // More than one 64-token group: the tiled GEMM (n_head and head_dim are
    // multiples of 16, so its output tiles divide the rows of wq_b).
    switch (indexer_gemm_tile(a.tokens, a.heads * a.head_dim)) {
      case 64: launch_gemm_shape<T, 64, 64, 2, 2>(a, stream); break;
      case 128: launch_gemm_shape<T, 128, 128, 2, 2>(a, stream); break;
      default: launch_gemm_shape<T, 256, 256, 2, 4>(a, stream);
    }
    return hipGetLastError();
  }
  const dim3 grid(static_cast<uint32_t>(q_tiles), static_cast<uint32_t>(ceil_div(a.tokens, kTokPerGroup)));
  launch_kernel(kKernIdxProject, indexer_project_kernel<T>, grid, dim3(kProjThreads), stream, a, q_tiles);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rope(const RopeArgs& a, hipStream_t stream) {
  const int64_t pairs = a.rows * (a.rope_dim / 2);
  launch_kernel(kKernIdxRope, indexer_rope_kernel<T>, dim3(static_cast<uint32_t>(ceil_div(pairs, 256))), dim3(256),
                stream, a);
  return hipGetLastError();
}

}  // namespace

int64_t indexer_k_chunk() { return kKChunk; }

// The GEMM's tile (64, 128 or 256: tokens and outputs of a workgroup) by the
// time that each would take, measured at 4096 outputs of K 2048: a launch's
// 64 x 64 tiles fill the chip's 256 CUs at 13 us and then cost 26.5 ns each,
// 128 x 128 ones 29.5 us and 75 ns, 256 x 256 ones 69 us per round of 256.
// 64-token groups / 64 / 128 / 256 tiles: 65 tokens 15.8 / 12.2 / 26 / 56 us,
// 512: 89 / 22 / 33 / 60, 1024: 174 / 34 / 29.5 / 59, 2048: 339 / 63 / 46 / 60,
// 4096: 675 / 120 / 85 / 69 us.  (Runs back to back; a trace says 74 to 78 us
// at 4096.)  K is not in the rule, which is fitted at that one: at K 256 to
// 7168, 256 to 16384 outputs and 65 to 16384 tokens the tile it takes runs in
// 0.08 to 0.94 of the groups' time.
int indexer_gemm_tile(int64_t tokens, int64_t outs) {
  const int64_t n64 = ceil_div(tokens, 64) * (outs / 64), n128 = ceil_div(tokens, 128) * (outs / 128);
  const int64_t n256 = ceil_div(tokens, 256) * (outs / 256);
  const double us64 = std::max(13.0, 7.0 + 0.0265 * n64), us128 = std::max(29.5, 8.0 + 0.075 * n128);
  const double us256 = 69.0 * ceil_div(n256, 256);
  if (us64 <= us128 && us64 <= us256) return 64;
  return us128 <= us256 ? 128 : 256;
}

hipError_t launch_indexer_project(const IndexerArgs& a, hipStream_t stream) {
  if (a.tokens == 0) return hipSuccess;
  return a.elem == Elem::kBf16 ? launch_project<Bf16>(a, stream) : launch_project<F16>(a, stream);
}

bool indexer_kw_supported(int64_t heads, int64_t hid) {
  return (heads == 16 || heads == 32 || heads == 64) && hid > 0 && hid % kGemmK == 0;
}

size_t indexer_kw_workspace_bytes(int64_t tokens, int64_t heads, int64_t hid, bool with_k) {
  return sizeof(float) * kw_slices(tokens, hid) * std::max<int64_t>(0, tokens) * ((with_k ? kKwDim : 0) + heads);
}

hipError_t launch_indexer_kw(const IndexerKwArgs& a, hipStream_t stream) {
  if (a.tokens == 0) return hipSuccess;
  if (a.wk != nullptr) return a.elem == Elem::kBf16 ? launch_kw<Bf16, true>(a, stream) : launch_kw<F16, true>(a, stream);
  return a.elem == Elem::kBf16 ? launch_kw<Bf16, false>(a, stream) : launch_kw<F16, false>(a, stream);
}

hipError_t launch_indexer_rope(const RopeArgs& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  return a.elem == Elem::kBf16 ? launch_rope<Bf16>(a, stream) : launch_rope<F16>(a, stream);
}

}  // namespace nvdsa
