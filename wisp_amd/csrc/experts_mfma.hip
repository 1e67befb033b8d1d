// Batched/prefill expert kernels on the bf16 MFMA units: a grouped GEMM over
// the slots present in the call.
//
// Replaces vLLM fused_experts for multi-token calls
// (src/wisp/integrations/vllm/fused_moe.py:1106-1118, 1155-1167); same
// arithmetic as the decode GEMV kernels:
//   act[p]  = bf16(silu(W13[s][:I] x[t]) * (W13[s][I:] x[t]))   p = (t, k)
//   y[p]    = W2[s] act[p]                                        (fp32)
//   out[t]  = bf16(sum_{k ascending} w[t,k] * y[(t, k)])
//
// Four launches (calls with many tokens per slot run 2 and 3 in block tiles,
// see there):
//   1. gather: per slot s, the ascending list of pairs routed to s and its
//      length (block-wide ballot compaction - stable, deterministic);
//   2. w13: block (i-panel of 64, slot s) streams the 64 gate rows and 64 up
//      rows of the panel once per 64 tokens of s and multiplies them against
//      those tokens, 16 per MFMA tile (v_mfma_f32_16x16x32_bf16); epilogue
//      silu(g) * u.  Both operands are staged through LDS by asynchronous
//      global->LDS copies (dma_pipeline.h);
//   3. w2: block (h-panel of 128, slot s) likewise over act, writing fp32 y;
//   4. combine: out[t] from y in routing order.
// Each output element is one MFMA dot product chain over K in a fixed order
// (ascending 32-column k-steps from a start column set by the output panel,
// wrapping around), independent of which other tokens share its tile, so a
// token's bytes do not depend on the grouping or the slot numbers: paged
// calls (split into token groups) give the same bytes as resident calls.
//
// At the Qwen3-30B-A3B shapes the expert weights are 9 MiB and a prefill
// chunk routes ~32 tokens to each expert, about 32 FLOP per weight byte: far
// below the bf16 ridge (~315 FLOP/B), so these kernels are HBM-bound and are
// built to stream each weight byte once per call.
#include <type_traits>

#include <algorithm>

#include "common.h"
#include "dma_pipeline.h"
#include "tile_pipeline.h"

namespace wisp {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kKAlign = 256;         // H and I must be multiples
constexpr int kPanel = 64;           // output columns per block: 4 waves x 16
// The LDS-staged w2 kernel's blocks own 128 output rows (4 waves x 32): a
// w2 row is only 12 chunks long at the Qwen3 shape, so per-block setup and
// the token tile weigh more than in w13, and 32 rows per wave halve both.
// Calls with enough (slot, panel) work for two rounds of blocks use 256 rows
// per block (two copy stages, two blocks per CU).
constexpr int kW2PanelsPer = 2;      // 64-row panels per LDS-staged w2 block
constexpr int kW2PanelsBig = 4;

// Work buffer carve-up (bytes, each piece 256-byte aligned).
struct WorkLayout {
  size_t lists, counts, y, total;
  WorkLayout(int P, int H, int nslots) {
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    lists = 0;
    counts = up((size_t)nslots * P * 4);
    y = counts + up((size_t)nslots * 4);
    total = y + up((size_t)P * H * 4);
  }
};

// ---------------------------------------------------------------------------
// 1. gather: lists[s * P + j] = j-th pair (ascending) with slots[p] == s, or,
// for a phase of a paged call, of the expert that slot s holds in it.
// grid = nslots; each iteration covers 8 consecutive pairs per thread and
// places the matches by a block-wide exclusive prefix of the per-thread
// counts (counts <= 8: four ballots per wave for the bits, one LDS exchange
// across the waves).  What bounds a long list is the chain of iterations, so
// the next one's pairs are loaded (16 bytes at a time where kVec) before this
// one's are placed, one barrier an iteration suffices (two sets of totals),
// and long lists take 16 waves instead of 8.  Measured with word loads and no
// look-ahead against this: 42 -> 11 us at 65536 pairs of 128 slots, 4.5 -> 2.8
// us at 4096.
// ---------------------------------------------------------------------------
constexpr int kGatherPer = 8;
constexpr int kGatherLong = 4096;  // pairs of one iteration of 8 waves

struct WholeCall {};  // no phase
struct Phase {
  const int32_t* ids;  // the pairs' experts
  PhaseTable t;
};

template <int NW, bool kVec, typename Ph>
__global__ __launch_bounds__(64 * NW) void gather_kernel(const int32_t* __restrict__ slots, int P,
                                                         int32_t* __restrict__ lists,
                                                         int32_t* __restrict__ counts, Ph phase) {
  __shared__ int wave_total[2][NW];
  const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int32_t* __restrict__ keys = slots;
  int key = s;
  if constexpr (std::is_same_v<Ph, Phase>) {
    const int e = phase.t.expert[s];
    if (e == PhaseTable::kNone) {
      if (tid == 0) counts[s] = 0;
      return;
    }
    if (e >= 0) {
      keys = phase.ids;
      key = e;
    }
  }
  int32_t* L = lists + (size_t)s * P;
  const uint64_t below = (1ull << lane) - 1ull;
  auto load = [&](int p0, int (&v)[kGatherPer]) {
    if (kVec && p0 + kGatherPer <= P) {
#pragma unroll
      for (int q = 0; q < kGatherPer; q += 4) {
        const int4 w = *reinterpret_cast<const int4*>(keys + p0 + q);
        v[q] = w.x, v[q + 1] = w.y, v[q + 2] = w.z, v[q + 3] = w.w;
      }
    } else {
#pragma unroll
      for (int q = 0; q < kGatherPer; ++q) v[q] = p0 + q < P ? keys[p0 + q] : -1;
    }
  };
  int n = 0;  // matches before this iteration (block-uniform)
  int v[kGatherPer], next[kGatherPer];
  load(tid * kGatherPer, v);
  for (int base = 0, it = 0; base < P; base += 64 * NW * kGatherPer, ++it) {
    const int p0 = base + tid * kGatherPer;
    load(p0 + 64 * NW * kGatherPer, next);
    unsigned hit = 0;
#pragma unroll
    for (int q = 0; q < kGatherPer; ++q) hit |= (unsigned)(v[q] == key) << q;
    const int c = __popc(hit);
    int pre = 0, tot = 0;
#pragma unroll
    for (int bit = 0; bit < 4; ++bit) {
      const uint64_t m = __ballot((c >> bit) & 1);
      pre += __popcll(m & below) << bit;
      tot += __popcll(m) << bit;
    }
    if (lane == 0) wave_total[it & 1][wave] = tot;
    // the totals of two iterations ago were read before the last barrier
    block_lds_sync();
    int off = n, all = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      off += w < wave ? wave_total[it & 1][w] : 0;
      all += wave_total[it & 1][w];
    }
    int o = off + pre;
#pragma unroll
    for (int q = 0; q < kGatherPer; ++q)
      if (hit >> q & 1u) L[o++] = p0 + q;
    n += all;
#pragma unroll
    for (int q = 0; q < kGatherPer; ++q) v[q] = next[q];
  }
  if (tid == 0) counts[s] = n;
}

// Where the k loop of an output panel starts.  Every block streams its rows
// chunk by chunk; when all blocks start at column 0, the reads in flight share
// their low address bits and crowd a few memory channels (a pure read of the
// Qwen3 w13 tensor in this order, non-temporal loads: 6.27 TB/s on MI355X).
// Starting each group of panels at its own multiple of 64 columns, evenly
// spread over the row, and wrapping around gives 6.99 TB/s.  The start depends
// only on the output column's group (64 columns of I in w13, 256 of H in w2),
// never on the slot, so an output's dot-product order is the same for any slot
// placement, token grouping or block size.
__device__ inline int k_rotation(unsigned group, unsigned groups, int Kdim) {
  return (int)(group * (unsigned)(Kdim / 64) / groups) * 64;
}

// The w2 kernel's rotation: by the block's 256-row group of H (NG 64-row
// panels per block, NG = 2 or 4), so that blocks of 128 and of 256 rows give
// every output row the same k order and the same bytes.
template <int NG>
__device__ inline int k_rotation_w2(int Kdim) {
  static_assert(NG == 2 || NG == 4, "64-row panels per w2 block");
  return k_rotation(blockIdx.x * NG / 4, gridDim.x * NG / 4, Kdim);
}

// Column of k-step offset k (0 <= k < Kdim) in a loop rotated by rot columns.
__device__ inline int k_col(int k, int rot, int Kdim) {
  const int c = k + rot;
  return c >= Kdim ? c - Kdim : c;
}

// ---------------------------------------------------------------------------
// w13 and w2 kernels: the chunk pipeline of dma_pipeline.h over 64-column
// (128-byte) chunks, two 32-column k-steps of MFMA per chunk, the k rotation
// of the output panel.  w13 blocks own a 64-row panel (each wave 16 gate and
// 16 up rows); w2 blocks own 128 rows (32 per wave).
// What bounds them: a pure read of the Qwen3 w13 tensor with these copies
// (non-temporal), chunk order, rotation and occupancy runs at 6.95 TB/s on
// MI355X and w13 here at 6.18 TB/s of weights; the w2 tensor reads at
// 6.45 TB/s and w2 here at 4.90 TB/s.
// ---------------------------------------------------------------------------

// The pass's GEMM over Kdim columns for mrows tokens (the pass's pair list
// held one entry per lane in `held`, dma::list_entries): acc[g][t] +=
// W(row group g) . A(token tile t)^T for the NT = ceil(mrows / 16) tiles the
// pass fills, NG row groups of 16 per wave, the k loop starting rot columns
// in.  A is the token matrix (leading dimension ld); with kTokenRows, pair p
// reads row p / K.  With the weights as the MFMA's first
// operand, lane l holds rows 4 (l / 16) + q, q < 4, of its group for token
// column l % 16: four consecutive outputs of one token, stored at once.
template <int NG, int S, bool kTokenRows>
__device__ inline void dma_gemm(unsigned char* smem,
                                const unsigned char* const (&wrow)[16 * NG / dma::kRowsPerCopy],
                                const uint16_t* __restrict__ A, int ld, int K, int held,
                                int mrows, int Kdim, int rot, bool first,
                                f32x4 (&acc)[NG][4]) {
  const int lane = threadIdx.x & 63;
  auto row_of = [&](int r) {
    const int p = dma::list_entry(held, r);
    return reinterpret_cast<const unsigned char*>(A + (size_t)(kTokenRows ? p / K : p) * ld);
  };
  auto off = [&](int c) { return (size_t)k_col(c * 64, rot, Kdim) * sizeof(uint16_t); };
  auto run = [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    dma::pass<16 * NG, S, NT>(
        smem, wrow, mrows, row_of, Kdim / 64, off,
        [&](const unsigned char* ws, const unsigned char* as, int) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int cb = u * 4 + (lane >> 4);
            bf16x8 b[NG], a[NT];
#pragma unroll
            for (int g = 0; g < NG; ++g)
              b[g] = *reinterpret_cast<const bf16x8*>(ws + dma::swz(g * 16 + (lane & 15), cb));
#pragma unroll
            for (int t = 0; t < NT; ++t)
              a[t] = *reinterpret_cast<const bf16x8*>(as + dma::swz(t * 16 + (lane & 15), cb));
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int g = 0; g < NG; ++g)
                acc[g][t] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[g], a[t], acc[g][t], 0, 0, 0);
          }
        },
        dma::NoSetup{}, first);
  };
  const int nt = (mrows + 15) >> 4;
  if (nt == 1)
    run(std::integral_constant<int, 1>{});
  else if (nt == 2)
    run(std::integral_constant<int, 2>{});
  else if (nt == 3)
    run(std::integral_constant<int, 3>{});
  else
    run(std::integral_constant<int, 4>{});
}

// The pairs of the token columns this lane stores after the pass (tile t,
// column lane % 16; columns past mrows repeat the last), from the pass's
// lane-held pair list.
__device__ inline void epilogue_pairs(int held, int mrows, int (&pr)[4]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < 4; ++t) pr[t] = dma::list_entry(held, min(t * 16 + (lane & 15), mrows - 1));
}

// bf16(silu(g) * u) of four consecutive columns, one 8-byte store at p.
__device__ inline void store_act4(uint16_t* p, const f32x4& g, const f32x4& u) {
  uint32_t h[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) h[q] = bf16_rne(silu(g[q]) * u[q]);
  *reinterpret_cast<uint2*>(p) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
}

template <int S>
__global__ __launch_bounds__(256) void mfma_w13_dma_kernel(
    const uint16_t* __restrict__ x, int H, int I, int K, int P, const int32_t* __restrict__ lists,
    const int32_t* __restrict__ counts, const uint16_t* __restrict__ w13, size_t w13_stride,
    uint16_t* __restrict__ act) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
  const int s = blockIdx.y;
  const int32_t* list = lists + (size_t)s * P;
  // the slot's count and the first pass's pair list, loaded together
  const int M = counts[s];
  int held = dma::list_entries(list, 0, P);
  if (M == 0) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i0 = blockIdx.x * kPanel + wave * 16;
  const uint16_t* W = w13 + (size_t)s * w13_stride;
  // this lane's weight copy rows: slice rows 0-15 gate, 16-31 up
  const unsigned char* wrow[32 / dma::kRowsPerCopy];
#pragma unroll
  for (int i = 0; i < 32 / dma::kRowsPerCopy; ++i) {
    const int r = i * dma::kRowsPerCopy + lane / dma::kLanesPerRow;
    wrow[i] = reinterpret_cast<const unsigned char*>(
        W + (size_t)(r < 16 ? i0 + r : I + i0 + r - 16) * H);
  }
  const int rot = k_rotation(blockIdx.x, gridDim.x, H);
  for (int m0 = 0; m0 < M; m0 += dma::kTokRows) {
    const int mrows = min(M - m0, dma::kTokRows);
    if (m0 > 0) held = dma::list_entries(list, m0, P);
    f32x4 acc[2][4];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int pr[4];
    epilogue_pairs(held, mrows, pr);
    dma_gemm<2, S, true>(dsm, wrow, x, H, K, held, mrows, H, rot, m0 == 0, acc);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (t * 16 + (lane & 15) < mrows)
        store_act4(act + (size_t)pr[t] * I + i0 + (lane >> 4) * 4, acc[0][t], acc[1][t]);
  }
}

template <int S, int NG>
__global__ __launch_bounds__(256) void mfma_w2_dma_kernel(
    const uint16_t* __restrict__ act, int H, int I, int P, const int32_t* __restrict__ lists,
    const int32_t* __restrict__ counts, const uint16_t* __restrict__ w2, size_t w2_stride,
    float* __restrict__ y) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
  const int s = blockIdx.y;
  const int32_t* list = lists + (size_t)s * P;
  // the slot's count and the first pass's pair list, loaded together
  const int M = counts[s];
  int held = dma::list_entries(list, 0, P);
  if (M == 0) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // NG row groups of 16 per wave
  const int h0 = blockIdx.x * kPanel * NG + wave * 16 * NG;
  const uint16_t* W = w2 + (size_t)s * w2_stride;
  const unsigned char* wrow[16 * NG / dma::kRowsPerCopy];
#pragma unroll
  for (int i = 0; i < 16 * NG / dma::kRowsPerCopy; ++i)
    wrow[i] = reinterpret_cast<const unsigned char*>(
        W + (size_t)(h0 + i * dma::kRowsPerCopy + lane / dma::kLanesPerRow) * I);
  const int rot = k_rotation_w2<NG>(I);
  for (int m0 = 0; m0 < M; m0 += dma::kTokRows) {
    const int mrows = min(M - m0, dma::kTokRows);
    if (m0 > 0) held = dma::list_entries(list, m0, P);
    f32x4 acc[NG][4];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int pr[4];
    epilogue_pairs(held, mrows, pr);
    dma_gemm<NG, S, false>(dsm, wrow, act, I, 1, held, mrows, I, rot, m0 == 0, acc);
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (t * 16 + (lane & 15) < mrows) {
        float* yr = y + (size_t)pr[t] * H + h0 + (lane >> 4) * 4;
#pragma unroll
        for (int g = 0; g < NG; ++g) *reinterpret_cast<f32x4*>(yr + g * 16) = acc[g][t];
      }
  }
}

// ---------------------------------------------------------------------------
// Large calls: the same two products in block tiles (tile_pipeline.h), 256
// weight rows (w13: 128 gate and 128 up rows) by up to 256 or 192 tokens,
// eight waves in persistent blocks, one per CU.  The matrix instruction and
// the k order of every output are those of the kernels above, so the bytes
// are too.
// What bounds them: at the Qwen3 8192-token chunk (512 tokens a slot) w13
// runs at 885 TFLOP/s and w2 at 637 (466 + 324 us; the 64-token blocks take
// 1322 + 790 us).  A build without the copies takes 354 + 204 us (a plain
// 8192^3 bf16 library product runs at 1209 TFLOP/s), one without the matrix
// instructions 410 + 315 us: staging 64 KB a chunk and block from L2, where
// 1 byte in 3 misses, is as long as the arithmetic and does not hide behind
// it entirely.  Measured and not better: four 64-byte stages (512 + 371 us),
// touching the lines three chunks ahead (557 + 361: the loads of a CU
// return in order), 320-token tiles (492 + 335, registers spill), 128 x 128
// tiles with two blocks per CU (545 + 351), no k rotation (447 + 329).
// These are figures of tiles whose halves started their k loops together.
// They start apart, each at its 64 columns' own place, because the 64-token
// blocks do: 2 or 3 of 32 chunks at this shape, in which one half of the waves
// has no products and its rows are not copied.  That costs w13 4 % here
// (rocprofv3: 505 -> 525 us) and 2 % at a 1000-token Mixtral chunk (585 -> 596).
// Peeling those steps off the loop, or the other assignment of waves to halves
// (both waves of a SIMD to one), changed nothing.
// ---------------------------------------------------------------------------
struct TileArgs {
  const uint16_t* A;  // token matrix: x (w13) or act (w2)
  int H, I, K, P, nslots;
  const int32_t* lists;
  const int32_t* counts;
  const uint16_t* W;
  size_t w_stride;
  void* out;
};

template <typename Sh, bool kW13>
struct TileLoop {
  static constexpr int NG = Sh::NG;
  static constexpr int kAhead = 3;  // 16-row groups a weight fragment is read ahead
  static constexpr int kRing = kAhead + 1;
  // groups of a chunk's second k-step left for after the next chunk's barrier
  static constexpr int kLeft = kAhead;
  static_assert(NG >= 4, "row groups of a wave");
  const TileArgs& a;
  unsigned char* smem;
  const tile::Table* tab;
  int N, Kdim, npanels, chunks;
  int wave, lane, wr, wt;
  uint32_t woff, wstep[Sh::kWCopies];
  // this lane's place, in a stage's weight (token) rows, of the fragment of
  // its wave's first row group (token tile) for either k-step
  int lw[2], lt[2];
  tile::Range tokens;
  int q = 0;  // chunks computed so far: chunk q lies in stage q % 2
  int j = 0;  // works taken so far
  int stored = 0;  // token tiles a wave stored of the tile before

  template <int NT>
  struct Frags {
    bf16x8 w[kRing], t[2][NT];
  };

  __device__ __attribute__((always_inline)) bool take(tile::Work* w) {
    const bool found = tile::find_work(tab, tile::work_of(blockIdx.x, j++), a.nslots, npanels, w);
    // wave-uniform by construction; the compiler sees it from here on
    w->slot = __builtin_amdgcn_readfirstlane(w->slot);
    w->panel = __builtin_amdgcn_readfirstlane(w->panel);
    w->m0 = __builtin_amdgcn_readfirstlane(w->m0);
    w->mrows = __builtin_amdgcn_readfirstlane(w->mrows);
    return __builtin_amdgcn_readfirstlane(found);
  }
  __device__ __attribute__((always_inline)) int copy_row(int i) const {
    return (i * Sh::kWaves + wave) * tile::kRowsPerCopy + lane / dma::kLanesPerRow;
  }
  // Weight row r of a panel, counted from the panel's first (gate) row.  w13:
  // each wave's rows are its gate rows, then the up rows of the same columns.
  __device__ __attribute__((always_inline)) int weight_row(int r) const {
    constexpr int half = NG * 8;
    if (!kW13) return r;
    return r / (2 * half) * half + r % half + (r % (2 * half) < half ? 0 : a.I);
  }
  // The pairs behind this lane's token copies.
  struct Pairs {
    int copy[Sh::kTCopies];
  };
  __device__ __attribute__((always_inline)) const int32_t* list(const tile::Work& w) const {
    return a.lists + (size_t)w.slot * a.P + w.m0;
  }
  __device__ __attribute__((always_inline)) void pairs(const tile::Work& w, Pairs* p) const {
    const int32_t* l = list(w);
#pragma unroll
    for (int i = 0; i < Sh::kTCopies; ++i) p->copy[i] = l[min(copy_row(i), w.mrows - 1)];
  }
  __device__ __attribute__((always_inline)) void source(const tile::Work& w, const Pairs& p,
                                                        tile::Source<Sh>* s) const {
    const int row0 = w.panel * (kW13 ? Sh::kRows / 2 : Sh::kRows);
    const uint32_t rb = (uint32_t)Kdim * 2;
    s->w = {a.W + (size_t)w.slot * a.w_stride + (size_t)row0 * Kdim, (uint32_t)(N - row0) * rb};
#pragma unroll
    for (int i = 0; i < Sh::kTCopies; ++i)
      s->toff[i] = (uint32_t)(kW13 ? p.copy[i] / a.K : p.copy[i]) * rb +
                   (((lane % dma::kLanesPerRow) ^ (copy_row(i) & 7)) << 4);
    constexpr int per = tile::kRowsPerCopy * Sh::kWaves, step = 16 * Sh::WT;
    s->tc = ((w.mrows + step - 1) / step * step + per - 1) / per;
    // a w13 panel's two halves (64 columns each) start their k loops apart
    const int half0 = kW13 ? 2 * w.panel : w.panel, halves = kW13 ? 2 * npanels : npanels;
    s->rot = k_rotation(half0, halves, Kdim) * 2;
    s->lag = kW13 ? (k_rotation(half0 + 1, halves, Kdim) * 2 - s->rot) / tile::kRowBytes : 0;
  }
  __device__ __attribute__((always_inline)) void issue(unsigned char* stage,
                                                       const tile::Source<Sh>& s, int c) const {
    // the first half's rows are not needed past its last chunk, nor the
    // second's before its first
    tile::copies<Sh>(stage, s, woff, wstep, tokens, wave, tile::chunk_byte(c, s.rot, Kdim * 2),
                     kW13 && c >= chunks ? Sh::kWCopies / 2 : 0,
                     kW13 && c < s.lag ? Sh::kWCopies / 2 : Sh::kWCopies);
  }
  template <int NT>
  __device__ __attribute__((always_inline)) void read_t(const unsigned char* stage, int u, int i,
                                                        Frags<NT>& f) const {
    f.t[u][i] = *reinterpret_cast<const bf16x8*>(
        stage + Sh::kRows * tile::kRowBytes + lt[u] + i * Sh::WT * 16 * tile::kRowBytes);
  }
  // Weight fragment n of a chunk: row group n % NG of k-step n / NG.
  template <int NT>
  __device__ __attribute__((always_inline)) void read_w(const unsigned char* stage, int n,
                                                        Frags<NT>& f) const {
    f.w[n % kRing] = *reinterpret_cast<const bf16x8*>(
        stage + lw[n / NG] + n % NG * 16 * tile::kRowBytes);
  }
  template <int NT>
  __device__ __attribute__((always_inline)) void mma(int n, const Frags<NT>& f,
                                                     f32x4 (&acc)[NG][NT]) const {
#pragma unroll
    for (int i = 0; i < NT; ++i)
      acc[n % NG][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[n % kRing], f.t[n / NG][i],
                                                               acc[n % NG][i], 0, 0, 0);
  }
  // One chunk, from stage `rds`, with the next chunk's copies into `wrs`
  // (distinct stages, see dma::step): fragment by fragment in the order of
  // the matrix instructions, each read kAhead groups before its use.  The
  // last kLeft groups of the chunk before (zeros before a tile's first) cover
  // the first reads, and this chunk's are left for the next call: all its
  // fragments are then in registers, so that its stage can be overwritten.
  // A wave that is not `active` has no products in this chunk.
  template <int NT>
  __device__ __attribute__((always_inline)) void chunk(unsigned char* __restrict__ wrs,
                                                       const unsigned char* __restrict__ rds,
                                                       const tile::Source<Sh>& cs, int cc,
                                                       bool active, Frags<NT>& f,
                                                       f32x4 (&acc)[NG][NT]) const {
    if (cc >= 0) issue(wrs, cs, cc);
    __builtin_amdgcn_sched_barrier(0);
    if (!active) return;
    // positions -kLeft .. 2 NG - kLeft - 1; before position n: token
    // fragments of the first k-step, then weight fragment n + kAhead
#pragma unroll
    for (int i = 0; i < NT; ++i) read_t<NT>(rds, 0, i, f);
#pragma unroll
    for (int n = -kLeft; n < 2 * NG - kLeft; ++n) {
      read_w<NT>(rds, n + kAhead, f);  // its place is free: group n - 1 was its last reader
      if (n >= 0 && n < NG - 1) {
#pragma unroll
        for (int i = n * NT / (NG - 1); i < (n + 1) * NT / (NG - 1); ++i)
          read_t<NT>(rds, 1, i, f);
      }
      mma<NT>(n >= 0 ? n : 2 * NG + n, f, acc);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Waits for the next chunk (this wave's copies of it) and for every wave's
  // reads of the one before.
  __device__ __attribute__((always_inline)) void wait() const {
    dma::wait_vm<0>();
    dma::lds_barrier();
  }
  // The same at a tile's first chunk, whose copies are older than the stores
  // of the tile before: those need not be waited for.  Every wave of a tile
  // with n token tiles a wave makes exactly n * kStores of them.
  static constexpr int kStores = kW13 ? NG / 2 : NG;
  template <int N = Sh::NT>
  __device__ __attribute__((always_inline)) void wait_first() const {
    if constexpr (N > 0) {
      if (stored != N) return wait_first<N - 1>();
    }
    dma::wait_vm<N * kStores>();
    dma::lds_barrier();
  }
  template <int NT>
  __device__ __attribute__((always_inline)) void next_chunk(const tile::Source<Sh>& cs, int cc,
                                                            bool active, Frags<NT>& f,
                                                            f32x4 (&acc)[NG][NT]) {
    chunk<NT>(smem + (~q & 1) * Sh::kStage, smem + (q & 1) * Sh::kStage, cs, cc, active, f, acc);
    ++q;
  }

  // One tile.  On entry the copies of its first chunk are issued; on return
  // those of the next tile's are, if any.  Its chunks + lag chunks start at
  // the first half's k rotation; the waves of the second half pass the first
  // `lag` of them, where their own rotation has not begun, and those of the
  // first half the last `lag`, which are past their end.
  template <int NT>
  __device__ __attribute__((always_inline)) void run(tile::Work& w, tile::Source<Sh>& src,
                                                     bool* more) {
    f32x4 acc[NG][NT];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    Frags<NT> f;
#pragma unroll
    for (int n = 2 * NG - kLeft; n < 2 * NG; ++n) f.w[n % kRing] = bf16x8{};
#pragma unroll
    for (int t = 0; t < NT; ++t) f.t[1][t] = bf16x8{};
    int pr[NT];
    Pairs np;
    tile::Work nw;
    tile::Source<Sh> ns;
    // The next tile's place and token rows are read behind the first chunk,
    // so that they are there without a wait when its copies start.
    wait_first();
    const bool next = take(&nw);
    if (next) pairs(nw, &np);
#pragma unroll
    for (int t = 0; t < NT; ++t)
      pr[t] = list(w)[min((t * Sh::WT + wt) * 16 + (lane & 15), w.mrows - 1)];
    const int lag = kW13 ? __builtin_amdgcn_readfirstlane(src.lag) : 0;
    const int begin = wr < Sh::WR / 2 ? 0 : lag, steps = chunks + lag;
    for (int c = 0; c < steps - 1; ++c) {
      next_chunk<NT>(src, c + 1, !kW13 || (c >= begin && c < begin + chunks), f, acc);
      wait();
    }
    if (next) source(nw, np, &ns);
    next_chunk<NT>(ns, next ? 0 : -1, begin == lag, f, acc);
#pragma unroll
    for (int n = 2 * NG - kLeft; n < 2 * NG; ++n) mma<NT>(n, f, acc);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      // columns past mrows hold, and store again, the last token's values
      if constexpr (kW13) {
        uint16_t* ar = (uint16_t*)a.out + (size_t)pr[t] * a.I + w.panel * (Sh::kRows / 2) +
                       wr * NG * 8 + (lane >> 4) * 4;
#pragma unroll
        for (int g = 0; g < NG / 2; ++g) {
          store_act4(ar + g * 16, acc[g][t], acc[g + NG / 2][t]);
          __builtin_amdgcn_sched_barrier(0);  // one store's temporaries at a time
        }
      } else {
        float* yr = (float*)a.out + (size_t)pr[t] * a.H + w.panel * Sh::kRows + wr * NG * 16 +
                    (lane >> 4) * 4;
#pragma unroll
        for (int g = 0; g < NG; ++g) *reinterpret_cast<f32x4*>(yr + g * 16) = acc[g][t];
      }
    }
    stored = NT;
    w = nw;
    src = ns;
    *more = next;
  }
};

template <typename Sh, bool kW13>
__global__ __launch_bounds__(64 * Sh::kWaves)
__attribute__((amdgpu_waves_per_eu(Sh::kWaves / 4, Sh::kWaves / 4))) void mfma_tile_kernel(
    TileArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char dsm[];
  tile::Table* tab = reinterpret_cast<tile::Table*>(dsm + Sh::kTable);
  TileLoop<Sh, kW13> L{a, dsm, tab};
  L.N = kW13 ? 2 * a.I : a.H;
  L.Kdim = kW13 ? a.H : a.I;
  L.npanels = L.N / Sh::kRows;
  L.chunks = L.Kdim * 2 / tile::kRowBytes;
  L.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  L.lane = threadIdx.x & 63;
  // (waves w and w + 4 share a SIMD: one of each half of the rows)
  static_assert(Sh::kWaves == 8 && Sh::WR % 2 == 0, "halves of the rows over the SIMDs");
  L.wr = L.wave / Sh::WT;
  L.wt = L.wave % Sh::WT;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    L.lw[u] = dma::swz(L.wr * Sh::NG * 16 + (L.lane & 15), u * 4 + (L.lane >> 4));
    L.lt[u] = dma::swz(L.wt * 16 + (L.lane & 15), u * 4 + (L.lane >> 4));
  }
  L.tokens = {a.A, (uint32_t)(kW13 ? a.P / a.K : a.P) * (uint32_t)(L.Kdim * 2)};
  // weight_row(64 i + r) is weight_row(64 i) + weight_row(r) for r < 64
  static_assert(Sh::kWaves * tile::kRowsPerCopy == 64 && Sh::NG % 4 == 0, "rows of a copy step");
  L.woff = (uint32_t)L.weight_row(L.copy_row(0)) * (uint32_t)(L.Kdim * 2) +
           (((L.lane % dma::kLanesPerRow) ^ (L.copy_row(0) & 7)) << 4);
#pragma unroll
  for (int i = 0; i < Sh::kWCopies; ++i)
    L.wstep[i] =
        (uint32_t)L.weight_row(i * Sh::kWaves * tile::kRowsPerCopy) * (uint32_t)(L.Kdim * 2);
  if (L.wave == 0) tile::fill_table(tab, a.counts, a.nslots, Sh::kToks);
  __syncthreads();
  tile::Work w;
  bool more = L.take(&w);
  if (!more) return;
  tile::Source<Sh> src;
  {
    typename TileLoop<Sh, kW13>::Pairs p;
    L.pairs(w, &p);
    L.source(w, p, &src);
  }
  L.issue(dsm, src, 0);
  while (more) {
    const int nt = (w.mrows + 16 * Sh::WT - 1) / (16 * Sh::WT);
    if (nt == 1)
      L.template run<1>(w, src, &more);
    else if (nt == 2)
      L.template run<2>(w, src, &more);
    else if (nt == 3)
      L.template run<3>(w, src, &more);
    else if (Sh::NT == 4 || nt == 4)
      L.template run<4>(w, src, &more);
    else if (nt == 5)
      L.template run<(Sh::NT > 4 ? 5 : 4)>(w, src, &more);
    else
      L.template run<(Sh::NT > 4 ? 6 : 4)>(w, src, &more);
  }
}

// ---------------------------------------------------------------------------
// 4. combine: out[t, h] = bf16(sum_k w[t,k] * y[(t,k), h]), k ascending,
// skipping pairs without a slot (their y rows are never written: selected
// out, not multiplied by zero).  8 columns per thread, every k's slot,
// weight and y loads issued before the sums.  A y of more than the last-level
// cache is read non-temporally (kStream), a smaller one comes from that cache.
// Measured at the Qwen3 shape, default against non-temporal loads (us): 9.1 /
// 9.9 at 768 tokens (50 MB), 14.4 / 15.8 at 1024, 23.0 / 26.2 at 2048, 49.1 /
// 49.9 at 4096 (268 MB), 119.5 / 99.0 at 8192.
// grid = (ceil(H / 2048), T).
// ---------------------------------------------------------------------------
constexpr int kCombineK = 16;  // top-k handled with all loads up front; more loop
constexpr size_t kCombineStream = 256ull << 20;  // bytes of y

template <bool kVecStore, bool kStream>
__global__ __launch_bounds__(256) void combine_kernel(const float* __restrict__ y, int H, int K,
                                                     int nslots, const float* __restrict__ topk_w,
                                                     const int32_t* __restrict__ slots,
                                                     uint16_t* __restrict__ out) {
  const int t = blockIdx.y;
  const int h = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (h >= H) return;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += kCombineK) {
    const int kn = min(K - k0, kCombineK);
    f32x4 lo[kCombineK], hi[kCombineK];
    float w[kCombineK];
    bool ok[kCombineK];
#pragma unroll
    for (int k = 0; k < kCombineK; ++k) {
      if (k < kn) {
        const int p = t * K + k0 + k;
        const int sl = slots[p];
        ok[k] = sl >= 0 && sl < nslots;
        w[k] = topk_w[p];
        const f32x4* yr = reinterpret_cast<const f32x4*>(y + (size_t)p * H + h);
        lo[k] = kStream ? __builtin_nontemporal_load(yr) : yr[0];
        hi[k] = kStream ? __builtin_nontemporal_load(yr + 1) : yr[1];
      }
    }
#pragma unroll
    for (int k = 0; k < kCombineK; ++k) {
      if (k < kn && ok[k]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[j] = fmaf(w[k], lo[k][j], acc[j]);
          acc[4 + j] = fmaf(w[k], hi[k][j], acc[4 + j]);
        }
      }
    }
  }
  uint16_t* o = out + (size_t)t * H + h;
  if constexpr (kVecStore) {
    u32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = (uint32_t)bf16_rne(acc[2 * j]) | ((uint32_t)bf16_rne(acc[2 * j + 1]) << 16);
    *reinterpret_cast<u32x4*>(o) = v;
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = bf16_rne(acc[j]);
  }
}

void launch_combine(const float* y, int T, int H, int K, int nslots, const float* topk_w,
                    const int32_t* slots, uint16_t* out, hipStream_t st) {
  const dim3 grid((H + 2047) / 2048, T);
  auto go = [&](auto* kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, y, H, K, nslots, topk_w, slots, out);
  };
  const bool vec = ((uintptr_t)out | ((size_t)H * 2)) % 16 == 0;
  if ((size_t)T * K * H * 4 >= kCombineStream)
    vec ? go(&combine_kernel<true, true>) : go(&combine_kernel<false, true>);
  else
    vec ? go(&combine_kernel<true, false>) : go(&combine_kernel<false, false>);
}

template <int S2, int NG>
hipError_t launch_w2_dma(const uint16_t* act, int H, int I, int P, int nslots,
                         const int32_t* lists, const int32_t* counts, const uint16_t* w2,
                         size_t w2_stride, float* y, hipStream_t st, hipEvent_t e2,
                         hipEvent_t e3) {
  constexpr unsigned b2 = dma::Smem<16 * NG, S2>::kBytes;
  static_assert(b2 <= 160 * 1024, "LDS per block");
  static std::atomic<uint64_t> big2{0};
  hipError_t e = allow_lds(&mfma_w2_dma_kernel<S2, NG>, b2, b2, &big2);
  if (e != hipSuccess) return e;
  launch_timed_lds(mfma_w2_dma_kernel<S2, NG>, dim3(H / (kPanel * NG), nslots), dim3(256), b2,
                   st, e2, e3, act, H, I, P, lists, counts, w2, w2_stride, y);
  return hipSuccess;
}

template <int S13>
hipError_t launch_dma(const uint16_t* x, int H, int I, int K, int P, int nslots,
                      const int32_t* lists, const int32_t* counts, const uint16_t* w13,
                      size_t w13_stride, const uint16_t* w2, size_t w2_stride, uint16_t* act,
                      float* y, hipStream_t st, const StageEvents* ev) {
  constexpr unsigned b13 = dma::Smem<32, S13>::kBytes;
  static_assert(b13 <= 160 * 1024, "LDS per block");
  static std::atomic<uint64_t> big13{0};
  hipError_t e = allow_lds(&mfma_w13_dma_kernel<S13>, b13, b13, &big13);
  if (e != hipSuccess) return e;
  hipEvent_t e0 = ev ? ev->ev[0] : nullptr, e1 = ev ? ev->ev[1] : nullptr;
  hipEvent_t e2 = ev ? ev->ev[2] : nullptr, e3 = ev ? ev->ev[3] : nullptr;
  launch_timed_lds(mfma_w13_dma_kernel<S13>, dim3(I / kPanel, nslots), dim3(256), b13, st, e0,
                   e1, x, H, I, K, P, lists, counts, w13, w13_stride, act);
  // 256-row w2 blocks (two stages) when the call's slots could give two
  // blocks per CU of them; else 128-row blocks (three stages).  Measured at
  // the Qwen3 512-token chunk: 83 against 89 us; the smaller blocks keep
  // calls with few slots (Mixtral, paged token groups) spread over the GPU.
  const int64_t busy = (int64_t)std::min(P, nslots) * (H / (kPanel * kW2PanelsBig));
  return busy >= 512 ? launch_w2_dma<2, kW2PanelsBig>(act, H, I, P, nslots, lists, counts, w2,
                                                      w2_stride, y, st, e2, e3)
                     : launch_w2_dma<3, kW2PanelsPer>(act, H, I, P, nslots, lists, counts, w2,
                                                      w2_stride, y, st, e2, e3);
}

template <typename Sh, bool kW13>
hipError_t launch_tile(const TileArgs& a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  constexpr unsigned lds = Sh::kTable + sizeof(tile::Table);
  static_assert(lds <= 160 * 1024, "LDS per block");
  static std::atomic<uint64_t> big{0};
  hipError_t e = allow_lds(&mfma_tile_kernel<Sh, kW13>, lds, lds, &big);
  if (e != hipSuccess) return e;
  launch_timed_lds(mfma_tile_kernel<Sh, kW13>, dim3(tile::kBlocks), dim3(64 * Sh::kWaves), lds, st,
                   e0, e1, a);
  return hipSuccess;
}

// Tiles of 256 tokens, unless they would leave CUs idle (one block per CU):
// then tiles of 192, which split the larger slots.  Measured at the Mixtral
// 1000-token chunk's w2 (8 slots of ~250 tokens, 16 panels): 392 against
// 341 us; at the Qwen3 8192-token chunk (128 slots of ~512, 8 panels) 324
// against 342 us, and its w13 466 against 509 us (before the halves of a w13
// tile started apart).
template <bool kW13>
hipError_t launch_tiles(const TileArgs& a, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  using Big = tile::Shape<2, 4, 8, 4>;
  using Small = tile::Shape<4, 2, 4, 6>;
  const int busy = std::min(a.P, a.nslots);
  const int64_t works = (int64_t)((kW13 ? 2 * a.I : a.H) / Big::kRows) * busy *
                        ((a.P / busy + Big::kToks - 1) / Big::kToks);
  return works >= tile::kBlocks ? launch_tile<Big, kW13>(a, st, e0, e1)
                              : launch_tile<Small, kW13>(a, st, e0, e1);
}

// Calls of at least this many pairs per slot take the block tiles.  The
// 64-token blocks stream a slot's weights once per 64 of its tokens, so their
// time steps up where slots start to need a second pass, while the tiles'
// hardly grows with the tokens until the matrix cores bound it.  Measured,
// 64-token blocks against tiles, w13 + w2 (us): Qwen3 48 / 64 / 96 / 128
// pairs per slot 254 / 362 / 458 / 617 against 266 / 285 / 303 / 317;
// Mixtral 50 / 64 / 100 / 250 508 / 728 / 981 / 2236 against
// 665 / 692 / 738 / 881.
constexpr int kTileMinPairs = 60;

// Whether a call takes the block tiles (their 32-bit row offsets must reach
// every byte of x, act and one expert's weights, and their buffer loads want
// 16-byte aligned rows).
bool tile_call(int P, int H, int I, int nslots, int spread, int T, uintptr_t addresses) {
  const uint64_t lim = 1ull << 32;
  return addresses % 16 == 0 && (int64_t)P >= (int64_t)kTileMinPairs * spread &&
         (uint64_t)T * H * 2 < lim &&
         (uint64_t)P * I * 2 < lim && (uint64_t)I * H * 4 < lim && nslots <= kMaxExperts;
}

}  // namespace

template <typename Ph>
static void gather(const int32_t* slots, int P, int nslots, int32_t* lists, int32_t* counts,
                   bool vec, const Ph& phase, hipStream_t st) {
  auto go = [&](auto nw) {
    constexpr int NW = decltype(nw)::value;
    if (vec)
      hipLaunchKernelGGL((gather_kernel<NW, true, Ph>), dim3(nslots), dim3(64 * NW), 0, st, slots,
                         P, lists, counts, phase);
    else
      hipLaunchKernelGGL((gather_kernel<NW, false, Ph>), dim3(nslots), dim3(64 * NW), 0, st, slots,
                         P, lists, counts, phase);
  };
  if (P > kGatherLong)
    go(std::integral_constant<int, 16>{});
  else
    go(std::integral_constant<int, 8>{});
}

void launch_gather(const int32_t* slots, int P, int nslots, int32_t* lists, int32_t* counts,
                   hipStream_t st) {
  gather(slots, P, nslots, lists, counts, (uintptr_t)slots % 16 == 0, WholeCall{}, st);
}

int experts_mfma_combine(int T, int H, int K, const float* topk_w, const int32_t* slots,
                         int nslots, const void* work, void* out, hipStream_t st);

size_t mfma_work_bytes(int T, int K, int H, int nslots) {
  if (T < 1 || K < 1 || H < 1 || nslots < 1) return 0;
  return WorkLayout(T * K, H, nslots).total;
}

// Shapes the MFMA path covers (else the caller uses the GEMV kernels).
bool mfma_supported(int H, int I) {
  return H >= kKAlign && I >= kKAlign && H % kKAlign == 0 && I % kKAlign == 0;
}

namespace {

// The pair lists, w13 and w2 of a call's pairs with a slot in [0, nslots):
// their fp32 rows of y in the work buffer.  `spread`: the number of experts
// the call's pairs spread over, for the choice of kernels.  With `phase`, the
// pairs of the experts that the slots hold in it.
int mfma_pairs(const void* x, int T, int H, int I, int K, const int32_t* slots, int nslots,
               const void* w13, size_t w13_stride, const void* w2, size_t w2_stride, void* act,
               void* work, size_t work_bytes, int spread, hipStream_t st,
               const StageEvents* ev, const Phase* phase = nullptr) {
  if (!mfma_supported(H, I)) {
    wisp_set_last_error("MFMA path needs hidden and intermediate sizes that are multiples of 256",
                        "MFMA experts");
    return WISP_ERR_UNSUPPORTED;
  }
  const int P = T * K;
  const WorkLayout W(P, H, nslots);
  if (nslots < 1 || nslots > 65535 || !work || work_bytes < W.total ||
      ((uintptr_t)work) % 256) {
    wisp_set_last_error("MFMA work buffer missing, misaligned or too small", "MFMA experts");
    return WISP_ERR_INVALID;
  }
  int32_t* lists = (int32_t*)((char*)work + W.lists);
  int32_t* counts = (int32_t*)((char*)work + W.counts);
  float* y = (float*)((char*)work + W.y);
  if (phase)
    gather(slots, P, nslots, lists, counts,
           ((uintptr_t)slots | (uintptr_t)phase->ids) % 16 == 0, *phase, st);
  else
    launch_gather(slots, P, nslots, lists, counts, st);
  // A slot holds a token at most once (a token's top-k experts are
  // distinct), so T bounds the rows of any slot.
  const uint16_t* xb = (const uint16_t*)x;
  const uint16_t* a13 = (const uint16_t*)w13;
  const uint16_t* a2 = (const uint16_t*)w2;
  uint16_t* ab = (uint16_t*)act;
  if (tile_call(P, H, I, nslots, spread, T, (uintptr_t)x | (uintptr_t)w13 | (uintptr_t)w2 |
                                                (uintptr_t)act | w13_stride * 2 |
                                                w2_stride * 2)) {
    const TileArgs t13{xb, H, I, K, P, nslots, lists, counts, a13, w13_stride, ab};
    const TileArgs t2{ab, H, I, K, P, nslots, lists, counts, a2, w2_stride, y};
    WISP_HIP_TRY((launch_tiles<true>(t13, st, ev ? ev->ev[0] : nullptr, ev ? ev->ev[1] : nullptr)));
    WISP_HIP_TRY((launch_tiles<false>(t2, st, ev ? ev->ev[2] : nullptr, ev ? ev->ev[3] : nullptr)));
  } else {
    // w13 with two copy stages (three blocks per CU: 241 against 244 us at the
    // Qwen3 512-token chunk), w2 with three (its shorter rows gain nothing from
    // a third block per CU).  Measured on MI355X, these kernels also beat
    // register-streaming ones at every call size, down to 4 tokens (71 against
    // 109 us at the Qwen3 shape).
    WISP_HIP_TRY((launch_dma<2>(xb, H, I, K, P, nslots, lists, counts, a13, w13_stride, a2,
                                w2_stride, ab, y, st, ev)));
  }
  WISP_HIP_TRY(hipGetLastError());
  return WISP_OK;
}

}  // namespace

int experts_mfma(const void* x, int T, int H, int I, int K, const float* topk_w,
                 const int32_t* slots, int nslots, const void* w13, size_t w13_stride,
                 const void* w2, size_t w2_stride, void* act, void* out, void* work,
                 size_t work_bytes, hipStream_t st, const StageEvents* ev) {
  if (T == 0) return WISP_OK;
  const int rc = mfma_pairs(x, T, H, I, K, slots, nslots, w13, w13_stride, w2, w2_stride, act,
                            work, work_bytes, nslots, st, ev);
  if (rc != WISP_OK) return rc;
  return experts_mfma_combine(T, H, K, topk_w, slots, nslots, work, out, st);
}

// The pairs of the experts that a phase of a paged call covers: their y rows
// in the work buffer.
int experts_mfma_phase(const void* x, int T, int H, int I, int K, const int32_t* ids,
                       const int32_t* slots, const PhaseTable& t, int nslots, int num_experts,
                       const void* w13, size_t w13_stride, const void* w2, size_t w2_stride,
                       void* act, void* work, size_t work_bytes, hipStream_t st,
                       const StageEvents* ev) {
  const Phase phase{ids, t};
  return mfma_pairs(x, T, H, I, K, slots, nslots, w13, w13_stride, w2, w2_stride, act, work,
                    work_bytes, num_experts, st, ev, &phase);
}

// out from the y rows of every pair with a slot.
int experts_mfma_combine(int T, int H, int K, const float* topk_w, const int32_t* slots,
                         int nslots, const void* work, void* out, hipStream_t st) {
  const WorkLayout W(T * K, H, nslots);
  launch_combine((const float*)((const char*)work + W.y), T, H, K, nslots, topk_w, slots,
                 (uint16_t*)out, st);
  WISP_HIP_TRY(hipGetLastError());
  return WISP_OK;
}

}  // namespace wisp
