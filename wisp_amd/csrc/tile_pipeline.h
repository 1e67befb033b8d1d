// Block-tile pipeline of the compute-bound grouped GEMMs (large calls).
//
// A block of WR x WT waves multiplies kRows weight rows with up to kToks
// token rows of one slot.  Both operands are staged through LDS by
// asynchronous global->LDS copies, one 128-byte chunk of every row at a
// time and one chunk ahead of its use.  Wave (wr, wt) reads the fragments of
// its NG groups of 16 weight rows and of the token tiles of 16 with index
// wt, wt + WT, ... from there, so a weight byte staged once serves kToks
// tokens and a token byte kRows rows.
#pragma once

#include "dma_pipeline.h"

namespace wisp {
namespace tile {

constexpr int kRowBytes = dma::kRowBytes;
constexpr int kRowsPerCopy = dma::kRowsPerCopy;
constexpr int kStages = 2;

template <int WR_, int WT_, int NG_, int NT_>
struct Shape {
  static constexpr int WR = WR_;  // waves over the weight rows
  static constexpr int WT = WT_;  // waves over the token tiles
  static constexpr int NG = NG_;  // 16-row groups of a wave
  static constexpr int NT = NT_;  // token tiles of a wave
  static constexpr int kWaves = WR * WT;
  static constexpr int kRows = WR * NG * 16;
  static constexpr int kToks = WT * NT * 16;
  static constexpr int kWCopies = kRows / kRowsPerCopy / kWaves;  // per wave
  static constexpr int kTCopies = kToks / kRowsPerCopy / kWaves;
  static_assert(kWCopies * kRowsPerCopy * kWaves == kRows, "weight copies split evenly");
  static_assert(kTCopies * kRowsPerCopy * kWaves == kToks, "token copies split evenly");
  static constexpr int kStage = (kRows + kToks) * kRowBytes;
  static constexpr int kTable = kStages * kStage;
};

// One output tile: a slot, an output panel, and mrows of the slot's tokens
// from m0 on.
struct Work {
  int slot, panel, m0, mrows;
};

// Blocks are persistent, one per CU: block b takes works work_of(b, 0), work_of(b, 1),
// ...  Blocks go to the XCDs round-robin, and each XCD takes runs of kRun
// consecutive works, so blocks that read the same weights or tokens share
// an L2.
constexpr int kBlocks = 256;
constexpr int kRun = 32;
__device__ inline int work_of(int b, int j) {
  const int i = (b >> 3) + j * ((int)gridDim.x >> 3);
  return ((i / kRun) * 8 + (b & 7)) * kRun + i % kRun;
}

// The slots' token counts and first tiles, in LDS.
struct Table {
  int base[kMaxExperts + 1];  // tiles of the slots before s
  int count[kMaxExperts];
};

// Works are ordered by slot, then panel, then token tile.  A slot of M
// tokens has ceil(M / toks) tiles of equal size (rounded up to 16 tokens).
// Called by one wave.
__device__ inline void fill_table(Table* tab, const int32_t* __restrict__ counts, int nslots,
                                  int toks) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int s0 = 0; s0 < nslots; s0 += 64) {
    const int M = s0 + lane < nslots ? counts[s0 + lane] : 0;
    const int n = (M + toks - 1) / toks;
    int incl = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d);
      incl += lane >= d ? o : 0;
    }
    if (s0 + lane < nslots) {
      tab->base[s0 + lane + 1] = base + incl;
      tab->count[s0 + lane] = M;
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  if (lane == 0) tab->base[0] = 0;
}

// Work w (every wave resolves it itself), or false past the last.
__device__ inline bool find_work(const Table* tab, int w, int nslots, int npanels, Work* out) {
  const int lane = threadIdx.x & 63;
  *out = Work{0, 0, 0, 1};
  const int j = w / npanels;  // a tile of the work's slot
  for (int s0 = 0; s0 < nslots; s0 += 64) {
    const int end = tab->base[min(s0 + lane, nslots - 1) + 1];
    const uint64_t hit = __ballot(end > j);
    if (hit) {
      const int s = s0 + __builtin_ctzll(hit);
      const int b = __builtin_amdgcn_readfirstlane(tab->base[s]);
      const int n = __builtin_amdgcn_readfirstlane(tab->base[s + 1]) - b;
      const int M = __builtin_amdgcn_readfirstlane(tab->count[s]);
      const int off = w - b * npanels;
      const int per = ((M + n - 1) / n + 15) & ~15;
      out->slot = s;
      out->panel = off / n;
      out->m0 = (off % n) * per;
      out->mrows = min(per, M - out->m0);
      return true;
    }
  }
  return false;
}

// A range of device memory copied from by a wave-uniform byte offset and one
// 32-bit offset per lane.
struct Range {
  const void* p;
  uint32_t bytes;
};

// r in scalar registers (it is the same for the whole wave, which the
// compiler does not always see).
__device__ __attribute__((always_inline)) inline Range scalar(const Range& r) {
  const uint64_t p = (uint64_t)r.p;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32));
  return Range{(const void*)(((uint64_t)hi << 32) | lo),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)r.bytes)};
}

// 16 bytes per lane from r, lane offset voff plus the wave's offset o, into
// LDS at dst + 16 * lane.
#ifdef __HIP_DEVICE_COMPILE__  // the host pass does not know these builtins
#define WISP_COPY_TO_LDS(size)                                                                   \
  __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                      \
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(r.p), 0, (int)r.bytes, 0x00027000),    \
      (dma::lds_void*)dst, size, (int)voff, o, 0, 0)
#else
#define WISP_COPY_TO_LDS(size)
#endif
__device__ __attribute__((always_inline)) inline void copy16(const Range& r, uint32_t voff, int o,
                                                             void* dst) {
  WISP_COPY_TO_LDS(16);
}
#undef WISP_COPY_TO_LDS

// Where a tile's rows are: the range its weight rows lie in, the byte of the
// row the chunk sequence starts at, and this lane's offset of each of its
// wave's token copies (copy i of wave w covers rows
// [(i * kWaves + w) * kRowsPerCopy, +kRowsPerCopy)).
template <typename Sh>
struct Source {
  Range w;
  uint32_t toff[Sh::kTCopies];
  int tc;  // token copies each wave makes
  int rot;
  int lag;  // chunks by which the second half of the weight rows starts later
};

__device__ inline int chunk_byte(int c, int rot, int row_bytes) {
  const int o = c * kRowBytes + rot;
  return o >= row_bytes ? o - row_bytes : o;
}

// One chunk's copies: weight copies [w0, w1) of each wave, and its tokens'.
template <typename Sh>
__device__ __attribute__((always_inline)) inline void copies(
    unsigned char* st, const Source<Sh>& src, uint32_t woff,
    const uint32_t (&wstep)[Sh::kWCopies], const Range& tokens, int wave, int o, int w0 = 0,
    int w1 = Sh::kWCopies) {
  const Range wr = scalar(src.w), tr = scalar(tokens);
  o = __builtin_amdgcn_readfirstlane(o);
#pragma unroll
  for (int i = 0; i < Sh::kWCopies; ++i)
    if (i >= w0 && i < w1)
      copy16(wr, woff, o + (int)wstep[i], st + (i * Sh::kWaves + wave) * 1024);
#pragma unroll
  for (int i = 0; i < Sh::kTCopies; ++i)
    if (i < src.tc)
      copy16(tr, src.toff[i], o, st + Sh::kRows * kRowBytes + (i * Sh::kWaves + wave) * 1024);
}

}  // namespace tile
}  // namespace wisp
