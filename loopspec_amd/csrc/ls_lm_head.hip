// Vocabulary head fused with the greedy argmax for gfx950.
//
// ids[m] = argmax_n sum_k hidden[m][k] * weight[n][k] (first index of the
// maximum, NaN first), without writing the [M, V] logits: the reference
// computes the logits with the vocabulary head (SGLang's LogitsProcessor over
// ParallelLMHead, sglang_recurrent/modeling/components.py:175-194) and then
// takes torch.argmax over every endpoint row
// (sglang_recurrent/loopspec/decisions.py:116).
//
// Both operands are K-contiguous (hidden [M, H] row-major, weight [V, H] as
// nn.Linear stores it), so each MFMA operand fragment is one 16-byte load.
// Up to 32 rows go to lm_head_rows_kernel (below): a read of the weight. More
// go to lm_head_kernel<MT>: one 512-lane workgroup computes a 64 MT-row x
// 192-column tile with v_mfma_f32_16x16x32_bf16, MT = 1..5 by the rows; eight
// waves (two per SIMD) form a 4 (rows) x 2 (columns) grid, each wave MT x 6
// tiles of 16 x 16. At MT = 5 a k-step reads 11 operand fragments from LDS for
// 30 MFMAs (a 5 x 3 tile per wave reads 8 for 15: about 30 % more LDS traffic
// per flop, above the LDS read rate at the MFMA peak). Both operands are staged
// through LDS in k-blocks of 64 (16-byte chunks XOR-swizzled by row) by direct
// global-to-LDS loads (global_load_lds_dwordx4): the weight two or three blocks
// ahead (non-temporal, see dma16_stream), so that those HBM reads are in flight while
// a block is multiplied and no registers hold them, the hidden rows
// (L2-resident, re-read by every column block) one or two blocks ahead. Each
// block ends with an explicit wait that leaves the newest loads in flight and a
// bare s_barrier (a workgroup fence would wait for them too). The loads bound
// the kernel (without the MFMAs it takes about 85 % of its time at 320 rows):
// a wave's loads return in order, so waiting for the next hidden block also
// waits for every weight load issued before it. Splitting the two operands'
// loads over different waves, with the next half block's fragments read during
// a half block's MFMAs, measured slower at 320 rows (68 us against 63): the
// weight loads of three waves take longer than the same loads spread over
// eight. Rows and time (H 2048, V 49152, with the finish kernel; before: one
// 320-row tile for any row count): 3: 61 -> 45 us, 64: 61 -> 50, 128: 61 -> 49,
// 192: 65 -> 53, 256: 65 -> 60, 320: 66 -> 66, 700: 188 -> 147.
// The epilogue reduces each row's (value, -index) key over the tile's columns
// (in-lane over the six column tiles, shuffles over the 16 lanes of a row, LDS
// over the two column waves) and writes one key per (column block, row); a
// second kernel reduces a row's keys to its index.
#include <string>

#include "ls_common.hpp"
#include "ls_runtime.hpp"

namespace ls {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kLmLanes = 512;
constexpr int kLmWaves = kLmLanes / 64;         // 8: 4 (rows) x 2 (columns)
constexpr int kLmNT = 6;                       // 16-column tiles per wave
constexpr int kLmColsPerWave = 16 * kLmNT;     // 96
constexpr int kLmMaxRows = 320;                // rows per workgroup at most (64 MT of them, MT = 1..5)
constexpr int kLmBN = 2 * kLmColsPerWave;      // 192 columns per workgroup
constexpr int kLmKB = 64;                      // k per LDS block
constexpr int kXcds = 8;
constexpr int kGridXLog2 = 22;                 // workgroups along x at most (see head_grid)
constexpr int kLmRowBytes = kLmKB * 2;         // 128 bytes of a row's k-block
constexpr int kLmBRounds = 3;  // 24 x 1 KB per B block over 8 waves

struct LmParams {
  const char* hidden;   // [M, H] bf16, row stride hs elements
  int64_t hs;
  const char* weight;   // [V, H] bf16, row stride ws elements
  int64_t ws;
  int64_t M, H, V;
  int nblk;             // column blocks (ceil(V / 192))
  int mblk;             // row blocks (ceil(M / 320); each of 64 MT rows, MT by the rows per block)
  uint64_t* keys;       // [nblk, M] partial keys
  int64_t* out;         // [M]
  void* logits;         // logits epilogue: [M, V] float32 or bf16, row stride los elements
  int64_t los;
};

// What a head workgroup writes from its tile: each row's partial key over
// the tile's columns (the argmax and verify paths), or the logits themselves.
enum LmEpilogue : int { kLmKeys = 0, kLmLogitsF32 = 1, kLmLogitsBF16 = 2 };

constexpr int kLmBBytes = kLmBN * kLmRowBytes;  // 24 KB
static_assert(kLmBRounds * kLmWaves * 1024 == kLmBBytes, "whole rounds per wave");

// Direct global-to-LDS load of 16 bytes per lane: lane l's bytes land at LDS
// address lds + 16 l (lds wave-uniform, passed in M0, which the compiler sets
// for the statement as an operand). Issued as an instruction the compiler does
// not track, so that its own LDS-hazard waits do not stall reads of the other
// buffers while the load is in flight; the caller waits for it explicitly
// (vmcnt) before the workgroup reads the buffer.
__device__ __forceinline__ void dma16(const void* src, uint32_t lds) {
  asm volatile("global_load_lds_dwordx4 %0, off" : : "v"(src), "{m0}"(lds) : "memory");
}

// The same with the non-temporal hint, for the weight: a line is read by the
// row blocks of one column block and then no more, while the hidden rows are
// re-read by every column block. After other traffic (2 GB written before each
// call; H 2048, V 49152) the hint is worth 102 -> 56 us at 65 rows, 114 -> 76
// at 320, 165 -> 149 at 700. Calls back to back, which nothing separates and
// which find part of the 201 MB weight in the Infinity Cache without it, take
// 66 us with it and 61 without at 320 rows, 144 and 138 at 700; a weight that
// does not fit there (1 GB, 1280 rows) 1100 and 1104.
__device__ __forceinline__ void dma16_stream(const void* src, uint32_t lds) {
  asm volatile("global_load_lds_dwordx4 %0, off nt" : : "v"(src), "{m0}"(lds) : "memory");
}

// A head workgroup's index. A launch dimension holds fewer than 2^32 lanes, so
// workgroups past the first 2^22 go along y; in dispatch order the index still
// counts up by one.
__device__ __forceinline__ int head_block() {
  return static_cast<int>(blockIdx.x + (blockIdx.y << kGridXLog2));
}

// Byte offset of 16-byte chunk c of row r in an A block.
__device__ __forceinline__ int a_off(int r, int c) { return r * kLmRowBytes + ((c ^ (r & 7)) << 4); }

// More than 32 rows; a workgroup takes kBM of them.
template <int MT, int EPI>
__global__ __launch_bounds__(kLmLanes) void lm_head_kernel(const LmParams p) {
  constexpr int kRowsPerWave = 16 * MT;
  constexpr int kBM = 4 * kRowsPerWave;
  constexpr int kABytes = kBM * kLmRowBytes;
  constexpr int kARounds = kABytes / 1024 / kLmWaves;  // 1 KB loads per wave and block
  // blocks of hidden rows and of weight in LDS: with up to 192 rows there is
  // room for a third (and up to 128 for a fourth weight block), so that a load
  // has two block times to arrive instead of one
  constexpr int kAStages = MT <= 3 ? 3 : 2, kBStages = MT <= 2 ? 4 : 3;
  constexpr int kALead = kAStages - 1, kBLead = kBStages - 1;  // blocks ahead
  // this wave's loads newer than block kb + 1's at the end of block kb
  constexpr int kNewer = (kALead - 1) * (kARounds + kLmBRounds) + (kBLead > kALead ? kLmBRounds : 0);
  __shared__ __attribute__((aligned(16))) uint8_t abuf[kAStages][kABytes];
  __shared__ __attribute__((aligned(16))) uint8_t bbuf[kBStages][kLmBBytes];
  const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
  const int wm = wid >> 1, wn = wid & 1;
  // Workgroups go to the eight XCDs in turn; the row blocks of one column block
  // follow each other on one XCD, so its weight comes from HBM once and the
  // other row blocks read it from that XCD's L2. (With the row block slowest
  // the whole weight was streamed once per row block: 1260 us against 1120 at
  // M 1280, H 4096, V 128256. Giving each XCD a run of column blocks of one row
  // block, for its hidden rows to stay in L2, measured 1160.)
  int m_blk = 0, nblk = head_block();
  if (p.mblk > 1) {
    const int xcd = nblk & (kXcds - 1), at = nblk / kXcds;
    m_blk = at % p.mblk;
    nblk = at / p.mblk * kXcds + xcd;
  }
  if (nblk >= p.nblk) return;
  const int64_t m_base = static_cast<int64_t>(m_blk) * kBM;
  const int64_t n_base = static_cast<int64_t>(nblk) * kLmBN;
  const int nkb = static_cast<int>(p.H / kLmKB);

  // Direct loads: round i of wave w puts lane l's 16 bytes at LDS chunk
  // j = (8i + w) * 64 + l, i.e. row j/8 of the buffer, swizzled chunk l & 7,
  // so the lane fetches logical chunk (l & 7) ^ (row & 7) of that row. A block
  // of hidden rows is 8 MT such 1 KB rounds (MT per wave), one of weight rows
  // 24 (three per wave). Rows past the matrix are clamped into it (their
  // results are never used). Byte offsets from the block's first row.
  const uint32_t lchunk = static_cast<uint32_t>(((lane & 7) ^ ((lane >> 3) & 7)) << 4);
  const char* abase = p.hidden + m_base * p.hs * 2;
  uint32_t aoff[kARounds];
#pragma unroll
  for (int i = 0; i < kARounds; ++i) {
    const int r = (i * kLmWaves + wid) * 8 + (lane >> 3);
    const int64_t rr = m_base + r < p.M ? r : p.M - 1 - m_base;
    aoff[i] = static_cast<uint32_t>(rr * p.hs * 2) + lchunk;
  }
  const char* bbase = p.weight + n_base * p.ws * 2;
  uint32_t boff[kLmBRounds];
#pragma unroll
  for (int i = 0; i < kLmBRounds; ++i) {
    const int r = (i * kLmWaves + wid) * 8 + (lane >> 3);
    const int64_t rr = n_base + r < p.V ? r : p.V - 1 - n_base;
    boff[i] = static_cast<uint32_t>(rr * p.ws * 2) + lchunk;
  }
  auto dma_a = [&](int kb, uint8_t* dst) {
    const char* base = abase + static_cast<int64_t>(kb) * kLmRowBytes;
#pragma unroll
    for (int i = 0; i < kARounds; ++i) {
      const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst)) + (i * kLmWaves + wid) * 1024;
      dma16(base + aoff[i], __builtin_amdgcn_readfirstlane(lds));
    }
  };
  auto dma_b = [&](int kb, uint8_t* dst) {
    const char* base = bbase + static_cast<int64_t>(kb) * kLmRowBytes;
#pragma unroll
    for (int i = 0; i < kLmBRounds; ++i) {
      const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst)) + (i * kLmWaves + wid) * 1024;
      dma16_stream(base + boff[i], __builtin_amdgcn_readfirstlane(lds));
    }
  };

  f32x4 acc[MT][kLmNT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int nt = 0; nt < kLmNT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // fragment rows: this wave's first row / column plus lane & 15 (tiles are a
  // multiple of 16 rows apart, so the swizzle is fixed per lane and the rest
  // is an immediate offset)
  const int fr_a = (wm * kRowsPerWave + (lane & 15)) * kLmRowBytes;
  const int fr_b = (wn * kLmColsPerWave + (lane & 15)) * kLmRowBytes;
  // One k-block: 2 k-steps x MT row tiles. Each tile's fragment (and each
  // k-step's column fragments) is read one tile ahead, before the current
  // tile's MFMAs, so the LDS latency overlaps them; a scheduling fence after
  // each tile keeps the compiler from hoisting every read.
  auto compute = [&](const uint8_t* abuf, const uint8_t* bbuf) {
    auto sw = [&](int ks) { return ((ks * 4 + (lane >> 4)) ^ (lane & 7)) << 4; };
    auto read_a = [&](int ks, int mt) {
      return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(abuf + fr_a + sw(ks) + mt * 16 * kLmRowBytes));
    };
    auto read_b = [&](int ks, bf16x8 (&b)[kLmNT]) {
      const uint8_t* const fb = bbuf + fr_b + sw(ks);
#pragma unroll
      for (int nt = 0; nt < kLmNT; ++nt)
        b[nt] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(fb + nt * 16 * kLmRowBytes));
    };
    bf16x8 acur, anext, bcur[kLmNT], bnext[kLmNT];
    read_b(0, bcur);
    acur = read_a(0, 0);
#pragma unroll
    for (int g = 0; g < 2 * MT; ++g) {
      const int ks = g / MT, mt = g % MT;
      if (g + 1 < 2 * MT) {
        const int ks1 = (g + 1) / MT, mt1 = (g + 1) % MT;
        if (ks1 != ks) read_b(ks1, bnext);
        anext = read_a(ks1, mt1);
      }
#pragma unroll
      for (int nt = 0; nt < kLmNT; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(acur, bcur[nt], acc[mt][nt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      acur = anext;
      if (g + 1 == MT) {
#pragma unroll
        for (int nt = 0; nt < kLmNT; ++nt) bcur[nt] = bnext[nt];
      }
    }
  };
  // End of block kb: block kb + 1 has landed in LDS (loads return in order;
  // the kNewer newer ones of this wave may be under way), this lane's LDS reads
  // are done, then the workgroup meets.
  auto block_end = [&](bool newer_in_flight) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (newer_in_flight) {
      __builtin_amdgcn_s_waitcnt((kNewer & 15) | ((kNewer >> 4) << 14) | 0x70);  // vmcnt(kNewer) lgkmcnt(0)
    } else {
      __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) expcnt(7) lgkmcnt(0)
    }
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };

  // block kb: hidden rows in abuf[kb % kAStages], weight rows in bbuf[kb %
  // kBStages]; unrolled so that every buffer is named statically. Per block,
  // the hidden rows of kb + kALead, then the weight rows of kb + kBLead, go out
  // before kb is multiplied, into buffers last read a barrier ago.
#pragma unroll
  for (int i = 0; i < kBLead; ++i) {
    if (i < kALead && i < nkb) dma_a(i, abuf[i]);
    if (i < nkb) dma_b(i, bbuf[i]);
  }
  block_end(false);
  constexpr int kUnroll = MT <= 2 ? 12 : (MT == 3 ? 3 : 6);  // whole turns of both rings
  static_assert(kUnroll % kAStages == 0 && kUnroll % kBStages == 0, "static buffers");
  for (int kb0 = 0; kb0 < nkb; kb0 += kUnroll) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int kb = kb0 + u;
      if (kb < nkb) {
        if (kb + kALead < nkb) dma_a(kb + kALead, abuf[(u + kALead) % kAStages]);
        const bool ahead = kb + kBLead < nkb;
        if (ahead) dma_b(kb + kBLead, bbuf[(u + kBLead) % kBStages]);
        compute(abuf[u % kAStages], bbuf[u % kBStages]);
        block_end(ahead);
      }
    }
  }

  if constexpr (EPI != kLmKeys) {
    // logits: accumulator i of tile (mt, nt) is row (lane / 16) * 4 + i, column
    // lane % 16 of the tile; 16 lanes store 16 consecutive columns of a row
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t m = m_base + wm * kRowsPerWave + mt * 16 + (lane >> 4) * 4 + i;
        if (m >= p.M) continue;
#pragma unroll
        for (int nt = 0; nt < kLmNT; ++nt) {
          const int64_t col = n_base + wn * kLmColsPerWave + nt * 16 + (lane & 15);
          if (col >= p.V) continue;
          if constexpr (EPI == kLmLogitsF32) {
            static_cast<float*>(p.logits)[m * p.los + col] = acc[mt][nt][i];
          } else {
            static_cast<__bf16*>(p.logits)[m * p.los + col] = static_cast<__bf16>(acc[mt][nt][i]);
          }
        }
      }
    }
    return;
  }
  uint64_t* const keys = reinterpret_cast<uint64_t*>(abuf);  // every read of it is behind the last barrier
  // epilogue: row keys over this wave's 96 columns, then over the 2 column waves
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint64_t best = 0;
#pragma unroll
      for (int nt = 0; nt < kLmNT; ++nt) {
        const int64_t col = n_base + wn * kLmColsPerWave + nt * 16 + (lane & 15);
        const uint64_t key = col < p.V ? argmax_key(acc[mt][nt][i], static_cast<uint32_t>(col)) : 0ull;
        best = key > best ? key : best;
      }
#pragma unroll
      for (int s = 1; s < 16; s <<= 1) {
        const uint64_t o = __shfl_xor(best, s);
        best = o > best ? o : best;
      }
      if ((lane & 15) == 0) keys[(wm * kRowsPerWave + mt * 16 + (lane >> 4) * 4 + i) * 2 + wn] = best;
    }
  }
  __syncthreads();
  for (int r = t; r < kBM; r += kLmLanes) {
    const int64_t m = m_base + r;
    if (m < p.M) {
      const uint64_t k0 = keys[r * 2], k1 = keys[r * 2 + 1];
      const uint64_t best = k1 > k0 ? k1 : k0;
      p.keys[static_cast<int64_t>(nblk) * p.M + m] = best;
    }
  }
}

// Up to 32 rows: the weight straight into registers.
//
// With few rows the head is a read of the weight (2 V H bytes for 2 M V H
// flops). Here each of twelve waves owns 16 of the 192 columns; its weight
// fragments are its own, so they need no LDS: a lane loads them four k-blocks
// of 64 ahead (8 loads, 32 registers; 96 KB in flight per CU; eight ahead
// measured the same), in order and without waiting for anything else. The
// hidden rows, shared by the waves, go through two LDS buffers of four
// k-blocks, one barrier per buffer. H 2048, V 49152, M = 3: 45 us with the
// finish kernel against 48.5 for lm_head_kernel<1>, M = 32: 45 against 46; past
// 32 rows the reads of the hidden rows by every wave cost more than the shared
// tile's (M = 64: 52 against 50). A read of the same bytes in the same pattern,
// and nothing else, takes 34.5 us.
constexpr int kDppRowRor8 = 0x128;
constexpr int kLrLanes = 768;
constexpr int kLrWaves = kLrLanes / 64;  // one per 16 columns
constexpr int kLrAhead = 4;              // k-blocks of weight in flight per wave, and per LDS buffer of hidden rows
static_assert(kLrWaves * 16 == kLmBN, "the same column blocks as lm_head_kernel (their keys share a layout)");

template <int MT, int EPI>
__global__ __launch_bounds__(kLrLanes) void lm_head_rows_kernel(const LmParams p) {
  constexpr int kRows = 16 * MT;
  constexpr int kStepBytes = kRows * kLmRowBytes;
  constexpr int kChunks = kLrAhead * kStepBytes / 16;
  constexpr int kRounds = (kChunks + kLrLanes - 1) / kLrLanes;
  __shared__ __attribute__((aligned(16))) uint8_t abuf[2][kLrAhead * kStepBytes];
  __shared__ uint64_t keys[kRows][kLrWaves];
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const int nblk = head_block();
  if (nblk >= p.nblk) return;
  const int64_t n_base = static_cast<int64_t>(nblk) * kLmBN;
  const int nkb = static_cast<int>(p.H / kLmKB);
  const int64_t col = n_base + w * 16 + (lane & 15);  // of this lane's accumulators
  // This lane's 16 bytes of weight rows lane & 7 and 8 + (lane & 7) of the
  // wave's sixteen (clamped: the results of columns past V are not used): one
  // load takes whole 128-byte lines of eight rows (half lines of sixteen, as the
  // MFMA has them, read at 4.9-5.3 TB/s instead of 5.8-6.5), lane l the chunk
  // l / 16 of the first half of its line, or of the second where bit 3 of l is
  // set.
  const char* bp[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t n = n_base + w * 16 + h * 8 + (lane & 7);
    bp[h] = p.weight + (n < p.V ? n : p.V - 1) * p.ws * 2 + (((lane >> 3) & 1) * 4 + (lane >> 4)) * 16;
  }
  const char* const none = p.weight;  // what a load past the last k-block reads

  // hidden rows: chunk i = t + 768 r of a buffer is 16 bytes of row (i / 8) mod
  // kRows of k-block i / (8 kRows), XOR-swizzled by row as in lm_head_kernel
  const char* ap[kRounds];
  int astep[kRounds];
  uint32_t aoff[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int i = t + r * kLrLanes;
    const int row = (i >> 3) & (kRows - 1), ch = i & 7;
    astep[r] = i / (8 * kRows);
    aoff[r] = static_cast<uint32_t>(astep[r] * kStepBytes + a_off(row, ch));
    ap[r] = p.hidden + (row < p.M ? row : p.M - 1) * p.hs * 2 + ch * 16;
  }
  u32x4 areg[kRounds];  // the next buffer of hidden rows on its way
  auto load_a = [&](int kb0, u32x4 (&d)[kRounds]) {  // the buffer of k-blocks kb0 .. (past the last: the last again, not used)
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      const int kb = kb0 + astep[r] < nkb ? kb0 + astep[r] : nkb - 1;
      d[r] = *reinterpret_cast<const u32x4*>(ap[r] + static_cast<int64_t>(kb) * kLmRowBytes);
    }
  };
  auto store_a = [&](uint8_t* buf, const u32x4 (&d)[kRounds]) {
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      if (kChunks % kLrLanes == 0 || t + r * kLrLanes < kChunks) *reinterpret_cast<u32x4*>(buf + aoff[r]) = d[r];
    }
  };
  auto meet = [&]() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); the weight loads stay in flight
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
  u32x4 b[kLrAhead][2];
  auto load_b = [&](int kb, u32x4 (&d)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const char* src = kb < nkb ? bp[h] + static_cast<int64_t>(kb) * kLmRowBytes : none;
      d[h] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src));
    }
  };
  // Fragments of a k-block's two halves: the first takes rows 0..7 from the
  // lanes below 8 of each sixteen and rows 8..15 from those lanes of the other
  // load (rotated by eight), the second the other way round.
  auto fragments = [&](const u32x4 (&d)[2], bf16x8 (&f)[2]) {
    u32x4 f0, f1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f0[i] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(d[0][i]), static_cast<int>(d[1][i]),
                                                                kDppRowRor8, 0xf, 0xc, false));
      f1[i] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(d[1][i]), static_cast<int>(d[0][i]),
                                                                kDppRowRor8, 0xf, 0x3, false));
    }
    f[0] = __builtin_bit_cast(bf16x8, f0);
    f[1] = __builtin_bit_cast(bf16x8, f1);
  };
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = (lane & 15) * kLmRowBytes;
  auto multiply = [&](const uint8_t* step, const u32x4 (&d)[2]) {
    bf16x8 b2[2];
    fragments(d, b2);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int sw = ((ks * 4 + (lane >> 4)) ^ (lane & 7)) << 4;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const bf16x8 a = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u32x4*>(step + fr + sw + mt * 16 * kLmRowBytes));
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b2[ks], acc[mt], 0, 0, 0);
      }
    }
  };

  // Loads return in order, so hidden rows asked for after a k-block's weight
  // arrive after it: those of a group go out before its weight, a group
  // ahead, or waiting for them would wait for all the weight under way.
  u32x4 first[kRounds];
  load_a(0, first);
#pragma unroll
  for (int u = 0; u < kLrAhead; ++u) {
    load_b(u, b[u]);
    if (u == kLrAhead - 1) load_a(kLrAhead, areg);
    __builtin_amdgcn_sched_barrier(0);
  }
  store_a(abuf[0], first);
  meet();
  int cur = 0;  // buffer of the k-blocks being multiplied
  int kb0 = 0;
  // whole groups of kLrAhead k-blocks with more to come: no branch inside, so
  // that the compiler's wait for one group's weight leaves the next in flight
  for (; kb0 + kLrAhead < nkb; kb0 += kLrAhead) {
#pragma unroll
    for (int u = 0; u < kLrAhead; ++u) {
      multiply(abuf[cur] + u * kStepBytes, b[u]);
      __builtin_amdgcn_sched_barrier(0);
      load_b(kb0 + u + kLrAhead, b[u]);
      if (u == kLrAhead - 1) {
        store_a(abuf[cur ^ 1], areg);
        load_a(kb0 + 2 * kLrAhead, areg);
        meet();
        cur ^= 1;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the last group (1 .. kLrAhead k-blocks)
#pragma unroll
  for (int u = 0; u < kLrAhead; ++u) {
    if (kb0 + u < nkb) multiply(abuf[cur] + u * kStepBytes, b[u]);
  }

  // accumulator i of row tile mt is row mt * 16 + (lane / 16) * 4 + i
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = mt * 16 + (lane >> 4) * 4 + i;
      if constexpr (EPI == kLmKeys) {
        uint64_t best = col < p.V ? argmax_key(acc[mt][i], static_cast<uint32_t>(col)) : 0ull;
#pragma unroll
        for (int sft = 1; sft < 16; sft <<= 1) {
          const uint64_t o = __shfl_xor(best, sft);
          best = o > best ? o : best;
        }
        if ((lane & 15) == 0) keys[m][w] = best;
      } else {
        if (m < p.M && col < p.V) {
          if constexpr (EPI == kLmLogitsF32) {
            static_cast<float*>(p.logits)[m * p.los + col] = acc[mt][i];
          } else {
            static_cast<__bf16*>(p.logits)[m * p.los + col] = static_cast<__bf16>(acc[mt][i]);
          }
        }
      }
    }
  }
  if constexpr (EPI == kLmKeys) {
    __syncthreads();
    if (t < kRows && t < p.M) {
      uint64_t best = keys[t][0];
#pragma unroll
      for (int i = 1; i < kLrWaves; ++i) best = keys[t][i] > best ? keys[t][i] : best;
      p.keys[static_cast<int64_t>(nblk) * p.M + t] = best;
    }
  }
}

// One wave per row: the maximum of the row's nblk keys.
__global__ __launch_bounds__(256) void lm_head_finish_kernel(const LmParams p) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t m = static_cast<int64_t>(blockIdx.x) * 4 + threadIdx.x / kWave;
  if (m >= p.M) return;
  uint64_t best = 0;
  for (int b = lane; b < p.nblk; b += kWave) {
    const uint64_t k = p.keys[static_cast<int64_t>(b) * p.M + m];
    best = k > best ? k : best;
  }
  best = wave_max_u64(best);
  if (lane == 0) p.out[m] = argmax_key_index(best);
}

// Greedy verify on the head's keys: one 256-lane workgroup per batch element
// g, whose rows are g * rpg + j (target positions j = 0..k, then the draft
// positions when the draft ids come from draft rows). Wave w reduces rows w,
// w + 4, ... to their ids; wave 0 then runs the accept-prefix scan (lane i
// compares draft position i, one ballot finds the first mismatch).
struct LmVerify {
  int k;
  int rpg;                       // rows per batch element: k + 1, or 2k + 1 with draft rows
  const int64_t* draft_tokens;   // [B, k] when the draft rows are not in the head's rows
  int32_t* accept_len;           // [B]
  int64_t* tokens;               // [B, k + 1]
  int64_t* row_argmax;           // optional [B, rpg]
};

constexpr int kLvLanes = 256;
constexpr int kLvMaxRows = 2 * 64 + 1;

__global__ __launch_bounds__(kLvLanes) void lm_head_verify_kernel(const LmParams p, const LmVerify v) {
  __shared__ int64_t ids[kLvMaxRows];
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int64_t g = blockIdx.x;
  for (int j = wid; j < v.rpg; j += kLvLanes / kWave) {
    const int64_t m = g * v.rpg + j;
    uint64_t best = 0;
    for (int b = lane; b < p.nblk; b += kWave) {
      const uint64_t key = p.keys[static_cast<int64_t>(b) * p.M + m];
      best = key > best ? key : best;
    }
    best = wave_max_u64(best);
    if (lane == 0) ids[j] = argmax_key_index(best);
  }
  __syncthreads();
  if (wid != 0) return;
  const int k = v.k;  // <= 64: draft position i is lane i
  const int64_t d = lane < k ? (v.draft_tokens ? v.draft_tokens[g * k + lane] : ids[k + 1 + lane]) : -1;
  const uint64_t bad = __ballot(lane < k && d != ids[lane < k ? lane : 0]);
  const int a = bad ? __builtin_ctzll(bad) : k;
  for (int pos = lane; pos <= k; pos += kWave) v.tokens[g * (k + 1) + pos] = pos <= a ? ids[pos] : -1;
  if (v.row_argmax) {
    for (int j = lane; j < v.rpg; j += kWave) v.row_argmax[g * v.rpg + j] = ids[j];
  }
  if (lane == 0) v.accept_len[g] = a;
}

}  // namespace
}  // namespace ls

using namespace ls;

extern "C" {

uint64_t ls_lm_head_argmax_workspace(int64_t rows, int64_t vocab) {
  if (rows <= 0 || vocab <= 0) return 0;
  const int64_t nblk = (vocab + kLmBN - 1) / kLmBN;
  return (static_cast<uint64_t>(nblk) * static_cast<uint64_t>(rows) * 8u + 255u) & ~255ull;
}

}  // extern "C"

namespace {

// Column blocks as launched: with several row blocks in groups of kXcds, each
// with its row blocks (see lm_head_kernel).
int64_t launched_cols(int64_t nblk, int64_t mblk) { return mblk > 1 ? (nblk + kXcds - 1) / kXcds * kXcds : nblk; }

// head_block's grid of n workgroups; those past n leave at once.
dim3 head_grid(int64_t n) {
  constexpr int64_t kMaxX = int64_t{1} << kGridXLog2;
  static_assert(kMaxX * kLrLanes < (int64_t{1} << 32) && kMaxX * kLmLanes < (int64_t{1} << 32), "lanes along x");
  return n <= kMaxX ? dim3(static_cast<unsigned>(n)) : dim3(kMaxX, static_cast<unsigned>((n + kMaxX - 1) / kMaxX));
}

// The kernel of a head call: a rule on the rows alone, so that every entry
// point forms a row's logits by the same products in the same order.
template <int EPI>
void launch_head(const LmParams& p, hipStream_t st) {
  if (p.M <= 32) {
    const dim3 grid = head_grid(p.nblk);
    if (p.M <= 16) {
      hipLaunchKernelGGL((lm_head_rows_kernel<1, EPI>), grid, dim3(kLrLanes), 0, st, p);
    } else {
      hipLaunchKernelGGL((lm_head_rows_kernel<2, EPI>), grid, dim3(kLrLanes), 0, st, p);
    }
    return;
  }
  const dim3 grid = head_grid(launched_cols(p.nblk, p.mblk) * p.mblk);
  const int64_t rows = (p.M + p.mblk - 1) / p.mblk;  // per row block
  if (rows <= 64) {
    hipLaunchKernelGGL((lm_head_kernel<1, EPI>), grid, dim3(kLmLanes), 0, st, p);
  } else if (rows <= 128) {
    hipLaunchKernelGGL((lm_head_kernel<2, EPI>), grid, dim3(kLmLanes), 0, st, p);
  } else if (rows <= 192) {
    hipLaunchKernelGGL((lm_head_kernel<3, EPI>), grid, dim3(kLmLanes), 0, st, p);
  } else if (rows <= 256) {
    hipLaunchKernelGGL((lm_head_kernel<4, EPI>), grid, dim3(kLmLanes), 0, st, p);
  } else {
    hipLaunchKernelGGL((lm_head_kernel<5, EPI>), grid, dim3(kLmLanes), 0, st, p);
  }
}

// Checks shared by the head's entry points; fills p and launches the head
// kernel (the caller launches the finish kernel it needs).
int lm_head_launch(const char* what, const void* hidden, int64_t hidden_stride, const void* weight,
                   int64_t weight_stride, int dtype, int64_t rows, int64_t hidden_size, int64_t vocab,
                   void* workspace, uint64_t ws_bytes, hipStream_t st, LmParams* out, int epi = kLmKeys,
                   void* logits = nullptr, int64_t logits_stride = 0) {
  const std::string w(what);
  if (dtype != LS_DTYPE_BF16) return fail(LS_ERR_VALUE, w + ": bf16 hidden states and weight only");
  if (rows < 0 || hidden_size <= 0 || vocab <= 0 || vocab > 0x7fffffffLL)
    return fail(LS_ERR_VALUE, w + ": need rows >= 0, hidden_size > 0, 0 < vocab < 2^31");
  if (hidden_size % kLmKB != 0) return fail(LS_ERR_VALUE, w + ": hidden_size must be a multiple of 64");
  if (rows == 0) return LS_OK;
  if (hidden == nullptr || weight == nullptr) return fail(LS_ERR_VALUE, w + ": NULL pointer");
  if (!aligned16(hidden) || !aligned16(weight) || hidden_stride % 8 != 0 || weight_stride % 8 != 0 ||
      hidden_stride < hidden_size || weight_stride < hidden_size)
    return fail(LS_ERR_VALUE, w + ": rows must be 16-byte aligned with strides >= hidden_size");
  const int64_t nblk = (vocab + kLmBN - 1) / kLmBN;
  const int64_t mblk = (rows + kLmMaxRows - 1) / kLmMaxRows;
  if (mblk > 65535) return fail(LS_ERR_VALUE, w + ": too many rows");
  // (their keys or logits would fill terabytes)
  if (launched_cols(nblk, mblk) * mblk > 0x7fffffffLL - (1LL << kGridXLog2))
    return fail(LS_ERR_VALUE, w + ": rows x vocab too large");
  if (epi == kLmKeys && (workspace == nullptr || ws_bytes < ls_lm_head_argmax_workspace(rows, vocab)))
    return fail(LS_ERR_VALUE, w + ": workspace too small");
  if (epi != kLmKeys && (logits == nullptr || logits_stride < vocab))
    return fail(LS_ERR_VALUE, w + ": logits must be [rows, vocab] with a row stride >= vocab");
  LmParams& p = *out;
  p = LmParams{};
  p.hidden = static_cast<const char*>(hidden);
  p.hs = hidden_stride;
  p.weight = static_cast<const char*>(weight);
  p.ws = weight_stride;
  p.M = rows;
  p.H = hidden_size;
  p.V = vocab;
  p.nblk = static_cast<int>(nblk);
  p.mblk = static_cast<int>(mblk);
  p.keys = static_cast<uint64_t*>(workspace);
  p.logits = logits;
  p.los = logits_stride;
  if (epi == kLmLogitsF32) {
    launch_head<kLmLogitsF32>(p, st);
  } else if (epi == kLmLogitsBF16) {
    launch_head<kLmLogitsBF16>(p, st);
  } else {
    launch_head<kLmKeys>(p, st);
  }
  return LS_OK;
}

}  // namespace

extern "C" {

int ls_lm_head_argmax(const void* hidden, int64_t hidden_stride, const void* weight, int64_t weight_stride,
                      int dtype, int64_t rows, int64_t hidden_size, int64_t vocab, int64_t* out, void* workspace,
                      uint64_t ws_bytes, ls_stream_t stream) {
  if (rows > 0 && out == nullptr) return fail(LS_ERR_VALUE, "lm_head_argmax: NULL pointer");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  LmParams p;
  const int rc = lm_head_launch("lm_head_argmax", hidden, hidden_stride, weight, weight_stride, dtype, rows,
                                hidden_size, vocab, workspace, ws_bytes, st, &p);
  if (rc != LS_OK || rows == 0) return rc;
  p.out = out;
  hipLaunchKernelGGL(lm_head_finish_kernel, dim3(static_cast<unsigned>((rows + 3) / 4)), dim3(256), 0, st, p);
  return check_launch("lm_head_argmax launch");
}

int ls_lm_head_logits(const void* hidden, int64_t hidden_stride, const void* weight, int64_t weight_stride,
                      int dtype, int64_t rows, int64_t hidden_size, int64_t vocab, void* logits,
                      int64_t logits_stride, int logits_dtype, ls_stream_t stream) {
  if (logits_dtype != LS_DTYPE_F32 && logits_dtype != LS_DTYPE_BF16)
    return fail(LS_ERR_VALUE, "lm_head_logits: float32 or bf16 logits only");
  if (rows > 0 && !aligned16(logits)) return fail(LS_ERR_VALUE, "lm_head_logits: logits must be 16-byte aligned");
  LmParams p;
  const int rc = lm_head_launch("lm_head_logits", hidden, hidden_stride, weight, weight_stride, dtype, rows,
                                hidden_size, vocab, nullptr, 0, static_cast<hipStream_t>(stream), &p,
                                logits_dtype == LS_DTYPE_F32 ? kLmLogitsF32 : kLmLogitsBF16, logits, logits_stride);
  if (rc != LS_OK || rows == 0) return rc;
  return check_launch("lm_head_logits launch");
}

int ls_lm_head_greedy_verify(const void* hidden, int64_t hidden_stride, const void* weight, int64_t weight_stride,
                             int dtype, int64_t batch, int64_t k, int64_t hidden_size, int64_t vocab,
                             const int64_t* draft_tokens, int32_t* accept_len, int64_t* tokens,
                             int64_t* row_argmax, void* workspace, uint64_t ws_bytes, ls_stream_t stream) {
  if (batch < 0 || k < 1 || k > 64 || batch > 65535)
    return fail(LS_ERR_VALUE, "lm_head_greedy_verify: need 0 <= batch <= 65535 and 1 <= k <= 64");
  if (batch == 0) return LS_OK;
  if (accept_len == nullptr || tokens == nullptr) return fail(LS_ERR_VALUE, "lm_head_greedy_verify: NULL pointer");
  const int64_t rpg = draft_tokens ? k + 1 : 2 * k + 1;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  LmParams p;
  const int rc = lm_head_launch("lm_head_greedy_verify", hidden, hidden_stride, weight, weight_stride, dtype,
                                batch * rpg, hidden_size, vocab, workspace, ws_bytes, st, &p);
  if (rc != LS_OK) return rc;
  LmVerify v{static_cast<int>(k), static_cast<int>(rpg), draft_tokens, accept_len, tokens, row_argmax};
  hipLaunchKernelGGL(lm_head_verify_kernel, dim3(static_cast<unsigned>(batch)), dim3(kLvLanes), 0, st, p, v);
  return check_launch("lm_head_greedy_verify launch");
}

}  // extern "C"
