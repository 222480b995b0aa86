// (a) logit processing and (c) lossless speculative sampling for gfx950.
//
// Launches per call: with a repetition penalty bitmap_kernel (each batch
// element's token history as a vocabulary bitmap) and stream_kernel, without
// one stream_reg_kernel; then fin_kernel (fin2_kernel when the units
// outnumber the CUs); then, for dense outputs only, dense_kernel.
//
// The stream kernels read every logit once: one wave per (row, 2048-element
// chunk) item, four independent waves per workgroup (stream_reg_kernel holds
// the chunk in registers only; stream_kernel stages it in LDS). A wave
//   * stages its chunk in LDS, decodes it, sets penalised tokens aside;
//   * computes the chunk max m_j, e = exp2m(fma(x, c, -mc_j)) and the chunk
//     mass M_j in the declared pairwise order; the penalised tokens' own max
//     and mass (pm_j, PM_j) from a list of them in index order that the
//     wave's lanes share (x / r or x * r);
//   * keeps the candidates: every element with RN32(x c - mref) >= -L, mref =
//     max(mc_j, pmc_j), L from a binary search on the chunk's vector maxima
//     (at most `cap` vectors reach it), lowered until at most `cap` elements
//     remain, written as (index, processed logit) into the chunk's slots;
//     and a 32-byte record.
// fin_kernel finalises one unit per workgroup. A unit is a pair (target row
// i, draft row i) of a batch element (spec, i < k), the bonus target row
// (spec, i = k) or one row (sample / dense):
//   * the records and every candidate slot of both rows are loaded together;
//     row constants mcmax, S and per chunk the largest p a non-candidate can
//     have (exact, because p is monotone in the logit);
//   * every candidate's p = RN(exp2p(RN32(fma64(x, cd, -mcmax))) / S) into
//     LDS, the exact top-p cutoffs of both rows by shared three-round radix
//     selects on the binary32 bits of p with 2^-46 fixed-point masses
//     (exact-mass top-p: sort + cumsum + searchsorted of
//     distributions.py:59-70 with the cumulative mass summed exactly; a row
//     whose binary32 cumsum in the reference crosses top_p at another index
//     than the exact mass keeps the exact set there);
//   * valid when the cutoff exceeds every chunk's non-candidate bound; else
//     the chunks whose bound reaches it are re-read and their {p >= cutoff}
//     replaces their candidates (exact, since that cutoff is a lower bound of
//     the row's); else the whole row is selected by passes over it;
//   * spec: the accept bit of x_i, the residual draw on rejection (draft
//     probabilities looked up through an LDS hash of the draft's entries),
//     the bonus draw for i = k; the last of the k+1 units of a batch element
//     writes its accepted length and tokens. sample: the draw. dense: the
//     statistics.
// The arithmetic is the declared arithmetic of ls_numerics.hpp, restated by
// oracle/sampling.py and oracle/native/ls_oracle.c, so every output is
// bit-identical to the oracle's.
#include <mutex>

#include "ls_common.hpp"
#include "ls_numerics.hpp"
#include "ls_runtime.hpp"

namespace ls {
namespace {

constexpr int kChunk = 2048;               // softmax chunk (declared arithmetic)
constexpr int kWG = 256;                   // stream_kernel workgroup
constexpr int kNW = kWG / kWave;           // waves per workgroup
constexpr int kMaxChunks = 128;            // vocab <= 262144
constexpr int kMaxVocab = kMaxChunks * kChunk;
constexpr int kRowCap = 2048;              // LDS entries per row in the finaliser
constexpr int kMaxLevel = 31;              // candidate levels: e >= 2^-L, L in [0, 31]
constexpr int64_t kMaxRows = 65536;
constexpr int64_t kMaxSpecBatch = 16384;
constexpr uint32_t kNone = 0xffffffffu;

enum Mode : int { kModeSpec = 0, kModeSample = 1, kModeDense = 2 };
// kChunkPenCands: penalised candidates follow the others, in no particular order
enum ChunkFlag : uint32_t { kChunkOverflow = 1u, kChunkHasTok = 2u, kChunkPenCands = 4u };
enum RowFlag : uint32_t { kRowFiltered = 1u, kRowList = 2u, kRowEmpty = 4u, kRowRefilled = 8u };

// Per-chunk result of the streaming pass.
struct ChunkRec {
  float m;          // max of the non-penalised x (-inf if none)
  float mass;       // M_j
  float pm;         // max of the penalised x (-inf if none)
  float pmass;      // PM_j
  int32_t level;    // candidates: RN32(x c - max(mc_j, pmc_j)) >= -level; -1 with kChunkOverflow
  uint32_t n;       // candidates written
  float xtok;       // processed logit of the row's draft token (kChunkHasTok)
  uint32_t flags;
};
static_assert(sizeof(ChunkRec) == 32, "ChunkRec layout");

// Published per-row statistics (dense mode).
struct RowStat {
  float mcmax, s, cutoff, mass;  // mass: binary32 retained mass (1 when unfiltered)
  uint32_t flags, pad;
  uint64_t mass_fx;
};
static_assert(sizeof(RowStat) == 32, "RowStat layout");

struct Params {
  const char* base0;           // target / row logits
  int64_t bstride0, pstride0;  // bytes
  const char* base1;           // draft logits (spec)
  int64_t bstride1, pstride1;
  int mode, k, rpg;            // rpg: rows per group (spec 2k+1, else 1)
  int vocab, nch, cap;         // chunks per row, candidate slots per chunk
  int items, groups, units;
  float c;                     // RN32(cd)
  double cd;                   // RN64(log2(e) / T)
  float pen;                   // repetition penalty
  int use_pen;
  float top_p;                 // >= 1: unfiltered
  int top_k;                   // 0: off, else 1 <= top_k < vocab
  const float* top_p_rows;     // optional per-row top_p (dense mode)
  const int32_t* hist;
  int64_t hist_stride;
  const int32_t* hist_len;
  int bm_words;                // bitmap words per group (nch * 64)
  // spec
  const int64_t* draft_tokens;  // [B, k]
  const float* uniforms;        // [B, 2k+1]
  int32_t* accept_len;
  int64_t* tokens;              // [B, k+1]
  // sample
  const float* row_uniforms;
  int64_t* row_tokens;
  // dense
  float* probs_out;
  int64_t probs_stride;
  float* filt_out;
  int64_t filt_stride;
  float* cutoff_out;
  float* mass_out;
  int vec_out;         // the rows of the dense outputs are 16-byte aligned
  int zero_out;        // filtered rows: zeros by the streaming pass, the support by the finaliser
  // workspace
  uint32_t* grp_cnt;   // [groups] (spec)
  ChunkRec* recs;      // [rows * nch]
  uint64_t* cands;     // [rows * nch * cap] of (index << 32 | bits(x))
  RowStat* stats;      // [rows]
  uint64_t* words;     // [groups * (k+1)] (spec)
  uint32_t* bitmap;    // [groups * bm_words]
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Declared arithmetic pieces
// ---------------------------------------------------------------------------

// 2^t for probabilities: the exp2q reduction with the polynomial in binary64,
// rounded once (monotone over every binary32 t). Coefficients: a discrete
// minimax fit of 2^r on [-1/2, 1/2] in relative error by linear programming,
// with p(0) = 1 and p(1/2) = 2 p(-1/2), kept in binary64 (oracle/exp2_fit.py).
constexpr double kP1 = 0x1.62e42920369e4p-1;
constexpr double kP2 = 0x1.ebf9bb8a817edp-3;
constexpr double kP3 = 0x1.c6b752e01b730p-5;
constexpr double kP4 = 0x1.3cea874a3c256p-7;
constexpr double kP5 = 0x1.5bba1349df24ap-10;

__device__ __forceinline__ float exp2p(float t) {
  const float tc = __builtin_fmaxf(t, kExp2Floor);
  const float kf = __builtin_rintf(tc);
  const double r = static_cast<double>(tc - kf);
  double q = kP5;
  q = __builtin_fma(q, r, kP4);
  q = __builtin_fma(q, r, kP3);
  q = __builtin_fma(q, r, kP2);
  q = __builtin_fma(q, r, kP1);
  q = __builtin_fma(q, r, 1.0);
  return __builtin_ldexpf(static_cast<float>(q), static_cast<int>(kf));
}

// The exponent of p: RN32(fma64(x, cd, -mcmax)).
__device__ __forceinline__ float p_exponent(float x, double cd, float mcmax) {
  return static_cast<float>(__builtin_fma(static_cast<double>(x), cd, -static_cast<double>(mcmax)));
}

// p(x) = S > 0 ? RN(exp2p(t) / S) : 0 (correctly rounded division).
__device__ __forceinline__ float p_of(float x, double cd, float mcmax, float s) {
  if (!(s > 0.0f)) return 0.0f;
  return exp2p(p_exponent(x, cd, mcmax)) / s;
}

// Repetition penalty of one logit (transformers' closed form).
__device__ __forceinline__ float penalise(float x, float pen) { return x < 0.0f ? x * pen : x / pen; }

// Row constants of one processed row.
struct RowK {
  float mcmax, s;
  double cd;
};

__device__ __forceinline__ float pval(const RowK& k, float x) { return p_of(x, k.cd, k.mcmax, k.s); }

__device__ __forceinline__ uint64_t pack_u32(uint32_t lo, uint32_t hi) {
  return static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32);
}

// The next binary32 value above t (t finite).
__device__ __forceinline__ float next_up(float t) {
  const uint32_t b = __float_as_uint(t);
  if (b == 0x80000000u || b == 0u) return __uint_as_float(1u);
  return __uint_as_float((b & 0x80000000u) ? b - 1u : b + 1u);
}

// ---------------------------------------------------------------------------
// Wave sums in the declared pairwise order (lanes 2i and 2i+1 first, then
// pairs of those ...): quad_perm swaps for distance 1 and 2, then the half-row
// and row mirrors (equivalent to distance 4 and 8 once every quad / half-row
// holds one value), then the row broadcasts.
// ---------------------------------------------------------------------------
constexpr int kDppQuadXor1 = 0xB1;      // quad_perm [1,0,3,2]
constexpr int kDppQuadXor2 = 0x4E;      // quad_perm [2,3,0,1]
constexpr int kDppRowHalfMirror = 0x141;
constexpr int kDppRowMirror = 0x140;

template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float v) {
  return __uint_as_float(dpp32<CTRL, ROWS>(0u, __float_as_uint(v))) + v;
}

// Pairwise sum over the 64 lanes (wave-uniform result).
__device__ __forceinline__ float wave_tree_sum(float v) {
  v = dpp_add<kDppQuadXor1, 0xf>(v);
  v = dpp_add<kDppQuadXor2, 0xf>(v);
  v = dpp_add<kDppRowHalfMirror, 0xf>(v);
  v = dpp_add<kDppRowMirror, 0xf>(v);
  v = dpp_add<kDppRowBcast15, 0xa>(v);  // rows 1, 3: r0 + r1, r2 + r3
  v = dpp_add<kDppRowBcast31, 0xc>(v);  // row 3: (r0 + r1) + (r2 + r3)
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(v), kWave - 1));
}

// Pairwise sum of N values held by one lane, adjacent pairs first.
template <int N>
__device__ __forceinline__ float lane_tree_sum(float (&a)[N]) {
#pragma unroll
  for (int w = 1; w < N; w *= 2) {
#pragma unroll
    for (int i = 0; i < N; i += 2 * w) a[i] = a[i] + a[i + w];
  }
  return a[0];
}

// ---------------------------------------------------------------------------
// Shared memory of stream_kernel: each wave's chunk as loaded
// ---------------------------------------------------------------------------
template <int DT>
struct StreamSh {
  u32x4 stage[kNW][kChunk / Elem<DT>::kPerVec];  // the chunk's 16-byte vectors
};


// ---------------------------------------------------------------------------
// Items
// ---------------------------------------------------------------------------
struct Item {
  int unit, row, chunk, group;
  int64_t tok;
  const char* rowp;
};

__device__ __forceinline__ Item item_of(const Params& p, int it) {
  Item r;
  if (p.mode == kModeSpec) {
    const int per_g = p.rpg * p.nch;
    const int g = it / per_g;
    const int q = it - g * per_g;
    const int two = 2 * p.nch;
    int i, slot, chunk;
    if (q < p.k * two) {
      i = q / two;
      const int w = q - i * two;
      slot = w >= p.nch ? 1 : 0;
      chunk = w - slot * p.nch;
    } else {
      i = p.k;
      slot = 0;
      chunk = q - p.k * two;
    }
    r.unit = g * (p.k + 1) + i;
    r.group = g;
    r.chunk = chunk;
    r.row = g * p.rpg + (slot == 0 ? i : p.k + 1 + i);
    r.rowp = slot == 0 ? p.base0 + g * p.bstride0 + i * p.pstride0 : p.base1 + g * p.bstride1 + i * p.pstride1;
    r.tok = i < p.k ? p.draft_tokens[static_cast<int64_t>(g) * p.k + i] : -1;
  } else {
    const int row = it / p.nch;
    r.unit = row;
    r.group = row;
    r.row = row;
    r.chunk = it - row * p.nch;
    r.rowp = p.base0 + static_cast<int64_t>(row) * p.bstride0;
    r.tok = -1;
  }
  return r;
}

// Logits row of row id r (spec rows: targets 0..k, then drafts 0..k-1).
__device__ __forceinline__ const char* row_ptr(const Params& p, int r) {
  if (p.mode != kModeSpec) return p.base0 + static_cast<int64_t>(r) * p.bstride0;
  const int g = r / p.rpg, jr = r - g * p.rpg;
  if (jr <= p.k) return p.base0 + g * p.bstride0 + jr * p.pstride0;
  return p.base1 + g * p.bstride1 + (jr - p.k - 1) * p.pstride1;
}

__device__ __forceinline__ const uint32_t* row_bitmap(const Params& p, int r) {
  return p.use_pen ? p.bitmap + static_cast<int64_t>(r / p.rpg) * p.bm_words : nullptr;
}

__device__ __forceinline__ float row_top_p(const Params& p, int r) {
  return p.top_p_rows ? p.top_p_rows[r] : p.top_p;
}

template <int DT>
__device__ __forceinline__ float decode_bits(uint32_t b) {
  return bits_to_float<DT>(b);
}

// Processed logit of element i of a row read from global memory.
template <int DT>
__device__ __forceinline__ float load_x(const Params& p, const char* rowp, const uint32_t* bm, int64_t i) {
  float x = decode_bits<DT>(load_bits<DT>(rowp, i));
  if (bm && ((bm[i >> 5] >> (i & 31)) & 1u)) x = penalise(x, p.pen);
  return x;
}

// ===========================================================================
// bitmap_kernel: the penalty bitmap of each group's token history
// ===========================================================================
constexpr int kBmB = 1024;
constexpr int kBmU = 8;  // history ids loaded per thread before any is used

__global__ __launch_bounds__(kBmB) void bitmap_kernel(const Params p) {
  __shared__ uint32_t bm[kMaxVocab / 32];
  const int t = threadIdx.x;
  const int64_t g = blockIdx.x;
  const int words = p.bm_words;
  // the length's load is in flight while the bitmap is cleared; a length
  // past the row stride (or negative) is clamped to the row
  const int64_t n_raw = p.hist_len[g];
  const int n = static_cast<int>(n_raw < 0 ? 0 : (n_raw > p.hist_stride ? p.hist_stride : n_raw));
  for (int w = t; w < words; w += kBmB) bm[w] = 0u;
  __syncthreads();
  const int32_t* h = p.hist + g * p.hist_stride;
  // every id of a batch of kBmU * kBmB is loaded before any is set, so a
  // history of up to 8192 ids costs one global-load latency, not one per
  // kBmB ids
  for (int i0 = 0; i0 < n; i0 += kBmB * kBmU) {
    int32_t id[kBmU];
#pragma unroll
    for (int u = 0; u < kBmU; ++u) {
      const int i = i0 + u * kBmB + t;
      id[u] = i < n ? h[i] : -1;
    }
#pragma unroll
    for (int u = 0; u < kBmU; ++u) {
      if (static_cast<unsigned>(id[u]) < static_cast<unsigned>(p.vocab))
        __hip_atomic_fetch_or(&bm[id[u] >> 5], 1u << (id[u] & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __syncthreads();
  uint32_t* out = p.bitmap + g * words;
  for (int w = t; w < words; w += kBmB) out[w] = bm[w];
}

// ===========================================================================
// Streaming pass
// ===========================================================================

// Loads of one item (lanes past the chunk end re-read its last vector), plus,
// with a penalty, the chunk's bitmap word t for lane t.
template <int DT, int NVC>
__device__ __forceinline__ void load_item(const Params& p, const Item& I, u32x4 (&d)[NVC], uint32_t& pw) {
  constexpr int EPV = Elem<DT>::kPerVec;
  const int c0 = I.chunk * kChunk;
  const int nel = p.vocab - c0 < kChunk ? p.vocab - c0 : kChunk;
  const int nvc = nel / EPV;
  const u32x4* src = reinterpret_cast<const u32x4*>(I.rowp) + c0 / EPV;
  const int t = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
    const int v = u * kWave + t;
    d[u] = __builtin_nontemporal_load(src + (v < nvc ? v : nvc - 1));
  }
  pw = 0u;
  if (p.use_pen) pw = p.bitmap[static_cast<int64_t>(I.group) * p.bm_words + I.chunk * (kChunk / 32) + t];
}

// Element li of the chunk staged in LDS, decoded.
template <int DT>
__device__ __forceinline__ float staged(const u32x4* st, int li) {
  if constexpr (DT == F32) {
    return __uint_as_float(reinterpret_cast<const uint32_t*>(st)[li]);
  } else {
    return decode_bits<DT>(reinterpret_cast<const uint16_t*>(st)[li]);
  }
}

// exp2q(t) for a finite t: the clamp at -200 changes nothing there (both
// forms give 0 below -200), so it is left out; a -inf or NaN operand gives
// NaN, which the caller detects in the sum.
__device__ __forceinline__ float exp2q_finite(float t) {
  const float kf = __builtin_rintf(t);
  const float r = t - kf;
  float q = kExp2C5;
  q = __builtin_fmaf(q, r, kExp2C4);
  q = __builtin_fmaf(q, r, kExp2C3);
  q = __builtin_fmaf(q, r, kExp2C2);
  q = __builtin_fmaf(q, r, kExp2C1);
  q = __builtin_fmaf(q, r, kExp2C0);
  int k;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(k) : "v"(kf));  // saturating conversion
  return __builtin_ldexpf(q, k);
}

// One chunk item, processed by wave w: its candidates and its record are
// stored (read by fin_kernel, after this kernel). The item is wave-uniform.
// The chunk's penalised elements (bits hb[u] of lane t's vector u) listed in
// index order into hl (chunk element indices); returns their number. Element
// e of vector u of lane t is chunk element (64 u + t) EPV + e, so index order
// is (u, lane, e): one packed wave scan of the per-vector counts (16-bit
// fields, four vectors per 64-bit word) places every lane's elements.
template <int EPV, int NVC>
__device__ __forceinline__ uint32_t list_hits(const uint32_t (&hb)[NVC], uint16_t* hl) {
  static_assert(NVC % 4 == 0 || NVC == 4, "vectors per lane");
  const int t = threadIdx.x & (kWave - 1);
  uint32_t base = 0;
#pragma unroll
  for (int u0 = 0; u0 < NVC; u0 += 4) {
    uint64_t packed = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) packed |= static_cast<uint64_t>(__builtin_popcount(hb[u0 + q])) << (16 * q);
    const uint64_t incl = wave_scan_add_u64(packed);
    const uint64_t tot = lane_bcast_u64(incl, kWave - 1);
    const uint64_t excl = incl - packed;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t pos = base + static_cast<uint32_t>((excl >> (16 * q)) & 0xffffu);
      uint32_t bits = hb[u0 + q];
      while (bits) {
        const int e = __builtin_ctz(bits);
        bits &= bits - 1u;
        hl[pos++] = static_cast<uint16_t>(((u0 + q) * kWave + t) * EPV + e);
      }
      base += static_cast<uint32_t>((tot >> (16 * q)) & 0xffffu);
    }
  }
  return base;
}

template <int DT>
__device__ __forceinline__ void stream_item(const Params& p, StreamSh<DT>& sh, int w, const Item& I,
                                            const u32x4 (&d)[Elem<DT>::kPerVec == 4 ? 8 : 4], uint32_t pw,
                                            uint16_t* hl) {
  constexpr int EPV = Elem<DT>::kPerVec;
  constexpr int NVC = kChunk / (kWave * EPV);
  constexpr int NE = NVC * EPV;
  static_assert(NE == 32, "32 elements per lane");
  int t = threadIdx.x & (kWave - 1);
  asm volatile("" : "+v"(t));
  const int c0 = I.chunk * kChunk;
  const int nel = p.vocab - c0 < kChunk ? p.vocab - c0 : kChunk;
  const int nvc = nel / EPV;
  const bool full = nel == kChunk;  // else the row's last chunk, past-the-end lanes at -inf

  // 1. stage the chunk as loaded
  u32x4* st = sh.stage[w];
#pragma unroll
  for (int u = 0; u < NVC; ++u) st[u * kWave + t] = d[u];

  // 2. penalised elements of this lane's vectors (bits of the chunk's
  //    bitmap words, which lane t loaded as word t)
  uint32_t hb[NVC];
  bool any_hit = false;
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
    const int i0 = (u * kWave + t) * EPV;
    const uint32_t word = static_cast<uint32_t>(__shfl(static_cast<int>(pw), i0 >> 5));
    hb[u] = (u * kWave + t < nvc) ? (word >> (i0 & 31)) & ((1u << EPV) - 1u) : 0u;
  }
  uint32_t a = 0;
#pragma unroll
  for (int u = 0; u < NVC; ++u) a |= hb[u];
  any_hit = __ballot(a != 0) != 0;

  // 3. decoded logits, penalised ones and lanes past the row end at -inf
  float x[NE];
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
#pragma unroll
    for (int e = 0; e < EPV; ++e) {
      float v = vec_elem<DT>(d[u], e);
      if ((hb[u] >> e) & 1u) v = -__builtin_inff();
      x[u * EPV + e] = v;
    }
  }
  if (!full) {
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      if (u * kWave + t >= nvc) {
#pragma unroll
        for (int e = 0; e < EPV; ++e) x[u * EPV + e] = -__builtin_inff();
      }
    }
  }

  // 4. vector maxima and the chunk max (NaN-propagating first; a NaN chunk
  //    is redone ignoring NaN)
  float vm[NVC];
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
    float mv = x[u * EPV];
#pragma unroll
    for (int e = 1; e < EPV; ++e) mv = nmax(mv, x[u * EPV + e]);
    vm[u] = mv;
  }
  float mx = vm[0];
#pragma unroll
  for (int u = 1; u < NVC; ++u) mx = nmax(mx, vm[u]);
  float m = wave_max_f32(mx);
  if (m != m) {
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      float mv = -__builtin_inff();
#pragma unroll
      for (int e = 0; e < EPV; ++e) mv = x[u * EPV + e] > mv ? x[u * EPV + e] : mv;
      vm[u] = mv;
    }
    mx = vm[0];
#pragma unroll
    for (int u = 1; u < NVC; ++u) mx = mx > vm[u] ? mx : vm[u];
    m = wave_max_f32(mx);
  }
  const float c = p.c;
  const float mc = m * c;

  // 5. the exponents t = fma(x, c, -mc) (replacing x), e = exp2m(t) and the
  //    chunk mass, before the penalised sub-chunk's loops (with those in
  //    between, the compiler re-decoded the staged chunk for the exponents;
  //    C4's stream pass 41.9 -> 41.0 us in this order)
  const float nmc = -mc;
#pragma unroll
  for (int i = 0; i < NE; ++i) x[i] = __builtin_fmaf(x[i], c, nmc);
  float ea[NE];
  float mass;
  // penalised elements sit at -inf: the clamped form
#pragma unroll
  for (int i = 0; i < NE; ++i) ea[i] = exp2q(x[i]);
  mass = wave_tree_sum(lane_tree_sum(ea));

  // 6. penalised sub-chunk: the hits listed in index order, hit h handled by
  //    lane h mod 64 (its penalised value kept in a register for the first
  //    64 hits, recomputed for later ones); the max of the penalised logits
  float pm = -__builtin_inff();
  uint32_t nh = 0;
  float xp0 = -__builtin_inff();  // the penalised value of hit t
  if (any_hit) {
    nh = list_hits<EPV, NVC>(hb, hl);
    float lm = -__builtin_inff();
    for (uint32_t h0 = 0; h0 < nh; h0 += kWave) {
      const uint32_t h = h0 + t;
      if (h < nh) {
        const float xp = penalise(staged<DT>(st, hl[h]), p.pen);
        if (h0 == 0) xp0 = xp;
        lm = xp > lm ? xp : lm;
      }
    }
    pm = wave_max_f32(lm);
  }
  const float pmc = pm * c;

  // 7. the level L: candidates are the elements with RN32(x c - mref) >= -L,
  //    mref = max(mc, pmc)
  const float mref = mc > pmc ? mc : pmc;
  const bool same = mref == mc && mc > -__builtin_inff();
  const int cap = p.cap;
  int L = -1;
  uint32_t mask = 0;  // bit 31 - i <-> element i (A elements)
  uint32_t cnt = 0;
  if (mref > -__builtin_inff()) {
    const float nref = -mref;
    if (!same) {
      // the penalised maximum lies above the rest (a penalty below 1, or
      // no other finite logit): the exponents relative to mref
#pragma unroll
      for (int u = 0; u < NVC; ++u) {
#pragma unroll
        for (int e = 0; e < EPV; ++e) {
          const int li = (u * kWave + t) * EPV + e;
          float v = staged<DT>(st, li);
          if (((hb[u] >> e) & 1u) || u * kWave + t >= nvc) v = -__builtin_inff();
          x[u * EPV + e] = __builtin_fmaf(v, c, nref);
        }
      }
    }
    // a start from the vector maxima: the largest L in [0, kMaxLevel] at
    // which at most cap of the lane vectors hold a candidate (binary search;
    // the count only grows with L)
    float tv[NVC];
#pragma unroll
    for (int u = 0; u < NVC; ++u) tv[u] = __builtin_fmaf(vm[u], c, nref);
    int lo = 0, hi = kMaxLevel;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      const float th = -static_cast<float>(mid);
      uint32_t nv = 0;
#pragma unroll
      for (int u = 0; u < NVC; ++u) nv += __builtin_popcountll(__ballot(tv[u] >= th));
      if (nv <= static_cast<uint32_t>(cap)) lo = mid; else hi = mid - 1;
    }
    for (L = lo; L >= 0; --L) {
      const float th = -static_cast<float>(L);
      // four interleaved chains of eight: m_q = 2 m_q + (t >= th), a compare
      // into VCC and one add with carry each
      uint32_t mq[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < NE / 4; ++i) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
              : "+v"(mq[q]) : "v"(x[(NE / 4) * q + i]), "v"(th) : "vcc");
        }
      }
      mask = (mq[0] << 24) | (mq[1] << 16) | (mq[2] << 8) | mq[3];
      cnt = static_cast<uint32_t>(__builtin_popcount(mask));
      uint32_t own = cnt;
      uint32_t pen_cnt = 0;
      // the penalised candidates at this level count against the same slots
      for (uint32_t h0 = 0; h0 < nh; h0 += kWave) {
        const uint32_t h = h0 + t;
        const float xp = h0 == 0 ? xp0 : (h < nh ? penalise(staged<DT>(st, hl[h]), p.pen) : -__builtin_inff());
        pen_cnt += static_cast<uint32_t>(__builtin_popcountll(__ballot(h < nh && __builtin_fmaf(xp, c, nref) >= th)));
      }
      const uint32_t tot = lane_bcast_u32(wave_scan_add_u32(own), kWave - 1) + pen_cnt;
      if (tot <= static_cast<uint32_t>(cap)) {
        cnt = tot;
        break;
      }
    }
    if (L < 0) {
      mask = 0;
      cnt = 0;
    }
  }

  // 8. A candidates in index order, (chunk index << 32 | bits(x)): element e
  //    of vector u of lane t is chunk element (64 u + t) EPV + e, so vector u
  //    of every lane precedes vector u + 1. Each lane's per-vector counts,
  //    8 bits apiece (a vector's total over the lanes is at most cap <= 64),
  //    go through one wave scan.
  uint64_t* out = p.cands + (static_cast<int64_t>(I.row) * p.nch + I.chunk) * p.cap;
  uint32_t nA = 0;
  if (L >= 0) {
    uint64_t packed = 0;
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      const uint32_t vb = (mask >> (32 - (u + 1) * EPV)) & ((1u << EPV) - 1u);
      packed |= static_cast<uint64_t>(__builtin_popcount(vb)) << (8 * u);
    }
    const uint64_t incl = wave_scan_add_u64(packed);
    const uint64_t tot = lane_bcast_u64(incl, kWave - 1);
    const uint64_t excl = incl - packed;
    uint32_t base = 0;
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      // bits of vector u, element 0 in the top bit
      uint32_t vb = (mask >> (32 - (u + 1) * EPV)) & ((1u << EPV) - 1u);
      uint32_t pos = base + static_cast<uint32_t>((excl >> (8 * u)) & 0xffu);
      while (vb) {
        const int e = __builtin_clz(vb) - (32 - EPV);
        vb &= ~(1u << (EPV - 1 - e));
        const int li = (u * kWave + t) * EPV + e;
        const float xv = staged<DT>(st, li);
        out[pos] = (static_cast<uint64_t>(c0 + li) << 32) | __float_as_uint(xv);
        ++pos;
      }
      base += static_cast<uint32_t>((tot >> (8 * u)) & 0xffu);
    }
    nA = base;
  }

  // 9. penalised sub-chunk: its mass (lane-sequential in (u, element) order,
  //    then the lanes pairwise) and its candidates (appended, any order)
  const uint32_t nA_plain = nA;
  float pmass = 0.0f;
  bool overflow = L < 0 && mref > -__builtin_inff();
  if (any_hit) {
    // PM_j: hit h added by lane h mod 64 in hit order, then the lanes
    // pairwise; the penalised candidates appended in hit order
    const float npmc = -pmc;
    const float nref = -mref;
    const float th = -static_cast<float>(L);
    float acc = 0.0f;
    uint32_t nB = 0;
    for (uint32_t h0 = 0; h0 < nh; h0 += kWave) {
      const uint32_t h = h0 + t;
      const bool in = h < nh;
      const uint32_t li = in ? hl[h] : 0u;
      const float xp = h0 == 0 ? xp0 : (in ? penalise(staged<DT>(st, li), p.pen) : -__builtin_inff());
      if (in) acc = acc + exp2q(__builtin_fmaf(xp, c, npmc));
      const bool cand = in && L >= 0 && __builtin_fmaf(xp, c, nref) >= th;
      const uint64_t m = __ballot(cand);
      const uint32_t q = nB + static_cast<uint32_t>(__builtin_popcountll(m & ((1ull << t) - 1ull)));
      if (cand && nA + q < static_cast<uint32_t>(cap))
        out[nA + q] = (static_cast<uint64_t>(c0 + li) << 32) | __float_as_uint(xp);
      nB += static_cast<uint32_t>(__builtin_popcountll(m));
    }
    pmass = wave_tree_sum(acc);
    if (nA + nB > static_cast<uint32_t>(cap)) overflow = true;
    nA += nB;
  }

  // 10. the row's draft token, processed
  float xtok = 0.0f;
  const bool has_tok = I.tok >= c0 && I.tok < c0 + nel;
  if (has_tok) {
    const int li = static_cast<int>(I.tok - c0);
    float xv = staged<DT>(st, li);
    const uint32_t word = static_cast<uint32_t>(__shfl(static_cast<int>(pw), li >> 5));
    if ((word >> (li & 31)) & 1u) xv = penalise(xv, p.pen);
    xtok = xv;
  }

  // 11. the record
  if (t == 0) {
    ChunkRec* rec = p.recs + static_cast<int64_t>(I.row) * p.nch + I.chunk;
    u32x4* r128 = reinterpret_cast<u32x4*>(rec);
    const uint32_t flags = (overflow ? kChunkOverflow : 0u) | (has_tok ? kChunkHasTok : 0u) |
                           (nA > nA_plain ? kChunkPenCands : 0u);
    r128[0] = u32x4{__float_as_uint(m), __float_as_uint(mass), __float_as_uint(pm), __float_as_uint(pmass)};
    r128[1] = u32x4{static_cast<uint32_t>(overflow ? -1 : L), overflow ? 0u : nA, __float_as_uint(xtok), flags};
  }
}

// The same item without a penalty, the chunk held in registers only (no LDS):
// the raw logits stay in x[], the exponents are recomputed where they are
// needed, and a candidate's value is selected among its vector's registers.
// Records and candidates as stream_item writes them for a row without
// penalised tokens; at most 64 VGPRs, so eight waves per SIMD fit where a
// staged form (32 KB of LDS per workgroup) fits five.
template <int DT>
__device__ __forceinline__ void stream_item_reg(const Params& p, const Item& I,
                                                const u32x4 (&d)[Elem<DT>::kPerVec == 4 ? 8 : 4]) {
  constexpr int EPV = Elem<DT>::kPerVec;
  constexpr int NVC = kChunk / (kWave * EPV);
  constexpr int NE = NVC * EPV;
  static_assert(NE == 32, "32 elements per lane");
  int t = threadIdx.x & (kWave - 1);
  asm volatile("" : "+v"(t));
  const int c0 = I.chunk * kChunk;
  const int nel = p.vocab - c0 < kChunk ? p.vocab - c0 : kChunk;
  const int nvc = nel / EPV;
  const bool full = nel == kChunk;

  // decoded logits, lanes past the row end at -inf
  float x[NE];
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
#pragma unroll
    for (int e = 0; e < EPV; ++e) x[u * EPV + e] = vec_elem<DT>(d[u], e);
  }
  if (!full) {
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      if (u * kWave + t >= nvc) {
#pragma unroll
        for (int e = 0; e < EPV; ++e) x[u * EPV + e] = -__builtin_inff();
      }
    }
  }

  // vector maxima and the chunk max (NaN-propagating; a NaN chunk is redone
  // ignoring NaN)
  float vm[NVC];
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
    float mv = x[u * EPV];
#pragma unroll
    for (int e = 1; e < EPV; ++e) mv = nmax(mv, x[u * EPV + e]);
    vm[u] = mv;
  }
  float mx = vm[0];
#pragma unroll
  for (int u = 1; u < NVC; ++u) mx = nmax(mx, vm[u]);
  float m = wave_max_f32(mx);
  if (m != m) {
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      float mv = -__builtin_inff();
#pragma unroll
      for (int e = 0; e < EPV; ++e) mv = x[u * EPV + e] > mv ? x[u * EPV + e] : mv;
      vm[u] = mv;
    }
    mx = vm[0];
#pragma unroll
    for (int u = 1; u < NVC; ++u) mx = mx > vm[u] ? mx : vm[u];
    m = wave_max_f32(mx);
  }
  const float c = p.c;
  const float mc = m * c;
  const float nmc = -mc;
  const int cap = p.cap;

  // a start for the level L (no penalty: mref = mc): the largest L in
  // [0, kMaxLevel] at which at most cap of the lane vectors hold a candidate
  // (binary search; the count only grows with L). Every vector that holds a
  // candidate at L adds one to the element count, so the L the element passes
  // below settle on is the largest at which at most cap elements qualify.
  int lo = 0;
  if (mc > -__builtin_inff()) {
#pragma unroll
    for (int u = 0; u < NVC; ++u) vm[u] = __builtin_fmaf(vm[u], c, nmc);
    int hi = kMaxLevel;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      const float th = -static_cast<float>(mid);
      uint32_t nv = 0;
#pragma unroll
      for (int u = 0; u < NVC; ++u) nv += __builtin_popcountll(__ballot(vm[u] >= th));
      if (nv <= static_cast<uint32_t>(cap)) lo = mid; else hi = mid - 1;
    }
  }

  // the chunk mass: e = exp2m(fma(x, c, -mc)) in the declared lane tree,
  // summed four elements at a time (the tree's subtrees of four, then of 8,
  // 16 and 32); each group's exponents wait for the previous group's sum, so
  // at most four values are in flight beside x
  float mass;
  {
    float nv = nmc;
    float s8[NE / 8], s16 = 0.0f, s4p = 0.0f;
#pragma unroll
    for (int g = 0; g < NE / 4; ++g) {
      float e4[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) e4[q] = exp2q_finite(__builtin_fmaf(x[4 * g + q], c, nv));
      const float s4 = (e4[0] + e4[1]) + (e4[2] + e4[3]);
      if (g & 1) {
        s8[g / 2] = s4p + s4;
        if ((g / 2) & 1) {
          const float a16 = s8[g / 2 - 1] + s8[g / 2];
          s16 = (g / 4) & 1 ? s16 + a16 : a16;
        }
      } else {
        s4p = s4;
      }
      asm volatile("" : "+v"(nv) : "v"(s4));
    }
    mass = wave_tree_sum(s16);
  }
  if (mass != mass) {
    float ea[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) ea[i] = exp2q(__builtin_fmaf(x[i], c, nmc));
    mass = wave_tree_sum(lane_tree_sum(ea));
  }

  // the level L: from the start down, the first at which at most cap
  // elements satisfy RN32(x c - mc) >= -L
  int L = -1;
  uint32_t mask = 0;  // bit 31 - i <-> element i
  if (mc > -__builtin_inff()) {
    for (L = lo; L >= 0; --L) {
      const float th = -static_cast<float>(L);
      // the exponent is formed inside the same asm (one temporary per
      // element at a time): fma, compare into VCC, add with carry
      uint32_t mq[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < NE / 4; ++i) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float tx;
          asm("v_fma_f32 %1, %2, %3, %4\n\tv_cmp_ge_f32_e32 vcc, %1, %5\n\t"
              "v_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
              : "+v"(mq[q]), "=&v"(tx) : "v"(x[(NE / 4) * q + i]), "s"(c), "v"(nmc), "v"(th) : "vcc");
        }
      }
      mask = (mq[0] << 24) | (mq[1] << 16) | (mq[2] << 8) | mq[3];
      const uint32_t tot = lane_bcast_u32(wave_scan_add_u32(static_cast<uint32_t>(__builtin_popcount(mask))), kWave - 1);
      if (tot <= static_cast<uint32_t>(cap)) break;
    }
    if (L < 0) mask = 0;
  }

  // candidates in index order, (chunk index << 32 | bits(x)); a candidate's
  // value is picked among its vector's EPV registers
  uint64_t* out = p.cands + (static_cast<int64_t>(I.row) * p.nch + I.chunk) * p.cap;
  uint32_t nA = 0;
  if (L >= 0) {
    uint64_t packed = 0;
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      const uint32_t vb = (mask >> (32 - (u + 1) * EPV)) & ((1u << EPV) - 1u);
      packed |= static_cast<uint64_t>(__builtin_popcount(vb)) << (8 * u);
    }
    const uint64_t incl = wave_scan_add_u64(packed);
    const uint64_t tot = lane_bcast_u64(incl, kWave - 1);
    const uint64_t excl = incl - packed;
    uint32_t base = 0;
#pragma unroll
    for (int u = 0; u < NVC; ++u) {
      uint32_t vb = (mask >> (32 - (u + 1) * EPV)) & ((1u << EPV) - 1u);
      uint32_t pos = base + static_cast<uint32_t>((excl >> (8 * u)) & 0xffu);
      while (vb) {
        const int e = __builtin_clz(vb) - (32 - EPV);
        vb &= ~(1u << (EPV - 1 - e));
        float xv = x[u * EPV];
#pragma unroll
        for (int q = 1; q < EPV; ++q) xv = e == q ? x[u * EPV + q] : xv;
        const int li = (u * kWave + t) * EPV + e;
        out[pos] = (static_cast<uint64_t>(c0 + li) << 32) | __float_as_uint(xv);
        ++pos;
      }
      base += static_cast<uint32_t>((tot >> (8 * u)) & 0xffu);
    }
    nA = base;
  }
  const bool overflow = L < 0 && mc > -__builtin_inff();

  // the row's draft token: element li of lane (li / EPV) mod 64
  float xtok = 0.0f;
  const bool has_tok = I.tok >= c0 && I.tok < c0 + nel;
  if (has_tok) {
    const int li = static_cast<int>(I.tok - c0);
    const int r = (li / (EPV * kWave)) * EPV + li % EPV;  // register index, wave-uniform
    float xv = x[0];
#pragma unroll
    for (int q = 1; q < NE; ++q) xv = r == q ? x[q] : xv;
    xtok = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(xv), (li / EPV) & (kWave - 1)));
  }

  if (t == 0) {
    ChunkRec* rec = p.recs + static_cast<int64_t>(I.row) * p.nch + I.chunk;
    u32x4* r128 = reinterpret_cast<u32x4*>(rec);
    const uint32_t flags = (overflow ? kChunkOverflow : 0u) | (has_tok ? kChunkHasTok : 0u);
    r128[0] = u32x4{__float_as_uint(m), __float_as_uint(mass), __float_as_uint(-__builtin_inff()), 0u};
    r128[1] = u32x4{static_cast<uint32_t>(overflow ? -1 : L), overflow ? 0u : nA, __float_as_uint(xtok), flags};
  }
}

// ===========================================================================
// stream_kernel: one (row, chunk) item per wave, four independent waves per
// workgroup
// ===========================================================================
template <int DT>
__global__ __launch_bounds__(kWG) void stream_kernel(const Params p) {
  constexpr int NVC = kChunk / (kWave * Elem<DT>::kPerVec);
  __shared__ StreamSh<DT> sh;
  __shared__ uint16_t hits[kNW][kChunk];  // each wave's penalised elements
  // the wave's item, wave-uniform (its decomposition runs on the scalar unit)
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int it = static_cast<int>(blockIdx.x) * kNW + w;
  if (it >= p.items) return;  // the waves of a workgroup share no barrier
  const Item I = item_of(p, it);
  u32x4 d[NVC];
  uint32_t pw;
  load_item<DT, NVC>(p, I, d, pw);
  stream_item<DT>(p, sh, w, I, d, pw, hits[w]);
}

// Without a penalty: the register-only item, eight waves per SIMD.
template <int DT>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(8, 8))) void stream_reg_kernel(const Params p) {
  constexpr int NVC = kChunk / (kWave * Elem<DT>::kPerVec);
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int it = static_cast<int>(blockIdx.x) * kNW + w;
  if (it >= p.items) return;
  const Item I = item_of(p, it);
  u32x4 d[NVC];
  const int c0 = I.chunk * kChunk;
  const u32x4* src = reinterpret_cast<const u32x4*>(I.rowp) + c0 / Elem<DT>::kPerVec;
  const int t = threadIdx.x & (kWave - 1);
  if (p.vocab - c0 >= kChunk) {
    // a whole chunk: one lane address, the vectors at fixed offsets
#pragma unroll
    for (int u = 0; u < NVC; ++u) d[u] = __builtin_nontemporal_load(src + t + u * kWave);
  } else {
    uint32_t pw;
    load_item<DT, NVC>(p, I, d, pw);
  }
  if (p.zero_out) {
    // this chunk of the filtered row, while the loads are under way
    f32x4* out = reinterpret_cast<f32x4*>(p.filt_out + static_cast<int64_t>(I.row) * p.filt_stride + c0);
    const int nvec = (p.vocab - c0 < kChunk ? p.vocab - c0 : kChunk) / 4;
#pragma unroll
    for (int u = 0; u < kChunk / 4 / kWave; ++u) {
      if (u * kWave + t < nvec) __builtin_nontemporal_store(f32x4{0.f, 0.f, 0.f, 0.f}, out + u * kWave + t);
    }
  }
  stream_item_reg<DT>(p, I, d);
}


// ===========================================================================
// Finaliser: fin_kernel, one workgroup per unit
// ===========================================================================
constexpr int kFW = 512;               // finaliser workgroup
constexpr int kFNW = kFW / kWave;
constexpr int kEPT = kRowCap / kFW;    // entries (and candidate slots) of one row per thread
constexpr int kPosPT = kChunk / kFW;   // chunk positions per thread in a draw
constexpr int kHash = 4096;            // draft-entry hash slots (at most half in use)
constexpr int kGather = kWave;         // a crossing bucket this small is finished by one wave
constexpr int kPackedUnits = 27;       // spec: up to this many units per batch element arrive with packed bits

struct RowAux {
  float mcmax, s, cut, mass_f;   // cutoff (0 unfiltered), binary32 retained mass
  uint64_t mass_fx;
  float bmax;                    // largest non-candidate bound
  float xtok;
  float ptok;                    // p of the draft token (0 without one)
  uint32_t n;                    // LDS entries
  uint32_t flags;
  uint32_t has_tok;
  float top_p;
};

// SB: bits per select digit; rounds on bits 29 .. 30 - SB, then the next SB
// bits, then the rest (11: 29..19, 18..8, 7..0; 10: 29..20, 19..10, 9..0).
template <int SB>
struct FinShT {
  static constexpr int kBits = SB;
  static constexpr int kBins = 1 << SB;         // radix digits per select round
  static constexpr int kPer = kBins / kFW;      // bins cleared per thread
  static constexpr int kCo = kBins / (kWave / 2);  // coarse bins of 32 radix bins (one per lane)
  union {
    uint64_t bins[2][kBins];     // radix bins of the unit's two rows (zero between selects)
    uint64_t pos[kChunk];        // a draw's weights by position in the chosen chunk
    struct {
      uint64_t cum[kRowCap];     // a draw's exclusive prefix masses by entry
    } dr;
    struct {
      float pv[kRowCap];         // a residual draw's P by entry
      float dv[kRowCap];         // and max(P - Q, 0)
    } res;
  } u;
  uint64_t coarse[2][kCo];       // sums of 32 consecutive bins (zero between selects)
  uint32_t gbits[2][kGather];    // a select's crossing bucket: bits of p and masses
  uint64_t gw[2][kGather];
  uint32_t gcount[2];
  uint32_t hash[kHash];          // slot 1's entries by vocabulary index (entry + 1, 0 = empty)
  struct Entries {
    uint32_t pbits[kRowCap];     // bits of p
    uint32_t eidx[kRowCap];      // vocabulary index
  } ent[2];
  uint64_t csum[kMaxChunks];     // per-chunk weight sums of a draw
  uint32_t cstart[2][kMaxChunks];  // each chunk's entries in the LDS list
  uint32_t ccount[2][kMaxChunks];
  float bound[2][kMaxChunks];    // per-chunk bound on the p of non-candidates
  uint8_t plain[2][kMaxChunks];  // the chunk's entries are in index order
  RowAux aux[2];
  uint64_t red[4][2 * kFNW];     // block scan slots (callers alternate buffers)
  uint32_t sel[2];               // radix select: crossing digit per row
  uint32_t selok[2];             // 0: the row's entries hold less than thr
  uint64_t sel64[2][2];          // (mass above the digit, the digit's mass)
  uint32_t fbits[2];             // a finished select's cutoff bits and retained mass
  uint64_t fmass[2];
  uint32_t pick;                 // a draw's chunk (kNone at zero total)
  uint64_t pick_rem;             // the target minus the mass before that chunk
  uint32_t last;                 // spec: this unit completes its batch element
  int64_t token;
};

static_assert(sizeof(FinShT<10>) <= 80 * 1024, "two finaliser workgroups per CU");

// With two finaliser workgroups per CU (128 registers) the whole-row passes need
// every vector register, and much of what the set-up keeps for them would spill
// there (24 to 32 bytes per lane still do; the finaliser had no scratch before it
// had these passes, and B 128, k 2, V 49152 f32, top-p 0.7 took 51.3 us a call
// then, 51.0 with them).
// uniform: a value every lane holds alike, in scalar registers. thread_index: the
// thread's index, opaque to the compiler, so that addresses formed from it are
// formed again where they are used. Where one workgroup has the CU both are left
// to the compiler (C3 0.4 us shorter).
template <class FS>
__device__ __forceinline__ float uniform(float v) {
  if constexpr (FS::kBits > 10) return v;
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
template <class FS>
__device__ __forceinline__ uint64_t uniform(uint64_t v) {
  if constexpr (FS::kBits > 10) return v;
  return pack_u32(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v))),
                  static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32))));
}

template <class FS>
__device__ __forceinline__ int thread_index() {
  int t = threadIdx.x;
  if constexpr (FS::kBits <= 10) asm volatile("" : "+v"(t));
  return t;
}

// Lanes below this one whose bit is set in a wave mask.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

// Block-wide inclusive scan of one u64 per thread; tot receives the total.
// red must not be in use by a scan whose reads may still be pending.
__device__ __forceinline__ uint64_t block_incl_scan(uint64_t v, uint64_t* red, uint64_t* tot) {
  const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
  const uint64_t inc = wave_scan_add_u64(v);
  if (lane == kWave - 1) red[wid] = inc;
  __syncthreads();
  uint64_t base = 0, all = 0;
#pragma unroll
  for (int i = 0; i < kFNW; ++i) {
    const uint64_t x = red[i];
    base += i < wid ? x : 0;
    all += x;
  }
  *tot = all;
  return base + inc;
}

__device__ __forceinline__ uint64_t block_sum(uint64_t v, uint64_t* red) {
  uint64_t tot;
  block_incl_scan(v, red, &tot);
  return tot;
}

// Block-wide sums of two u64 per thread with one barrier (red: 2 kFNW slots).
__device__ __forceinline__ void block_sum2(uint64_t a, uint64_t b, uint64_t* red, uint64_t* sa, uint64_t* sb) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  a = wave_sum_u64(a);
  b = wave_sum_u64(b);
  if (lane == 0) {
    red[wid] = a;
    red[kFNW + wid] = b;
  }
  __syncthreads();
  uint64_t x = 0, y = 0;
#pragma unroll
  for (int i = 0; i < kFNW; ++i) {
    x += red[i];
    y += red[kFNW + i];
  }
  *sa = x;
  *sb = y;
}

// ---------------------------------------------------------------------------
// Draft-entry hash: open addressing over kHash slots, at most kRowCap keys.
// ---------------------------------------------------------------------------
static_assert(kHash == 4096 && kRowCap <= kHash / 2, "hash size");
__device__ __forceinline__ uint32_t hash_slot(uint32_t x) { return (x * 2654435761u) >> 20; }

template <class FS>
__device__ __forceinline__ void hash_insert(FS& f, uint32_t x, uint32_t e) {
  uint32_t h = hash_slot(x);
  for (int probe = 0; probe < kHash; ++probe) {
    if (atomicCAS(&f.hash[h], 0u, e + 1u) == 0u) return;
    h = (h + 1u) & (kHash - 1);
  }
}

// The entry of slot 1 holding vocabulary index x, or kNone.
template <class FS>
__device__ __forceinline__ uint32_t hash_find(const FS& f, uint32_t x) {
  uint32_t h = hash_slot(x);
  for (int probe = 0; probe < kHash; ++probe) {
    const uint32_t v = f.hash[h];
    if (v == 0u) return kNone;
    if (f.ent[1].eidx[v - 1u] == x) return v - 1u;
    h = (h + 1u) & (kHash - 1);
  }
  return kNone;
}

// Builds the hash over slot 1's support entries (p >= its cutoff): the only
// ones whose filtered probability is not zero. The hash is zero on entry.
template <class FS>
__device__ __forceinline__ void hash_support(FS& f) {
  const uint32_t n = f.aux[1].n;
  const float cut = f.aux[1].cut;
  for (uint32_t e = threadIdx.x; e < n; e += kFW) {
    const uint32_t pb = f.ent[1].pbits[e];
    if (pb != 0u && __uint_as_float(pb) >= cut) hash_insert(f, f.ent[1].eidx[e], e);
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// Unit set-up: records, row constants, LDS entries
// ---------------------------------------------------------------------------

// Records of chunks 2l and 2l+1 of a row for lane l (zero past nch).
struct RecPair {
  u32x4 a0, a1, b0, b1;
};

__device__ __forceinline__ RecPair load_recs(const Params& p, int row) {
  const int lane = threadIdx.x & (kWave - 1);
  const u32x4* base = reinterpret_cast<const u32x4*>(p.recs + static_cast<int64_t>(row) * p.nch);
  const u32x4 z{0u, 0u, 0u, 0u};
  RecPair r{z, z, z, z};
  const int ja = 2 * lane, jb = ja + 1;
  if (ja < p.nch) {
    r.a0 = base[2 * ja];
    r.a1 = base[2 * ja + 1];
  }
  if (jb < p.nch) {
    r.b0 = base[2 * jb];
    r.b1 = base[2 * jb + 1];
  }
  return r;
}

// Row constants and per-chunk data of row slot s from its records (wave s).
template <class FS>
__device__ __forceinline__ void row_setup(const Params& p, FS& f, int s, const RecPair& rp, float top_p) {
  const int lane = threadIdx.x & (kWave - 1);
  const int nch = p.nch;
  const float c = p.c;
  ChunkRec ra, rb;
  {
    u32x4 wa[2] = {rp.a0, rp.a1}, wb[2] = {rp.b0, rp.b1};
    __builtin_memcpy(&ra, wa, 32);
    __builtin_memcpy(&rb, wb, 32);
  }
  const int ja = 2 * lane, jb = ja + 1;
  const bool ia = ja < nch, ib = jb < nch;
  const float ninf = -__builtin_inff();
  const float mca = ia ? ra.m * c : ninf, pmca = ia ? ra.pm * c : ninf;
  const float mcb = ib ? rb.m * c : ninf, pmcb = ib ? rb.pm * c : ninf;
  float lm = mca;
  lm = pmca > lm ? pmca : lm;
  lm = mcb > lm ? mcb : lm;
  lm = pmcb > lm ? pmcb : lm;
  const float mcmax = wave_max_f32(lm);
  // slots 4l..4l+3 = (A, B) of chunks 2l and 2l+1: the first two pairwise
  // levels of the normaliser's sum
  const float sa = ia ? exp2q(mca - mcmax) * ra.mass : 0.0f;
  const float sb = ia ? exp2q(pmca - mcmax) * ra.pmass : 0.0f;
  const float sc = ib ? exp2q(mcb - mcmax) * rb.mass : 0.0f;
  const float sd = ib ? exp2q(pmcb - mcmax) * rb.pmass : 0.0f;
  const float S = wave_tree_sum((sa + sb) + (sc + sd));
  // largest p of a non-candidate: candidates are RN32(x c - mref) >= -L, so
  // every other x has x c < mref - L and p(x) <= p at the exponent
  // (mref - L) cd / c - mcmax, rounded up
  auto bound = [&](const ChunkRec& r, float mcj, float pmcj) -> float {
    if (r.flags & kChunkOverflow) return __builtin_inff();
    const float mref = mcj > pmcj ? mcj : pmcj;
    if (!(mref > ninf) || !(S > 0.0f)) return 0.0f;
    const double a = static_cast<double>(mref) - static_cast<double>(r.level);
    const double tb = a * (p.cd / static_cast<double>(c)) - static_cast<double>(mcmax);
    const float tf = next_up(static_cast<float>(tb));
    return exp2p(tf) / S;
  };
  const float ba = ia ? bound(ra, mca, pmca) : 0.0f;
  const float bb = ib ? bound(rb, mcb, pmcb) : 0.0f;
  // counts read back from the workspace never exceed the chunk's slots
  const uint32_t capu = static_cast<uint32_t>(p.cap);
  const uint32_t na = ia ? (ra.n < capu ? ra.n : capu) : 0u, nb = ib ? (rb.n < capu ? rb.n : capu) : 0u;
  const uint32_t own = na + nb;
  const uint32_t incl = wave_scan_add_u32(own);
  const uint32_t ntot = lane_bcast_u32(incl, kWave - 1);
  if (ia) {
    f.bound[s][ja] = ba;
    f.cstart[s][ja] = incl - own;
    f.ccount[s][ja] = na;
    f.plain[s][ja] = (ra.flags & kChunkPenCands) ? 0 : 1;
  }
  if (ib) {
    f.bound[s][jb] = bb;
    f.cstart[s][jb] = incl - own + na;
    f.ccount[s][jb] = nb;
    f.plain[s][jb] = (rb.flags & kChunkPenCands) ? 0 : 1;
  }
  const float bmax = wave_max_f32(ba > bb ? ba : bb);
  const bool ta = ia && (ra.flags & kChunkHasTok), tb2 = ib && (rb.flags & kChunkHasTok);
  const uint64_t tk = __ballot(ta || tb2);
  float xt = ta ? ra.xtok : (tb2 ? rb.xtok : 0.0f);
  const int tl = tk ? __builtin_ctzll(tk) : 0;
  xt = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__float_as_uint(xt), tl));
  const float pt = tk ? p_of(xt, p.cd, mcmax, S) : 0.0f;
  if (lane == 0) {
    RowAux& a = f.aux[s];
    a.mcmax = mcmax;
    a.s = S;
    a.bmax = bmax;
    a.n = ntot;
    a.has_tok = tk != 0;
    a.xtok = xt;
    a.ptok = pt;
    a.flags = S > 0.0f ? 0u : kRowEmpty;
    a.cut = 0.0f;
    a.mass_f = 1.0f;
    a.mass_fx = 0;
    a.top_p = top_p;
  }
}

// Candidate slots i = t + q kFW of the unit's rows, loaded before the records
// were known, placed into the LDS entries when the record's count covers
// them: entry cstart + k holds (bits of p, vocabulary index). The bits of p
// and their masses stay in eb / ew (zero for an unused slot); the rows in
// `hist` add their masses (kCount: their numbers, for the select by counts that
// comes first with top-k) to the bins of the first select round (bits 29..20
// of p) and to their coarse sums, which are zero on entry.
template <bool kCount, class FS>
__device__ __forceinline__ void place_entries(const Params& p, FS& f, int nr, const uint64_t (&sl)[2][kEPT],
                                              uint32_t hist, uint32_t (&eb)[2][kEPT], uint64_t (&ew)[2][kEPT]) {
  const int t = threadIdx.x;
  const int nslot = p.nch * p.cap;
  const int lc = __builtin_ctz(static_cast<unsigned>(p.cap));
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const RowK K{f.aux[s].mcmax, f.aux[s].s, p.cd};
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      eb[s][q] = 0u;
      ew[s][q] = 0u;
      const int i = t + q * kFW;
      if (s < nr && i < nslot) {
        const int j = i >> lc;
        const uint32_t k = static_cast<uint32_t>(i & (p.cap - 1));
        if (k < f.ccount[s][j]) {
          const uint32_t e = f.cstart[s][j] + k;
          const uint32_t idx = static_cast<uint32_t>(sl[s][q] >> 32);
          const bool ok = idx < static_cast<uint32_t>(p.vocab);  // always, for a well-formed workspace
          const uint32_t pb = ok ? __float_as_uint(pval(K, __uint_as_float(static_cast<uint32_t>(sl[s][q])))) : 0u;
          f.ent[s].pbits[e] = pb;
          f.ent[s].eidx[e] = ok ? idx : 0u;
          eb[s][q] = pb;
          ew[s][q] = fx46(__uint_as_float(pb));
        }
      }
    }
    if ((hist >> s) & 1u) {
#pragma unroll
      for (int q = 0; q < kEPT; ++q) {
        const uint64_t w = kCount ? (eb[s][q] != 0u ? 1u : 0u) : ew[s][q];
        if (w && (eb[s][q] >> 30) == 0u) {
          __hip_atomic_fetch_add(&f.u.bins[s][eb[s][q] >> (30 - FS::kBits)], w, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
          __hip_atomic_fetch_add(&f.coarse[s][eb[s][q] >> (35 - FS::kBits)], w, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Top-p cutoffs
// ---------------------------------------------------------------------------

// Exact top-p cutoffs over the entries of the rows in `mask` (bit s for slot
// s): c_s = max{v : sum over entries with p >= v of fx46(p) >= thr_s}. Every
// thread holds kEPT entries of each row in registers (eb: bits of p, ew: their
// masses; zero for an unused slot), any partition of the row's entries over
// the threads. Radix rounds on the bits of p (p <= 1, so bits < 2^30): bits
// 29..20, 19..10 and 9..0. In each round wave s alone finds row s's crossing
// digit (lane l < 32 reads the coarse sum of the 32 bins below FS::kBins - 32 l,
// which every mass added to a bin also went into; one wave scan finds the
// lane and a second one, over those 32 bins, the digit); the entries of that
// digit are then gathered and, when at most kGather, finished by wave s,
// which also stores the row's cutoff and retained mass in f.aux[s] (set[s];
// not with kStore false, for a select by counts). ok[s] is false
// when the entries hold less than thr_s. Entries of zero mass never decide
// the cutoff and are skipped. hist: round 0's masses are already in the bins
// and coarse bins (which are otherwise cleared here first).
template <bool kStore = true, class FS>
__device__ __forceinline__ void select_entries(FS& f, uint32_t mask, const uint64_t (&thr)[2],
                                               const uint32_t (&eb)[2][kEPT], const uint64_t (&ew)[2][kEPT],
                                               bool hist, float (&cut)[2], uint64_t (&mass)[2],
                                               bool (&ok)[2], bool (&set)[2]) {
  const int t = thread_index<FS>(), lane = t & (kWave - 1), wid = t / kWave;
  bool live[2] = {(mask & 1u) != 0, (mask & 2u) != 0};
  ok[0] = live[0];
  ok[1] = live[1];
  set[0] = false;
  set[1] = false;
  if (!hist) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (live[s]) {
#pragma unroll
        for (int q = 0; q < FS::kPer; ++q) f.u.bins[s][FS::kPer * t + q] = 0;
        if (t < FS::kCo) f.coarse[s][t] = 0;
      }
    }
    __syncthreads();
  }
  uint32_t prefix[2] = {0u, 0u};  // the resolved high bits: bits >> hshift
  uint64_t above[2] = {0u, 0u};   // mass strictly above the resolved prefix
  for (int round = 0; round < 3 && (live[0] || live[1]); ++round) {
    const int shift = round == 0 ? 30 - FS::kBits : (round == 1 ? 30 - 2 * FS::kBits : 0);
    const int width = round == 2 ? 30 - 2 * FS::kBits : FS::kBits;
    const int hshift = shift + width;
    // 1. masses into the bins of this round's digit
    if (round > 0 || !hist) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (!live[s]) continue;
#pragma unroll
        for (int q = 0; q < kEPT; ++q) {
          if (ew[s][q] && (eb[s][q] >> hshift) == prefix[s]) {
            const uint32_t dg = (eb[s][q] >> shift) & ((1u << width) - 1u);
            __hip_atomic_fetch_add(&f.u.bins[s][dg], ew[s][q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(&f.coarse[s][dg >> 5], ew[s][q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
      }
      __syncthreads();
    }
    // 2. the crossing digit of row s, by wave s
    if (wid < 2 && live[wid]) {
      const int s = wid;
      const uint64_t* bs = f.u.bins[s];
      // lane l < FS::kCo: the 32 bins below FS::kBins - 32 l, whose sum is
      // coarse[FS::kCo - 1 - l]
      const uint64_t own = lane < FS::kCo ? f.coarse[s][FS::kCo - 1 - lane] : 0u;
      const uint64_t incl = wave_scan_add_u64(own);
      const uint64_t tot = lane_bcast_u64(incl, kWave - 1);
      const uint64_t need = thr[s] - above[s];  // > 0: above < thr
      if (tot < need) {
        if (lane == 0) f.selok[s] = 0u;
      } else {
        const int c = __builtin_ctzll(__ballot(incl >= need));
        const uint64_t before = lane_bcast_u64(incl - own, c);
        const int bin = FS::kBins - 1 - kWave / 2 * c - lane;
        const uint64_t v = lane < kWave / 2 ? bs[bin] : 0u;
        const uint64_t inc2 = wave_scan_add_u64(v);
        const int d = __builtin_ctzll(__ballot(lane < kWave / 2 && before + inc2 >= need));
        if (lane == d) {
          f.sel[s] = static_cast<uint32_t>(bin);
          f.sel64[s][0] = above[s] + before + inc2 - v;
          f.sel64[s][1] = v;
          f.selok[s] = 1u;
        }
      }
      if (lane == 0) f.gcount[s] = 0;
    }
    __syncthreads();
    // 3. the crossing digit's entries gathered (ballot-compacted, one LDS
    //    atomic per wave and row); the bins cleared for the next round (their
    //    reads are all before the last barrier)
    uint64_t binmass[2] = {0u, 0u};
    uint64_t gm[2][kEPT];
    uint32_t gcnt[2] = {0u, 0u};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (!live[s]) continue;
      if (!f.selok[s]) {
        // the entries hold less than thr (uniform over the workgroup)
        live[s] = false;
        ok[s] = false;
        continue;
      }
      prefix[s] = (prefix[s] << width) | f.sel[s];
      above[s] = f.sel64[s][0];
      binmass[s] = f.sel64[s][1];
#pragma unroll
      for (int q = 0; q < kEPT; ++q) {
        gm[s][q] = __ballot(ew[s][q] && (eb[s][q] >> shift) == prefix[s]);
        gcnt[s] += static_cast<uint32_t>(__builtin_popcountll(gm[s][q]));
      }
#pragma unroll
      for (int q = 0; q < FS::kPer; ++q) f.u.bins[s][FS::kPer * t + q] = 0;
      if (t < FS::kCo) f.coarse[s][t] = 0;
    }
    uint32_t gbase[2] = {0u, 0u};
    if (lane == 0) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (live[s] && gcnt[s])
          gbase[s] = __hip_atomic_fetch_add(&f.gcount[s], gcnt[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (!live[s] || !gcnt[s]) continue;
      uint32_t at = lane_bcast_u32(gbase[s], 0);
#pragma unroll
      for (int q = 0; q < kEPT; ++q) {
        const uint32_t k = at + lanes_below(gm[s][q]);
        if (((gm[s][q] >> lane) & 1ull) && k < static_cast<uint32_t>(kGather)) {
          f.gbits[s][k] = eb[s][q];
          f.gw[s][k] = ew[s][q];
        }
        at += static_cast<uint32_t>(__builtin_popcountll(gm[s][q]));
      }
    }
    __syncthreads();
    // 4. a small bucket is finished by wave s: lane l holds entry l, its
    //    mass at and above it A_l; the cutoff is the largest p with A >= thr
    bool fin[2] = {false, false};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (!live[s]) continue;
      const uint32_t cnt = f.gcount[s];
      if (cnt <= static_cast<uint32_t>(kGather)) {
        fin[s] = true;
        if (wid == s) {
          const bool in = static_cast<uint32_t>(lane) < cnt;
          const uint32_t b = in ? f.gbits[s][lane] : 0u;
          uint64_t A = above[s];
          for (uint32_t j0 = 0; j0 < cnt; j0 += 8) {
            uint32_t bj[8];
            uint64_t wj[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const bool v = j0 + q < cnt;
              bj[q] = f.gbits[s][v ? j0 + q : 0];
              wj[q] = v ? f.gw[s][j0 + q] : 0u;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) A += bj[q] >= b ? wj[q] : 0u;
          }
          const bool good = in && A >= thr[s];
          const uint64_t best = wave_max_u64(good ? b : 0u);
          const uint64_t at = wave_max_u64(good && b == static_cast<uint32_t>(best) ? A : 0u);
          if (lane == 0) {
            f.fbits[s] = static_cast<uint32_t>(best);
            f.fmass[s] = at;
            if (kStore) {
              RowAux& a = f.aux[s];
              a.flags = kRowFiltered | kRowList;
              a.cut = __uint_as_float(static_cast<uint32_t>(best));
              a.mass_fx = at;
              a.mass_f = mass_to_f32(at);
            }
          }
        }
      } else if (round == 2) {
        // every entry of the bucket has the same bits
        cut[s] = __uint_as_float(prefix[s]);
        mass[s] = above[s] + binmass[s];
        live[s] = false;
      }
    }
    if (fin[0] || fin[1]) {
      __syncthreads();
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (!fin[s]) continue;
        cut[s] = __uint_as_float(f.fbits[s]);
        mass[s] = f.fmass[s];
        live[s] = false;
        set[s] = kStore;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Whole-row passes: rows whose support is not among their candidates
// ---------------------------------------------------------------------------
constexpr int kQueue = kHash / kFNW;  // words of LDS (the draft hash's) a wave queues logits in

// Logits that bracket an element's p without forming it. p = RN(e / S) with
// e = RN(E), E the unrounded power of two: a relative rounding moves p by 2^-24,
// but where p or e is subnormal it moves it by up to half of 2^-149, any number
// of octaves of the smallest ones. So p >= v means e / S >= v - h and
// E >= S (v - h) - h with h = 2^-150, and p < v means e / S <= v - h and
// E <= S (v - h) + h (both exact in binary64 where h matters). The relative
// roundings (of p, of E's polynomial and exponent: under 2^-16 octaves) are
// covered by 2^-10 octaves of slack.
constexpr double kHalfUlp0 = 0x1p-150;
constexpr double kLogSlack = 0x1p-10;

// A logit no element with p >= v lies below.
__device__ __forceinline__ float x_floor(const RowK& K, float v) {
  const double s = static_cast<double>(K.s);
  const double e = __builtin_fma(s, static_cast<double>(v) - kHalfUlp0, -kHalfUlp0);
  if (!(e > 0.0)) return -__builtin_inff();
  const float x = static_cast<float>((log2(e) - kLogSlack + static_cast<double>(K.mcmax)) / K.cd);
  return -next_up(-x);
}

// A logit no element with p < v lies above (v > 0).
__device__ __forceinline__ float x_ceil(const RowK& K, float v) {
  const double s = static_cast<double>(K.s);
  const double e = __builtin_fma(s, static_cast<double>(v) - kHalfUlp0, kHalfUlp0);
  return next_up(static_cast<float>((log2(e) + kLogSlack + static_cast<double>(K.mcmax)) / K.cd));
}

// Orders a wave's own LDS traffic (the LDS serves a wave in order; this keeps
// the compiler from moving it).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// What travels with a queued logit: nothing, the second row's logit at the
// same index, or the index.
enum Beside : int { kAlone = 0, kPairX = 1, kIndex = 2 };

// A piece of a row as one wave loads it: four vectors per lane, vector u of
// lane t (words 4 u .. of its registers) the piece's vector 64 u + t (lanes past
// the row's end re-read its last vector); 1024 elements in f32 (two pieces to a
// chunk), 2048 in 16 bits. bits: with a penalty, the bitmap word of each vector.
// The passes below loop over a piece's elements a few at a time with a uniform
// register index, not unrolled: the same time, and a third of the code.
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
template <int DT>
struct Piece {
  static constexpr int kVecs = 4;
  static constexpr int kElems = kVecs * kWave * Elem<DT>::kPerVec;
  static constexpr int kPerChunk = kChunk / kElems;
  u32x16 d;
  u32x4 bits;
};

// Piece q of a row (element q * kElems on), or its vectors u0 .. u1 - 1 only (the
// others' registers then hold vector u0 again: with a branch around each load
// instead, the loads of a whole piece waited for one another; B 64, k 2, V 49152
// f32, top-p 0.9, 157 us a call against 147).
template <int DT>
__device__ __forceinline__ void load_piece(const Params& p, const char* rowp, const uint32_t* bm, int q, Piece<DT>& c,
                                           int u0 = 0, int u1 = Piece<DT>::kVecs) {
  constexpr int EPV = Elem<DT>::kPerVec;
  const int lane = threadIdx.x & (kWave - 1);
  const int v0 = q * Piece<DT>::kElems / EPV, nv = p.vocab / EPV;
  const u32x4* src = reinterpret_cast<const u32x4*>(rowp);
#pragma unroll
  for (int u = 0; u < Piece<DT>::kVecs; ++u) {
    const int at = v0 + (u < u0 || u >= u1 ? u0 : u) * kWave + lane, v = at < nv ? at : nv - 1;
    const u32x4 x = src[v];
#pragma unroll
    for (int k = 0; k < 4; ++k) c.d[4 * u + k] = x[k];
    if (bm) c.bits[u] = bm[(v * EPV) >> 5];
  }
}

// kStep elements of a lane from a piece's registers, processed: those from its
// kStep * st 'th on, whose index in the row is *i0 onwards.
template <int DT, int kStep>
__device__ __forceinline__ void piece_step(const Params& p, const Piece<DT>& c, u32x4 bits, bool pen, int q, int st,
                                           float (&x)[kStep], int* i0) {
  constexpr int EPV = Elem<DT>::kPerVec;
  constexpr int kPerWord = EPV / 4;
  const int lane = threadIdx.x & (kWave - 1);
  const int u = st * kStep / EPV, e0 = st * kStep % EPV;
  const int i = q * Piece<DT>::kElems + (u * kWave + lane) * EPV + e0;
#pragma unroll
  for (int w = 0; w < kStep / kPerWord; ++w) {
    const uint32_t word = c.d[st * (kStep / kPerWord) + w];
    if constexpr (DT == F32) {
      x[w] = __uint_as_float(word);
    } else {
      x[2 * w] = bits_to_float<DT>(word & 0xffffu);
      x[2 * w + 1] = bits_to_float<DT>(word >> 16);
    }
  }
  if (pen) {
    const uint32_t pb = bits[u] >> (i & 31);
#pragma unroll
    for (int e = 0; e < kStep; ++e) x[e] = (pb >> e) & 1u ? penalise(x[e], p.pen) : x[e];
  }
  *i0 = i;
}

// What fn of a pass gets at a time: kN queued logits per lane, so that with
// one workgroup per CU (two waves per SIMD) the exact p of several are under
// way together; with two workgroups one (their registers are few, and the other
// waves cover a dependent chain's latency).
template <int kBeside, class FS>
struct Batch {
  static constexpr int kN = FS::kBits > 10 ? (kBeside == kAlone ? 4 : 2) : 1;
  float x[kN];
  uint32_t beside[kN];
  bool valid[kN];
};

// A piece as piece_pass takes it: kStep elements of every lane, kSteps times.
template <int DT, int kBeside>
struct Pass {
  static constexpr int kStep = kBeside == kAlone ? 4 : 2;  // elements between drains
  static constexpr int kSteps = Piece<DT>::kElems / kWave / kStep;
};

// One wave over loaded piece q of a row: fn(batch) on the elements whose
// processed logit lies in [lo, hi] (a NaN counts as inside), in no particular
// order. fn evaluates p exactly (some 32 instructions, in binary64), and a pass
// wants few of the elements, so each element's test only appends it to the
// wave's queue in LDS and fn runs on full waves of queued ones. The piece's
// elements are all done on return. Of the piece's steps st0 .. st1 - 1 are taken.
// kWhole: with lo = -inf every element is wanted, and goes to fn without the
// queue.
template <int DT, int kBeside, bool kWhole, class FS, typename Fn>
__device__ __forceinline__ void piece_pass(const Params& p, const Piece<DT>& c, const Piece<DT>& c1, int q, float lo,
                                           float hi, uint32_t* queue, Fn fn, int st0 = 0,
                                           int st1 = Pass<DT, kBeside>::kSteps) {
  using B = Batch<kBeside, FS>;
  constexpr int kWords = kBeside == kAlone ? 1 : 2;
  constexpr int kStep = Pass<DT, kBeside>::kStep;
  static_assert((kStep + B::kN) * kWave * kWords <= kQueue, "queue size");
  const int lane = threadIdx.x & (kWave - 1);
  const bool pen = p.use_pen != 0;
  uint32_t n = 0;  // queued (wave-uniform)
#pragma unroll 1
  for (int st = st0; st < st1; ++st) {
    float x[kStep], x1[kStep];
    int i0;
    piece_step<DT, kStep>(p, c, c.bits, pen, q, st, x, &i0);
    if constexpr (kBeside == kPairX) piece_step<DT, kStep>(p, c1, c.bits, pen, q, st, x1, &i0);
    const bool in_row = i0 < p.vocab;
    if constexpr (kWhole) {
      if (lo == -__builtin_inff()) {
#pragma unroll
        for (int e = 0; e < kStep; e += B::kN) {
          B b;
#pragma unroll
          for (int k = 0; k < B::kN; ++k) {
            b.valid[k] = in_row;
            b.x[k] = x[e + k];
            b.beside[k] = kBeside == kPairX ? __float_as_uint(x1[e + k]) : 0u;
          }
          fn(b);
        }
        continue;
      }
    }
#pragma unroll
    for (int e = 0; e < kStep; ++e) {
      const bool in = in_row && !(x[e] < lo) && !(x[e] > hi);
      const uint64_t m = __ballot(in);
      if (in) {
        const uint32_t at = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), n)) * kWords;
        queue[at] = __float_as_uint(x[e]);
        if constexpr (kBeside == kPairX) queue[at + 1] = __float_as_uint(x1[e]);
        if constexpr (kBeside == kIndex) queue[at + 1] = static_cast<uint32_t>(i0 + e);
      }
      n += static_cast<uint32_t>(__builtin_popcountll(m));
    }
    wave_lds_fence();
    // whole batches; after the last step also the rest
    const uint32_t most = st == st1 - 1 ? 0u : B::kN * kWave - 1;
#pragma unroll 1
    while (n > most) {
      const uint32_t take = n < static_cast<uint32_t>(B::kN * kWave) ? n : static_cast<uint32_t>(B::kN * kWave);
      n -= take;
      B b;
#pragma unroll
      for (int k = 0; k < B::kN; ++k) {
        const uint32_t i = static_cast<uint32_t>(k * kWave + lane);
        b.valid[k] = i < take;
        const uint32_t at = (n + (b.valid[k] ? i : 0u)) * kWords;
        b.x[k] = __uint_as_float(queue[at]);
        b.beside[k] = kWords > 1 ? queue[at + kWords - 1] : 0u;
      }
      wave_lds_fence();
      fn(b);
    }
  }
}

// The piece's registers hold their loads' results from here on (otherwise the
// compiler waits for the loads of the next piece too wherever this one is read).
template <int DT>
__device__ __forceinline__ void piece_arrived(Piece<DT>& c) {
  asm volatile("" : "+v"(c.d));
}

// each(q, piece, piece1) over every piece of a row (kPair: and of a second
// row), in chunk order, wave w on chunks w, w + kFNW, ... With one workgroup per
// CU the next piece's loads are in flight while a piece is worked on; with two
// the other waves cover them.
template <int DT, bool kPair, class FS, typename Each>
__device__ __forceinline__ void each_piece(const Params& p, const char* row0, const char* row1, const uint32_t* bm,
                                           Each each) {
  constexpr bool kAhead = FS::kBits > 10;
  constexpr int kPer = Piece<DT>::kPerChunk;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int total = (p.vocab + Piece<DT>::kElems - 1) / Piece<DT>::kElems;  // pieces of the row
  // the piece after q of this wave's chunks
  auto after = [&](int q) { return kPer == 1 || q % kPer == kPer - 1 ? q + 1 + (kFNW - 1) * kPer : q + 1; };
  Piece<DT> c, c1, next, next1;
  int q = w * kPer;
  if (q < total) {
    load_piece<DT>(p, row0, bm, q, c);
    if constexpr (kPair) load_piece<DT>(p, row1, nullptr, q, c1);
  }
#pragma unroll 1
  while (q < total) {
    const int qn = after(q);
    piece_arrived<DT>(c);
    if constexpr (kPair) piece_arrived<DT>(c1);
    if constexpr (kAhead) {
      if (qn < total) {
        load_piece<DT>(p, row0, bm, qn, next);
        if constexpr (kPair) load_piece<DT>(p, row1, nullptr, qn, next1);
      }
    }
    each(q, c, c1);
    if constexpr (kAhead) {
      c = next;
      if constexpr (kPair) c1 = next1;
    } else if (qn < total) {
      load_piece<DT>(p, row0, bm, qn, c);
      if constexpr (kPair) load_piece<DT>(p, row1, nullptr, qn, c1);
    }
    q = qn;
  }
}

template <class FS>
__device__ __forceinline__ uint32_t* wave_queue(FS& f) {
  return f.hash + __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave) * kQueue;
}

// piece_pass over a whole row.
template <int DT, class FS, typename Fn>
__device__ __forceinline__ void row_pass(const Params& p, FS& f, int row, float lo, float hi, Fn fn) {
  uint32_t* queue = wave_queue(f);
  each_piece<DT, false, FS>(p, row_ptr(p, row), nullptr, row_bitmap(p, row),
                            [&](int q, const Piece<DT>& c, const Piece<DT>&) {
                              piece_pass<DT, kAlone, false, FS>(p, c, c, q, lo, hi, queue, fn);
                            });
}

// The smallest processed logit of a row (a NaN, whose p is 0, as -inf), per lane.
template <int DT, class FS>
__device__ __forceinline__ float lane_row_min(const Params& p, int row) {
  constexpr int kStep = 4;
  float mn = __builtin_inff();
  each_piece<DT, false, FS>(p, row_ptr(p, row), nullptr, row_bitmap(p, row),
                            [&](int q, const Piece<DT>& c, const Piece<DT>&) {
#pragma unroll 1
    for (int st = 0; st < Piece<DT>::kElems / kWave / kStep; ++st) {
      float x[kStep];
      int i0;
      piece_step<DT, kStep>(p, c, c.bits, p.use_pen != 0, q, st, x, &i0);
      if (i0 >= p.vocab) continue;
#pragma unroll
      for (int e = 0; e < kStep; ++e) mn = x[e] != x[e] ? -__builtin_inff() : (x[e] < mn ? x[e] : mn);
    }
  });
  return mn;
}

// Slot s's list entries 0 .. n - 1 selected for `thr` (kCount: by counts).
template <bool kCount, class FS>
__device__ __forceinline__ bool select_list(FS& f, int s, uint32_t n, uint64_t thr, float* cut, uint64_t* mass) {
  const int t = thread_index<FS>();
  uint32_t eb[2][kEPT];
  uint64_t ew[2][kEPT];
#pragma unroll
  for (int s1 = 0; s1 < 2; ++s1) {
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const uint32_t e = static_cast<uint32_t>(t + kFW * q);
      const bool in = s1 == s && e < n;
      eb[s1][q] = in ? f.ent[s].pbits[e] : 0u;
      ew[s1][q] = !in ? 0u : (kCount ? 1u : fx46(__uint_as_float(eb[s1][q])));
    }
  }
  const uint64_t t2[2] = {thr, thr};
  float c1[2];
  uint64_t m1[2];
  bool o1[2], set1[2];
  __syncthreads();  // every lane has read the list and its count
  select_entries<false>(f, 1u << s, t2, eb, ew, false, c1, m1, o1, set1);
  *cut = s == 0 ? c1[0] : c1[1];
  *mass = s == 0 ? m1[0] : m1[1];
  return s == 0 ? o1[0] : o1[1];
}

// Lanes with `hit` append b to slot s's list (entries past kRowCap are counted
// only); e: the entry's index in the vocabulary, stored with kIndexed.
template <bool kIndexed, class FS>
__device__ __forceinline__ void list_append(FS& f, int s, uint32_t* count, bool hit, uint32_t b, uint32_t e) {
  const uint64_t m = __ballot(hit);
  if (m == 0) return;
  uint32_t at = 0;
  if ((threadIdx.x & (kWave - 1)) == 0)
    at = __hip_atomic_fetch_add(count, static_cast<uint32_t>(__builtin_popcountll(m)), __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_WORKGROUP);
  at = lane_bcast_u32(at, 0) + lanes_below(m);
  if (hit && at < static_cast<uint32_t>(kRowCap)) {
    f.ent[s].pbits[at] = b;
    if constexpr (kIndexed) f.ent[s].eidx[at] = e;
  }
}

// The largest bin (searching down from the top) at which the bins' sum reaches
// need: its index and the sum above it and in it; false when the total is less.
// Ends with a barrier. bins: kFW * kPer values.
template <int kPer, class FS>
__device__ __forceinline__ bool crossing_bin(FS& f, const uint64_t* bins, uint64_t need, uint64_t* red, uint32_t* bin,
                                             uint64_t* above, uint64_t* in, uint64_t* total) {
  const int g0 = kPer * (kFW - 1 - static_cast<int>(threadIdx.x));
  uint64_t own = 0;
#pragma unroll
  for (int q = 0; q < kPer; ++q) own += bins[g0 + q];
  const uint64_t incl = block_incl_scan(own, red, total);
  if (*total < need) {
    __syncthreads();
    return false;
  }
  if (incl >= need && incl - own < need) {
    uint64_t acc = incl - own;
    int d = g0;
#pragma unroll
    for (int q = kPer - 1; q >= 0; --q) {
      const uint64_t bq = bins[g0 + q];
      if (acc + bq >= need) {
        d = g0 + q;
        break;
      }
      acc += bq;
    }
    f.sel[0] = static_cast<uint32_t>(d);
    f.sel64[0][0] = acc;
    f.sel64[0][1] = bins[d];
  }
  __syncthreads();
  *bin = f.sel[0];
  *above = f.sel64[0][0];
  *in = f.sel64[0][1];
  return true;
}

// A whole row's cutoff in two passes, the usual way for a support beyond the
// LDS entries. The first bins approximate masses (hardware exp2 of the exponent
// in units of 2^-31, 1/16 octave per bin; binary32 LDS atomics took four times
// as long as integer ones) of the elements p >= v_min and finds the bin where
// they reach thr; the second, over the elements of the
// bins beside it and above, forms the exact mass above those bins and gathers
// theirs, which decide the cutoff exactly. The first pass only chooses the
// window: it is checked against the exact masses, and false is returned (the
// exact digit rounds of select_row follow) when the cutoff is not inside or the
// window holds more than the list.
constexpr int kWinShift = 19;                                      // bits of a float above 4 mantissa bits
constexpr int kWinBins = 2 * kFW;                                  // 64 octaves
constexpr int kWinBase = (0x4f000000 >> kWinShift) - kWinBins + 16;  // bin 0; p = 1 (2^31 units) lies below the top 16

template <int DT, class FS>
__device__ __forceinline__ bool select_window(const Params& p, FS& f, int s, int row, const RowK& K, uint64_t thr,
                                              float v_min, float* cut, uint64_t* mass) {
  constexpr int kStep = 4;
  const int t = thread_index<FS>();
  uint32_t* fb = reinterpret_cast<uint32_t*>(f.u.bins[1]);
  uint64_t* bins = f.u.bins[0];
  const float inf = __builtin_inff();
  __syncthreads();  // earlier reads of the bins and of the list
#pragma unroll
  for (int q = 0; q < 2; ++q) fb[2 * t + q] = 0u;
  if (t == 0) f.gcount[s] = 0;
  __syncthreads();
  {
    const float lo = x_floor(K, v_min);
    // exponents of p in units of 2^-31
    const float c = p.c, nm = 31.0f - K.mcmax - __builtin_amdgcn_logf(K.s);
    each_piece<DT, false, FS>(p, row_ptr(p, row), nullptr, row_bitmap(p, row),
                              [&](int pq, const Piece<DT>& pc, const Piece<DT>&) {
#pragma unroll 1
      for (int st = 0; st < Piece<DT>::kElems / kWave / kStep; ++st) {
        float x[kStep];
        int i0;
        piece_step<DT, kStep>(p, pc, pc.bits, p.use_pen != 0, pq, st, x, &i0);
        const float lo_in = i0 < p.vocab ? lo : inf;
#pragma unroll
        for (int e = 0; e < kStep; ++e) {
          if (x[e] >= lo_in) {
            const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(x[e], c, nm));
            int b = static_cast<int>(__float_as_uint(w) >> kWinShift) - kWinBase;
            b = b < 0 ? 0 : (b > kWinBins - 1 ? kWinBins - 1 : b);
            __hip_atomic_fetch_add(&fb[b], static_cast<uint32_t>(w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
      }
    });
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q)
    bins[2 * t + q] = static_cast<uint64_t>(fb[2 * t + q]) << (kFxBits - 31);
  __syncthreads();
  uint32_t d;
  uint64_t above, in, tot;
  if (!crossing_bin<2>(f, bins, thr, f.red[0], &d, &above, &in, &tot)) return false;
  if (d < 2u || d > static_cast<uint32_t>(kWinBins - 3)) return false;
  const float v_lo = __uint_as_float((d - 1u + kWinBase) << kWinShift) * 0x1p-31f;
  const float v_hi = __uint_as_float((d + 2u + kWinBase) << kWinShift) * 0x1p-31f;
  uint64_t own = 0;
  row_pass<DT>(p, f, row, x_floor(K, v_lo), inf, [&](const Batch<kAlone, FS>& b) {
    float v[b.kN];
#pragma unroll
    for (int k = 0; k < b.kN; ++k) {
      v[k] = pval(K, b.x[k]);
      own += b.valid[k] && v[k] >= v_hi ? fx46(v[k]) : 0u;
    }
#pragma unroll
    for (int k = 0; k < b.kN; ++k)
      list_append<false>(f, s, &f.gcount[s], b.valid[k] && v[k] >= v_lo && v[k] < v_hi, __float_as_uint(v[k]), 0u);
  });
  const uint64_t hi = block_sum(own, f.red[1]);
  const uint32_t n = f.gcount[s];  // every append precedes the sum's barrier
  if (hi >= thr || n > static_cast<uint32_t>(kRowCap)) return false;
  uint64_t m;
  if (!select_list<false>(f, s, n, thr - hi, cut, &m)) return false;
  *mass = hi + m;
  return true;
}

// Exact cutoff of a whole row: c = max{v : sum over the row's p >= v of
// fx46(p) >= thr} (kCount: every element weighs 1, so thr = k gives the k-th
// largest p, duplicates counted), *mass the sum at and above it. v_min: a p the
// cutoff does not lie below (masses: probably not). Masses take select_window's
// two passes first. What those leave undecided, and counts, take radix rounds on the bits
// of p as in select_entries: a pass over the row bins the masses of the current
// digit, the crossing digit's elements are gathered by a second pass into slot
// s's entries and finished by select_entries when they fit, else the next digit
// is binned. A row that holds less than thr in all keeps everything (the
// reference clamps to the last sorted value, the row minimum). The draft hash
// and slot s's entries are overwritten.
template <int DT, bool kCount, class FS>
__device__ __forceinline__ void select_row(const Params& p, FS& f, int s, int row, const RowK& K, uint64_t thr,
                                           float v_min, float* cut, uint64_t* mass) {
  const int t = thread_index<FS>();
  if constexpr (!kCount) {
    if (select_window<DT>(p, f, s, row, K, thr, v_min, cut, mass)) return;
  }
  uint64_t* bins = f.u.bins[0];
  const float inf = __builtin_inff();
  float lo = kCount ? x_floor(K, v_min) : -inf, hi = inf;
  uint32_t prefix = 0;
  uint64_t above = 0;
#pragma unroll 1
  for (int round = 0; round < 3; ++round) {
    const int shift = round == 0 ? 30 - FS::kBits : (round == 1 ? 30 - 2 * FS::kBits : 0);
    const int width = round == 2 ? 30 - 2 * FS::kBits : FS::kBits;
    __syncthreads();  // earlier reads of the bins and of the list
#pragma unroll
    for (int q = 0; q < FS::kPer; ++q) bins[FS::kPer * t + q] = 0;
    if (t == 0) f.gcount[s] = 0;
    __syncthreads();
    row_pass<DT>(p, f, row, lo, hi, [&](const Batch<kAlone, FS>& b) {
#pragma unroll
      for (int k = 0; k < b.kN; ++k) {
        const uint32_t v = __float_as_uint(pval(K, b.x[k]));
        const uint64_t w = kCount ? uint64_t{1} : fx46(__uint_as_float(v));
        if (b.valid[k] && w && (v >> (shift + width)) == prefix)
          __hip_atomic_fetch_add(&bins[(v >> shift) & ((1u << width) - 1u)], w, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    });
    __syncthreads();
    uint32_t d;
    uint64_t ab, in, tot;
    if (!crossing_bin<FS::kPer>(f, bins, thr - above, f.red[round & 1], &d, &ab, &in, &tot)) {
      // the row holds less than thr (only in the first round)
      const float mn = -block_max_f32<kFW>(-lane_row_min<DT, FS>(p, row), reinterpret_cast<float*>(f.red[2]));
      *cut = pval(K, mn);
      *mass = tot;
      return;
    }
    prefix = (prefix << width) | d;
    above += ab;
    if (round == 2) {
      *cut = __uint_as_float(prefix);
      *mass = above + in;
      return;
    }
    // the crossing digit's elements (p from prefix << shift up to the next digit)
    lo = prefix ? x_floor(K, __uint_as_float(prefix << shift)) : -inf;
    hi = x_ceil(K, __uint_as_float((prefix + 1u) << shift));
    row_pass<DT>(p, f, row, lo, hi, [&](const Batch<kAlone, FS>& b) {
#pragma unroll
      for (int k = 0; k < b.kN; ++k) {
        const uint32_t v = __float_as_uint(pval(K, b.x[k]));
        list_append<false>(f, s, &f.gcount[s],
                           b.valid[k] && (v >> shift) == prefix && (kCount || fx46(__uint_as_float(v)) != 0), v, 0u);
      }
    });
    __syncthreads();
    const uint32_t n = f.gcount[s];
    if (n <= static_cast<uint32_t>(kRowCap)) {
      uint64_t m;
      select_list<kCount>(f, s, n, thr - above, cut, &m);
      *mass = above + m;
      return;
    }
  }
}

// Appends the elements p >= c of the chunks whose non-candidates may reach c
// to slot s's entries, in no order, in place of those chunks' candidates
// (whose p becomes 0). False when they do not fit. Uses the draft hash's LDS.
template <int DT, class FS>
__device__ __forceinline__ bool refill_chunks(const Params& p, FS& f, int s, int row, const RowK& K, float c) {
  const int t = thread_index<FS>(), lane = t & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const char* rowp = row_ptr(p, row);
  const uint32_t* bm = row_bitmap(p, row);
  const float lo = x_floor(K, c);
  uint32_t* q = wave_queue(f);
  // the chunks to re-read (lane l's bounds are chunk l's and chunk 64 + l's),
  // dealt to the waves in turn: whole ones, or, when they are fewer than the
  // waves, as many parts of each as give every wave one (a chunk read by one
  // wave while the others waited took 1.5 us longer)
  uint64_t need[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int j = h * kWave + lane;
    need[h] = __ballot(j < p.nch && f.bound[s][j < p.nch ? j : 0] >= c);
  }
  const int chunks = __builtin_popcountll(need[0]) + __builtin_popcountll(need[1]);
  const int parts = chunks > 4 ? 1 : (chunks > 2 ? 2 : (chunks == 2 ? 4 : 8));
  constexpr int kPer = Piece<DT>::kPerChunk;
  constexpr int kStep = Pass<DT, kIndex>::kStep, kSteps = Pass<DT, kIndex>::kSteps;
  static_assert(kSteps * kPer % 8 == 0 && kFNW == 8, "whole steps per part");
  const int per_part = kSteps * kPer / parts;
  int turn = 0;
#pragma unroll 1
  while (need[0] | need[1]) {
    const int hi = need[0] ? 0 : 1;
    const int j = hi * kWave + __builtin_ctzll(hi ? need[1] : need[0]);
    if (hi) need[1] &= need[1] - 1; else need[0] &= need[0] - 1;
    const int part = (w - turn) & (kFNW - 1);
    turn += parts;
    if (part >= parts) continue;
    Piece<DT> cd[kPer];
    int st0[kPer], st1[kPer];  // this wave's steps of each piece
#pragma unroll
    for (int h = 0; h < kPer; ++h) {
      const int a = part * per_part - h * kSteps, b = a + per_part;
      st0[h] = a < 0 ? 0 : a;
      st1[h] = b > kSteps ? kSteps : b;
      load_piece<DT>(p, rowp, bm, j * kPer + h, cd[h], st0[h] * kStep / Elem<DT>::kPerVec,
                     (st1[h] * kStep + Elem<DT>::kPerVec - 1) / Elem<DT>::kPerVec);
    }
    if (part == 0) {
      const uint32_t e0 = f.cstart[s][j], e1 = e0 + f.ccount[s][j];
      for (uint32_t e = e0 + lane; e < e1; e += kWave) f.ent[s].pbits[e] = 0u;
    }
#pragma unroll
    for (int h = 0; h < kPer; ++h) {
      piece_pass<DT, kIndex, false, FS>(p, cd[h], cd[h], j * kPer + h, lo, __builtin_inff(), q,
                                 [&](const Batch<kIndex, FS>& b) {
        float v[b.kN];
#pragma unroll
        for (int k = 0; k < b.kN; ++k) v[k] = pval(K, b.x[k]);
#pragma unroll
        for (int k = 0; k < b.kN; ++k)
          list_append<true>(f, s, &f.aux[s].n, b.valid[k] && v[k] >= c, __float_as_uint(v[k]), b.beside[k]);
      }, st0[h], st1[h]);
    }
  }
  __syncthreads();
  return f.aux[s].n <= static_cast<uint32_t>(kRowCap);
}

// A p the top-p cutoff of a row probably does not lie below: every element
// below it together holds less than half of 1 - top_p.
__device__ __forceinline__ float cutoff_guess(const Params& p, uint64_t thr) {
  const float rest = static_cast<float>(kFxOne - static_cast<double>(thr)) * static_cast<float>(1.0 / kFxOne);
  return rest > 0.0f ? 0.5f * rest / static_cast<float>(p.vocab) : 0.0f;
}

// A resolved row's state (one thread).
__device__ __forceinline__ void store_row(RowAux& a, uint32_t flags, float cut, uint64_t mass) {
  a.flags = flags;
  a.cut = cut;
  a.mass_fx = mass;
  a.mass_f = mass_to_f32(mass);
}

// Resolves the cutoffs of the unit's rows: list mode (kRowList: the support
// is in the LDS entries) or dense (the support is {p >= cut} of the whole
// row). The rows in `mask` are filtered (thr: their thresholds); their first
// selects share their rounds, over the entries in eb / ew, whose first-round
// masses are in the bins already with `hist`. Unfiltered rows keep row_setup's
// state. A select over the entries is the row's when its cutoff lies above
// every chunk's non-candidate bound. Otherwise that cutoff, when the entries
// hold thr, is a lower bound of the row's: the chunks whose bound reaches it
// are re-read and the entries selected again; a row they do not fit,
// or whose entries hold less than thr, is selected whole.
template <int DT, class FS>
__device__ __forceinline__ void resolve_rows(const Params& p, FS& f, const int (&rows)[2], const RowK (&K)[2], uint32_t mask,
                                            const uint64_t (&thr)[2], const uint32_t (&eb)[2][kEPT],
                                            const uint64_t (&ew)[2][kEPT], bool hist) {
  float cut[2] = {0.0f, 0.0f};
  uint64_t mass[2] = {0u, 0u};
  bool ok[2] = {false, false}, set[2] = {false, false};
  if (!mask) return;
  select_entries(f, mask, thr, eb, ew, hist, cut, mass, ok, set);
  uint32_t late = 0, whole = 0;  // list rows not stored yet; rows to select whole
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (!((mask >> s) & 1u)) continue;  // unfiltered: P = p over the whole row
    if (!ok[s] || !(cut[s] > f.aux[s].bmax)) {
      whole |= 1u << s;
    } else if (!set[s]) {
      late |= 1u << s;
    }
  }
  if (!(late | whole)) return;
  __syncthreads();  // every read of the rows' state above precedes the stores
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if ((late >> s) & 1u) store_row(f.aux[s], kRowFiltered | kRowList, cut[s], mass[s]);
    }
  }
  const float g0 = uniform<FS>(ok[0] ? cut[0] : cutoff_guess(p, thr[0]));
  const float g1 = uniform<FS>(ok[1] ? cut[1] : cutoff_guess(p, thr[1]));
#pragma unroll 1
  for (int s = 0; s < 2; ++s) {
    if (!((whole >> s) & 1u)) continue;
    const int row = s == 0 ? rows[0] : rows[1];
    const RowK Ks = s == 0 ? K[0] : K[1];
    const uint64_t th = s == 0 ? thr[0] : thr[1];
    const float g = s == 0 ? g0 : g1;
    float c;
    uint64_t m;
    uint32_t flags = kRowFiltered;
    if ((s == 0 ? ok[0] : ok[1]) && refill_chunks<DT>(p, f, s, row, Ks, g) &&
        select_list<false>(f, s, f.aux[s].n, th, &c, &m)) {
      flags |= kRowList | kRowRefilled;
    } else {
      select_row<DT, false>(p, f, s, row, Ks, th, g, &c, &m);
    }
    __syncthreads();
    if (threadIdx.x == 0) store_row(f.aux[s], flags, c, m);
  }
  // the draft hash is empty again (its LDS held the waves' queues)
  for (int h = threadIdx.x; h < kHash; h += kFW) f.hash[h] = 0u;
  __syncthreads();
}

// sum_{p >= c[s]} fx46(p) over the entries of the slots in `mask`, both slots
// in one block reduction.
template <class FS>
__device__ __forceinline__ void entries_mass2(FS& f, uint32_t mask, const float (&c)[2], uint64_t (&out)[2]) {
  uint64_t own[2] = {0u, 0u};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (!((mask >> s) & 1u)) continue;
    const uint32_t n = f.aux[s].n;
    for (uint32_t e = threadIdx.x; e < n; e += kFW) {
      const float v = __uint_as_float(f.ent[s].pbits[e]);
      if (v >= c[s]) own[s] += fx46(v);
    }
  }
  block_sum2(own[0], own[1], f.red[2], &out[0], &out[1]);
  __syncthreads();
}

// sum_{p >= c} fx46(p) over slot s's list entries 0 .. n - 1 (kCount: the number of them).
template <bool kCount, class FS>
__device__ __forceinline__ uint64_t list_mass(FS& f, int s, uint32_t n, float c) {
  uint64_t own = 0;
  for (uint32_t e = threadIdx.x; e < n; e += kFW) {
    const float v = __uint_as_float(f.ent[s].pbits[e]);
    if (v >= c) own += kCount ? uint64_t{1} : fx46(v);
  }
  const uint64_t tot = block_sum(own, f.red[2]);
  __syncthreads();
  return tot;
}

// The elements p >= c of a whole row into slot s's entries, in no order and
// without their indices; returns their number (past kRowCap they are counted only).
template <int DT, class FS>
__device__ __forceinline__ uint32_t gather_row(const Params& p, FS& f, int s, int row, const RowK& K, float c) {
  __syncthreads();  // earlier reads of the list
  if (threadIdx.x == 0) f.gcount[s] = 0;
  __syncthreads();
  row_pass<DT>(p, f, row, x_floor(K, c), __builtin_inff(), [&](const Batch<kAlone, FS>& b) {
#pragma unroll
    for (int k = 0; k < b.kN; ++k) {
      const float v = pval(K, b.x[k]);
      list_append<false>(f, s, &f.gcount[s], b.valid[k] && v >= c, __float_as_uint(v), 0u);
    }
  });
  __syncthreads();
  return f.gcount[s];
}

// sum_{p >= c} fx46(p) over a whole row.
template <int DT, class FS>
__device__ __forceinline__ uint64_t row_mass(const Params& p, FS& f, int row, const RowK& K, float c) {
  uint64_t own = 0;
  row_pass<DT>(p, f, row, x_floor(K, c), __builtin_inff(), [&](const Batch<kAlone, FS>& b) {
#pragma unroll
    for (int k = 0; k < b.kN; ++k) {
      const float v = pval(K, b.x[k]);
      own += b.valid[k] && v >= c ? fx46(v) : 0u;
    }
  });
  const uint64_t tot = block_sum(own, f.red[2]);
  __syncthreads();
  return tot;
}

// Cutoffs of the unit's rows with top-k (1 <= p.top_k < V): max(k-th largest
// p, top-p cutoff) -- the joint rule of distributions.py:72-86, or the k-th
// largest alone for the rows not in `mask` (top_p = 1) -- with ties kept and
// one renormalisation over {p >= cutoff}. rmask: the rows with any mass, whose
// entries are counted in the bins already. The k-th largest ck of the entries
// comes first, by a select by counts over both rows. Above every chunk's non-candidate bound it is the row's, and every element at or
// above it is an entry, so the top-p cutoff cp is decided there too: the
// entries' mass at and above ck falls short of thr exactly when cp < ck (the
// cutoff is ck), and otherwise cp >= ck is the entries' own. So a row whose
// top-p support is far larger than its candidates needs no pass over the row
// when its k largest are among them (one sequence, k = 4, V = 32000, T 0.8,
// top_p 0.95, top_k 50: the finaliser took 25 to 164 us with top-p resolved
// first). Rows whose k largest are not all candidates take their top-p cutoff
// first, and keep it when no more than k elements reach it. Otherwise the
// k-th largest of those elements is the cutoff: of the entries, counted again
// where chunks were re-read into them or the row's support was gathered, or of
// the whole row (B 64, k 2, V 49152
// f32, T 0.7, top_p 0.95, top_k 1000, chunks re-read: 140 us a call with the
// whole row selected twice instead).
template <int DT, class FS>
__device__ __forceinline__ void resolve_top_k(const Params& p, FS& f, const int (&rows)[2], const RowK (&K)[2],
                                              uint32_t rmask, uint32_t mask, const uint64_t (&thr)[2],
                                              const uint32_t (&eb)[2][kEPT], const uint64_t (&ew)[2][kEPT]) {
  const uint64_t kk = static_cast<uint64_t>(p.top_k);
  if (!rmask) return;
  const float bmax[2] = {f.aux[0].bmax, f.aux[1].bmax};
  float ck[2];
  bool okk[2];
  {
    uint64_t one[2][kEPT], m1[2];
    bool set1[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int q = 0; q < kEPT; ++q) one[s][q] = eb[s][q] != 0u ? 1u : 0u;
    }
    const uint64_t k2[2] = {kk, kk};
    select_entries<false>(f, rmask, k2, eb, one, true, ck, m1, okk, set1);
  }
  uint32_t kmask = 0;  // rows whose k largest are entries
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (((rmask >> s) & 1u) && okk[s] && ck[s] > bmax[s]) kmask |= 1u << s;
  }
  uint64_t mass[2] = {0u, 0u};
  if (kmask) entries_mass2(f, kmask, ck, mass);
  // rows that still need a top-p select: those whose mass at and above ck
  // reaches thr, and those whose ck is not known to be the row's
  uint32_t pmask = 0;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (((mask >> s) & 1u) && !(((kmask >> s) & 1u) && mass[s] < thr[s])) pmask |= 1u << s;
  }
  if (pmask) resolve_rows<DT>(p, f, rows, K, pmask, thr, eb, ew, false);
  uint32_t store = 0, emask = 0, whole = 0;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (!((rmask >> s) & 1u)) continue;
    if ((kmask >> s) & 1u) {
      if (!((pmask >> s) & 1u)) store |= 1u << s;  // else cp >= ck: as resolved
    } else if (((pmask >> s) & 1u) && (f.aux[s].flags & kRowList)) {
      if (okk[s] && ck[s] > f.aux[s].cut) emask |= 1u << s;
    } else {
      whole |= 1u << s;
    }
  }
#pragma unroll 1
  for (int s = 0; s < 2; ++s) {
    // re-read rows: the elements at and above cp in the list, and where they
    // are more than k the k-th largest of the list (its dead entries count at
    // p = 0, below any cutoff)
    if (!((pmask >> s) & 1u) || !(f.aux[s].flags & kRowRefilled)) continue;
    const uint32_t n = f.aux[s].n;
    const float cp = f.aux[s].cut;
    emask &= ~(1u << s);
    if (list_mass<true>(f, s, n, cp) <= kk) continue;
    float c;
    uint64_t m;
    select_list<true>(f, s, n, kk, &c, &m);
    if (c > cp) emask |= 1u << s;
    if (s == 0) ck[0] = c;
    else ck[1] = c;
  }
  if (emask) {
    uint64_t em[2];
    entries_mass2(f, emask, ck, em);
    if (emask & 1u) mass[0] = em[0];
    if (emask & 2u) mass[1] = em[1];
  }
  __syncthreads();  // every read of the rows' state above precedes the stores
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (((store | emask) >> s) & 1u)
        store_row(f.aux[s], kRowFiltered | kRowList | (f.aux[s].flags & kRowRefilled), ck[s], mass[s]);
    }
  }
#pragma unroll 1
  for (int s = 0; s < 2; ++s) {
    if (!((whole >> s) & 1u)) continue;
    // the k-th largest of the whole row by passes over it
    const int row = s == 0 ? rows[0] : rows[1];
    const RowK Ks = s == 0 ? K[0] : K[1];
    const float lower = ((pmask >> s) & 1u) ? uniform<FS>(f.aux[s].cut) : 0.0f;
    float c;
    uint64_t m;
    bool listed = false;  // the elements at and above cp, all of them
    if (lower > 0.0f) {
      const uint32_t n = gather_row<DT>(p, f, s, row, Ks, lower);
      if (n <= kk) continue;
      listed = n <= static_cast<uint32_t>(kRowCap);
      if (listed) {
        select_list<true>(f, s, n, kk, &c, &m);
        m = list_mass<false>(f, s, n, c);
      }
    }
    if (!listed) {
      select_row<DT, true>(p, f, s, row, Ks, kk, lower, &c, &m);
      m = row_mass<DT>(p, f, row, Ks, c);
    }
    if (threadIdx.x == 0) store_row(f.aux[s], kRowFiltered, c, m);
  }
  __syncthreads();
}

// Filtered probability of a row at p (P = p when unfiltered).
__device__ __forceinline__ float filtered_of(const RowAux& a, float pv) {
  if (!(a.flags & kRowFiltered)) return pv;
  if (a.mass_fx == 0) return 0.0f;
  return pv >= a.cut ? pv / a.mass_f : 0.0f;
}

// ---------------------------------------------------------------------------
// Draws: the first index j (in vocabulary order) with
// sum_{i <= j} W_i > floor(u * sum W), W_i = fx46 of the normalised weight;
// index 0 at zero total (categorical_pick).
// ---------------------------------------------------------------------------

// Chunk j* holding the target, from f.csum: lane l of wave 0 holds chunks
// 2l and 2l+1. Writes f.pick_rem = target - mass before j*, f.pick = j*
// (kNone at zero total). Ends with a barrier.
template <class FS>
__device__ __forceinline__ void pick_chunk(const Params& p, FS& f, float u) {
  const int t = threadIdx.x;
  if (t < kWave) {
    const int ja = 2 * t, jb = ja + 1;
    const uint64_t a = ja < p.nch ? f.csum[ja] : 0, b = jb < p.nch ? f.csum[jb] : 0;
    const uint64_t incl = wave_scan_add_u64(a + b);
    const uint64_t total = lane_bcast_u64(incl, kWave - 1);
    const uint64_t target = floor_u_times(u, total);
    const uint64_t ex = incl - a - b;
    // the first chunk whose inclusive mass exceeds the target
    const bool in_a = ja < p.nch && ex <= target && ex + a > target;
    const bool in_b = jb < p.nch && ex + a <= target && ex + a + b > target;
    if (total == 0) {
      if (t == 0) f.pick = kNone;
    } else if (in_a) {
      f.pick = static_cast<uint32_t>(ja);
      f.pick_rem = target - ex;
    } else if (in_b) {
      f.pick = static_cast<uint32_t>(jb);
      f.pick_rem = target - ex - a;
    }
  }
  __syncthreads();
}

// Within a chunk of 2048 positions: thread t owns positions kPosPT t .. +
// kPosPT - 1 with weights w; the first position whose inclusive mass exceeds
// `rem` (the target minus the mass before the chunk) goes to f.token as c0 + pos.
template <class FS>
__device__ __forceinline__ void pick_in_chunk(FS& f, int64_t c0, const uint64_t (&w)[kPosPT], uint64_t rem) {
  const int t = threadIdx.x;
  uint64_t own = 0;
#pragma unroll
  for (int q = 0; q < kPosPT; ++q) own += w[q];
  uint64_t tot;
  const uint64_t incl = block_incl_scan(own, f.red[3], &tot);
  const uint64_t ex = incl - own;
  if (ex <= rem && incl > rem) {
    uint64_t acc = ex;
#pragma unroll
    for (int q = 0; q < kPosPT; ++q) {
      if (acc + w[q] > rem) {
        f.token = c0 + kPosPT * t + q;
        break;
      }
      acc += w[q];
    }
  }
  __syncthreads();
}

// List-mode draw over slot 0's entries, thread t weighing entries kEPT t + q
// by wl[q]. With each chunk's entries contiguous and the chunks in order
// (`ordered`: no chunk was refilled), a scan over the list finds the entry
// holding the target, which is the draw when its chunk's entries are in index
// order; otherwise (per-chunk sums find the chunk when not `ordered`) the
// chunk's entries are scattered to their positions (indices are distinct
// among entries of nonzero weight) and scanned there.
template <class FS>
__device__ __forceinline__ int64_t draw_list(const Params& p, FS& f, const uint64_t (&wl)[kEPT], float u,
                                             bool ordered) {
  const int t = thread_index<FS>();
  const uint32_t n = f.aux[0].n;
  uint32_t js;
  uint64_t rem;
  if (ordered) {
    uint64_t own = 0;
#pragma unroll
    for (int q = 0; q < kEPT; ++q) own += wl[q];
    uint64_t total;
    const uint64_t incl = block_incl_scan(own, f.red[3], &total);
    if (total == 0) return 0;
    const uint64_t target = floor_u_times(u, total);
    uint64_t run = incl - own;
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const uint32_t e = kEPT * t + q;
      if (e < n) {
        f.u.dr.cum[e] = run;
        if (run <= target && target < run + wl[q]) f.pick = e;
      }
      run += wl[q];
    }
    __syncthreads();
    // the entry holding the target; in a chunk whose entries are in index
    // order it is the draw
    const uint32_t idx = f.ent[0].eidx[f.pick];
    js = idx >> 11;
    if (f.plain[0][js]) return static_cast<int64_t>(idx);
    rem = target - f.u.dr.cum[f.cstart[0][js]];
    __syncthreads();  // every read of f.u.dr precedes the position scatter
  } else {
    for (int j = t; j < p.nch; j += kFW) f.csum[j] = 0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const uint32_t e = kEPT * t + q;
      if (e < n && wl[q])
        __hip_atomic_fetch_add(&f.csum[f.ent[0].eidx[e] >> 11], wl[q], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    pick_chunk(p, f, u);
    js = f.pick;
    if (js == kNone) return 0;
    rem = f.pick_rem;
  }
  // chunk js by positions
#pragma unroll
  for (int q = 0; q < kPosPT; ++q) f.u.pos[kPosPT * t + q] = 0;
  if (t == 0) f.token = 0;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kEPT; ++q) {
    const uint32_t e = kEPT * t + q;
    if (e < n && wl[q]) {
      const uint32_t ix = f.ent[0].eidx[e];
      if ((ix >> 11) == js) f.u.pos[ix & (kChunk - 1)] = wl[q];
    }
  }
  __syncthreads();
  uint64_t w[kPosPT];
#pragma unroll
  for (int q = 0; q < kPosPT; ++q) w[q] = f.u.pos[kPosPT * t + q];
  pick_in_chunk(f, static_cast<int64_t>(js) * kChunk, w, rem);
  return f.token;
}

// Dense-mode draw over the whole vocabulary with weights wfn(x0, x1), zero
// for every x0 below lo (kPair: x1 is row1's logit at the same index): each
// chunk's mass by one wave, then the chunk holding the target by positions.
template <int DT, bool kPair, typename WFn, class FS>
__device__ __forceinline__ int64_t draw_dense(const Params& p, FS& f, int row0, int row1, float lo, float u, WFn wfn) {
  const int t = thread_index<FS>();
  const char* r0 = row_ptr(p, row0);
  const char* r1 = kPair ? row_ptr(p, row1) : nullptr;
  const uint32_t* bm = row_bitmap(p, row0);
  uint32_t* q = wave_queue(f);
  if (t == 0) f.token = 0;
  uint64_t own = 0;  // of the chunk
  each_piece<DT, kPair, FS>(p, r0, r1, bm, [&](int pq, const Piece<DT>& c, const Piece<DT>& c1) {
    constexpr int kBeside = kPair ? kPairX : kAlone;
    constexpr int kPer = Piece<DT>::kPerChunk;
    piece_pass<DT, kBeside, true, FS>(p, c, c1, pq, lo, __builtin_inff(), q, [&](const Batch<kBeside, FS>& b) {
#pragma unroll
      for (int k = 0; k < b.kN; ++k) own += b.valid[k] ? wfn(b.x[k], __uint_as_float(b.beside[k])) : 0u;
    });
    if (pq % kPer == kPer - 1 || (pq + 1) * Piece<DT>::kElems >= p.vocab) {
      own = wave_sum_u64(own);
      if ((t & (kWave - 1)) == 0) f.csum[pq / kPer] = own;
      own = 0;
    }
  });
  __syncthreads();
  pick_chunk(p, f, u);
  const uint32_t js = f.pick;
  if (js == kNone) return 0;
  const int64_t c0 = static_cast<int64_t>(js) * kChunk;
  uint64_t wt[kPosPT];
#pragma unroll
  for (int r = 0; r < kPosPT; ++r) {
    const int64_t i = c0 + kPosPT * t + r;
    wt[r] = i < p.vocab ? wfn(load_x<DT>(p, r0, bm, i), kPair ? load_x<DT>(p, r1, bm, i) : 0.0f) : 0u;
  }
  pick_in_chunk(f, c0, wt, f.pick_rem);
  return f.token;
}

// Filtered draft probability Q at vocabulary index x (slot 1).
template <int DT, class FS>
__device__ __forceinline__ float q_at(const Params& p, const FS& f, const RowK& K1, int row1, uint32_t x) {
  const RowAux& a = f.aux[1];
  if (a.flags & kRowEmpty) return 0.0f;
  if (a.flags & kRowList) {
    // every draft element with q >= its cutoff is an entry
    const uint32_t e = hash_find(f, x);
    return e == kNone ? 0.0f : filtered_of(a, __uint_as_float(f.ent[1].pbits[e]));
  }
  return filtered_of(a, pval(K1, load_x<DT>(p, row_ptr(p, row1), row_bitmap(p, row1), x)));
}

// A logit every element of the row's support lies at or above.
__device__ __forceinline__ float support_floor(const RowAux& a, const RowK& K) {
  return (a.flags & kRowFiltered) ? x_floor(K, a.cut) : -__builtin_inff();
}

// Draw from slot 0's filtered distribution P (bonus / sample).
template <int DT, class FS>
__device__ __forceinline__ int64_t draw_target(const Params& p, FS& f, int row0, const RowK& K0, float u) {
  const RowAux& a = f.aux[0];
  if (a.flags & kRowList) {
    uint64_t wl[kEPT];
    const uint32_t n = a.n;
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const uint32_t e = kEPT * threadIdx.x + q;
      wl[q] = e < n ? fx46(filtered_of(a, __uint_as_float(f.ent[0].pbits[e]))) : 0;
    }
    return draw_list(p, f, wl, u, !(a.flags & kRowRefilled));
  }
  return draw_dense<DT, false>(p, f, row0, row0, support_floor(a, K0), u,
                               [&](float x, float) { return fx46(filtered_of(a, pval(K0, x))); });
}

// Residual draw at a rejected position: normalize(max(P - Q, 0)), falling
// back to normalize(P) at zero mass (rejection.py:60-69).
template <int DT, class FS>
__device__ __forceinline__ int64_t draw_residual(const Params& p, FS& f, int row0, int row1, const RowK& K0, const RowK& K1,
                                 float u) {
  const int t = thread_index<FS>();
  const RowAux& a = f.aux[0];
  if (a.flags & kRowList) {
    const uint32_t n = a.n;
    const RowAux& a1 = f.aux[1];
    // P and d = max(P - Q, 0) at the entries t + kFW q (every wave takes a
    // share), Q where P > 0; in list mode the first hash probes of all of
    // them go out together and only a collision walks on
    float P[kEPT], Q[kEPT];
    uint32_t ix[kEPT];
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const uint32_t e = t + kFW * q;
      P[q] = e < n ? filtered_of(a, __uint_as_float(f.ent[0].pbits[e])) : 0.0f;
      ix[q] = e < n ? f.ent[0].eidx[e] : 0u;
      Q[q] = 0.0f;
    }
    if ((a1.flags & kRowList) && !(a1.flags & kRowEmpty)) {
      uint32_t v[kEPT], m[kEPT];
#pragma unroll
      for (int q = 0; q < kEPT; ++q) v[q] = P[q] > 0.0f ? f.hash[hash_slot(ix[q])] : 0u;
#pragma unroll
      for (int q = 0; q < kEPT; ++q) m[q] = v[q] ? f.ent[1].eidx[v[q] - 1u] : 0u;
#pragma unroll
      for (int q = 0; q < kEPT; ++q) {
        if (v[q] && m[q] != ix[q]) v[q] = hash_find(f, ix[q]) + 1u;  // kNone + 1 = 0: absent
        if (v[q]) Q[q] = filtered_of(a1, __uint_as_float(f.ent[1].pbits[v[q] - 1u]));
      }
    } else {
#pragma unroll
      for (int q = 0; q < kEPT; ++q) {
        if (P[q] > 0.0f) Q[q] = q_at<DT>(p, f, K1, row1, ix[q]);
      }
    }
    uint64_t dsum = 0, psum = 0;
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      float d = P[q] - Q[q];
      d = P[q] > 0.0f && d > 0.0f ? d : 0.0f;
      const uint32_t e = t + kFW * q;
      if (e < n) {
        f.u.res.pv[e] = P[q];
        f.u.res.dv[e] = d;
      }
      dsum += fx46(d);
      psum += fx46(P[q]);
    }
    uint64_t dtot, ptot;
    block_sum2(dsum, psum, f.red[1], &dtot, &ptot);
    const bool use_d = dtot > 0;
    const float den = use_d ? mass_to_f32(dtot) : (ptot > 0 ? mass_to_f32(ptot) : 1.0f);
    // the draw's weights at this thread's entries kEPT t + q
    uint64_t wl[kEPT];
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const uint32_t e = kEPT * t + q;
      wl[q] = e < n ? fx46((use_d ? f.u.res.dv[e] : f.u.res.pv[e]) / den) : 0u;
    }
    return draw_list(p, f, wl, u, !(a.flags & kRowRefilled));
  }
  // dense target support: passes over both rows
  const RowAux a1 = f.aux[1];
  auto pair = [&](float x0, float x1, float* P) -> float {
    *P = filtered_of(a, pval(K0, x0));
    const float Q = (a1.flags & kRowEmpty) ? 0.0f : filtered_of(a1, pval(K1, x1));
    const float d = *P - Q;
    return *P > 0.0f && d > 0.0f ? d : 0.0f;
  };
  const float lo = support_floor(a, K0);
  const char* r1 = row_ptr(p, row1);
  const uint32_t* bm = row_bitmap(p, row0);
  uint32_t* qu = wave_queue(f);
  uint64_t dsum = 0, psum = 0;
  each_piece<DT, true, FS>(p, row_ptr(p, row0), r1, bm, [&](int pq, const Piece<DT>& c, const Piece<DT>& c1) {
    piece_pass<DT, kPairX, true, FS>(p, c, c1, pq, lo, __builtin_inff(), qu, [&](const Batch<kPairX, FS>& b) {
#pragma unroll
      for (int k = 0; k < b.kN; ++k) {
        float P;
        const float d = pair(b.x[k], __uint_as_float(b.beside[k]), &P);
        dsum += b.valid[k] ? fx46(d) : 0u;
        psum += b.valid[k] ? fx46(P) : 0u;
      }
    });
  });
  uint64_t dtot, ptot;
  block_sum2(dsum, psum, f.red[1], &dtot, &ptot);
  const bool use_d = dtot > 0;
  const float den = use_d ? mass_to_f32(dtot) : (ptot > 0 ? mass_to_f32(ptot) : 1.0f);
  return draw_dense<DT, true>(p, f, row0, row1, lo, u, [&](float x0, float x1) -> uint64_t {
    float P;
    const float d = pair(x0, x1, &P);
    return fx46((use_d ? d : P) / den);
  });
}

// ---------------------------------------------------------------------------
// fin_kernel: unit blockIdx.x, after stream_kernel wrote every record
// ---------------------------------------------------------------------------
template <int DT, bool kTopK, class FS>
__device__ __forceinline__ void fin_unit(const Params& p, FS& f) {
  const int t = threadIdx.x, w = t / kWave;
  const int unit = blockIdx.x;
  int g, i, nr;
  int rows[2];
  if (p.mode == kModeSpec) {
    g = unit / (p.k + 1);
    i = unit - g * (p.k + 1);
    nr = i < p.k ? 2 : 1;
    rows[0] = g * p.rpg + i;
    rows[1] = g * p.rpg + p.k + 1 + i;
  } else {
    g = unit;
    i = 0;
    nr = 1;
    rows[0] = unit;
    rows[1] = unit;
  }
  // the unit's uniforms and draft token, wanted only at the end: loaded now
  float u_acc = 0.0f, u_draw = 0.0f;
  int64_t xdraft = 0;
  if (p.mode == kModeSpec) {
    const float* ug = p.uniforms + static_cast<int64_t>(g) * (2 * p.k + 1);
    if (i < p.k) {
      u_acc = ug[i];
      u_draw = ug[p.k + i];
      xdraft = p.draft_tokens[static_cast<int64_t>(g) * p.k + i];
    } else {
      u_draw = ug[2 * p.k];
    }
  } else if (p.mode == kModeSample) {
    u_draw = p.row_uniforms[rows[0]];
  }
  const float tp0 = row_top_p(p, rows[0]);
  const float tp1 = nr == 2 ? row_top_p(p, rows[1]) : 1.0f;
  // every load of the set-up issued before any result is used: the records
  // (wave s < nr, row s) first, then every candidate slot of both rows
  RecPair rp;
  if (w < nr) rp = load_recs(p, rows[w]);
  const int nslot = p.nch * p.cap;
  uint64_t sl[2][kEPT];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const uint64_t* cb = p.cands + static_cast<int64_t>(rows[s]) * nslot;
#pragma unroll
    for (int q = 0; q < kEPT; ++q) {
      const int e = t + q * kFW;
      sl[s][q] = (s < nr && e < nslot) ? cb[e] : 0u;
    }
  }
  // cleared while the loads are in flight: the draft hash and the radix bins
  if (nr == 2) {
    for (int h = t; h < kHash; h += kFW) f.hash[h] = 0u;
  }
#pragma unroll
  for (int q = 0; q < FS::kPer; ++q) {
    f.u.bins[0][FS::kPer * t + q] = 0;
    f.u.bins[1][FS::kPer * t + q] = 0;
  }
  if (t < FS::kCo) {
    f.coarse[0][t] = 0;
    f.coarse[1][t] = 0;
  }
  if (w < nr) row_setup(p, f, w, rp, w == 0 ? tp0 : tp1);
  __syncthreads();
  // the filtered rows and their thresholds
  uint32_t mask = 0;
  uint64_t thr[2] = {0u, 0u};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float tp = s == 0 ? tp0 : tp1;
    if (s < nr && tp < 1.0f && !(f.aux[s].flags & kRowEmpty)) {
      mask |= 1u << s;
      // a threshold of 0 (top_p < 2^-46) selects the largest p, as 1 does
      // whenever that p has a nonzero mass
      const uint64_t tf = fx46(tp);
      thr[s] = uniform<FS>(tf > 0 ? tf : 1);
    }
  }
  uint32_t eb[2][kEPT];
  uint64_t ew[2][kEPT];
  uint32_t rmask = 0;  // rows with any mass (with top-k, all of them are selected)
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (s < nr && !(f.aux[s].flags & kRowEmpty)) rmask |= 1u << s;
  }
  place_entries<kTopK>(p, f, nr, sl, kTopK ? rmask : mask, eb, ew);
  __syncthreads();
  RowK K[2];
  for (int s = 0; s < 2; ++s) K[s] = RowK{uniform<FS>(f.aux[s < nr ? s : 0].mcmax), uniform<FS>(f.aux[s < nr ? s : 0].s), p.cd};
  if constexpr (kTopK) {
    resolve_top_k<DT>(p, f, rows, K, rmask, mask, thr, eb, ew);
  } else {
    resolve_rows<DT>(p, f, rows, K, mask, thr, eb, ew, true);
  }

  if (p.mode == kModeSpec) {
    const int k = p.k;
    int64_t token;
    bool acc = false;
    if (i == k) {
      token = draw_target<DT>(p, f, rows[0], K[0], u_draw);
    } else {
      const RowAux& a0 = f.aux[0];
      const RowAux& a1 = f.aux[1];
      const float P = a0.has_tok ? filtered_of(a0, a0.ptok) : 0.0f;
      const float Q = a1.has_tok ? filtered_of(a1, a1.ptok) : 0.0f;
      acc = accept_draw(u_acc, P, Q);
      // the draft's support by vocabulary index, for the residual's Q lookups
      if (!acc && (a0.flags & kRowList) && (a1.flags & kRowList)) hash_support(f);
      token = acc ? xdraft : draw_residual<DT>(p, f, rows[0], rows[1], K[0], K[1], u_draw);
    }
    // publish, then the last of the batch element's k+1 units completes the
    // outputs
    int64_t* tg = p.tokens + static_cast<int64_t>(g) * (k + 1);
    if (k + 1 <= kPackedUnits) {
      // each unit stores its token where it belongs and arrives with its
      // rejection bit (bits 0..4 count the arrivals, bit 5 + i is position
      // i's rejection): the last arrival holds every bit and only replaces
      // the positions after the first rejection by -1
      if (t == 0) {
        store_sc64(reinterpret_cast<uint64_t*>(tg + i), static_cast<uint64_t>(token));
        drain_stores();
        const uint32_t mine = 1u + (acc || i == k ? 0u : 1u << (5 + i));
        const uint32_t old = atomic_add_u32(p.grp_cnt + g, mine);
        if ((old & 31u) == static_cast<uint32_t>(k)) {
          const uint32_t rej = (old + mine) >> 5;
          const int a = rej ? __builtin_ctz(rej) : k;
          for (int pos = a + 1; pos <= k; ++pos) store_sc64(reinterpret_cast<uint64_t*>(tg + pos), ~0ull);
          p.accept_len[g] = a;
          atomic_store_u32(p.grp_cnt + g, 0u);
        }
      }
    } else {
      if (t == 0) {
        store_sc64(p.words + static_cast<int64_t>(g) * (k + 1) + i,
                   static_cast<uint64_t>(token) | (acc ? (1ull << 63) : 0ull));
        drain_stores();
        const uint32_t old = atomic_arrive(p.grp_cnt + g);
        f.last = old == static_cast<uint32_t>(k) ? 1u : 0u;
      }
      __syncthreads();
      if (f.last && t < kWave) {
        // accepted length: the first rejected position (k if none), 64 positions per pass
        const uint64_t* wg = p.words + static_cast<int64_t>(g) * (k + 1);
        int a = k;
        for (int b0 = 0; b0 < k && a == k; b0 += kWave) {
          const int pos = b0 + t;
          const uint64_t wd = pos < k ? load_sc64(wg + pos) : (1ull << 63);
          const uint64_t rej = __ballot(!(wd >> 63));
          if (rej) a = b0 + __builtin_ctzll(rej);
        }
        for (int b0 = 0; b0 <= k; b0 += kWave) {
          const int pos = b0 + t;
          if (pos <= k) {
            const int64_t tokv = pos <= a ? static_cast<int64_t>(load_sc64(wg + pos) & 0x7fffffffffffffffull) : -1;
            tg[pos] = tokv;
          }
        }
        if (t == 0) {
          p.accept_len[g] = a;
          atomic_store_u32(p.grp_cnt + g, 0u);
        }
      }
    }
  } else if (p.mode == kModeSample) {
    const int64_t token = draw_target<DT>(p, f, rows[0], K[0], u_draw);
    if (t == 0) p.row_tokens[rows[0]] = token;
  } else {
    // the support into the row of zeros that the streaming pass wrote; dense_kernel
    // writes the rows whose support is not in the list
    if (p.zero_out && (f.aux[0].flags & kRowList)) {
      const RowAux& a = f.aux[0];
      float* out = p.filt_out + static_cast<int64_t>(rows[0]) * p.filt_stride;
      const uint32_t n = a.n;
      for (uint32_t e = t; e < n; e += kFW) {
        const float P = filtered_of(a, __uint_as_float(f.ent[0].pbits[e]));
        if (P > 0.0f) out[f.ent[0].eidx[e]] = P;
      }
    }
    if (t == 0) {
      const RowAux& a = f.aux[0];
      RowStat st;
      st.mcmax = a.mcmax;
      st.s = a.s;
      st.cutoff = a.cut;
      st.mass = a.mass_f;
      st.flags = a.flags;
      st.pad = 0;
      st.mass_fx = a.mass_fx;
      p.stats[rows[0]] = st;
      const bool filt = a.flags & kRowFiltered;
      if (p.cutoff_out) p.cutoff_out[rows[0]] = filt ? a.cut : 0.0f;
      if (p.mass_out) p.mass_out[rows[0]] = filt ? a.mass_f : 1.0f;
    }
  }
}

// One workgroup per CU when every unit has a CU of its own. kTopK: the build
// with the top-k step (launched only for calls with 1 <= top_k < V, so that
// the other calls run code without it).
template <int DT, bool kTopK>
__global__ __launch_bounds__(kFW) __attribute__((amdgpu_flat_work_group_size(kFW, kFW)))
void fin_kernel(const Params p) {
  __shared__ FinShT<11> f;
  fin_unit<DT, kTopK>(p, f);
}

// Two workgroups per CU (the LDS is under 80 KB; at most 128 registers) for
// calls with more units than CUs: one round instead of two.
template <int DT, bool kTopK>
__global__ __launch_bounds__(kFW) __attribute__((amdgpu_flat_work_group_size(kFW, kFW), amdgpu_waves_per_eu(4, 4)))
void fin2_kernel(const Params p) {
  __shared__ FinShT<10> f;
  fin_unit<DT, kTopK>(p, f);
}
// ===========================================================================
// dense_kernel: p and the filtered distribution for one (row, chunk) item
// ===========================================================================
constexpr int kCB = 256;

// N consecutive floats (N a multiple of 4), 16 bytes at a time where the rows allow.
template <int N>
__device__ __forceinline__ void store_floats(float* out, const float (&v)[N], bool vec) {
  if (vec) {
#pragma unroll
    for (int e = 0; e < N; e += 4)
      __builtin_nontemporal_store(f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]}, reinterpret_cast<f32x4*>(out + e));
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) out[e] = v[e];
  }
}

template <int DT>
__global__ __launch_bounds__(kCB) void dense_kernel(const Params p) {
  constexpr int EPV = Elem<DT>::kPerVec;
  constexpr int NVC = kChunk / (kCB * EPV);
  const int t = threadIdx.x;
  const int item = blockIdx.x;
  const int64_t r = item / p.nch;
  const int cj = item - static_cast<int>(r) * p.nch;
  const RowStat st = p.stats[r];
  if (p.zero_out && (st.flags & kRowList)) return;  // the finaliser wrote the row
  const char* rowp = p.base0 + r * p.bstride0;
  const int c0 = cj * kChunk;
  const int nel = p.vocab - c0 < kChunk ? p.vocab - c0 : kChunk;
  const int nvc = nel / EPV;
  const u32x4* src = reinterpret_cast<const u32x4*>(rowp) + c0 / EPV;
  const RowK K{st.mcmax, st.s, p.cd};
  RowAux a{};
  a.flags = st.flags;
  a.cut = st.cutoff;
  a.mass_f = st.mass;
  a.mass_fx = st.mass_fx;
  u32x4 d[NVC];
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
    const int v = u * kCB + t;
    d[u] = __builtin_nontemporal_load(src + (v < nvc ? v : nvc - 1));
  }
#pragma unroll
  for (int u = 0; u < NVC; ++u) {
    const int v = u * kCB + t;
    if (v < nvc) {
      float pv[EPV], fv[EPV];
#pragma unroll
      for (int e = 0; e < EPV; ++e) {
        pv[e] = pval(K, vec_elem<DT>(d[u], e));
        fv[e] = filtered_of(a, pv[e]);
      }
      const int64_t i = c0 + static_cast<int64_t>(v) * EPV;
      if (p.probs_out) store_floats(p.probs_out + r * p.probs_stride + i, pv, p.vec_out);
      if (p.filt_out) store_floats(p.filt_out + r * p.filt_stride + i, fv, p.vec_out);
    }
  }
}

// ===========================================================================
// Host side
// ===========================================================================
struct Layout {
  uint64_t grp_cnt, recs, cands, stats, words, bitmap, total;
};

int nch_for(int64_t vocab) { return static_cast<int>((vocab + kChunk - 1) / kChunk); }
int cap_for(int nch) { return nch <= 32 ? 64 : (nch <= 64 ? 32 : 16); }

// Workspace: [group counters] -- at a fixed place sized for the largest call,
// so that calls of any shape on one workspace find them zero (each call leaves
// them zero) -- then, shaped by the call, [chunk records] [candidate slots]
// [row statistics] [published words] [penalty bitmaps].
Layout ws_layout(int64_t rows, int64_t words, int64_t groups, int nch) {
  auto al = [](uint64_t x) { return (x + 255u) & ~255ull; };
  Layout l{};
  uint64_t off = 0;
  l.grp_cnt = off;
  off = al(off + static_cast<uint64_t>(kMaxSpecBatch) * 4u);
  l.recs = off;
  off = al(off + static_cast<uint64_t>(rows) * nch * sizeof(ChunkRec));
  l.cands = off;
  off = al(off + static_cast<uint64_t>(rows) * nch * cap_for(nch) * 8u);
  l.stats = off;
  off = al(off + static_cast<uint64_t>(rows) * sizeof(RowStat));
  l.words = off;
  off = al(off + static_cast<uint64_t>(words) * 8u);
  l.bitmap = off;
  off = al(off + static_cast<uint64_t>(groups) * nch * (kChunk / 32) * 4u);
  l.total = off;
  return l;
}

void bind_workspace(Params& p, void* ws, const Layout& l) {
  char* b = static_cast<char*>(ws);
  p.grp_cnt = reinterpret_cast<uint32_t*>(b + l.grp_cnt);
  p.recs = reinterpret_cast<ChunkRec*>(b + l.recs);
  p.cands = reinterpret_cast<uint64_t*>(b + l.cands);
  p.stats = reinterpret_cast<RowStat*>(b + l.stats);
  p.words = reinterpret_cast<uint64_t*>(b + l.words);
  p.bitmap = reinterpret_cast<uint32_t*>(b + l.bitmap);
}

template <int DT>
void launch_dt(const Params& p, hipStream_t st) {
  if (p.use_pen) hipLaunchKernelGGL(bitmap_kernel, dim3(static_cast<unsigned>(p.groups)), dim3(kBmB), 0, st, p);
  const dim3 sgrid(static_cast<unsigned>((p.items + kNW - 1) / kNW));
  if (p.use_pen) {
    hipLaunchKernelGGL((stream_kernel<DT>), sgrid, dim3(kWG), 0, st, p);
  } else {
    hipLaunchKernelGGL((stream_reg_kernel<DT>), sgrid, dim3(kWG), 0, st, p);
  }
  const dim3 fgrid(static_cast<unsigned>(p.units));
  if (p.units > device_cu_count()) {
    if (p.top_k) {
      hipLaunchKernelGGL((fin2_kernel<DT, true>), fgrid, dim3(kFW), 0, st, p);
    } else {
      hipLaunchKernelGGL((fin2_kernel<DT, false>), fgrid, dim3(kFW), 0, st, p);
    }
  } else if (p.top_k) {
    hipLaunchKernelGGL((fin_kernel<DT, true>), fgrid, dim3(kFW), 0, st, p);
  } else {
    hipLaunchKernelGGL((fin_kernel<DT, false>), fgrid, dim3(kFW), 0, st, p);
  }
  if (p.mode == kModeDense && (p.probs_out || p.filt_out)) {
    hipLaunchKernelGGL((dense_kernel<DT>), dim3(static_cast<unsigned>(p.items)), dim3(kCB), 0, st, p);
  }
}

int launch(const Params& p, int dtype, hipStream_t st) {
  switch (dtype) {
    case LS_DTYPE_F32: launch_dt<F32>(p, st); break;
    case LS_DTYPE_BF16: launch_dt<BF16>(p, st); break;
    case LS_DTYPE_F16: launch_dt<F16>(p, st); break;
    default: return fail(LS_ERR_VALUE, "unsupported logits dtype");
  }
  return check_launch("sampling kernel launch");
}

// Shared argument validation / setup for the processing options.
int setup_common(Params& p, int dtype, int64_t rows, int64_t vocab, float temperature, float top_p, int64_t top_k,
                 float penalty, const int32_t* history, int64_t history_stride, const int32_t* history_len) {
  const int eb = dtype_bytes(dtype);
  if (eb == 0) return fail(LS_ERR_VALUE, "unsupported logits dtype");
  if (vocab <= 0 || vocab > kMaxVocab) return fail(LS_ERR_VALUE, "vocabulary size must be in [1, 262144]");
  if ((vocab * eb) % 16 != 0) return fail(LS_ERR_VALUE, "vocabulary row bytes must be a multiple of 16");
  if (rows > kMaxRows) return fail(LS_ERR_VALUE, "at most 65536 logit rows per call");
  if (!(temperature > 0.0f)) return fail(LS_ERR_VALUE, "temperature must be > 0");
  if (!(top_p > 0.0f) || top_p > 1.0f) return fail(LS_ERR_VALUE, "top_p must be in (0, 1]");
  if (top_k < 0) return fail(LS_ERR_VALUE, "top_k must be >= 0");
  if (!(penalty > 0.0f)) return fail(LS_ERR_VALUE, "repetition penalty must be > 0");
  if (penalty != 1.0f && (history == nullptr || history_len == nullptr))
    return fail(LS_ERR_VALUE, "repetition penalty needs a token history");
  if (penalty != 1.0f && (history_stride < 0 || history_stride > 0x7fffffffLL))
    return fail(LS_ERR_VALUE, "history_stride must be in [0, 2^31)");
  p.vocab = static_cast<int>(vocab);
  p.nch = nch_for(vocab);
  p.cap = cap_for(p.nch);
  p.bm_words = p.nch * (kChunk / 32);
  p.items = static_cast<int>(rows * p.nch);
  p.cd = kLog2eD / static_cast<double>(temperature);
  p.c = static_cast<float>(p.cd);
  p.use_pen = penalty != 1.0f;
  p.pen = penalty;
  p.top_p = top_p;
  p.top_k = top_k > 0 && top_k < vocab ? static_cast<int>(top_k) : 0;
  p.hist = history;
  p.hist_stride = history_stride;
  p.hist_len = history_len;
  return LS_OK;
}

// Zeroes n 32-bit words (a kernel, not a memset, so that it may be captured
// into a graph and replayed).
__global__ void zero_words_kernel(uint32_t* p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

}  // namespace
}  // namespace ls

// ---------------------------------------------------------------------------
// Static scratch of ls_spec_verify_noalloc: the workspace of one call, kept in
// this GPU's copy of a file-scope array for the life of the process. Host code
// uses the address hipGetSymbolAddress returns for the current device, never
// the array's name.
// ---------------------------------------------------------------------------
constexpr uint64_t kNoAllocScratchBytes = 16ull << 20;  // 16 MiB per GPU
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices];  // per device, null until set up

// The current device's scratch address. The first call on a device looks it
// up and zeroes the group counters there (on `st`); every call leaves them
// zero again.
int scratch_for_current_device(hipStream_t st, void** out) {
  int dev = -1;
  LS_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxScratchDevices) return ls::fail(LS_ERR_RUNTIME, "spec_verify_noalloc: device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return ls::hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return ls::fail(LS_ERR_RUNTIME, "spec_verify_noalloc: no scratch address");
    const int64_t words = ls::kMaxSpecBatch;  // the group counters at the workspace's start
    hipLaunchKernelGGL(ls::zero_words_kernel, dim3(static_cast<unsigned>((words + 255) / 256)), dim3(256), 0, st,
                       static_cast<uint32_t*>(p), words);
    const int rc = ls::check_launch("spec_verify_noalloc scratch set-up");
    if (rc) return rc;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return LS_OK;
}
}  // namespace

using namespace ls;

extern "C" {

uint64_t ls_spec_verify_workspace(int64_t batch, int64_t k, int64_t vocab) {
  if (batch <= 0 || k < 1 || vocab <= 0) return 0;
  return ws_layout(batch * (2 * k + 1), batch * (k + 1), batch, nch_for(vocab)).total;
}

int ls_spec_verify(const void* target_logits, int64_t target_batch_stride, int64_t target_pos_stride,
                   const void* draft_logits, int64_t draft_batch_stride, int64_t draft_pos_stride,
                   const int64_t* draft_tokens, const float* uniforms, int dtype, int64_t batch, int64_t k,
                   int64_t vocab, float temperature, float top_p, int64_t top_k, float penalty,
                   const int32_t* history, int64_t history_stride, const int32_t* history_len,
                   int32_t* accept_len, int64_t* tokens, void* workspace, uint64_t ws_bytes, ls_stream_t stream) {
  if (batch < 0 || batch > kMaxSpecBatch || k < 1 || k > 64)
    return fail(LS_ERR_VALUE, "spec_verify: need 0 <= batch <= 16384 and 1 <= k <= 64");
  if (batch == 0) return LS_OK;
  if (!target_logits || !draft_logits || !draft_tokens || !uniforms || !accept_len || !tokens)
    return fail(LS_ERR_VALUE, "spec_verify: NULL pointer");
  Params p{};
  const int64_t rows = batch * (2 * k + 1);
  int rc = setup_common(p, dtype, rows, vocab, temperature, top_p, top_k, penalty, history, history_stride,
                        history_len);
  if (rc) return rc;
  const int eb = dtype_bytes(dtype);
  p.base0 = static_cast<const char*>(target_logits);
  p.bstride0 = target_batch_stride * eb;
  p.pstride0 = target_pos_stride * eb;
  p.base1 = static_cast<const char*>(draft_logits);
  p.bstride1 = draft_batch_stride * eb;
  p.pstride1 = draft_pos_stride * eb;
  if (!aligned16(target_logits) || !aligned16(draft_logits) || p.bstride0 % 16 || p.pstride0 % 16 ||
      p.bstride1 % 16 || p.pstride1 % 16)
    return fail(LS_ERR_VALUE, "spec_verify: logits rows must be 16-byte aligned");
  p.mode = kModeSpec;
  p.k = static_cast<int>(k);
  p.rpg = static_cast<int>(2 * k + 1);
  p.groups = static_cast<int>(batch);
  p.units = static_cast<int>(batch * (k + 1));
  p.draft_tokens = draft_tokens;
  p.uniforms = uniforms;
  p.accept_len = accept_len;
  p.tokens = tokens;
  const Layout l = ws_layout(rows, batch * (k + 1), batch, p.nch);
  if (!workspace || ws_bytes < l.total) return fail(LS_ERR_VALUE, "spec_verify: workspace too small");
  bind_workspace(p, workspace, l);
  return launch(p, dtype, static_cast<hipStream_t>(stream));
}

int ls_spec_verify_noalloc(const void* target_logits, int64_t target_batch_stride, int64_t target_pos_stride,
                           const void* draft_logits, int64_t draft_batch_stride, int64_t draft_pos_stride,
                           const int64_t* draft_tokens, const float* uniforms, int dtype, int64_t batch, int64_t k,
                           int64_t vocab, float temperature, float top_p, int64_t top_k, float penalty,
                           const int32_t* history, int64_t history_stride, const int32_t* history_len,
                           int32_t* accept_len, int64_t* tokens, ls_stream_t stream) {
  const uint64_t need = (batch > 0 && k >= 1 && vocab > 0) ? ls_spec_verify_workspace(batch, k, vocab) : 0;
  if (need > kNoAllocScratchBytes)
    return fail(LS_ERR_VALUE, "spec_verify_noalloc: the call needs " + std::to_string(need) +
                                  " bytes of scratch, above the 16 MiB static scratch; use ls_spec_verify with a workspace");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  void* ws = nullptr;
  const int rc = scratch_for_current_device(st, &ws);
  if (rc) return rc;
  return ls_spec_verify(target_logits, target_batch_stride, target_pos_stride, draft_logits, draft_batch_stride,
                        draft_pos_stride, draft_tokens, uniforms, dtype, batch, k, vocab, temperature, top_p, top_k,
                        penalty, history, history_stride, history_len, accept_len, tokens, ws, kNoAllocScratchBytes,
                        stream);
}

uint64_t ls_sample_logits_workspace(int64_t rows, int64_t vocab) {
  if (rows <= 0 || vocab <= 0) return 0;
  return ws_layout(rows, 0, rows, nch_for(vocab)).total;
}

int ls_sample_logits(const void* logits, int64_t row_stride, int dtype, int64_t rows, int64_t vocab,
                     float temperature, float top_p, int64_t top_k, float penalty, const int32_t* history,
                     int64_t history_stride, const int32_t* history_len, const float* uniforms,
                     int64_t* out_tokens, void* workspace, uint64_t ws_bytes, ls_stream_t stream) {
  if (rows < 0 || rows > kMaxRows) return fail(LS_ERR_VALUE, "sample_logits: need 0 <= rows <= 65536");
  if (rows == 0) return LS_OK;
  if (!logits || !uniforms || !out_tokens) return fail(LS_ERR_VALUE, "sample_logits: NULL pointer");
  Params p{};
  int rc = setup_common(p, dtype, rows, vocab, temperature, top_p, top_k, penalty, history, history_stride,
                        history_len);
  if (rc) return rc;
  const int eb = dtype_bytes(dtype);
  p.base0 = static_cast<const char*>(logits);
  p.bstride0 = row_stride * eb;
  if (!aligned16(logits) || p.bstride0 % 16) return fail(LS_ERR_VALUE, "sample_logits: rows must be 16-byte aligned");
  p.mode = kModeSample;
  p.rpg = 1;
  p.k = 0;
  p.groups = static_cast<int>(rows);
  p.units = static_cast<int>(rows);
  p.row_uniforms = uniforms;
  p.row_tokens = out_tokens;
  const Layout l = ws_layout(rows, 0, rows, p.nch);
  if (!workspace || ws_bytes < l.total) return fail(LS_ERR_VALUE, "sample_logits: workspace too small");
  bind_workspace(p, workspace, l);
  return launch(p, dtype, static_cast<hipStream_t>(stream));
}

uint64_t ls_filter_logits_workspace(int64_t rows, int64_t vocab) {
  if (rows <= 0 || vocab <= 0) return 0;
  return ws_layout(rows, 0, rows, nch_for(vocab)).total;
}

int ls_filter_logits(const void* logits, int64_t row_stride, int dtype, int64_t rows, int64_t vocab,
                     float temperature, float top_p, const float* top_p_rows, int64_t top_k, float* probs_out,
                     int64_t probs_stride, float* filtered_out, int64_t filtered_stride, float* cutoff_out,
                     float* mass_out, void* workspace, uint64_t ws_bytes, ls_stream_t stream) {
  if (rows < 0 || rows > kMaxRows) return fail(LS_ERR_VALUE, "filter_logits: need 0 <= rows <= 65536");
  if (rows == 0) return LS_OK;
  if (!logits) return fail(LS_ERR_VALUE, "filter_logits: NULL logits");
  Params p{};
  int rc = setup_common(p, dtype, rows, vocab, temperature, top_p, top_k, 1.0f, nullptr, 0, nullptr);
  if (rc) return rc;
  const int eb = dtype_bytes(dtype);
  p.base0 = static_cast<const char*>(logits);
  p.bstride0 = row_stride * eb;
  if (!aligned16(logits) || p.bstride0 % 16) return fail(LS_ERR_VALUE, "filter_logits: rows must be 16-byte aligned");
  p.mode = kModeDense;
  p.rpg = 1;
  p.k = 0;
  p.groups = static_cast<int>(rows);
  p.units = static_cast<int>(rows);
  p.top_p_rows = top_p < 1.0f ? top_p_rows : nullptr;
  p.probs_out = probs_out;
  p.probs_stride = probs_stride;
  p.filt_out = filtered_out;
  p.filt_stride = filtered_stride;
  p.cutoff_out = cutoff_out;
  p.mass_out = mass_out;
  p.vec_out = (!probs_out || (aligned16(probs_out) && probs_stride % 4 == 0)) &&
              (!filtered_out || (aligned16(filtered_out) && filtered_stride % 4 == 0));
  // Without the unfiltered rows, a filtered row is zeros but for its support,
  // which the finaliser holds: no second pass over the logits (64 rows, V 49152
  // f32, T 1, top-p 0.7: 23.5 us a call with dense_kernel writing every row, 21.3
  // so; 200 rows, V 128256 bf16 128.5 and 120.6). The rule cannot know the
  // supports: a row whose support is not in the finaliser's list is written
  // twice, the zeros for nothing (top-p 0.95: 50.9 and 53.7; 115.4 and 129.2;
  // unfiltered rows, by a top_p_rows of 1, 18.5 and 21.0).
  // Not where the output overlaps the logits, which the finaliser may read again.
  auto disjoint = [&](const void* x, int64_t xs, int64_t xb, const void* y, int64_t ys, int64_t yb) {
    const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), y0 = reinterpret_cast<uintptr_t>(y);
    const uintptr_t x1 = x0 + static_cast<uintptr_t>(((rows - 1) * xs + vocab) * xb);
    const uintptr_t y1 = y0 + static_cast<uintptr_t>(((rows - 1) * ys + vocab) * yb);
    return x1 <= y0 || y1 <= x0;
  };
  p.zero_out = filtered_out && !probs_out && p.vec_out && (top_p < 1.0f || p.top_k) && row_stride >= 0 &&
               filtered_stride >= vocab && disjoint(logits, row_stride, eb, filtered_out, filtered_stride, 4);
  const Layout l = ws_layout(rows, 0, rows, p.nch);
  if (!workspace || ws_bytes < l.total) return fail(LS_ERR_VALUE, "filter_logits: workspace too small");
  bind_workspace(p, workspace, l);
  return launch(p, dtype, static_cast<hipStream_t>(stream));
}

}  // extern "C"
