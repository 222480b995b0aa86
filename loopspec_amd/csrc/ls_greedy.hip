// (b) Greedy verification for gfx950.
//
// One launch covers every row of the step. Rows are cut into `splits` equal
// segments, with splits chosen so that the segments spread evenly over the CUs
// (C2: 320 rows x 4 segments = 5 workgroups on each of 256 CUs) and every lane
// issues all of its 16-byte non-temporal loads up front (J loads per lane, a
// template constant when the segment is an exact multiple of the workgroup).
// A lane keeps a (vector-max, vector) candidate, resolves the first index of
// the maximum inside the winning vector, and the block reduces packed
// (value, -index) keys. Segments meet in the fused epilogue without
// same-address contention: each workgroup writes its key to its own slot with
// a device-coherent store and arrives on its batch element's
// counter; the last arriver loads the element's keys, takes the per-row
// maximum over segments and runs the accept-prefix scan.
//
// Reference semantics: torch.argmax over the endpoint rows
// (sglang_recurrent/loopspec/decisions.py:116) and the final-endpoint rule
// (decisions.py:157-170) applied along the accept prefix (pipeline.py:365-412).
#include "ls_common.hpp"
#include "ls_runtime.hpp"

namespace ls {
namespace {

constexpr int kUnroll = 8;
// Arrival counters sit one 64-byte line apart: device-scope atomics on one
// line serialise, and adjacent counters of concurrently finishing groups
// measured several microseconds of queueing on MI355X. They live at a fixed
// place (the first kMaxGroups lines of the workspace) so that the key slots of
// a call with another shape never overlap them.
constexpr int kCounterStride = 16;
constexpr int64_t kMaxGroups = 16384;
// Workspace: the counter lines, one 256-byte line holding the sticky status
// word, then the key slots.
constexpr uint64_t kStatusOffset = static_cast<uint64_t>(kMaxGroups) * kCounterStride * 4u;
constexpr uint64_t kSlotsOffset = kStatusOffset + 256u;
// Status bit: some split's key was not visible within the poll limit, so a
// row's maximum was taken without it.
constexpr uint32_t kStatusKeyTimeout = 1u;
constexpr int kMaxSplits = 16;
constexpr int kMaxRowsPerGroup = 2 * 64 + 1;

struct GreedyParams {
  const char* target;        // row (b, i) at target + b*t_bstride + i*t_pstride (bytes)
  int64_t t_bstride, t_pstride;
  const char* draft;         // NULL when draft ids are supplied
  int64_t d_bstride, d_pstride;
  const int64_t* draft_tokens;
  int64_t vocab;
  int64_t nvec;              // 16-byte vectors per row (at most, for rows at any element)
  int64_t seg;               // vectors per split
  int k;                     // draft positions (verify mode); 0 in argmax mode
  int rows_per_group;        // argmax: 1; verify: (k+1) [+ k when draft logits given]
  int splits;                // workgroups per row
  int direct;                // argmax mode with splits == 1: write out[] directly
  int64_t* out;              // argmax mode output [rows]
  int32_t* accept_len;       // verify outputs
  int64_t* tokens;
  int64_t* row_argmax;
  uint64_t* slots;           // workspace: one key per (row, split)
  uint32_t* counters;        // workspace: one arrival counter per group, kCounterStride apart
  uint32_t* status;          // workspace: sticky status bits (kStatusKeyTimeout)
};

// Row j of group g (verify rows: target positions 0..k, then draft positions
// 0..k-1; argmax mode: row g).
__device__ __forceinline__ const char* row_ptr(const GreedyParams& p, int64_t g, int j) {
  if (j <= p.k) return p.target + g * p.t_bstride + j * p.t_pstride;
  return p.draft + g * p.d_bstride + (j - p.k - 1) * p.d_pstride;
}

// First-index argmax key of this lane's share of vectors [v0, v1) of a row.
// The lane's vectors are v0 + lane + j*BLOCK for j < n. Loads go through a
// clamped address (lanes past their last vector re-read it and ignore the
// result), so a batch of loads is issued without branches and each vector is
// consumed as soon as its own load returns. J > 0: the whole share is one batch
// of exactly J loads (J = n for every lane when the segment is J*BLOCK
// vectors); J == 0: batches of kUnroll.
template <int DT, int BLOCK, int J>
__device__ __forceinline__ uint64_t thread_argmax_vec(const u32x4* __restrict__ src, int64_t v0, int64_t v1) {
  constexpr int EPV = Elem<DT>::kPerVec;
  constexpr int kBatch = J > 0 ? J : kUnroll;
  const int64_t first = v0 + threadIdx.x;
  if (first >= v1) return 0;
  const int n = J > 0 ? J : static_cast<int>((v1 - first + BLOCK - 1) / BLOCK);
  const u32x4* __restrict__ p = src + first;
  float best = -__builtin_inff();
  int bestj = 0;
  u32x4 bestd = {0u, 0u, 0u, 0u};
  for (int j0 = 0; j0 < n; j0 += kBatch) {
    u32x4 d[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int j = J > 0 ? u : (j0 + u < n ? j0 + u : n - 1);
      d[u] = __builtin_nontemporal_load(p + static_cast<int64_t>(j) * BLOCK);
    }
    // Every load of the batch is issued before any of them is consumed: the
    // scheduler would otherwise interleave the first vectors' decoding with
    // the issue and wait on them before the last loads leave.
    __builtin_amdgcn_sched_barrier(0);
    // Seeding with the lane's first vector makes an all -inf share resolve to
    // its first element without a sentinel.
    if (j0 == 0) bestd = d[0];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const float g = vec_max<DT>(d[u]);
      // Vectors arrive in increasing index order, so a strict '>' keeps the
      // earliest vector holding the maximum; a NaN beats any number once.
      const bool in = J > 0 ? true : (j0 + u < n);
      const bool take = in & ((g > best) | ((g != g) & (best == best)));
      best = take ? g : best;
      bestj = take ? j0 + u : bestj;
      bestd = take ? d[u] : bestd;
    }
    if constexpr (J > 0) break;
  }
  // First element of the winning vector equal to the maximum (or the first
  // NaN), by selects from the last element down.
  const bool is_nan = best != best;
  int e = 0;
#pragma unroll
  for (int q = EPV - 1; q >= 0; --q) {
    const float x = vec_elem<DT>(bestd, q);
    const bool hit = (x == best) | (is_nan & (x != x));
    e = hit ? q : e;
  }
  const int64_t v = first + static_cast<int64_t>(bestj) * BLOCK;
  return argmax_key(best, static_cast<uint32_t>(v * EPV + e));
}

// The same over a row that starts or ends at any element, segment `split` of
// `splits` segments of `seg` vectors: 16-byte vectors from the row's first
// 16-byte boundary on (the boundary differs from row to row when the row size is
// not a multiple of 16 bytes); the elements before it are the first segment's,
// one per lane, those after the last whole vector the last segment's. Nothing
// outside the row is read. (One element per lane and step, as rows like these
// went before: B 96, k 3, V 50257 in f16, 38.6 MB, 38.5 us a call against 10.9;
// B 200, k 8, V 32003 in bf16 134 against 38.)
template <int DT, int BLOCK>
__device__ __forceinline__ uint64_t thread_argmax_any(const char* row, int64_t vocab, int split, int splits,
                                                      int64_t seg) {
  constexpr int EPV = Elem<DT>::kPerVec, EB = Elem<DT>::kBytes;
  const int64_t to_boundary = static_cast<int64_t>((16u - (reinterpret_cast<uintptr_t>(row) & 15u)) & 15u) / EB;
  const int64_t head = to_boundary < vocab ? to_boundary : vocab;
  const int64_t nvec = (vocab - head) / EPV;
  const int64_t v0 = split * seg, v1 = v0 + seg < nvec ? v0 + seg : nvec;
  uint64_t key = thread_argmax_vec<DT, BLOCK, 0>(reinterpret_cast<const u32x4*>(row + head * EB), v0, v1);
  if (key) key -= static_cast<uint64_t>(head);  // the key's low word is ~index
  const int64_t t = threadIdx.x;
  auto element = [&](int64_t i) {
    const uint64_t k = argmax_key(load_elem<DT>(row, i), static_cast<uint32_t>(i));
    key = k > key ? k : key;
  };
  if (split == 0 && t < head) element(t);
  const int64_t tail = head + nvec * EPV;
  if (split == splits - 1 && tail + t < vocab) element(tail + t);
  return key;
}

// A published key is never zero (its low word is ~index with index < 2^31),
// so an empty slot reads as 0. Keys are stored without waiting for the store
// to complete before the arrival: the last arriver polls each slot until its
// key is visible (every store it waits for was issued before the matching
// arrival, so the wait ends; the poll count is bounded regardless) and clears
// it for the next call. A poll that runs out sets kStatusKeyTimeout in the
// sticky status word, which ls_greedy_workspace_status reports; it then
// clears the word and every key slot (a late key could otherwise be read by
// the next launch).
constexpr int kPollLimit = 1 << 22;

__device__ __forceinline__ uint64_t take_key(uint64_t* slot, uint32_t* status) {
  uint64_t v = load_sc64(slot);
  for (int n = 0; v == 0 && n < kPollLimit; ++n) {
    __builtin_amdgcn_s_sleep(1);
    v = load_sc64(slot);
  }
  if (v == 0) atomic_or_u32(status, kStatusKeyTimeout);
  store_sc64(slot, 0);
  return v;
}

// Wave 0 of the last workgroup of group g when the group has at most 64
// keys: lane i holds key i (this workgroup's own from registers, the others
// from `pre` when already loaded, else polled for). Row j's key is the maximum over its splits' keys; the accept-prefix
// scan is lane-parallel (lane i compares draft position i, one ballot finds
// the first mismatch, lane i writes output position i).
__device__ __forceinline__ void finalize_small(const GreedyParams& p, int64_t g, int own, uint64_t own_key,
                                               uint64_t pre) {
  const int lane = threadIdx.x & (kWave - 1);
  const int k = p.k;
  const int rpg = p.rows_per_group, splits = p.splits;
  const int nkeys = rpg * splits;
  uint64_t* slots = p.slots + g * nkeys;
  const int64_t dtok = (k > 0 && !p.draft && lane < k) ? p.draft_tokens[g * k + lane] : -1;
  uint64_t key = 0;
  if (lane == own) {
    key = own_key;
  } else if (lane < nkeys) {
    // take_key polls until the key is visible and clears the slot; a key
    // already loaded is visible, so clearing it now comes after its store
    if (pre != 0) {
      key = pre;
      store_sc64(slots + lane, 0);
    } else {
      key = take_key(slots + lane, p.status);
    }
  }
  // this workgroup's slot is cleared by the lane that stored it (program order)
  if (lane == 0) store_sc64(slots + own, 0);
  uint64_t best = 0;
  for (int s = 0; s < splits; ++s) {
    const uint64_t o = __shfl(key, lane < rpg ? lane * splits + s : 0);
    best = o > best ? o : best;
  }
  const int64_t id = lane < rpg ? static_cast<int64_t>(argmax_key_index(best)) : -1;
  if (lane == 0) store_sc(p.counters + g * kCounterStride, 0u);
  if (k == 0) {
    if (lane == 0) p.out[g] = id;
    return;
  }
  // draft id of position lane: the draft row's argmax or the caller's id
  const int64_t d = p.draft ? __shfl(id, lane < k ? k + 1 + lane : 0) : dtok;
  const uint64_t bad = __ballot(lane < k && d != id);
  const int a = bad ? __builtin_ctzll(bad) : k;
  if (lane <= k) p.tokens[g * (k + 1) + lane] = lane <= a ? id : -1;
  if (p.row_argmax) {
    if (lane <= k) p.row_argmax[g * (2 * k + 1) + lane] = id;
    if (lane < k) p.row_argmax[g * (2 * k + 1) + k + 1 + lane] = d;
  }
  if (lane == 0) p.accept_len[g] = a;
}

// Runs on every lane of the last workgroup of group g (a block-uniform
// branch), when the group has more than 64 keys. Row j's key is the maximum over its splits' keys. The
// accept-prefix scan is lane-parallel: lane i compares draft position i, the
// first mismatch comes from one ballot, and lane i writes output position i,
// so no store waits on another. When the group has at most 64 keys, wave 0
// alone does all of it in registers (no workgroup barrier).
template <int BLOCK>
__device__ void finalize_group(const GreedyParams& p, int64_t g, int own, uint64_t own_key, int64_t* ids,
                               uint64_t* keys) {
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int k = p.k;
  const int rpg = p.rows_per_group, splits = p.splits;
  const int nkeys = rpg * splits;
  uint64_t* slots = p.slots + g * nkeys;
  // the thread that stored this workgroup's key clears it (same address, same
  // thread: the stores land in program order)
  if (t == 0) store_sc64(slots + own, 0);
  if (nkeys <= kWave) {
    if (t >= kWave) return;
    const int64_t dtok = (k > 0 && !p.draft && lane < k) ? p.draft_tokens[g * k + lane] : -1;
    // this workgroup's own key is taken from registers (its store may still be in flight)
    const uint64_t key = lane == own ? own_key : (lane < nkeys ? take_key(slots + lane, p.status) : 0);
    uint64_t best = 0;
    for (int s = 0; s < splits; ++s) {
      const uint64_t o = __shfl(key, lane < rpg ? lane * splits + s : 0);
      best = o > best ? o : best;
    }
    const int64_t id = lane < rpg ? static_cast<int64_t>(argmax_key_index(best)) : -1;
    if (lane == 0) store_sc(p.counters + g * kCounterStride, 0u);
    if (k == 0) {
      if (lane == 0) p.out[g] = id;
      return;
    }
    // draft id of position lane: the draft row's argmax or the caller's id
    const int64_t d = p.draft ? __shfl(id, lane < k ? k + 1 + lane : 0) : dtok;
    const uint64_t bad = __ballot(lane < k && d != id);
    const int a = bad ? __builtin_ctzll(bad) : k;
    if (lane <= k) p.tokens[g * (k + 1) + lane] = lane <= a ? id : -1;
    if (p.row_argmax) {
      if (lane <= k) p.row_argmax[g * (2 * k + 1) + lane] = id;
      if (lane < k) p.row_argmax[g * (2 * k + 1) + k + 1 + lane] = d;
    }
    if (lane == 0) p.accept_len[g] = a;
    return;
  }
  // caller-supplied draft ids go where the draft rows' argmax would be
  if (k > 0 && !p.draft && t < k) ids[k + 1 + t] = p.draft_tokens[g * k + t];
  for (int i = t; i < nkeys; i += BLOCK) keys[i] = i == own ? own_key : take_key(slots + i, p.status);
  __syncthreads();
  for (int j = t; j < rpg; j += BLOCK) {
    uint64_t best = 0;
    for (int s = 0; s < splits; ++s) best = keys[j * splits + s] > best ? keys[j * splits + s] : best;
    ids[j] = argmax_key_index(best);
  }
  __syncthreads();
  if (t == 0) store_sc(p.counters + g * kCounterStride, 0u);
  if (k == 0) {
    if (t == 0) p.out[g] = ids[0];
    return;
  }
  // every wave forms the same mask over draft positions 0..k-1 (k <= 64)
  const uint64_t bad = __ballot(lane < k && ids[k + 1 + lane] != ids[lane]);
  const int a = bad ? __builtin_ctzll(bad) : k;
  if (t <= k) p.tokens[g * (k + 1) + t] = t <= a ? ids[t] : -1;
  if (p.row_argmax) {
    if (t <= k) p.row_argmax[g * (2 * k + 1) + t] = ids[t];
    if (t < k) p.row_argmax[g * (2 * k + 1) + k + 1 + t] = ids[k + 1 + t];
  }
  if (t == 0) p.accept_len[g] = a;
}

// Grid: direct mode (argmax, one workgroup per row) is 1-D over rows;
// otherwise (splits, rows_per_group, groups), so no index division is needed.
template <int DT, bool VEC, int BLOCK, int J>
__global__ __launch_bounds__(BLOCK) void greedy_kernel(GreedyParams p) {
  __shared__ uint64_t red[BLOCK / kWave];
  __shared__ int64_t ids[kMaxRowsPerGroup];
  __shared__ uint64_t keys[kMaxRowsPerGroup * 4];
  __shared__ int last;
  // The row address is formed with selects from parameters that are all
  // fetched in one round of scalar loads (a branch on the row kind would
  // chain dependent kernel-argument loads ahead of the first logits load).
  int64_t tbs = p.t_bstride, tps = p.t_pstride, dbs = p.d_bstride, dps = p.d_pstride;
  int kk = p.k, direct = p.direct;
  asm volatile("" : "+s"(tbs), "+s"(tps), "+s"(dbs), "+s"(dps), "+s"(kk), "+s"(direct));
  const char* tbase = p.target;
  const char* dbase = p.draft;
  const int split = direct ? 0 : static_cast<int>(blockIdx.x);
  const int j = direct ? 0 : static_cast<int>(blockIdx.y);
  const int64_t g = direct ? static_cast<int64_t>(blockIdx.x) : static_cast<int64_t>(blockIdx.z);
  const bool is_t = j <= kk;
  const char* row = (is_t ? tbase : dbase) + g * (is_t ? tbs : dbs) +
                    static_cast<int64_t>(is_t ? j : j - kk - 1) * (is_t ? tps : dps);

  uint64_t key;
  if constexpr (VEC) {
    const int64_t v0 = split * p.seg;
    const int64_t v1 = v0 + p.seg < p.nvec ? v0 + p.seg : p.nvec;
    key = thread_argmax_vec<DT, BLOCK, J>(reinterpret_cast<const u32x4*>(row), v0, v1);
  } else {
    key = thread_argmax_any<DT, BLOCK>(row, p.vocab, split, p.splits, p.seg);
  }
  key = block_max_u64<BLOCK>(key, red);

  if (direct) {
    if (threadIdx.x == 0) p.out[g] = argmax_key_index(key);
    return;
  }
  const int own = j * p.splits + split;
  const int nkeys = p.rows_per_group * p.splits;
  if (nkeys <= kWave) {
    // Wave 0 alone (the other waves are done): thread 0 publishes the key and
    // arrives; the last arriver takes the other keys. (Loading them in every
    // workgroup alongside the arrival, to save the last one a round trip,
    // measured slower: 20 workgroups then read the lines others store to.)
    if (threadIdx.x >= kWave) return;
    uint32_t prev = 0;
    if (threadIdx.x == 0) {
      store_sc64(p.slots + g * nkeys + own, key);
      prev = atomic_arrive(p.counters + g * kCounterStride);
    }
    prev = lane_bcast_u32(prev, 0);
    if (prev != static_cast<uint32_t>(nkeys - 1)) return;
    finalize_small(p, g, own, key, 0);
    return;
  }
  if (threadIdx.x == 0) {
    store_sc64(p.slots + g * nkeys + own, key);
    const uint32_t prev = atomic_arrive(p.counters + g * kCounterStride);
    last = prev == static_cast<uint32_t>(nkeys - 1);
  }
  __syncthreads();
  if (last) finalize_group<BLOCK>(p, g, own, key, ids, keys);
}

// Read-ceiling calibration: greedy_kernel's grid, row addressing and loads
// (every lane issues its J non-temporal 16-byte loads at once), with only an
// exclusive-or of the loaded words kept, one word per wave. It bounds from
// below what any kernel reading the same rows in the same pattern can take.
template <int BLOCK, int J>
__global__ __launch_bounds__(BLOCK) void read_probe_kernel(GreedyParams p, uint32_t* out) {
  int64_t tbs = p.t_bstride, tps = p.t_pstride, dbs = p.d_bstride, dps = p.d_pstride;
  int kk = p.k;
  asm volatile("" : "+s"(tbs), "+s"(tps), "+s"(dbs), "+s"(dps), "+s"(kk));
  const int split = static_cast<int>(blockIdx.x);
  const int j = static_cast<int>(blockIdx.y);
  const int64_t g = static_cast<int64_t>(blockIdx.z);
  const bool is_t = j <= kk;
  const char* row = (is_t ? p.target : p.draft) + g * (is_t ? tbs : dbs) +
                    static_cast<int64_t>(is_t ? j : j - kk - 1) * (is_t ? tps : dps);
  const int64_t v0 = split * p.seg;
  const int64_t v1 = v0 + p.seg < p.nvec ? v0 + p.seg : p.nvec;
  const int64_t first = v0 + threadIdx.x;
  uint32_t acc = 0;
  if (first < v1) {
    const u32x4* src = reinterpret_cast<const u32x4*>(row) + first;
    u32x4 d[J];
#pragma unroll
    for (int u = 0; u < J; ++u) d[u] = __builtin_nontemporal_load(src + static_cast<int64_t>(u) * BLOCK);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < J; ++u) acc ^= d[u][0] ^ d[u][1] ^ d[u][2] ^ d[u][3];
  }
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) acc ^= static_cast<uint32_t>(__shfl_xor(static_cast<int>(acc), m));
  if ((threadIdx.x & (kWave - 1)) == 0) {
    const int64_t wg = (g * p.rows_per_group + j) * p.splits + split;
    out[wg * (BLOCK / kWave) + threadIdx.x / kWave] = acc;
  }
}

// Workspace: kMaxGroups counter lines, the status line, then rows * kMaxSplits
// key slots.
uint64_t workspace_bytes(int64_t rows) {
  const uint64_t slots = static_cast<uint64_t>(rows) * kMaxSplits * 8u;
  return (kSlotsOffset + slots + 255u) & ~255ull;
}

void bind_workspace(GreedyParams& p, void* workspace) {
  char* base = static_cast<char*>(workspace);
  p.counters = reinterpret_cast<uint32_t*>(base);
  p.status = reinterpret_cast<uint32_t*>(base + kStatusOffset);
  p.slots = reinterpret_cast<uint64_t*>(base + kSlotsOffset);
}

struct Shape {
  int block;
  int splits;
  int j;  // loads per lane as a template constant (0: generic batches)
};

// Workgroup shape. Each row is cut into `splits` equal segments; the split
// count minimises the bytes on the busiest CU, ceil(rows*splits / CUs)
// segments of ceil(nvec/splits) vectors each, preferring fewer splits on
// near-ties (each split adds one key to the epilogue). Measured on MI355X
// (C2: 320 bf16 rows of 49152): 4 splits = 5 equal workgroups per CU, 6 loads
// per lane, all in flight at once.
Shape choose_shape(int64_t rows, int64_t vocab, int elem_bytes, int rows_per_group) {
  const int64_t nvec = vocab * elem_bytes / 16 > 0 ? vocab * elem_bytes / 16 : 1;
  int64_t block = option("greedy_block");
  if (block != 256 && block != 512 && block != 1024) block = 256;
  const int64_t max_by_len = nvec / block > 1 ? nvec / block : 1;  // >= one vector per lane
  int64_t max_s = max_by_len < kMaxSplits ? max_by_len : kMaxSplits;
  const int64_t max_by_lds = 4 * kMaxRowsPerGroup / rows_per_group;  // finalizer key buffer
  if (max_s > max_by_lds) max_s = max_by_lds;
  int64_t s = option("greedy_splits");
  if (s <= 0) {
    const int64_t cus = static_cast<int64_t>(device_cu_count());
    double best = 0.0;
    s = 1;
    for (int64_t c = 1; c <= max_s; ++c) {
      const double busiest = static_cast<double>((rows * c + cus - 1) / cus) * static_cast<double>((nvec + c - 1) / c);
      if (c == 1 || busiest < best * 0.97) {
        best = busiest;
        s = c;
      }
    }
  }
  if (s > max_s) s = max_s;
  if (s < 1) s = 1;
  const int64_t seg = (nvec + s - 1) / s;
  int j = 0;
  if (block == 256 && seg % 256 == 0 && seg / 256 >= 1 && seg / 256 <= 8 && nvec % s == 0) j = static_cast<int>(seg / 256);
  return Shape{static_cast<int>(block), static_cast<int>(s), j};
}

template <int DT, bool VEC, int BLOCK, int J>
void launch_one(const GreedyParams& p, int64_t groups, hipStream_t st) {
  const dim3 grid = p.direct ? dim3(static_cast<unsigned>(groups))
                             : dim3(static_cast<unsigned>(p.splits), static_cast<unsigned>(p.rows_per_group),
                                    static_cast<unsigned>(groups));
  hipLaunchKernelGGL((greedy_kernel<DT, VEC, BLOCK, J>), grid, dim3(BLOCK), 0, st, p);
}

template <int DT>
void launch_dt(const GreedyParams& p, const Shape& sh, int64_t groups, bool vec, hipStream_t st) {
  if (!vec) {
    if (sh.block == 1024) {
      launch_one<DT, false, 1024, 0>(p, groups, st);
    } else if (sh.block == 512) {
      launch_one<DT, false, 512, 0>(p, groups, st);
    } else {
      launch_one<DT, false, 256, 0>(p, groups, st);
    }
    return;
  }
  if (sh.block == 1024) {
    launch_one<DT, true, 1024, 0>(p, groups, st);
  } else if (sh.block == 512) {
    launch_one<DT, true, 512, 0>(p, groups, st);
  } else {
    switch (sh.j) {
      case 1: launch_one<DT, true, 256, 1>(p, groups, st); break;
      case 2: launch_one<DT, true, 256, 2>(p, groups, st); break;
      case 3: launch_one<DT, true, 256, 3>(p, groups, st); break;
      case 4: launch_one<DT, true, 256, 4>(p, groups, st); break;
      case 5: launch_one<DT, true, 256, 5>(p, groups, st); break;
      case 6: launch_one<DT, true, 256, 6>(p, groups, st); break;
      case 7: launch_one<DT, true, 256, 7>(p, groups, st); break;
      case 8: launch_one<DT, true, 256, 8>(p, groups, st); break;
      default: launch_one<DT, true, 256, 0>(p, groups, st); break;
    }
  }
}

int launch(const GreedyParams& p, int dtype, const Shape& sh, int64_t groups, bool vec, hipStream_t st) {
  switch (dtype) {
    case LS_DTYPE_F32: launch_dt<F32>(p, sh, groups, vec, st); break;
    case LS_DTYPE_BF16: launch_dt<BF16>(p, sh, groups, vec, st); break;
    case LS_DTYPE_F16: launch_dt<F16>(p, sh, groups, vec, st); break;
    default: return fail(LS_ERR_VALUE, "unsupported logits dtype");
  }
  return check_launch("greedy kernel launch");
}

}  // namespace
}  // namespace ls

using namespace ls;

extern "C" {

uint64_t ls_argmax_rows_workspace(int64_t rows, int64_t vocab) {
  (void)vocab;
  return rows > 0 ? workspace_bytes(rows < kMaxGroups ? rows : kMaxGroups) : 0;
}

int ls_argmax_rows(const void* logits, int dtype, int64_t rows, int64_t vocab, int64_t row_stride,
                   int64_t* out, void* workspace, uint64_t ws_bytes, ls_stream_t stream) {
  const int eb = dtype_bytes(dtype);
  if (eb == 0) return fail(LS_ERR_VALUE, "unsupported logits dtype");
  if (rows < 0 || vocab <= 0 || vocab > 0x7fffffffLL) return fail(LS_ERR_VALUE, "argmax: invalid rows/vocab");
  if (rows == 0) return LS_OK;
  if (logits == nullptr || out == nullptr) return fail(LS_ERR_VALUE, "argmax: NULL pointer");
  if (rows > 0x7fffffffLL) return fail(LS_ERR_VALUE, "argmax: too many rows");
  GreedyParams p{};
  p.target = static_cast<const char*>(logits);
  p.t_bstride = row_stride * eb;  // argmax rows are groups of one row
  p.vocab = vocab;
  p.k = 0;
  p.rows_per_group = 1;
  const bool vec = aligned16(logits) && ((row_stride * eb) % 16 == 0) && ((vocab * eb) % 16 == 0);
  Shape shape = choose_shape(rows, vocab, eb, 1);
  if (shape.splits > 1 && (rows > kMaxGroups || workspace == nullptr || ws_bytes < workspace_bytes(rows))) {
    // Without scratch (or beyond the counter area) one workgroup per row.
    shape.splits = 1;
    shape.j = 0;
  }
  if (!vec) shape.j = 0;
  p.splits = shape.splits;
  p.direct = p.splits == 1;
  p.out = out;
  p.nvec = vocab * eb / 16;
  p.seg = (p.nvec + p.splits - 1) / p.splits;
  if (!p.direct) bind_workspace(p, workspace);
  return launch(p, dtype, shape, rows, vec, static_cast<hipStream_t>(stream));
}

uint64_t ls_greedy_verify_workspace(int64_t batch, int64_t k, int64_t vocab) {
  (void)vocab;
  if (batch <= 0 || k < 0) return 0;
  return workspace_bytes(batch * (2 * k + 1));
}

int ls_greedy_verify(const void* target_logits, int64_t target_batch_stride, int64_t target_pos_stride,
                     const void* draft_logits, int64_t draft_batch_stride, int64_t draft_pos_stride,
                     const int64_t* draft_tokens, int dtype, int64_t batch, int64_t k, int64_t vocab,
                     int32_t* accept_len, int64_t* tokens, int64_t* row_argmax, void* workspace,
                     uint64_t ws_bytes, ls_stream_t stream) {
  const int eb = dtype_bytes(dtype);
  if (eb == 0) return fail(LS_ERR_VALUE, "unsupported logits dtype");
  if (batch < 0 || batch > kMaxGroups || k < 1 || k > 64 || vocab <= 0 || vocab > 0x7fffffffLL)
    return fail(LS_ERR_VALUE, "greedy_verify: need 0 <= batch <= 16384, 1 <= k <= 64, 0 < vocab < 2^31");
  if (batch == 0) return LS_OK;
  if (target_logits == nullptr || accept_len == nullptr || tokens == nullptr)
    return fail(LS_ERR_VALUE, "greedy_verify: NULL pointer");
  if (draft_logits == nullptr && draft_tokens == nullptr)
    return fail(LS_ERR_VALUE, "greedy_verify: need draft logits or draft tokens");
  const int rpg = static_cast<int>(draft_logits ? 2 * k + 1 : k + 1);
  const int64_t total = batch * rpg;
  if (workspace == nullptr || ws_bytes < workspace_bytes(total))
    return fail(LS_ERR_VALUE, "greedy_verify: workspace too small");
  GreedyParams p{};
  p.target = static_cast<const char*>(target_logits);
  p.t_bstride = target_batch_stride * eb;
  p.t_pstride = target_pos_stride * eb;
  p.draft = static_cast<const char*>(draft_logits);
  p.d_bstride = draft_batch_stride * eb;
  p.d_pstride = draft_pos_stride * eb;
  p.draft_tokens = draft_tokens;
  p.vocab = vocab;
  p.k = static_cast<int>(k);
  p.rows_per_group = rpg;
  bool vec = aligned16(target_logits) && (p.t_bstride % 16 == 0) && (p.t_pstride % 16 == 0) &&
             ((vocab * eb) % 16 == 0);
  if (draft_logits)
    vec = vec && aligned16(draft_logits) && (p.d_bstride % 16 == 0) && (p.d_pstride % 16 == 0);
  Shape shape = choose_shape(total, vocab, eb, rpg);
  if (!vec) shape.j = 0;
  p.splits = shape.splits;
  p.direct = 0;
  p.nvec = vocab * eb / 16;
  p.seg = (p.nvec + p.splits - 1) / p.splits;
  p.accept_len = accept_len;
  p.tokens = tokens;
  p.row_argmax = row_argmax;
  bind_workspace(p, workspace);
  return launch(p, dtype, shape, batch, vec, static_cast<hipStream_t>(stream));
}

uint64_t ls_stream_read_probe_words(int64_t batch, int64_t k) {
  if (batch <= 0 || k < 1) return 0;
  return static_cast<uint64_t>(batch * (2 * k + 1)) * kMaxSplits * 4u;
}

int ls_stream_read_probe(const void* target_logits, int64_t target_batch_stride, int64_t target_pos_stride,
                         const void* draft_logits, int64_t draft_batch_stride, int64_t draft_pos_stride, int dtype,
                         int64_t batch, int64_t k, int64_t vocab, uint32_t* out, uint64_t out_words,
                         ls_stream_t stream) {
  const int eb = dtype_bytes(dtype);
  if (eb == 0) return fail(LS_ERR_VALUE, "unsupported logits dtype");
  if (batch <= 0 || batch > kMaxGroups || k < 1 || k > 64 || vocab <= 0 || vocab > 0x7fffffffLL)
    return fail(LS_ERR_VALUE, "stream_read_probe: need 0 < batch <= 16384, 1 <= k <= 64, 0 < vocab < 2^31");
  if (!target_logits || !draft_logits || !out) return fail(LS_ERR_VALUE, "stream_read_probe: NULL pointer");
  if (out_words < ls_stream_read_probe_words(batch, k))
    return fail(LS_ERR_VALUE, "stream_read_probe: output too small");
  GreedyParams p{};
  p.target = static_cast<const char*>(target_logits);
  p.t_bstride = target_batch_stride * eb;
  p.t_pstride = target_pos_stride * eb;
  p.draft = static_cast<const char*>(draft_logits);
  p.d_bstride = draft_batch_stride * eb;
  p.d_pstride = draft_pos_stride * eb;
  p.k = static_cast<int>(k);
  p.rows_per_group = static_cast<int>(2 * k + 1);
  const bool vec = aligned16(target_logits) && aligned16(draft_logits) && (p.t_bstride % 16 == 0) &&
                   (p.t_pstride % 16 == 0) && (p.d_bstride % 16 == 0) && (p.d_pstride % 16 == 0) &&
                   ((vocab * eb) % 16 == 0);
  const Shape shape = choose_shape(batch * p.rows_per_group, vocab, eb, p.rows_per_group);
  if (!vec || shape.block != 256 || shape.j == 0)
    return fail(LS_ERR_VALUE, "stream_read_probe: needs the greedy kernel's exact vector shape (aligned rows, "
                              "segments of 256..2048 vectors)");
  p.splits = shape.splits;
  p.nvec = vocab * eb / 16;
  p.seg = p.nvec / p.splits;
  const dim3 grid(static_cast<unsigned>(p.splits), static_cast<unsigned>(p.rows_per_group),
                  static_cast<unsigned>(batch));
  const hipStream_t st = static_cast<hipStream_t>(stream);
  switch (shape.j) {
    case 1: hipLaunchKernelGGL((read_probe_kernel<256, 1>), grid, dim3(256), 0, st, p, out); break;
    case 2: hipLaunchKernelGGL((read_probe_kernel<256, 2>), grid, dim3(256), 0, st, p, out); break;
    case 3: hipLaunchKernelGGL((read_probe_kernel<256, 3>), grid, dim3(256), 0, st, p, out); break;
    case 4: hipLaunchKernelGGL((read_probe_kernel<256, 4>), grid, dim3(256), 0, st, p, out); break;
    case 5: hipLaunchKernelGGL((read_probe_kernel<256, 5>), grid, dim3(256), 0, st, p, out); break;
    case 6: hipLaunchKernelGGL((read_probe_kernel<256, 6>), grid, dim3(256), 0, st, p, out); break;
    case 7: hipLaunchKernelGGL((read_probe_kernel<256, 7>), grid, dim3(256), 0, st, p, out); break;
    default: hipLaunchKernelGGL((read_probe_kernel<256, 8>), grid, dim3(256), 0, st, p, out); break;
  }
  return check_launch("stream read probe launch");
}

uint64_t ls_greedy_status_offset(void) { return kStatusOffset; }

int ls_greedy_workspace_status(void* workspace, uint64_t ws_bytes, uint32_t* status, ls_stream_t stream) {
  if (workspace == nullptr || status == nullptr) return fail(LS_ERR_VALUE, "greedy_status: NULL pointer");
  if (ws_bytes < kSlotsOffset) return fail(LS_ERR_VALUE, "greedy_status: not a greedy workspace");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  uint32_t* word = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + kStatusOffset);
  hipError_t err = hipStreamSynchronize(st);
  if (err != hipSuccess) return hip_fail(err, "greedy_status: stream");
  err = hipMemcpy(status, word, sizeof(uint32_t), hipMemcpyDeviceToHost);
  if (err != hipSuccess) return hip_fail(err, "greedy_status: copy");
  if (*status != 0) {
    // a timed-out key may have landed in its slot after the slot was cleared
    // (the stream is drained now, so every such store is done): clear the
    // status line and every key slot so the next launch reads only new keys
    err = hipMemset(word, 0, ws_bytes - kStatusOffset);
    if (err != hipSuccess) return hip_fail(err, "greedy_status: clear");
  }
  return LS_OK;
}

}  // extern "C"
