// Device-side building blocks: Philox4x32-10, open-addressing probes, wave64 /
// block scans.  gfx950 only (64-wide wavefronts).
#pragma once

#include "common.hpp"
#include "lookback.hpp"

namespace lmi {

// ------------------------------------------------------------------ Philox
// Philox4x32-10 (Salmon et al. 2011); constants as published.
struct Philox4 {
  uint32_t x, y, z, w;
};

__device__ __forceinline__ Philox4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                 uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    // one 32 x 32 -> 64 product each (v_mad_u64_u32) instead of a high and a low one
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    c0 = hi1 ^ c1 ^ k0;
    c1 = lo1;
    c2 = hi0 ^ c3 ^ k1;
    c3 = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return Philox4{c0, c1, c2, c3};
}

// The sampler's draw: key = 64-bit batch seed, counter = (node, hop, slot, 0).
__device__ __forceinline__ uint32_t sample_draw(uint64_t seed, uint32_t hop, uint32_t node,
                                                uint32_t slot) {
  return philox4x32_10(node, hop, slot, 0u, (uint32_t)seed, (uint32_t)(seed >> 32)).x;
}

// What lane R of each lane group of G lanes holds, in every lane of the group, R a constant (G <= 16) or the same in the
// whole wavefront: moves between registers, where a shuffle goes through the LDS unit and its latency.
template <int G, int R>
__device__ __forceinline__ uint32_t group_lane(uint32_t v) {
  static_assert(G == 4 || G == 8 || G == 16, "lane groups inside a row of 16 lanes");
  if constexpr (G == 4) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, R * 0x55, 0xf, 0xf, true);  // quad_perm R,R,R,R
  } else {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + R, 0xf, 0xf, true);  // row_newbcast
    if constexpr (G == 16) return lo;
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + ((R + 8) & 15), 0xf, 0xf, true);
    return (threadIdx.x & 8) ? hi : lo;
  }
}
template <int G>
__device__ __forceinline__ uint32_t group_lane(uint32_t v, int r) {
  static_assert(G == 32 || G == 64, "lane groups of several rows");
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)v, r);
  if constexpr (G == 64) return lo;
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)v, r + 32);
  return (threadIdx.x & 32) ? hi : lo;
}

// Floyd's rule within a lane group: lane s drew t out of [0, j], j = deg - fanout + s; its pick is t unless an earlier
// lane picked that already, and j then.  All lanes of the group call; lanes from `fanout` on hold t = 0xFFFFFFFF.
// One step per lane, each waiting for the one before: through shuffles a step took the LDS unit's latency (24 of them
// for a fanout of 25).
template <int G, int R>
__device__ __forceinline__ void floyd_step(uint32_t t, uint32_t j, int lane, int fanout, bool &dup) {
  if constexpr (R + 1 < G) {
    if (R + 1 < fanout) {
      const uint32_t p = group_lane<G, R>(dup ? j : t);
      dup = dup || (lane > R && t == p);
      floyd_step<G, R + 1>(t, j, lane, fanout, dup);
    }
  }
}
template <int G>
__device__ __forceinline__ uint32_t floyd_pick(uint32_t t, uint32_t j, int lane, int fanout) {
  bool dup = false;
  if constexpr (G <= 16) {
    floyd_step<G, 0>(t, j, lane, fanout, dup);
  } else {
    for (int r = 0; r + 1 < fanout; ++r) {
      const uint32_t p = group_lane<G>(dup ? j : t, r);
      dup = dup || (lane > r && t == p);
    }
  }
  return dup ? j : t;
}

// ------------------------------------------------------------------ faults
// A condition the host must hear about: recorded in the batch state (read back by
// lmi_batch_counters) and in the server's sticky fault word, which lives in pinned host
// memory and is never cleared by a later batch, so the host sees it without reading the
// device (lmi_server_status).
struct FaultTo {    // where a condition of this batch is recorded
  int32_t serial;   // number of the batch
  int32_t *sticky;  // the server's words, or null
};
__device__ __forceinline__ void raise_fault(DevState *st, int which, FaultTo to) {
  if (which == kFaultBadId) st->bad_id = to.serial; else st->scan_fault = to.serial;
  if (to.sticky) __hip_atomic_store(&to.sticky[which], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ FaultTo fault_to(const DevState *st) { return FaultTo{st->serial, st->fault}; }

__device__ __forceinline__ void note_seen(SeenWord *word, int count, int seeds) {
  *word = (SeenWord)(uint32_t)seeds << 32 | (uint32_t)count;
}

// -------------------------------------------------------------- hash table
__device__ __forceinline__ uint32_t hash_id(int32_t key, int log2cap) {
  return ((uint32_t)key * 0x9E3779B1u) >> (32 - log2cap);
}

// A stored key is `key | tag`: the tag (an epoch number in the bits above the widest id)
// says which batch wrote the slot.  A slot whose tag bits differ from the current tag is
// free -- never written (key -1: every tag bit set) or left by an earlier batch -- so the
// table needs no clearing between batches until the epochs run out.  Untagged tables use
// tag 0 with the sign bit as mask: only the empty key -1 is free.
// Insert `key` (if absent) and lower its value to min(value, cand); returns the
// slot index.  One 8-byte load reads key and value together; a free slot is claimed
// with one 8-byte compare-and-swap that writes key and value at once.  Within a batch
// a slot only ever goes free -> key, so a stale non-free read is still correct and a
// stale free read is resolved by the CAS.  Values only ever decrease, so a stale value
// is never too low: when the value read is already <= cand the atomic can be skipped,
// which removes almost all same-address atomics on frequently sampled hub nodes.
// The slot index comes back with kKnownRepeat set when the insert already saw a lower
// value: such a candidate is certainly not the key's first occurrence, and whoever asks
// later need not read the slot to learn that.  (Without the bit it may or may not be.)
constexpr uint32_t kKnownRepeat = 0x80000000u;
__device__ __forceinline__ uint32_t table_insert_min(HashSlot *slots, int log2cap, int32_t key, int32_t cand,
                                                     int32_t tag = 0, int32_t tag_mask = kUntaggedMask) {
  const uint32_t mask = (1u << log2cap) - 1u;
  const int32_t stored = key | tag;
  uint32_t h = hash_id(key, log2cap);
  const unsigned long long mine = (unsigned long long)(uint32_t)stored | ((unsigned long long)(uint32_t)cand << 32);
  while (true) {
    unsigned long long *word = reinterpret_cast<unsigned long long *>(&slots[h]);
    unsigned long long raw = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (((int32_t)(uint32_t)raw & tag_mask) != tag) {  // free: claim it with key and value together
      const unsigned long long was = atomicCAS(word, raw, mine);
      if (was == raw) return h;
      raw = was;  // somebody else took it: this is what it holds now
    }
    if ((int32_t)(uint32_t)raw == stored) {
      if ((int32_t)(uint32_t)(raw >> 32) > cand) {
        atomicMin(&slots[h].val, cand);
        return h;
      }
      return h | kKnownRepeat;  // a lower candidate is already there: this one cannot be the minimum
    }
    h = (h + 1) & mask;
  }
}

// Read-only probe: value or -1.  FRESH: other tiles of the same launch insert too, possibly on another die, whose L2 this
// one does not see.
template <bool FRESH = false>
__device__ __forceinline__ int32_t table_find(const HashSlot *slots, int log2cap, int32_t key, int32_t tag = 0,
                                              int32_t tag_mask = kUntaggedMask) {
  const uint32_t mask = (1u << log2cap) - 1u;
  const int32_t stored = key | tag;
  uint32_t h = hash_id(key, log2cap);
  while (true) {
    int2 kv;
    if constexpr (FRESH) {
      const unsigned long long raw = __hip_atomic_load(reinterpret_cast<const unsigned long long *>(&slots[h]),
                                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      kv = make_int2((int32_t)(uint32_t)raw, (int32_t)(uint32_t)(raw >> 32));
    } else {
      kv = *reinterpret_cast<const int2 *>(&slots[h]);
    }
    if (kv.x == stored) return kv.y;
    if ((kv.x & tag_mask) != tag) return -1;
    h = (h + 1) & mask;
  }
}

// Bitmap + rank table: the slot of a cached node is the number of cached nodes
// with a smaller id = rank at the start of its 64-id word + set bits below it.
__device__ __forceinline__ int32_t rank_find(const uint4 *tab, int32_t id) {
  const uint4 e = tab[id >> 6];
  const uint64_t bits = (uint64_t)e.x | ((uint64_t)e.y << 32);
  const int b = id & 63;
  if (!((bits >> b) & 1ull)) return -1;
  return (int32_t)e.z + __popcll(bits & ((1ull << b) - 1ull));
}

// The id -> slot table of the static / int8 caches.
struct SlotTable {
  int kind;  // LMI_TABLE_*, or -1: no cache
  const HashSlot *slots;
  int log2cap;
  const int32_t *slot_of;
  const uint4 *rank_tab;
};
__device__ __forceinline__ int32_t static_find(const SlotTable &t, int32_t id) {
  if (t.kind < 0) return -1;
  if (t.kind == LMI_TABLE_RANK) return rank_find(t.rank_tab, id);
  if (t.kind == LMI_TABLE_DIRECT) return t.slot_of[id];
  return table_find(t.slots, t.log2cap, id);
}

// The dynamic cache.  A set's record is its keys followed by its ticks (one 64-byte line for 8 ways), so the tick of a
// hit is written into the line its key was just read from.
struct LruSets {
  const int32_t *keys;  // first record
  int32_t *use;         // its ticks
  int32_t *head;        // first row of each set's list of misses, -1: none
  int64_t sets;
  int ways;
};
// Slot of `id` or -1; a hit is marked as used at `tick`.
__device__ __forceinline__ int32_t lru_find(const LruSets &t, int32_t id, int32_t tick) {
  const int set = (int)((uint32_t)id % (uint32_t)t.sets);
  const int64_t rec = (int64_t)set * 2 * t.ways;
  int way = -1;
  if ((t.ways & 3) == 0) {  // a set's keys start on a 16-byte boundary: four ways per load
    for (int w = 0; w < t.ways; w += 4) {
      const int4 k = *reinterpret_cast<const int4 *>(t.keys + rec + w);
      if (k.x == id) way = w;
      if (k.y == id) way = w + 1;
      if (k.z == id) way = w + 2;
      if (k.w == id) way = w + 3;
    }
  } else {
    for (int w = 0; w < t.ways; ++w)
      if (t.keys[rec + w] == id) way = w;
  }
  if (way < 0) return -1;
  t.use[rec + way] = tick;
  return set * t.ways + way;  // sets * ways < 2^31
}
// Puts a miss on its set's list.
__device__ __forceinline__ void lru_chain(const LruSets &t, int32_t *next, int row, int32_t id) {
  next[row] = atomicExch(&t.head[(uint32_t)id % (uint32_t)t.sets], row);
}

// Last step of a hop: the local id of every edge source is the value its table slot
// holds once the hop's first occurrences have published theirs.  Strided over the
// `n_threads` threads that take part, `tid` being this thread's place among them.
struct FillArgs {
  const DevState *st;
  const HashSlot *slots;
  const int32_t *eslot;  // table slot per edge of hop `hop` (| kKnownRepeat)
  int32_t *agg_src_off;
  int hop = -1;          // -1: nothing to fill
};

__device__ __forceinline__ void fill_local_ids(const FillArgs &f, int64_t tid, int64_t n_threads) {
  if (f.hop < 0) return;
  const int n = f.st->edge_counter[9 + f.hop + 1];
  const int eoff = f.st->edge_counter[12 + f.hop + 1];
  // four edges in flight per thread: the two dependent reads of each overlap those of the others
  for (int64_t e = tid; e < n; e += 4 * n_threads) {
    int32_t slot[4], val[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) slot[u] = (e + u * n_threads < n) ? (f.eslot[e + u * n_threads] & (int32_t)~kKnownRepeat) : 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) val[u] = (e + u * n_threads < n) ? f.slots[slot[u]].val : 0;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (e + u * n_threads < n) f.agg_src_off[eoff + e + u * n_threads] = val[u];
  }
}

// A launch that serves n pipes interleaves them over blockIdx.x (grid_row).
#define LMI_GRID_ROW(n_rows)                                                   \
  const GridRow lmi_gr_ = grid_row(blockIdx.x, (unsigned)(n_rows));            \
  const int row = lmi_gr_.row;                                                 \
  const int bx = lmi_gr_.bx;                                                   \
  const int gx = (int)(gridDim.x / (unsigned)(n_rows));                        \
  (void)gx

// ------------------------------------------------------------------- scans
// Moves between registers (DPP: four shifts within a row of 16 lanes, then the rows' last lanes broadcast) instead of
// shuffles, each of which goes through the LDS unit.  The whole wavefront calls.
__device__ __forceinline__ int wave_inclusive_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15, into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31, into rows 2 and 3
  return v;
}
// Sum over the wavefront, in every lane.
__device__ __forceinline__ int wave_sum(int v) {
  return __builtin_amdgcn_readlane(wave_inclusive_scan(v), kWave - 1);
}

// Exclusive scan over a block of BLOCK threads; `total` = sum over the block.
// lds must hold BLOCK / 64 + 1 ints.  Contains __syncthreads: call uniformly.
template <int BLOCK>
__device__ __forceinline__ int block_exclusive_scan(int v, int *lds, int &total) {
  constexpr int NW = BLOCK / kWave;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int inc = wave_inclusive_scan(v);
  if (lane == kWave - 1) lds[wid] = inc;
  __syncthreads();
  if (wid == 0) {
    int w = (lane < NW) ? lds[lane] : 0;
    const int winc = wave_inclusive_scan(w);
    if (lane < NW) lds[lane] = winc - w;
    if (lane == NW - 1) lds[NW] = winc;
  }
  __syncthreads();
  const int res = inc - v + lds[wid];
  total = lds[NW];
  __syncthreads();
  return res;
}

// The same with one barrier: every wavefront adds up the others' sums itself.  lds holds BLOCK / 64 ints that are not
// written again before the block has passed another barrier.
template <int BLOCK>
__device__ __forceinline__ int block_exclusive_scan_once(int v, int *lds, int &total) {
  constexpr int NW = BLOCK / kWave;
  const int lane = threadIdx.x & (kWave - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int inc = wave_inclusive_scan(v);
  if (lane == kWave - 1) lds[wid] = inc;
  __syncthreads();
  const int w = lane < NW ? lds[lane] : 0;
  const int winc = wave_inclusive_scan(w);
  total = __builtin_amdgcn_readlane(winc, kWave - 1);
  return inc - v + __builtin_amdgcn_readlane(winc - w, wid);
}

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & (kWave - 1);
  return (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
}

}  // namespace lmi
