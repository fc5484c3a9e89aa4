// The gather of feature rows by a grid of blocks: as a launch of its own (cache.hip), and for rows known early in blocks of a
// hop's launch (sampler.hip).
#pragma once

#include "device.hpp"

namespace lmi {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));  // a 16-byte access at a 4-byte-aligned address

constexpr int kFlatTileMax = 256;  // rows per tile
// About 8 KB worth of rows for 256 threads, two at least.
inline int flat_tile_rows(int64_t row_bytes) {
  return (int)std::max<int64_t>(2, std::min<int64_t>(64, 8192 / row_bytes));
}

struct RowSources {
  const uint8_t *cache;  // row of a slot, slots [0, n_cache)
  const uint8_t *table;  // MISSES: row of a node id, ids [0, n_table)
  uint32_t n_cache, n_table;
  int64_t pitch;  // bytes of a row, in both
};

// Output rows [first, n) of fp32 / fp16 rows of every size from 16 bytes up, source row = src_index[row] (a cache slot;
// outside [0, n_cache) = nothing to move).  A block takes a
// tile of consecutive rows and its BLOCK threads walk the tile's 16-byte units in flat order -- unit f is
// piece f % upr of row f / upr -- U units per lane and pass: the U slots (lanes of one row read the
// same word: one cache line per wavefront), then the U row pieces, then the U stores, each step
// issued whole before the next waits.  Lanes without a unit, or whose row is a miss, issue nothing
// (every access they would make costs the memory pipeline a cycle whether or not HBM sees it).
// Nothing else stands between a block and its bytes: no LDS, no barrier.  Measured against the same
// loop with computed source rows on one output buffer, this shape keeps 90 % of its rate; staging a
// tile's rows through LDS first kept 70 %.  A row that is no multiple of 16 bytes ends with a unit
// that overlaps the one before it (both write the same bytes), so every access is 16 bytes wide, at
// 4-byte alignment when the row length demands it (V16 says which).
// MISSES: a row without a slot is read from the feature table by its node id in the same pass (gather_in_line says
// when).  The table may lie behind the host link: the wavefronts that hold such rows then wait for the link, which
// bounds the launch, while the hits of all others stream past.
// look: the slots are not known yet: a block looks its tile's rows up first, a thread each (tiles of at most BLOCK and
// kFlatTileMax rows), and hands slots and ids to the others through LDS (s_rows: kSlotLds ints), and slots to look_index
// unless that is null.  One read in a row more per tile instead of a launch and a pass over the ids.
// FRESH (with look): another block of the same launch wrote the ids.
constexpr int kSlotLds = 2 * kFlatTileMax;
template <typename V16, int BLOCK, int U, bool NT, bool MISSES, bool FRESH = false>
__device__ __forceinline__ void gather_rows(const RowSources &from, const int32_t *__restrict__ src_index,
                                            const int32_t *__restrict__ ids, uint8_t *__restrict__ dst, int first, int n,
                                            int upr, int last_off, int rows_per_tile, int64_t dst_pitch, int bx, int gx,
                                            bool look, const SlotTable &slots, int32_t *look_index, int *s_rows) {
  const int dq = BLOCK / upr, dr = BLOCK % upr;  // what BLOCK units further means in (row, piece)
  const int r0 = (int)threadIdx.x / upr, u0 = (int)threadIdx.x % upr;
  for (int tile = bx; tile * rows_per_tile < n - first; tile += gx) {
    const int row0 = first + tile * rows_per_tile;
    const int nr = n - row0 < rows_per_tile ? n - row0 : rows_per_tile;
    const int lim = nr * upr;
    if (look) {
      __syncthreads();  // the tile before is done with its slots
      if ((int)threadIdx.x < nr) {
        const int32_t node = FRESH ? __hip_atomic_load(&ids[row0 + threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                   : ids[row0 + threadIdx.x];
        const int32_t found = (uint32_t)node < from.n_table ? static_find(slots, node) : -1;
        s_rows[threadIdx.x] = found;
        s_rows[kFlatTileMax + threadIdx.x] = node;
        if (look_index) look_index[row0 + threadIdx.x] = found;
      }
      __syncthreads();
    }
    int rr = r0, uu = u0;
    for (int f0 = threadIdx.x; f0 < lim; f0 += BLOCK * U) {
      int slot[U], id[U], off[U];
      int64_t da[U];
      V16 v[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int i = row0 + rr;
        slot[k] = id[k] = -1;
        if (f0 + BLOCK * k < lim) {
          slot[k] = look ? s_rows[rr] : src_index[i];
          // beside the slot, not behind it: a miss waits for one read, not for two
          if (MISSES) id[k] = look ? s_rows[kFlatTileMax + rr] : ids[i];
        }
        off[k] = (uu == upr - 1) ? last_off : 16 * uu;
        da[k] = (int64_t)i * dst_pitch + off[k];
        uu += dr;
        rr += dq;
        if (uu >= upr) {
          uu -= upr;
          ++rr;
        }
      }
      const uint8_t *at[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        at[k] = (uint32_t)slot[k] < from.n_cache ? from.cache + (int64_t)slot[k] * from.pitch + off[k] : nullptr;
        if (MISSES && !at[k] && (uint32_t)id[k] < from.n_table) at[k] = from.table + (int64_t)id[k] * from.pitch + off[k];
      }
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (at[k]) v[k] = __builtin_nontemporal_load(reinterpret_cast<const V16 *>(at[k]));
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (at[k]) {
          V16 *d = reinterpret_cast<V16 *>(dst + da[k]);
          if (NT) __builtin_nontemporal_store(v[k], d);
          else *d = v[k];
        }
    }
  }
}

}  // namespace lmi
