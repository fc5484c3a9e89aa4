// Feature caches: static hot-set, LRU dynamic, int8-compressed; the id->slot
// lookup; and the row gather (HBM rows on hits, zero-copy pinned host rows on
// misses, dequantisation fused for int8 rows).
//
// Reference semantics (Legion-IBP, sampling_server/src):
//   cache/cache_impl.cuh:239-303        gather: row i of the output belongs to ids[i];
//                                       hit -> cache row, miss -> host row of the id
//   cache/cache.cu:314-338              FindFeat: id -> slot for one frontier segment
//   cache/cache.cu:559-656              FillUp: choose rows, copy them, build the map
//   comp_cache/static_cache_kernel.cuh:6-29,185-266   set = id mod n_sets, ways contiguous
// What differs on purpose: hot set = top rows by (out-degree desc, id asc) found
// with a histogram of the keys and two scans (no sort, no presampling); our own
// open-addressing table (or a direct map) instead of the vendored cuckoo table;
// a batch-synchronous LRU (the reference's LRU source is absent); int8 + per-row
// scale instead of the un-vendored lossless codec; one lane moves 16 bytes and
// several rows are in flight per lane instead of one float per thread.
#include <algorithm>
#include <vector>

#include <hip/hip_ext.h>

#include "gather.hpp"
#include "scan.hpp"

namespace lmi {

// ------------------------------------------------------------------ gather
// Generic row mover over work items j in [*first_ptr, *n_ptr).  Entry j of the work
// list is a pair (output row i, source row); without a list i = j.  With SRC_FROM_LIST the source row is the pair's
// second word, so the only dependent load in front of the row itself is the pair;
// otherwise it is src_index[i] (or i).  The destination row is dst_index[i] (or
// i); a negative source or destination skips the row.  LPR lanes cooperate on a
// row, each moving sizeof(V) bytes per step, with U rows in flight per lane.
// HOSTLINK only names the instantiation that reads over the host link, so that
// profiles list the HBM gather and the host-link gather as two kernels.
// One launch can serve several pipes (output buffers): their blocks interleave over
// blockIdx.x like those of the sampling kernels, and the source table is shared.
struct MoveRow {
  const int2 *list;
  const int32_t *first_ptr, *n_ptr, *src_index, *dst_index;
  const int32_t *ids;  // gather_rows_flat_kernel<.., MISSES>: node id per row
  int32_t *look_index; // gather_rows_flat_kernel<.., LOOK>: receives the slot per row
  uint8_t *dst;
  int note_seeds;  // Pipe::note_seeds
  // the HBM gathers of a batch carry its last steps (MoveGroup::tail_blocks)
  FillArgs fill;        // last hop's local ids (hop -1: already there)
  HeaderCopy headers;   // where the batch's headers go besides its state (nodes null: nowhere)
};
struct MoveGroup {
  MoveRow p[LMI_MAX_GROUP];
  int n;
  int tail_blocks;  // blocks [0, tail_blocks) of each pipe finish the batch, the rest gather
};

// The last steps of a batch in blocks of the gather: the fill is bound by random reads of the dedup table that leave
// HBM's streams to the gather (four papers100M-shaped batches from a table in HBM: gather 152 us, with the fill 160).
__device__ __forceinline__ void batch_tail(const MoveRow &r, int bx, int tail_blocks) {
  if (bx == 0 && r.headers.nodes && threadIdx.x < 32) {
    const int t = threadIdx.x & 15;
    const DevState *st = r.fill.st;
    if (threadIdx.x < 16) r.headers.nodes[t] = st->node_counter[t];
    else r.headers.edges[t] = st->edge_counter[t];
  }
  fill_local_ids(r.fill, (int64_t)bx * blockDim.x + threadIdx.x, (int64_t)tail_blocks * blockDim.x);
}

// LMI_GRID_ROW for a kernel that carries batch_tail: those blocks leave, bx and gx count the others.
#define LMI_GRID_ROW_TAIL(g)                                                          \
  const GridRow lmi_gr_ = grid_row(blockIdx.x, (unsigned)(g).n);                      \
  const int row = lmi_gr_.row;                                                        \
  if (lmi_gr_.bx < (g).tail_blocks) {                                                 \
    batch_tail((g).p[row], lmi_gr_.bx, (g).tail_blocks);                              \
    return;                                                                           \
  }                                                                                   \
  const int bx = lmi_gr_.bx - (g).tail_blocks;                                        \
  const int gx = (int)(gridDim.x / (unsigned)(g).n) - (g).tail_blocks

template <typename V, int LPR, int U, bool NT, bool HOSTLINK>
static __global__ __launch_bounds__(256) void move_rows_kernel(
    MoveGroup g, int src_from_list, const uint8_t *src, int chunks, int64_t src_row_bytes, int64_t dst_row_bytes,
    unsigned long long *row_counter) {
  LMI_GRID_ROW(g.n);
  const MoveRow &r = g.p[row];
  const int2 *list = r.list;
  const int32_t *src_index = r.src_index, *dst_index = r.dst_index;
  uint8_t *dst = r.dst;
  const int n = *r.n_ptr;
  const int first = r.first_ptr ? *r.first_ptr : 0;
  if (row_counter && bx == 0 && threadIdx.x == 0 && n > first)
    atomicAdd(row_counter, (unsigned long long)(n - first));  // work items offered to this launch (profiling)
  const int lane = threadIdx.x & (LPR - 1);
  const int group = (bx * blockDim.x + threadIdx.x) / LPR;
  const int n_groups = gx * blockDim.x / LPR;
  for (int j0 = first + group; j0 < n; j0 += n_groups * U) {
    int64_t so[U], dofs[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * n_groups;
      so[u] = -1;
      dofs[u] = -1;
      if (j < n) {
        int i = j, si;
        if (list) {
          const int2 pr = list[j];
          i = pr.x;
          si = pr.y;
        }
        if (!list || !src_from_list) si = src_index ? src_index[i] : i;
        const int di = dst_index ? dst_index[i] : i;
        if (si >= 0 && di >= 0) {
          so[u] = (int64_t)si * src_row_bytes;
          dofs[u] = (int64_t)di * dst_row_bytes;
        }
      }
    }
    for (int c = lane; c < chunks; c += LPR) {
      V v[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (so[u] >= 0) v[u] = __builtin_nontemporal_load(reinterpret_cast<const V *>(src + so[u] + (int64_t)c * sizeof(V)));
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (so[u] >= 0) {
          V *d = reinterpret_cast<V *>(dst + dofs[u] + (int64_t)c * sizeof(V));
          if (NT) __builtin_nontemporal_store(v[u], d);
          else *d = v[u];
        }
    }
  }
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Row mover for rows that a power-of-two lane group does not fit: 400-byte rows (25 chunks of
// 16 bytes would leave 7 of 32 lanes idle), rows that are no multiple of 16 bytes, rows whose
// start is only 4-byte aligned.  A row is `cpr` 16-byte units followed by `tail` 4-byte units.
// A block takes a tile of TILE consecutive work items in two steps.  Staging: one thread per
// work item resolves it (list entry, source row, destination row: the only dependent loads)
// and the items that have something to move -- cache hits, when the source index is the
// cache slot -- are compacted into LDS by ballot + prefix popcount, as (source offset,
// destination offset) pairs.  Moving: the 256 threads walk the units of the staged rows in
// flat order, unit f = staged row f / units, place f % units inside it, offsets from LDS, so
// every lane of every pass but the last has a unit, misses cost no lanes, and the row loads
// of a pass depend on nothing but LDS.  Consecutive lanes touch consecutive bytes of a row,
// and of the next row when the destination rows are contiguous.  V16 says whether the 16-byte
// accesses may assume 16-byte alignment.  Work items, lists and index arrays mean what they
// mean in move_rows_kernel.
constexpr int kTileWaves = 4;  // wavefronts of a 256-thread block
template <typename V16, int TILE, int U, bool NT, bool HOSTLINK>
static __global__ __launch_bounds__(256) void move_rows_tiled_kernel(
    MoveGroup g, int src_from_list, const uint8_t *src, int cpr, int tail, int tile_rows, int64_t src_row_bytes,
    int64_t dst_row_bytes, unsigned long long *row_counter) {
  static_assert(TILE == 64 || TILE == 256, "a tile is at most one work item per lane of one wavefront, or of the block");
  __shared__ int64_t s_src[TILE], s_dst[TILE];
  __shared__ int s_cnt[kTileWaves];
  LMI_GRID_ROW(g.n);
  const MoveRow &r = g.p[row];
  const int2 *list = r.list;
  const int32_t *src_index = r.src_index, *dst_index = r.dst_index;
  uint8_t *dst = r.dst;
  const int n = *r.n_ptr;
  const int first = r.first_ptr ? *r.first_ptr : 0;
  if (row_counter && bx == 0 && threadIdx.x == 0 && n > first)
    atomicAdd(row_counter, (unsigned long long)(n - first));  // work items offered to this launch (profiling)
  const int units = cpr + tail;
  const int dq = 256 / units, dr = 256 % units;  // what 256 units further means in (row, place)
  const int r0 = (int)threadIdx.x / units, u0 = (int)threadIdx.x % units;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int n_tiles = (n - first + tile_rows - 1) / tile_rows;  // tile_rows <= TILE
  for (int tile = bx; tile < n_tiles; tile += gx) {
    // ---- staging
    bool ok = false;
    int64_t so = 0, dof = 0;
    if ((int)threadIdx.x < tile_rows) {
      const int j = first + tile * tile_rows + (int)threadIdx.x;
      if (j < n) {
        int i = j, si;
        if (list) {
          const int2 pr = list[j];
          i = pr.x;
          si = pr.y;
        }
        if (!list || !src_from_list) si = src_index ? src_index[i] : i;
        const int di = dst_index ? dst_index[i] : i;
        ok = si >= 0 && di >= 0;
        so = (int64_t)si * src_row_bytes;
        dof = (int64_t)di * dst_row_bytes;
      }
    }
    int n_rows;
    if (TILE == 64) {
      if (wid == 0) {
        const uint64_t m = __ballot(ok);
        if (ok) {
          const int pos = __popcll(m & lanemask_lt());
          s_src[pos] = so;
          s_dst[pos] = dof;
        }
        if (lane == 0) s_cnt[0] = __popcll(m);
      }
      __syncthreads();
      n_rows = s_cnt[0];
    } else {
      const uint64_t m = __ballot(ok);
      if (lane == 0) s_cnt[wid] = __popcll(m);
      __syncthreads();
      int base = 0, total = 0;
#pragma unroll
      for (int w = 0; w < kTileWaves; ++w) {
        const int c = s_cnt[w];
        if (w < wid) base += c;
        total += c;
      }
      if (ok) {
        const int pos = base + __popcll(m & lanemask_lt());
        s_src[pos] = so;
        s_dst[pos] = dof;
      }
      __syncthreads();
      n_rows = total;
    }
    // ---- moving
    const int lim = n_rows * units;
    int rr = r0, uu = u0;
    for (int f0 = threadIdx.x; f0 < lim; f0 += 256 * U) {
      int64_t sa[U], da[U];
      int kind[U];  // 0: nothing, 1: 16 bytes, 2: 4 bytes
#pragma unroll
      for (int q = 0; q < U; ++q) {
        kind[q] = 0;
        if (f0 + q * 256 < lim) {
          const int off = uu < cpr ? 16 * uu : 16 * cpr + 4 * (uu - cpr);
          sa[q] = s_src[rr] + off;
          da[q] = s_dst[rr] + off;
          kind[q] = uu < cpr ? 1 : 2;
        }
        uu += dr;
        rr += dq;
        if (uu >= units) {
          uu -= units;
          ++rr;
        }
      }
      V16 v[U];
      uint32_t w[U];
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (kind[q] == 1) v[q] = __builtin_nontemporal_load(reinterpret_cast<const V16 *>(src + sa[q]));
        else if (kind[q] == 2) w[q] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(src + sa[q]));
      }
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (kind[q] == 1) {
          V16 *d = reinterpret_cast<V16 *>(dst + da[q]);
          if (NT) __builtin_nontemporal_store(v[q], d);
          else *d = v[q];
        } else if (kind[q] == 2) {
          uint32_t *d = reinterpret_cast<uint32_t *>(dst + da[q]);
          if (NT) __builtin_nontemporal_store(w[q], d);
          else *d = w[q];
        }
      }
    }
    __syncthreads();  // the next tile's staging overwrites the offsets
  }
}

// The HBM gather as a launch of its own (gather_rows).  LOOK: the slots are not known yet (`look` there).
// rows_seen (pinned host memory, or null): the launch leaves each pipe's row count there for the host
// to size later grids by (see launch_gather_flat).
template <typename V16, int U, bool NT, bool MISSES, bool LOOK>
static __global__ __launch_bounds__(256) void gather_rows_flat_kernel(MoveGroup g, RowSources from, int upr, int last_off,
                                                                      int rows_per_tile, int64_t dst_pitch,
                                                                      unsigned long long *row_counter,
                                                                      SeenWord *rows_seen, SlotTable look) {
  __shared__ int s_slot[LOOK ? kSlotLds : 1];
  LMI_GRID_ROW_TAIL(g);
  const MoveRow &r = g.p[row];
  const int n = *r.n_ptr;
  const int first = r.first_ptr ? *r.first_ptr : 0;
  if (bx == 0 && threadIdx.x == 0) {
    if (row_counter && n > first) atomicAdd(row_counter, (unsigned long long)(n - first));  // profiling
    if (rows_seen && r.note_seeds > 0) note_seen(&rows_seen[row], n - first, r.note_seeds);
  }
  gather_rows<V16, 256, U, NT, MISSES>(from, r.src_index, r.ids, r.dst, first, n, upr, last_off, rows_per_tile, dst_pitch, bx, gx,
                                       LOOK, look, r.look_index, s_slot);
}

// Grid of a gather whose real row count only the device knows.  The worst case of a batch is about
// ten times what a batch holds, and a block that finds no tile is not free: the device starts about one
// workgroup per clock, so the 8 000 idle blocks of a worst-case grid cost a 40 us launch a seventh of
// its time.  The gather kernels leave the row count of every launch in pinned host memory
// (rows_seen); the largest of the last launch in proportion to the seeds, with an eighth on top, sizes the next grid.  The
// kernels stride over their tiles by the grid, so a grid that turns out small is slower, not wrong.
// Whole batches use the first LMI_MAX_GROUP words; a gather of one segment (operator by operator) has a word of its own,
// or the seeds' 800 rows would size the grid of the last hop's 44 000 (284 instead of 190 us for the operators of a batch).
int64_t hinted_rows(const Server *s, int64_t n_max, int word, Pipe *const *pp, int n) {
  if (!s->rows_seen_host || !s->gather_adaptive) return n_max;
  const int seeds = most_seeds(pp, n);
  int64_t seen = 0;
  const int words = word == 0 ? LMI_MAX_GROUP : 1;
  for (int k = 0; k < words; ++k) seen = std::max(seen, seen_count(&s->rows_seen_host[word + k], seeds));
  if (seen <= 0) return n_max;  // nothing seen yet
  return std::min<int64_t>(n_max, seen + seen / 8 + 64);
}

static int rows_word(const Server *s, int seg, int seg_last) {
  return seg_last == s->cfg.hops && (seg == 0 || seg != seg_last) ? 0 : LMI_MAX_GROUP + seg_last;
}

struct MoveArgs {
  MoveGroup g;     // per pipe: work list, bounds, index arrays, destination
  int src_from_list;
  int max_blocks;  // per pipe; 0 = fill the device
  int unroll;      // 0 = the server's gather_unroll
  int host_link;   // the source is pinned host memory read over the host link
  unsigned long long *row_counter;  // device counter that receives the number of work items, or null
  hipEvent_t ev_start, ev_stop;     // stamped with the kernel's begin and end when not null (profiling)
  const uint8_t *src;
  int64_t n_src;                    // rows of src (flat gather: indexes at or beyond it move nothing)
  const uint8_t *table;             // flat gather: the feature table rows without a slot are read from, or null
  int64_t n_table;                  // node ids below this have a row there
  int look;                         // flat gather with a table: look the slots up on the way
  int note_rows;                    // flat gather: the word of rows_seen that receives the row counts, or -1
  int64_t rows_hint;                // note_rows >= 0: how many rows are expected (hinted_rows)
  int64_t src_row_bytes, dst_row_bytes, row_bytes;  // row_bytes = bytes moved per row
  int64_t n_max;   // per pipe
};

template <typename V, int LPR, int U>
static void launch_move_vlu(hipStream_t st, const MoveArgs &a, int grid, bool nt) {
  const int chunks = (int)(a.row_bytes / sizeof(V));
  // with profiling on, the launch carries its own start / stop events
#define LMI_MOVE(NT_, HL_)                                                                                      \
  if (a.ev_start || a.ev_stop)                                                                                  \
    hipExtLaunchKernelGGL((move_rows_kernel<V, LPR, U, NT_, HL_>), dim3(grid * a.g.n), dim3(256), 0, st,         \
                          a.ev_start, a.ev_stop, 0, a.g, a.src_from_list, a.src, chunks, a.src_row_bytes,        \
                          a.dst_row_bytes, a.row_counter);                                                       \
  else                                                                                                          \
    hipLaunchKernelGGL((move_rows_kernel<V, LPR, U, NT_, HL_>), dim3(grid * a.g.n), dim3(256), 0, st, a.g,       \
                       a.src_from_list, a.src, chunks, a.src_row_bytes, a.dst_row_bytes, a.row_counter)
  if (a.host_link) {
    LMI_MOVE(true, true);
  } else if (nt) {
    LMI_MOVE(true, false);
  } else {
    LMI_MOVE(false, false);
  }
#undef LMI_MOVE
}

template <typename V, int LPR>
static void launch_move_vl(hipStream_t st, const MoveArgs &a, int grid, bool nt, int unroll) {
  switch (unroll) {
    case 1: launch_move_vlu<V, LPR, 1>(st, a, grid, nt); break;
    case 2: launch_move_vlu<V, LPR, 2>(st, a, grid, nt); break;
    case 8: launch_move_vlu<V, LPR, 8>(st, a, grid, nt); break;
    default: launch_move_vlu<V, LPR, 4>(st, a, grid, nt); break;
  }
}

template <typename V>
static void launch_move_v(hipStream_t st, const MoveArgs &a, int grid, bool nt, int unroll, int lpr) {
  switch (lpr) {
    case 1: launch_move_vl<V, 1>(st, a, grid, nt, unroll); break;  // thread per row (measurement only)
    case 4: launch_move_vl<V, 4>(st, a, grid, nt, unroll); break;
    case 8: launch_move_vl<V, 8>(st, a, grid, nt, unroll); break;
    case 16: launch_move_vl<V, 16>(st, a, grid, nt, unroll); break;
    case 32: launch_move_vl<V, 32>(st, a, grid, nt, unroll); break;
    default: launch_move_vl<V, 64>(st, a, grid, nt, unroll); break;
  }
}

// Grid of an HBM gather whose worst case needs `want` blocks: a sixteenth of that, between 8
// and 64 blocks per CU.
static int64_t auto_gather_blocks(const Server *s, int64_t want) {
  return std::min<int64_t>(std::max<int64_t>(want / 16, (int64_t)s->n_cu * 8), (int64_t)s->n_cu * 64);
}

template <typename V16, int TILE, int U>
static void launch_tiled_vtu(hipStream_t st, const MoveArgs &a, int grid, bool nt, int cpr, int tail, int tile_rows) {
#define LMI_TILED(NT_, HL_)                                                                                         \
  if (a.ev_start || a.ev_stop)                                                                                      \
    hipExtLaunchKernelGGL((move_rows_tiled_kernel<V16, TILE, U, NT_, HL_>), dim3(grid * a.g.n), dim3(256), 0, st,    \
                          a.ev_start, a.ev_stop, 0, a.g, a.src_from_list, a.src, cpr, tail, tile_rows,              \
                          a.src_row_bytes, a.dst_row_bytes, a.row_counter);                                          \
  else                                                                                                              \
    hipLaunchKernelGGL((move_rows_tiled_kernel<V16, TILE, U, NT_, HL_>), dim3(grid * a.g.n), dim3(256), 0, st, a.g,  \
                       a.src_from_list, a.src, cpr, tail, tile_rows, a.src_row_bytes, a.dst_row_bytes, a.row_counter)
  if (a.host_link) {
    LMI_TILED(true, true);
  } else if (nt) {
    LMI_TILED(true, false);
  } else {
    LMI_TILED(false, false);
  }
#undef LMI_TILED
}

template <typename V16, int TILE>
static void launch_tiled_vt(hipStream_t st, const MoveArgs &a, int grid, bool nt, int cpr, int tail, int tile_rows,
                            int unroll) {
  if (unroll >= 4) launch_tiled_vtu<V16, TILE, 4>(st, a, grid, nt, cpr, tail, tile_rows);
  else if (unroll >= 2) launch_tiled_vtu<V16, TILE, 2>(st, a, grid, nt, cpr, tail, tile_rows);
  else launch_tiled_vtu<V16, TILE, 1>(st, a, grid, nt, cpr, tail, tile_rows);
}

// Rows of a tile of the tiled movers: about 8 KB of rows, so that a batch of long rows still
// makes thousands of tiles and short tiles even out the blocks that run beside host-link reads;
// between 2 and 64 (a wavefront stages them), or the block's 256 when rows are so short that 64
// of them do not give every thread a unit.  Measured, share of HBM peak: 400-byte rows 16 rows
// 47 %, 32 44 %, 64 42 %; 5 732-byte rows 2 rows 52 %, 4 48 %, 8 49 %, 16 41 %.
static int tiled_tile_rows(Server *s, int64_t row_bytes) {
  if (s->gather_tile_rows > 0) return std::min(s->gather_tile_rows, row_bytes < 128 ? 256 : 64);
  if (row_bytes < 128) return 256;
  int t = 64;
  while (t > 2 && (int64_t)t * row_bytes > 8192) t >>= 1;
  return t;
}

static int launch_gather_flat(Server *s, hipStream_t st, const MoveArgs &a, bool nt, bool aligned16) {
  const int upr = (int)((a.row_bytes + 15) / 16);
  const int last_off = (int)a.row_bytes - 16;
  const int u_want = s->gather_unroll > 0 ? s->gather_unroll : 2;
  const int U = u_want >= 4 ? 4 : u_want >= 2 ? 2 : 1;
  int rpt = flat_tile_rows(a.row_bytes);
  if (s->gather_tile_rows > 0) rpt = std::min(s->gather_tile_rows, kFlatTileMax);
  const int64_t want = ceil_div(a.note_rows >= 0 ? a.rows_hint : a.n_max, rpt);
  const int64_t cap = a.max_blocks > 0 ? a.max_blocks : s->gather_blocks > 0 ? s->gather_blocks : (int64_t)s->n_cu * 64;
  const int grid = (int)std::max<int64_t>(1, std::min(want, cap)) + a.g.tail_blocks;
  const SlotTable look = slot_table(s);
  const RowSources from{a.src, a.table, (uint32_t)a.n_src, (uint32_t)a.n_table, a.src_row_bytes};
#define LMI_FLAT(V_, U_, NT_, M_, L_)                                                                                      \
  if (a.ev_start || a.ev_stop)                                                                                         \
    hipExtLaunchKernelGGL((gather_rows_flat_kernel<V_, U_, NT_, M_, L_>), dim3(grid * a.g.n), dim3(256), 0, st,             \
                          a.ev_start, a.ev_stop, 0, a.g, from, upr, last_off, rpt, a.dst_row_bytes, a.row_counter, \
                          a.note_rows >= 0 ? s->rows_seen_dev + a.note_rows : nullptr, look); \
  else                                                                                                                 \
    hipLaunchKernelGGL((gather_rows_flat_kernel<V_, U_, NT_, M_, L_>), dim3(grid * a.g.n), dim3(256), 0, st, a.g, from, upr, \
                       last_off, rpt, a.dst_row_bytes, a.row_counter, a.note_rows >= 0 ? s->rows_seen_dev + a.note_rows : nullptr, look)
#define LMI_FLAT_U(V_, NT_)                        \
  if (a.look) { LMI_FLAT(V_, 2, NT_, true, true); }         \
  else if (a.table) { LMI_FLAT(V_, 2, NT_, true, false); }  \
  else if (U == 4) { LMI_FLAT(V_, 4, NT_, false, false); } \
  else if (U == 2) { LMI_FLAT(V_, 2, NT_, false, false); } \
  else { LMI_FLAT(V_, 1, NT_, false, false); }
  if (aligned16 && nt) { LMI_FLAT_U(u32x4, true) }
  else if (aligned16) { LMI_FLAT_U(u32x4, false) }
  else if (nt) { LMI_FLAT_U(u32x4_a4, true) }
  else { LMI_FLAT_U(u32x4_a4, false) }
#undef LMI_FLAT_U
#undef LMI_FLAT
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

static int launch_move_rows_tiled(Server *s, hipStream_t st, const MoveArgs &a, bool nt, bool aligned16) {
  const int cpr = (int)(a.row_bytes / 16), tail = (int)(a.row_bytes % 16) / 4;
  const int tile = tiled_tile_rows(s, a.row_bytes);
  const int64_t want = ceil_div(a.n_max, tile);
  const int64_t cap = a.max_blocks > 0 ? a.max_blocks : s->gather_blocks > 0 ? s->gather_blocks : auto_gather_blocks(s, want);
  const int grid = (int)std::max<int64_t>(1, std::min(want, cap));
  // two units in flight per lane unless the caller or the knob says otherwise (400-byte rows: 1 -> 42 %
  // of HBM peak, 2 -> 44 %, 4 -> 34 %)
  const int unroll = a.unroll > 0 ? a.unroll : s->gather_unroll > 0 ? s->gather_unroll : 2;
  if (aligned16 && tile <= 64) launch_tiled_vt<u32x4, 64>(st, a, grid, nt, cpr, tail, tile, unroll);
  else if (aligned16) launch_tiled_vt<u32x4, 256>(st, a, grid, nt, cpr, tail, tile, unroll);
  else if (tile <= 64) launch_tiled_vt<u32x4_a4, 64>(st, a, grid, nt, cpr, tail, tile, unroll);
  else launch_tiled_vt<u32x4_a4, 256>(st, a, grid, nt, cpr, tail, tile, unroll);
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// measurement knobs of the lane-group mover
static bool lane_group_knobs(const Server *s, bool host_link) { return s->gather_vec != 0 || (s->gather_lpr != 0 && !host_link); }

// Picks the widest vector that divides the row and all base addresses, and a
// power-of-two lane group that covers one row when possible; rows such a group does not
// fit exactly go to the tiled mover.
static int launch_move_rows(Server *s, hipStream_t st, const MoveArgs &a, bool nt) {
  if (a.n_max <= 0 || a.row_bytes <= 0) return LMI_OK;
  if (a.g.n < 1 || a.g.n > LMI_MAX_GROUP) LMI_FAIL(LMI_ERR_ARG, "a row move serves 1..LMI_MAX_GROUP pipes");
  uintptr_t align = (uintptr_t)a.src | (uintptr_t)a.table | (uintptr_t)a.src_row_bytes | (uintptr_t)a.dst_row_bytes | (uintptr_t)a.row_bytes;
  for (int k = 0; k < a.g.n; ++k) align |= (uintptr_t)a.g.p[k].dst;
  int vec = (align % 16 == 0) ? 16 : (align % 8 == 0) ? 8 : 4;
  if (align % 4 != 0) LMI_FAIL(LMI_ERR_ARG, "feature rows must be 4-byte aligned");
  {
    // a lane group fits exactly when the row is 8, 16, 32 or 64 aligned 16-byte chunks (128 .. 1024 bytes)
    const int64_t c16 = a.row_bytes / 16;
    const bool exact = vec == 16 && (c16 == 8 || c16 == 16 || c16 == 32 || c16 == 64);
    const bool knobs = lane_group_knobs(s, a.host_link != 0);
    // HBM gather (gather_flat): 0 or 3 the flat gather, 1 the LDS-tiled mover, 2 lane groups; host-link
    // gather (miss_flat): the LDS-tiled mover 0 when no lane group fits, 1 always, 2 never
    const int flat = a.host_link ? s->miss_flat : s->gather_flat;
    bool direct = !a.host_link && a.row_bytes >= 16;  // rows walked directly, source row = src_index[row]: the hits
    for (int k = 0; k < a.g.n; ++k) direct = direct && !a.g.p[k].list && a.g.p[k].src_index && !a.g.p[k].dst_index;
    if (direct && !knobs && (flat == 0 || flat == 3)) return launch_gather_flat(s, st, a, nt, vec == 16);
    if (a.row_bytes >= 16 && (flat == 1 || (flat == 0 && !exact && !knobs)))
      return launch_move_rows_tiled(s, st, a, nt, vec == 16);
  }
  if (s->gather_vec == 4 || (s->gather_vec == 8 && vec == 16)) vec = s->gather_vec;  // narrower on request
  const int64_t chunks = a.row_bytes / vec;
  int lpr = a.host_link ? 0 : s->gather_lpr;  // the knob is about the HBM gather
  if (lpr != 1 && lpr != 4 && lpr != 8 && lpr != 16 && lpr != 32 && lpr != 64) {
    lpr = 8;
    while (lpr < chunks && lpr < 64) lpr <<= 1;
  }
  const int unroll = a.unroll > 0 ? a.unroll : s->gather_unroll > 0 ? s->gather_unroll : 1;
  const int64_t groups_per_block = 256 / lpr;
  int64_t want = ceil_div(a.n_max, groups_per_block * (unroll > 0 ? unroll : 1));
  // Many small blocks rather than one resident wave of them: blocks that run beside host-link reads
  // are slowed unevenly, and the dispatcher evens that out (paper100m-shaped, 4 batches per launch:
  // 8 blocks per CU and pipe 62 % of HBM peak, 32 66 %, 64 67 %, 128 66 %, 256 57 %).  A batch holds
  // about a tenth of its worst-case rows, and blocks without rows are not free (products-shaped:
  // 40 % of peak on 2048 blocks per pipe, 36 % on 16384), hence the sixteenth.
  int64_t cap = a.max_blocks > 0 ? a.max_blocks : s->gather_blocks > 0 ? s->gather_blocks : auto_gather_blocks(s, want);
  const int grid = (int)std::max<int64_t>(1, std::min(want, cap));
  if (vec == 16) launch_move_v<u32x4>(st, a, grid, nt, unroll, lpr);
  else if (vec == 8) launch_move_v<u32x2>(st, a, grid, nt, unroll, lpr);
  else launch_move_v<uint32_t>(st, a, grid, nt, unroll, lpr);
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// ------------------------------------------------------------- int8 codec
__device__ __forceinline__ float load_elem(const uint8_t *row, int i, int dtype) {
  if (dtype == LMI_F16) return __half2float(reinterpret_cast<const __half *>(row)[i]);
  return reinterpret_cast<const float *>(row)[i];
}

// One wavefront per row: absmax over the row, scale = absmax / 127,
// q = clamp(rint(x / scale), -127, 127).  The row usually lies in pinned host memory, whose link bounds the build: rows
// of up to 64 * KEEP elements stay in registers between the two passes over them, longer ones (KEEP 0) are read twice.
__device__ __forceinline__ int8_t quantize_elem(float x, float absmax, float sc) {
  float v = (absmax == 0.0f) ? 0.0f : rintf(x / sc);
  v = fminf(127.0f, fmaxf(-127.0f, v));
  return (int8_t)v;
}
template <int KEEP>
static __global__ __launch_bounds__(256) void quantize_rows_kernel(
    const int32_t *row_ids, int64_t n_rows, const uint8_t *feat, int dim, int dtype, int64_t row_bytes,
    int8_t *q, float *scale) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t n_waves = (int64_t)gridDim.x * blockDim.x / kWave;
  for (int64_t r = wave; r < n_rows; r += n_waves) {
    const uint8_t *row = feat + (int64_t)row_ids[r] * row_bytes;
    float x[KEEP > 0 ? KEEP : 1];
    float a = 0.0f;
    if constexpr (KEEP > 0) {
#pragma unroll
      for (int k = 0; k < KEEP; ++k) x[k] = lane + k * kWave < dim ? load_elem(row, lane + k * kWave, dtype) : 0.0f;
#pragma unroll
      for (int k = 0; k < KEEP; ++k) a = fmaxf(a, fabsf(x[k]));
    } else {
      for (int i = lane; i < dim; i += kWave) a = fmaxf(a, fabsf(load_elem(row, i, dtype)));
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) a = fmaxf(a, __shfl_xor(a, d, kWave));
    const float sc = a / 127.0f;
    if (lane == 0) scale[r] = sc;
    if constexpr (KEEP > 0) {
#pragma unroll
      for (int k = 0; k < KEEP; ++k)
        if (lane + k * kWave < dim) q[r * dim + lane + k * kWave] = quantize_elem(x[k], a, sc);
    } else {
      for (int i = lane; i < dim; i += kWave) q[r * dim + i] = quantize_elem(load_elem(row, i, dtype), a, sc);
    }
  }
}

// y = float(q) * scale for the four int8 values packed in `w`, bit for bit what
// __fmul_rn((float)q, scale) gives, in two instructions per element instead of three:
// the byte, biased by 128, converts as an unsigned byte in one instruction, and one fused
// multiply-add takes the bias out again -- (q + 128) * scale - 128 * scale is q * scale
// exactly before the single rounding, because 128 * scale is exact (a power of two; the
// caller takes the plain path when it would overflow).
__device__ __forceinline__ void dequant4(uint32_t w, float sc, float bias /* -128 * sc */, bool plain, float y[4]) {
  if (plain) {
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = __fmul_rn((float)(int8_t)((w >> (e * 8)) & 0xFF), sc);
    return;
  }
  const uint32_t u = w ^ 0x80808080u;
  y[0] = __fmaf_rn((float)(u & 0xFFu), sc, bias);
  y[1] = __fmaf_rn((float)((u >> 8) & 0xFFu), sc, bias);
  y[2] = __fmaf_rn((float)((u >> 16) & 0xFFu), sc, bias);
  y[3] = __fmaf_rn((float)(u >> 24), sc, bias);
}

// Dequantising gather for hits of the int8 cache, 16 elements per lane:
// y = float(q) * scale, rounded to the output type (RNE for fp16).
// Like the row mover, one launch serves several pipes (MoveGroup: src_index = slot per row,
// dst = the pipe's output rows).
template <typename OUT, int LPR>
static __global__ __launch_bounds__(256) void gather_int8_kernel(MoveGroup g, const int8_t *q, const float *scale,
                                                                 int dim, unsigned long long *row_counter) {
  LMI_GRID_ROW(g.n);
  const int32_t *cache_index = g.p[row].src_index;
  OUT *out = reinterpret_cast<OUT *>(g.p[row].dst);
  const int n = *g.p[row].n_ptr;
  const int first = g.p[row].first_ptr ? *g.p[row].first_ptr : 0;
  if (row_counter && bx == 0 && threadIdx.x == 0 && n > first)
    atomicAdd(row_counter, (unsigned long long)(n - first));
  const int lane = threadIdx.x & (LPR - 1);
  const int group = (bx * blockDim.x + threadIdx.x) / LPR;
  const int n_groups = gx * blockDim.x / LPR;
  const int chunks = dim / 16;
  for (int i = first + group; i < n; i += n_groups) {
    const int slot = cache_index[i];
    if (slot < 0) continue;
    const float sc = scale[slot];
    const bool plain = !(sc < 1.0e30f);  // 128 * scale must stay finite (also catches a NaN scale)
    const float bias = -128.0f * sc;
    const int8_t *src = q + (int64_t)slot * dim;
    OUT *dst = out + (int64_t)i * dim;
    for (int c = lane; c < chunks; c += LPR) {
      const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src + c * 16));
      union alignas(16) {
        OUT y[16];
        u32x4 v[sizeof(OUT)];
      } pk;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float f[4];
        dequant4(w[k], sc, bias, plain, f);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (sizeof(OUT) == 2) pk.y[4 * k + e] = __float2half_rn(f[e]);
          else pk.y[4 * k + e] = f[e];
        }
      }
      u32x4 *d4 = reinterpret_cast<u32x4 *>(dst + c * 16);
#pragma unroll
      for (int k = 0; k < (int)sizeof(OUT); ++k) __builtin_nontemporal_store(pk.v[k], d4 + k);
    }
  }
}

// The same gather in the shape of move_rows_tiled_kernel: the hits of a tile of 64 rows are
// staged in LDS as (output row, slot, scale), then the block walks their EPL-element units in
// flat order.  EPL = 16 / sizeof(OUT) makes every lane's output one 16-byte store and a
// wavefront's store one contiguous kilobyte.  U units in flight per lane.
template <int BYTES> struct RawVec;
template <> struct RawVec<16> { typedef u32x4 type; };
template <> struct RawVec<8> { typedef u32x2 type; };
template <> struct RawVec<4> { typedef uint32_t type; };

template <typename OUT, int EPL, int U>
static __global__ __launch_bounds__(256) void gather_int8_tiled_kernel(MoveGroup g, const int8_t *q, const float *scale,
                                                                       int dim, int tile_rows,
                                                                       unsigned long long *row_counter,
                                                                       SeenWord *rows_seen) {
  typedef typename RawVec<EPL>::type IN;
  constexpr int OUT_VECS = EPL * (int)sizeof(OUT) / 16;
  constexpr int TILE = 64;
  __shared__ int s_row[TILE], s_slot[TILE];
  __shared__ float s_scale[TILE];
  __shared__ int s_cnt;
  LMI_GRID_ROW_TAIL(g);
  const int32_t *cache_index = g.p[row].src_index;
  OUT *out = reinterpret_cast<OUT *>(g.p[row].dst);
  const int n = *g.p[row].n_ptr;
  const int first = g.p[row].first_ptr ? *g.p[row].first_ptr : 0;
  if (bx == 0 && threadIdx.x == 0) {
    if (row_counter && n > first) atomicAdd(row_counter, (unsigned long long)(n - first));
    // for the host to size the next grids by (hinted_rows)
    if (rows_seen && g.p[row].note_seeds > 0) note_seen(&rows_seen[row], n - first, g.p[row].note_seeds);
  }
  const int units = dim / EPL;
  const int dq = 256 / units, dr = 256 % units;
  const int r0 = (int)threadIdx.x / units, u0 = (int)threadIdx.x % units;
  const int n_tiles = (n - first + tile_rows - 1) / tile_rows;  // tile_rows <= TILE
  for (int tile = bx; tile < n_tiles; tile += gx) {
    if (threadIdx.x < TILE) {
      const int i = first + tile * tile_rows + (int)threadIdx.x;
      const int slot = ((int)threadIdx.x < tile_rows && i < n) ? cache_index[i] : -1;
      const uint64_t m = __ballot(slot >= 0);
      if (slot >= 0) {
        const int pos = __popcll(m & lanemask_lt());
        s_row[pos] = i;
        s_slot[pos] = slot;
        s_scale[pos] = scale[slot];
      }
      if (threadIdx.x == 0) s_cnt = __popcll(m);
    }
    __syncthreads();
    const int lim = s_cnt * units;
    int rr = r0, uu = u0;
    for (int f0 = threadIdx.x; f0 < lim; f0 += 256 * U) {
      int at[U], c[U];
      bool on[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        on[k] = f0 + k * 256 < lim;
        at[k] = rr;
        c[k] = uu;
        uu += dr;
        rr += dq;
        if (uu >= units) {
          uu -= units;
          ++rr;
        }
      }
      union {
        IN v;
        uint32_t w[EPL / 4];
      } in[U];
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (on[k])
          in[k].v = __builtin_nontemporal_load(reinterpret_cast<const IN *>(q + (int64_t)s_slot[at[k]] * dim + c[k] * EPL));
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (on[k]) {
          union alignas(16) {
            OUT y[EPL];
            u32x4 v[OUT_VECS];
          } pk;
          const float sc = s_scale[at[k]];
          const bool plain = !(sc < 1.0e30f);
          const float bias = -128.0f * sc;
#pragma unroll
          for (int e4 = 0; e4 < EPL / 4; ++e4) {
            float f[4];
            dequant4(in[k].w[e4], sc, bias, plain, f);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (sizeof(OUT) == 2) pk.y[4 * e4 + e] = __float2half_rn(f[e]);
              else pk.y[4 * e4 + e] = f[e];
            }
          }
          u32x4 *d4 = reinterpret_cast<u32x4 *>(out + (int64_t)s_row[at[k]] * dim + c[k] * EPL);
#pragma unroll
          for (int e = 0; e < OUT_VECS; ++e) __builtin_nontemporal_store(pk.v[e], d4 + e);
        }
    }
    __syncthreads();
  }
}

// Element-wise fallback for row lengths that are not a multiple of 16.
template <typename OUT>
static __global__ __launch_bounds__(256) void gather_int8_generic_kernel(MoveGroup g, const int8_t *q,
                                                                         const float *scale, int dim,
                                                                         unsigned long long *row_counter) {
  LMI_GRID_ROW(g.n);
  const int32_t *cache_index = g.p[row].src_index;
  OUT *out = reinterpret_cast<OUT *>(g.p[row].dst);
  const int n = *g.p[row].n_ptr;
  const int first = g.p[row].first_ptr ? *g.p[row].first_ptr : 0;
  if (row_counter && bx == 0 && threadIdx.x == 0 && n > first)
    atomicAdd(row_counter, (unsigned long long)(n - first));
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = (bx * blockDim.x + threadIdx.x) / kWave;
  const int n_waves = gx * blockDim.x / kWave;
  for (int i = first + wave; i < n; i += n_waves) {
    const int slot = cache_index[i];
    if (slot < 0) continue;
    const float sc = scale[slot];
    for (int c = lane; c < dim; c += kWave) {
      const float f = __fmul_rn((float)q[(int64_t)slot * dim + c], sc);
      if constexpr (sizeof(OUT) == 2) out[(int64_t)i * dim + c] = __float2half_rn(f);
      else out[(int64_t)i * dim + c] = f;
    }
  }
}

// ------------------------------------------------------------------ lookup
struct LookupArgs {
  const int32_t *ids;
  int64_t n_nodes;
  int kind;
  SlotTable table;
  LruSets lru;
  int32_t *cache_index, *lru_fill;
  int2 *miss_list;  // null: no list wanted
  DevState *st;
  int seg_first, seg_last, seg;
  const HashSlot *dedup;  // the batch's dedup table: value of a seed id = its first row; null: it was in LDS and is gone
  int dedup_log2cap;
  int lookup_blocks;  // blocks [0, lookup_blocks) look rows up, the rest carry `fill`
  FillArgs fill;      // last step of the hop sampled just before (hop -1: none)
};

// Whether seed row i repeats an earlier one, by looking (a batch small enough for LDS has few seeds).
__device__ __forceinline__ bool seed_repeats(const int32_t *ids, int i) {
  const int32_t id = ids[i];
  for (int j = 0; j < i; ++j)
    if (ids[j] == id) return true;
  return false;
}

// id -> slot for rows [first, last) of the batch -> cache_index[].  Rows that
// miss are appended to the segment's miss list as (row, id) pairs: ballot +
// prefix popcount inside each wavefront, one LDS pass over the 16 wavefronts of
// the block, one atomic per block.  The HBM gather needs no list: it walks the
// rows directly and skips the misses.  List order is arbitrary; it only
// schedules the host-link gather.
constexpr int kLookupBlock = 1024;
struct LookupGroup {  // blocks interleave over the pipes, as in the sampling kernels
  LookupArgs p[LMI_MAX_GROUP];
  int n;
};

static __global__ __launch_bounds__(kLookupBlock) void lookup_kernel(LookupGroup g) {
  LMI_GRID_ROW(g.n);
  const LookupArgs &a = g.p[row];
  __shared__ int wave_cnt[kLookupBlock / kWave];
  __shared__ int block_base;
  if (bx >= a.lookup_blocks) {
    fill_local_ids(a.fill, (int64_t)(bx - a.lookup_blocks) * blockDim.x + threadIdx.x,
                   (int64_t)(gx - a.lookup_blocks) * blockDim.x);
    return;
  }
  const int first = (a.seg_first == 0) ? 0 : a.st->node_counter[9 + a.seg_first - 1];
  const int last = a.st->node_counter[9 + a.seg_last];
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int stride = a.lookup_blocks * blockDim.x;
  for (int b = first + bx * blockDim.x; b < last; b += stride) {
    const int i = b + threadIdx.x;
    bool miss = false;
    int32_t id = -1;
    if (i < last) {
      id = a.ids[i];
      int slot = -1;
      if (id >= 0 && id < a.n_nodes) {
        if (a.kind == LMI_CACHE_LRU) {
          slot = lru_find(a.lru, id, a.st->lru_tick);
          // a repeated seed keeps both rows, but the id is offered for insertion once, by its first row
          const bool repeat =
              i < a.st->n_seeds &&
              (a.dedup ? table_find(a.dedup, a.dedup_log2cap, id, a.st->table_tag, a.st->table_mask) != i : seed_repeats(a.ids, i));
          a.lru_fill[i] = repeat ? -2 : -1;
        } else if (a.kind != LMI_CACHE_NONE) {
          slot = static_find(a.table, id);
        }
        miss = slot < 0;
      }
      a.cache_index[i] = slot;
    }
    if (!a.miss_list) continue;
    const uint64_t mm = __ballot(miss);
    if (lane == 0) wave_cnt[wid] = __popcll(mm);
    __syncthreads();
    if (threadIdx.x == 0) {
      int t = 0;
#pragma unroll
      for (int w = 0; w < kLookupBlock / kWave; ++w) {
        const int c = wave_cnt[w];
        wave_cnt[w] = t;
        t += c;
      }
      block_base = t ? atomicAdd(&a.st->n_miss[a.seg], t) : 0;
    }
    __syncthreads();
    if (miss) a.miss_list[block_base + wave_cnt[wid] + __popcll(mm & lanemask_lt())] = make_int2(i, id);
    __syncthreads();
  }
}

int launch_lookup(Server *s, Pipe *const *pp, int n, hipStream_t st, int seg_first, int seg_last, bool with_list) {
  LookupGroup g{};
  g.n = n;
  const int64_t n_max = s->node_cap[seg_last];
  const int lookup_blocks = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n_max, kLookupBlock), (int64_t)s->n_cu * 2));
  int grid = lookup_blocks;
  const int pending = pp[0]->fill_pending;  // the hop sampled last left its local ids to this kernel
  if (pending >= 0) grid += fill_blocks(s->edge_cap[pending], kLookupBlock);
  for (int k = 0; k < n; ++k) {
    Pipe &p = *pp[k];
    LookupArgs &a = g.p[k];
    a.ids = p.ids;
    a.n_nodes = s->n_nodes;
    a.kind = s->cache_kind;
    a.table = slot_table(s);
    a.lru = lru_sets(s);
    a.cache_index = p.cache_index;
    a.miss_list = with_list ? p.miss_list + miss_list_base(s, seg_first) : nullptr;
    a.lru_fill = p.lru_fill;
    a.dedup = p.table_in_lds ? nullptr : p.dedup.slots;
    a.dedup_log2cap = p.dedup.log2cap;
    a.st = p.st;
    a.seg_first = seg_first;
    a.seg_last = seg_last;
    a.seg = seg_first;
    a.lookup_blocks = lookup_blocks;
    a.fill.hop = -1;
    if (pending >= 0) a.fill = fill_args(p, pending);
    p.fill_pending = -1;
  }
  hipLaunchKernelGGL(lookup_kernel, dim3(grid * n), dim3(kLookupBlock), 0, st, g);
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// Orders `st` behind the pipe's last batch.  Its side-stream work ends with the event `join_of`; a
// wait on another queue's event holds a stream up for about 10 us even when the event fired long
// ago, so that wait is only queued when the host cannot already see the event as complete.  Work
// of the batch that `join_of` does not cover sits on the caller's stream that carried the batch:
// the same stream orders itself.  Another one waits for the batch's own end where that was marked
// (tail_event), so that it does not wait for batches queued behind it and does not need that stream
// any more; else, as between operators, for an event recorded there now (at that stream's present
// tail, which is at or behind the batch's last kernel).
int pipe_handover(Pipe &p, hipStream_t st) {
  if (!p.tail_unjoined || p.last_stream == st || !p.handover) return LMI_OK;
  if (p.tail_event) {
    const bool done = hipEventQuery(p.tail_event) == hipSuccess;
    if (!done) {
      (void)hipGetLastError();  // "not ready" is an answer, not a failure
      LMI_HIP(hipStreamWaitEvent(st, p.tail_event, 0));
    }
    if (p.tail_follow) p.tail_event = nullptr;
    else if (done) p.tail_unjoined = false;
  } else {
    LMI_HIP(hipEventRecord(p.handover, p.last_stream));
    LMI_HIP(hipStreamWaitEvent(st, p.handover, 0));
  }
  p.last_stream = st;  // `st` now carries the order
  return LMI_OK;
}

int pipe_join(Pipe &p, hipStream_t st) {
  LMI_TRY(pipe_handover(p, st));
  if (!p.side_pending || (p.join_waited && p.join_waiter == st)) return LMI_OK;
  if (hipEventQuery(p.join_of) == hipSuccess) {
    p.side_pending = false;  // complete: no stream has to wait any more
    return LMI_OK;
  }
  (void)hipGetLastError();  // "not ready" is an answer, not a failure
  LMI_HIP(hipStreamWaitEvent(st, p.join_of, 0));
  p.join_waited = true;  // this stream is in order; another one that names the pipe later still has to wait
  p.join_waiter = st;
  return LMI_OK;
}

// A join event was just recorded for the pipe on the side stream.
static void pipe_side_owes(Pipe &p, hipEvent_t join_of) {
  p.join_of = join_of;
  p.side_pending = true;
  p.join_waited = false;
}

int pipes_join(Pipe *const *pp, int n, hipStream_t st) {
  hipEvent_t seen[LMI_MAX_GROUP];
  bool done[LMI_MAX_GROUP];
  int n_seen = 0;
  for (int k = 0; k < n; ++k) {
    Pipe &p = *pp[k];
    LMI_TRY(pipe_handover(p, st));
    if (!p.side_pending) continue;
    int dup = -1;
    for (int j = 0; j < n_seen; ++j)
      if (seen[j] == p.join_of) dup = j;
    if (dup >= 0) {  // `st` already waits for this event, or has seen it complete
      if (done[dup]) p.side_pending = false;
      else p.join_waited = true, p.join_waiter = st;
      continue;
    }
    LMI_TRY(pipe_join(p, st));
    if (n_seen < LMI_MAX_GROUP) {
      seen[n_seen] = p.join_of;
      done[n_seen++] = !p.side_pending;
    }
  }
  return LMI_OK;
}

// int8 rows: dequantised inside the gather.
static int launch_hits_int8(Server *s, const MoveGroup &g, int64_t rows_hint, hipStream_t st, int seg, int seg_last, hipEvent_t end) {
  const int64_t n_max = s->node_cap[seg_last];
  const int dim = s->cfg.feat_dim;
  const int64_t want = ceil_div(n_max, 4);
  const int64_t cap = s->gather_blocks > 0 ? s->gather_blocks : auto_gather_blocks(s, want);
  const int grid = g.n * (int)std::max<int64_t>(1, std::min<int64_t>(want, cap));
  const int8_t *q = (const int8_t *)s->cache_data;
  unsigned long long *rc = s->prof_on ? s->d_prof_rows : nullptr;
  hipEvent_t e0, e1;
  prof_kernel_events(s, PROF_GATHER_HIT, &e0, &e1);
  if (end) e1 = end;
#define LMI_INT8(KERN)                                                                                   \
  if (e0 || e1)                                                                                          \
    hipExtLaunchKernelGGL((KERN), dim3(grid), dim3(256), 0, st, e0, e1, 0, g, q, s->cache_scale, dim, rc); \
  else                                                                                                   \
    hipLaunchKernelGGL((KERN), dim3(grid), dim3(256), 0, st, g, q, s->cache_scale, dim, rc)
  const bool half = s->cfg.feat_dtype == LMI_F16;
  if (dim % 16 == 0 && s->gather_flat != 2) {
    // elements per lane: by default as many as make one 16-byte store (8 fp16, 4 fp32)
    int epl = s->int8_epl > 0 ? s->int8_epl : (half ? 8 : 4);
    if (epl != 16 && epl != 8 && epl != 4) epl = half ? 8 : 4;
    if (half && epl == 4) epl = 8;  // fewer than 16 output bytes per lane are not offered
    // 768-element fp16 rows, share of HBM peak: 8 rows per tile 45 %, 16 51 %, 32 54 %, 64 52 %
    const int tile_rows = s->gather_tile_rows > 0 ? std::min(64, s->gather_tile_rows) : 32;
    // sized by the rows the last launches held (hinted_rows): a block without a tile is not free
    const int64_t want_f = ceil_div(rows_hint, tile_rows);
    const int64_t cap_f = s->gather_blocks > 0 ? s->gather_blocks
                          : s->gather_adaptive ? (int64_t)s->n_cu * 64 : auto_gather_blocks(s, want_f);
    const int grid_f = g.n * ((int)std::max<int64_t>(1, std::min<int64_t>(want_f, cap_f)) + g.tail_blocks);
#define LMI_INT8_FLAT(KERN)                                                                                   \
  if (e0 || e1)                                                                                               \
    hipExtLaunchKernelGGL((KERN), dim3(grid_f), dim3(256), 0, st, e0, e1, 0, g, q, s->cache_scale, dim,        \
                          tile_rows, rc, s->rows_seen_dev + rows_word(s, seg, seg_last));                      \
  else                                                                                                        \
    hipLaunchKernelGGL((KERN), dim3(grid_f), dim3(256), 0, st, g, q, s->cache_scale, dim, tile_rows, rc,       \
                       s->rows_seen_dev + rows_word(s, seg, seg_last))
#define LMI_INT8_FLAT_U(OUT_, EPL_)                                    \
  if (s->gather_unroll >= 4) {                                         \
    LMI_INT8_FLAT((gather_int8_tiled_kernel<OUT_, EPL_, 4>));           \
  } else if (s->gather_unroll != 1) {                                  \
    LMI_INT8_FLAT((gather_int8_tiled_kernel<OUT_, EPL_, 2>));           \
  } else {                                                             \
    LMI_INT8_FLAT((gather_int8_tiled_kernel<OUT_, EPL_, 1>));           \
  }
    if (half && epl == 16) {
      LMI_INT8_FLAT_U(__half, 16)
    } else if (half) {
      LMI_INT8_FLAT_U(__half, 8)
    } else if (epl == 16) {
      LMI_INT8_FLAT_U(float, 16)
    } else if (epl == 8) {
      LMI_INT8_FLAT_U(float, 8)
    } else {
      LMI_INT8_FLAT_U(float, 4)
    }
#undef LMI_INT8_FLAT_U
#undef LMI_INT8_FLAT
  } else if (dim % 16 == 0) {
    // lanes per row: 16 or 32, several 16-element chunks per lane when the row is longer (768-d rows,
    // beside the host-link gather: 64 lanes, 48 of them busy, 39 % of HBM peak; 32 lanes x 2 steps 48 %;
    // 16 lanes x 3 steps 49 %; 8 lanes x 6 steps 46 %), or what the measurement knob asks for
    int lpr = s->gather_lpr;
    if (lpr != 8 && lpr != 16 && lpr != 32 && lpr != 64) lpr = dim / 16 <= 16 ? 16 : 32;
#define LMI_INT8_L(OUT_)                                   \
  if (lpr == 8) {                                          \
    LMI_INT8((gather_int8_kernel<OUT_, 8>));               \
  } else if (lpr == 16) {                                  \
    LMI_INT8((gather_int8_kernel<OUT_, 16>));              \
  } else if (lpr == 32) {                                  \
    LMI_INT8((gather_int8_kernel<OUT_, 32>));              \
  } else {                                                 \
    LMI_INT8((gather_int8_kernel<OUT_, 64>));              \
  }
    if (half) {
      LMI_INT8_L(__half)
    } else {
      LMI_INT8_L(float)
    }
#undef LMI_INT8_L
  } else if (half) {
    LMI_INT8((gather_int8_generic_kernel<__half>));
  } else {
    LMI_INT8((gather_int8_generic_kernel<float>));
  }
#undef LMI_INT8
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// Hands the batches' last steps to a launch over `g`.
static void tail_args(Server *s, Pipe *const *pp, int n, const HeaderCopy *headers, MoveGroup *g) {
  const int pending = pp[0]->fill_pending;  // the pipes are in step
  if (pending < 0 && !headers) return;
  g->tail_blocks = pending >= 0 ? fill_blocks(s->edge_cap[pending], 256) : 1;
  for (int k = 0; k < n; ++k) {
    g->p[k].fill = fill_args(*pp[k], pending);
    if (headers) g->p[k].headers = *headers;
    pp[k]->fill_pending = -1;
  }
}

static __global__ __launch_bounds__(256) void batch_tail_kernel(MoveGroup g) {
  LMI_GRID_ROW(g.n);
  batch_tail(g.p[row], bx, g.tail_blocks);
}

// ... or to a launch of their own, if anything is left.
static int launch_batch_tail(Server *s, Pipe *const *pp, int n, hipStream_t st, const HeaderCopy *headers) {
  MoveGroup g{};
  g.n = n;
  tail_args(s, pp, n, headers, &g);
  if (g.tail_blocks == 0) return LMI_OK;
  hipLaunchKernelGGL(batch_tail_kernel, dim3(g.tail_blocks * n), dim3(256), 0, st, g);
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// No cache and the table behind the host link: every row of a batch comes over the link.
static bool all_rows_over_link(const Server *s) { return s->cache_kind == LMI_CACHE_NONE && s->feat_loc == LMI_LOC_HOST; }

// Gather of rows [first, last) on stream `st`, for all n pipes in one launch: the cache hits from HBM, and with
// `misses` the other rows from the feature table in the same pass (only where gather_in_line allows it).  end: an event
// that marks the end of the launch (not with a profiled gather, which carries events of its own).
static int launch_hits(Server *s, Pipe *const *pp, int n, hipStream_t st, int seg, int seg_last, bool misses = false,
                       const HeaderCopy *headers = nullptr, bool look = false, hipEvent_t end = nullptr) {
  LMI_TRY(lru_wait_copied(s, st));
  // what is left of the batch rides in the flat and the tiled int8 gather; a profiled gather is timed by itself
  // (launch_gather_group)
  const bool carries = !s->prof_on && (s->cache_kind == LMI_CACHE_INT8
                                           ? s->cfg.feat_dim % 16 == 0 && s->gather_flat != 2
                                           : s->row_bytes >= 16 && !lane_group_knobs(s, false) &&
                                                 (s->gather_flat == 0 || s->gather_flat == 3));
  if (!carries) LMI_TRY(launch_batch_tail(s, pp, n, st, headers));
  const int64_t n_max = s->node_cap[seg_last];
  const bool have_cache = s->cache_kind != LMI_CACHE_NONE;
  MoveArgs m{};
  m.g.n = n;
  for (int k = 0; k < n; ++k) {
    const Pipe &p = *pp[k];
    MoveRow &r = m.g.p[k];
    r.list = nullptr;  // rows [first, n) directly; cache_index < 0 (a miss) skips the row
    r.first_ptr = seg == 0 ? nullptr : &p.st->node_counter[9 + seg - 1];
    r.n_ptr = &p.st->node_counter[9 + seg_last];
    r.src_index = have_cache ? p.cache_index : p.ids;
    r.ids = p.ids;
    r.look_index = p.cache_index;
    r.dst = (uint8_t *)p.features;
    r.note_seeds = p.note_seeds;
    r.fill.hop = -1;
  }
  if (carries) tail_args(s, pp, n, headers, &m.g);
  m.note_rows = rows_word(s, seg, seg_last);
  m.rows_hint = hinted_rows(s, n_max, m.note_rows, pp, n);
  if (s->cache_kind == LMI_CACHE_INT8) return launch_hits_int8(s, m.g, m.rows_hint, st, seg, seg_last, end);
  m.src = have_cache ? s->cache_data : s->feat;
  m.n_src = have_cache ? s->cache_rows : s->n_nodes;
  if (misses && have_cache) {
    m.table = s->feat;
    m.n_table = s->n_nodes;
    m.look = look ? 1 : 0;
  }
  if (all_rows_over_link(s)) {
    // A grid that fills the link, not the device: more reads in flight cost the link a tenth (3 400 rows of 4 096 bytes,
    // us on the whole grid 309, 256 blocks 278, 128 273, 96 273, 64 278, 48 285; 24 000 rows of 256 bytes 182, 171, 168,
    // 169, 168, 173; four batches of 24 000 rows of 3 072 bytes, on all of the blocks, 5 558, 5 396, 5 604, 5 548, 5 434, 5 508).
    const int blocks = s->miss_blocks > 0 ? s->miss_blocks : s->miss_blocks == 0 ? s->n_cu : 96;
    m.max_blocks = std::max(1, (blocks + n - 1) / n);  // per pipe
  }
  m.src_row_bytes = m.dst_row_bytes = m.row_bytes = s->row_bytes;
  m.n_max = n_max;
  m.row_counter = s->prof_on ? s->d_prof_rows : nullptr;  // all rows of the segment: hits + misses
  prof_kernel_events(s, PROF_GATHER_HIT, &m.ev_start, &m.ev_stop);
  if (end) m.ev_stop = end;
  return launch_move_rows(s, st, m, s->gather_nt != 0);
}

// Gather of the rows on the segment's miss list from the feature table, on a
// small grid when the table sits behind the host link (few bytes in flight fill it).
// One launch for all n pipes; the small grid is then shared between them.
static int launch_misses(Server *s, Pipe *const *pp, int n, hipStream_t st, int seg, int seg_last, int blocks_override = 0,
                         hipEvent_t end = nullptr) {
  MoveArgs m{};
  m.g.n = n;
  for (int k = 0; k < n; ++k) {
    MoveRow &r = m.g.p[k];
    r.list = pp[k]->miss_list + miss_list_base(s, seg);
    r.n_ptr = &pp[k]->st->n_miss[seg];
    r.dst = (uint8_t *)pp[k]->features;
  }
  m.src_from_list = 1;
  m.src = s->feat;
  m.src_row_bytes = m.dst_row_bytes = m.row_bytes = s->row_bytes;
  m.n_max = s->node_cap[seg_last];
  if (s->feat_loc == LMI_LOC_HOST) {
    // (listed rows without a cache: nothing runs beside them)
    const int usual = s->miss_blocks >= 0 ? s->miss_blocks : all_rows_over_link(s) ? 64 : n >= 4 ? 40 : 32;
    const int blocks = blocks_override > 0 ? blocks_override : usual > 0 ? usual : s->n_cu;
    m.max_blocks = std::max(1, (blocks + n - 1) / n);  // per pipe
    m.unroll = s->miss_unroll;
    m.host_link = 1;
  }
  m.row_counter = s->prof_on ? s->d_prof_rows + 1 : nullptr;  // misses
  prof_kernel_events(s, PROF_GATHER_MISS, &m.ev_start, &m.ev_stop);
  if (end) m.ev_stop = end;
  return launch_move_rows(s, st, m, s->gather_nt != 0);
}

// Every node has a slot: no batch has a miss.
static bool no_miss_possible(const Server *s) {
  return (s->cache_kind == LMI_CACHE_STATIC || s->cache_kind == LMI_CACHE_INT8) && s->cache_rows >= s->n_nodes;
}

// Hits and misses in one pass of the flat gather: full-width cache rows (an int8 hit and a miss are moved in
// different ways) of at least 16 bytes, no measurement knob that asks for another mover.  A profiled batch keeps
// two launches, so that each gather is timed by itself.  Where all rows come over the link, rows of more than a block's
// 256 lanes of 16 bytes are listed and left to the LDS-tiled mover, which keeps whole rows in flight (us of a batch of
// 24 000 rows in one pass / listed: 4 096 bytes 1 829 / 1 855, 5 732 bytes 2 760 / 2 626, 8 192 bytes 3 717 / 3 606).
bool one_pass_gather(const Server *s) {
  return s->cache_kind != LMI_CACHE_INT8 && s->row_bytes >= 16 && !lane_group_knobs(s, false) &&
         (s->gather_flat == 0 || s->gather_flat == 3) && !s->prof_on && !(all_rows_over_link(s) && s->row_bytes > 4096);
}

// Whether the misses are gathered on the caller's stream like the hits (profiled batches too, in two launches).  A side
// stream for them costs a fork and a
// join: 26 us on the device where a second launch on the same stream costs 5, and 11 us of the host's time for each
// wait it queues.  It pays when it lets the misses of a batch overlap the sampling of the next one -- so not
//  * when the table lies in HBM, or there is no cache, or no row can miss;
//  * when what a batch can miss at all takes the link less time than the fork and join (1 MB: 20 us);
//  * when the caller takes a batch in order, on the batch's own stream, before it issues the next (lmi_batch_wait
//    on that stream, or reading the batch back): nothing is left to overlap.  The batch before tells.
// ogbn-products-shaped, one batch of 800 seeds at a time with a wait on the same stream: 160 us with the side
// stream, 122 us with everything on one and hits and misses in one launch (inference of 16 seeds: 70 and 36 us).
bool gather_in_line(const Server *s, Pipe *const *pp, int n, int seg_last) {
  if (s->split_miss == 0 || s->feat_loc != LMI_LOC_HOST || s->cache_kind == LMI_CACHE_NONE) return true;
  if (no_miss_possible(s)) return true;
  if (s->split_miss != 1 || s->protect_hits) return false;
  constexpr int64_t kFewBytes = 1 << 20;
  if (n * s->node_cap[seg_last] * s->row_bytes <= kFewBytes) return true;
  for (int k = 0; k < n; ++k)
    if (!pp[k]->taken_in_order) return false;
  return true;
}

// Whether the hops' launches gather the rows that a batch knows before them (early_rows), and the last hop's tiles the rows
// they add (tile_rows), in place of a gather behind the hops: where the misses come over the host link on the caller's
// stream, in one pass with the hits.  The link, which bounds such a batch, then works while the hops are sampled, and starts
// on a tile's misses while others are still being ranked; a launch and a pass over ids and slots go.  Not with the LRU
// cache, whose batches miss little, and not from a table in HBM, whose reads the hops' own wait for.
// Blocks and tiles of a hop move hits more slowly than a grid of the gather's own, which shows for long rows where most are
// hits.  So early_rows up to 4 KB, above 512 bytes only where enough rows miss, and tile_rows where a thread has few bytes to
// move and the link is busy for longer than that takes.  The limits are fits, not derived: 512 and 4 096 bytes, 1.8 % of
// misses, 450 and 1 300 bytes a thread, and a microsecond of link for every ten of these, to the batches below; that 2.2 times
// the keys outside the cache miss (Server::miss_share; the distinct nodes of a batch are drawn more evenly than its edges are)
// to synthetic graphs of Zipf-distributed degrees whose neighbours are drawn in proportion to them.  Elsewhere the rules may
// take the slower way.  us a batch of 800 seeds, 10,5, gathered behind the hops / early_rows / both
// (bytes a thread of the last hop's tiles, us over the link as estimated here), by bytes of a row and share of nodes cached:
//   400: 20 % 61 / 57 / 54 (122, 34), 50 % 55 / 54 / 51 (98, 18), 90 % 39 / 38 / 39 (98, 2);  1 024, 4 000 seeds, 5,4: 50 % 113 / 111 / 105
//   (370, 47);  1 536: 80 % 43 / 38 / 48 (470, 8);  2 408: 20 % 208 / 198 / 196 (736, 207), 60 % 75 / 72 / 70 (736, 38), 70 % 62 / 58 / 62
//   (736, 23), 80 % 50 / 49 / 59 (736, 12);  4 096: 60 % 102 / 98 / 103 (1 253, 65);  5 732: 20 % 441 / 437 / 449, 80 % 73 / 87 / 118
//   (1 753, 28);  no cache: 3 072 870 / 857 / 829 (939, 804), 4 096 1 116 / 1 101 / 1 098 (1 253, 1 072);
//   156 seeds, 10,5, 1 024: 26 % 36 / 28 / 39 (400, 16);  65 seeds, 25,15, 2 408: 62 % 38 / 31 / 50 (815, 9).

// Bytes a second, of 400-byte rows, for rows of every length in these rules (aligned rows of 512 bytes come at 55e9, of 200 bytes
// at 31e9).
constexpr double kLinkRate = 41e9;
static double miss_estimate(const Server *s) {
  if (s->cache_kind == LMI_CACHE_NONE) return 1.0;
  return std::min(1.0, s->policy_built == LMI_POLICY_PRESAMPLED ? s->miss_share : 2.2 * s->miss_share);
}
// A gather that a knob shapes stays a launch of its own: rows in the hops and beside small batches take their tiles and grid
// from those launches, and are stored non-temporally.  (Rows in flight per lane follow their knob only without a cache.)
bool gather_knobs(const Server *s) {
  return s->gather_tile_rows > 0 || s->gather_blocks > 0 || !s->gather_nt ||
         (s->gather_unroll > 0 && s->cache_kind == LMI_CACHE_NONE);
}
bool early_rows(const Server *s, bool in_line) {
  return in_line && !gather_knobs(s) && one_pass_gather(s) && s->feat_loc == LMI_LOC_HOST && !no_miss_possible(s) && s->fuse_count && !s->lds_dedup &&
         (s->cache_kind == LMI_CACHE_STATIC || s->cache_kind == LMI_CACHE_NONE) &&
         (s->row_bytes <= 512 || (s->row_bytes <= 4096 && miss_estimate(s) >= 0.018));
}
// `n` batches of `added` new rows each, out of `tiles` tiles of `shape` each.
bool tile_rows(const Server *s, int n, int64_t added, int64_t tiles, const HopShape &shape) {
  const double bytes = (double)n * (double)added * (double)s->row_bytes;
  // (with several nodes per lane group a thread has half as much under way)
  const double thread = bytes / (double)(n * tiles * shape.block) * (shape.passes == 1 ? 1 : 2);
  const double link_us = bytes * miss_estimate(s) / kLinkRate * 1e6;
  return thread <= (s->cache_kind == LMI_CACHE_NONE ? 1300 : 450) && link_us >= 0.1 * thread;
}
// Their blocks (of 256 threads), for all batches of a launch: a grid that fills the link, as in launch_hits; more where the
// rows, most of which are hits, would take such a grid longer than a hop takes.
int early_rows_blocks(const Server *s, int64_t rows) {
  const int64_t link = s->miss_blocks > 0 ? s->miss_blocks : s->miss_blocks == 0 ? s->n_cu : 96;
  if (s->cache_kind == LMI_CACHE_NONE) return (int)link;
  return (int)std::max<int64_t>(link, std::min<int64_t>(ceil_div(rows * s->row_bytes, 1 << 17), 2048));
}

// Lookup and gather of one segment in one launch (operator by operator; gather_in_line and one_pass_gather hold): a static
// cache with full-width rows.  The operators of a products-shaped batch: 126 us with
// three lookup launches (and one more at the start of the batch), 109 without.
bool lookup_rides_in_gather(const Server *s) { return s->cache_kind == LMI_CACHE_STATIC; }
int launch_lookup_gather(Server *s, Pipe &p, hipStream_t st, int seg) {
  Pipe *pp[1] = {&p};
  p.tail_unjoined = true;  // everything is on the caller's stream
  ++s->routes.gather_lookups;
  return launch_hits(s, pp, 1, st, seg, seg, true, nullptr, true);
}

// The host-link gather of segments [seg, seg_last], released ahead of the batch's later hops.
int launch_misses_early(Server *s, Pipe *const *pp, int n, hipStream_t st, int seg, int seg_last) {
  hipEvent_t fork = pp[0]->fork_early;
  LMI_HIP(hipEventRecord(fork, st));
  LMI_HIP(hipStreamWaitEvent(s->side, fork, 0));
  if (n > 1 && s->group_miss) return launch_misses(s, pp, n, s->side, seg, seg_last, s->miss_blocks_early);
  for (int k = 0; k < n; ++k) LMI_TRY(launch_misses(s, pp + k, 1, s->side, seg, seg_last, s->miss_blocks_early));
  return LMI_OK;  // the join event that launch_gather_group records behind the batch's last misses covers these
}

// Whether a side stream's join event ends batches like this one: behind that nobody follows the stream that takes a batch, so
// neither where the gather is in line only because that side stream would have nothing to overlap.
static bool batch_sided(const Server *s, bool early_fork) {
  return s->feat_loc == LMI_LOC_HOST && s->cache_kind != LMI_CACHE_NONE && (s->split_miss == 2 || (s->split_miss == 1 && !early_fork));
}
static bool early_forked(const Server *s, int n) { return s->early_fork == 1 || (s->early_fork == 2 && n > 1); }

void rows_gathered(Server *s, Pipe *const *pp, int n, hipEvent_t end) {
  s->routes.one_pass_gathers += n;
  for (int k = 0; k < n; ++k) {
    pp[k]->tail_follow = !batch_sided(s, early_forked(s, n));
    pp[k]->tail_unjoined = true;
    pp[k]->tail_event = end;
  }
}

// Gathers the rows [first, last) of a segment into each pipe's feature buffer:
// cache hits from HBM, misses from the feature table, over the host link where it lies
// in host memory.  With several pipes, the hits of all are one launch and so are the
// misses (group_miss).  Schedules (tuning key "split_miss"):
//   0  both on the caller's stream, in one pass where one_pass_gather allows it;
//   1  hits on the caller's stream, misses on the server's side stream, where they
//      overlap the next batch's sampling.  A wide host-link gather beside HBM gathers
//      cuts their bandwidth by more than half: it runs on a small grid (miss_blocks);
//   2  both on the side stream (a gather stage behind the sampling stage): the
//      caller's stream is free for the next batch's sampling as soon as the lookup
//      is done.
// gather_in_line says when schedule 0 is taken whatever the knob says: nothing is left
// then for a side stream to overlap, and a wide grid has no neighbour to slow.
// With 1 and 2 the caller's stream does not wait here: the next call on this pipe,
// or lmi_batch_wait, joins.  A segment of an LRU batch joins at once (a later call
// inserts the gathered rows).
int launch_gather_group(Server *s, Pipe *const *pp, int n, hipStream_t st, int seg, int seg_last, int lru_lists,
                        bool same_stream, int hit_seg_first, const HeaderCopy *headers, bool early_rows) {
  if (early_rows) seg = seg_last;  // the hops' launches took the rows before the last hop's
  const int hit_seg = hit_seg_first >= 0 ? hit_seg_first : seg;  // the hits of segments whose misses went ahead
  const bool have_cache = s->cache_kind != LMI_CACHE_NONE;
  const bool in_line = same_stream || gather_in_line(s, pp, n, seg_last);
  int mode = in_line ? 0 : s->split_miss;
  // The gather kernels carry their own profiling events (prof_kernel_events); a bracket
  // left open by the sampling phase ends here, with the last hop's fill.
  if (s->prof_on) LMI_TRY(launch_batch_tail(s, pp, n, st, headers));
  prof_phase(s, st, &s->prof_open, -1);
  // What a batch leaves on the caller's stream ends with a kernel of its gather, which carries an event that says so (the
  // first pipe's for all pipes of a group): recorded behind it the event would be a packet of its own, and recorded when
  // another stream asks it would stand for whatever is queued by then.  Not for a segment: its batch goes on.
  const bool whole = (hit_seg == 0 || early_rows) && seg_last == s->cfg.hops;
  const hipEvent_t end = whole && !s->prof_on ? pp[0]->handover : nullptr;
  // LRU batches are host-link-bound (a fifth of their rows miss): their host-link gather starts
  // beside the HBM gather instead of behind it.  The insertion that follows it on the side stream
  // only overwrites ways this batch's lookup did not touch, so the hits never read a row it writes.
  const bool early = (lru_lists > 0 && s->lru_early_miss) ||
                     (lru_lists == 0 && early_forked(s, n));
  for (int k = 0; k < n; ++k) pp[k]->tail_follow = !batch_sided(s, early);
  if (mode == 0) {
    const bool last_hits = lru_lists == 0 && (one_pass_gather(s) || no_miss_possible(s));
    for (int k = 0; k < n; ++k) {
      pp[k]->tail_unjoined = true;
      pp[k]->tail_event = end;
    }
    if (one_pass_gather(s)) {
      s->routes.one_pass_gathers += n;
      LMI_TRY(launch_hits(s, pp, n, st, seg, seg_last, true, headers, false, last_hits ? end : nullptr));
    } else {
      if (have_cache) LMI_TRY(launch_hits(s, pp, n, st, seg, seg_last, false, headers, false, last_hits ? end : nullptr));
      else LMI_TRY(launch_batch_tail(s, pp, n, st, headers));
      if (!no_miss_possible(s)) LMI_TRY(launch_misses(s, pp, n, st, seg, seg_last, 0, lru_lists == 0 ? end : nullptr));
    }
    for (int k = 0; k < n && lru_lists > 0; ++k) LMI_TRY(launch_lru_insert(s, *pp[k], st, lru_lists, end));
    return LMI_OK;
  }
  hipEvent_t fork = nullptr;
  if (mode == 2) {
    LMI_TRY(launch_batch_tail(s, pp, n, st, nullptr));
    for (int k = 0; k < n; ++k) pp[k]->tail_unjoined = false;  // both gathers run behind the fork
  }
  if (mode == 1) {
    // Host-link reads in flight halve the HBM gather's bandwidth: optionally hold the hits back
    // until the side stream has drained the host-link gathers issued before (other pipes').
    if (s->protect_hits && s->side_busy) {
      if (hipEventQuery(s->side_idle) != hipSuccess) {
        (void)hipGetLastError();
        LMI_HIP(hipStreamWaitEvent(st, s->side_idle, 0));
      } else {
        s->side_busy = false;
      }
    }
    // behind a late fork the join event covers the whole batch; ahead of an early one the HBM gather stays
    // on the caller's stream alone
    for (int k = 0; k < n; ++k) {
      pp[k]->tail_unjoined = early;
      pp[k]->tail_event = early ? end : nullptr;
    }
    if (early) {
      fork = pp[0]->fork;
      LMI_HIP(hipEventRecord(fork, st));
    }
    // one launch for the group
    LMI_TRY(launch_hits(s, pp, n, st, hit_seg, seg_last, false, nullptr, false, early ? end : nullptr));
  }
  if (!fork) {  // one fork for the whole group
    fork = pp[0]->fork;
    LMI_HIP(hipEventRecord(fork, st));
  }
  LMI_HIP(hipStreamWaitEvent(s->side, fork, 0));
  // the group's host-link gathers as one launch when nothing has to come between them
  const bool misses_together = n > 1 && mode == 1 && lru_lists == 0 && s->group_miss;
  if (misses_together) LMI_TRY(launch_misses(s, pp, n, s->side, seg, seg_last));
  if (misses_together) {  // nothing else of the group goes to the side stream: one event for all its pipes
    LMI_HIP(hipEventRecord(pp[0]->join, s->side));
    for (int k = 0; k < n; ++k) pipe_side_owes(*pp[k], pp[0]->join);
  }
  for (int k = 0; k < n && !misses_together; ++k) {
    Pipe &p = *pp[k];
    if (mode == 2) LMI_TRY(launch_hits(s, pp + k, 1, s->side, seg, seg_last));
    LMI_TRY(launch_misses(s, pp + k, 1, s->side, seg, seg_last));
    if (lru_lists > 0) LMI_TRY(launch_lru_insert(s, p, s->side, lru_lists));  // reads the rows just gathered
    LMI_HIP(hipEventRecord(p.join, s->side));
    pipe_side_owes(p, p.join);
    // an LRU insertion that comes later on the caller's stream copies the gathered rows: join now
    if (s->cache_kind == LMI_CACHE_LRU && lru_lists == 0) LMI_TRY(pipe_join(p, st));
  }
  if (s->protect_hits) {
    LMI_HIP(hipEventRecord(s->side_idle, s->side));
    s->side_busy = true;
  }
  return LMI_OK;
}

int launch_gather_seg(Server *s, Pipe &p, hipStream_t st, int seg, int seg_last, int lru_lists) {
  Pipe *pp[1] = {&p};
  return launch_gather_group(s, pp, 1, st, seg, seg_last, lru_lists);
}

// --------------------------------------------------------------- LRU insert
// Batch-synchronous insertion in two launches.  lru_chain_kernel threads the misses of
// every set into a list (head[set] -> row -> next[row] ...; one atomic exchange per miss,
// on as many addresses as there are sets).  lru_place_kernel: the thread of the row at a
// list's head serves its set alone -- the set's misses in ascending row order each take
// the way with the smallest (last_use, way) among ways not touched in this batch, until
// no way is left; the rest are refused (-2).  A list is as long as the batch has misses
// in that set (one or two for any useful geometry), and the walk is serial, so a cache of
// very few sets pays for its collisions in time, not in correctness.
struct LruArgs {
  const int32_t *ids;
  const int2 *miss_list[LMI_MAX_HOPS + 1];
  const DevState *st;
  int n_lists;
  int32_t *keys, *use, *head, *next, *fill;
  int64_t sets;
  int ways;
};

// Not needed where the lookup has chained the misses already (LOOK_LRU).
static __global__ __launch_bounds__(256) void lru_chain_kernel(LruArgs a, LruSets t) {
  for (int l = 0; l < a.n_lists; ++l) {
    const int n = a.st->n_miss[l];
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
      const int2 pr = a.miss_list[l][j];  // (row, id)
      const int i = pr.x;
      if (a.fill[i] != -1) continue;  // the later row of a repeated seed
      lru_chain(t, a.next, i, pr.y);
    }
  }
}

// Serves the set of the miss `pr` (row, id) if its row is at the head of the set's list; granted(row, slot) for every row
// that gets a way.
template <typename F>
__device__ __forceinline__ void lru_place(const LruArgs &a, int2 pr, int tick, F granted) {
  const int i = pr.x;
  const int64_t set = (uint32_t)pr.y % (uint32_t)a.sets;  // sets < 2^31
  if (a.head[set] != i) return;  // some other row's thread serves this set
  const int64_t base = set * a.ways;     // the set's first slot (row of the cache)
  const int64_t rec = set * 2 * a.ways;  // the set's record: keys, then ticks
  int last = -1;  // the row placed last; the next one is the smallest row above it
  for (int placed = 0; placed < a.ways; ++placed) {
    int row = kIntMax;
    for (int r = i; r != -1; r = a.next[r])
      if (r > last && r < row) row = r;
    if (row == kIntMax) break;  // everybody is placed
    int best = -1, best_use = kIntMax;
    if ((a.ways & 3) == 0) {  // four ways per load, same order of preference (lowest way wins a tie)
      for (int w = 0; w < a.ways; w += 4) {
        const int4 u = *reinterpret_cast<const int4 *>(a.use + rec + w);
        if (u.x < tick && u.x < best_use) best = w, best_use = u.x;
        if (u.y < tick && u.y < best_use) best = w + 1, best_use = u.y;
        if (u.z < tick && u.z < best_use) best = w + 2, best_use = u.z;
        if (u.w < tick && u.w < best_use) best = w + 3, best_use = u.w;
      }
    } else {
      for (int w = 0; w < a.ways; ++w) {
        const int u = a.use[rec + w];
        if (u < tick && u < best_use) best = w, best_use = u;
      }
    }
    if (best < 0) break;  // every way was touched in this batch
    a.keys[rec + best] = a.ids[row];
    a.use[rec + best] = tick;
    a.fill[row] = (int)(base + best);
    granted(row, (int)(base + best));
    last = row;
  }
  for (int r = i; r != -1; r = a.next[r])
    if (a.fill[r] == -1) a.fill[r] = -2;  // no way left for these
  a.head[set] = -1;  // ready for the next batch
}

static __global__ __launch_bounds__(256) void lru_place_kernel(LruArgs a) {
  const int tick = a.st->lru_tick;
  for (int l = 0; l < a.n_lists; ++l) {
    const int n = a.st->n_miss[l];
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
      lru_place(a, a.miss_list[l][j], tick, [](int, int) {});
  }
}

// Placement and copy in one launch, for an insertion whose end nobody waits for half-way (on the caller's stream): the
// first kLruTile threads of a block each serve a miss, the block copies the rows they granted (at most 64 ways each).  A
// tile this small makes some hundred blocks of a few thousand misses, whose serial walks overlap.  Rows of 16 bytes and
// more, as in gather_rows_flat_kernel.
constexpr int kLruTile = 32;
static __global__ __launch_bounds__(256) void lru_place_copy_kernel(LruArgs a, const uint8_t *rows, uint8_t *cache,
                                                                    int64_t row_bytes) {
  __shared__ int2 s_row[kLruTile * 64];
  __shared__ int s_n;
  const int tick = a.st->lru_tick;
  const int upr = (int)((row_bytes + 15) / 16);
  const int n = a.st->n_miss[0];
  for (int j0 = blockIdx.x * kLruTile; j0 < n; j0 += gridDim.x * kLruTile) {
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    if ((int)threadIdx.x < kLruTile && j0 + (int)threadIdx.x < n)
      lru_place(a, a.miss_list[0][j0 + threadIdx.x], tick,
                [&](int row, int slot) { s_row[atomicAdd(&s_n, 1)] = make_int2(row, slot); });
    __syncthreads();
    const int units = s_n * upr;
    for (int f = threadIdx.x; f < units; f += 256) {
      const int2 r = s_row[f / upr];
      const int u = f % upr;
      const int64_t off = u == upr - 1 ? row_bytes - 16 : 16 * u;
      *reinterpret_cast<u32x4_a4 *>(cache + r.y * row_bytes + off) =
          *reinterpret_cast<const u32x4_a4 *>(rows + r.x * row_bytes + off);
    }
    __syncthreads();
  }
}

int launch_lru_insert(Server *s, Pipe &p, hipStream_t st, int n_lists, hipEvent_t end) {
  if (s->cache_kind != LMI_CACHE_LRU) return LMI_OK;
  LruArgs a{};
  a.ids = p.ids;
  for (int l = 0; l < n_lists; ++l) a.miss_list[l] = p.miss_list + miss_list_base(s, l);
  a.st = p.st;
  a.n_lists = n_lists;
  a.keys = s->lru_keys;
  a.use = s->lru_use;
  a.fill = p.lru_fill;
  a.next = p.lru_next;
  a.head = s->lru_head;
  a.sets = s->lru_sets;
  a.ways = s->lru_ways;
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(s->max_nodes, 256), (int64_t)s->n_cu * 4));
  if (!p.lru_chained) hipLaunchKernelGGL(lru_chain_kernel, dim3(grid), dim3(256), 0, st, a, lru_sets(s));
  p.lru_chained = false;
  if (n_lists == 1 && st != s->side && s->row_bytes >= 16) {
    const int tiles = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(s->max_nodes, kLruTile), (int64_t)s->n_cu * 8));
    s->lru_keyed = s->lru_done = end ? end : s->lru_ready;
    hipExtLaunchKernelGGL(lru_place_copy_kernel, dim3(tiles), dim3(256), 0, st, nullptr, s->lru_done, 0, a,
                          (const uint8_t *)p.features, s->cache_data, s->row_bytes);
    LMI_HIP(hipGetLastError());
    ++s->routes.lru_place_copies;
    s->lru_pending = s->lru_copy_pending = true;
    s->lru_stream = st;
    return LMI_OK;
  }
  s->lru_keyed = s->lru_ready;
  s->lru_done = end ? end : s->lru_copied;
  // The events are the kernels' own completions: recorded behind them they were packets of their own and cost 6 us each.
  // keys and ticks are final: the next batch's lookup may start while the rows are still copied
  hipExtLaunchKernelGGL(lru_place_kernel, dim3(grid), dim3(256), 0, st, nullptr, s->lru_ready, 0, a);
  LMI_HIP(hipGetLastError());
  s->lru_pending = true;
  s->lru_stream = st;
  // copy the granted rows from the output buffer (already gathered) into the cache
  for (int l = 0; l < n_lists; ++l) {
    MoveArgs m{};
    m.g.n = 1;
    MoveRow &r = m.g.p[0];
    r.list = p.miss_list + miss_list_base(s, l);
    r.n_ptr = &p.st->n_miss[l];
    r.src_index = nullptr;
    m.src_from_list = 0;
    r.dst_index = p.lru_fill;
    m.src = (const uint8_t *)p.features;
    r.dst = s->cache_data;
    m.src_row_bytes = m.dst_row_bytes = m.row_bytes = s->row_bytes;
    m.n_max = s->node_cap[s->cfg.hops];
    if (l == n_lists - 1) m.ev_stop = s->lru_done;
    LMI_TRY(launch_move_rows(s, st, m, false));
  }
  s->lru_copy_pending = true;
  return LMI_OK;
}

// The LRU state is batch-synchronous: a lookup sees the cache after the previous batch's
// insertion.  Sampling does not touch the cache, so only the lookup has to wait.  The event is asked for also where the
// insertion ran on a stream of the same handle: that stream may be gone and the handle another stream's by now, and on
// the stream itself the wait costs nothing.
int lru_wait_ready(Server *s, hipStream_t st) {
  if (s->cache_kind != LMI_CACHE_LRU || !s->lru_pending) return LMI_OK;
  if (hipEventQuery(s->lru_keyed) == hipSuccess) {
    s->lru_pending = false;
    return LMI_OK;
  }
  (void)hipGetLastError();  // "not ready" is an answer, not a failure
  LMI_HIP(hipStreamWaitEvent(st, s->lru_keyed, 0));
  return LMI_OK;
}

// The rows the previous batch's insertion granted must be in the cache before a gather reads it.
int lru_wait_copied(Server *s, hipStream_t st) {
  if (s->cache_kind != LMI_CACHE_LRU || !s->lru_copy_pending) return LMI_OK;
  if (hipEventQuery(s->lru_done) == hipSuccess) {
    s->lru_copy_pending = false;
    return LMI_OK;
  }
  (void)hipGetLastError();
  LMI_HIP(hipStreamWaitEvent(st, s->lru_done, 0));
  return LMI_OK;
}

// -------------------------------------------------------- static cache build
// Ranking key of a node: its out-degree, or how often presampling touched it.
__device__ __forceinline__ int64_t rank_key(const int64_t *indptr, const uint32_t *hot, int64_t v) {
  return hot ? (int64_t)hot[v] : indptr[v + 1] - indptr[v];
}

// Presampling hotness (reference: HotnessMeasure, cache/cache_impl.cuh:190-198): one
// count per appearance of a node among a batch's sampled ids.
// Extra blocks finish a hop left pending.
static __global__ __launch_bounds__(256) void hotness_kernel(const int32_t *ids, const DevState *st, int64_t n_nodes,
                                                             uint32_t *hot, FillArgs fill, int fill_grid) {
  const int bx = (int)blockIdx.x - fill_grid, gx = (int)gridDim.x - fill_grid;
  if (bx < 0) {
    fill_local_ids(fill, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, (int64_t)fill_grid * blockDim.x);
    return;
  }
  const int n = st->node_counter[7];
  for (int i = bx * blockDim.x + threadIdx.x; i < n; i += gx * blockDim.x) {
    const int32_t v = ids[i];
    if (v >= 0 && v < n_nodes) atomicAdd(&hot[v], 1u);
  }
}

int launch_hotness(Server *s, Pipe &p, hipStream_t st) {
  if (!s->hot) {
    LMI_HIP(hipMalloc(&s->hot, (size_t)s->n_nodes * 4));
    LMI_HIP(hipMemsetAsync(s->hot, 0, (size_t)s->n_nodes * 4, st));
  }
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(s->max_nodes, 256), (int64_t)s->n_cu * 4));
  const int pending = p.fill_pending, extra = pending >= 0 ? fill_blocks(s->edge_cap[pending], 256) : 0;
  hipLaunchKernelGGL(hotness_kernel, dim3(grid + extra), dim3(256), 0, st, p.ids, p.st, s->n_nodes, s->hot,
                     fill_args(p, pending), extra);
  p.fill_pending = -1;
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// Histogram of the ranking keys in [lo, hi): bin (key - lo) >> shift, or with shift < 0 the key's bit length.  A block
// counts in LDS and adds its bins once: one same-address atomic per wavefront, as a count of the keys above a bound
// needs, took 190 us for 2.4 M nodes, this 12.
constexpr int kRankBins = 4096;
static __global__ __launch_bounds__(1024) void rank_histogram_kernel(const int64_t *indptr, const uint32_t *hot, int64_t n,
                                                                     int64_t lo, int64_t hi, int shift,
                                                                     unsigned long long *bins) {
  __shared__ unsigned int s_bin[kRankBins];
  for (int b = threadIdx.x; b < kRankBins; b += blockDim.x) s_bin[b] = 0;
  __syncthreads();
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const int64_t key = rank_key(indptr, hot, v);
    if (key < lo || key >= hi) continue;
    atomicAdd(&s_bin[shift < 0 ? (key == 0 ? 0 : 64 - __clzll(key)) : (int)((key - lo) >> shift)], 1u);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kRankBins; b += blockDim.x)
    if (s_bin[b]) atomicAdd(&bins[b], (unsigned long long)s_bin[b]);
}

// mode 0: cnt[v] = (deg == thr);  mode 1: cnt[v] = member flag using tie ranks.
static __global__ __launch_bounds__(kScanBlock) void member_flag_kernel(
    const int64_t *indptr, const uint32_t *hot, const int32_t *n_ptr, int64_t thr, int mode,
    const int32_t *tie_rank, int64_t ties_taken, int32_t *cnt, int32_t *tile_sums) {
  __shared__ int lds[kScanBlock / kWave];
  const int n = *n_ptr;
  const int n_tiles = (n + kScanTile - 1) / kScanTile;
  for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int base = tile * kScanTile + threadIdx.x * kScanItems;
    int sum = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
      const int v = base + j;
      if (v < n) {
        const int64_t d = rank_key(indptr, hot, v);
        int f;
        if (mode == 0) f = (d == thr);
        else f = (d > thr) || (d == thr && (int64_t)tie_rank[v] < ties_taken);
        cnt[v] = f;
        sum += f;
      }
    }
    tile_reduce_store(sum, tile_sums, tile, lds);
  }
}

// sums[0] += keys of the members, sums[1] += all keys: what share of the accesses, were they in proportion to the keys, the
// cache serves.  One pair of atomics a block.
static __global__ __launch_bounds__(1024) void key_mass_kernel(const int64_t *indptr, const uint32_t *hot, const int32_t *member,
                                                               int64_t n, unsigned long long *sums) {
  __shared__ unsigned long long s_sum[2];
  if (threadIdx.x < 2) s_sum[threadIdx.x] = 0;
  __syncthreads();
  unsigned long long in = 0, all = 0;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const unsigned long long key = (unsigned long long)rank_key(indptr, hot, v);
    all += key;
    if (member[v]) in += key;
  }
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) in += __shfl_xor(in, d, kWave), all += __shfl_xor(all, d, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    atomicAdd(&s_sum[0], in);
    atomicAdd(&s_sum[1], all);
  }
  __syncthreads();
  if (threadIdx.x < 2) atomicAdd(&sums[threadIdx.x], s_sum[threadIdx.x]);
}

static __global__ __launch_bounds__(256) void publish_slots_kernel(const int32_t *member, const int32_t *slot,
                                                                   int64_t n, int table_kind, HashSlot *slots,
                                                                   int log2cap, int32_t *slot_of,
                                                                   int32_t *cached_ids) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const bool m = member[v] != 0;
    if (table_kind == LMI_TABLE_DIRECT) slot_of[v] = m ? slot[v] : -1;
    if (m) {
      cached_ids[slot[v]] = (int32_t)v;
      if (table_kind == LMI_TABLE_HASH) {
        const uint32_t h = table_insert_min(slots, log2cap, (int32_t)v, slot[v]);
        (void)h;
      }
    }
  }
}

// One thread per 64-id word of the bitmap + rank table.
static __global__ __launch_bounds__(256) void publish_rank_kernel(const int32_t *member, const int32_t *slot,
                                                                  int64_t n, uint4 *tab) {
  const int64_t n_words = (n + 63) / 64;
  for (int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; w < n_words; w += (int64_t)gridDim.x * blockDim.x) {
    uint64_t bits = 0;
    const int64_t v0 = w * 64;
    for (int b = 0; b < 64 && v0 + b < n; ++b)
      if (member[v0 + b]) bits |= 1ull << b;
    tab[w] = make_uint4((uint32_t)bits, (uint32_t)(bits >> 32), (uint32_t)slot[v0], 0u);
  }
}

static __global__ void fill_i32_kernel(int32_t *p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

static __global__ void fill_slots_kernel(HashSlot *p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = HashSlot{kEmptyKey, kIntMax};
}

int launch_table_clear(Table &t, hipStream_t st) {
  const int64_t n = int64_t(1) << t.log2cap;
  hipLaunchKernelGGL(fill_slots_kernel, dim3((int)std::min<int64_t>(ceil_div(n, 256), 4096)), dim3(256), 0, st,
                     t.slots, n);
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

// No cache any more, and no batch in flight that still reads it; its buffers stay for the build that follows.
static void cache_drop(Server *s) {
  (void)hipDeviceSynchronize();  // batches in flight (side stream included) still read the old cache
  s->lru_pending = s->lru_copy_pending = false;
  if (s->lru_keys) (void)hipFree(s->lru_keys);  // one allocation: lru_use points into it
  if (s->lru_head) (void)hipFree(s->lru_head);
  s->lru_keys = s->lru_use = s->lru_head = nullptr;
  s->cache_kind = LMI_CACHE_NONE;
  s->cache_rows = 0;
}

void cache_free(Server *s) {
  cache_drop(s);
  if (s->cache_data) (void)hipFree(s->cache_data);
  if (s->cache_scale) (void)hipFree(s->cache_scale);
  if (s->id_table.slots) (void)hipFree(s->id_table.slots);
  if (s->slot_of) (void)hipFree(s->slot_of);
  if (s->rank_tab) (void)hipFree(s->rank_tab);
  s->cache_data = nullptr;
  s->cache_scale = nullptr;
  s->id_table = Table{};
  s->slot_of = nullptr;
  s->rank_tab = nullptr;
  if (s->build_scratch) (void)hipFree(s->build_scratch);
  s->build_scratch = nullptr;
  s->build_scratch_bytes = 0;
  for (size_t &b : s->cache_buf) b = 0;
}

// The largest key `thr` that at least `cap` nodes (1 <= cap <= nodes) reach, and how many lie above it: the octave of
// keys first, then 4096 bins at a time of what is left (two passes for keys below 8192).
static int rank_threshold(const Server *s, int64_t cap, unsigned long long *d_bins, int64_t *thr, int64_t *above) {
  std::vector<unsigned long long> bins(kRankBins);
  int64_t lo = 0, size = INT64_MAX;
  int shift = -1;
  *above = 0;
  while (true) {
    LMI_HIP(hipMemsetAsync(d_bins, 0, kRankBins * 8, 0));
    hipLaunchKernelGGL(rank_histogram_kernel, dim3(s->n_cu), dim3(1024), 0, 0, s->indptr,
                       s->policy == LMI_POLICY_PRESAMPLED ? s->hot : nullptr, s->n_nodes, lo,
                       size == INT64_MAX ? size : lo + size, shift, d_bins);
    LMI_HIP(hipGetLastError());
    LMI_HIP(hipMemcpy(bins.data(), d_bins, kRankBins * 8, hipMemcpyDeviceToHost));
    int b = kRankBins - 1;
    for (; b > 0 && *above + (int64_t)bins[b] < cap; --b) *above += (int64_t)bins[b];
    if (shift < 0) {
      lo = b == 0 ? 0 : int64_t(1) << (b - 1);  // bit length b: keys [2^(b-1), 2^b)
      size = b == 0 ? 1 : lo;
    } else {
      lo += (int64_t)b << shift;
      size = int64_t(1) << shift;
    }
    if (size == 1) break;
    shift = 0;
    while ((size >> shift) > kRankBins) ++shift;
  }
  *thr = lo;
  return LMI_OK;
}

// A buffer of the cache: kept when it has the size already (a cache that is built again), else allocated.
static int cache_buffer(void **p, size_t *have, size_t want) {
  if (*p && *have == want) return LMI_OK;
  if (*p) (void)hipFree(*p);
  *p = nullptr;
  *have = 0;
  if (want == 0) return LMI_OK;
  LMI_HIP(hipMalloc(p, want));
  *have = want;
  return LMI_OK;
}

// Hot set = first `capacity_rows` nodes under (out-degree desc, id asc):
// everything above the threshold degree plus the lowest-id ties at the threshold.
// slot(v) = number of cached nodes with a smaller id.
int cache_build_static(Server *s, int64_t capacity_rows, int table_kind, bool int8) {
  if (!s->indptr || !s->feat) LMI_FAIL(LMI_ERR_STATE, "load the graph and attach features before building a cache");
  if (table_kind != LMI_TABLE_HASH && table_kind != LMI_TABLE_DIRECT && table_kind != LMI_TABLE_RANK)
    LMI_FAIL(LMI_ERR_ARG, "bad table kind");
  if (s->n_nodes >= (int64_t(1) << 31) - kScanTile) LMI_FAIL(LMI_ERR_CAPACITY, "too many nodes");
  cache_drop(s);
  const int64_t N = s->n_nodes;
  const int64_t cap = std::max<int64_t>(0, std::min(capacity_rows, N));
  s->table_kind = table_kind;
  s->cache_row_bytes = int8 ? s->cfg.feat_dim : s->row_bytes;
  const bool presampled = s->policy == LMI_POLICY_PRESAMPLED;
  int lg = 4;
  while ((int64_t(1) << lg) < 2 * cap) ++lg;
  if (cap == 0 || (presampled && !s->hot) || (table_kind == LMI_TABLE_HASH && lg > 31)) {
    cache_free(s);
    if (cap == 0) LMI_FAIL(LMI_ERR_ARG, "cache capacity must be at least one row");
    if (presampled && !s->hot)
      LMI_FAIL(LMI_ERR_STATE, "the presampled policy needs lmi_presample (or presampling operators) first");
    LMI_FAIL(LMI_ERR_CAPACITY, "cache too large for the hash table");
  }
  const uint32_t *hot_key = presampled ? s->hot : nullptr;
  // What the cache before had in another size goes first, so that the two never lie in memory together.  (Taking
  // 40 MB of scratch anew costs a build 0.5 ms.)
  const size_t want[kCacheBufs] = {(size_t)cap * s->cache_row_bytes, int8 ? (size_t)cap * 4 : 0,
                                   table_kind == LMI_TABLE_HASH ? size_t(8) << lg : 0,
                                   table_kind == LMI_TABLE_DIRECT ? (size_t)N * 4 : 0,
                                   table_kind == LMI_TABLE_RANK ? (size_t)ceil_div(N, 64) * 16 : 0};
  void **const buf[kCacheBufs] = {(void **)&s->cache_data, (void **)&s->cache_scale, (void **)&s->id_table.slots,
                                  (void **)&s->slot_of, (void **)&s->rank_tab};
  for (int k = 0; k < kCacheBufs; ++k)
    if (s->cache_buf[k] != want[k]) LMI_TRY(cache_buffer(buf[k], &s->cache_buf[k], 0));

  // build-time scratch in one allocation: released on every return path, or kept for the next build when it is small
  struct Scratch {
    Server *s;
    uint8_t *base = nullptr;
    size_t bytes = 0;
    ~Scratch() {
      if (s->build_scratch_bytes > kKeepBuildScratch) {
        (void)hipFree(s->build_scratch);
        s->build_scratch = nullptr;
        s->build_scratch_bytes = 0;
      }
    }
    size_t take(size_t n) {
      const size_t at = bytes;
      bytes += (n + 255) / 256 * 256;
      return at;
    }
  } scratch{s};
  const size_t o_bins = scratch.take(kRankBins * 8), o_cnt = scratch.take((N + 1) * 4), o_tie = scratch.take((N + 1) * 4),
               o_slot = scratch.take((N + 1) * 4), o_tiles = scratch.take((ceil_div(N, kScanTile) + 1) * 4),
               o_n = scratch.take(24), o_cached = scratch.take(cap * 4);
  LMI_TRY(cache_buffer(&s->build_scratch, &s->build_scratch_bytes, scratch.bytes));
  scratch.base = (uint8_t *)s->build_scratch;
  unsigned long long *d_bins = (unsigned long long *)(scratch.base + o_bins);
  int32_t *d_cnt = (int32_t *)(scratch.base + o_cnt), *d_tie = (int32_t *)(scratch.base + o_tie),
          *d_slot = (int32_t *)(scratch.base + o_slot), *d_tiles = (int32_t *)(scratch.base + o_tiles),
          *d_n = (int32_t *)(scratch.base + o_n), *d_cached = (int32_t *)(scratch.base + o_cached);
  struct {  // at d_n: the nodes, the total of a scan, key_mass_kernel's sums
    int32_t n, total;
    unsigned long long mass[2];
  } counts = {(int32_t)N, 0, {0, 0}};
  static_assert(sizeof(counts) == 24, "o_n");
  LMI_HIP(hipMemcpy(d_n, &counts, sizeof(counts), hipMemcpyHostToDevice));

  int64_t thr = 0, above = 0;
  LMI_TRY(rank_threshold(s, cap, d_bins, &thr, &above));
  const int64_t ties_taken = cap - above;

  const int grid = scan_grid(N);
  hipLaunchKernelGGL(member_flag_kernel, dim3(grid), dim3(kScanBlock), 0, 0, s->indptr, hot_key, d_n, thr, 0, nullptr,
                     (int64_t)0, d_cnt, d_tiles);
  LMI_TRY(launch_scan_phases(0, d_cnt, d_tie, d_tiles, d_n, N, SCAN_EPI_NONE, nullptr, 0, d_n + 1));
  hipLaunchKernelGGL(member_flag_kernel, dim3(grid), dim3(kScanBlock), 0, 0, s->indptr, hot_key, d_n, thr, 1, d_tie,
                     ties_taken, d_cnt, d_tiles);
  LMI_TRY(launch_scan_phases(0, d_cnt, d_slot, d_tiles, d_n, N, SCAN_EPI_NONE, nullptr, 0, d_n + 1));
  if (!int8)  // int8 rows are not gathered in the hops, which is what asks for it
    hipLaunchKernelGGL(key_mass_kernel, dim3((int)std::min<int64_t>(s->n_cu, ceil_div(N, 1024))), dim3(1024), 0, 0, s->indptr,
                       hot_key, d_cnt, N, (unsigned long long *)(d_n + 2));
  LMI_HIP(hipMemcpy(&counts, d_n, sizeof(counts), hipMemcpyDeviceToHost));
  if (counts.total != cap)
    LMI_FAIL(LMI_ERR_HIP, "static cache selection picked %d rows, expected %lld", counts.total, (long long)cap);
  s->miss_share = counts.mass[1] ? 1.0 - (double)counts.mass[0] / (double)counts.mass[1] : 1.0 - (double)cap / (double)N;
  s->policy_built = s->policy;

  for (int k = 0; k < kCacheBufs; ++k) LMI_TRY(cache_buffer(buf[k], &s->cache_buf[k], want[k]));
  if (table_kind == LMI_TABLE_HASH) {
    s->id_table.log2cap = lg;
    LMI_TRY(launch_table_clear(s->id_table, 0));
  } else if (table_kind == LMI_TABLE_RANK) {
    hipLaunchKernelGGL(publish_rank_kernel, dim3(s->n_cu * 8), dim3(256), 0, 0, d_cnt, d_slot, N, s->rank_tab);
  }
  hipLaunchKernelGGL(publish_slots_kernel, dim3(s->n_cu * 8), dim3(256), 0, 0, d_cnt, d_slot, N, table_kind,
                     s->id_table.slots, s->id_table.log2cap, s->slot_of, d_cached);
  LMI_HIP(hipGetLastError());

  // rows
  int32_t cap32[2] = {(int32_t)cap, 0};
  LMI_HIP(hipMemcpy(d_n, cap32, 8, hipMemcpyHostToDevice));
  if (int8) {
#define LMI_QUANT(KEEP_)                                                                                              \
  hipLaunchKernelGGL(quantize_rows_kernel<KEEP_>, dim3(s->n_cu * 8), dim3(256), 0, 0, d_cached, cap, s->feat,          \
                     s->cfg.feat_dim, s->cfg.feat_dtype, s->row_bytes, (int8_t *)s->cache_data, s->cache_scale)
    if (s->cfg.feat_dim <= 4 * kWave) LMI_QUANT(4);
    else if (s->cfg.feat_dim <= 12 * kWave) LMI_QUANT(12);
    else if (s->cfg.feat_dim <= 24 * kWave) LMI_QUANT(24);
    else LMI_QUANT(0);
#undef LMI_QUANT
    LMI_HIP(hipGetLastError());
  } else {
    MoveArgs m{};
    m.g.n = 1;
    m.g.p[0].n_ptr = d_n;
    m.g.p[0].src_index = d_cached;
    m.g.p[0].dst = s->cache_data;
    m.src = s->feat;
    m.n_src = N;
    m.note_rows = -1;
    m.src_row_bytes = m.dst_row_bytes = m.row_bytes = s->row_bytes;
    m.n_max = cap;
    // Over the link a block per CU: more reads in flight cost it a few percent, except of rows so long that few of them are
    // (us a build on the device's grid / 256 blocks / 96: 735 000 rows of 400 bytes 6 778 / 6 574 / 6 476, of 512 6 985 / 6 785 /
    // 6 800; 1.2 M of 64 bytes 2 510 / 2 357 / 2 455; 160 000 of 3 072 8 980 / 8 744 / 8 998; 120 000 of 5 732 13 280 / 13 497 /
    // 14 075).
    if (s->feat_loc == LMI_LOC_HOST && s->row_bytes <= 4096) m.max_blocks = s->n_cu;
    LMI_TRY(launch_move_rows(s, 0, m, false));
  }
  LMI_HIP(hipDeviceSynchronize());
  s->cache_rows = cap;
  s->cache_kind = int8 ? LMI_CACHE_INT8 : LMI_CACHE_STATIC;
  return LMI_OK;
}

// Empty LRU records: key -1 and tick 0 in every way.
static __global__ __launch_bounds__(256) void lru_init_kernel(int32_t *rec, int64_t n_words, int ways) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_words; i += (int64_t)gridDim.x * blockDim.x)
    rec[i] = ((i / ways) & 1) ? 0 : -1;
}

int cache_build_lru(Server *s, int64_t n_sets, int32_t ways) {
  if (!s->feat) LMI_FAIL(LMI_ERR_STATE, "attach features before building a cache");
  if (n_sets < 1 || ways < 1 || ways > 64 || n_sets * ways >= (int64_t(1) << 31))
    LMI_FAIL(LMI_ERR_ARG, "bad LRU geometry (sets=%lld ways=%d)", (long long)n_sets, ways);
  cache_free(s);
  const int64_t rows = n_sets * ways;
  LMI_HIP(hipMalloc(&s->lru_keys, rows * 8));  // per set: `ways` keys, then `ways` ticks
  s->lru_use = s->lru_keys + ways;
  LMI_HIP(hipMalloc(&s->lru_head, n_sets * 4));
  LMI_TRY(cache_buffer((void **)&s->cache_data, &s->cache_buf[0], (size_t)rows * s->row_bytes));
  const int g = 2048;
  hipLaunchKernelGGL(lru_init_kernel, dim3(g), dim3(256), 0, 0, s->lru_keys, rows * 2, ways);
  hipLaunchKernelGGL(fill_i32_kernel, dim3(g), dim3(256), 0, 0, s->lru_head, n_sets, -1);
  LMI_HIP(hipDeviceSynchronize());
  s->lru_sets = n_sets;
  s->lru_ways = ways;
  s->lru_tick = 0;
  s->cache_rows = rows;
  s->cache_row_bytes = s->row_bytes;
  s->cache_kind = LMI_CACHE_LRU;
  return LMI_OK;
}

static __global__ void dump_static_kernel(SlotTable table, int64_t n, int32_t *out) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x)
    out[v] = static_find(table, (int32_t)v);
}

int cache_dump(Server *s, int32_t *slot_of, int64_t n, int32_t *aux) {
  if (s->cache_kind == LMI_CACHE_NONE) LMI_FAIL(LMI_ERR_STATE, "no cache built");
  LMI_HIP(hipDeviceSynchronize());
  if (s->cache_kind == LMI_CACHE_LRU) {
    if (n != s->cache_rows) LMI_FAIL(LMI_ERR_ARG, "LRU dump needs n == sets*ways");
    std::vector<int32_t> rec((size_t)n * 2);
    LMI_HIP(hipMemcpy(rec.data(), s->lru_keys, (size_t)n * 8, hipMemcpyDeviceToHost));
    const int64_t ways = s->lru_ways;
    for (int64_t slot = 0; slot < n; ++slot) {  // slot = set * ways + way
      const int64_t at = slot / ways * 2 * ways + slot % ways;
      slot_of[slot] = rec[at];
      if (aux) aux[slot] = rec[at + ways];
    }
    return LMI_OK;
  }
  if (n != s->n_nodes) LMI_FAIL(LMI_ERR_ARG, "dump needs n == n_nodes");
  // through the scratch of the build where that was kept
  const bool kept = s->build_scratch_bytes >= (size_t)n * 4;
  int32_t *d = (int32_t *)s->build_scratch;
  if (!kept) LMI_HIP(hipMalloc(&d, n * 4));
  hipLaunchKernelGGL(dump_static_kernel, dim3(s->n_cu * 4), dim3(256), 0, 0, slot_table(s), n, d);
  const hipError_t e = hipMemcpy(slot_of, d, n * 4, hipMemcpyDeviceToHost);
  if (!kept) (void)hipFree(d);
  LMI_HIP(e);
  return LMI_OK;
}

}  // namespace lmi
