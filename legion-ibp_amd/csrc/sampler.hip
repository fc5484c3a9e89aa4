// Seed staging and the per-hop sampling / dedup / relabel kernels.
//
// Reference semantics (Legion-IBP, sampling_server/src/engine/operator_impl.cu):
//   batch_generate :28-56    seeds become local ids 0..n-1 in batch order
//   random_sample  :178-302  hop k samples from ALL nodes known so far; a row with
//                            deg <= fanout is taken whole in CSR order; edges run
//                            neighbour -> node
//   construct_graph:304-317  edges relabelled to local ids
//   counter_update :58-91    16-int headers
// What differs on purpose: Philox4x32-10 keyed by (seed, hop, node, slot) with
// Floyd's without-replacement rule instead of a per-node default-seeded
// minstd_rand; an open-addressing hash table in HBM instead of an N-bit bitmap
// plus an N-entry position map; scans instead of atomics for placement, so the
// edge order is (node, slot) and local ids follow first occurrence in that order.
//
// A hop is one launch (hop_kernel): per-node output counts -> block-CSR row pointers, draws, edges, inserts of the sources
// into the dedup table, first occurrences -> ranks, ids[] and local ids of the new nodes, their cache lookup; for hop 0 it
// also stages the seeds.  What is left is the local id of every edge source = its table slot's value: inside a batch that
// rides in extra blocks of the next kernel (the next hop, or the gather); hop_fill_kernel does it alone.
// (Also available as three launches: hop_count_scan, hop_sample, hop_flag_scan.)
// Batches expected to be small go through one workgroup instead (small.hip).
#include <algorithm>

#include <hip/hip_ext.h>

#include "gather.hpp"
#include "scan.hpp"

namespace lmi {

struct HopShared {  // what the pipes of a launch have in common
  // graph
  const int64_t *indptr;
  const int32_t *indices;
  int64_t n_nodes;
  int fanout, hop, hops;
  int log2cap;      // dedup tables
  int max_tiles;
  int stage_seeds;  // hop 0 only: the seeds have not been staged by batch_generate_kernel yet
  int begin;        // hop 0 only: no batch_begin_kernel ran, the parameters are in HopArgs::bp and the state is set up here
  int tile_blocks;  // hop_kernel: blocks [0, tile_blocks) own tiles, the rest fill; hop_flag_scan: own edge tiles, the rest
                    // look the seeds up
  int node_cap;     // nodes a batch can know before the hop
  SeenWord *nodes_seen;  // pinned host memory: receives how many the batch `note_row` knew, and behind the last hop its rows
  int note_row;
  int note_total;        // (its rows: only then)
  int seed_tiles;   // hop_kernel: the first tiles stage 256 seeds each
  // cache lookup of the nodes the hop adds
  int look_mode, miss_seg;
  SlotTable cache;
  LruSets lru;  // LOOK_LRU
  // hop_kernel: its first blocks gather the rows that the batch knew before the hop and that no launch before gathered
  int gather_blocks, upr, last_off, rows_per_tile;
  int tile_rows;  // last hop: every tile gathers the rows it adds and fills in its edges' local ids, and the batch is complete
  RowSources rows;
};
struct HopArgs {
  DevState *st;
  int32_t *ids, *labels;
  int32_t *row_ptr;  // block CSR row pointers of this hop
  int32_t *agg_src_ids, *agg_src_off, *agg_dst_off;
  HashSlot *slots;
  int32_t *eslot;   // table slot per edge of this hop (| kKnownRepeat)
  unsigned long long *scan_words;
  FillArgs fill;    // the previous hop's last step, carried by hop_kernel (hop -1: none)
  BatchParams bp;   // HopShared::begin
  int32_t *cache_index;
  int2 *miss_list;
  int32_t *lru_fill, *lru_next;
  uint8_t *features;
  HeaderCopy headers;  // HopShared::tile_rows: where the headers go besides the state (nodes null: nowhere)
};

// Several mini-batches (pipes) can share every launch of the sampling phase: block b
// works on pipe b mod n (LMI_GRID_ROW).  The kernels are latency-bound, so a second batch
// in the same launch costs far less than a second launch.
constexpr int kMaxGroup = LMI_MAX_GROUP;
struct HopGroup {
  HopShared c;
  HopArgs p[kMaxGroup];
  int n;
};
static_assert(sizeof(HopGroup) <= 4096, "a kernel's arguments");
// A batch's parameters where the argument segment of a kernel whose first argument is a HopGroup holds them.  Read through
// this address space because a choice between them and the state's (HopShared::begin), were both behind ordinary pointers,
// may become a choice of pointers, for which the compiler copies all arguments to scratch memory (a hop took ten times as
// long).
typedef const __attribute__((address_space(4))) HopGroup ArgHopGroup;
typedef const __attribute__((address_space(4))) BatchParams ArgParams;
__device__ __forceinline__ ArgParams &arg_params(int row) {
  return ((ArgHopGroup *)__builtin_amdgcn_kernarg_segment_ptr())->p[row].bp;
}
struct FillGroup {
  FillArgs p[kMaxGroup];
  int n;
};
struct BeginPipe {
  HashSlot *slots;
  DevState *st;
  unsigned long long *scan_words;
  BatchParams bp;
};
struct BeginGroup {
  BeginPipe p[kMaxGroup];
  int n;
};

// ------------------------------------------------------------ batch start
// Clears the dedup table (key = -1, value = INT_MAX), resets the pipe state and
// the scan words, and stores the per-batch parameters where later kernels read them.  Most batches do without this
// launch (2-9 us): their table needs no wiping, scan words of earlier batches mean nothing, and the first hop's kernel can
// set up the state (HopShared::begin).
static __global__ __launch_bounds__(256) void batch_begin_kernel(BeginGroup g, int64_t n_slots, int hops,
                                                                 int max_tiles) {
  LMI_GRID_ROW(g.n);
  HashSlot *slots = g.p[row].slots;
  DevState *st = g.p[row].st;
  const BatchParams &bp = g.p[row].bp;
  const int64_t tid = (int64_t)bx * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gx * blockDim.x;
  // two slots (16 bytes) per store
  if (bp.clear_table) {
    const int4 fill = make_int4(kEmptyKey, kIntMax, kEmptyKey, kIntMax);
    int4 *p = reinterpret_cast<int4 *>(slots);
    for (int64_t i = tid; i < n_slots / 2; i += stride) p[i] = fill;
  }
  for (int64_t i = tid; i < (int64_t)kScanChains * max_tiles; i += stride) g.p[row].scan_words[i] = 0ull;
  if (tid == 0) {
    state_begin(st, bp, hops);
    misses_begin(st);
    st->scan_fault = st->bad_id = 0;
  }
}

// Stage the seeds on their own (operator-by-operator use, where the seeds' cache
// lookup runs before the first hop): ids[i] = seed, labels, table[seed] = min(i).
// `begin`: the table needs no wiping, and this launch sets the batch up too (hops >= 1), from its arguments.
static __global__ __launch_bounds__(256) void batch_generate_kernel(int64_t n_nodes, int32_t *ids, int32_t *labels,
                                                                    int log2cap, BeginPipe p, int begin, int hops) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const BatchParams &bp = p.bp;
  if (begin && i == 0) {
    state_begin(p.st, bp, hops);
    misses_begin(p.st);
  }
  if (i >= bp.n_seeds) return;
  const int32_t id = bp.seeds[i];
  ids[i] = id;
  labels[i] = bp.labels ? bp.labels[i] : -1;
  if (id < 0 || id >= n_nodes) {
    raise_fault(p.st, kFaultBadId, FaultTo{bp.serial, bp.fault});
    return;
  }
  table_insert_min(p.slots, log2cap, id, i, bp.table_tag, bp.table_mask);
}

// ------------------------------------------------------------- hop, phase 1
// row_ptr[i] = exclusive prefix of min(deg(ids[i]), fanout) over every node known
// so far; the total is the hop's edge count.  Hop 0 first stages the seeds:
// ids[i] = seed, labels, and table[seed] = min(i) so that a repeated seed resolves
// to its first row.
template <int ITEMS>
static __global__ __launch_bounds__(kScanBlock) void hop_count_scan_kernel(HopGroup g) {
  LMI_GRID_ROW(g.n);
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  constexpr int TILE = kScanBlock * ITEMS;
  __shared__ int lds[kScanBlock / kWave + 1];
  __shared__ int s_prefix;
  DevState *st = a.st;
  const FaultTo fault = fault_to(st);
  const ScanChain nodes = scan_chain(a.scan_words, g.c.max_tiles, 0);
  const uint32_t stamp = scan_stamp(fault.serial, g.c.hop);
  const int n = st->node_counter[9 + g.c.hop];
  const int n_tiles = (n + TILE - 1) / TILE;
  if (n_tiles == 0) {
    if (bx == 0 && threadIdx.x == 0) {
      a.row_ptr[0] = 0;
      scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, 0);
    }
    return;
  }
  const int tile = bx;
  if (tile < n_tiles) {
    const int base = tile * TILE + threadIdx.x * ITEMS;
    int32_t id[ITEMS];
    // 1. node ids (hop 0: stage the seeds)
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const int i = base + j;
      id[j] = -1;
      if (i < n) {
        if (g.c.stage_seeds) {
          id[j] = st->seeds[i];
          a.ids[i] = id[j];
          a.labels[i] = st->labels_in ? st->labels_in[i] : -1;
        } else {
          id[j] = a.ids[i];
        }
        if (id[j] < 0 || id[j] >= g.c.n_nodes) {
          if (g.c.stage_seeds) raise_fault(st, kFaultBadId, fault);
          id[j] = -1;
        }
      }
    }
    // 2. all row-pointer loads in flight together
    int64_t lo[ITEMS], hi[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      lo[j] = hi[j] = 0;
      if (id[j] >= 0) {
        lo[j] = g.c.indptr[id[j]];
        hi[j] = g.c.indptr[id[j] + 1];
      }
    }
    if (g.c.stage_seeds) {
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
        if (id[j] >= 0) table_insert_min(a.slots, g.c.log2cap, id[j], base + j, st->table_tag, st->table_mask);
    }
    int v[ITEMS], sum = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const int64_t deg = hi[j] - lo[j];
      v[j] = (int)(deg < (int64_t)g.c.fanout ? deg : (int64_t)g.c.fanout);
      sum += v[j];
    }
    int total;
    const int ex = block_exclusive_scan<kScanBlock>(sum, lds, total);
    if (threadIdx.x == 0) scan_tile_announce(nodes, stamp, tile, total);
    const int prefix = scan_tile_prefix(nodes, stamp, tile, total, &s_prefix, st, fault);
    if (prefix == kScanFaultPrefix) return;  // the whole block: no offset, no writes
    int run = prefix + ex;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (base + j < n) a.row_ptr[base + j] = run;
      run += v[j];
    }
    if (tile == n_tiles - 1 && threadIdx.x == 0) {
      a.row_ptr[n] = prefix + total;
      scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, prefix + total);
    }
  }
}

// ------------------------------------------------------------- hop, phase 2
// One group of G lanes per node, one lane per output slot.  Rows no longer than
// the fanout are copied whole; longer rows draw `fanout` distinct positions with
// Floyd's rule, the group resolving collisions slot by slot through shuffles.
// Every sampled edge is inserted into the dedup table with candidate value
// n_prev + e (e = edge index inside the hop); atomicMin keeps the first edge.
template <int G>
static __global__ __launch_bounds__(256) void hop_sample_kernel(HopGroup g) {
  LMI_GRID_ROW(g.n);
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  const DevState *st = a.st;
  const int64_t flat = (int64_t)bx * blockDim.x + threadIdx.x;
  const uint64_t seed = (uint64_t)st->rng_lo | ((uint64_t)st->rng_hi << 32);
  const int32_t tag = st->table_tag, tag_mask = st->table_mask;
  const int n_prev = st->node_counter[9 + g.c.hop];
  const int eoff = st->edge_counter[12 + g.c.hop + 1];
  const int fanout = g.c.fanout;
  const int lane = threadIdx.x & (G - 1);
  const int group = (int)(flat / G);
  const int n_groups = gx * blockDim.x / G;
  for (int i = group; i < n_prev; i += n_groups) {
    const int32_t v = a.ids[i];
    if (v < 0 || v >= g.c.n_nodes) continue;
    const int64_t beg = g.c.indptr[v];
    const int64_t deg = g.c.indptr[v + 1] - beg;
    const int base = a.row_ptr[i];
    int64_t pick = lane;
    int count;
    if (deg <= (int64_t)fanout) {
      count = (int)deg;
    } else {
      count = fanout;
      const uint32_t j = (uint32_t)(deg - fanout) + (uint32_t)lane;
      uint32_t t = 0xFFFFFFFFu;
      if (lane < fanout) t = __umulhi(sample_draw(seed, (uint32_t)g.c.hop, (uint32_t)v, (uint32_t)lane), j + 1u);
      pick = floyd_pick<G>(t, j, lane, fanout);
    }
    if (lane < count) {
      const int32_t nbr = g.c.indices[beg + pick];
      const int e = base + lane;
      a.agg_src_ids[eoff + e] = nbr;
      a.agg_dst_off[eoff + e] = i;
      a.eslot[e] = (int)table_insert_min(a.slots, g.c.log2cap, nbr, n_prev + e, tag, tag_mask);
    }
  }
}

// Variant with LDS-staged probes: the (up to 256) edges a block draws in one step are
// first deduplicated in a 512-entry LDS hash table; only the lowest edge of each
// distinct neighbour probes the HBM table, the other lanes copy its slot.  Same
// results (the HBM table still sees the minimum edge index per key).
template <int G>
static __global__ __launch_bounds__(256) void hop_sample_lds_kernel(HopGroup g) {
  LMI_GRID_ROW(g.n);
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  constexpr int TAB = 512;
  __shared__ int32_t lds_key[TAB];
  __shared__ int32_t lds_min[TAB];
  __shared__ int32_t lds_slot[TAB];
  const DevState *st = a.st;
  const int64_t flat = (int64_t)bx * blockDim.x + threadIdx.x;
  const uint64_t seed = (uint64_t)st->rng_lo | ((uint64_t)st->rng_hi << 32);
  const int n_prev = st->node_counter[9 + g.c.hop];
  const int eoff = st->edge_counter[12 + g.c.hop + 1];
  const int fanout = g.c.fanout;
  const int lane = threadIdx.x & (G - 1);
  const int group = (int)(flat / G);
  const int n_groups = gx * blockDim.x / G;
  const int groups_per_block = 256 / G;
  // uniform trip count per block: the block's first group decides
  for (int i0 = bx * groups_per_block; i0 < n_prev; i0 += n_groups) {
    const int i = i0 + (group - bx * groups_per_block);
    for (int t = threadIdx.x; t < TAB; t += 256) {
      lds_key[t] = kEmptyKey;
      lds_min[t] = kIntMax;
    }
    __syncthreads();
    bool active = false;
    int32_t nbr = -1;
    int e = 0, h = 0;
    if (i < n_prev) {
      const int32_t v = a.ids[i];
      if (v >= 0 && v < g.c.n_nodes) {
        const int64_t beg = g.c.indptr[v];
        const int64_t deg = g.c.indptr[v + 1] - beg;
        const int base = a.row_ptr[i];
        int64_t pick = lane;
        int count;
        if (deg <= (int64_t)fanout) {
          count = (int)deg;
        } else {
          count = fanout;
          const uint32_t j = (uint32_t)(deg - fanout) + (uint32_t)lane;
          uint32_t t = 0xFFFFFFFFu;
          if (lane < fanout) t = __umulhi(sample_draw(seed, (uint32_t)g.c.hop, (uint32_t)v, (uint32_t)lane), j + 1u);
          pick = floyd_pick<G>(t, j, lane, fanout);
        }
        if (lane < count) {
          active = true;
          nbr = g.c.indices[beg + pick];
          e = base + lane;
          a.agg_src_ids[eoff + e] = nbr;
          a.agg_dst_off[eoff + e] = i;
          h = (int)(((uint32_t)nbr * 0x9E3779B1u) >> 23);  // 9 bits
          while (true) {
            const int32_t k = atomicCAS(&lds_key[h], kEmptyKey, nbr);
            if (k == kEmptyKey || k == nbr) break;
            h = (h + 1) & (TAB - 1);
          }
          atomicMin(&lds_min[h], e);
        }
      }
    }
    __syncthreads();
    if (active && lds_min[h] == e)
      lds_slot[h] = (int)table_insert_min(a.slots, g.c.log2cap, nbr, n_prev + e, st->table_tag, st->table_mask);
    __syncthreads();
    // an edge that lost inside the block is a repeat whatever the table said to the winner
    if (active) a.eslot[e] = (lds_min[h] == e) ? lds_slot[h] : (lds_slot[h] | (int32_t)kKnownRepeat);
    __syncthreads();
  }
}

__device__ __forceinline__ int32_t hop_lookup(const HopGroup &g, const HopArgs &a, int32_t id, int32_t lru_tick) {
  return g.c.look_mode == LOOK_LRU ? lru_find(g.c.lru, id, lru_tick) : static_find(g.c.cache, id);
}
// Cache lookup of the rows a block adds to the batch, ITEMS a thread (`look`): node, row, slot found.  In the kernels that add
// them because the id is in a register there and the random read of the cache's table hides behind the other tiles'
// look-back: as a kernel of its own the lookup was a launch and a pass over the ids: 30 us, its part of the last fill
// included, for a group of four papers100M-shaped batches.
template <int ITEMS, int BLOCK>
__device__ __forceinline__ void rows_looked_up(const HopGroup &g, const HopArgs &a, bool seed_rows, const int32_t *node,
                                               const int32_t *local, const int32_t *slot_of, bool *look, int32_t tag,
                                               int32_t tag_mask, int *lds, int *lds_at) {
  int misses = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (look[j]) a.cache_index[local[j]] = slot_of[j];
    look[j] = look[j] && slot_of[j] < 0 && node[j] >= 0 && node[j] < g.c.n_nodes;  // from here on: a miss
    misses += look[j] ? 1 : 0;
  }
  if (g.c.look_mode == LOOK_LRU) {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (!look[j]) continue;
      // a repeated seed keeps both rows, but the id is offered for insertion once, by its first row
      const bool repeat = seed_rows && table_find<true>(a.slots, g.c.log2cap, node[j], tag, tag_mask) != local[j];
      a.lru_fill[local[j]] = repeat ? -2 : -1;
      if (!repeat) lru_chain(g.c.lru, a.lru_next, local[j], node[j]);
    }
  }
  if (g.c.look_mode >= LOOK_LIST) {  // one atomic per block: one per wavefront on the same counter costs 24 ns each
    int total;
    int at = block_exclusive_scan<BLOCK>(misses, lds, total);
    if (total == 0) return;
    if (threadIdx.x == 0) *lds_at = atomicAdd(&a.st->n_miss[g.c.miss_seg], total);
    __syncthreads();
    at += *lds_at;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (look[j]) a.miss_list[at++] = make_int2(local[j], node[j]);
  }
}

// Copies the headers, which the block has just left in the state, to where the caller wants them too.
__device__ __forceinline__ void headers_copy(const HopGroup &g, const HopArgs &a, int t) {
  if (!g.c.tile_rows || !a.headers.nodes) return;
  __syncthreads();
  if (t < 16) a.headers.nodes[t] = a.st->node_counter[t];
  else if (t < 32) a.headers.edges[t - 16] = a.st->edge_counter[t - 16];
}

// ------------------------------------------------------------- hop, one launch
// All of a hop by tiles of NPB nodes, G lanes per node: row pointers and counts (wavefront 0), draws and neighbour reads,
// inserts into the dedup table, the tile's edge offset (look-back), first occurrences and their ranks (look-back), ids and
// local ids, cache lookup.  An edge is a first occurrence iff no earlier edge and no known node has its source, which the
// tile can tell as soon as every EARLIER tile has inserted its edges -- later ones hold larger candidates.  So a tile
// announces its edge count only when its inserts are complete, and the look-back over the counts is that wait too: like the
// other one it needs no block that has not been dispatched.  The candidates themselves need no offset: i * fanout + slot
// grows like the edge's index does.  The first hop's seeds, which come before all edges, are staged by tiles of their own
// ahead of the others (HopShared::seed_tiles).  What tiles tell each other inside the launch -- table slots, scan words, the
// miss count -- goes through device-scope atomics, which all dies see alike; wait_memory stands between a tile's inserts and
// its word.
// Bound by latency: eight dependent reads and two look-backs in a row (800 seeds, 25,10: 13 and 17 us for the two hops), and
// by random accesses where a hop has 10^5 edges.  As two launches (sampling, then the flags from the edges' slots in memory)
// a hop paid a launch and three dependent reads more.  us a pass, two launches per hop / one: 800 seeds, 25,10, a third of
// the rows cached 110.6 / 102.4; 8 000 seeds, all rows cached 80.9 / 73.7; four such batches from a table in HBM 303 / 290;
// 1 024 seeds, 15,10,5, four batches in a row through the LRU cache 350 / 298.
// Rows (early_rows, tile_rows say when): blocks ahead of the tiles gather what was known before the hop, the last hop's tiles
// what they add, and those then fill in their edges' local ids behind a third look-back, for tiles whose rows are published:
// the batch ends with the hop.  The first of the two cases above is bound by 2.9 MB over the host link (70 us): 102.4 us with
// a gather of its own, 94.9 with early rows, 89.5 with both.
// 64 registers and 96 scalar ones at most, so that two blocks of 1024 threads share a CU: the last tiles of a hop otherwise
// waited for the first to end.
template <int G, int BLOCK, int PASSES>
static __global__ __launch_bounds__(BLOCK, 8) void hop_kernel(HopGroup g) {
  const GridRow grid = grid_row(blockIdx.x, (unsigned)g.n);
  const int row = grid.row, bx = grid.bx - g.c.gather_blocks, gx = (int)(gridDim.x / (unsigned)g.n) - g.c.gather_blocks;
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  constexpr int PER_PASS = BLOCK / G, NPB = PER_PASS * PASSES, WAVES = BLOCK / kWave;
  static_assert(NPB <= BLOCK, "a thread per node");
  __shared__ int32_t s_id[NPB];
  __shared__ int64_t s_beg[NPB], s_deg[NPB];
  __shared__ int s_row[NPB];
  __shared__ int s_total, s_edge0, s_rank0, s_miss0, s_published, s_added;
  __shared__ int s_cnt[PASSES * WAVES];
  __shared__ int s_scan[WAVES + 1];
  __shared__ int s_slot[kSlotLds];
  DevState *st = a.st;
  if (bx >= g.c.tile_blocks) {  // extra blocks: the previous hop's local ids
    fill_local_ids(a.fill, (int64_t)(bx - g.c.tile_blocks) * blockDim.x + threadIdx.x,
                   (int64_t)(gx - g.c.tile_blocks) * blockDim.x);
    return;
  }
  if (bx < 0) {  // the blocks ahead of the tiles: rows known before this hop (early_rows)
    ArgParams &bp = arg_params(row);
    const bool first_hop = g.c.hop == 0;
    const int first = first_hop ? 0 : st->node_counter[9 + g.c.hop - 1];
    const int n = first_hop && g.c.begin ? bp.n_seeds : st->node_counter[9 + g.c.hop];
    const int32_t *ids = !first_hop ? a.ids : g.c.begin ? bp.seeds : st->seeds;
    gather_rows<u32x4_a4, BLOCK, 2, true, true>(g.c.rows, a.cache_index, ids, a.features, first, n, g.c.upr, g.c.last_off,
                                                g.c.rows_per_tile, g.c.rows.pitch, bx + g.c.gather_blocks, g.c.gather_blocks,
                                                first_hop, g.c.cache, nullptr, s_slot);
    return;
  }
  const int seed_tiles = g.c.seed_tiles;
  const int tile = bx, t = threadIdx.x;
  const int my = (tile - seed_tiles) * NPB + t;  // wavefront 0: the thread's node
  // a batch that starts here takes its parameters from the arguments (nobody in this launch may read the state that one
  // of its threads sets up), any other from the state
  const bool begin = g.c.begin != 0;
  ArgParams &bp = arg_params(row);
  int32_t id = -1;
  if (!g.c.stage_seeds && t < NPB && my < g.c.node_cap) id = a.ids[my];  // beside the state, not behind it
  const FaultTo fault = begin ? FaultTo{bp.serial, bp.fault} : fault_to(st);
  const int n_prev = begin ? bp.n_seeds : st->node_counter[9 + g.c.hop];
  const int n_tiles = seed_tiles + (n_prev + NPB - 1) / NPB;
  if (tile >= n_tiles) {
    if (n_tiles == 0 && tile == 0) {
      if (t == 0) {
        a.row_ptr[0] = 0;
        scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, 0);
        scan_epilogue(SCAN_EPI_HOP_NODES, st, g.c.hop, 0);
      }
      headers_copy(g, a, t);
    }
    return;
  }
  const bool last = tile == n_tiles - 1;
  if (begin && tile == 0 && t == 0) misses_begin(st);  // complete before any tile gets past this one's inserts
  const uint32_t stamp = scan_stamp(fault.serial, g.c.hop);
  const ScanChain edges = scan_chain(a.scan_words, g.c.max_tiles, 0), firsts = scan_chain(a.scan_words, g.c.max_tiles, 1),
                  published = scan_chain(a.scan_words, g.c.max_tiles, 2);
  const int32_t tag = begin ? bp.table_tag : st->table_tag, tag_mask = begin ? bp.table_mask : st->table_mask;
  const int32_t *seeds = g.c.stage_seeds ? (begin ? bp.seeds : st->seeds) : nullptr;
  const int look_mode = g.c.look_mode;
  int32_t node[PASSES], local[PASSES], slot_of[PASSES];
  bool look[PASSES];  // a row that the tile adds to the batch
#pragma unroll
  for (int u = 0; u < PASSES; ++u) node[u] = local[u] = slot_of[u] = -1, look[u] = false;

  if (tile < seed_tiles) {
    const int i = tile * BLOCK + t;
    if (t == 0) {
      scan_tile_announce(firsts, stamp, tile, 0);
      scan_tile_announce(published, stamp, tile, 0);
    }
    if (i < n_prev) {
      const int32_t *labels = begin ? bp.labels : st->labels_in;
      node[0] = seeds[i];
      local[0] = i;
      look[0] = true;
      a.ids[i] = node[0];
      a.labels[i] = labels ? labels[i] : -1;
      if (node[0] < 0 || node[0] >= g.c.n_nodes) raise_fault(st, kFaultBadId, fault);
      else table_insert_min(a.slots, g.c.log2cap, node[0], i, tag, tag_mask);
    }
    wait_memory();
    __syncthreads();
    if (t == 0) scan_tile_announce(edges, stamp, tile, 0);
    if (look_mode != LOOK_NOT && look[0] && node[0] >= 0 && node[0] < g.c.n_nodes)
      slot_of[0] = hop_lookup(g, a, node[0], begin ? bp.lru_tick : st->lru_tick);
    if (begin && tile == 0 && t == 0) state_params(st, bp);
    if (scan_tile_prefix(edges, stamp, tile, 0, &s_edge0, st, fault) == kScanFaultPrefix) return;
    if (last) {  // no seeds at all
      s_added = 0;
      if (t == 0) a.row_ptr[0] = 0;
      if (begin) {
        if (t < 32) headers_first_hop(st, t, g.c.hops, 0, 0, 0);
      } else if (t == 0) {
        scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, 0);
        scan_epilogue(SCAN_EPI_HOP_NODES, st, g.c.hop, 0);
      }
    }
  } else {
    // ---- counts
    if (seeds && t < NPB && my < n_prev) id = seeds[my];
    if (t >= NPB || my >= n_prev || id < 0 || id >= g.c.n_nodes) id = -1;
    int64_t lo = 0, hi = 0;
    if (id >= 0) {
      lo = g.c.indptr[id];
      hi = g.c.indptr[id + 1];
    }
    const int64_t deg = hi - lo;
    const int cnt = (int)(deg < (int64_t)g.c.fanout ? deg : (int64_t)g.c.fanout);
    if (t < NPB) {
      s_id[t] = id;
      s_beg[t] = lo;
      s_deg[t] = deg;
    }
    int ex, total;
    if constexpr (NPB <= kWave) {
      ex = wave_inclusive_scan(cnt) - cnt;
      if (t == kWave - 1) s_total = ex + cnt;
      if (t < NPB) s_row[t] = ex;
      __syncthreads();
      total = s_total;
    } else {
      ex = block_exclusive_scan<BLOCK>(cnt, s_scan, total);
      if (t < NPB) s_row[t] = ex;
      __syncthreads();
    }
    // ---- draws, neighbour reads, inserts
    const uint64_t seed = begin ? bp.rng_seed : (uint64_t)st->rng_lo | ((uint64_t)st->rng_hi << 32);
    // the edge offset of the hop is fixed by the hops before it
    const int eoff = (g.c.hop == 0) ? 0 : st->edge_counter[12 + g.c.hop] + st->edge_counter[9 + g.c.hop];
    const int fanout = g.c.fanout;
    const int lane = t & (G - 1);
    const int node0 = (tile - seed_tiles) * NPB + t / G;  // local id of the lane group's first node
    bool on[PASSES];
#pragma unroll
    for (int u = 0; u < PASSES; ++u) {
      const int q = t / G + u * PER_PASS;
      const int32_t v = s_id[q];  // -1 behind the last node
      const int64_t beg = s_beg[q], deg = s_deg[q];
      int64_t pick = lane;
      on[u] = v >= 0 && lane < fanout && (int64_t)lane < deg;
      if (deg > (int64_t)fanout) {
        const uint32_t j = (uint32_t)(deg - fanout) + (uint32_t)lane;
        uint32_t d = 0xFFFFFFFFu;
        if (lane < fanout) d = __umulhi(sample_draw(seed, (uint32_t)g.c.hop, (uint32_t)v, (uint32_t)lane), j + 1u);
        pick = floyd_pick<G>(d, j, lane, fanout);
      }
      if (on[u]) node[u] = g.c.indices[beg + pick];
    }
    uint32_t slot[PASSES];
#pragma unroll
    for (int u = 0; u < PASSES; ++u)
      slot[u] = on[u] ? table_insert_min(a.slots, g.c.log2cap, node[u], n_prev + (node0 + u * PER_PASS) * fanout + lane, tag, tag_mask)
                      : kKnownRepeat;
    wait_memory();
    __syncthreads();
    if (t == 0) scan_tile_announce(edges, stamp, tile, total);
    const int edge0 = scan_tile_prefix(edges, stamp, tile, total, &s_edge0, st, fault);
    if (edge0 == kScanFaultPrefix) return;  // the whole block: no offset, no writes
    // ---- first occurrences, in edge order: pass by pass, threads in order
    int32_t val[PASSES];
#pragma unroll
    for (int u = 0; u < PASSES; ++u)
      val[u] = (slot[u] & kKnownRepeat) ? -1 : __hip_atomic_load(&a.slots[slot[u]].val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint64_t m[PASSES];
#pragma unroll
    for (int u = 0; u < PASSES; ++u) {
      look[u] = !(slot[u] & kKnownRepeat) && val[u] == n_prev + (node0 + u * PER_PASS) * fanout + lane;
      m[u] = __ballot(look[u]);
      if ((t & (kWave - 1)) == 0) s_cnt[u * WAVES + t / kWave] = __popcll(m[u]);
    }
    __syncthreads();
    int added = 0;
    if constexpr (PASSES * WAVES <= 16) {
#pragma unroll
      for (int k = 0; k < PASSES * WAVES; ++k) {
        const int c = s_cnt[k];
        if (k % WAVES == t / kWave) local[k / WAVES] = added;
        added += c;
      }
    } else {  // at most a wavefront of counts: every wavefront scans them
      const int lane64 = t & (kWave - 1);
      const int c = lane64 < PASSES * WAVES ? s_cnt[lane64] : 0;
      const int inc = wave_inclusive_scan(c);
      added = __builtin_amdgcn_readlane(inc, kWave - 1);
#pragma unroll
      for (int u = 0; u < PASSES; ++u) local[u] = __shfl(inc - c, u * WAVES + t / kWave, kWave);
    }
    if (t == 0) scan_tile_announce(firsts, stamp, tile, added);
    // ---- edges, lookups
#pragma unroll
    for (int u = 0; u < PASSES; ++u) {
      if (look_mode != LOOK_NOT && look[u] && node[u] >= 0 && node[u] < g.c.n_nodes)
        slot_of[u] = hop_lookup(g, a, node[u], begin ? bp.lru_tick : st->lru_tick);
      if (!on[u]) continue;
      const int e = edge0 + s_row[t / G + u * PER_PASS] + lane;
      a.agg_src_ids[eoff + e] = node[u];
      a.agg_dst_off[eoff + e] = node0 + u * PER_PASS;
      if (!g.c.tile_rows) a.eslot[e] = (int)slot[u];
    }
    if (t < NPB && my < n_prev) a.row_ptr[my] = edge0 + ex;
    const int rank0 = scan_tile_prefix(firsts, stamp, tile, added, &s_rank0, st, fault);
    if (rank0 == kScanFaultPrefix) return;  // the whole block: no ranks
#pragma unroll
    for (int u = 0; u < PASSES; ++u) {
      local[u] += n_prev + rank0 + __popcll(m[u] & lanemask_lt());
      if (look[u]) {
        a.ids[local[u]] = node[u];
        // later edges of the same node compare this with their own, larger, candidates either way
        __hip_atomic_store(&a.slots[slot[u]].val, local[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (last) {
      s_added = rank0 + added;
      if (t == 0) a.row_ptr[n_prev] = edge0 + total;
      if (begin) {
        if (t < 32) headers_first_hop(st, t, g.c.hops, n_prev, edge0 + total, rank0 + added);
      } else if (t == 0) {
        scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, edge0 + total);
        scan_epilogue(SCAN_EPI_HOP_NODES, st, g.c.hop, rank0 + added);
      }
    }
    if (g.c.tile_rows) {
      if (look_mode != LOOK_NOT)
        rows_looked_up<PASSES, BLOCK>(g, a, false, node, local, slot_of, look, tag, tag_mask, s_scan, &s_miss0);
      wait_memory();
      __syncthreads();
      if (t == 0) scan_tile_announce(published, stamp, tile, 0);
      const int row0 = n_prev + rank0;
      gather_rows<u32x4_a4, BLOCK, PASSES == 1 ? 4 : 2, true, true>(g.c.rows, a.cache_index, a.ids, a.features, row0, row0 + added, g.c.upr,
                                                  g.c.last_off, added, g.c.rows.pitch, 0, 1, false, g.c.cache, nullptr,
                                                  s_slot);
      // the first occurrence of an edge's source lies in this tile or in an earlier one
      if (scan_tile_prefix(published, stamp, tile, 0, &s_published, st, fault) == kScanFaultPrefix) return;
#pragma unroll
      for (int u = 0; u < PASSES; ++u) {
        if (!on[u]) continue;
        const int e = edge0 + s_row[t / G + u * PER_PASS] + lane;
        a.agg_src_off[eoff + e] = __hip_atomic_load(&a.slots[slot[u] & ~kKnownRepeat].val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (last) headers_copy(g, a, t);
  if (t == 0 && row == g.c.note_row && g.c.nodes_seen) {  // for the host to shape later launches by
    const int n_seeds = g.c.hop == 0 ? n_prev : st->node_counter[9];
    if (g.c.note_total && last) note_seen(g.c.nodes_seen + 1, n_prev + s_added, n_seeds);
    if (tile == 0) note_seen(g.c.nodes_seen, n_prev, n_seeds);
  }
  if (look_mode != LOOK_NOT && !(g.c.tile_rows && tile >= seed_tiles))
    rows_looked_up<PASSES, BLOCK>(g, a, tile < seed_tiles, node, local, slot_of, look, tag, tag_mask, s_scan, &s_miss0);
}

// ------------------------------------------------------------- hop, step 2
// An edge is the first occurrence of a new node iff the table value of its source names
// the edge itself (n_prev + e).  Its rank among first occurrences (single-pass scan) is the
// node's place after the n_prev known nodes: the edge appends the node to ids[] and
// publishes the local id in the table.  Publishing while other tiles still read is safe: a
// later edge of the same node compares the value with its own, larger, index either way.
template <int ITEMS>
static __global__ __launch_bounds__(kScanBlock) void hop_flag_scan_kernel(HopGroup g) {
  LMI_GRID_ROW(g.n);
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  constexpr int TILE = kScanBlock * ITEMS;
  __shared__ int lds[kScanBlock / kWave + 1];
  __shared__ int s_prefix;
  DevState *st = a.st;
  int32_t local[ITEMS], node[ITEMS], slot_of[ITEMS];
  bool look[ITEMS];  // a row to look up
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) local[j] = node[j] = slot_of[j] = -1, look[j] = false;
  const int look_mode = g.c.look_mode;
  if (bx >= g.c.tile_blocks) {  // extra blocks: the seeds' lookup (ids[] holds them since the hop's first kernel)
    const int i = (bx - g.c.tile_blocks) * kScanBlock + (int)threadIdx.x;
    if (i < st->n_seeds) {
      node[0] = a.ids[i];
      local[0] = i;
      look[0] = true;
      if (look_mode != LOOK_NOT && node[0] >= 0 && node[0] < g.c.n_nodes) slot_of[0] = hop_lookup(g, a, node[0], st->lru_tick);
    }
  } else {
    const FaultTo fault = fault_to(st);
    const ScanChain edges = scan_chain(a.scan_words, g.c.max_tiles, 1);
    const uint32_t stamp = scan_stamp(fault.serial, g.c.hop);
    const int n_prev = st->node_counter[9 + g.c.hop];
    const int n = st->edge_counter[9 + g.c.hop + 1];
    const int eoff = st->edge_counter[12 + g.c.hop + 1];
    const int n_tiles = (n + TILE - 1) / TILE;
    if (n_tiles == 0 && bx == 0 && threadIdx.x == 0) scan_epilogue(SCAN_EPI_HOP_NODES, st, g.c.hop, 0);
    const int tile = bx;
    if (tile >= n_tiles) return;
    const int base = tile * TILE + threadIdx.x * ITEMS;
    int v[ITEMS], slot[ITEMS], sum = 0;
    // the source ids beside the slots, and the lookups ahead of the look-back: two reads less in a row
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const int e = base + j;
      int flag = 0;
      slot[j] = 0;
      if (e < n) {
        const int32_t es = a.eslot[e];  // sign bit = kKnownRepeat: no need to look
        slot[j] = es & (int32_t)~kKnownRepeat;
        if (es >= 0) {
          node[j] = a.agg_src_ids[eoff + e];
          flag = (a.slots[slot[j]].val == n_prev + e) ? 1 : 0;
        }
      }
      v[j] = flag;
      sum += flag;
    }
    int total;
    const int ex = block_exclusive_scan<kScanBlock>(sum, lds, total);
    if (threadIdx.x == 0) scan_tile_announce(edges, stamp, tile, total);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      look[j] = v[j] != 0;
      if (look_mode != LOOK_NOT && look[j] && node[j] >= 0 && node[j] < g.c.n_nodes)
        slot_of[j] = hop_lookup(g, a, node[j], st->lru_tick);
    }
    const int prefix = scan_tile_prefix(edges, stamp, tile, total, &s_prefix, st, fault);
    if (prefix == kScanFaultPrefix) return;  // the whole block: no ranks, no writes
    int run = n_prev + prefix + ex;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      local[j] = run;
      run += v[j];
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (look[j]) {
        a.ids[local[j]] = node[j];
        a.slots[slot[j]].val = local[j];
      }
    if (tile == n_tiles - 1 && threadIdx.x == 0) scan_epilogue(SCAN_EPI_HOP_NODES, st, g.c.hop, prefix + total);
  }
  if (look_mode != LOOK_NOT)
    rows_looked_up<ITEMS, kScanBlock>(g, a, bx >= g.c.tile_blocks, node, local, slot_of, look, st->table_tag, st->table_mask, lds, &s_prefix);
}

// ------------------------------------------------------------- hop, step 3
static __global__ __launch_bounds__(256) void hop_fill_kernel(FillGroup g) {
  LMI_GRID_ROW(g.n);
  const FillArgs &f = g.p[row];
  fill_local_ids(f, (int64_t)bx * blockDim.x + threadIdx.x, (int64_t)gx * blockDim.x);
}

// ---------------------------------------------------------------- launchers
SlotTable slot_table(const Server *s) {
  return SlotTable{s->cache_kind == LMI_CACHE_NONE ? -1 : s->table_kind, s->id_table.slots, s->id_table.log2cap, s->slot_of,
                   s->rank_tab};
}

LruSets lru_sets(const Server *s) { return LruSets{s->lru_keys, s->lru_use, s->lru_head, s->lru_sets, s->lru_ways}; }

static int begin_grid(const Pipe &p) {
  const int64_t n_slots = int64_t(1) << p.dedup.log2cap;
  return (int)std::min<int64_t>(ceil_div(n_slots / 2, 256), 2048);
}

static BeginGroup begin_group(Pipe *const *pp, const BatchParams *bps, int n) {
  BeginGroup g{};
  g.n = n;
  for (int k = 0; k < n; ++k) {
    g.p[k].slots = pp[k]->dedup.slots;
    g.p[k].st = pp[k]->st;
    g.p[k].scan_words = pp[k]->scan_words;
    g.p[k].bp = bps[k];
  }
  return g;
}

// First kernel of a batch for each of the n pipes (one launch); stage_seeds also stages the
// seeds in a kernel of their own (operator-by-operator use, one pipe).
int launch_batch_generate(Server *s, Pipe *const *pp, const BatchParams *bps, int n, hipStream_t st, bool stage_seeds) {
  Pipe &p0 = *pp[0];
  const int64_t n_slots = int64_t(1) << p0.dedup.log2cap;
  const BeginGroup g = begin_group(pp, bps, n);
  const bool together = stage_seeds && n == 1 && !bps[0].clear_table;  // 9.6 us as two launches, 4.5 as one
  if (!together)
    hipLaunchKernelGGL(batch_begin_kernel, dim3((begin_grid(p0)) * n), dim3(256), 0, st, g, n_slots, s->cfg.hops,
                       p0.max_tiles);
  if (stage_seeds) {
    for (int k = 0; k < n; ++k)
      hipLaunchKernelGGL(batch_generate_kernel, dim3((int)ceil_div(s->cfg.batch_size, 256)), dim3(256), 0, st, s->n_nodes, pp[k]->ids,
                         pp[k]->labels, pp[k]->dedup.log2cap, g.p[k], together ? 1 : 0, s->cfg.hops);
  }
  LMI_HIP(hipGetLastError());
  for (int k = 0; k < n; ++k) {
    pipe_seeds(s, *pp[k], bps[k].n_seeds);
    pp[k]->hops_done = 0;
    pp[k]->fill_pending = -1;
    pp[k]->table_in_lds = false;
  }
  return LMI_OK;
}

// Re-points the captured graph's first kernel at this batch's parameters.
int graph_update_begin(Server *s, Pipe &p, const BatchParams &bp) {
  Pipe *pp[1] = {&p};
  BeginGroup g = begin_group(pp, &bp, 1);
  int64_t n_slots = int64_t(1) << p.dedup.log2cap;
  int hops = s->cfg.hops;
  int max_tiles = p.max_tiles;
  void *args[4] = {&g, &n_slots, &hops, &max_tiles};
  hipKernelNodeParams kp{};
  kp.func = reinterpret_cast<void *>(batch_begin_kernel);
  kp.gridDim = dim3(begin_grid(p));
  kp.blockDim = dim3(256);
  kp.sharedMemBytes = 0;
  kp.kernelParams = args;
  kp.extra = nullptr;
  LMI_HIP(hipGraphExecKernelNodeSetParams(p.graph_exec, p.begin_node, &kp));
  pipe_seeds(s, p, bp.n_seeds);
  p.hops_done = s->cfg.hops;
  return LMI_OK;
}

// Only the fused first kernel of a hop can set the batch up.
bool hop_sets_up(const Server *s) { return s->fuse_count && !s->lds_dedup; }

// Which tile a hop of n batches takes.  Tiles wait for each other twice, each time the longer the more of them there are:
// as small as leaves one tile per CU, then several nodes per lane group, with the largest for what does not fit the device
// anyway.  us a pass by tile (threads x nodes per lane group) and the hop's tiles with it:
//   800 seeds, fanouts 25,10, second hop (7 068 nodes): 256x1 442 tiles 105.6, 512x1 221 102.8, 1024x1 111 104.1;
//   8 000 seeds, first hop: 256x1 1 000 83.5, 512x1 500 80.9, 1024x1 250 76.7, 512x4 125 82.8;
//   their second (31 700 nodes): 1024x1 496 79.6, 512x2 496 74.8, 512x4 248 73.7, 1024x4 124 76.8;
//   four such batches, second hop: 512x4 1 172 278.6, 1024x4 586 274.7, 256x4 2 344 285.4, 256x1 355.6;
//   1 024 seeds, 15,10,5, third hop (20 000 nodes): 256x1 625 295.3, 1024x1 157 281.6, 512x4 78 284.7.
// The nodes of a hop are in proportion to those that the last batches knew there; before the first, the graph's mean degree
// tells, 2 to 17 times too many on graphs of heavy-tailed degrees: its tiles are larger, and tile_rows decides on the same
// number (us a pass by that estimate and grids for the worst case, as a call captured on a new server keeps them / by what
// batches met: 800 seeds into the caller's buffers 111 / 103; 8 000 seeds, all rows cached 92 / 86; two launches a hop, which the
// worst case shaped, took 127 and 97).
static int64_t hop_nodes(const Server *s, int hop, int n_seeds) {
  const int64_t seen = hop > 0 && s->nodes_seen_host ? seen_count(&s->nodes_seen_host[hop], n_seeds) : 0;  // hop == hops: the batch's rows
  int64_t nodes = seen > 0 ? seen : n_seeds;
  const double mean = s->n_nodes > 0 ? (double)s->n_edges / (double)s->n_nodes : 0;
  for (int k = 0; k < hop && seen <= 0; ++k) nodes += (int64_t)((double)nodes * std::min<double>(mean, s->cfg.fanout[k]));
  return std::max<int64_t>(1, std::min(nodes, s->node_cap[hop]));
}
HopShape hop_shape(const Server *s, int n, int hop, int n_seeds, int G) {
  const int64_t nodes = hop_nodes(s, hop, n_seeds);
  constexpr HopShape kOnePass[] = {{256, 1}, {512, 1}, {1024, 1}}, kMore[] = {{512, 2}, {512, 4}};
  for (const HopShape &h : kOnePass)
    if (n * ceil_div(nodes, h.block / G) <= s->n_cu) return h;
  for (const HopShape &h : kMore)
    if (n * ceil_div(nodes, h.block / G * h.passes) <= 2 * s->n_cu) return h;
  return HopShape{1024, 4};
}

// One hop for each of the n pipes, all in the same launches (the pipes are in step: same hop,
// same pending fill).
int launch_hop(Server *s, Pipe *const *pp, int n, hipStream_t st, int hop, bool stage_seeds, bool defer_fill,
               const BatchParams *begin, HopLookup look) {
  const int f = s->cfg.fanout[hop];
  const int64_t n_max = s->node_cap[hop], e_max = s->edge_cap[hop];
  Pipe &p0 = *pp[0];
  HopGroup g{};
  g.n = n;
  g.c.indptr = s->indptr;
  g.c.indices = s->indices;
  g.c.n_nodes = s->n_nodes;
  g.c.fanout = f;
  g.c.hop = hop;
  g.c.hops = s->cfg.hops;
  g.c.log2cap = p0.dedup.log2cap;
  g.c.max_tiles = p0.max_tiles;
  g.c.node_cap = (int)n_max;
  g.c.stage_seeds = (hop == 0 && stage_seeds) ? 1 : 0;
  g.c.begin = begin ? 1 : 0;
  g.c.look_mode = look.mode;
  g.c.miss_seg = look.miss_seg;
  g.c.cache = slot_table(s);
  g.c.lru = lru_sets(s);
  for (int k = 0; k < n; ++k) {
    Pipe &p = *pp[k];
    HopArgs &a = g.p[k];
    a.st = p.st;
    a.ids = p.ids;
    a.labels = p.labels;
    a.row_ptr = p.blk_indptr[hop];
    a.agg_src_ids = p.agg_src_ids;
    a.agg_src_off = p.agg_src_off;
    a.agg_dst_off = p.agg_dst_off;
    a.slots = p.dedup.slots;
    a.eslot = p.eslot[hop & 1];
    a.scan_words = p.scan_words;
    a.fill.hop = -1;
    a.cache_index = p.cache_index;
    a.miss_list = p.miss_list + miss_list_base(s, look.miss_seg);
    a.lru_fill = p.lru_fill;
    a.lru_next = p.lru_next;
    a.features = (uint8_t *)p.features;
    if (look.mode == LOOK_LRU) p.lru_chained = true;
    if (begin) {
      a.bp = begin[k];
      pipe_seeds(s, p, begin[k].n_seeds);
      p.hops_done = 0;
      p.fill_pending = -1;
      p.table_in_lds = false;
    }
  }
  for (int k = 1; k < n; ++k)
    if (pp[k]->note_seeds > pp[g.c.note_row]->note_seeds) g.c.note_row = k;
  if (s->nodes_seen_dev && pp[g.c.note_row]->note_seeds > 0) g.c.nodes_seen = s->nodes_seen_dev + hop;
  int G = 4;
  while (G < f) G <<= 1;
  const bool fused = s->fuse_count && !s->lds_dedup;
  if (!fused) LMI_TRY(launch_fill(s, pp, n, st));
  if (fused) {
    // one tile of nodes per block; a hop left pending gets its local ids filled in by extra blocks behind the tile blocks
    const int n_seeds = most_seeds(pp, n);
    const HopShape shape = hop_shape(s, n, hop, n_seeds, G);
    const auto [block, passes] = shape;
    const int npb = block / G * passes;
    g.c.seed_tiles = g.c.stage_seeds ? (int)ceil_div(s->cfg.batch_size, block) : 0;
    g.c.tile_blocks = g.c.seed_tiles + (int)ceil_div(std::max<int64_t>(n_max, 1), npb);
    int grid = g.c.tile_blocks;
    if (p0.fill_pending >= 0) grid += fill_blocks(s->edge_cap[p0.fill_pending], block);
    if (look.early_rows) {
      g.c.rows = RowSources{s->cache_data, s->feat, (uint32_t)s->cache_rows, (uint32_t)s->n_nodes, s->row_bytes};
      g.c.upr = (int)((s->row_bytes + 15) / 16);
      g.c.last_off = (int)s->row_bytes - 16;
      g.c.rows_per_tile = flat_tile_rows(s->row_bytes) * (block / 256);
      g.c.gather_blocks = std::max(1, early_rows_blocks(s, n * hop_nodes(s, hop, n_seeds)) * 256 / block / n);
      grid += g.c.gather_blocks;
      const int64_t nodes = hop_nodes(s, hop, n_seeds);
      g.c.note_total = hop == s->cfg.hops - 1;
      g.c.tile_rows = hop == s->cfg.hops - 1 &&
                      tile_rows(s, n, std::max<int64_t>(1, hop_nodes(s, hop + 1, n_seeds) - nodes), ceil_div(nodes, npb), shape);
      for (int k = 0; k < n; ++k) {
        if (look.headers) g.p[k].headers = *look.headers;
        pp[k]->rows_done = g.c.tile_rows != 0;
      }
      if (hop == 0) s->row_routes.early_rows += n;
      if (g.c.tile_rows) s->row_routes.tile_rows += n;
    }
    s->row_routes.hop_threads[hop] = block;
    s->row_routes.hop_nodes[hop] = npb;
    const hipEvent_t end = g.c.tile_rows ? look.end : nullptr;
    for (int k = 0; k < n; ++k) {
      if (pp[k]->fill_pending >= 0) g.p[k].fill = fill_args(*pp[k], pp[k]->fill_pending);
      pp[k]->fill_pending = -1;
    }
#define LMI_HOP2(GG, BB, PP)                                                                                       \
  else if (block == BB && passes == PP) {                                                                          \
    if (end) hipExtLaunchKernelGGL((hop_kernel<GG, BB, PP>), dim3(grid * n), dim3(BB), 0, st, nullptr, end, 0, g); \
    else hipLaunchKernelGGL((hop_kernel<GG, BB, PP>), dim3(grid * n), dim3(BB), 0, st, g);                         \
  }
#define LMI_HOP(GG)                                                                                                         \
  if (false) {}                                                                                                             \
  LMI_HOP2(GG, 256, 1) LMI_HOP2(GG, 512, 1) LMI_HOP2(GG, 1024, 1) LMI_HOP2(GG, 512, 2) LMI_HOP2(GG, 512, 4) LMI_HOP2(GG, 1024, 4) \
  else LMI_FAIL(LMI_ERR_STATE, "no hop kernel of %d threads, %d passes", block, passes);
    switch (G) {
      case 4: LMI_HOP(4) break;
      case 8: LMI_HOP(8) break;
      case 16: LMI_HOP(16) break;
      case 32: LMI_HOP(32) break;
      default: LMI_HOP(64) break;
    }
#undef LMI_HOP
#undef LMI_HOP2
  } else {
    // one tile per block (blocks past the real item count leave at once); few items per
    // thread while that keeps the tile count near a thousand: the row-pointer reads are
    // dependent random accesses, so parallelism matters more than per-thread work
    const int64_t nm = std::max<int64_t>(n_max, 1);
    if (nm <= 256 * 1024)
      hipLaunchKernelGGL(hop_count_scan_kernel<1>, dim3(((int)ceil_div(nm, kScanBlock)) * n), dim3(kScanBlock), 0, st, g);
    else if (nm <= 512 * 1024)
      hipLaunchKernelGGL(hop_count_scan_kernel<2>, dim3(((int)ceil_div(nm, kScanBlock * 2)) * n), dim3(kScanBlock), 0, st, g);
    else if (nm <= 1024 * 1024)
      hipLaunchKernelGGL(hop_count_scan_kernel<4>, dim3(((int)ceil_div(nm, kScanBlock * 4)) * n), dim3(kScanBlock), 0, st, g);
    else
      hipLaunchKernelGGL(hop_count_scan_kernel<8>, dim3(((int)ceil_div(nm, kScanBlock * 8)) * n), dim3(kScanBlock), 0, st, g);
    const int grid = (int)std::min<int64_t>(ceil_div(n_max * G, 256), 8192);
    if (s->lds_dedup) {
      switch (G) {
        case 4: hipLaunchKernelGGL(hop_sample_lds_kernel<4>, dim3((grid) * n), dim3(256), 0, st, g); break;
        case 8: hipLaunchKernelGGL(hop_sample_lds_kernel<8>, dim3((grid) * n), dim3(256), 0, st, g); break;
        case 16: hipLaunchKernelGGL(hop_sample_lds_kernel<16>, dim3((grid) * n), dim3(256), 0, st, g); break;
        case 32: hipLaunchKernelGGL(hop_sample_lds_kernel<32>, dim3((grid) * n), dim3(256), 0, st, g); break;
        default: hipLaunchKernelGGL(hop_sample_lds_kernel<64>, dim3((grid) * n), dim3(256), 0, st, g); break;
      }
    } else {
      switch (G) {
        case 4: hipLaunchKernelGGL(hop_sample_kernel<4>, dim3((grid) * n), dim3(256), 0, st, g); break;
        case 8: hipLaunchKernelGGL(hop_sample_kernel<8>, dim3((grid) * n), dim3(256), 0, st, g); break;
        case 16: hipLaunchKernelGGL(hop_sample_kernel<16>, dim3((grid) * n), dim3(256), 0, st, g); break;
        case 32: hipLaunchKernelGGL(hop_sample_kernel<32>, dim3((grid) * n), dim3(256), 0, st, g); break;
        default: hipLaunchKernelGGL(hop_sample_kernel<64>, dim3((grid) * n), dim3(256), 0, st, g); break;
      }
    }
    const int64_t em = std::max<int64_t>(e_max, 1);
    const int seed_blocks = (hop == 0 && look.mode != LOOK_NOT) ? (int)ceil_div(s->cfg.batch_size, kScanBlock) : 0;
#define LMI_FLAG(I_)                                                                                                 \
    {                                                                                                                  \
      g.c.tile_blocks = (int)ceil_div(em, kScanBlock * I_);                                                            \
      hipLaunchKernelGGL(hop_flag_scan_kernel<I_>, dim3((g.c.tile_blocks + seed_blocks) * n), dim3(kScanBlock), 0, st, g); \
    }
    if (em <= 1024 * 1024) LMI_FLAG(2)
    else if (em <= 2560 * 1024) LMI_FLAG(4)
    else LMI_FLAG(8)
#undef LMI_FLAG
  }
  LMI_HIP(hipGetLastError());
  if (hop == 0 && look.mode != LOOK_NOT) (look.mode == LOOK_LRU ? s->routes.lru_scan_lookups : s->routes.scan_lookups) += n;
  for (int k = 0; k < n; ++k) {
    pp[k]->fill_pending = g.c.tile_rows ? -1 : hop;
    pp[k]->hops_done = hop + 1;
  }
  if (!defer_fill) LMI_TRY(launch_fill(s, pp, n, st));
  return LMI_OK;
}

FillArgs fill_args(const Pipe &p, int hop) {
  FillArgs f{};
  f.st = p.st;
  f.slots = p.dedup.slots;
  f.eslot = p.eslot[hop & 1];
  f.agg_src_off = p.agg_src_off;
  f.hop = hop;
  return f;
}

int fill_blocks(int64_t e_max, int block) {  // four edges per thread
  return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(e_max, (int64_t)block * 4), 1024));
}

int launch_fill(Server *s, Pipe *const *pp, int n, hipStream_t st) {
  const int hop = pp[0]->fill_pending;
  if (hop < 0) return LMI_OK;
  FillGroup g{};
  g.n = n;
  for (int k = 0; k < n; ++k) {
    g.p[k] = fill_args(*pp[k], hop);
    pp[k]->fill_pending = -1;
  }
  hipLaunchKernelGGL(hop_fill_kernel, dim3((fill_blocks(s->edge_cap[hop], 256)) * n), dim3(256), 0, st, g);
  LMI_HIP(hipGetLastError());
  return LMI_OK;
}

}  // namespace lmi
