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
// A hop is three steps:
//   1. hop_count_sample per-node output counts -> block-CSR row pointers (single-pass
//                       scan), draw positions, write edges, insert sources into the dedup
//                       table; for hop 0 it also stages the seeds.  (Also available as
//                       two kernels, hop_count_scan + hop_sample.)
//   2. hop_flag_scan    first-occurrence flags -> ranks (single-pass scan); first
//                       occurrences append their node to ids[] and publish its local id
//                       in the table; new node count.  The cache lookup of the appended
//                       nodes (hop 0: of the seeds too) rides along.
//   3. fill             local id of every edge source = its table slot's value.  Inside a
//                       batch this rides in extra blocks of the next kernel (the next
//                       hop's step 1, or the gather); hop_fill_kernel does it alone.
// Batches expected to be small go through one workgroup instead (small.hip).
#include <algorithm>

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
  int tile_blocks;  // hop_count_sample: blocks [0, tile_blocks) own node tiles, the rest fill; hop_flag_scan: own edge
                    // tiles, the rest look the seeds up
  // cache lookup of the nodes the hop adds (hop_flag_scan)
  int look_mode, miss_seg;
  SlotTable cache;
  LruSets lru;  // LOOK_LRU
};
struct HopArgs {
  DevState *st;
  int32_t *ids, *labels;
  int32_t *row_ptr;  // block CSR row pointers of this hop
  int32_t *agg_src_ids, *agg_dst_off;
  HashSlot *slots;
  int32_t *eslot;   // table slot per edge of this hop (| kKnownRepeat)
  ScanChain chain_nodes, chain_edges;
  FillArgs fill;    // the previous hop's last step, carried by hop_count_sample (hop -1: none)
  BatchParams bp;   // HopShared::begin
  int32_t *cache_index;
  int2 *miss_list;
  int32_t *lru_fill, *lru_next;
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
struct FillGroup {
  FillArgs p[kMaxGroup];
  int n;
};
struct BeginPipe {
  HashSlot *slots;
  DevState *st;
  ScanChain chain_nodes, chain_edges;
  BatchParams bp;
};
struct BeginGroup {
  BeginPipe p[kMaxGroup];
  int n;
};

// ------------------------------------------------------------ batch start
// Clears the dedup table (key = -1, value = INT_MAX), resets the pipe state and
// the scan chains, and stores the per-batch parameters where later kernels read them.  Most batches do without this
// launch (2-9 us): their table needs no wiping, the last flag scan of the batch before left chain_nodes clean, every
// hop's first kernel resets chain_edges, and the first hop's first kernel can set up the state (HopShared::begin).
static __global__ __launch_bounds__(256) void batch_begin_kernel(BeginGroup g, int64_t n_slots, int hops,
                                                                 int max_tiles) {
  LMI_GRID_ROW(g.n);
  HashSlot *slots = g.p[row].slots;
  DevState *st = g.p[row].st;
  const ScanChain chain_nodes = g.p[row].chain_nodes, chain_edges = g.p[row].chain_edges;
  const BatchParams &bp = g.p[row].bp;
  const int64_t tid = (int64_t)bx * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gx * blockDim.x;
  // two slots (16 bytes) per store
  if (bp.clear_table) {
    const int4 fill = make_int4(kEmptyKey, kIntMax, kEmptyKey, kIntMax);
    int4 *p = reinterpret_cast<int4 *>(slots);
    for (int64_t i = tid; i < n_slots / 2; i += stride) p[i] = fill;
  }
  scan_chain_reset(chain_nodes, max_tiles, tid, stride);
  scan_chain_reset(chain_edges, max_tiles, tid, stride);
  if (tid == 0) {
    state_begin(st, bp, hops);
    st->scan_fault = st->bad_id = 0;
  }
}

// Stage the seeds on their own (operator-by-operator use, where the seeds' cache
// lookup runs before the first hop): ids[i] = seed, labels, table[seed] = min(i).
// `begin`: the table needs no wiping, and this launch sets the batch up too (hops >= 1), from its arguments.
static __global__ __launch_bounds__(256) void batch_generate_kernel(int64_t n_nodes, int32_t *ids, int32_t *labels,
                                                                    int log2cap, BeginPipe p, int begin, int hops,
                                                                    int max_tiles) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const BatchParams &bp = p.bp;
  if (begin) {
    scan_chain_reset(p.chain_nodes, max_tiles, i, (int64_t)gridDim.x * blockDim.x);
    scan_chain_reset(p.chain_edges, max_tiles, i, (int64_t)gridDim.x * blockDim.x);
    if (i == 0) state_begin(p.st, bp, hops);
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
    if (threadIdx.x == 0) scan_tile_announce(a.chain_nodes, tile, total);
    const int prefix = scan_tile_prefix(a.chain_nodes, tile, total, &s_prefix, st, fault);
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
  scan_chain_reset(a.chain_edges, g.c.max_tiles, flat, (int64_t)gx * blockDim.x);
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
  scan_chain_reset(a.chain_edges, g.c.max_tiles, flat, (int64_t)gx * blockDim.x);
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

// ------------------------------------------------- hop, phases 1 and 2 in one launch
// One tile of NPB nodes per block.  Wavefront 0 loads the tile's row pointers, scans
// min(deg, fanout) across its lanes and obtains the tile's edge offset by look-back
// over the earlier tiles; then the whole block samples the tile's nodes, G lanes per
// node, from the row bounds kept in LDS.  Same outputs as hop_count_scan_kernel
// followed by hop_sample_kernel, one launch and one row-pointer read less.
template <int G, int NPB>
static __global__ __launch_bounds__(256) void hop_count_sample_kernel(HopGroup g) {
  LMI_GRID_ROW(g.n);
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  static_assert(NPB <= kWave && NPB >= 256 / G, "tile = one wavefront of nodes at most, one pass at least");
  __shared__ int32_t s_id[NPB];
  __shared__ int64_t s_beg[NPB], s_deg[NPB];
  __shared__ int s_row[NPB];
  __shared__ int s_prefix;
  DevState *st = a.st;
  const int64_t flat = (int64_t)bx * blockDim.x + threadIdx.x;
  scan_chain_reset(a.chain_edges, g.c.max_tiles, flat, (int64_t)gx * blockDim.x);
  if (bx >= g.c.tile_blocks) {  // extra blocks: the previous hop's local ids
    fill_local_ids(a.fill, (int64_t)(bx - g.c.tile_blocks) * blockDim.x + threadIdx.x,
                   (int64_t)(gx - g.c.tile_blocks) * blockDim.x);
    return;
  }
  // a batch that starts here takes its parameters from the arguments (nobody in this launch may read the state that one
  // of its threads sets up), any other from the state
  const bool begin = g.c.begin != 0;
  const BatchParams &bp = a.bp;
  const FaultTo fault = begin ? FaultTo{bp.serial, bp.fault} : fault_to(st);
  const int n_prev = begin ? bp.n_seeds : st->node_counter[9 + g.c.hop];
  const int n_tiles = (n_prev + NPB - 1) / NPB;
  if (n_tiles == 0) {
    if (bx == 0 && threadIdx.x == 0) {
      if (begin) state_begin(st, bp, g.c.hops);
      a.row_ptr[0] = 0;
      scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, 0);
    }
    return;
  }
  const int tile = bx;
  if (tile >= n_tiles) return;
  const int t = threadIdx.x;
  if (begin && tile == n_tiles - 1 && t == 0) state_begin(st, bp, g.c.hops);  // the thread that updates the headers below
  const int32_t tag = begin ? bp.table_tag : st->table_tag, tag_mask = begin ? bp.table_mask : st->table_mask;
  // ---- counts, tile scan (wavefront 0)
  const int my = tile * NPB + t;
  int cnt = 0, ex = 0, total = 0;
  int32_t id = -1;
  int64_t lo = 0, hi = 0;
  if (t < kWave) {
    if (t < NPB && my < n_prev) {
      if (g.c.stage_seeds) {
        const int32_t *labels = begin ? bp.labels : st->labels_in;
        id = (begin ? bp.seeds : st->seeds)[my];
        a.ids[my] = id;
        a.labels[my] = labels ? labels[my] : -1;
      } else {
        id = a.ids[my];
      }
      if (id < 0 || id >= g.c.n_nodes) {
        if (g.c.stage_seeds) raise_fault(st, kFaultBadId, fault);
        id = -1;
      }
    }
    if (id >= 0) {
      lo = g.c.indptr[id];
      hi = g.c.indptr[id + 1];
      if (g.c.stage_seeds) table_insert_min(a.slots, g.c.log2cap, id, my, tag, tag_mask);
    }
    const int64_t deg = hi - lo;
    cnt = (int)(deg < (int64_t)g.c.fanout ? deg : (int64_t)g.c.fanout);
    const int inc = wave_inclusive_scan(cnt);
    ex = inc - cnt;
    total = __shfl(inc, kWave - 1, kWave);
  }
  if (t == 0) scan_tile_announce(a.chain_nodes, tile, total);
  if (t < NPB) {
    s_id[t] = id;
    s_beg[t] = lo;
    s_deg[t] = hi - lo;
    s_row[t] = ex;
  }
  __syncthreads();
  // ---- sampling.  What is drawn depends on no other tile: the draws are made and the neighbour reads of up to PASSES
  // nodes per lane group are issued before the look-back, which hides behind them; only where the edges go needs it.
  const uint64_t seed = begin ? bp.rng_seed : (uint64_t)st->rng_lo | ((uint64_t)st->rng_hi << 32);
  // the edge offset of the hop is fixed by the hops before it
  const int eoff = (g.c.hop == 0) ? 0 : st->edge_counter[12 + g.c.hop] + st->edge_counter[9 + g.c.hop];
  const int fanout = g.c.fanout;
  const int lane = t & (G - 1);
  constexpr int PER_PASS = 256 / G, PASSES = NPB / PER_PASS < 4 ? NPB / PER_PASS : 4;
  int prefix = 0;
  for (int q0 = t / G; q0 < NPB; q0 += PER_PASS * PASSES) {
    int32_t nbr[PASSES];
    bool on[PASSES];
#pragma unroll
    for (int u = 0; u < PASSES; ++u) {
      const int q = q0 + u * PER_PASS;
      const int32_t v = s_id[q];  // -1 behind the last node
      const int64_t beg = s_beg[q], deg = s_deg[q];
      int64_t pick = lane;
      nbr[u] = -1;
      on[u] = v >= 0 && lane < fanout && (int64_t)lane < deg;
      if (deg > (int64_t)fanout) {
        const uint32_t j = (uint32_t)(deg - fanout) + (uint32_t)lane;
        uint32_t d = 0xFFFFFFFFu;
        if (lane < fanout) d = __umulhi(sample_draw(seed, (uint32_t)g.c.hop, (uint32_t)v, (uint32_t)lane), j + 1u);
        pick = floyd_pick<G>(d, j, lane, fanout);
      }
      if (on[u]) nbr[u] = g.c.indices[beg + pick];
    }
    if (q0 == t / G) {  // the first time round, all threads alike
      prefix = scan_tile_prefix(a.chain_nodes, tile, total, &s_prefix, st, fault);
      if (prefix == kScanFaultPrefix) return;  // the whole block: no offset, no writes
      if (t < NPB && my < n_prev) a.row_ptr[my] = prefix + ex;
      if (tile == n_tiles - 1 && t == 0) {
        a.row_ptr[n_prev] = prefix + total;
        scan_epilogue(SCAN_EPI_HOP_EDGES, st, g.c.hop, prefix + total);
      }
    }
#pragma unroll
    for (int u = 0; u < PASSES; ++u) {
      if (!on[u]) continue;
      const int q = q0 + u * PER_PASS;
      const int e = prefix + s_row[q] + lane;
      a.agg_src_ids[eoff + e] = nbr[u];
      a.agg_dst_off[eoff + e] = tile * NPB + q;
      a.eslot[e] = (int)table_insert_min(a.slots, g.c.log2cap, nbr[u], n_prev + e, tag, tag_mask);
    }
  }
}

// ------------------------------------------------------------- hop, step 2
// An edge is the first occurrence of a new node iff the table value of its source names
// the edge itself (n_prev + e).  Its rank among first occurrences (single-pass scan) is the
// node's place after the n_prev known nodes: the edge appends the node to ids[] and
// publishes the local id in the table.  Publishing while other tiles still read is safe: a
// later edge of the same node compares the value with its own, larger, index either way.
__device__ __forceinline__ int32_t hop_lookup(const HopGroup &g, const HopArgs &a, int32_t id) {
  return g.c.look_mode == LOOK_LRU ? lru_find(g.c.lru, id, a.st->lru_tick) : static_find(g.c.cache, id);
}
template <int ITEMS>
static __global__ __launch_bounds__(kScanBlock) void hop_flag_scan_kernel(HopGroup g) {
  LMI_GRID_ROW(g.n);
  const HopArgs &a = g.p[row];  // this block's pipe (mini-batch)
  constexpr int TILE = kScanBlock * ITEMS;
  __shared__ int lds[kScanBlock / kWave + 1];
  __shared__ int s_prefix;
  DevState *st = a.st;
  const int64_t flat = (int64_t)bx * blockDim.x + threadIdx.x;
  scan_chain_reset(a.chain_nodes, g.c.max_tiles, flat, (int64_t)gx * blockDim.x);  // for the next hop
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
      if (look_mode != LOOK_NOT && node[0] >= 0 && node[0] < g.c.n_nodes) slot_of[0] = hop_lookup(g, a, node[0]);
    }
  } else {
    const FaultTo fault = fault_to(st);
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
    if (threadIdx.x == 0) scan_tile_announce(a.chain_edges, tile, total);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      look[j] = v[j] != 0;
      if (look_mode != LOOK_NOT && look[j] && node[j] >= 0 && node[j] < g.c.n_nodes)
        slot_of[j] = hop_lookup(g, a, node[j]);
    }
    const int prefix = scan_tile_prefix(a.chain_edges, tile, total, &s_prefix, st, fault);
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
  // ---- cache lookup of the rows the block holds.  In this kernel because the id is in a register here and the random
  // read of the cache's table hides behind the other tiles' look-back: as a kernel of its own the lookup was a launch
  // and a pass over the ids: 30 us, its part of the last fill included, for a group of four papers100M-shaped
  // batches, whose flag scans did not get slower (31 + 12 us).
  if (look_mode == LOOK_NOT) return;
  int misses = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    if (look[j]) a.cache_index[local[j]] = slot_of[j];
    look[j] = look[j] && slot_of[j] < 0 && node[j] >= 0 && node[j] < g.c.n_nodes;  // from here on: a miss
    misses += look[j] ? 1 : 0;
  }
  if (look_mode == LOOK_LRU) {
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (!look[j]) continue;
      // a repeated seed keeps both rows, but the id is offered for insertion once, by its first row
      const bool repeat = bx >= g.c.tile_blocks &&
                          table_find(a.slots, g.c.log2cap, node[j], st->table_tag, st->table_mask) != local[j];
      a.lru_fill[local[j]] = repeat ? -2 : -1;
      if (!repeat) lru_chain(g.c.lru, a.lru_next, local[j], node[j]);
    }
  }
  if (look_mode >= LOOK_LIST) {  // one atomic per block: one per wavefront on the same counter costs 24 ns each
    int total;
    int at = block_exclusive_scan<kScanBlock>(misses, lds, total);
    if (total == 0) return;
    if (threadIdx.x == 0) s_prefix = atomicAdd(&st->n_miss[g.c.miss_seg], total);
    __syncthreads();
    at += s_prefix;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (look[j]) a.miss_list[at++] = make_int2(local[j], node[j]);
  }
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

static ScanChain chain_of(const Pipe &p, int which) { return ScanChain{p.chain_status[which]}; }

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
    g.p[k].chain_nodes = chain_of(*pp[k], 0);
    g.p[k].chain_edges = chain_of(*pp[k], 1);
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
    const int64_t threads = together ? std::max<int64_t>(s->cfg.batch_size, p0.max_tiles) : s->cfg.batch_size;
    for (int k = 0; k < n; ++k)
      hipLaunchKernelGGL(batch_generate_kernel, dim3((int)ceil_div(threads, 256)), dim3(256), 0, st, s->n_nodes, pp[k]->ids,
                         pp[k]->labels, pp[k]->dedup.log2cap, g.p[k], together ? 1 : 0, s->cfg.hops, p0.max_tiles);
  }
  LMI_HIP(hipGetLastError());
  for (int k = 0; k < n; ++k) {
    pp[k]->n_seeds = bps[k].n_seeds;
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
  p.n_seeds = bp.n_seeds;
  p.hops_done = s->cfg.hops;
  return LMI_OK;
}

// Only the fused first kernel of a hop can set the batch up.
bool hop_sets_up(const Server *s) { return s->fuse_count && !s->lds_dedup; }

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
    a.agg_dst_off = p.agg_dst_off;
    a.slots = p.dedup.slots;
    a.eslot = p.eslot[hop & 1];
    a.chain_nodes = chain_of(p, 0);
    a.chain_edges = chain_of(p, 1);
    a.fill.hop = -1;
    a.cache_index = p.cache_index;
    a.miss_list = p.miss_list + miss_list_base(s, look.miss_seg);
    a.lru_fill = p.lru_fill;
    a.lru_next = p.lru_next;
    if (look.mode == LOOK_LRU) p.lru_chained = true;
    if (begin) {
      a.bp = begin[k];
      p.n_seeds = begin[k].n_seeds;
      p.hops_done = 0;
      p.fill_pending = -1;
      p.table_in_lds = false;
    }
  }
  int G = 4;
  while (G < f) G <<= 1;
  const bool fused = s->fuse_count && !s->lds_dedup;
  if (!fused) LMI_TRY(launch_fill(s, pp, n, st));
  if (fused) {
    // counts, scan and sampling in one launch, one tile of nodes per block; a hop left
    // pending gets its local ids filled in by extra blocks behind the tile blocks
    const int npb = hop_tile_nodes(n_max, G, s->fuse_small_max);
    const int tile_blocks = (int)ceil_div(std::max<int64_t>(n_max, 1), npb);
    int grid = tile_blocks;
    if (p0.fill_pending >= 0) grid += fill_blocks(s->edge_cap[p0.fill_pending], 256);
    g.c.tile_blocks = tile_blocks;
    for (int k = 0; k < n; ++k) {
      if (pp[k]->fill_pending >= 0) g.p[k].fill = fill_args(*pp[k], pp[k]->fill_pending);
      pp[k]->fill_pending = -1;
    }
#define LMI_FUSED(GG)                                                                                   \
  if (npb == 64)                                                                                        \
    hipLaunchKernelGGL((hop_count_sample_kernel<GG, 64>), dim3((grid) * n), dim3(256), 0, st, g);          \
  else                                                                                                  \
    hipLaunchKernelGGL((hop_count_sample_kernel<GG, (256 / GG)>), dim3((grid) * n), dim3(256), 0, st, g);
    switch (G) {
      case 4: LMI_FUSED(4) break;
      case 8: LMI_FUSED(8) break;
      case 16: LMI_FUSED(16) break;
      case 32: LMI_FUSED(32) break;
      default: LMI_FUSED(64) break;
    }
#undef LMI_FUSED
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
  LMI_HIP(hipGetLastError());
  if (hop == 0 && look.mode != LOOK_NOT) (look.mode == LOOK_LRU ? s->routes.lru_scan_lookups : s->routes.scan_lookups) += n;
  for (int k = 0; k < n; ++k) {
    pp[k]->fill_pending = hop;
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
