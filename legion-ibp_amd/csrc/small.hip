// The whole sampling phase of a small batch in one workgroup.
//
// A small batch is bound by latency: in the general path every hop is a launch whose blocks pass counts through
// HBM (look-back) and deduplicate through atomics on a table in HBM, two launches and a gather of 5-13 us each for 16 seeds
// that touch 500 nodes.  One workgroup of 1024 threads has all of it within a barrier's reach instead: the dedup table, the
// slots of a hop's edges and the nodes being sampled lie in LDS, the scans are block scans, and one launch per group of
// batches (a workgroup each) does the seeds, every hop, the relabelling, the cache lookup and the headers.  What is left
// of HBM is the chain seed -> row pointers -> neighbours -> row pointers ... that no kernel can shorten.
// Its rows, where they are all gathered in one pass on the caller's stream, are looked up and gathered by other workgroups of
// the launch, each tile as soon as the sampling workgroup has published its ids: a launch, the lookups of the last hop and the
// host link's latency for the rows of the hops before leave the chain (us a batch, gather behind / inside: 16 seeds, 10,5, a
// third cached 18.4 / 16.6, 96 seeds 30.0 / 25.4; one hop of 20, 64 seeds 16.1 / 13.9; 64 seeds of a Cora-shaped graph,
// 13 MB of rows 25.3 / 23.8, half of them over the link 130 / 116).
// us per batch, gather behind the launch in both, by the hops' launches and here: 16 seeds, fanouts 10,5 (445 edges in the
// last hop): 30 / 19;
// 64 seeds of a Cora-shaped graph, 25,10 (3 680 edges): 27 / 25, 96 (5 185): 28 / 31, 128 (6 979): 30 / 35; 64 seeds, 10,5
// (2 332): 33 / 26; three hops 5,4,3, 16 seeds (846): 45 / 25, 64 (3 918): 44 / 44; one hop of 20, 128 seeds (1 003): 22 / 18,
// 256 (1 918): 22 / 25.  1024 threads, because draws and probes fill the CU's four SIMDs: with 512 the second of these took
// a sixth more, with 256 three quarters.  A barrier of sixteen wavefronts is a tenth of a microsecond: scans take one each
// (three before: 0.7 us a batch of two hops).
// Outputs are those of the general path, bit for bit (same draws, same candidates in the dedup table, same ranks).
#include <algorithm>

#include <hip/hip_ext.h>

#include "gather.hpp"
#include "scan.hpp"

namespace lmi {

constexpr int kSmallBlock = 1024;
constexpr int kSmallItems = 4;  // edges per thread and step of the flag scan
constexpr int kSmallNodes = 2;  // nodes in flight per lane group
constexpr int64_t kSmallLds = 160 * 1024;

struct SmallPipe {
  DevState *st;
  int32_t *ids, *labels;
  int32_t *row_ptr[LMI_MAX_HOPS];
  int32_t *agg_src_ids, *agg_src_off, *agg_dst_off;
  int32_t *cache_index;
  int2 *miss_list;
  uint8_t *features;
  unsigned long long *known;  // with gather workgroups: how many rows they may gather (small_publish), and behind it whether
                              // one of them has left its rows (small_leave)
  int note_seeds;  // Pipe::note_seeds
  BatchParams bp;
};
struct SmallGroup {
  const int64_t *indptr;
  const int32_t *indices;
  int64_t n_nodes;
  int fanout[LMI_MAX_HOPS];
  int hops;
  int log2t;      // LDS dedup table
  int look_mode;
  SlotTable cache;
  // workgroups per batch that look up and gather its rows, beside the one that samples it; 0: a launch behind this one does
  int n, workers, upr, last_off, rows_per_tile;
  int patience;  // reads of SmallPipe::known before a gather workgroup leaves
  RowSources rows;
  SeenWord *rows_seen;  // hinted_rows
  SmallPipe p[LMI_MAX_GROUP];
};
static_assert(sizeof(SmallGroup) <= 4096, "a kernel's arguments");

// The block's LDS, carved by hand: its sizes follow the batch.
struct SmallLds {
  int64_t *beg, *deg;  // [kSmallBlock] rows of the nodes being sampled; those of the first kSmallBlock nodes stay for the
                       // next hop, which then starts without a read
  int32_t *key, *val;  // dedup table: id, lowest candidate (later: local id)
  int *base, *node;    // [kSmallBlock] place of the node's first edge, its id
  int *scan;           // block scans (kSmallScan ints), which take its halves in turn; the last one counts misses
  uint16_t *order;     // [kSmallBlock] the nodes being sampled, those that draw first
  uint16_t *eslot;     // table slot of each edge of the hop
};
constexpr int kSmallScan = 2 * kSmallBlock / kWave + 4;
__host__ __device__ inline int64_t small_lds_bytes(int log2t, int64_t edges) {
  return (int64_t(8) << log2t) + kSmallBlock * 26 + kSmallScan * 4 + 2 * ((edges + 7) / 8 * 8);
}

// Slot of `id`, its value lowered to at most `cand`.  The table is no larger than the distinct ids a valid graph can
// give a batch need; neighbour ids outside the graph could fill it, so the probe is bounded and reports them.
__device__ __forceinline__ int small_insert(const SmallLds &l, int log2t, int32_t id, int cand, bool *full) {
  const int mask = (1 << log2t) - 1;
  int h = (int)hash_id(id, log2t);
  for (int probes = 0; probes <= mask; ++probes) {
    int32_t k = l.key[h];
    if (k == kEmptyKey) k = atomicCAS(&l.key[h], kEmptyKey, id);
    if (k == kEmptyKey || k == id) {
      atomicMin(&l.val[h], cand);
      return h;
    }
    h = (h + 1) & mask;
  }
  *full = true;
  return 0;
}

// `shared`: other workgroups of the launch read the id.
__device__ __forceinline__ void id_store(int32_t *p, int32_t id, bool shared) {
  if (shared) __hip_atomic_store(p, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = id;
}

// Samples the n_here staged nodes, a lane group per node and kSmallNodes nodes in flight, so that their neighbour reads
// overlap.  The nodes come in the order of SmallLds::order, those that draw first: a wavefront computes draws for all its
// groups if one of them needs any, and draws are what one CU is slow at.  (64 seeds of a Cora-shaped graph, where a
// quarter of the nodes draw: 30.4 us in plain order, 27.0 in this one, gather and launches included, both in one run.)
template <int G>
__device__ __forceinline__ void small_sample(const SmallLds &l, const SmallGroup &g, const SmallPipe &a, int hop, int n_here,
                                             int c0, int n_known, int eoff, bool *full) {
  const int lane = threadIdx.x & (G - 1), per_pass = kSmallBlock / G, fanout = g.fanout[hop];
  for (int k0 = threadIdx.x / G; k0 < n_here; k0 += per_pass * kSmallNodes) {
    int32_t nbr[kSmallNodes];
    int at[kSmallNodes];  // the node, or -1 in a lane without an edge
#pragma unroll
    for (int u = 0; u < kSmallNodes; ++u) {
      at[u] = -1;
      nbr[u] = -1;
      if (k0 + u * per_pass >= n_here) continue;
      const int q = n_here > per_pass ? l.order[k0 + u * per_pass] : k0;
      const int64_t deg = l.deg[q];
      uint32_t pick = (uint32_t)lane;
      if (deg > (int64_t)fanout) {
        const uint32_t j = (uint32_t)(deg - fanout) + (uint32_t)lane;
        uint32_t d = 0xFFFFFFFFu;
        if (lane < fanout)
          d = __umulhi(sample_draw(a.bp.rng_seed, (uint32_t)hop, (uint32_t)l.node[q], (uint32_t)lane), j + 1u);
        bool dup = false;  // Floyd's rule (floyd_pick); a loop, for code that runs once per batch is paid for by its length
#pragma unroll 1
        for (int r = 0; r + 1 < fanout; ++r) {
          const uint32_t p = __shfl(dup ? j : d, r, G);
          dup = dup || (lane > r && d == p);
        }
        pick = dup ? j : d;
      }
      if ((int64_t)lane < deg && lane < fanout) {
        at[u] = q;
        nbr[u] = g.indices[l.beg[q] + pick];
      }
    }
#pragma unroll
    for (int u = 0; u < kSmallNodes; ++u) {
      if (at[u] < 0) continue;
      const int e = l.base[at[u]] + lane;
      a.agg_src_ids[eoff + e] = nbr[u];
      a.agg_dst_off[eoff + e] = c0 + at[u];
      l.eslot[e] = (uint16_t)small_insert(l, g.log2t, nbr[u], n_known + e, full);
    }
  }
}

// The rows of a batch whose ids are in memory by now, for the workgroups that gather them: a scan word that only this kernel
// uses, `last` when there will be no more.  One thread calls, behind wait_memory and a barrier.
constexpr int kSmallStampHop = 3;  // a hop that no batch has
static_assert(LMI_MAX_HOPS <= kSmallStampHop, "the stamp would be a hop's");
__device__ __forceinline__ void small_publish(const SmallPipe &a, int rows, bool last) {
  scan_publish(ScanChain{a.known}, scan_stamp(a.bp.serial, kSmallStampHop), 0, last ? kScanInclusive : kScanSum, rows);
}

// A gather workgroup leaves, and its rows to the sampling one, where its wait does not end: one of the two has to see what the
// other has written.  Both are device-scope accesses, each complete before the read of the other's word.
__device__ __forceinline__ unsigned long long small_known(const SmallPipe &a) {
  return __hip_atomic_load(a.known, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void small_leave(const SmallPipe &a) {
  scan_publish(ScanChain{a.known}, scan_stamp(a.bp.serial, kSmallStampHop), 1, kScanInclusive, 0);
  wait_memory();
}
__device__ __forceinline__ bool small_left(const SmallPipe &a) {
  wait_memory();
  return (uint32_t)(__hip_atomic_load(a.known + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 34) ==
         scan_stamp(a.bp.serial, kSmallStampHop);
}

// A workgroup that gathers: every `step`-th tile of rows from `tile` on, each as soon as the sampling workgroup has published
// its ids (`all`: they all are, `known` of them).
// The sampling workgroup has a lower number, but each die starts its share of the workgroups by itself: launches of several
// streams can fill a die with waiting ones while the sampling ones that they wait for stand in line at other dies, filled by
// one another's.  So a wait that lasts (SmallGroup::patience: half a millisecond; an ordinary one is tens of microseconds)
// ends with the workgroup leaving, which gives its place to one that somebody waits for, and the sampling workgroup, which
// waits for nobody, then gathers all the batch's rows itself: some twice, with the same bytes.
__device__ __forceinline__ void small_gather(const SmallGroup &g, const SmallPipe &a, int tile, int step, int known, bool all,
                                             int *lds) {
  const uint32_t stamp = scan_stamp(a.bp.serial, kSmallStampHop);
  int *s_known = lds + kSlotLds;  // rows, whether they are all
  for (int64_t row0 = (int64_t)tile * g.rows_per_tile;; row0 += (int64_t)step * g.rows_per_tile) {
    if (!all && known < row0 + g.rows_per_tile) {
      __syncthreads();  // everybody has read s_known
      if (threadIdx.x == 0) {
        for (int reads = 0;; ++reads) {
          if (reads == g.patience) small_leave(a);
          const unsigned long long w = small_known(a);
          if ((uint32_t)(w >> 34) == stamp) {
            known = (int)(unsigned)w;
            all = ((unsigned)(w >> 32) & 3u) == kScanInclusive;
            if (all || (known >= row0 + g.rows_per_tile && reads < g.patience)) break;
          }
          if (reads >= g.patience) {
            known = 0;
            all = true;
            break;
          }
          __builtin_amdgcn_s_sleep(2);
        }
        s_known[0] = known;
        s_known[1] = all ? 1 : 0;
      }
      __syncthreads();
      known = s_known[0];
      all = s_known[1] != 0;
    }
    if (row0 >= known) return;  // all of them are known by now
    const int n = (int)(known - row0 < g.rows_per_tile ? known : row0 + g.rows_per_tile);
    gather_rows<u32x4_a4, kSmallBlock, 2, true, true, true>(g.rows, nullptr, a.ids, a.features, (int)row0, n, g.upr, g.last_off,
                                                            g.rows_per_tile, g.rows.pitch, 0, 1, true, g.cache, a.cache_index, lds);
  }
}

// The batch's sampling, by one workgroup: the rows it ends with.  WORKERS: others gather them beside it.
template <bool WORKERS>
__device__ __forceinline__ int small_sampled(const SmallGroup &g, const SmallPipe &a, int row, unsigned char *smem) {
  const BatchParams &bp = a.bp;
  const int t = threadIdx.x, T = 1 << g.log2t;
  SmallLds l;
  l.beg = reinterpret_cast<int64_t *>(smem);
  l.deg = l.beg + kSmallBlock;
  l.key = reinterpret_cast<int32_t *>(l.deg + kSmallBlock);
  l.val = l.key + T;
  l.base = reinterpret_cast<int *>(l.val + T);
  l.node = l.base + kSmallBlock;
  l.scan = l.node + kSmallBlock;
  l.order = reinterpret_cast<uint16_t *>(l.scan + kSmallScan);
  l.eslot = l.order + kSmallBlock;
  int *n_miss = l.scan + kSmallScan - 1;
  int scans = 0;
  const auto block_scan = [&](int v, int &total) {  // a barrier each
    return block_exclusive_scan_once<kSmallBlock>(v, l.scan + (scans++ & 1) * (kSmallBlock / kWave), total);
  };
  const FaultTo fault{bp.serial, bp.fault};
  for (int i = t; i < T; i += kSmallBlock) {
    l.key[i] = kEmptyKey;
    l.val[i] = kIntMax;
  }
  if (t == 0) {
    *n_miss = 0;
    state_begin(a.st, bp, g.hops);
    misses_begin(a.st);
  }
  __syncthreads();
  bool full = false;
  // Rows [first, last) of the batch by a thread each: the cache lookup, the miss list (its order is arbitrary) and, where
  // the next hop will sample them from LDS, their row pointers, all in flight together.  Hop -1: the seeds.
  const auto rows = [&](int hop, int first, int last) {
    const bool stay = hop + 1 < g.hops;
    for (int i0 = first; i0 < last; i0 += kSmallBlock) {
      const int i = i0 + t;
      bool miss = false;
      int32_t id = -1;
      if (i < last) {
        id = hop < 0 ? bp.seeds[i] : i < kSmallBlock ? l.node[i] : a.ids[i];
        const bool good = id >= 0 && id < g.n_nodes;
        int64_t lo = 0, hi = 0;
        if (stay && i < kSmallBlock && good) {
          lo = g.indptr[id];
          hi = g.indptr[id + 1];
        }
        int32_t slot = -1;
        if (g.look_mode != LOOK_NOT && good) slot = static_find(g.cache, id);
        if (hop < 0) {
          id_store(&a.ids[i], id, WORKERS);
          a.labels[i] = bp.labels ? bp.labels[i] : -1;
          if (i < kSmallBlock) l.node[i] = id;
          if (good) small_insert(l, g.log2t, id, i, &full);
          else raise_fault(a.st, kFaultBadId, fault);
        }
        if (stay && i < kSmallBlock) {
          l.beg[i] = lo;
          l.deg[i] = hi - lo;
        }
        if (g.look_mode != LOOK_NOT) a.cache_index[i] = slot;
        miss = good && slot < 0;
      }
      if (g.look_mode == LOOK_LIST) {
        const uint64_t m = __ballot(miss);
        int at = 0;
        if ((t & (kWave - 1)) == 0 && m) at = atomicAdd(n_miss, __popcll(m));
        at = __shfl(at, 0, kWave) + __popcll(m & lanemask_lt());
        if (miss) a.miss_list[at] = make_int2(i, id);
      }
    }
  };
  rows(-1, 0, bp.n_seeds);
  __syncthreads();
  int n_known = bp.n_seeds, eoff = 0;
  for (int hop = 0; hop < g.hops; ++hop) {
    const int fanout = g.fanout[hop];
    int G = 4;
    while (G < fanout) G <<= 1;
    int32_t *row_ptr = a.row_ptr[hop];
    // ---- sampling, kSmallBlock nodes at a time: all nodes known so far, in order
    int n_edges = 0;
    const bool here = n_known <= kSmallBlock;  // all their rows are in LDS
    for (int c0 = 0; c0 < n_known; c0 += kSmallBlock) {
      const int my = c0 + t;
      int64_t deg = 0;
      if (here) {
        if (my < n_known) deg = l.deg[t];
      } else {
        int32_t id = -1;
        int64_t lo = 0, hi = 0;
        if (my < n_known) id = a.ids[my];
        if (id >= 0 && id < g.n_nodes) {
          lo = g.indptr[id];
          hi = g.indptr[id + 1];
        }
        l.beg[t] = lo;
        l.deg[t] = deg = hi - lo;
        l.node[t] = id;
      }
      // one scan for the edges (at most 2^16) and, above them, for the places in the order: nodes that draw from the front,
      // the others from the back
      const int n_here = n_known - c0 < kSmallBlock ? n_known - c0 : kSmallBlock;
      const bool draws = deg > (int64_t)fanout;
      int total;
      const int ex = block_scan((draws ? fanout | 1 << 20 : (int)deg), total);
      const int base = n_edges + (ex & 0xfffff), drawn = ex >> 20;
      total &= 0xfffff;
      if (my < n_known) {
        row_ptr[my] = base;
        l.order[draws ? drawn : n_here - 1 - (t - drawn)] = (uint16_t)t;
      }
      l.base[t] = base;
      __syncthreads();
      switch (G) {
        case 4: small_sample<4>(l, g, a, hop, n_here, c0, n_known, eoff, &full); break;
        case 8: small_sample<8>(l, g, a, hop, n_here, c0, n_known, eoff, &full); break;
        case 16: small_sample<16>(l, g, a, hop, n_here, c0, n_known, eoff, &full); break;
        case 32: small_sample<32>(l, g, a, hop, n_here, c0, n_known, eoff, &full); break;
        default: small_sample<64>(l, g, a, hop, n_here, c0, n_known, eoff, &full); break;
      }
      n_edges += total;
      __syncthreads();  // the next nodes overwrite these; the table is complete behind the last ones
    }
    if (t == 0) {
      row_ptr[n_known] = n_edges;
      scan_epilogue(SCAN_EPI_HOP_EDGES, a.st, hop, n_edges);
    }
    // ---- first occurrences: ranks in edge order, ids, local ids.  An edge is one iff the value of its slot names the
    // edge (a published local id never does: it is at most the candidate it replaces, see hop_kernel).
    int n_new = 0;
    for (int e0 = 0; e0 < n_edges; e0 += kSmallBlock * kSmallItems) {
      const int e = e0 + t * kSmallItems;
      int slot[kSmallItems], first[kSmallItems], sum = 0;
#pragma unroll
      for (int u = 0; u < kSmallItems; ++u) {
        slot[u] = e + u < n_edges ? (int)l.eslot[e + u] : 0;
        first[u] = e + u < n_edges && l.val[slot[u]] == n_known + e + u ? 1 : 0;
        sum += first[u];
      }
      int total;
      int at = n_known + n_new + block_scan(sum, total);
      n_new += total;
#pragma unroll
      for (int u = 0; u < kSmallItems; ++u)
        if (first[u]) {
          const int32_t id = l.key[slot[u]];
          l.val[slot[u]] = at;
          id_store(&a.ids[at], id, WORKERS);
          if (at < kSmallBlock) l.node[at] = id;
          ++at;
        }
    }
    const bool last = hop + 1 == g.hops;
    if (WORKERS && last) wait_memory();
    __syncthreads();
    if (WORKERS && last && t == 0) small_publish(a, n_known + n_new, true);
    // ---- local ids of the edges' sources, lookup of the new rows
    for (int e = t; e < n_edges; e += kSmallBlock) a.agg_src_off[eoff + e] = l.val[l.eslot[e]];
    if (!(WORKERS && last)) rows(hop, n_known, n_known + n_new);
    if (t == 0) scan_epilogue(SCAN_EPI_HOP_NODES, a.st, hop, n_new);
    n_known += n_new;
    eoff += n_edges;
    if (WORKERS && !last) wait_memory();  // behind the reads of the new nodes' rows, which took as long
    __syncthreads();  // the next hop overwrites the edges' slots, and reads what was written here
    if (WORKERS && !last && t == 0) small_publish(a, n_known, false);
  }
  if (full) raise_fault(a.st, kFaultBadId, fault);
  if (t == 0) {
    a.st->n_miss[0] = *n_miss;
    if (WORKERS && g.rows_seen && a.note_seeds > 0) note_seen(&g.rows_seen[row], n_known, a.note_seeds);
  }
  return n_known;
}

// WORKERS: with gather workgroups (SmallGroup::workers).  Not a branch: a kernel that might gather samples 0.8 us more slowly.
template <bool WORKERS>
static __global__ __launch_bounds__(kSmallBlock) void batch_small_kernel(SmallGroup g) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int row = WORKERS ? (int)blockIdx.x % g.n : (int)blockIdx.x;
  const SmallPipe &a = g.p[row];
  if constexpr (!WORKERS) {
    small_sampled<false>(g, a, row, smem);
  } else {
    int tile = (int)blockIdx.x / g.n - 1, step = g.workers, known = 0;
    const bool sampler = tile < 0;
    if (sampler) {
      known = small_sampled<true>(g, a, row, smem);
      int *s_left = reinterpret_cast<int *>(smem);
      if (threadIdx.x == 0) *s_left = small_left(a) ? 1 : 0;
      __syncthreads();
      if (*s_left == 0) return;
      tile = 0;
      step = 1;
    }
    small_gather(g, a, tile, step, known, sampler, reinterpret_cast<int *>(smem));
  }
}

// Distinct ids bound the table: a batch's worst case or, in a small graph, its nodes.  Load at most 0.95 in a worst case
// that real batches, which fill a quarter of it, do not come near.
static int small_log2t(const Server *s) {
  const int64_t distinct = std::min(s->max_nodes, s->n_nodes);
  int lg = 6;
  while ((int64_t(1) << lg) * 95 < 100 * distinct) ++lg;
  return lg;
}

// Edges of the largest hop as the graph's mean degree has it (a quarter more for the degrees of neighbours).
static double small_expected_edges(const Server *s) {
  const double mean = 1.25 * (double)s->n_edges / (double)s->n_nodes;
  double nodes = s->cfg.batch_size, most = 0;
  for (int k = 0; k < s->cfg.hops; ++k) {
    const double e = nodes * std::min<double>(mean, s->cfg.fanout[k]);
    most = std::max(most, e);
    nodes += e;
  }
  return most;
}

// Which batches: those whose largest hop is expected to hold at most small_edges edges, half as many where it is the only
// hop (where one workgroup, on one CU, is still faster than a launch a hop over the whole device), and whose table and edges
// fit the LDS of a CU in the worst case.  Not with the LRU cache: its lookup waits for the insertion before and asks the dedup table in HBM for repeated
// seeds.
bool small_batch(const Server *s) {
  const int lg = small_log2t(s);
  const double most = (double)s->small_edges * (s->cfg.hops == 1 ? 0.5 : 1.0);
  return s->cache_kind != LMI_CACHE_LRU && lg <= 15 && small_lds_bytes(lg, s->max_edges_hop) <= kSmallLds &&
         small_expected_edges(s) <= most && !s->lds_dedup && s->fuse_count;
}

int launch_small(Server *s, Pipe *const *pp, const BatchParams *bps, int n, hipStream_t st, HopLookup look) {
  SmallGroup g{};
  g.indptr = s->indptr;
  g.indices = s->indices;
  g.n_nodes = s->n_nodes;
  g.hops = s->cfg.hops;
  for (int k = 0; k < s->cfg.hops; ++k) g.fanout[k] = s->cfg.fanout[k];
  g.log2t = small_log2t(s);
  g.look_mode = look.mode;
  g.cache = slot_table(s);
  g.n = n;
  for (int k = 0; k < n; ++k) pipe_seeds(s, *pp[k], bps[k].n_seeds);
  const int64_t lds = small_lds_bytes(g.log2t, s->max_edges_hop);
  int64_t workers = 0;
  if (look.early_rows) {
    g.rows = RowSources{s->cache_data, s->feat, (uint32_t)(s->cache_kind == LMI_CACHE_NONE ? 0 : s->cache_rows),
                        (uint32_t)s->n_nodes, s->row_bytes};
    g.upr = (int)((s->row_bytes + 15) / 16);
    g.last_off = (int)s->row_bytes - 16;
    // A workgroup's one pass.  A batch of its own takes up to a workgroup per CU (64 seeds of a Cora-shaped graph on 255 / 127 /
    // 63: 23.8 / 27.8 / 36.0 us).  A CU has room for one, of sixteen wavefronts with more than 96 scalar registers, and those of
    // a group wait with several sampling ones: no more of them than leave room for another such launch beside it, or a launch
    // behind this one gathers (us a group at most half of the CUs / a quarter: eight batches of 32 seeds, 10,5, all rows cached
    // 17.1 / 19.0, four of 96 23.8 / 27.2; four streams of the first kind, one group each: 40 / 52).  Where yet more streams
    // wait on each other, small_gather ends it.
    const int64_t tile_bytes = n == 1 ? 16 * 1024 : 32 * 1024;
    g.rows_per_tile = (int)std::max<int64_t>(1, std::min<int64_t>(kFlatTileMax, tile_bytes / s->row_bytes));
    const int64_t tiles = ceil_div(hinted_rows(s, s->max_nodes, 0, pp, n), g.rows_per_tile);
    const int64_t room = s->n_cu / 2 / n - 1;
    workers = n == 1 ? std::min<int64_t>(tiles, s->n_cu - 1) : 2 * room >= tiles ? std::min(tiles, room) : 0;
    if (s->cache_kind == LMI_CACHE_NONE && s->feat_loc == LMI_LOC_HOST)  // a grid that fills the link
      workers = std::min<int64_t>(workers, std::max(1, early_rows_blocks(s, 0) * 256 / kSmallBlock / n));
    if (workers > 0) {
      g.rows_seen = s->rows_seen_dev;
      g.look_mode = LOOK_NOT;
    }
  }
  g.workers = (int)workers;
  g.patience = s->small_patience;
  for (int k = 0; k < n; ++k) {
    Pipe &p = *pp[k];
    SmallPipe &a = g.p[k];
    a.st = p.st;
    a.ids = p.ids;
    a.labels = p.labels;
    for (int h = 0; h < LMI_MAX_HOPS; ++h) a.row_ptr[h] = p.blk_indptr[h];
    a.agg_src_ids = p.agg_src_ids;
    a.agg_src_off = p.agg_src_off;
    a.agg_dst_off = p.agg_dst_off;
    a.cache_index = p.cache_index;
    a.miss_list = p.miss_list;
    a.features = (uint8_t *)p.features;
    a.known = p.scan_words;
    a.bp = bps[k];
    a.note_seeds = p.note_seeds;
    p.hops_done = s->cfg.hops;
    p.fill_pending = -1;
    p.table_in_lds = true;
    p.rows_done = g.workers > 0;
    if (bps[k].clear_table) p.table_dirty = true;  // this batch leaves the table in HBM as it is
  }
  const dim3 grid(n * (1 + g.workers));
  if (workers > 0 && look.end)
    hipExtLaunchKernelGGL(batch_small_kernel<true>, grid, dim3(kSmallBlock), (size_t)lds, st, nullptr, look.end, 0, g);
  else if (workers > 0)
    hipLaunchKernelGGL(batch_small_kernel<true>, grid, dim3(kSmallBlock), (size_t)lds, st, g);
  else
    hipLaunchKernelGGL(batch_small_kernel<false>, grid, dim3(kSmallBlock), (size_t)lds, st, g);
  LMI_HIP(hipGetLastError());
  s->routes.small_batches += n;
  if (workers > 0) s->row_routes.small_rows += n;
  return LMI_OK;
}

}  // namespace lmi
