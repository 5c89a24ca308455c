// BFS on gfx950: unweighted levels from `src`, INT_MAX for unreachable.
//
// Reference family: codes/cuda/bfs-cuda (180 variants).  The styles below
// cover its axes on wave64 hardware:
//   v_topo_push_*   [C-BVT] BFS_CUDA_V_Topo_Push_..._Thread:46-119 (warp/block
//                   siblings map to one wave64 / one 256-lane workgroup)
//   v_topo_pull_*   BFS_CUDA_V_Topo_Pull_..._Thread:56-78
//   *_determ        level-synchronous rule `if (s == iter)` (Determ siblings :65)
//   *_cas / *_seqcst  CAS-loop and seq_cst/system-scope atomicMin (the
//                   reference's Atomic vs CudaAtomic axis)
//   v_data_push_*   [C-BVD]:46-139 worklist with NonDup stamps
//   e_topo_push_*   [C-BET]:56-115 one edge per item
//   e_data_push_*   [C-BED]:46-140 edge worklist, stamps on edge ids
//   do_hybrid       direction-optimizing BFS (no reference counterpart):
//                   top-down from a chunked queue, bottom-up over unvisited
//                   vertices, switched per level on the device
// All styles produce identical level arrays (BFS levels are unique).
#include "igx_internal.hpp"
#include "igx_frontier.hpp"

namespace igx {
namespace {

enum Gran { kThread = 0, kWaveG = 1, kBlockG = 2 };

__global__ void __launch_bounds__(kBlock) bfs_init(int src, int* __restrict__ dist, int n)
{
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n) dist[v] = (v == src) ? 0 : kInf;
}

__global__ void __launch_bounds__(kBlock) fill_int(int* __restrict__ p, int value, long long count)
{
  const long long stride = (long long)gridDim.x * kBlock;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < count; i += stride) p[i] = value;
}

// --------------------------------------------------- vertex, topology ----
template <int G, int AK, bool DETERM, bool PERSIST>
__global__ void __launch_bounds__(kBlock) bfs_vtopo_push(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, int n,
                                                          int* __restrict__ dist, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int iter = ctl->iter;
  bool updated = false;
  if constexpr (G == kThread) {
    const int stride = gridDim.x * kBlock;
    for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
      const int s = dist[v];
      if (s != kInf && (!DETERM || s == iter)) {
        const int nd = s + 1;
        for (int i = nindex[v]; i < nindex[v + 1]; i++) {
          if (atomic_min_k<AK>(&dist[nlist[i]], nd) > nd) updated = true;
        }
      }
    }
  } else if constexpr (G == kWaveG) {
    const int waves = gridDim.x * kWavesPerBlock;
    const int lane = lane_id();
    for (int v = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; v < n; v += waves) {
      const int s = dist[v];
      if (s != kInf && (!DETERM || s == iter)) {
        const int nd = s + 1;
        for (int i = nindex[v] + lane; i < nindex[v + 1]; i += kWave) {
          if (atomic_min_k<AK>(&dist[nlist[i]], nd) > nd) updated = true;
        }
      }
    }
  } else {
    for (int v = blockIdx.x; v < n; v += gridDim.x) {
      const int s = dist[v];
      if (s != kInf && (!DETERM || s == iter)) {
        const int nd = s + 1;
        for (int i = nindex[v] + (int)threadIdx.x; i < nindex[v + 1]; i += kBlock) {
          if (atomic_min_k<AK>(&dist[nlist[i]], nd) > nd) updated = true;
        }
      }
    }
  }
  raise_flag(ctl, updated);
}

template <int G>
__global__ void __launch_bounds__(kBlock) bfs_vtopo_pull(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, int n,
                                                          int* __restrict__ dist, Ctl* ctl)
{
  if (round_done(ctl)) return;
  bool updated = false;
  if constexpr (G == kThread) {
    const int stride = gridDim.x * kBlock;
    for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
      const int d0 = dist[v];
      int d = d0;
      for (int i = nindex[v]; i < nindex[v + 1]; i++) {
        const int s = load_relaxed(&dist[nlist[i]]);
        if (s != kInf && s + 1 < d) d = s + 1;
      }
      if (d < d0) {
        store_relaxed(&dist[v], d);
        updated = true;
      }
    }
  } else {
    const int waves = gridDim.x * kWavesPerBlock;
    const int lane = lane_id();
    for (int v = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; v < n; v += waves) {
      const int d0 = dist[v];
      int d = d0;
      for (int i = nindex[v] + lane; i < nindex[v + 1]; i += kWave) {
        const int s = load_relaxed(&dist[nlist[i]]);
        if (s != kInf && s + 1 < d) d = s + 1;
      }
      #pragma unroll
      for (int k = kWave / 2; k > 0; k >>= 1) d = min(d, __shfl_xor(d, k, kWave));
      if (d < d0) {
        if (lane == 0) store_relaxed(&dist[v], d);
        updated = true;
      }
    }
  }
  raise_flag(ctl, updated);
}

// ------------------------------------------------------- edge, topology ----
template <int AK>
__global__ void __launch_bounds__(kBlock) bfs_etopo_push(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                          int m, int* __restrict__ dist, Ctl* ctl)
{
  if (round_done(ctl)) return;
  bool updated = false;
  const int stride = gridDim.x * kBlock;
  for (int e = blockIdx.x * kBlock + threadIdx.x; e < m; e += stride) {
    const int s = dist[sp[e]];
    if (s != kInf) {
      const int nd = s + 1;
      const int dst = nlist[e];
      if (dist[dst] > nd && atomic_min_k<AK>(&dist[dst], nd) > nd) updated = true;
    }
  }
  raise_flag(ctl, updated);
}

// ------------------------------------------------------- vertex, data ----
__global__ void __launch_bounds__(kBlock) bfs_vdata_init(int src, int* __restrict__ wl, Ctl* ctl)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    wl[0] = src;
    ctl->wl_count[0] = 1;
    ctl->wl_count[1] = 0;
  }
}

template <int G>
__global__ void __launch_bounds__(kBlock) bfs_vdata_push(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, int* __restrict__ dist,
                                                          int* __restrict__ wl0, int* __restrict__ wl1,
                                                          int* __restrict__ stamp, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int iter = ctl->iter;
  const int p = iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  int* wl_out = p ? wl0 : wl1;
  int* out_count = &ctl->wl_count[p ^ 1];
  const int tag = iter + 1;
  if constexpr (G == kThread) {
    const int stride = gridDim.x * kBlock;
    for (int idx = blockIdx.x * kBlock + threadIdx.x; idx < count; idx += stride) {
      const int v = wl_in[idx];
      const int s = dist[v];
      if (s != kInf) {
        const int nd = s + 1;
        for (int i = nindex[v]; i < nindex[v + 1]; i++) {
          const int dst = nlist[i];
          bool push = false;
          if (dist[dst] > nd && atomic_min_relaxed(&dist[dst], nd) > nd) {
            push = atomic_max_relaxed(&stamp[dst], tag) != tag;
          }
          const int slot = wave_push_slot(out_count, push);
          if (push) wl_out[slot] = dst;
        }
      }
    }
  } else {
    const int waves = gridDim.x * kWavesPerBlock;
    const int lane = lane_id();
    for (int idx = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; idx < count; idx += waves) {
      const int v = wl_in[idx];
      const int s = dist[v];
      if (s != kInf) {
        const int nd = s + 1;
        const int beg = nindex[v], end = nindex[v + 1];
        for (int base = beg; base < end; base += kWave) {
          const int i = base + lane;
          bool push = false;
          if (i < end) {
            const int dst = nlist[i];
            if (dist[dst] > nd && atomic_min_relaxed(&dist[dst], nd) > nd) {
              push = atomic_max_relaxed(&stamp[dst], tag) != tag;
            }
            const int slot = wave_push_slot(out_count, push);
            if (push) wl_out[slot] = dst;
          }
        }
      }
    }
  }
}

// --------------------------------------------------------- edge, data ----
__global__ void __launch_bounds__(kBlock) bfs_edata_init(int src, const int* __restrict__ nindex,
                                                          int* __restrict__ wl, Ctl* ctl)
{
  if (blockIdx.x != 0) return;
  const int beg = nindex[src], end = nindex[src + 1];
  for (int i = beg + (int)threadIdx.x; i < end; i += kBlock) wl[i - beg] = i;
  if (threadIdx.x == 0) {
    ctl->wl_count[0] = end - beg;
    ctl->wl_count[1] = 0;
  }
}

// One thread per worklist edge.  When dst improves, all of dst's edges are
// queued for the next round at once, so the NonDup test is kept per source
// vertex (vstamp[dst] == tag), admitting exactly the edges that per-edge
// stamps admit; the ids are written wave-cooperatively.
__global__ void __launch_bounds__(kBlock) bfs_edata_push(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, const int* __restrict__ sp,
                                                          int* __restrict__ dist, int* __restrict__ wl0,
                                                          int* __restrict__ wl1, int* __restrict__ vstamp, Ctl* ctl)
{
  __shared__ ListLds s_list;
  if (round_done(ctl)) return;
  const int iter = ctl->iter;
  const int p = iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  int* wl_out = p ? wl0 : wl1;
  int* out_count = &ctl->wl_count[p ^ 1];
  const int tag = iter + 1;
  const int per = list_items_per_thread(count);
  const long long step = (long long)gridDim.x * kBlock * per;
  with_list_items(per, [&](auto items) {
    constexpr int kPer = decltype(items)::value;
    for (long long base = (long long)blockIdx.x * kBlock * per; base < count; base += step) {  // uniform per workgroup
      int e[kPer], rbeg[kPer], rlen[kPer];
      #pragma unroll
      for (int k = 0; k < kPer; k++) {
        const long long idx = base + k * kBlock + (int)threadIdx.x;
        e[k] = (k < per && idx < count) ? wl_in[idx] : -1;
        rbeg[k] = rlen[k] = 0;
      }
      int s[kPer], dst[kPer], d[kPer];
      #pragma unroll
      for (int k = 0; k < kPer; k++) {
        s[k] = (e[k] >= 0) ? dist[sp[e[k]]] : kInf;
        dst[k] = (e[k] >= 0) ? nlist[e[k]] : 0;
      }
      #pragma unroll
      for (int k = 0; k < kPer; k++) d[k] = (e[k] >= 0) ? dist[dst[k]] : 0;
      #pragma unroll
      for (int k = 0; k < kPer; k++) {
        if (s[k] == kInf) continue;
        const int nd = s[k] + 1;
        if (d[k] > nd && atomic_min_relaxed(&dist[dst[k]], nd) > nd && atomic_max_relaxed(&vstamp[dst[k]], tag) != tag) {
          rbeg[k] = nindex[dst[k]];
          rlen[k] = nindex[dst[k] + 1] - rbeg[k];
        }
      }
      block_push_edge_ranges(wl_out, out_count, rbeg, rlen, count <= kListAlone, s_list);
    }
  });
}

// ------------------------------------------ direction-optimizing hybrid ----
// Per level one kernel: top-down expansion of the frontier, or bottom-up over
// every vertex.  The last block picks the next direction with Beamer's rule
// (top-down -> bottom-up when the next frontier's edges exceed the unvisited
// edges / kAlpha; back when the frontier has < n / kBeta vertices).
//
// Frontier representation.  Three bitmaps rotate: bm[level % 3] holds the
// current frontier, bm[(level + 1) % 3] receives the next one and
// bm[(level + 2) % 3] (the previous frontier) is cleared for the level after.
// The bitmaps are always complete.  A top-down level whose frontier has at
// most kQueueEdges edges also appends the discovered vertices' chunks to a
// segmented queue (few appends, so the queue is cheaper to read than the
// bitmap); larger top-down levels and all bottom-up levels produce the bitmap
// only -- no queue atomics at all.  A top-down level reads the queue when the
// previous level wrote one (ctl->in_bits == 0), else the bitmap: 64-vertex
// tiles whose rows of at most kChunk edges one wave expands, and the
// precomputed chunks of the longer rows, filtered by the bitmap.
constexpr int kAlpha = 14;
constexpr int kBeta = 24;
constexpr long long kQueueEdges = 1 << 16;

// Narrow levels.  A level costs two dependent launches, about 12 us on this
// chip however few vertices it has, and a mesh has thousands of levels of a
// few hundred.  So the workgroup that ends a level goes on by itself while the
// frontier has at most kNarrowEdges edges: the frontier's edges are a list in
// LDS (no owner search), a level is one pass over it by 1024 threads, and
// nothing is written to memory but the levels themselves.  What bounds such a
// level is the chain nlist -> dist -> compare-and-swap -> nindex, about 4 us
// (grid 512 x 512 without long edges: 1018 levels in 3.9 ms).  At 4096 edges
// it takes about as long as the two launches (a limit of 8192 measured the
// same), since one CU takes in about one cache line a cycle.  A launch ends
// after kNarrowLevels levels, so that the host can look at its time limit.
// Levels from a queue above the limit run on few workgroups, one per
// kLevelEdges edges.  Grid 1024 x 1024, whole run: 21.3 -> 11.0 ms.
constexpr int kNarrowEdges = 4 * kFinBlock;
constexpr int kNarrowLevels = 512;
constexpr int kFewEdges = 1 << 20;  // graphs below it seldom need more than four levels beyond the narrow ones
constexpr long long kLevelEdges = 256;  // frontier edges per workgroup of a level from a queue
constexpr int kNarrowShift = 21;  // a wave's edges, cut off: 256 * (kNarrowEdges + 1) < 2^21; its vertices above
typedef int NarrowRow __attribute__((ext_vector_type(2), aligned(4)));  // a row's two offsets in one load

// Clears the control block and prepares the run: dist, bitmaps 0 and 1 (2 is
// cleared during level 0) with src in 0, and src's chunks in queue segment 0.
__global__ void __launch_bounds__(kBlock) bfs_do_init(int src, const int* __restrict__ nindex, int n, int m,
                                                       int* __restrict__ dist, Entry* __restrict__ q0,
                                                       unsigned* __restrict__ bm, int words, Ctl* ctl)
{
  const int stride = gridDim.x * kBlock;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  for (int v = t; v < n; v += stride) dist[v] = (v == src) ? 0 : kInf;
  for (int i = t; i < 2 * words; i += stride) bm[i] = (i == (src >> 5)) ? (1u << (src & 31)) : 0u;
  if (blockIdx.x != 0) return;
  const int beg = nindex[src], end = nindex[src + 1];
  const int c = chunks_of(end - beg);
  for (int k = threadIdx.x; k < c; k += kBlock) {
    const int b = beg + k * kChunk;
    q0[k] = Entry{src, b, (b + kChunk < end) ? b + kChunk : end, 0};
  }
  if ((int)threadIdx.x < kGroups) {
    GroupSlot* gs = ctl_groups(ctl) + threadIdx.x;
    gs->qcount[0] = (threadIdx.x == 0) ? c : 0;
    gs->qcount[1] = 0;
    gs->tiles = 0;
  }
  if (threadIdx.x == 0) {
    Ctl z = {};
    z.n = n;
    z.edges_next = end - beg;  // edges of the current frontier
    z.edges_unvisited = (long long)m - (end - beg);
    *ctl = z;
  }
}

__device__ __forceinline__ bool in_bits(const unsigned* __restrict__ bits, int w)
{
  return (bits[w >> 5] >> (w & 31)) & 1u;
}

__global__ void __launch_bounds__(kBlock) bfs_do_level(const int* __restrict__ nindex,
                                                        const int* __restrict__ nlist, int n,
                                                        int* __restrict__ dist, SegQ q0, SegQ q1,
                                                        const Entry* __restrict__ bigq,
                                                        const int* __restrict__ bigq_count,
                                                        unsigned* __restrict__ bm, int words, bool short_rows,
                                                        Ctl* ctl)
{
  __shared__ int s_excl[kWavesPerBlock][kWave];
  __shared__ Entry s_ent[kWavesPerBlock][kWave];
  __shared__ long long s_red[kWavesPerBlock * kStats];
  if (round_done(ctl)) return;
  // a level from a small queue runs on the first `active` workgroups only
  const int active = (ctl->active > 0) ? ctl->active : (int)gridDim.x;
  if ((int)blockIdx.x >= active) return;
  const int level = ctl->level;
  const int mode = ctl->mode;
  const int in_b = ctl->in_bits;
  const bool out_b = (mode == 1) || (ctl->edges_next > kQueueEdges);
  const int p = level & 1;
  const SegQ q_in = p ? q1 : q0;
  const SegQ q_out = p ? q0 : q1;
  Entry* q_mine = segq_mine(q_out);
  int* out_count = segq_counter(ctl, p ^ 1, my_group());
  const int turn = level + ctl->bm_phase;
  const unsigned* cur = bm + (size_t)(turn % 3) * words;
  unsigned* next = bm + (size_t)((turn + 1) % 3) * words;
  unsigned* stale = bm + (size_t)((turn + 2) % 3) * words;
  const int nd = level + 1;
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  const int gw = blockIdx.x * kWavesPerBlock + w;
  const int nwaves = active * kWavesPerBlock;
  {
    const int stride = active * kBlock;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < words; i += stride) stale[i] = 0u;
  }
  long long found_v = 0, found_e = 0;
  if (mode == 0) {
    auto discover = [&](const Entry&, int e) {
      const int u = nlist[e];
      bool disc = false;
      int ub = 0, ue = 0;
      if (dist[u] == kInf) {
        int expected = kInf;
        disc = __hip_atomic_compare_exchange_strong(&dist[u], &expected, nd, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        if (disc) {
          atomicOr(&next[u >> 5], 1u << (u & 31));
          ub = nindex[u];
          ue = nindex[u + 1];
          found_v += 1;
          found_e += ue - ub;
        }
      }
      if (!out_b) push_vertex_chunks(q_mine, out_count, disc && ue > ub, u, ub, ue);
    };
    if (!in_b) {
      const SegPrefix pre = segq_prefix(ctl, p);
      wave_expand_with(pre.pre[kGroups], gw, nwaves, s_excl[w], s_ent[w],
                       [&](int i) { return segq_at(q_in, pre, i); }, discover);
    } else {
      // rows of at most kChunk edges, the non-empty 64-vertex tiles of the bitmap
      for_each_bitmap_tile(cur, n, gw, nwaves, [&](int v0, bool in) {
        const int u = v0 + lane;
        Entry ent = Entry{0, 0, 0, 0};
        if (in) {
          const int b = nindex[u], e = nindex[u + 1];
          if (e - b <= kChunk) ent = Entry{u, b, e, 0};
        }
        const int len = ent.end - ent.beg;
        const int incl = wave_incl_scan(len);
        const int total = wave_bcast(incl, kWave - 1);
        if (total == 0) return;  // uniform
        __builtin_amdgcn_wave_barrier();
        s_excl[w][lane] = incl - len;
        s_ent[w][lane] = ent;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        for (int tb = 0; tb < total; tb += kWave) {
          const int t = tb + lane;
          if (t < total) {
            int lo = 0, hi = kWave;
            while (hi - lo > 1) {
              const int mid = (lo + hi) >> 1;
              if (s_excl[w][mid] <= t) lo = mid;
              else hi = mid;
            }
            const Entry& en = s_ent[w][lo];
            discover(en, en.beg + (t - s_excl[w][lo]));
          }
        }
        __builtin_amdgcn_wave_barrier();
      });
      // longer rows: their precomputed chunks, kept when the row is in the frontier
      wave_expand_with(*bigq_count, gw, nwaves, s_excl[w], s_ent[w],
                       [&](int i) {
                         Entry en = bigq[i];
                         if (!in_bits(cur, en.v)) en.end = en.beg;
                         return en;
                       },
                       discover);
    }
  } else {
    // kSub 64-vertex sub-tiles per step, their loads issued together (the
    // chain dist -> row -> first neighbours -> frontier bits is latency-bound),
    // side by side on a large graph and one grid apart on a small one, so that
    // every wave has some.  Rows that go on: by their lanes, kStep neighbours
    // at once up to kLaneRow, and only the rest by the wave, one after the
    // other (Erdos-Renyi n = 20 k, average degree 8, all by the wave: the whole
    // run 158 us, 97 us this way); on a large graph with long rows, where few
    // go past the first four, by the wave at once (R-MAT 22 219 -> 217 us)
    constexpr int kFirst = 4;
    constexpr int kSub = 4;
    constexpr int kStep = 4;
    constexpr int kLaneRow = 36;
    const int ntiles = (n + kWave - 1) / kWave;
    auto bottom_up = [&](auto dense) {
      constexpr bool kDense = decltype(dense)::value;
      const int apart = kDense ? 1 : nwaves;
      const bool by_lanes = !kDense || short_rows;
      for (int tile0 = gw * (kDense ? kSub : 1); tile0 < ntiles; tile0 += nwaves * kSub) {  // uniform per wave
        bool unvisited[kSub], found[kSub];
        int ub[kSub], ue[kSub];
        #pragma unroll
        for (int s = 0; s < kSub; s++) {
          const long long u = ((long long)tile0 + (long long)s * apart) * kWave + lane;
          unvisited[s] = (u < n) && dist[u] == kInf;
          found[s] = false;
          ub[s] = ue[s] = 0;
        }
        #pragma unroll
        for (int s = 0; s < kSub; s++) {
          const long long u = ((long long)tile0 + (long long)s * apart) * kWave + lane;
          if (unvisited[s]) {
            ub[s] = nindex[u];
            ue[s] = nindex[u + 1];
          }
        }
        int nb[kSub][kFirst];
        #pragma unroll
        for (int s = 0; s < kSub; s++) {
          #pragma unroll
          for (int k = 0; k < kFirst; k++) nb[s][k] = (unvisited[s] && ub[s] + k < ue[s]) ? nlist[ub[s] + k] : -1;
        }
        #pragma unroll
        for (int s = 0; s < kSub; s++) {
          #pragma unroll
          for (int k = 0; k < kFirst; k++) found[s] = found[s] || (nb[s][k] >= 0 && in_bits(cur, nb[s][k]));
        }
        #pragma unroll
        for (int s = 0; s < kSub; s++) {
          const long long tile = (long long)tile0 + (long long)s * apart;
          if (tile >= ntiles) break;  // uniform
          int at = ub[s] + kFirst;
          const int stop = by_lanes ? min(ue[s], ub[s] + kLaneRow) : at;
          while (unvisited[s] && !found[s] && at < stop) {
            int u[kStep];
            #pragma unroll
            for (int k = 0; k < kStep; k++) u[k] = (at + k < stop) ? nlist[at + k] : -1;
            #pragma unroll
            for (int k = 0; k < kStep; k++) found[s] = found[s] || (u[k] >= 0 && in_bits(cur, u[k]));
            at += kStep;
          }
          uint64_t pending = ballot(unvisited[s] && !found[s] && ue[s] > stop);
          while (pending != 0) {
            const int L = __ffsll((unsigned long long)pending) - 1;
            pending &= pending - 1;
            const int s0 = __shfl(stop, L, kWave);
            const int e0 = __shfl(ue[s], L, kWave);
            bool hit = false;
            for (int i0 = s0; i0 < e0; i0 += kWave) {
              const int i = i0 + lane;
              const bool h = (i < e0) && in_bits(cur, nlist[i]);
              if (ballot(h) != 0) {
                hit = true;
                break;
              }
            }
            if (lane == L) found[s] = hit;
          }
          if (found[s]) {
            dist[tile * kWave + lane] = nd;
            found_v += 1;
            found_e += ue[s] - ub[s];
          }
          const uint64_t mask = ballot(found[s]);
          const long long wd = tile * 2;
          if (lane == 0) next[wd] = (unsigned)mask;
          if (lane == 1) next[wd + 1] = (unsigned)(mask >> 32);
        }
      }
    };
    if (ntiles >= nwaves * kSub) bottom_up(std::true_type{});
    else bottom_up(std::false_type{});
  }
  round_partials(ctl, found_v, found_e, 0, 0, s_red);
}

// Level decision (thread 0 of bfs_do_finish after each bfs_do_level): totals
// s[0] = vertices found, s[1] = their edges.
struct FinBfsDo {
  __device__ void operator()(Ctl* ctl, const RoundTotals& t) const
  {
    const long long nf = t.s[0];
    const long long mf = t.s[1];
    const int p = ctl->level & 1;
    const bool out_b = (ctl->mode == 1) || (ctl->edges_next > kQueueEdges);
    ctl->edges_unvisited -= mf;
    if (nf == 0) {
      ctl->done = 1;
    } else if (ctl->mode == 0) {
      if (mf > ctl->edges_unvisited / kAlpha) ctl->mode = 1;
    } else {
      if (nf < (long long)ctl->n / kBeta) ctl->mode = 0;
    }
    ctl->in_bits = out_b ? 1 : 0;
    ctl->edges_next = mf;
    GroupSlot* gs = ctl_groups(ctl);
    for (int g = 0; g < kGroups; g++) gs[g].qcount[p] = 0;
    ctl->level += 1;
    ctl->iter += 1;
  }
};

// Ends a level (after_level; the first launch of a run has none to end) and
// runs the narrow levels that follow it, see kNarrowEdges.  One workgroup.
//
// The frontier comes from the queue and, when the narrow levels end with one
// left, goes back to it (segment 0) and to its bitmap, in the state that
// bfs_do_level expects.  In between the bitmaps are not kept: the entry
// frontier's bits are cleared, which leaves the bitmap of the frontier before
// it the only one with bits, and bm_phase is set so that at the end this one
// is the stale bitmap again.
__global__ void __launch_bounds__(kFinBlock) bfs_do_finish(const int* __restrict__ nindex,
                                                            const int* __restrict__ nlist, int* __restrict__ dist,
                                                            SegQ q0, SegQ q1, unsigned* __restrict__ bm, int words,
                                                            int nparts, bool after_level, Ctl* ctl)
{
  __shared__ int s_edge[2][kNarrowEdges];  // edges of the current and of the next frontier
  __shared__ int s_vert[kNarrowEdges];     // vertices of the next frontier (at most one per edge walked)
  __shared__ unsigned long long s_found;   // vertices (high half) and edges of the next frontier
  __shared__ int s_edges, s_over, s_chunks;
  __shared__ int s_go;
  if (round_done(ctl)) return;
  const int tid = threadIdx.x;
  if (after_level) {
    const RoundTotals tot = round_totals<0x3>(ctl, nparts);
    if (tid == 0) FinBfsDo{}(ctl, tot);
  }
  // workgroups of the next level: a queue level takes one per kLevelEdges edges, at least 64
  auto set_active = [&]() {
    const long long want = (ctl->edges_next + kLevelEdges - 1) / kLevelEdges;
    const bool few = ctl->mode == 0 && ctl->in_bits == 0 && want < nparts;
    ctl->active = few ? (int)max(want, 64LL) : 0;
  };
  if (tid == 0) {
    s_go = !ctl->done && ctl->in_bits == 0 && ctl->edges_next <= kNarrowEdges;
    s_edges = 0;
    s_chunks = 0;
    if (!s_go) set_active();
  }
  __syncthreads();
  if (!s_go) return;
  const int level0 = ctl->level;
  const int phase0 = ctl->bm_phase;
  long long unvisited = ctl->edges_unvisited;
  {
    const int p = level0 & 1;
    const SegQ q_in = p ? q1 : q0;
    unsigned* cur = bm + (size_t)((level0 + phase0) % 3) * words;
    const SegPrefix pre = segq_prefix(ctl, p);
    for (int i = tid; i < pre.pre[kGroups]; i += kFinBlock) {
      const Entry en = segq_at(q_in, pre, i);
      cur[en.v >> 5] = 0u;
      const int len = en.end - en.beg;
      const int at = atomicAdd(&s_edges, len);
      for (int k = 0; k < len; k++) s_edge[0][at + k] = en.beg + k;
    }
  }
  int level = level0;
  int count = 0;
  int found = 1;
  __syncthreads();
  count = s_edges;
  __syncthreads();
  if (tid < kGroups) ctl_groups(ctl)[tid].qcount[level0 & 1] = 0;
  for (;;) {  // uniform
    if (tid == 0) {
      s_found = 0;
      s_over = 0;
    }
    __syncthreads();
    const int* in = s_edge[(level - level0) & 1];
    int* out = s_edge[((level - level0) & 1) ^ 1];
    const int nd = level + 1;
    with_narrow_items(count, [&](auto items) {
      constexpr int kPer = decltype(items)::value;
      if ((tid & ~(kWave - 1)) >= count) return;  // uniform per wave
      int u[kPer], d[kPer];
      #pragma unroll
      for (int k = 0; k < kPer; k++) {
        const int i = k * kFinBlock + tid;
        u[k] = (i < count) ? nlist[in[i]] : -1;
      }
      #pragma unroll
      for (int k = 0; k < kPer; k++) d[k] = (u[k] >= 0) ? dist[u[k]] : 0;
      bool won[kPer];
      #pragma unroll
      for (int k = 0; k < kPer; k++) {
        won[k] = false;
        if (d[k] == kInf) {
          int expected = kInf;
          won[k] = __hip_atomic_compare_exchange_strong(&dist[u[k]], &expected, nd, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      // the rows of the winners only: one CU takes in about one cache line a
      // cycle, and with thousands of scattered edges that rate is the level's time
      NarrowRow row[kPer];
      #pragma unroll
      for (int k = 0; k < kPer; k++) row[k] = won[k] ? *(const NarrowRow*)(nindex + u[k]) : NarrowRow{0, 0};
      // places for the thread's winners and their edges: one scan and one LDS
      // atomic per wave, of (winners, edges) in one number; lengths enter it cut
      // off just above kNarrowEdges, what is cut goes to s_over
      unsigned mine = 0;
      #pragma unroll
      for (int k = 0; k < kPer; k++) {
        const int len = row[k][1] - row[k][0];
        if (won[k]) mine += (1u << kNarrowShift) + (unsigned)min(len, kNarrowEdges + 1);
        if (len > kNarrowEdges + 1) atomicAdd(&s_over, len - (kNarrowEdges + 1));
      }
      if (ballot(mine != 0) != 0) {
        const unsigned incl = (unsigned)wave_incl_scan((int)mine);
        unsigned long long base = 0;
        if (lane_id() == kWave - 1) {
          base = atomicAdd(&s_found, ((unsigned long long)(incl >> kNarrowShift) << 32) |
                                         (incl & ((1u << kNarrowShift) - 1u)));
        }
        base = __shfl(base, kWave - 1, kWave);
        const unsigned excl = incl - mine;
        int vat = (int)(base >> 32) + (int)(excl >> kNarrowShift);
        int eat = (int)(base & 0xffffffffull) + (int)(excl & ((1u << kNarrowShift) - 1u));
        #pragma unroll
        for (int k = 0; k < kPer; k++) {
          if (!won[k]) continue;
          s_vert[vat++] = u[k];
          const int len = min(row[k][1] - row[k][0], kNarrowEdges + 1);
          if (eat <= kNarrowEdges - len) {  // else the frontier is not narrow: the list is not used
            for (int j = 0; j < len; j++) out[eat + j] = row[k][0] + j;
          }
          eat += len;
        }
      }
    });
    __syncthreads();
    count = (int)(s_found & 0xffffffffull) + s_over;
    found = (int)(s_found >> 32);
    __syncthreads();
    level++;
    unvisited -= count;
    if (found == 0 || count > kNarrowEdges || level - level0 >= kNarrowLevels) break;
  }
  if (found != 0) {
    const int p = level & 1;
    const SegQ q = p ? q1 : q0;
    unsigned* cur = bm + (size_t)((level0 + phase0) % 3) * words;  // empty since the entry
    for (int i = tid; i < found; i += kFinBlock) {
      const int v = s_vert[i];
      const int vb = nindex[v], ve = nindex[v + 1];
      atomicOr(&cur[v >> 5], 1u << (v & 31));
      const int c = chunks_of(ve - vb);
      const int at = atomicAdd(&s_chunks, c);
      for (int k = 0; k < c; k++) {
        const int x = vb + k * kChunk;
        q.base[at + k] = Entry{v, x, (x + kChunk < ve) ? x + kChunk : ve, 0};
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    ctl->iter += level - level0;
    ctl->level = level;
    ctl->bm_phase = (phase0 + 2 * (level - level0)) % 3;  // level + bm_phase stays the same modulo 3
    ctl->edges_unvisited = unvisited;
    ctl->edges_next = count;
    ctl->done = (found == 0) ? 1 : 0;
    ctl->mode = (count > kNarrowEdges && count > unvisited / kAlpha) ? 1 : 0;
    ctl_groups(ctl)[0].qcount[level & 1] = s_chunks;
    set_active();
  }
}

// ------------------------------------------------------------ host side ----
struct Bufs {
  int* wl0;
  int* wl1;
  int* stamp;
};

template <typename K>
int run_topo(const igx_graph* g, int src, int* d_dist, igx_run_info* info, int grid, long long max_rounds,
             K kernel_launch)
{
  Runtime& R = rt();
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(bfs_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, src, d_dist, g->nodes);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        kernel_launch(grid);
        launch_fin_flag();
      },
      max_rounds, &rounds, &launches);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

template <int G, int AK, bool DETERM, bool PERSIST>
int style_vtopo_push(const igx_graph* g, int src, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* dist = (int*)out;
  int grid = R.persist_blocks;
  if (!PERSIST) {
    grid = (G == kThread) ? blocks_for(g->nodes, kBlock)
                          : (G == kWaveG ? blocks_for(g->nodes, kWavesPerBlock) : g->nodes);
  }
  return run_topo(g, src, dist, info, grid, (long long)g->nodes + 2,
                  [&](int gr) {
                    hipLaunchKernelGGL((bfs_vtopo_push<G, AK, DETERM, PERSIST>), dim3(gr), dim3(kBlock), 0, R.stream,
                                       g->nindex, g->nlist, g->nodes, dist, R.d_ctl);
                  });
}

template <int G>
int style_vtopo_pull(const igx_graph* g, int src, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* dist = (int*)out;
  return run_topo(g, src, dist, info, R.persist_blocks, (long long)g->nodes + 2,
                  [&](int gr) {
                    hipLaunchKernelGGL((bfs_vtopo_pull<G>), dim3(gr), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                                       g->nodes, dist, R.d_ctl);
                  });
}

template <int AK>
int style_etopo_push(const igx_graph* g, int src, void* out, const void* aux, igx_run_info* info)
{
  Runtime& R = rt();
  int* dist = (int*)out;
  const int* sp = (const int*)aux;
  return run_topo(g, src, dist, info, R.persist_blocks, (long long)g->nodes + 2,
                  [&](int gr) {
                    hipLaunchKernelGGL((bfs_etopo_push<AK>), dim3(gr), dim3(kBlock), 0, R.stream, g->nlist, sp,
                                       g->edges, dist, R.d_ctl);
                  });
}

int get_worklists(size_t items, size_t stamp_items, Bufs* b)
{
  void* p = nullptr;
  IGX_TRY(ws_get(WS_A, sizeof(int) * items, &p));
  b->wl0 = (int*)p;
  IGX_TRY(ws_get(WS_B, sizeof(int) * items, &p));
  b->wl1 = (int*)p;
  IGX_TRY(ws_get(WS_C, sizeof(int) * stamp_items, &p));
  b->stamp = (int*)p;
  return IGX_OK;
}

template <int G>
int style_vdata_push(const igx_graph* g, int src, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* dist = (int*)out;
  const size_t items = (size_t)std::max(g->edges, g->nodes);
  Bufs b;
  IGX_TRY(get_worklists(items, (size_t)g->nodes, &b));
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(bfs_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, src, dist, g->nodes);
  hipLaunchKernelGGL(fill_int, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, b.stamp, 0,
                     (long long)g->nodes);
  hipLaunchKernelGGL(bfs_vdata_init, dim3(1), dim3(64), 0, R.stream, src, b.wl0, R.d_ctl);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        hipLaunchKernelGGL((bfs_vdata_push<G>), dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex,
                           g->nlist, dist, b.wl0, b.wl1, b.stamp, R.d_ctl);
        launch_fin_worklist();
      },
      (long long)g->nodes + 2, &rounds, &launches);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

int style_edata_push(const igx_graph* g, int src, void* out, const void* aux, igx_run_info* info)
{
  Runtime& R = rt();
  int* dist = (int*)out;
  const int* sp = (const int*)aux;
  const size_t items = (size_t)std::max(g->edges, g->nodes);
  Bufs b;
  IGX_TRY(get_worklists(items, (size_t)g->nodes, &b));
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(bfs_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, src, dist, g->nodes);
  hipLaunchKernelGGL(fill_int, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, b.stamp, 0,
                     (long long)g->nodes);
  hipLaunchKernelGGL(bfs_edata_init, dim3(1), dim3(kBlock), 0, R.stream, src, g->nindex, b.wl0, R.d_ctl);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        hipLaunchKernelGGL(bfs_edata_push, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                           sp, dist, b.wl0, b.wl1, b.stamp, R.d_ctl);
        launch_fin_worklist();
      },
      (long long)g->nodes + 2, &rounds, &launches);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

int style_do_hybrid(const igx_graph* g, int src, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* dist = (int*)out;
  const long long cap = (long long)g->nodes + g->edges / kChunk + 64;  // chunks of all rows
  const int words = ((g->nodes + kWave - 1) / kWave) * 2;
  void *p0 = nullptr, *p1 = nullptr, *pb = nullptr, *pq = nullptr, *pc = nullptr;
  IGX_TRY(ws_get(WS_D, sizeof(Entry) * (size_t)cap * kGroups, &p0));
  IGX_TRY(ws_get(WS_E, sizeof(Entry) * (size_t)cap * kGroups, &p1));
  IGX_TRY(ws_get(WS_F, sizeof(unsigned) * 3 * (size_t)words, &pb));
  // chunks of the rows longer than kChunk: at most 2 * edges / kChunk
  IGX_TRY(ws_get(WS_G, sizeof(Entry) * (2 * (size_t)(g->edges / kChunk) + 64), &pq));
  IGX_TRY(ws_get(WS_H, sizeof(int) * 64, &pc));
  const SegQ q0{(Entry*)p0, cap}, q1{(Entry*)p1, cap};
  IGX_TRY(timer_start());
  hipLaunchKernelGGL(bfs_do_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, src, g->nindex,
                     g->nodes, g->edges, dist, (Entry*)p0, (unsigned*)pb, words, R.d_ctl);
  IGX_TRY(big_rows(g, pq, (int*)pc));
  auto finish = [&](bool after_level) {
    hipLaunchKernelGGL(bfs_do_finish, dim3(1), dim3(kFinBlock), 0, R.stream, g->nindex, g->nlist, dist, q0, q1,
                       (unsigned*)pb, words, R.persist_blocks, after_level, R.d_ctl);
  };
  // the timed region of a level is the level and the narrow ones that the
  // kernel that ends it runs; the first has those before it too
  ktimer_begin("bfs_do_level");
  finish(false);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        ktimer_begin("bfs_do_level");
        hipLaunchKernelGGL(bfs_do_level, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                           g->nodes, dist, q0, q1, (const Entry*)pq, (const int*)pc, (unsigned*)pb, words,
                           g->edges / 16 < g->nodes, R.d_ctl);
        finish(true);
        ktimer_end("bfs_do_level");
      },
      (long long)g->nodes + 2, &rounds, &launches, g->edges < kFewEdges ? 4 : 6);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

const StyleEntry kStyles[] = {
    {"v_topo_push_thread", style_vtopo_push<kThread, kAtomicRelaxed, false, true>, 0},
    {"v_topo_push_wave", style_vtopo_push<kWaveG, kAtomicRelaxed, false, true>, 0},
    {"v_topo_push_block", style_vtopo_push<kBlockG, kAtomicRelaxed, false, true>, 0},
    {"v_topo_push_thread_nonpersist", style_vtopo_push<kThread, kAtomicRelaxed, false, false>, 0},
    {"v_topo_push_thread_determ", style_vtopo_push<kThread, kAtomicRelaxed, true, true>, 0},
    {"v_topo_push_thread_cas", style_vtopo_push<kThread, kAtomicCas, false, true>, 0},
    {"v_topo_push_thread_seqcst", style_vtopo_push<kThread, kAtomicSeqCst, false, true>, 0},
    {"v_topo_pull_thread", style_vtopo_pull<kThread>, 0},
    {"v_topo_pull_wave", style_vtopo_pull<kWaveG>, 0},
    {"v_data_push_thread", style_vdata_push<kThread>, 0},
    {"v_data_push_wave", style_vdata_push<kWaveG>, 0},
    {"e_topo_push_thread", style_etopo_push<kAtomicRelaxed>, 1},
    {"e_data_push_thread", style_edata_push, 1},
    {"do_hybrid", style_do_hybrid, 0},
};

}  // namespace

const StyleEntry* bfs_styles(int* count)
{
  *count = (int)(sizeof(kStyles) / sizeof(kStyles[0]));
  return kStyles;
}

}  // namespace igx
