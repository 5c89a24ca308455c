// Frontier machinery shared by the data-driven kernels (BFS, SSSP).
//
// A frontier is a queue of edge chunks: each entry names a vertex and a range
// of at most kChunk of its edges.  Vertices with more edges are split into
// several entries when they are pushed, so the expansion below can balance
// hubs (R-MAT vertex 0 has ~1.6e5 neighbours at scale 22) across many waves.
//
// Expansion is wave-level merge path: a wave loads 64 entries, scans their
// lengths, and then walks the concatenated edge space 64 edges at a time;
// every lane finds its entry by binary search over the 64 exclusive prefixes
// kept in LDS.  All lanes stay busy regardless of the degree mix.
#pragma once

#include <type_traits>

#include "igx_device.hpp"

namespace igx {

constexpr int kChunk = 256;

struct Entry {
  int v;    // vertex owning the edges
  int beg;  // first edge (index into nlist)
  int end;  // one past the last edge
  int pad;
};

__device__ __forceinline__ int chunks_of(int deg) { return (deg + kChunk - 1) / kChunk; }

// Push the chunks of vertex v (edge range [beg, end)) into q.  Lanes with
// exactly one chunk share one wave-aggregated atomic, lanes with several
// share a second one (their runs are laid out in lane order), then all active
// lanes write the multi-chunk runs together (a hub has hundreds of chunks).
// Safe in divergent code.
__device__ __forceinline__ void push_vertex_chunks(Entry* __restrict__ q, int* counter, bool pred, int v, int beg,
                                                   int end)
{
  const int deg = end - beg;
  const int c = pred ? chunks_of(deg) : 0;
  const int slot = wave_push_slot(counter, c == 1);
  if (c == 1) q[slot] = Entry{v, beg, end, 0};
  uint64_t big = ballot(c > 1);
  if (big != 0) {
    // lane-ordered offsets of the multi-chunk runs (serial over those lanes)
    const int lane = lane_id();
    int total = 0, off = 0;
    for (uint64_t b = big; b != 0; b &= b - 1) {
      const int L = __ffsll((unsigned long long)b) - 1;
      if (lane == L) off = total;
      total += __shfl(c, L, kWave);
    }
    const int leader = __ffsll((unsigned long long)big) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(counter, total);
    base = __shfl(base, leader, kWave) + off;
    const uint64_t act = ballot(true);
    const int P = __popcll(act);
    const int r = mbcnt(act);
    while (big != 0) {
      const int L = __ffsll((unsigned long long)big) - 1;
      big &= big - 1;
      const int bv = __shfl(v, L, kWave), bb = __shfl(beg, L, kWave), be = __shfl(end, L, kWave);
      const int bbase = __shfl(base, L, kWave), bc = __shfl(c, L, kWave);
      for (int k = r; k < bc; k += P) {
        const int b = bb + k * kChunk;
        q[bbase + k] = Entry{bv, b, (b + kChunk < be) ? b + kChunk : be, 0};
      }
    }
  }
}

// ----------------------------------------------------- segmented queues ----
// A chunk queue split into kGroups segments of `cap` entries each.  Workgroup
// b appends to segment b % kGroups, whose size lives in that group's control
// slot, so pushes from the whole grid spread over kGroups counters; readers
// walk the concatenation of the segments.  Each segment can hold a full
// round's output on its own.
struct SegQ {
  Entry* base;
  long long cap;
};

__device__ __forceinline__ Entry* segq_mine(const SegQ& q) { return q.base + (long long)my_group() * q.cap; }
__device__ __forceinline__ int* segq_counter(Ctl* ctl, int parity, int seg)
{
  return &ctl_groups(ctl)[seg].qcount[parity];
}

// prefix offsets of the kGroups segment sizes (kept in registers by the reader)
struct SegPrefix {
  int pre[kGroups + 1];
};
__device__ __forceinline__ SegPrefix segq_prefix(Ctl* ctl, int parity)
{
  SegPrefix sp;
  sp.pre[0] = 0;
  #pragma unroll
  for (int g = 0; g < kGroups; g++) sp.pre[g + 1] = sp.pre[g] + load_relaxed(segq_counter(ctl, parity, g));
  return sp;
}
__device__ __forceinline__ Entry segq_at(const SegQ& q, const SegPrefix& sp, int idx)
{
  // constant indices only, so that the prefixes stay in registers
  int s = 0, base = 0;
  #pragma unroll
  for (int g = 1; g < kGroups; g++) {
    if (idx >= sp.pre[g]) {
      s = g;
      base = sp.pre[g];
    }
  }
  return q.base[(long long)s * q.cap + (idx - base)];
}

// Visit every 64-vertex tile [v0, v0 + 64) that holds at least one set bit of
// the bitmap, one wave per tile: body(v0, bit) with `bit` this lane's vertex
// v0 + lane.  A wave loads 64 words (2048 vertices) at once and skips empty
// tiles without further loads, so a sparse frontier costs one coalesced pass
// over the bitmap; a bitmap of fewer words than that gives all waves work is
// read in smaller pieces (300 k vertices are 147 pieces of 64 words for 8192
// waves: a push round took 180 us).  All lanes of the wave call this together;
// bits at or past n must be clear.
template <typename F>
__device__ __forceinline__ void for_each_bitmap_tile(const unsigned* __restrict__ bits, int n, int gw, int nwaves,
                                                     F body)
{
  const int lane = lane_id();
  const int nwords = (n + 31) >> 5;
  int piece = kWave;
  while (piece > 2 && (long long)nwaves * piece > nwords) piece >>= 1;
  for (int wb = gw * piece; wb < nwords; wb += nwaves * piece) {  // uniform
    const int wi = wb + lane;
    const unsigned word = (lane < piece && wi < nwords) ? bits[wi] : 0u;
    const uint64_t nz = ballot(word != 0u);
    uint64_t pair = (nz | (nz >> 1)) & 0x5555555555555555ull;  // even j: word j or j + 1 non-empty
    while (pair != 0) {
      const int j = __ffsll((unsigned long long)pair) - 1;
      pair &= pair - 1;
      const unsigned w0 = __shfl(word, j, kWave), w1 = __shfl(word, j + 1, kWave);
      const unsigned mine = (lane < 32) ? w0 : w1;
      body((wb + j) * 32, ((mine >> (lane & 31)) & 1u) != 0u);
    }
  }
}

// Edge worklists: a workgroup takes up to kListPer * kBlock consecutive items
// per step (fewer when the list is short, so that it still spreads over the
// grid) and appends what they queue together.  Items per thread and step:
constexpr int kListPer = 4;
__device__ __forceinline__ int list_items_per_thread(int count)
{
  const long long lanes = (long long)gridDim.x * kBlock;
  const long long per = (count + lanes - 1) / lanes;
  return (int)(per < kListPer ? (per < 1 ? 1 : per) : kListPer);
}

// The items per thread as a constant for the loops over them: body(1) for a
// short list, whose rounds are latency alone, else body(kListPer).
template <typename F>
__device__ __forceinline__ void with_list_items(int per, F body)
{
  if (per == 1) body(std::integral_constant<int, 1>{});
  else body(std::integral_constant<int, kListPer>{});
}

// Edges per thread of a narrow level or round (bfs_do_finish, sssp_do_finish),
// as a constant for the loops over them.  One workgroup's instructions are much
// of the time of such a level, so no thread goes through the loops for edges
// that are not there.
template <typename F>
__device__ __forceinline__ void with_narrow_items(int count, F body)
{
  if (count <= kFinBlock) body(std::integral_constant<int, 1>{});
  else if (count <= 2 * kFinBlock) body(std::integral_constant<int, 2>{});
  else body(std::integral_constant<int, 4>{});
}

// LDS of block_push_edge_ranges
struct ListLds {
  int excl[kWavesPerBlock][kWave];
  int beg[kWavesPerBlock][kWave];
  int total[kWavesPerBlock];
  int base;
};

// Append the edge ids [beg[k], beg[k] + len[k]) of every thread to an edge
// worklist.  One atomic per workgroup reserves the places: the counter is one
// address, where an atomic per 64 items took 11 ns each and was the time of
// the large rounds (R-MAT 20, SSSP edge worklist: 300 k of them in a round of
// 3.3 ms).  A short list (`alone`, at most kListAlone items) has few waves to
// meet there, and each reserves for itself, without the workgroup's barriers.
// Then each wave writes its ranges one k after the other, its 64 lanes
// together: those of at most kListLong ids as one concatenation, each lane
// finding its range by binary search over the exclusive prefixes in LDS, and
// longer ones one by one without a search (a hub's neighbours are the other
// hubs, in the same few waves: a million ids each on R-MAT 20, 3.3 ms of
// searches in the first round).  All threads of the workgroup call this
// together; threads with nothing to push pass len = 0.
constexpr int kListAlone = 1 << 16;
constexpr int kListLong = 256;

template <int kPer>
__device__ __forceinline__ void block_push_edge_ranges(int* __restrict__ out, int* counter, const int (&beg)[kPer],
                                                       const int (&len)[kPer], bool alone, ListLds& L)
{
  const int lane = lane_id();
  const int w = threadIdx.x / kWave;
  int incl[kPer];  // inclusive prefix of the short ranges
  int total = 0;
  #pragma unroll
  for (int k = 0; k < kPer; k++) {
    incl[k] = 0;
    if (ballot(len[k] != 0) != 0) {  // uniform per wave
      incl[k] = wave_incl_scan((len[k] <= kListLong) ? len[k] : 0);
      total += wave_bcast(incl[k], kWave - 1);
      if (ballot(len[k] > kListLong) != 0) total += wave_sum((len[k] > kListLong) ? len[k] : 0);
    }
  }
  int base = 0;
  if (alone) {
    if (total == 0) return;
    if (lane == 0) base = atomicAdd(counter, total);
    base = wave_bcast(base, 0);
  } else {
    if (lane == 0) L.total[w] = total;
    __syncthreads();
    int before = 0, all = 0;
    #pragma unroll
    for (int k = 0; k < kWavesPerBlock; k++) {
      if (k < w) before += L.total[k];
      all += L.total[k];
    }
    if (threadIdx.x == 0 && all != 0) L.base = atomicAdd(counter, all);
    __syncthreads();
    base = L.base + before;
  }
  int* excl = L.excl[w];
  int* rbeg = L.beg[w];
  #pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int sum = wave_bcast(incl[k], kWave - 1);
    if (sum != 0) {  // uniform per wave
      __builtin_amdgcn_wave_barrier();
      excl[lane] = incl[k] - ((len[k] <= kListLong) ? len[k] : 0);
      rbeg[lane] = beg[k];
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int t = lane; t < sum; t += kWave) {
        int lo = 0, hi = kWave;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (excl[mid] <= t) lo = mid;
          else hi = mid;
        }
        out[base + t] = rbeg[lo] + (t - excl[lo]);
      }
      base += sum;
      __builtin_amdgcn_wave_barrier();
    }
    for (uint64_t todo = ballot(len[k] > kListLong); todo != 0; todo &= todo - 1) {
      const int owner = __ffsll((unsigned long long)todo) - 1;
      const int b = __shfl(beg[k], owner, kWave), n = __shfl(len[k], owner, kWave);
      #pragma unroll 4
      for (int t = lane; t < n; t += kWave) out[base + t] = b + t;
      base += n;
    }
  }
  if (!alone) __syncthreads();
}

// Walk all edges of the queue entries [0, qsize) with the calling wave among
// `nwaves` waves (wave index `gw`).  lds_excl / lds_ent must point at this
// wave's 64-slot LDS arrays.  visit(ent, e) is called once per edge; all lanes
// of the wave call this function together (the loops are wave-uniform).
// Entries per wave group: 64 when the queue is long; fewer (a power of two)
// when it is short, so that a handful of hub chunks still spreads over all
// waves instead of over qsize / 64 of them.
__device__ __forceinline__ int group_entries(int qsize, int nwaves)
{
  if (qsize >= nwaves * kWave) return kWave;
  const int per = (qsize + nwaves - 1) / nwaves;
  int g = 1;
  while (g < per) g <<= 1;
  return g;
}

// Expansion over any indexable source of entries: fetch(idx) returns entry
// idx of [0, qsize); entries with end == beg are skipped at no cost.
template <typename Fetch, typename F>
__device__ __forceinline__ void wave_expand_with(int qsize, int gw, int nwaves, int* lds_excl, Entry* lds_ent,
                                                 Fetch fetch, F visit)
{
  const int lane = lane_id();
  const int G = group_entries(qsize, nwaves);
  for (int gbase = gw * G; gbase < qsize; gbase += nwaves * G) {
    const int idx = gbase + lane;
    Entry ent = Entry{0, 0, 0, 0};
    if (lane < G && idx < qsize) ent = fetch(idx);
    const int len = ent.end - ent.beg;
    const int incl = wave_incl_scan(len);
    const int total = wave_bcast(incl, kWave - 1);
    if (total == 0) continue;  // uniform
    __builtin_amdgcn_wave_barrier();
    lds_excl[lane] = incl - len;
    lds_ent[lane] = ent;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    for (int tb = 0; tb < total; tb += kWave) {
      const int t = tb + lane;
      if (t < total) {
        // last k with excl[k] <= t (zero-length entries share the next prefix)
        int lo = 0, hi = kWave;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (lds_excl[mid] <= t) lo = mid;
          else hi = mid;
        }
        const Entry& en = lds_ent[lo];
        visit(en, en.beg + (t - lds_excl[lo]));
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// The same walk with the entries dealt out round-robin: lane l of wave gw
// takes entry gw + (64 s + l) * nwaves in step s, so consecutive entries go
// to consecutive waves.  For a list in which the live entries come in long
// runs (the chunks of a few hub rows among the chunks of every long row),
// the consecutive grouping above hands a whole run to one wave; here a run
// of c chunks spreads over c waves.
template <typename Fetch, typename F>
__device__ __forceinline__ void wave_expand_strided(int qsize, int gw, int nwaves, int* lds_excl, Entry* lds_ent,
                                                    Fetch fetch, F visit)
{
  const int lane = lane_id();
  const long long step = (long long)kWave * nwaves;
  for (long long base = gw; base < qsize; base += step) {
    const long long idx = base + (long long)lane * nwaves;
    Entry ent = Entry{0, 0, 0, 0};
    if (idx < qsize) ent = fetch((int)idx);
    const int len = ent.end - ent.beg;
    const int incl = wave_incl_scan(len);
    const int total = wave_bcast(incl, kWave - 1);
    if (total == 0) continue;  // uniform
    __builtin_amdgcn_wave_barrier();
    lds_excl[lane] = incl - len;
    lds_ent[lane] = ent;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    for (int tb = 0; tb < total; tb += kWave) {
      const int t = tb + lane;
      if (t < total) {
        int lo = 0, hi = kWave;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (lds_excl[mid] <= t) lo = mid;
          else hi = mid;
        }
        const Entry& en = lds_ent[lo];
        visit(en, en.beg + (t - lds_excl[lo]));
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <typename F>
__device__ __forceinline__ void wave_expand(const Entry* __restrict__ q, int qsize, int gw, int nwaves,
                                            int* lds_excl, Entry* lds_ent, F visit)
{
  wave_expand_with(qsize, gw, nwaves, lds_excl, lds_ent, [&](int i) { return q[i]; }, visit);
}

}  // namespace igx
