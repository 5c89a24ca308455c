// Maximal independent set on gfx950.  Priorities are the reference's hash of
// (v + 712313887) compared as UNSIGNED with ties broken toward the larger id
// (codes/omp MIS init and mis_vertex_omp.h:127-132; the CUDA variants compare
// them as signed int and produce a different set).  With fixed priorities
// every style converges to the same set: the greedy MIS in descending
// (priority, id) order.  Output: int32 status, 1 = in the set, 2 = not.
// Self loops are ignored (the reference never terminates on them).
//
// Reference family: codes/cuda/mis-cuda (112 variants), codes/omp/mis-omp.
//   v_topo_push_*  [C-MVT] MIS_CUDA_V_Topo_Push_..._Thread:45-128 / [O-MIS]
//   v_topo_pull_*  V_Topo_Pull siblings (exclude self when a neighbour is in)
//   v_data_pull_*  V_Data_Pull siblings: worklist of undecided vertices
//   e_topo_thread  [C-MET]:57-127 / [O-MISe]:52-94 edge pass + vertex pass
//   e_data_thread  [C-MED]:45-213 worklist of edges, edge pass + vertex pass
//   e_data_thread_{copy,merge}determ  MIS_OMP_E_Data_..._{Copy,Merge}Determ:
//                  the same passes over a second status buffer, published
//                  after each pass
//   v_resume_pull  (no reference counterpart) pull over the outranking
//                  neighbours only, resuming where the last round stopped
#include "igx_internal.hpp"
#include "igx_frontier.hpp"

namespace igx {
namespace {

constexpr int kUndecided = 0;
constexpr int kIncluded = 1;
constexpr int kExcluded = 2;

// u outranks v under the unsigned-priority order with id tie-break
__device__ __forceinline__ bool outranks(uint32_t pu, int u, uint32_t pv, int v)
{
  return (pu > pv) || (pu == pv && u > v);
}

__global__ void __launch_bounds__(kBlock) mis_init(int* __restrict__ status, int n)
{
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n) status[v] = kUndecided;
}

// [C-MVT] mis():56-80 with unsigned priorities
template <bool WAVE>
__global__ void __launch_bounds__(kBlock) mis_vtopo_push(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, int n,
                                                          int* __restrict__ status, Ctl* ctl)
{
  if (round_done(ctl)) return;
  bool pending = false;
  if constexpr (!WAVE) {
    const int stride = gridDim.x * kBlock;
    for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
      if (load_relaxed(&status[v]) != kUndecided) continue;
      const uint32_t pv = mis_priority(v);
      const int beg = nindex[v], end = nindex[v + 1];
      int i = beg;
      while (i < end) {
        const int u = nlist[i];
        if (u != v && load_relaxed(&status[u]) != kExcluded && outranks(mis_priority(u), u, pv, v)) break;
        i++;
      }
      if (i < end) {
        pending = true;
      } else {
        store_relaxed(&status[v], kIncluded);
        for (int j = beg; j < end; j++) {
          const int u = nlist[j];
          if (u != v) store_relaxed(&status[u], kExcluded);
        }
      }
    }
  } else {
    const int waves = gridDim.x * kWavesPerBlock;
    const int lane = lane_id();
    for (int v = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; v < n; v += waves) {
      if (load_relaxed(&status[v]) != kUndecided) continue;
      const uint32_t pv = mis_priority(v);
      const int beg = nindex[v], end = nindex[v + 1];
      bool blocked = false;
      for (int i = beg + lane; i < end; i += kWave) {
        const int u = nlist[i];
        if (u != v && load_relaxed(&status[u]) != kExcluded && outranks(mis_priority(u), u, pv, v)) blocked = true;
      }
      if (ballot(blocked) != 0) {
        if (lane == 0) pending = true;
      } else {
        if (lane == 0) store_relaxed(&status[v], kIncluded);
        for (int j = beg + lane; j < end; j += kWave) {
          const int u = nlist[j];
          if (u != v) store_relaxed(&status[u], kExcluded);
        }
      }
    }
  }
  raise_flag(ctl, pending);
}

// pull: a vertex excludes itself when a neighbour is in the set and includes
// itself when every outranking neighbour is excluded
__device__ __forceinline__ int mis_pull_decide(const int* __restrict__ nindex, const int* __restrict__ nlist,
                                               const int* __restrict__ status, int v)
{
  const uint32_t pv = mis_priority(v);
  bool best = true;
  for (int i = nindex[v]; i < nindex[v + 1]; i++) {
    const int u = nlist[i];
    if (u == v) continue;
    const int su = load_relaxed(&status[u]);
    if (su == kIncluded) return kExcluded;
    if (su != kExcluded && outranks(mis_priority(u), u, pv, v)) best = false;
  }
  return best ? kIncluded : kUndecided;
}

__global__ void __launch_bounds__(kBlock) mis_vtopo_pull(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, int n,
                                                          int* __restrict__ status, Ctl* ctl)
{
  if (round_done(ctl)) return;
  bool pending = false;
  const int stride = gridDim.x * kBlock;
  for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
    if (load_relaxed(&status[v]) != kUndecided) continue;
    const int d = mis_pull_decide(nindex, nlist, status, v);
    if (d == kUndecided) pending = true;
    else store_relaxed(&status[v], d);
  }
  raise_flag(ctl, pending);
}

__global__ void __launch_bounds__(kBlock) mis_seed(int* __restrict__ wl, int n, Ctl* ctl)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) wl[i] = i;
  if (i == 0) {
    ctl->wl_count[0] = n;
    ctl->wl_count[1] = 0;
  }
}

__global__ void __launch_bounds__(kBlock) mis_vdata_pull(const int* __restrict__ nindex,
                                                          const int* __restrict__ nlist, int* __restrict__ status,
                                                          int* __restrict__ wl0, int* __restrict__ wl1, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int p = ctl->iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  int* wl_out = p ? wl0 : wl1;
  int* out_count = &ctl->wl_count[p ^ 1];
  const int stride = gridDim.x * kBlock;
  for (int base = blockIdx.x * kBlock; base < count; base += stride) {
    const int idx = base + threadIdx.x;
    bool keep = false;
    int v = 0;
    if (idx < count) {
      v = wl_in[idx];
      if (load_relaxed(&status[v]) == kUndecided) {
        const int d = mis_pull_decide(nindex, nlist, status, v);
        if (d == kUndecided) keep = true;
        else store_relaxed(&status[v], d);
      }
    }
    const int slot = wave_push_slot(out_count, keep);
    if (keep) wl_out[slot] = v;
  }
}

// [O-MISe]:52-77 edge pass: exclude the neighbours of included vertices and
// mark the lower-ranked endpoint of an undecided pair as lost
__global__ void __launch_bounds__(kBlock) mis_edge_pass(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                         int m, int* __restrict__ status, int* __restrict__ lost,
                                                         Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int stride = gridDim.x * kBlock;
  for (int e = blockIdx.x * kBlock + threadIdx.x; e < m; e += stride) {
    const int src = sp[e];
    const int dst = nlist[e];
    if (src == dst) continue;
    const int ss = load_relaxed(&status[src]);
    const int sd = load_relaxed(&status[dst]);
    if (ss == kIncluded) {
      store_relaxed(&status[dst], kExcluded);
    } else if (sd == kIncluded) {
      store_relaxed(&status[src], kExcluded);
    } else if (ss != kExcluded && sd != kExcluded) {
      const bool dst_wins = outranks(mis_priority(dst), dst, mis_priority(src), src);
      store_relaxed(&lost[dst_wins ? src : dst], 1);
    }
  }
}

// [O-MISe]:79-94 vertex pass: include every undecided vertex that did not lose
__global__ void __launch_bounds__(kBlock) mis_vertex_pass(int n, int* __restrict__ status, int* __restrict__ lost,
                                                           Ctl* ctl)
{
  if (round_done(ctl)) return;
  bool pending = false;
  const int stride = gridDim.x * kBlock;
  for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
    if (lost[v] == 0) {
      if (status[v] == kUndecided) status[v] = kIncluded;
    } else {
      pending = true;
      lost[v] = 0;
    }
  }
  raise_flag(ctl, pending);
}

// ------------------------------------------------------ edge, data-driven ----
// [C-MED] init():45-62, mis():64-91, mis_vertex_pass():93-126,
// mis_last_pass():128-137: a worklist of edges, each
// undirected edge once (src < dst), shrinks as both endpoints get decided.
// Per round an edge pass excludes the other endpoint of an included vertex and
// marks the lower-ranked endpoint of an undecided pair as lost; a vertex pass
// over the same edges includes every undecided endpoint that did not lose and
// keeps the edges that still have an undecided endpoint.  A vertex left
// undecided at the end has no edge to anyone else and joins.
//
// `lost` holds the number of the round in which a vertex lost (rounds count
// from 1), so it never needs clearing; the reference clears a 0/1 flag array
// every round.  Statuses use one array, as in the topology-driven edge style:
// an edge pass sees every inclusion of earlier rounds (the kernel boundary
// publishes them) and, within the pass, a stale "undecided" only adds a lost
// mark, which delays a vertex by a round and never decides one wrongly.  The
// worklist never holds an edge twice, so the reference's per-edge time stamps
// that suppress duplicate pushes are not needed.
__global__ void __launch_bounds__(kBlock) mis_edata_seed(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                          int m, int* __restrict__ wl, Ctl* ctl)
{
  const int stride = gridDim.x * kBlock;
  for (int base = blockIdx.x * kBlock; base < m; base += stride) {  // uniform per wave
    const int e = base + threadIdx.x;
    const bool keep = e < m && sp[e] < nlist[e];
    const int slot = wave_push_slot(&ctl->wl_count[0], keep);
    if (keep) wl[slot] = e;
  }
}

__global__ void __launch_bounds__(kBlock) mis_edata_edge(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                          int* __restrict__ status, int* __restrict__ lost,
                                                          const int* __restrict__ wl0, const int* __restrict__ wl1,
                                                          Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int p = ctl->iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  const int stamp = ctl->iter + 1;
  const int stride = gridDim.x * kBlock;
  for (int idx = blockIdx.x * kBlock + threadIdx.x; idx < count; idx += stride) {
    const int e = wl_in[idx];
    const int src = sp[e];
    const int dst = nlist[e];
    const int ss = status[src];
    const int sd = status[dst];
    if (ss == kIncluded) {
      status[dst] = kExcluded;
    } else if (sd == kIncluded) {
      status[src] = kExcluded;
    } else if (ss == kUndecided && sd == kUndecided) {
      const bool dst_wins = outranks(mis_priority(dst), dst, mis_priority(src), src);
      lost[dst_wins ? src : dst] = stamp;
    }
  }
}

__global__ void __launch_bounds__(kBlock) mis_edata_vertex(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                            int* __restrict__ status, const int* __restrict__ lost,
                                                            int* __restrict__ wl0, int* __restrict__ wl1, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int p = ctl->iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  int* wl_out = p ? wl0 : wl1;
  int* out_count = &ctl->wl_count[p ^ 1];
  const int stamp = ctl->iter + 1;
  const int stride = gridDim.x * kBlock;
  for (int base = blockIdx.x * kBlock; base < count; base += stride) {  // uniform per wave
    const int idx = base + threadIdx.x;
    bool keep = false;
    int e = 0;
    if (idx < count) {
      e = wl_in[idx];
      const int src = sp[e];
      const int dst = nlist[e];
      const int ss = status[src];
      const int sd = status[dst];
      if (ss == kUndecided && lost[src] != stamp) status[src] = kIncluded;
      if (sd == kUndecided && lost[dst] != stamp) status[dst] = kIncluded;
      keep = ss == kUndecided || sd == kUndecided;
    }
    const int slot = wave_push_slot(out_count, keep);
    if (keep) wl_out[slot] = e;
  }
}

__global__ void __launch_bounds__(kBlock) mis_edata_last(int* __restrict__ status, int n)
{
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n && status[v] == kUndecided) status[v] = kIncluded;
}

// Determ forms of the edge worklist style: MIS_OMP_E_Data_IntType_Atomic_
// CopyDeterm_Default_NoFieldBug.cpp OMPmis_edge() and its MergeDeterm sibling
// (include/mis_edge_omp.h:151-163 updateFromWorklist).  Each pass reads
// `status` only and writes its decisions into `status_n`; a publish kernel
// after the pass copies them to `status`: every vertex (Copy), or the
// endpoints of the round's worklist edges, the only vertices a pass can
// change (Merge).  No read in a pass sees a write of the same pass, so every
// round's decisions are fixed by the round before.  status_n equals status
// at the start of every pass.
__global__ void __launch_bounds__(kBlock) mis_determ_edge(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                           const int* __restrict__ status,
                                                           int* __restrict__ status_n, int* __restrict__ lost,
                                                           const int* __restrict__ wl0, const int* __restrict__ wl1,
                                                           Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int p = ctl->iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  const int stamp = ctl->iter + 1;
  const int stride = gridDim.x * kBlock;
  for (int idx = blockIdx.x * kBlock + threadIdx.x; idx < count; idx += stride) {
    const int e = wl_in[idx];
    const int src = sp[e];
    const int dst = nlist[e];
    const int ss = status[src];
    const int sd = status[dst];
    if (ss == kIncluded) {
      status_n[dst] = kExcluded;
    } else if (sd == kIncluded) {
      status_n[src] = kExcluded;
    } else if (ss == kUndecided && sd == kUndecided) {
      const bool dst_wins = outranks(mis_priority(dst), dst, mis_priority(src), src);
      lost[dst_wins ? src : dst] = stamp;
    }
  }
}

__global__ void __launch_bounds__(kBlock) mis_determ_vertex(const int* __restrict__ nlist, const int* __restrict__ sp,
                                                             const int* __restrict__ status,
                                                             int* __restrict__ status_n, const int* __restrict__ lost,
                                                             int* __restrict__ wl0, int* __restrict__ wl1, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int p = ctl->iter & 1;
  const int count = ctl->wl_count[p];
  const int* wl_in = p ? wl1 : wl0;
  int* wl_out = p ? wl0 : wl1;
  int* out_count = &ctl->wl_count[p ^ 1];
  const int stamp = ctl->iter + 1;
  const int stride = gridDim.x * kBlock;
  for (int base = blockIdx.x * kBlock; base < count; base += stride) {  // uniform per wave
    const int idx = base + threadIdx.x;
    bool keep = false;
    int e = 0;
    if (idx < count) {
      e = wl_in[idx];
      const int src = sp[e];
      const int dst = nlist[e];
      const int ss = status[src];
      const int sd = status[dst];
      if (ss == kUndecided && lost[src] != stamp) status_n[src] = kIncluded;
      if (sd == kUndecided && lost[dst] != stamp) status_n[dst] = kIncluded;
      keep = ss == kUndecided || sd == kUndecided;
    }
    const int slot = wave_push_slot(out_count, keep);
    if (keep) wl_out[slot] = e;
  }
}

// status <- status_n after a pass: all n vertices (Copy) or the endpoints of
// the round's input worklist edges (Merge)
template <bool MERGE>
__global__ void __launch_bounds__(kBlock) mis_determ_publish(const int* __restrict__ nlist,
                                                              const int* __restrict__ sp,
                                                              const int* __restrict__ status_n,
                                                              int* __restrict__ status, int n,
                                                              const int* __restrict__ wl0,
                                                              const int* __restrict__ wl1, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int stride = gridDim.x * kBlock;
  if constexpr (MERGE) {
    const int p = ctl->iter & 1;
    const int count = ctl->wl_count[p];
    const int* wl_in = p ? wl1 : wl0;
    for (int idx = blockIdx.x * kBlock + threadIdx.x; idx < count; idx += stride) {
      const int e = wl_in[idx];
      const int src = sp[e];
      const int dst = nlist[e];
      status[src] = status_n[src];
      status[dst] = status_n[dst];
    }
  } else {
    for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) status[v] = status_n[v];
  }
}

// ------------------------------------------------------- resumable pull ----
// Only the neighbours that outrank v matter for v joining the set: v joins
// once all of them are excluded.  A vertex that joins excludes all its
// neighbours itself (a push: plain stores, every one of them is either
// lower-ranked, and so cannot join while v is undecided or in, or already
// excluded), so an undecided vertex only has to wait: it walks its
// outranking neighbours in list order and stops at the first one that is not
// excluded (in the set -> v is excluded; undecided -> v waits).  Where it
// stopped is kept in pos[v] (every outranking neighbour before it is excluded,
// which is final), so later rounds resume there instead of rescanning.
// Statuses are read and written with plain loads and stores, not agent-scope
// atomics (on gfx950 those bypass the XCD's L2 and made the first round 8x
// slower): a status only ever moves from undecided to in or out, so a stale
// read can only say "undecided", and then v waits a round; every decision is
// taken on a value that was true.  The kernel boundary publishes the round.
// A round is bound by chains of dependent gathers (row, neighbours, their
// statuses), so they are kept short and wide: a vertex a lane, its first
// kMisFirst neighbours at once, then kMisStep at once up to kMisLane; what is
// longer is finished by the whole wave, 64 neighbours per step.  The
// neighbours of the vertices that joined are excluded over the concatenated
// rows of the wave's vertices (owner by binary search in LDS), so no lane
// pushes a row by itself; rows of more than kMisPush edges go to a list of
// pieces that all waves share at the start of the next round (a hub that joins
// would keep one wave busy for the rest of its round), which is early enough,
// since a neighbour that has not been told meets the hub in its own walk.  The
// fixed point is the same greedy set; only the round in which a vertex is
// decided can differ from the full-scan styles.  R-MAT 22: 1.28 -> 0.59 ms;
// Erdos-Renyi n = 1 M, average degree 16: 1.31 -> 0.25 ms, of which about 0.9
// ms was the waves' stores to the flag (raise_flag).  Handing the tiles out by
// counters (0.75-1.2 ms on R-MAT 22), tiles mixed from four quarters of the
// graph (0.61) and two or four tiles a step (0.65, 0.80) measured slower.
constexpr int kMisLane = 32;
constexpr int kMisFirst = 4;
constexpr int kMisStep = 8;
constexpr int kMisPush = 1024;

// End of a round: the flag rule, and the list of pieces it consumed is empty.
// On a dense graph up to kMisNow new pieces are worked off here, before the next
// round and not beside it, whose walks meet the row's neighbours everywhere:
// those that pass before the pieces do go the long way or wait a round more (a
// clique of 2000: 3 rounds, 196 us -> 2 rounds, 69 us; Erdos-Renyi n = 4096,
// average degree 1500: 11 rounds, 257 us -> 6 rounds, 154 us).  On a sparse
// graph a row covers little of it and the next round's waves are the better
// place (R-MAT 20 275 us, 285 here); so are they for many pieces.
constexpr int kMisNow = 16;
constexpr int kMisDense = 256;  // average degree of a dense graph
__global__ void __launch_bounds__(kFinBlock) mis_resume_end(const int* __restrict__ nlist, int* __restrict__ status,
                                                             const Entry* __restrict__ push0,
                                                             const Entry* __restrict__ push1, bool dense, Ctl* ctl)
{
  if (round_done(ctl)) return;
  const int p = ctl->iter & 1;
  const int pieces = ctl->wl_count[p ^ 1];
  const bool now = dense && pieces <= kMisNow;
  if (now) {
    static_assert(kFinBlock == kMisPush, "a piece a step");
    const Entry* push = p ? push0 : push1;
    #pragma unroll 4
    for (int k = 0; k < pieces; k++) {
      const Entry en = push[k];
      const int j = en.beg + (int)threadIdx.x;
      const int u = (j < en.end) ? nlist[j] : en.v;
      if (u != en.v) status[u] = kExcluded;
    }
  }
  __syncthreads();  // the control block has been read by all
  if (threadIdx.x != 0) return;
  ctl->wl_count[p] = 0;
  if (now) ctl->wl_count[p ^ 1] = 0;
  finalize_flag_round(ctl);
}

__global__ void __launch_bounds__(kBlock) mis_resume_init(const int* __restrict__ nindex, int* __restrict__ status,
                                                           int* __restrict__ pos, int n)
{
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n) {
    status[v] = kUndecided;
    pos[v] = nindex[v];
  }
}

__global__ void __launch_bounds__(kBlock) mis_resume_pull(const int* __restrict__ nindex,
                                                           const int* __restrict__ nlist, int n,
                                                           int* status, int* __restrict__ pos,
                                                           Entry* __restrict__ push0, Entry* __restrict__ push1,
                                                           Ctl* ctl)
{
  __shared__ int s_excl[kWavesPerBlock][kWave];
  __shared__ int s_beg[kWavesPerBlock][kWave];
  __shared__ int s_own[kWavesPerBlock][kWave];
  if (round_done(ctl)) return;
  const int lane = lane_id();
  const int w = threadIdx.x / kWave;
  int* excl = s_excl[w];
  int* rbeg = s_beg[w];
  int* rown = s_own[w];
  const int gw = blockIdx.x * kWavesPerBlock + w;
  const int nwaves = gridDim.x * kWavesPerBlock;
  const int p = ctl->iter & 1;
  const Entry* push_in = p ? push1 : push0;
  Entry* push_out = p ? push0 : push1;
  int* push_count = &ctl->wl_count[p ^ 1];
  const int pieces = ctl->wl_count[p];
  for (int k = gw; k < pieces; k += nwaves) {  // uniform per wave
    const Entry en = push_in[k];
    #pragma unroll 4
    for (int j = en.beg + lane; j < en.end; j += kWave) {
      const int u = nlist[j];
      if (u != en.v) status[u] = kExcluded;
    }
  }
  bool pending = false;
  const int ntiles = (n + kWave - 1) / kWave;
  for (int tile = gw; tile < ntiles; tile += nwaves) {  // uniform
    const long long vl = (long long)tile * kWave + lane;
    const int v = (vl < n) ? (int)vl : n;  // n: no vertex
    const bool undec = v < n && status[v] == kUndecided;
    if (ballot(undec) == 0) continue;
    const uint32_t pv = mis_priority((uint32_t)v);
    int i = undec ? pos[v] : 0;
    const int end = undec ? nindex[v + 1] : 0;
    int result = kUndecided;
    bool walk = undec, more = false;
    {
      int nb[kMisFirst], su[kMisFirst];
      #pragma unroll
      for (int k = 0; k < kMisFirst; k++) nb[k] = (i + k < end) ? nlist[i + k] : -1;
      #pragma unroll
      for (int k = 0; k < kMisFirst; k++) {
        const int u = nb[k];
        const bool above = u >= 0 && u != v && outranks(mis_priority((uint32_t)u), u, pv, v);
        su[k] = above ? status[u] : kExcluded;
      }
      int go = kMisFirst;
      #pragma unroll
      for (int k = kMisFirst - 1; k >= 0; k--) {
        if (su[k] != kExcluded) {
          go = k;
          result = (su[k] == kIncluded) ? kExcluded : kUndecided;  // in the set, or v waits for it
          walk = false;
        }
      }
      i = min(i + go, end);
      if (walk && i >= end) {
        result = kIncluded;
        walk = false;
      }
    }
    if (walk) {
      const int stop = min(end, i + kMisLane);
      bool waits = false;
      while (i < stop && result == kUndecided && !waits) {
        int u[kMisStep], x[kMisStep];
        #pragma unroll
        for (int k = 0; k < kMisStep; k++) u[k] = (i + k < stop) ? nlist[i + k] : v;
        #pragma unroll
        for (int k = 0; k < kMisStep; k++) {
          const bool above = u[k] != v && outranks(mis_priority((uint32_t)u[k]), u[k], pv, v);
          x[k] = above ? status[u[k]] : kExcluded;
        }
        int go = kMisStep;
        #pragma unroll
        for (int k = kMisStep - 1; k >= 0; k--) {
          if (x[k] != kExcluded) {
            go = k;
            result = (x[k] == kIncluded) ? kExcluded : kUndecided;
            waits = x[k] == kUndecided;
          }
        }
        i = min(i + go, stop);
      }
      if (result == kUndecided && !waits && i >= end) result = kIncluded;
      more = result == kUndecided && !waits;
    }
    for (uint64_t todo = ballot(more); todo != 0; todo &= todo - 1) {
      const int L = __ffsll((unsigned long long)todo) - 1;
      const int vL = __shfl(v, L, kWave);
      const uint32_t pvL = mis_priority((uint32_t)vL);
      const int s0 = __shfl(i, L, kWave), e0 = __shfl(end, L, kWave);
      int r = kIncluded, stop = e0;
      for (int i0 = s0; i0 < e0; i0 += kWave) {
        const int idx = i0 + lane;
        int x = kExcluded;
        if (idx < e0) {
          const int u = nlist[idx];
          if (u != vL && outranks(mis_priority((uint32_t)u), u, pvL, vL)) x = status[u];
        }
        const uint64_t hit = ballot(x != kExcluded);
        if (hit != 0) {
          const int first = __ffsll((unsigned long long)hit) - 1;
          r = (__shfl(x, first, kWave) == kIncluded) ? kExcluded : kUndecided;
          stop = i0 + first;
          break;
        }
      }
      if (lane == L) {
        result = r;
        i = stop;
      }
    }
    if (undec) {
      if (result != kUndecided) {
        status[v] = result;
      } else {
        pos[v] = i;
        pending = true;
      }
    }
    // a vertex that joined excludes its neighbours
    const bool joined = undec && result == kIncluded;
    if (ballot(joined) == 0) continue;
    const int rb = joined ? nindex[v] : 0;
    int len = joined ? end - rb : 0;
    if (len > kMisPush) {
      const int c = (len + kMisPush - 1) / kMisPush;
      const int slot = atomicAdd(push_count, c);
      for (int k = 0; k < c; k++) {
        const int b = rb + k * kMisPush;
        push_out[slot + k] = Entry{v, b, min(b + kMisPush, end), 0};
      }
      len = 0;
    }
    const int incl = wave_incl_scan(len);
    const int total = wave_bcast(incl, kWave - 1);
    __builtin_amdgcn_wave_barrier();
    excl[lane] = incl - len;
    rbeg[lane] = rb;
    rown[lane] = v;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    constexpr int kIlp = 4;
    for (int tb = 0; tb < total; tb += kIlp * kWave) {
      int u[kIlp], own[kIlp];
      #pragma unroll
      for (int k = 0; k < kIlp; k++) {
        const int t = tb + k * kWave + lane;
        u[k] = own[k] = 0;
        if (t < total) {
          int lo = 0, hi = kWave;
          while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (excl[mid] <= t) lo = mid;
            else hi = mid;
          }
          u[k] = nlist[rbeg[lo] + (t - excl[lo])];
          own[k] = rown[lo];
        }
      }
      #pragma unroll
      for (int k = 0; k < kIlp; k++) {
        if (tb + k * kWave + lane < total && u[k] != own[k]) status[u[k]] = kExcluded;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  raise_flag(ctl, pending);
}

// ------------------------------------------------------------ host side ----
// worklist: the round ends by the data-driven rule, else by the flag rule
template <typename K>
int mis_rounds(const igx_graph* g, igx_run_info* info, K launch, bool worklist = false)
{
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        launch();
        if (worklist) launch_fin_worklist();
        else launch_fin_flag();
      },
      (long long)g->nodes + 2, &rounds, &launches);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

template <bool WAVE>
int style_vtopo_push(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, status, g->nodes);
  return mis_rounds(g, info, [&] {
    hipLaunchKernelGGL((mis_vtopo_push<WAVE>), dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex,
                       g->nlist, g->nodes, status, R.d_ctl);
  });
}

int style_vtopo_pull(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, status, g->nodes);
  return mis_rounds(g, info, [&] {
    hipLaunchKernelGGL(mis_vtopo_pull, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                       g->nodes, status, R.d_ctl);
  });
}

int style_vdata_pull(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  void *p0 = nullptr, *p1 = nullptr;
  IGX_TRY(ws_get(WS_A, sizeof(int) * (size_t)g->nodes, &p0));
  IGX_TRY(ws_get(WS_B, sizeof(int) * (size_t)g->nodes, &p1));
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, status, g->nodes);
  hipLaunchKernelGGL(mis_seed, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, (int*)p0, g->nodes,
                     R.d_ctl);
  return mis_rounds(g, info, [&] {
    ktimer_begin("mis_vdata_pull");
    hipLaunchKernelGGL(mis_vdata_pull, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                       status, (int*)p0, (int*)p1, R.d_ctl);
    ktimer_end("mis_vdata_pull");
  }, true);
}

int style_resume_pull(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  void *pp = nullptr, *p0 = nullptr, *p1 = nullptr;
  // pieces of rows longer than kMisPush: fewer than 2 * edges / kMisPush
  const size_t cap = 2 * ((size_t)g->edges / kMisPush) + 64;
  IGX_TRY(ws_get(WS_A, sizeof(int) * (size_t)g->nodes, &pp));
  IGX_TRY(ws_get(WS_B, sizeof(Entry) * cap, &p0));
  IGX_TRY(ws_get(WS_C, sizeof(Entry) * cap, &p1));
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(mis_resume_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, g->nindex, status,
                     (int*)pp, g->nodes);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        ktimer_begin("mis_resume_pull");
        hipLaunchKernelGGL(mis_resume_pull, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                           g->nodes, status, (int*)pp, (Entry*)p0, (Entry*)p1, R.d_ctl);
        ktimer_end("mis_resume_pull");
        hipLaunchKernelGGL(mis_resume_end, dim3(1), dim3(kFinBlock), 0, R.stream, g->nlist, status, (const Entry*)p0,
                           (const Entry*)p1, g->edges / kMisDense >= g->nodes, R.d_ctl);
      },
      (long long)g->nodes + 2, &rounds, &launches, 6);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

int style_etopo(const igx_graph* g, int, void* out, const void* aux, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  const int* sp = (const int*)aux;
  void* pl = nullptr;
  IGX_TRY(ws_get(WS_A, sizeof(int) * (size_t)g->nodes, &pl));
  int* lost = (int*)pl;
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, status, g->nodes);
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, lost, g->nodes);
  return mis_rounds(g, info, [&] {
    hipLaunchKernelGGL(mis_edge_pass, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nlist, sp, g->edges,
                       status, lost, R.d_ctl);
    hipLaunchKernelGGL(mis_vertex_pass, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nodes, status, lost,
                       R.d_ctl);
  });
}

int style_edata(const igx_graph* g, int, void* out, const void* aux, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  const int* sp = (const int*)aux;
  const size_t wl_items = (size_t)(g->edges > 0 ? g->edges : 1);
  void *pl = nullptr, *p0 = nullptr, *p1 = nullptr;
  IGX_TRY(ws_get(WS_A, sizeof(int) * (size_t)g->nodes, &pl));
  IGX_TRY(ws_get(WS_B, sizeof(int) * wl_items, &p0));
  IGX_TRY(ws_get(WS_C, sizeof(int) * wl_items, &p1));
  int* lost = (int*)pl;
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, status, g->nodes);
  hipLaunchKernelGGL(mis_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, lost, g->nodes);
  hipLaunchKernelGGL(mis_edata_seed, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nlist, sp, g->edges,
                     (int*)p0, R.d_ctl);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        hipLaunchKernelGGL(mis_edata_edge, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nlist, sp, status,
                           lost, (const int*)p0, (const int*)p1, R.d_ctl);
        hipLaunchKernelGGL(mis_edata_vertex, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nlist, sp,
                           status, (const int*)lost, (int*)p0, (int*)p1, R.d_ctl);
        launch_fin_worklist();
      },
      (long long)g->nodes + 2, &rounds, &launches);
  hipLaunchKernelGGL(mis_edata_last, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, status,
                     g->nodes);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

template <bool MERGE>
int style_edata_determ(const igx_graph* g, int, void* out, const void* aux, igx_run_info* info)
{
  Runtime& R = rt();
  int* status = (int*)out;
  const int* sp = (const int*)aux;
  const size_t wl_items = (size_t)(g->edges > 0 ? g->edges : 1);
  void *pl = nullptr, *p0 = nullptr, *p1 = nullptr, *pn = nullptr;
  IGX_TRY(ws_get(WS_A, sizeof(int) * (size_t)g->nodes, &pl));
  IGX_TRY(ws_get(WS_B, sizeof(int) * wl_items, &p0));
  IGX_TRY(ws_get(WS_C, sizeof(int) * wl_items, &p1));
  IGX_TRY(ws_get(WS_D, sizeof(int) * (size_t)g->nodes, &pn));
  int* lost = (int*)pl;
  int* status_n = (int*)pn;
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  const dim3 vb(blocks_for(g->nodes, kBlock));
  hipLaunchKernelGGL(mis_init, vb, dim3(kBlock), 0, R.stream, status, g->nodes);
  hipLaunchKernelGGL(mis_init, vb, dim3(kBlock), 0, R.stream, status_n, g->nodes);
  hipLaunchKernelGGL(mis_init, vb, dim3(kBlock), 0, R.stream, lost, g->nodes);
  hipLaunchKernelGGL(mis_edata_seed, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nlist, sp, g->edges,
                     (int*)p0, R.d_ctl);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        const dim3 grid(R.persist_blocks), blk(kBlock);
        hipLaunchKernelGGL(mis_determ_edge, grid, blk, 0, R.stream, g->nlist, sp, (const int*)status, status_n, lost,
                           (const int*)p0, (const int*)p1, R.d_ctl);
        hipLaunchKernelGGL((mis_determ_publish<MERGE>), grid, blk, 0, R.stream, g->nlist, sp,
                           (const int*)status_n, status, g->nodes, (const int*)p0, (const int*)p1, R.d_ctl);
        hipLaunchKernelGGL(mis_determ_vertex, grid, blk, 0, R.stream, g->nlist, sp, (const int*)status, status_n,
                           (const int*)lost, (int*)p0, (int*)p1, R.d_ctl);
        hipLaunchKernelGGL((mis_determ_publish<MERGE>), grid, blk, 0, R.stream, g->nlist, sp,
                           (const int*)status_n, status, g->nodes, (const int*)p0, (const int*)p1, R.d_ctl);
        launch_fin_worklist();
      },
      (long long)g->nodes + 2, &rounds, &launches);
  hipLaunchKernelGGL(mis_edata_last, vb, dim3(kBlock), 0, R.stream, status, g->nodes);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  return rc;
}

const StyleEntry kStyles[] = {
    {"v_topo_push_thread", style_vtopo_push<false>, 0},
    {"v_topo_push_wave", style_vtopo_push<true>, 0},
    {"v_topo_pull_thread", style_vtopo_pull, 0},
    {"v_data_pull_thread", style_vdata_pull, 0},
    {"e_topo_thread", style_etopo, 1},
    {"v_resume_pull", style_resume_pull, 0},
    {"e_data_thread", style_edata, 1},
    {"e_data_thread_copydeterm", style_edata_determ<false>, 1},
    {"e_data_thread_mergedeterm", style_edata_determ<true>, 1},
};

}  // namespace

const StyleEntry* mis_styles(int* count)
{
  *count = (int)(sizeof(kStyles) / sizeof(kStyles[0]));
  return kStyles;
}

}  // namespace igx
