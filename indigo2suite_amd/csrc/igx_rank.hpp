// Degree ranks and flat passes over the edges, shared by the kernels that
// work in degree order (triangle counting, PageRank).
//
// A vertex's rank is its place when the vertices are sorted by degree, highest
// first, by counting: three launches (histogram of degree bins, first rank of
// each bin, assignment), no sort.  Vertices of one bin are in no particular
// order, so any order of a bin must serve the caller.
//
// A flat pass gives every workgroup kEdgeTile consecutive edges, whatever the
// rows, and finds each edge's row in LDS (edge_tile_rows), so that no edge ->
// row map goes through memory.
#pragma once

#include "igx_device.hpp"
#include "igx_scan.hpp"

namespace igx {

constexpr int kEdgeTile = 2048;  // edges per workgroup of a flat pass
constexpr int kEdgePer = kEdgeTile / kBlock;
constexpr int kRankExact = 2048;  // degrees below it have a bin of their own
constexpr int kRankBins = kRankExact + 21 * 64;
constexpr int kRankRows = 4096;  // vertices per workgroup of the rank passes

// degree -> bin: exact below kRankExact, then 64 per octave.  Any order of the
// vertices within a bin is a valid order of the whole.
__device__ __forceinline__ int rank_bin(int deg)
{
  if (deg < kRankExact) return deg;
  const int e = 31 - __clz(deg);
  return kRankExact + (e - 11) * 64 + ((deg >> (e - 6)) & 63);
}

// bins[k] += vertices of bin k, and tile_row[t] = the row that holds edge
// t * kEdgeTile
static __global__ void __launch_bounds__(kBlock) rank_hist(const int* __restrict__ nindex, int n, int* __restrict__ bins,
                                                   int* __restrict__ tile_row)
{
  __shared__ int s_bin[kRankBins];
  for (int i = threadIdx.x; i < kRankBins; i += kBlock) s_bin[i] = 0;
  __syncthreads();
  const long long base = (long long)blockIdx.x * kRankRows;
  constexpr int kPer = kRankRows / kBlock;
  int b[kPer], e[kPer];  // loaded together
  #pragma unroll
  for (int k = 0; k < kPer; k++) {
    const long long v = base + k * kBlock + threadIdx.x;
    b[k] = (v < n) ? nindex[v] : 0;
    e[k] = (v < n) ? nindex[v + 1] : 0;
  }
  #pragma unroll
  for (int k = 0; k < kPer; k++) {
    const long long v = base + k * kBlock + threadIdx.x;
    if (v < n) atomicAdd(&s_bin[rank_bin(e[k] - b[k])], 1);
    for (int t = (int)(((long long)b[k] + kEdgeTile - 1) / kEdgeTile); (long long)t * kEdgeTile < e[k]; t++) {
      tile_row[t] = (int)v;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kRankBins; i += kBlock) {
    if (s_bin[i] != 0) atomicAdd(&bins[i], s_bin[i]);
  }
}

// the vertices whose bins lie whole within the first `ranks` ranks
struct RankHead {
  long long edges;   // their edges, at least
  long long degree;  // their least degree; INT_MAX: there are none
};

// bins become the first rank of each (highest degree first); *above = number
// of vertices of degree above `limit` (below kRankExact); *head, if asked for,
// describes the first `ranks` ranks.  One workgroup.
static __global__ void __launch_bounds__(kBlock) rank_bins(int* __restrict__ bins, int limit, int* __restrict__ above,
                                                            int ranks, RankHead* __restrict__ head)
{
  __shared__ int s_red[kWavesPerBlock];
  __shared__ long long s_edges[kWavesPerBlock], s_degree[kWavesPerBlock];
  constexpr int kPerT = (kRankBins + kBlock - 1) / kBlock;
  int c[kPerT];
  int local = 0;
  #pragma unroll
  for (int k = 0; k < kPerT; k++) {
    const int i = kRankBins - 1 - ((int)threadIdx.x * kPerT + k);
    c[k] = (i >= 0) ? bins[i] : 0;
    local += c[k];
  }
  int tot = 0;
  int run = block_excl_scan(local, s_red, &tot);
  long long edges = 0;  // of the head, by the least degree of each bin
  long long least = INT_MAX;
  #pragma unroll
  for (int k = 0; k < kPerT; k++) {
    const int i = kRankBins - 1 - ((int)threadIdx.x * kPerT + k);
    if (i >= 0) {
      bins[i] = run;
      const int over = i - kRankExact;
      const long long deg = (over < 0) ? i : ((long long)(64 + (over & 63)) << (5 + over / 64));
      if (c[k] > 0 && run + c[k] <= ranks) {
        edges += deg * c[k];
        least = min(least, deg);
      }
    }
    if (i == limit && above != nullptr) *above = run;
    run += c[k];
  }
  if (head == nullptr) return;
  edges = wave_sum_ll(edges);
  least = wave_min_ll(least);
  if (lane_id() == 0) {
    s_edges[threadIdx.x / kWave] = edges;
    s_degree[threadIdx.x / kWave] = least;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    RankHead h{0, INT_MAX};
    for (int k = 0; k < kWavesPerBlock; k++) {
      h.edges += s_edges[k];
      h.degree = min(h.degree, s_degree[k]);
    }
    *head = h;
  }
}

// rank[v] and its inverse order[] (and the degrees in rank order, when asked
// for): a workgroup reserves a run of ranks in each bin for its vertices.
static __global__ void __launch_bounds__(kBlock) rank_assign(const int* __restrict__ nindex, int n, int* __restrict__ bins,
                                                   int* __restrict__ rank, int* __restrict__ order,
                                                   int* __restrict__ degree)
{
  __shared__ int s_bin[kRankBins];
  if (degree != nullptr && blockIdx.x == 0 && threadIdx.x == 0) degree[n] = 0;  // closes a scan
  for (int i = threadIdx.x; i < kRankBins; i += kBlock) s_bin[i] = 0;
  __syncthreads();
  const long long base = (long long)blockIdx.x * kRankRows;
  int bin[kRankRows / kBlock];
  #pragma unroll
  for (int k = 0; k < kRankRows / kBlock; k++) {
    const long long v = base + k * kBlock + threadIdx.x;
    bin[k] = (v < n) ? rank_bin(nindex[v + 1] - nindex[v]) : 0;
    if (v < n) atomicAdd(&s_bin[bin[k]], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kRankBins; i += kBlock) {
    if (s_bin[i] != 0) s_bin[i] = atomicAdd(&bins[i], s_bin[i]);
  }
  __syncthreads();
  #pragma unroll
  for (int k = 0; k < kRankRows / kBlock; k++) {
    const long long v = base + k * kBlock + threadIdx.x;
    if (v < n) {
      const int r = atomicAdd(&s_bin[bin[k]], 1);
      rank[v] = r;
      order[r] = (int)v;
      if (degree != nullptr) degree[r] = nindex[v + 1] - nindex[v];
    }
  }
}

// s_row[i] = row of edge base + i, minus r0 (the row of edge base), for the
// tile's kEdgeTile edges: the rows that start inside the tile mark their first
// edge, and a running maximum carries each to the next.  r1: the row of the
// next tile's first edge (n - 1 for the last tile).  Between the two there may
// be any number of empty rows (the vertices that a graph keeps but does not
// use), which one workgroup would walk alone: 16 million of them after the
// edges of an R-MAT 16 took 18 ms.  So beyond kTileRows rows every edge finds
// its row by a binary search.
constexpr int kTileRows = 4 * kEdgeTile;
__device__ __forceinline__ void edge_tile_rows(const int* __restrict__ nindex, int base, int r0, int r1, int* s_row,
                                             int* s_red)
{
  const int tid = threadIdx.x;
  if (r1 - r0 > kTileRows) {  // uniform
    constexpr int kAtOnce = 4;
    #pragma unroll 1
    for (int i0 = tid; i0 < kEdgeTile; i0 += kAtOnce * kBlock) {
      int at[kAtOnce] = {};  // the last row that starts at or before the edge
      for (int len = r1 - r0 + 1; len > 1;) {
        const int half = len >> 1;
        #pragma unroll
        for (int k = 0; k < kAtOnce; k++) at[k] += (nindex[r0 + at[k] + half] <= base + i0 + k * kBlock) ? half : 0;
        len -= half;
      }
      #pragma unroll
      for (int k = 0; k < kAtOnce; k++) s_row[i0 + k * kBlock] = at[k];
    }
    __syncthreads();
    return;
  }
  for (int i = tid; i < kEdgeTile; i += kBlock) s_row[i] = 0;
  __syncthreads();
  for (int r = r0 + 1 + tid; r <= r1; r += kBlock) {
    const int p = nindex[r] - base;  // empty rows share the place of the row after them, the larger one stays
    if (p < kEdgeTile) atomicMax(&s_row[p], r - r0);
  }
  __syncthreads();
  int x[kEdgePer];
  int mx = 0;
  #pragma unroll
  for (int k = 0; k < kEdgePer; k++) {
    mx = max(mx, s_row[tid * kEdgePer + k]);
    x[k] = mx;
  }
  int incl = mx;
  #pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int t = __shfl_up(incl, d, kWave);
    if (lane_id() >= d) incl = max(incl, t);
  }
  const int w = tid / kWave;
  if (lane_id() == kWave - 1) s_red[w] = incl;
  int before = __shfl_up(incl, 1, kWave);
  if (lane_id() == 0) before = 0;
  __syncthreads();
  for (int k = 0; k < w; k++) before = max(before, s_red[k]);
  #pragma unroll
  for (int k = 0; k < kEdgePer; k++) s_row[tid * kEdgePer + k] = max(before, x[k]);
  __syncthreads();
}

}  // namespace igx
