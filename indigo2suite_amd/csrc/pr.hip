// PageRank (pull, Jacobi) on gfx950, following pr_cuda.h / [C-PRt]:
//   s0 = 1/n;  s_v <- (1 - d)/n + d * sum_{u in N(v)} s_u / deg(u),  d = 0.85
// with no dangling-mass redistribution, stopping when the L1 change of an
// iteration falls below eps or after max_iter iterations.
//
// Precision: scores and contributions are FP32; every neighbour sum is
// compensated (TwoSum per addition; partial sums are merged as (sum, error)
// pairs), and the per-iteration L1 residual that decides convergence is
// accumulated exactly: each row's |change| is computed in FP64 and rounded to
// a multiple of 2^-50, and those integers are summed in 64 bits, so the
// residual does not depend on which wave handled which row (below 1e-9 from
// the FP64 sum for a million rows).  Results are checked against an FP64 host
// oracle.
//
// Reference family: codes/cuda/pr-cuda (54 variants).
//   pull_thread_kahan   [C-PRt] contrib:41-47 + pull:49-70 (thread per vertex)
//   pull_wave_kahan     PR_CUDA_Pull_..._Warp siblings (one wave64 per vertex)
//   pull_block_kahan    PR_CUDA_Pull_..._Block siblings (one workgroup per vertex)
//   pull_balanced_kahan (no reference counterpart) rows classed by degree:
//                       small rows streamed in runs of consecutive rows and
//                       summed in edge order by their lane, longer rows split
//                       into chunks of at most kChunk edges (one wave each)
//                       whose compensated partial sums are merged in chunk
//                       order
//   push_fixed_{thread,wave,block}  [C-PRpush] Push siblings: contributions
//                       pushed to the neighbours' totals with 64-bit
//                       fixed-point atomic adds (exact, order-independent)
// The contribution of the next iteration (score / degree) is written by the
// same kernel that produces the score, so one pass per iteration remains.
#include "igx_internal.hpp"
#include "igx_frontier.hpp"
#include "igx_rank.hpp"
#include "igx_scan.hpp"

namespace igx {
namespace {

constexpr float kDamp = 0.85f;  // pr_cuda.h:43
constexpr int kSmallRow = 32;    // rows streamed in runs by pr_bal_main; longer ones by chunks
constexpr int kSlice = 512;      // edges per streamed slice
constexpr double kResScale = 1125899906842624.0;  // 2^50: fixed-point unit of the residual

struct Pair {
  float s;  // running sum
  float e;  // accumulated rounding error (true sum ~ s + e)
};

__device__ __forceinline__ void two_sum_add(Pair& p, float x)
{
  const float t = p.s + x;
  const float bp = t - p.s;
  const float err = (p.s - (t - bp)) + (x - bp);
  p.s = t;
  p.e += err;
}

__device__ __forceinline__ Pair pair_merge(Pair a, Pair b)
{
  Pair r;
  r.s = a.s + b.s;
  const float bp = r.s - a.s;
  const float err = (a.s - (r.s - bp)) + (b.s - bp);
  r.e = a.e + b.e + err;
  return r;
}

__device__ __forceinline__ Pair wave_merge(Pair p)
{
  #pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    Pair o;
    o.s = __shfl_xor(p.s, d, kWave);
    o.e = __shfl_xor(p.e, d, kWave);
    // merge in a lane-order-independent way: lower half first
    p = ((lane_id() & d) == 0) ? pair_merge(p, o) : pair_merge(o, p);
  }
  return p;
}

__global__ void __launch_bounds__(kBlock) pr_init(const int* __restrict__ nindex, int n, float* __restrict__ score,
                                                   float* __restrict__ contrib)
{
  const int v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n) {
    const float s0 = 1.0f / (float)n;  // pr_cuda.h:133
    score[v] = s0;
    contrib[v] = s0 / (float)(nindex[v + 1] - nindex[v]);
  }
}

// finish one vertex: new score, next contribution, residual term (|change|
// in units of 2^-50, rounded to nearest)
__device__ __forceinline__ long long pr_finish(int v, Pair acc, float base, const int* __restrict__ nindex,
                                               float* __restrict__ score, float* __restrict__ contrib_next)
{
  const float sum = acc.s + acc.e;
  const float value = base + kDamp * sum;
  const float old = score[v];
  score[v] = value;
  contrib_next[v] = value / (float)(nindex[v + 1] - nindex[v]);
  return (long long)(fabs((double)value - (double)old) * kResScale + 0.5);
}


// End of an iteration (run by round_finalize): the L1 residual is the exact
// integer sum of the per-block partials (slot 0: rows scored by the main
// kernel, slot 1: rows merged from chunks, slot 2: rows of one chunk of a
// renumbered graph), scaled back from 2^-50 units.  Also tells the host
// whether the balanced style's merging kernel has work on this graph.
struct FinPr {
  double eps;
  int max_iter;
  const int* big_rows;
  __device__ void operator()(Ctl* ctl, const RoundTotals& t) const
  {
    ctl->aux_ll[0] = (big_rows != nullptr) ? *big_rows : 0;
    const double r = (double)(t.s[0] + t.s[1] + t.s[2]) / kResScale;
    ctl->res_last = r;
    ctl->iter += 1;
    if (r < eps || ctl->iter >= max_iter) ctl->done = 1;
  }
};

enum Gran { kThread = 0, kWaveG = 1, kBlockG = 2 };

template <int G>
__global__ void __launch_bounds__(kBlock) pr_pull(const int* __restrict__ nindex, const int* __restrict__ nlist,
                                                   int n, float base, float* __restrict__ score,
                                                   const float* __restrict__ contrib_cur,
                                                   float* __restrict__ contrib_next, Ctl* ctl, double eps,
                                                   int max_iter)
{
  __shared__ long long s_red[kWavesPerBlock];
  __shared__ Pair s_pair[kWavesPerBlock];
  if (round_done(ctl)) return;
  long long err = 0;
  if constexpr (G == kThread) {
    const int stride = gridDim.x * kBlock;
    for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
      Pair acc{0.0f, 0.0f};
      for (int i = nindex[v]; i < nindex[v + 1]; i++) two_sum_add(acc, contrib_cur[nlist[i]]);
      err += pr_finish(v, acc, base, nindex, score, contrib_next);
    }
  } else if constexpr (G == kWaveG) {
    const int waves = gridDim.x * kWavesPerBlock;
    const int lane = lane_id();
    for (int v = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; v < n; v += waves) {
      Pair acc{0.0f, 0.0f};
      for (int i = nindex[v] + lane; i < nindex[v + 1]; i += kWave) two_sum_add(acc, contrib_cur[nlist[i]]);
      acc = wave_merge(acc);
      if (lane == 0) err += pr_finish(v, acc, base, nindex, score, contrib_next);
    }
  } else {
    const int w = threadIdx.x / kWave;
    for (int v = blockIdx.x; v < n; v += gridDim.x) {
      Pair acc{0.0f, 0.0f};
      for (int i = nindex[v] + (int)threadIdx.x; i < nindex[v + 1]; i += kBlock) two_sum_add(acc, contrib_cur[nlist[i]]);
      acc = wave_merge(acc);
      if (lane_id() == 0) s_pair[w] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        Pair t = s_pair[0];
        for (int k = 1; k < kWavesPerBlock; k++) t = pair_merge(t, s_pair[k]);
        err += pr_finish(v, t, base, nindex, score, contrib_next);
      }
      __syncthreads();
    }
  }
  round_partial_ll(ctl, 0, err, s_red);
}

// ------------------------------------------------------------- balanced ----
// Row classes are built once per run: every row longer than kSmallRow is cut
// into chunks of at most kChunk edges (its pieces in edge order, in a
// contiguous run of chunk slots).  A row of one chunk is finished by the wave
// that sums it (Entry::pad = -1); the others leave compensated partial sums
// that pr_bal_big merges in a fixed order, so the result does not depend on
// the schedule.
struct BigRow {
  int v;
  int first;  // first chunk slot
  int count;  // number of chunks
};

// Degree order.  An iteration is bound by its gathers, one contribution per
// edge.  On a graph with hubs most of them go to few vertices, the head (the
// kHotRanks vertices of highest degree; a contribution each: 64 KB of LDS),
// which may lie all over the contribution array, a cache line each.  Such a
// graph is worked on as a copy renumbered by degree rank: the head's
// contributions lie side by side and the chunks find them in LDS.  Rows keep
// their edges in the order they had, and their chunks, so a row of one chunk
// sums the same values in the same order.  R-MAT 20: the iterations without the
// hot values in LDS 190 -> 139 us, the copy 210 us per run.
//
// The rule.  Copied are graphs whose head
// * takes a quarter of the edges, and 1.5 times its share of the vertices:
//   without the second, every graph of up to 65,536 vertices has such a head
//   (Erdos-Renyi n = 65,536, average degree 64: 344 us as given, 459 copied);
// * is met by long rows, which are the ones that look in LDS (kMinHits of
//   kSamples edges): a star's are met by its leaves (300,000 vertices, 40 hubs:
//   1576 / 2497 us), a mesh and a sparse random graph have none (200 x 200
//   mesh 351 / 657 us);
// * is scattered, where the contributions exceed an XCD's L2 (kNearNodes):
//   Chung-Lu ids are in degree order already (n = 2 M, degree 16, exponent
//   2.3: 3479 / 3853 us; R-MAT 22, edge factor 4: 7718 / 4285 us).  Below, the
//   copy pays there too, since rows of one length side by side make long runs
//   for pr_bal_main (n = 400 k: 1321 / 1075 us);
// * is that of a graph with an edge a vertex, as the copy also passes over the
//   vertices.
// The host decides, from the degree bins and the sample, while pr_classify
// prepares a graph that is not copied (and is empty for one that is): a graph
// that is not copied paid 60 us for launches that found nothing to do when the
// device decided (Erdos-Renyi n = 300 k, average degree 9: 520 -> 502 us).
constexpr int kHotRanks = 16384;
constexpr int kRelabelMinNodes = 2 * kHotRanks;  // below, most of the array is close by anyway
constexpr int kNearNodes = 1 << 20;              // contributions of an XCD's L2 (4 MB)
constexpr int kSamples = 4096;
constexpr int kMinHits = kSamples / 50;

__host__ __device__ inline bool pr_head_counts(int n, int m, long long head_edges)
{
  return head_edges >= m / 4 && (double)head_edges * n >= 1.5 * kHotRanks * m;
}

// what pr_sample counts; zero where the head is too small
struct PrSample {
  int hits;   // edges of long rows whose neighbour is in the head
  int heads;  // edges whose neighbour is in the head
  int mates;  // of the three vertices next to such a neighbour (ids equal but for the lowest two bits), those in it
};

__host__ __device__ inline bool pr_renumber_pays(int n, int m, const int* sample)
{
  const PrSample s = *(const PrSample*)sample;
  const bool scattered = 4LL * s.mates < 3LL * 3 * s.heads;  // fewer than three quarters
  return s.hits >= kMinHits && m >= n && (n <= kNearNodes || scattered || m < 8LL * n);
}

// The graph a run works on: as given, or the renumbered copy.
struct PrGraph {
  const int* nindex;
  const int* nlist;
  float* score;
};

// kSamples evenly spaced edges against the head, added to *out; nothing is
// looked at where the head is too small anyway
__global__ void __launch_bounds__(kBlock) pr_sample(const int* __restrict__ nindex, const int* __restrict__ nlist, int n,
                                                     int m, const int* __restrict__ tile_row,
                                                     const RankHead* __restrict__ head, PrSample* __restrict__ out)
{
  if (!pr_head_counts(n, m, head->edges)) return;
  const int e = (int)((long long)m * (blockIdx.x * kBlock + threadIdx.x) / kSamples);
  const int tile = e / kEdgeTile;
  int lo = tile_row[tile], hi = ((long long)(tile + 1) * kEdgeTile < m) ? tile_row[tile + 1] + 1 : n;
  // the last row that starts at or before e
  while (hi - lo > 1) {
    const int mid = lo + (hi - lo) / 2;
    if (nindex[mid] <= e) lo = mid;
    else hi = mid;
  }
  const int u = nlist[e];
  auto in_head = [&](int v) { return v < n && nindex[v + 1] - nindex[v] >= head->degree; };
  const bool hot = in_head(u);
  int mates = 0;
  for (int k = 1; k < 4; k++) mates += (hot && in_head(u ^ k)) ? 1 : 0;
  mates = wave_sum(mates);
  const int hits = __popcll(ballot(hot && nindex[lo + 1] - nindex[lo] > kSmallRow));
  const int heads = __popcll(ballot(hot));
  if (lane_id() == 0) {
    atomicAdd(&out->hits, hits);
    atomicAdd(&out->heads, heads);
    atomicAdd(&out->mates, mates);
  }
}

__global__ void __launch_bounds__(kBlock) pr_zero(int* __restrict__ p, int count)
{
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < count; i += gridDim.x * kBlock) p[i] = 0;
}

// the renumbered lists: edge (v, u) to the place it has in row rank[v]
__global__ void __launch_bounds__(kBlock) pr_relabel(const int* __restrict__ nindex, const int* __restrict__ nlist, int n,
                                                      int m, const int* __restrict__ rank,
                                                      const int* __restrict__ tile_row,
                                                      const int* __restrict__ nindex1, int* __restrict__ nlist1)
{
  __shared__ __align__(16) int s_row[kEdgeTile];
  __shared__ int s_red[kWavesPerBlock];
  const int tile = blockIdx.x;
  const int base = tile * kEdgeTile;
  const int r0 = tile_row[tile];
  const int r1 = (tile + 1 < (int)gridDim.x) ? tile_row[tile + 1] : n - 1;
  int u[kEdgePer], ru[kEdgePer];
  #pragma unroll
  for (int k = 0; k < kEdgePer; k++) {
    const int i = k * kBlock + (int)threadIdx.x;
    u[k] = (i < m - base) ? nlist[base + i] : -1;
  }
  #pragma unroll
  for (int k = 0; k < kEdgePer; k++) ru[k] = (u[k] >= 0) ? rank[u[k]] : 0;
  edge_tile_rows(nindex, base, r0, r1, s_row, s_red);
  #pragma unroll
  for (int k = 0; k < kEdgePer; k++) {
    if (u[k] >= 0) {
      const int i = k * kBlock + (int)threadIdx.x;
      const int v = r0 + s_row[i];
      nlist1[nindex1[rank[v]] + (base + i - nindex[v])] = ru[k];
    }
  }
}

// scores of a renumbered graph back in the caller's order
__global__ void __launch_bounds__(kBlock) pr_scores_out(const float* __restrict__ score, int n, const int* __restrict__ order,
                                                         float* __restrict__ out)
{
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r < n) out[order[r]] = score[r];
}

// counts[1]: rows of several chunks (big); counts[2]: chunks.  kClassRows
// consecutive rows per workgroup, which reserves their slots with one atomic
// on each counter (one per wave had 170 us of them on R-MAT 20); the chunks
// of a longer row are written by its wave together.  Also the first scores and
// contributions: one launch and one read of the row starts less (7 us at
// n = 1,000,000).
constexpr int kClassPer = 2;
constexpr int kClassRows = kClassPer * kBlock;
__global__ void __launch_bounds__(kBlock) pr_classify(PrGraph g, int n, int m, float* __restrict__ contrib, int* __restrict__ counts,
                                                       Entry* __restrict__ chunks, BigRow* __restrict__ big,
                                                       const int* __restrict__ sample)
{
  __shared__ int s_red[kWavesPerBlock];
  __shared__ int s_first, s_big;
  if (sample != nullptr && pr_renumber_pays(n, m, sample)) return;  // the copy is classified instead
  int beg[kClassPer], end[kClassPer], c[kClassPer];
  int nc = 0, nb = 0;
  #pragma unroll
  for (int k = 0; k < kClassPer; k++) {
    const long long v = (long long)blockIdx.x * kClassRows + k * kBlock + threadIdx.x;
    beg[k] = (v < n) ? g.nindex[v] : 0;
    end[k] = (v < n) ? g.nindex[v + 1] : 0;
    if (v < n) {
      const float s0 = 1.0f / (float)n;  // pr_cuda.h:133
      g.score[v] = s0;
      contrib[v] = s0 / (float)(end[k] - beg[k]);
    }
    c[k] = (end[k] - beg[k] > kSmallRow) ? chunks_of(end[k] - beg[k]) : 0;
    nc += c[k];
    nb += (c[k] > 1) ? 1 : 0;
  }
  int tc = 0, tb = 0;
  int first = block_excl_scan(nc, s_red, &tc);
  if (tc == 0) return;  // uniform
  int bs = block_excl_scan(nb, s_red, &tb);
  if (threadIdx.x == 0) {
    s_first = atomicAdd(&counts[2], tc);
    s_big = (tb > 0) ? atomicAdd(&counts[1], tb) : 0;
  }
  __syncthreads();
  first += s_first;
  bs += s_big;
  #pragma unroll
  for (int k = 0; k < kClassPer; k++) {
    const int v = blockIdx.x * kClassRows + k * kBlock + (int)threadIdx.x;
    if (c[k] == 1) chunks[first] = Entry{v, beg[k], end[k], -1};
    if (c[k] > 1) big[bs++] = BigRow{v, first, c[k]};
    for (uint64_t todo = ballot(c[k] > 1); todo != 0; todo &= todo - 1) {
      const int L = __ffsll((unsigned long long)todo) - 1;
      const int rb = __shfl(beg[k], L, kWave), re = __shfl(end[k], L, kWave), rc = __shfl(c[k], L, kWave);
      const int rf = __shfl(first, L, kWave), rv = __shfl(v, L, kWave);
      for (int j = lane_id(); j < rc; j += kWave) {
        const int b = rb + j * kChunk;
        chunks[rf + j] = Entry{rv, b, (b + kChunk < re) ? b + kChunk : re, 0};
      }
    }
    first += c[k];
  }
}

// One chunk's compensated sum by the wave, its values gathered by `value`
// (kChunk / 64 loads per lane issued together); the row's score when the chunk
// is the whole row.  Returns the residual term on lane 0.
template <typename F>
__device__ __forceinline__ long long pr_chunk(const Entry& en, int k, const PrGraph& g, float base,
                                              float* __restrict__ contrib_next, Pair* __restrict__ partial, F value)
{
  constexpr int kPer = kChunk / kWave;
  const int lane = lane_id();
  int u[kPer];
  #pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int i = en.beg + j * kWave + lane;
    u[j] = (i < en.end) ? g.nlist[i] : -1;
  }
  float x[kPer];
  value(u, x);
  Pair acc{0.0f, 0.0f};
  #pragma unroll
  for (int j = 0; j < kPer; j++) {
    if (u[j] >= 0) two_sum_add(acc, x[j]);
  }
  acc = wave_merge(acc);
  if (lane == 0) {
    if (en.pad < 0) return pr_finish(en.v, acc, base, g.nindex, g.score, contrib_next);
    partial[k] = acc;
  }
  return 0;
}

// The chunks of a renumbered graph, with the kHotRanks hot contributions in
// LDS (64 KB, so two workgroups of 16 waves fill a CU).  A gather that misses
// LDS moves a cache line from L2, which is what an iteration is bound by:
// R-MAT 20 (57% of the edges hot): 128 -> 104 us an iteration together with
// the small rows.
constexpr int kHotBlock = 1024;
__global__ void __launch_bounds__(kHotBlock) pr_hot_chunks(PrGraph g, int n, float base,
                                                            const float* __restrict__ contrib_cur,
                                                            float* __restrict__ contrib_next,
                                                            const int* __restrict__ counts,
                                                            const Entry* __restrict__ chunks,
                                                            Pair* __restrict__ partial, int nparts, Ctl* ctl)
{
  __shared__ float s_hot[kHotRanks];
  __shared__ long long s_red[kHotBlock / kWave];
  if (round_done(ctl)) return;
  // partial slots past this grid (the round's other kernels have a wider one)
  if (blockIdx.x == 0) {
    for (int i = gridDim.x + threadIdx.x; i < nparts; i += kHotBlock) ctl_parts(ctl)[(size_t)2 * kMaxParts + i] = 0;
  }
  long long err = 0;
  for (int i = threadIdx.x; i < kHotRanks && i < n; i += kHotBlock) s_hot[i] = contrib_cur[i];
  __syncthreads();
  const int nch = counts[2];
  const int waves = gridDim.x * (kHotBlock / kWave);
  for (int k = blockIdx.x * (kHotBlock / kWave) + threadIdx.x / kWave; k < nch; k += waves) {  // uniform per wave
    err += pr_chunk(chunks[k], k, g, base, contrib_next, partial, [&](const int* u, float* x) {
      #pragma unroll
      for (int j = 0; j < kChunk / kWave; j++) x[j] = (u[j] >= kHotRanks) ? contrib_cur[u[j]] : 0.0f;
      #pragma unroll
      for (int j = 0; j < kChunk / kWave; j++) {
        if (u[j] >= 0 && u[j] < kHotRanks) x[j] = s_hot[u[j]];
      }
    });
  }
  round_partial_ll(ctl, 2, err, s_red);
}

// One iteration's sums: first the chunks, unless pr_hot_chunks does them (one
// wave each; chunks are at most kChunk edges, so a fixed round-robin share
// balances), then the small rows in 64-row tiles, also round robin.  Small
// rows: consecutive small rows form runs whose edges are contiguous, streamed
// kSlice at a time (independent loads, values parked in LDS); each lane then
// adds its own row's values in edge order.
__global__ void __launch_bounds__(kBlock) pr_bal_main(PrGraph g, bool chunks_done, int n, float base,
                                                       const float* __restrict__ contrib_cur,
                                                       float* __restrict__ contrib_next,
                                                       const int* __restrict__ counts,
                                                       const Entry* __restrict__ chunks, Pair* __restrict__ partial,
                                                       Ctl* ctl)
{
  __shared__ long long s_red[kWavesPerBlock];
  __shared__ float s_val[kWavesPerBlock][kSlice];
  if (round_done(ctl)) return;
  const int* __restrict__ nindex = g.nindex;
  const int* __restrict__ nlist = g.nlist;
  float* __restrict__ score = g.score;
  long long err = 0;
  const int waves = gridDim.x * kWavesPerBlock;
  const int gw = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  const int lane = lane_id();
  const int nch = chunks_done ? 0 : counts[2];
  for (int k = gw; k < nch; k += waves) {  // uniform per wave
    err += pr_chunk(chunks[k], k, g, base, contrib_next, partial, [&](const int* u, float* x) {
      #pragma unroll
      for (int j = 0; j < kChunk / kWave; j++) x[j] = (u[j] >= 0) ? contrib_cur[u[j]] : 0.0f;
    });
  }
  float* vbuf = s_val[threadIdx.x / kWave];
  for (int v0 = gw * kWave; v0 < n; v0 += waves * kWave) {  // uniform per wave
    const int v = v0 + lane;
    int rb = 0, re = 0;
    if (v < n) {
      rb = nindex[v];
      re = nindex[v + 1];
    }
    const bool small = (v < n) && (re - rb <= kSmallRow);
    Pair acc{0.0f, 0.0f};
    uint64_t todo = ballot(small);
    while (todo != 0) {  // one run of consecutive small rows
      const int first = __ffsll((unsigned long long)todo) - 1;
      const uint64_t from = todo >> first;
      const int cnt = (~from == 0) ? (kWave - first) : (__ffsll((unsigned long long)~from) - 1);
      const int last = first + cnt - 1;
      todo &= (cnt + first >= kWave) ? ((1ull << first) - 1) : ~(((1ull << cnt) - 1) << first);
      const int r0 = __shfl(rb, first, kWave), r1 = __shfl(re, last, kWave);
      const bool mine = lane >= first && lane <= last;
      for (int c0 = r0; c0 < r1; c0 += kSlice) {
        const int c1 = (r1 - c0 < kSlice) ? r1 : c0 + kSlice;
        int uu[kSlice / kWave];
        #pragma unroll
        for (int k = 0; k < kSlice / kWave; k++) {
          const int e = c0 + k * kWave + lane;
          uu[k] = (e < c1) ? nlist[e] : -1;
        }
        float xx[kSlice / kWave];
        #pragma unroll
        for (int k = 0; k < kSlice / kWave; k++) xx[k] = (uu[k] >= 0) ? contrib_cur[uu[k]] : 0.0f;
        __builtin_amdgcn_wave_barrier();
        #pragma unroll
        for (int k = 0; k < kSlice / kWave; k++) vbuf[k * kWave + lane] = xx[k];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (mine) {
          const int lo = (rb > c0) ? rb : c0;
          const int hi = (re < c1) ? re : c1;
          for (int i = lo; i < hi; i++) two_sum_add(acc, vbuf[i - c0]);
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (small) err += pr_finish(v, acc, base, nindex, score, contrib_next);
  }
  round_partial_ll(ctl, 0, err, s_red);
}

// The partial sums of the rows of several chunks, kBigLanes lanes a row: each
// merges every kBigLanes-th one, then the lanes merge in lane order.  (One
// lane a row left the longest row's chain, 273 merges on R-MAT 20, as the
// kernel's time: 29 us.)
constexpr int kBigLanes = 8;
__global__ void __launch_bounds__(kBlock) pr_bal_big(PrGraph g, float base, float* __restrict__ contrib_next,
                                                      const BigRow* __restrict__ big, const int* __restrict__ counts,
                                                      const Pair* __restrict__ partial, Ctl* ctl)
{
  __shared__ long long s_red[kWavesPerBlock];
  if (round_done(ctl)) return;
  long long err = 0;
  const int nb = counts[1];
  const int l = threadIdx.x % kBigLanes;
  const int stride = gridDim.x * (kBlock / kBigLanes);
  for (int i = blockIdx.x * (kBlock / kBigLanes) + threadIdx.x / kBigLanes; i < nb; i += stride) {
    const BigRow b = big[i];
    Pair acc{0.0f, 0.0f};
    for (int k = l; k < b.count; k += kBigLanes) acc = pair_merge(acc, partial[b.first + k]);
    #pragma unroll
    for (int d = 1; d < kBigLanes; d <<= 1) {
      Pair o;
      o.s = __shfl_xor(acc.s, d, kWave);
      o.e = __shfl_xor(acc.e, d, kWave);
      acc = ((l & d) == 0) ? pair_merge(acc, o) : pair_merge(o, acc);
    }
    if (l == 0) err += pr_finish(b.v, acc, base, g.nindex, g.score, contrib_next);
  }
  round_partial_ll(ctl, 1, err, s_red);
}

// ----------------------------------------------------------------- push ----
// [C-PRpush] contrib():41-48, push():50-63, compute():65-77: every vertex adds
// its contribution score / degree to each neighbour's incoming total, then
// every vertex turns its total into its new score.  The reference adds floats
// atomically, so its totals depend on the order in which the atomics land.
// Here each contribution is rounded once to a multiple of 2^-60 (a float
// contribution of at least 2^-37 already is one, so typical contributions are
// not rounded at all) and added as a 64-bit integer: integer addition is
// associative, so every total, and with it the iteration count, is the same
// whatever the schedule, and it is the exact sum of the rounded contributions.
// A total is at most the sum of all scores (at most 1 = 2^60 units), far from
// the int64 limit.  The compute pass reads each total once, clears it for the
// next iteration, and writes the score, the next contribution and the
// residual exactly like the pull styles.
constexpr double kFixScale = 1152921504606846976.0;  // 2^60: fixed-point unit of the totals

__device__ __forceinline__ unsigned long long pr_fixed(float c)
{
  return (unsigned long long)((double)c * kFixScale + 0.5);
}

template <int G>
__global__ void __launch_bounds__(kBlock) pr_push(const int* __restrict__ nindex, const int* __restrict__ nlist,
                                                   int n, const float* __restrict__ contrib,
                                                   unsigned long long* __restrict__ incoming, Ctl* ctl)
{
  if (round_done(ctl)) return;
  if constexpr (G == kThread) {
    const int stride = gridDim.x * kBlock;
    for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
      const int beg = nindex[v], end = nindex[v + 1];
      if (beg == end) continue;  // a vertex of degree 0 has an infinite contribution and no edge
      const unsigned long long q = pr_fixed(contrib[v]);
      for (int i = beg; i < end; i++) atomicAdd(&incoming[nlist[i]], q);
    }
  } else if constexpr (G == kWaveG) {
    const int waves = gridDim.x * kWavesPerBlock;
    const int lane = lane_id();
    for (int v = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; v < n; v += waves) {
      const int beg = nindex[v], end = nindex[v + 1];
      if (beg == end) continue;
      const unsigned long long q = pr_fixed(contrib[v]);
      for (int i = beg + lane; i < end; i += kWave) atomicAdd(&incoming[nlist[i]], q);
    }
  } else {
    for (int v = blockIdx.x; v < n; v += gridDim.x) {
      const int beg = nindex[v], end = nindex[v + 1];
      if (beg == end) continue;
      const unsigned long long q = pr_fixed(contrib[v]);
      for (int i = beg + (int)threadIdx.x; i < end; i += kBlock) atomicAdd(&incoming[nlist[i]], q);
    }
  }
}

__global__ void __launch_bounds__(kBlock) pr_push_compute(const int* __restrict__ nindex, int n, float base,
                                                           float* __restrict__ score, float* __restrict__ contrib,
                                                           unsigned long long* __restrict__ incoming, Ctl* ctl)
{
  __shared__ long long s_red[kWavesPerBlock];
  if (round_done(ctl)) return;
  long long err = 0;
  const int stride = gridDim.x * kBlock;
  for (int v = blockIdx.x * kBlock + threadIdx.x; v < n; v += stride) {
    const float total = (float)((double)incoming[v] / kFixScale);
    incoming[v] = 0;
    err += pr_finish(v, Pair{total, 0.0f}, base, nindex, score, contrib);
  }
  round_partial_ll(ctl, 0, err, s_red);
}

__global__ void __launch_bounds__(kBlock) pr_zero_ull(unsigned long long* __restrict__ p, int n)
{
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ------------------------------------------------------------ host side ----
int pr_buffers(const igx_graph* g, float** c0, float** c1)
{
  void *p0 = nullptr, *p1 = nullptr;
  IGX_TRY(ws_get(WS_F, sizeof(float) * (size_t)g->nodes, &p0));
  IGX_TRY(ws_get(WS_G, sizeof(float) * (size_t)g->nodes, &p1));
  *c0 = (float*)p0;
  *c1 = (float*)p1;
  return IGX_OK;
}

template <int G>
int style_pull(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  float* score = (float*)out;
  float *c0 = nullptr, *c1 = nullptr;
  IGX_TRY(pr_buffers(g, &c0, &c1));
  const PrParams P = pr_params();
  const float base = (1.0f - kDamp) / (float)g->nodes;  // pr_cuda.h:140
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(g->nodes));
  hipLaunchKernelGGL(pr_init, dim3(blocks_for(g->nodes, kBlock)), dim3(kBlock), 0, R.stream, g->nindex, g->nodes,
                     score, c0);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long r) {
        float* cur = (r & 1) ? c1 : c0;
        float* nxt = (r & 1) ? c0 : c1;
        hipLaunchKernelGGL((pr_pull<G>), dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist,
                           g->nodes, base, score, cur, nxt, R.d_ctl, P.eps, P.max_iter);
        launch_finalize<0x1>(R.persist_blocks, FinPr{P.eps, P.max_iter, nullptr});
      },
      P.max_iter, &rounds, &launches);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  info->residual = R.h_ctl->res_last;
  return rc == IGX_ERR_LIMIT ? IGX_OK : rc;
}

int style_balanced(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  float *c0 = nullptr, *c1 = nullptr;
  IGX_TRY(pr_buffers(g, &c0, &c1));
  const int n = g->nodes;
  const int m = g->edges;
  // rows above kSmallRow: at most edges / (kSmallRow + 1) of them, each with
  // at most deg / kChunk + 1 chunks
  const size_t nrows = (size_t)m / (kSmallRow + 1) + 64;
  const size_t nchunks = (size_t)m / kChunk + nrows;
  constexpr int kSmall = 64 + kRankBins;  // counters and the degree bins
  const int tiles = (int)(((long long)m + kEdgeTile - 1) / kEdgeTile);
  void *pcnt = nullptr, *pch = nullptr, *pbig = nullptr, *ppart = nullptr, *ptile = nullptr;
  IGX_TRY(ws_get(WS_B, sizeof(int) * kSmall, &pcnt));
  IGX_TRY(ws_get(WS_D, sizeof(Entry) * nchunks, &pch));
  IGX_TRY(ws_get(WS_C, sizeof(BigRow) * nrows, &pbig));
  IGX_TRY(ws_get(WS_H, sizeof(Pair) * nchunks, &ppart));
  // without the memory for the renumbered copy the run does without it
  const bool may = n >= kRelabelMinNodes && m > 0 &&
                   ws_get(WS_BLOCKS, sizeof(int) * ((size_t)tiles + scan_tiles_for(n + 1) + 64), &ptile) == IGX_OK;
  int* counts = (int*)pcnt;
  int* bins = counts + 64;
  int* tile_row = (int*)ptile;
  int* tile_sum = tile_row + tiles;
  PrGraph from = {g->nindex, g->nlist, (float*)out};
  const PrParams P = pr_params();
  const float base = (1.0f - kDamp) / (float)n;
  const int rank_blocks = blocks_for(n, kRankRows);
  auto zero = [&](int count) {
    hipLaunchKernelGGL(pr_zero, dim3(blocks_for(count, kBlock)), dim3(kBlock), 0, R.stream, counts, count);
  };
  auto classify = [&](const int* sample) {
    hipLaunchKernelGGL(pr_classify, dim3(blocks_for(n, kClassRows)), dim3(kBlock), 0, R.stream, from, n, m, c0, counts,
                       (Entry*)pch, (BigRow*)pbig, sample);
  };
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(n));
  zero(kSmall);
  if (may) {
    hipLaunchKernelGGL(rank_hist, dim3(rank_blocks), dim3(kBlock), 0, R.stream, g->nindex, n, bins, tile_row);
    RankHead* head = (RankHead*)R.d_ctl->aux_ll;
    hipLaunchKernelGGL(rank_bins, dim3(1), dim3(kBlock), 0, R.stream, bins, 0, (int*)nullptr, kHotRanks, head);
    hipLaunchKernelGGL(pr_sample, dim3(kSamples / kBlock), dim3(kBlock), 0, R.stream, g->nindex, g->nlist, n, m,
                       (const int*)tile_row, (const RankHead*)head, (PrSample*)R.d_ctl->sample);
    IGX_TRY(batch_mark(0));
  }
  classify(may ? R.d_ctl->sample : nullptr);  // under way while the host waits
  bool hot = false;
  int* order = nullptr;
  if (may) {
    IGX_TRY(batch_wait(0));
    void *pr1 = nullptr, *pl1 = nullptr;
    const bool pays = pr_renumber_pays(n, m, R.h_ctl->sample);
    hot = pays && ws_get(WS_A, sizeof(int) * 5 * ((size_t)n + 1), &pr1) == IGX_OK &&
          ws_get(WS_E, sizeof(int) * (size_t)m, &pl1) == IGX_OK;
    if (hot) {
      int* rank = (int*)pr1;
      order = rank + n;
      int* degree = order + n;        // n + 1
      int* nindex1 = degree + n + 1;  // n + 1
      hipLaunchKernelGGL(rank_assign, dim3(rank_blocks), dim3(kBlock), 0, R.stream, g->nindex, n, bins, rank, order,
                         degree);
      exclusive_scan(degree, nindex1, n + 1, tile_sum, tile_sum + scan_tiles_for(n + 1), R.stream);
      hipLaunchKernelGGL(pr_relabel, dim3(tiles), dim3(kBlock), 0, R.stream, g->nindex, g->nlist, n, m,
                         (const int*)rank, (const int*)tile_row, (const int*)nindex1, (int*)pl1);
      from = PrGraph{nindex1, (const int*)pl1, (float*)(nindex1 + n + 1)};
    }
    if (pays) classify(nullptr);
  }
  // Iterations to 1e-6 fall with the degree: 14 at an average of 16, 11 at 32,
  // 8 at 64, 5 at 300.  So a second batch goes in before the first is waited
  // for up to a degree of 32 (Chung-Lu n = 400 k, degree 16, exponent 2.9:
  // 1187 -> 1156 us), unless the iterations are so short that the merging
  // kernel, which the host does not yet know to be idle, costs as much as the
  // wait (200 x 200 mesh 350 -> 356 us).
  const int first_batch = (m > 128LL * n) ? 5 : 4;
  const bool behind = hot || (m <= 32LL * n && m >= (1 << 21));
  const int unseen = first_batch + (behind ? kAheadRounds : 0);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long r) {
        float* cur = (r & 1) ? c1 : c0;
        float* nxt = (r & 1) ? c0 : c1;
        // once a batch of iterations on the graph as given has come back, the
        // merging kernel is left out where it has nothing to do
        const bool big = hot || r < unseen || R.h_ctl->aux_ll[0] != 0;
        ktimer_begin("pr_bal_main");
        if (hot) {
          ktimer_begin("pr_hot_chunks");
          hipLaunchKernelGGL(pr_hot_chunks, dim3(2 * R.cus), dim3(kHotBlock), 0, R.stream, from, n, base, cur, nxt,
                             (const int*)counts, (const Entry*)pch, (Pair*)ppart, R.persist_blocks, R.d_ctl);
          ktimer_end("pr_hot_chunks");
        }
        hipLaunchKernelGGL(pr_bal_main, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, from, hot, n, base, cur, nxt,
                           (const int*)counts, (const Entry*)pch, (Pair*)ppart, R.d_ctl);
        ktimer_end("pr_bal_main");
        if (big) {
          hipLaunchKernelGGL(pr_bal_big, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, from, base, nxt,
                             (const BigRow*)pbig, (const int*)counts, (const Pair*)ppart, R.d_ctl);
        }
        const FinPr fin{P.eps, P.max_iter, counts + 1};
        if (hot) launch_finalize<0x7>(R.persist_blocks, fin);
        else if (big) launch_finalize<0x3>(R.persist_blocks, fin);
        else launch_finalize<0x1>(R.persist_blocks, fin);
      },
      P.max_iter, &rounds, &launches, first_batch, behind);
  if (hot) {
    hipLaunchKernelGGL(pr_scores_out, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, R.stream,
                       (const float*)from.score, n, (const int*)order, (float*)out);
  }
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  info->residual = R.h_ctl->res_last;
  return rc == IGX_ERR_LIMIT ? IGX_OK : rc;
}

// One contribution buffer suffices: the push pass reads it and the compute
// pass, a separate launch, rewrites it.
template <int G>
int style_push(const igx_graph* g, int, void* out, const void*, igx_run_info* info)
{
  Runtime& R = rt();
  float* score = (float*)out;
  const int n = g->nodes;
  void *pc = nullptr, *pin = nullptr;
  IGX_TRY(ws_get(WS_F, sizeof(float) * (size_t)n, &pc));
  IGX_TRY(ws_get(WS_H, sizeof(unsigned long long) * (size_t)n, &pin));
  float* contrib = (float*)pc;
  unsigned long long* incoming = (unsigned long long*)pin;
  const PrParams P = pr_params();
  const float base = (1.0f - kDamp) / (float)n;
  IGX_TRY(timer_start());
  IGX_TRY(ctl_reset(n));
  hipLaunchKernelGGL(pr_init, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, R.stream, g->nindex, n, score, contrib);
  hipLaunchKernelGGL(pr_zero_ull, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, R.stream, incoming, n);
  int rounds = 0, launches = 0;
  const int rc = run_rounds(
      [&](long long) {
        ktimer_begin("pr_push");
        hipLaunchKernelGGL((pr_push<G>), dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, g->nlist, n,
                           contrib, incoming, R.d_ctl);
        ktimer_end("pr_push");
        hipLaunchKernelGGL(pr_push_compute, dim3(R.persist_blocks), dim3(kBlock), 0, R.stream, g->nindex, n, base,
                           score, contrib, incoming, R.d_ctl);
        launch_finalize<0x1>(R.persist_blocks, FinPr{P.eps, P.max_iter, nullptr});
      },
      P.max_iter, &rounds, &launches);
  IGX_TRY(timer_stop(&info->seconds));
  info->iterations = rounds;
  info->launches = launches;
  info->residual = R.h_ctl->res_last;
  return rc == IGX_ERR_LIMIT ? IGX_OK : rc;
}

const StyleEntry kStyles[] = {
    {"pull_thread_kahan", style_pull<kThread>, 0},
    {"pull_wave_kahan", style_pull<kWaveG>, 0},
    {"pull_block_kahan", style_pull<kBlockG>, 0},
    {"pull_balanced_kahan", style_balanced, 0},
    {"push_fixed_thread", style_push<kThread>, 0},
    {"push_fixed_wave", style_push<kWaveG>, 0},
    {"push_fixed_block", style_push<kBlockG>, 0},
};

}  // namespace

const StyleEntry* pr_styles(int* count)
{
  *count = (int)(sizeof(kStyles) / sizeof(kStyles[0]));
  return kStyles;
}

}  // namespace igx
