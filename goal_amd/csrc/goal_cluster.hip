// One-kernel assembly of residual and Jacobian for neo-Hookean quadratic tets
// with four points, FP64: a workgroup forms all CSR rows of one run of nodes
// (goal_cluster.hpp) from the nodal values, so no element matrix goes through
// memory.
//
// Tangent in spatial form.  With F^{-T} dN/dX = f and F dN/dX = h per node,
// c = mu J^{-2/3}, P = c F + s F^{-T}, s = p J - c tr(F F^T) / 3,
// s2 = p J + 2/9 c tr(F F^T), pi = F^{-T} grad p, t = tau J (the closed form of
// goal_device.hpp contracted with node a's gradient G_a):
//   K(ai,bk) = s2 f_ai f_bk - 2/3 c (h_ai f_bk + f_ai h_bk) - s f_ak f_bi + c d_ik G_a.G_b
//   K(ai,b3) = N_b J f_ai
//   K(a3,bk) = N_a beta f_bk + t (f_a.pi f_bk - pi_k f_a.f_b - f_ak f_b.pi)
//   K(a3,b3) = N_a N_b / kappa + t f_a.f_b
//   R(ai) = c h_ai + s f_ai,   R(a3) = N_a r1 + t f_a.pi     (all times w dv, summed over the points)
//
// One lane forms the two 4 x 4 CSR blocks of a pair of nodes: it runs over the
// elements that hold both and sums the blocks over their points in registers.
//
// Measured on the P2 64^3 cube (1.57 M tets; 7.8 GB of CSR values): 5.6 ms
// against 12.7 ms for the element pass and the gather, whose 20.6 GB of element
// matrices were written and read once.  HBM traffic 10.8 GB instead of 51.
// Leaving out the blocks' sums takes 1.0-1.6 ms off, the point states 1.6-1.9,
// the stores 1.4-1.7, and all three leave 1.1 ms: with four workgroups per CU
// (LDS) the phases' latencies add up: the vector ALUs are busy 52% of the time,
// LDS 34%, with 2.3 waves a SIMD resident, which wait 57% of theirs.
// Also measured:
//   - sums in LDS by FP64 atomics, one lane per (element, row): 8.2 ms; an
//     LDS FP64 atomic of a wave takes 48 cycles, half of them conflicts
//   - one lane per block instead of per pair of blocks: 7.9 ms
//   - a persistent grid, with the next chunk's plan fetched ahead or its point
//     states formed by waves of their own: 9.5-9.9 ms
//   - four waves per workgroup and at most two visits a lane: 5.9 ms; three
//     waves, two visits: 5.7; the blocks stored by one lane each: 5.7;
//     nontemporal stores: 9.5 (L2 no longer joins the rows' 32-byte pieces)
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "goal_cluster.hpp"
#include "goal_device.hpp"
#include "goal_kernels.hpp"

namespace goal {
namespace {

// ------------------------------------------------------------------- plan
constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n) { return (unsigned)std::min<int64_t>(std::max<int64_t>((n + kBlock - 1) / kBlock, 1), 65536); }

__device__ inline int edge_lo(int k) { return k < 3 ? k : k - 3; }  // edges 01, 12, 20, 03, 13, 23
__device__ inline int edge_hi(int k) { return k < 3 ? (k == 2 ? 0 : k + 1) : 3; }

// A double's bits as an integer that orders as the double does.
__device__ inline unsigned long long ordered_bits(double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ inline double from_ordered(unsigned long long u) {
  return __longlong_as_double((long long)((u >> 63) ? (u & 0x7fffffffffffffffull) : ~u));
}

// box[0..2], [3..5]: smallest and largest coordinates (ordered_bits), ~0 and zero
// before.  One atomic per workgroup and bound: with one per wave their turns on
// six addresses took 280 us for 275 K nodes.
__global__ __launch_bounds__(kBlock) void cluster_box_kernel(const double* X, int64_t nn, unsigned long long* box) {
  __shared__ unsigned long long part[kBlock / 64][6];
  unsigned long long lo[3] = {~0ull, ~0ull, ~0ull}, hi[3] = {0, 0, 0};
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nn; i += (int64_t)gridDim.x * kBlock)
    for (int c = 0; c < 3; ++c) {
      const unsigned long long u = ordered_bits(X[3 * i + c]);
      lo[c] = min(lo[c], u);
      hi[c] = max(hi[c], u);
    }
  for (int c = 0; c < 3; ++c) {
    for (int off = 32; off > 0; off >>= 1) {
      lo[c] = min(lo[c], (unsigned long long)__shfl_xor((long long)lo[c], off, 64));
      hi[c] = max(hi[c], (unsigned long long)__shfl_xor((long long)hi[c], off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
      part[threadIdx.x >> 6][c] = lo[c];
      part[threadIdx.x >> 6][3 + c] = hi[c];
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    unsigned long long v = part[0][threadIdx.x];
    for (int w = 1; w < kBlock / 64; ++w)
      v = threadIdx.x < 3 ? min(v, part[w][threadIdx.x]) : max(v, part[w][threadIdx.x]);
    if (threadIdx.x < 3) atomicMin(&box[threadIdx.x], v);
    else atomicMax(&box[threadIdx.x], v);
  }
}

__device__ inline uint32_t spread3(uint32_t v) {  // ten bits, three apart
  v = (v | (v << 16)) & 0x030000ff;
  v = (v | (v << 8)) & 0x0300f00f;
  v = (v | (v << 4)) & 0x030c30c3;
  return (v | (v << 2)) & 0x09249249;
}

// Each node's place on a Morton curve through the mesh's box (cubic cells).
__global__ __launch_bounds__(kBlock) void cluster_morton_kernel(const double* X, int64_t nn,
                                                                const unsigned long long* box, uint32_t* code,
                                                                int32_t* iota) {
  double lo[3], size = 0.0;
  for (int c = 0; c < 3; ++c) {
    lo[c] = from_ordered(box[c]);
    size = fmax(size, from_ordered(box[3 + c]) - lo[c]);
  }
  const double scale = size > 0.0 ? 1024.0 / size : 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nn; i += (int64_t)gridDim.x * kBlock) {
    uint32_t v = 0;
    for (int c = 0; c < 3; ++c) v |= spread3((uint32_t)fmin(fmax((X[3 * i + c] - lo[c]) * scale, 0.0), 1023.0)) << c;
    code[i] = v;
    iota[i] = (int32_t)i;
  }
}

// pass 0: every node its own rank; 1: edge nodes cleared; 2: edge nodes the
// smaller rank of their edge's vertices
__global__ __launch_bounds__(kBlock) void cluster_keys_kernel(const int32_t* conn, int64_t ne, int64_t nn, int pass,
                                                              const int32_t* rank, int32_t* keys, int32_t* iota) {
  const int64_t n = pass == 0 ? nn : 6 * ne;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    if (pass == 0) {
      keys[i] = rank[i];
      iota[i] = (int32_t)i;
      continue;
    }
    const int32_t* c = conn + 10 * (i / 6);
    const int k = (int)(i % 6);
    if (pass == 1) keys[c[4 + k]] = INT32_MAX;
    else atomicMin(&keys[c[4 + k]], min(rank[c[edge_lo(k)]], rank[c[edge_hi(k)]]));
  }
}

__global__ __launch_bounds__(kBlock) void cluster_segments_kernel(const int32_t* keys, int64_t nn, int64_t* seg) {
  for (int64_t a = (int64_t)blockIdx.x * kBlock + threadIdx.x; a <= nn; a += (int64_t)gridDim.x * kBlock) {
    int64_t lo = 0, hi = nn;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (keys[mid] < a) lo = mid + 1;
      else hi = mid;
    }
    seg[a] = lo;
  }
}

__global__ __launch_bounds__(kBlock) void cluster_place_kernel(const int32_t* nodes, int64_t nn, int32_t* place) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nn; i += (int64_t)gridDim.x * kBlock)
    place[nodes[i]] = (int32_t)i;
}

// One wavefront walks a key's part of the nodes.  Bound by the latency of a
// node's loads.  P2 8^3: 25 us each, 64^3: 1.0 and 1.2 ms; one thread a key, which
// looked an element up in its list entry by entry, took 270 us and 2.0 ms.
__global__ __launch_bounds__(kBlock) void cluster_count_kernel(ClusterMesh m, const int64_t* seg, int64_t nn,
                                                               int32_t* runs, int32_t* more, int32_t* recs,
                                                               int32_t* most) {
  const int64_t waves = (int64_t)gridDim.x * (kBlock / 64);
  for (int64_t a = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); a <= nn; a += waves) {
    ClusterCount c;
    const int64_t lo = a < nn ? seg[a] : 0, hi = a < nn ? seg[a + 1] : 0;
    if (lo < hi) walk_cluster(m, lo, hi, c);
    if (threadIdx.x & 63) continue;
    runs[a] = c.runs;
    more[a] = c.chunks > c.runs ? c.chunks - c.runs : 0;
    recs[a] = c.recs;
    if (c.most > *most) atomicMax(most, c.most);
  }
}

__global__ __launch_bounds__(kBlock) void cluster_fill_kernel(ClusterMesh m, const int64_t* seg, int64_t nn,
                                                              const int32_t* runs, const int32_t* more,
                                                              const int32_t* recs, int64_t num_runs, int4* run_tab,
                                                              int4* chunk_tab, int2* span_tab, uint32_t* elem_tab,
                                                              int2* rec_tab) {
  const int64_t waves = (int64_t)gridDim.x * (kBlock / 64);
  for (int64_t a = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); a < nn; a += waves) {
    const int64_t lo = seg[a], hi = seg[a + 1];
    if (lo == hi) continue;
    ClusterFill f;
    f.runs = run_tab;
    f.chunks = chunk_tab;
    f.spans = span_tab;
    f.elems = elem_tab;
    f.recs = rec_tab;
    f.r = runs[a];
    f.x = (int)num_runs + more[a];
    f.k = recs[a];
    f.writes = (threadIdx.x & 63) == 0;
    walk_cluster(m, lo, hi, f);
  }
}

// out: four totals, for one read-back.
__global__ void cluster_totals_kernel(const int32_t* a, const int32_t* b, const int32_t* c, const int32_t* d,
                                      int4* out) {
  *out = int4{*a, *b, *c, *d};
}

// First lane of every pair (block s < nb with cnt[s] > 0 visits): the pairs in
// order of cluster_rank, then of s.  By groups of 64 blocks: a group's pairs of a
// rank are counted by ballot, and the lanes before them are a prefix over ranks
// and groups.  With one thread a pair that counted the pairs before it and then
// looked through its node's incidences once a lane, the tables of 1.57 M linear
// tets took 2 x 2.2 ms (sizes, then tables) and those of 83 K quadratic ones 2 x
// 0.55; now 0.3 (linear_split counts the lanes too) and 1.1, and 2 x 0.26.
constexpr int kRanks = 9, kGroups = kClusterSlots / 64;
static_assert(kRanks * kGroups <= 128 && kGroups <= 64, "two entries a lane");
__device__ void order_pairs(const int* cnt, int nb, int* before, uint16_t* at) {  // before: [kRanks * kGroups]
  const int tid = threadIdx.x, lane = tid & 63;
  for (int g = tid >> 6; g < kGroups; g += kBlock / 64) {
    const int s = 64 * g + lane, rank = s < nb ? cluster_rank(cnt[s]) : kRanks;
    for (int k = 0; k < kRanks; ++k) {
      const unsigned long long b = __ballot(rank == k);
      if (rank == k) at[s] = (uint16_t)(cluster_lanes_of_rank(k) * __popcll(b & ((1ull << lane) - 1)));
      if (lane == 0) before[kGroups * k + g] = cluster_lanes_of_rank(k) * __popcll(b);
    }
  }
  __syncthreads();
  if (tid < 64) {
    int carry = 0;
    for (int i0 = 0; i0 < kRanks * kGroups; i0 += 64) {
      const int i = i0 + lane, v = i < kRanks * kGroups ? before[i] : 0;
      int sum = v;
      for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(sum, off, 64);
        if (lane >= off) sum += o;
      }
      if (i < kRanks * kGroups) before[i] = carry + sum - v;
      carry += __shfl(sum, 63, 64);
    }
  }
  __syncthreads();
  for (int s = tid; s < nb; s += kBlock)
    if (cnt[s]) at[s] = (uint16_t)(at[s] + before[kGroups * cluster_rank(cnt[s]) + s / 64]);
  __syncthreads();
}

// The lanes that cnt's pairs take, added to *total (zero before).
__device__ void count_lanes(int mine, int* total) {
  for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off, 64);
  if ((threadIdx.x & 63) == 0) atomicAdd(total, mine);
  __syncthreads();
}

// One workgroup per run: the pairs of each of its chunks, one thread per visit
// (row node's incidence, element node), the visits of a pair in incidence order.
__global__ __launch_bounds__(kBlock) void cluster_lanes_kernel(ClusterMesh m, const int4* run_tab, int4* chunk_tab,
                                                               const int2* span_tab, const uint32_t* elem_tab,
                                                               const int2* recs, int32_t* nlanes,
                                                               ClusterLane* lanes) {
  constexpr int kRecs = 10 * kClusterElems;                // a chunk's incidences, at most
  __shared__ int first[kClusterNodes + 1];                 // first block of a node
  __shared__ int rlo[kClusterNodes];                       // a node's first incidence in the chunk
  __shared__ uint16_t rpos[kRecs * 10];                    // their positions
  __shared__ int rinfo[kRecs];                             // element slot | local node << 8 | run-local node << 16
  __shared__ int cnt[kClusterSlots];                       // visits of a block's pair
  __shared__ int before[kRanks * kGroups];
  __shared__ uint16_t at[kClusterSlots], src[kRecs * 10];  // first lane of a pair; a lane's first visit
  __shared__ unsigned long long work[kRecs * 10];          // the visits of every lane
  __shared__ int total;
  const int tid = threadIdx.x;
  const int4 run = run_tab[blockIdx.x];
  const int nn = run.y - run.x;
  if (tid < nn) {
    const int64_t n = m.nodes[run.x + tid];
    first[tid + 1] = (int)((m.row_ptr[4 * n + 1] - m.row_ptr[4 * n]) / 4);
  }
  if (tid == 0) first[0] = 0;
  __syncthreads();
  if (tid == 0)
    for (int i = 0; i < nn; ++i) first[i + 1] += first[i];
  __syncthreads();
  const int nb = first[nn];
  for (int c = (int)blockIdx.x, nxt = run.z;; c = nxt++) {
    const int2 span = span_tab[c];
    const int nr = span.y - span.x;
    if (tid < nn) rlo[tid] = 0;
    if (tid == 0) total = 0;
    for (int s = tid; s < nb; s += kBlock) cnt[s] = 0;
    for (int t = tid; t < nr; t += kBlock) rinfo[t] = recs[span.x + t].y;
    for (int t = tid; t < 10 * nr; t += kBlock) rpos[t] = m.posi[10 * (int64_t)recs[span.x + t / 10].x + t % 10];
    __syncthreads();
    for (int t = tid; t < nr; t += kBlock) {
      const int node = rinfo[t] >> 16;
      if (t == 0 || (rinfo[t - 1] >> 16) != node) rlo[node] = t;
    }
    for (int t = tid; t < 10 * nr; t += kBlock) atomicAdd(&cnt[first[rinfo[t / 10] >> 16] + rpos[t]], 1);
    __syncthreads();
    int own = 0;
    for (int s = tid; s < nb; s += kBlock) {
      const int n = cnt[s];
      if (!n) continue;
      int node = 0;
      while (first[node + 1] <= s) ++node;
      const int64_t ga = m.nodes[run.x + node], gb = m.cols[m.row_ptr[4 * ga] + 4 * (s - first[node])] / 4;
      if (m.place[gb] < m.place[ga]) cnt[s] = 0;  // the pair is b's run's
      else own += 1 << cluster_log_lanes(n);
    }
    count_lanes(own, &total);
    if (!lanes) {
      if (tid == 0) nlanes[c] = (total + 63) / 64 * 64;
    } else {
      order_pairs(cnt, nb, before, at);
      for (int l = tid; l < total; l += kBlock) work[l] = 0;
      __syncthreads();
      for (int i = tid; i < 10 * nr; i += kBlock) {
        const int t = i / 10, b = i % 10, node = rinfo[t] >> 16, pos = rpos[i], n = cnt[first[node] + pos];
        if (!n) continue;
        int v = 0;  // visits of the pair before this one
        for (int u = 10 * rlo[node]; u < i; ++u) v += rpos[u] == pos;
        const int lg = cluster_log_lanes(n), lane = at[first[node] + pos] + (v & ((1 << lg) - 1));
        const int code = (rinfo[t] & 31) | (((rinfo[t] >> 8) & 15) << 5) | (b << 9);
        atomicOr(&work[lane], (unsigned long long)code << (13 * (v >> lg)));
        if (!(v >> lg)) src[lane] = (uint16_t)i;
      }
      __syncthreads();
      const int base = nlanes[c], end = nlanes[c + 1];
      if (tid == 0) {
        chunk_tab[c].y = base;
        chunk_tab[c].z = end;
      }
      for (int l = tid; l < end - base; l += kBlock) {
        ClusterLane o = {0, 0};  // idle lanes: no visits
        if (l < total) {
          const int i = src[l], t = i / 10, b = i % 10, node = rinfo[t] >> 16, pos = rpos[i], s = first[node] + pos;
          const int a = (rinfo[t] >> 8) & 15, lg = cluster_log_lanes(cnt[s]), j = l - at[s];
          const int k = (cnt[s] - j + (1 << lg) - 1) >> lg;  // visits j, j + 2^lg, ..
          const int64_t ga = m.nodes[run.x + node], gb = m.cols[m.row_ptr[4 * ga] + 4 * pos] / 4;
          // an earlier chunk of the run that adds to this pair holds an earlier incidence of its node
          bool earlier = false;
          for (int64_t r = m.inc_ptr[ga]; r < recs[span.x + rlo[node]].x; ++r)
            for (int q = 0; q < 10; ++q) earlier |= m.posi[10 * r + q] == pos;
          const int64_t e = elem_tab[(int64_t)c * kClusterElems + (rinfo[t] & 31)] & ~kClusterOwned;
          const int pos_t = m.pos[(10 * e + b) * 10 + a];
          const int64_t rb = m.row_ptr[4 * gb];
          o.x = work[l] | ((uint64_t)k << kLaneCount) | ((uint64_t)pos << kLanePos) | ((uint64_t)node << kLaneNode) |
                ((uint64_t)lg << kLaneLog) | (earlier ? 0 : kLaneFirst) | (ga == gb ? kLaneDiag : 0);
          o.y = (uint64_t)(rb / 16) | ((uint64_t)((m.row_ptr[4 * gb + 1] - rb) / 4) << kLaneDegT) |
                ((uint64_t)pos_t << kLanePosT);
        }
        lanes[base + l] = o;
      }
    }
    __syncthreads();
    if (nxt >= run.w) break;
  }
}

__global__ __launch_bounds__(kBlock) void cluster_conn_kernel(int64_t num_chunks, const int4* chunk_tab,
                                                              const uint32_t* elem_tab, const int32_t* conn,
                                                              int32_t* chunk_conn) {
  const int64_t n = num_chunks * kClusterElems * 10;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
    const int64_t s = i / 10, c = s / kClusterElems;
    const bool live = s % kClusterElems < chunk_tab[c].x;
    chunk_conn[i] = live ? conn[10 * (int64_t)(elem_tab[s] & ~kClusterOwned) + i % 10] : 0;
  }
}

// --------------------------------------------------------------- assembly
constexpr double kA = 0.5854101966249685, kB = 0.1381966011250105;  // lambda of the four points

// LDS table of one element, per point: f_a = F^{-T} grad N_a of the ten nodes
// (three each), dev(F F^T) (xx xy xz yy yz zz) and the scalars below (times
// w dv: c, c tr(F F^T)/3, p J, J, beta, tau J, 1/kappa, r1; and pi).  Odd
// strides spread the elements over the LDS banks.
enum : int { oF = 0, oDev = 30, oC = 36, oCT, oPJ, oJ, oBeta, oT, oPi, oKap = oPi + 3, oR1, kPt };
constexpr int kElemStride = 4 * kPt + 1;
static_assert(kPt == 47 && kElemStride % 2 == 1, "odd strides");
__device__ constexpr int sym(int i, int j) { return (i < j ? i : j) + (i > j ? i : j) + (i > 0 && j > 0 ? 1 : 0); }

__device__ inline double lam_at(int v, int q) { return v == q ? kA : kB; }

__device__ inline int64_t run_of(int64_t it, int64_t n, int remap) {
  const int64_t nb = gridDim.x, b = blockIdx.x;
  if (!remap || (nb & 7)) {
    const int64_t g = b + it * nb;
    return g < n ? g : -1;
  }
  // XCD x (workgroups go round the eight XCDs) takes the x-th eighth of the runs
  const int64_t per = (n + 7) >> 3, g = (b >> 3) + it * (nb >> 3);
  if (g >= per) return -1;
  const int64_t r = (b & 7) * per + g;
  return r < n ? r : -1;
}

// Stage ends: pin() forces a value here, stage_end() keeps later loads and
// arithmetic behind.  Left alone, the compiler starts the loads of all stages
// at once and spills at the 168 registers that three waves per SIMD leave
// (13 spilled registers were 3 GB of scratch traffic per assembly; with the
// stages apart the kernel takes 140 and spills none).
__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }
template <int N>
__device__ __forceinline__ void pin(double (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) pin(v[k]);
}
__device__ __forceinline__ void stage_end() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// The state of point q of element e (nodes ec), into its part of the element's
// table.
__device__ __forceinline__ void point_state(const ClusterArgs& a, int64_t e, const int32_t* ec, int q, bool owned,
                                            double* pe) {
  const MatParams mp = a.mats[a.elem_set ? a.elem_set[e] : 0];
  double lam[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) lam[v] = lam_at(v, q);
  // U[v] = sum_n (dN_n / d lambda_v) x_n, so that grad x = sum_v U[v] grad lambda_v
  double U[4][4], p = 0.0;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const double* xn = a.x + 4 * (int64_t)ec[v];
#pragma unroll
    for (int i = 0; i < 4; ++i) U[v][i] = (4.0 * lam[v] - 1.0) * xn[i];
    p += lam[v] * (2.0 * lam[v] - 1.0) * xn[3];
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    if (k == 2) stage_end();
    const int i = k < 3 ? k : k - 3, j = k < 3 ? (k == 2 ? 0 : k + 1) : 3;
    const double* xn = a.x + 4 * (int64_t)ec[4 + k];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      U[i][d] += 4.0 * lam[j] * xn[d];
      U[j][d] += 4.0 * lam[i] * xn[d];
    }
    p += 4.0 * lam[i] * lam[j] * xn[3];
  }
  // differences first (the four gradients sum to zero): a rigid part of x drops out exactly
  double D[12];
#pragma unroll
  for (int v = 1; v < 4; ++v)
#pragma unroll
    for (int i = 0; i < 4; ++i) D[4 * (v - 1) + i] = U[v][i] - U[0][i];
  pin(D);
  pin(p);
  stage_end();
  double F[9], gp[3], gl[4][3], tau, det;
  {
    double X[4][3];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int c = 0; c < 3; ++c) X[v][c] = a.coords[3 * (int64_t)ec[v] + c];
    det = dev::tet_gradlambda(X, gl);
    tau = a.stabilization ? dev::stab_tau(X, mp) : 0.0;
  }
#pragma unroll
  for (int J = 0; J < 3; ++J) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
      F[3 * i + J] = (i == J ? 1.0 : 0.0) + (D[i] * gl[1][J] + D[4 + i] * gl[2][J] + D[8 + i] * gl[3][J]);
    gp[J] = D[3] * gl[1][J] + D[7] * gl[2][J] + D[11] * gl[3][J];
  }
  pin(F);
  pin(gp);
  pin(tau);
  pin(det);
  stage_end();
  double* o = pe + kPt * q;
  const double J = dev::det3(F), iJ = 1.0 / J, W = det / 24.0;
  {
    double b[6];  // F F^T
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = i; j < 3; ++j)
        b[sym(i, j)] = F[3 * i] * F[3 * j] + F[3 * i + 1] * F[3 * j + 1] + F[3 * i + 2] * F[3 * j + 2];
    const double trb = b[0] + b[3] + b[5], third = trb / 3.0;
    b[0] -= third;
    b[3] -= third;
    b[5] -= third;
    const double Jm13 = 1.0 / cbrt(J), Jm23 = Jm13 * Jm13;
    if (owned) {
      const double m = mp.mu * (Jm23 * Jm23 * Jm13);
      double* sg = a.sigma + 4 * e + q;
#pragma unroll
      for (int k = 0; k < 9; ++k) sg[k * 4 * a.num_elems] = m * b[sym(k / 3, k % 3)] + (k % 4 == 0 ? p : 0.0);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) o[oDev + k] = b[k];
    const double C = W * (mp.mu * Jm23);
    o[oC] = C;
    o[oCT] = C * third;
  }
  o[oPJ] = W * (p * J);
  o[oJ] = W * J;
  o[oBeta] = W * (-0.5 * (J + iJ));
  o[oT] = W * J * tau;
  o[oKap] = W / mp.kappa;
  o[oR1] = W * (p / mp.kappa - 0.5 * (J - iJ));
  stage_end();
  double Fi[9], phi[4][3];
  dev::inv3(F, J, Fi);
#pragma unroll
  for (int k = 0; k < 3; ++k) o[oPi + k] = Fi[k] * gp[0] + Fi[3 + k] * gp[1] + Fi[6 + k] * gp[2];
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      phi[v][k] = Fi[k] * gl[v][0] + Fi[3 + k] * gl[v][1] + Fi[6 + k] * gl[v][2];
      o[oF + 3 * v + k] = (4.0 * lam[v] - 1.0) * phi[v][k];
    }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const int i = k < 3 ? k : k - 3, j = k < 3 ? (k == 2 ? 0 : k + 1) : 3;
#pragma unroll
    for (int d = 0; d < 3; ++d) o[oF + 12 + 3 * k + d] = 4.0 * (lam[i] * phi[j][d] + lam[j] * phi[i][d]);
  }
}

// N_a at point q (vertices: lambda (2 lambda - 1), edges: 4 lambda_i lambda_j).
__device__ inline double shape_at(int a, int q) {
  if (a < 4) return lam_at(a, q) * (2.0 * lam_at(a, q) - 1.0);
  return 4.0 * lam_at(edge_lo(a - 4), q) * lam_at(edge_hi(a - 4), q);
}

// The sums of a pair {a, b}: uu[3 i + k] = K(ai, bk) (= K(bk, ai)), pp = K(a3,
// b3), and both blocks' pressure columns and rows; r: the residual of a = b.
struct PairSum {
  double uu[9], pp, ab_c[3], ab_r[3], ba_c[3], ba_r[3], r[4];
  template <typename F>
  __device__ __forceinline__ void each(F f) {
#pragma unroll
    for (int k = 0; k < 9; ++k) f(uu[k]);
    f(pp);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      f(ab_c[k]);
      f(ab_r[k]);
      f(ba_c[k]);
      f(ba_r[k]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) f(r[k]);
  }
  template <typename F>
  __device__ __forceinline__ void all(F f) {
    each(f);
  }
};

// Adds one visit: element table P, local nodes la and lb; shape[4 a + q] = N_a
// at point q.
__device__ __forceinline__ void visit(const double* P, const double* shape, int la, int lb, bool diag, PairSum& s) {
#pragma unroll 1
  for (int q = 0; q < 4; ++q) {
    const double* p = P + kPt * q;
    double fa[3], fb[3], ha[3], hb[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      fa[k] = p[oF + 3 * la + k];
      fb[k] = p[oF + 3 * lb + k];
    }
    {
      double dv[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) dv[k] = p[oDev + k];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        ha[j] = dv[sym(j, 0)] * fa[0] + dv[sym(j, 1)] * fa[1] + dv[sym(j, 2)] * fa[2];
        hb[j] = dv[sym(j, 0)] * fb[0] + dv[sym(j, 1)] * fb[1] + dv[sym(j, 2)] * fb[2];
      }
    }
    const double d = fa[0] * fb[0] + fa[1] * fb[1] + fa[2] * fb[2];
    {
      const double C = p[oC], CT = p[oCT], PJ = p[oPJ];
      const double hd = ha[0] * fb[0] + ha[1] * fb[1] + ha[2] * fb[2];
      const double m = (-2.0 / 3.0) * C, A = PJ - (2.0 / 3.0) * CT, S = CT - PJ, gg = C * hd + CT * d;
      if (diag) {
#pragma unroll
        for (int i = 0; i < 3; ++i) s.r[i] += C * ha[i] + PJ * fa[i];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const double u = m * ha[i] + A * fa[i], v = m * fa[i], w = S * fb[i];
#pragma unroll
        for (int k = 0; k < 3; ++k) s.uu[3 * i + k] += u * fb[k] + v * hb[k] + w * fa[k];
        s.uu[4 * i] += gg;
      }
    }
    pin(s.uu);
    stage_end();
    const double Na = shape[4 * la + q], Nb = shape[4 * lb + q];
    const double J = p[oJ], be = p[oBeta], t = p[oT];
    const double pi[3] = {p[oPi], p[oPi + 1], p[oPi + 2]};
    const double pa = pi[0] * fa[0] + pi[1] * fa[1] + pi[2] * fa[2];
    const double pb = pi[0] * fb[0] + pi[1] * fb[1] + pi[2] * fb[2];
    const double td = t * d, ta = t * pa, tb = t * pb;
    const double ja = J * Na, jb = J * Nb, al = be * Na + ta, bl = be * Nb + tb;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      s.ab_c[i] += jb * fa[i];
      s.ba_c[i] += ja * fb[i];
      const double tp = td * pi[i];
      s.ab_r[i] += al * fb[i] - tb * fa[i] - tp;
      s.ba_r[i] += bl * fa[i] - ta * fb[i] - tp;
    }
    s.pp += td + p[oKap] * (Na * Nb);
    if (diag) s.r[3] += p[oR1] * Na + ta;
  }
}

// v + the partner's v for lanes that share a block, by step: 0: lane ^ 1, 1:
// lane ^ 2, 2 and 3: the mirrored lane of 8 and of 16 (whose sums agree with
// lane ^ 4 and ^ 8 by then).
template <int STEP>
__device__ inline double partner(double v) {
  if constexpr (STEP >= 4) {  // lane ^ 16, lane ^ 32: pairs with more than 48 visits
    return __shfl_xor(v, 1 << STEP, 64);
  } else {
    constexpr int ctrl = STEP == 0 ? 0xB1 : STEP == 1 ? 0x4E : STEP == 2 ? 0x141 : 0x140;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), ctrl, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), ctrl, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
  }
}
template <int STEP, typename Sum>
__device__ __forceinline__ void join(int lg, Sum& s) {
  s.all([&](double& v) {
    const double o = partner<STEP>(v);
    if (lg > STEP) v += o;
  });
}

// Where a lane's 4 x 4 block goes: rows len apart, 32-byte aligned; at = 0: none.
struct BlockPlace {
  uint64_t at;
  int len, set;  // set: store, else add
  __device__ __forceinline__ BlockPlace other() const {  // the neighbour lane's (lane ^ 1)
    BlockPlace o;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)at, 0xB1, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(at >> 32), 0xB1, 0xF, 0xF, true);
    o.at = lo | ((uint64_t)hi << 32);
    o.len = __builtin_amdgcn_update_dpp(0, len, 0xB1, 0xF, 0xF, true);
    o.set = __builtin_amdgcn_update_dpp(0, set, 0xB1, 0xF, 0xF, true);
    return o;
  }
  __device__ __forceinline__ void put(int i, int half, double2 v) const {
    if (!at) return;
    double2* o = reinterpret_cast<double2*>(at) + (int64_t)i * (len / 2) + half;
    if (!set) {
      const double2 w = *o;
      v.x += w.x;
      v.y += w.y;
    }
    *o = v;
  }
};

// Stores the lanes' blocks, two lanes to a block: a row of a block is 32 bytes,
// and one lane's two 16-byte stores reach L2 as two requests where the two
// lanes' one store is a single one.
__device__ __forceinline__ void put_block(const BlockPlace& mine, int half, const double* uu, bool transpose,
                                          const double* col, const double* row, double pp) {
  const BlockPlace other = mine.other();
  const BlockPlace even = half ? other : mine, odd = half ? mine : other;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = i < 3 ? (k < 3 ? (transpose ? uu[3 * k + i] : uu[3 * i + k]) : col[i]) : k < 3 ? row[k] : pp;
    const double2 got = {partner<0>(half ? v[0] : v[2]), partner<0>(half ? v[1] : v[3])};
    const double2 lo = {v[0], v[1]}, hi = {v[2], v[3]};
    even.put(i, half, half ? got : lo);
    odd.put(i, half, half ? hi : got);
  }
}

constexpr int kClusterThreads = 192;
static_assert(4 * kClusterElems <= kClusterThreads && kClusterNodes <= 64, "one thread per point, one per node");

// A barrier for what the workgroup shares in LDS: __syncthreads() would also
// wait until every store of the chunk's blocks has reached memory.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A pending clear of the functional's derivative goes along with the runs, each
// node being in one: a launch less (162 tets 34.4 -> 32.6 us, 3,072 quadratic
// ones 51.1 -> 46.6).
__device__ __forceinline__ void clear_node(double* zero, int32_t n) {
  double2* z = reinterpret_cast<double2*>(zero + 4 * (int64_t)n);
  z[0] = z[1] = double2{0.0, 0.0};
}

// The chunks of a workgroup's runs, one after the other: chunk r is run r's
// first, its further ones are r.z .. r.w.
struct ClusterCursor {
  int64_t it = 0, run, c;
  int4 r;
  int x;
  __device__ __forceinline__ explicit ClusterCursor(const ClusterArgs& a) { load(a); }
  __device__ __forceinline__ void load(const ClusterArgs& a) {
    c = run = run_of(it, a.num_runs, a.xcd_remap);
    if (run < 0) return;
    r = a.runs[run];
    x = r.z;
  }
  __device__ __forceinline__ bool valid() const { return run >= 0; }
  __device__ __forceinline__ void next(const ClusterArgs& a) {
    if (x < r.w) {
      c = x++;
      return;
    }
    ++it;
    load(a);
  }
};

template <bool TR>
__global__ __launch_bounds__(kClusterThreads, 3) void cluster_kernel(ClusterArgs a) {
  __shared__ double pe[kClusterElems * kElemStride];
  __shared__ double shape[40];
  __shared__ int64_t nbase[kClusterNodes];
  __shared__ int32_t nid[kClusterNodes], nlen[kClusterNodes];
  const int tid = threadIdx.x, lane = tid & 63, el = tid >> 2;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 40) shape[tid] = shape_at(tid >> 2, tid & 3);

  ClusterCursor cur(a);
  if (!cur.valid()) return;  // the whole workgroup
  for (;;) {
    const int4 ch = a.chunks[cur.c];
    ClusterCursor nxt = cur;
    nxt.next(a);
    if (wave == 2 && lane < cur.r.y - cur.r.x) {  // the run's nodes: CSR base and row length
      const int32_t n = a.nodes[cur.r.x + lane];
      const int64_t b = a.row_ptr[4 * (int64_t)n];
      nid[lane] = n;
      if (a.zero) clear_node(a.zero, n);
      nbase[lane] = b;
      nlen[lane] = (int)(a.row_ptr[4 * (int64_t)n + 1] - b);
    }
    int q = tid & 3;
    asm volatile("" : "+v"(q));  // what hangs on it is formed here, not kept in registers over the loop
    if (el < ch.x) {
      const int64_t s = cur.c * kClusterElems + el;
      const uint32_t w = a.chunk_elems[s];
      point_state(a, (int64_t)(w & ~kClusterOwned), a.chunk_conn + 10 * s, q, a.save_state && (w & kClusterOwned),
                  pe + kElemStride * el);
    }
    lds_barrier();  // point states and node table are there
    for (int g = ch.y + 64 * wave; g < ch.z; g += kClusterThreads) {
      const ClusterLane e = a.lanes[g + lane];
      const int n = (int)(e.x >> kLaneCount) & 3, lg = (int)(e.x >> kLaneLog) & 7;
      const bool diag = e.x & kLaneDiag;
      PairSum s;
      s.each([](double& v) { v = 0.0; });
      uint64_t code = e.x;
      for (int v = 0; v < n; ++v, code >>= 13)
        visit(pe + kElemStride * (int)(code & 31), shape, (int)(code >> 5) & 15, (int)(code >> 9) & 15, diag, s);
      const int most = __builtin_amdgcn_readfirstlane(lg);  // the first lane's pair has the most lanes
      if (most > 0) join<0>(lg, s);
      if (most > 1) join<1>(lg, s);
      if (most > 2) join<2>(lg, s);
      if (most > 3) join<3>(lg, s);
      const bool mine = n > 0 && !(lane & ((1 << lg) - 1));
      const int nl = (int)(e.x >> kLaneNode) & 31;
      const bool first = e.x & kLaneFirst;
      BlockPlace ab = {0, nlen[nl], a.overwrite_vals && first}, ba = ab;
      if (mine) ab.at = reinterpret_cast<uint64_t>(a.vals + nbase[nl] + 4 * ((int)(e.x >> kLanePos) & 511));
      if (mine && !diag) {
        ba.at = reinterpret_cast<uint64_t>(a.vals + 16 * (int64_t)(e.y & ((uint64_t(1) << kLaneDegT) - 1)) +
                                           4 * (int64_t)(e.y >> kLanePosT));
        ba.len = 4 * ((int)(e.y >> kLaneDegT) & 4095);
      }
      // block (a, b); of the transpose, what the matrix has at (b, a), transposed
      put_block(ab, lane & 1, s.uu, false, TR ? s.ba_r : s.ab_c, TR ? s.ba_c : s.ab_r, s.pp);
      put_block(ba, lane & 1, s.uu, true, TR ? s.ab_r : s.ba_c, TR ? s.ab_c : s.ba_r, s.pp);
      if (mine && diag) {
        double* o = a.R + 4 * (int64_t)nid[nl];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = ((a.overwrite_R && first) ? 0.0 : o[i]) + s.r[i];
      }
    }
    if (!nxt.valid()) break;
    if (nxt.run == cur.run) __threadfence();  // the next chunk may add to this one's blocks
    lds_barrier();                          // the point states are free
    cur = nxt;
  }
}

// ----------------------------------------------------------- linear tets
// One workgroup per run of nodes [lo, hi): its incidences in LDS, the distinct
// elements among them numbered by first appearance.
struct LinearRun {
  int nodes[kLinearNodes], first[kLinearNodes + 1], rec0[kLinearNodes + 1];
  alignas(16) int elem[kLinearRecs];
  int info[kLinearRecs];  // first incidence of the element << 2 | local node
  alignas(8) uint16_t pos[4 * kLinearRecs];
  uint16_t slot[kLinearRecs];
  uint8_t node[kLinearRecs];
  int ne;
};
// false: too many incidences or blocks (nothing else is set then)
__device__ bool linear_load(const ClusterMesh& m, int64_t lo, int64_t hi, LinearRun& r) {
  static_assert(kLinearNodes == 8, "prefixes over eight lanes");
  const int tid = threadIdx.x, nn = (int)(hi - lo);
  __syncthreads();
  if (tid < 64) {
    // no overflow: eight terms of at most 2^20, which is over both limits; a node without elements ends here too
    constexpr int64_t kMany = 1 << 20;
    int deg = 0, inc = 0;
    if (tid < nn) {
      const int64_t n = m.nodes[lo + tid], d = (m.row_ptr[4 * n + 1] - m.row_ptr[4 * n]) / 4,
                    k = m.inc_ptr[n + 1] - m.inc_ptr[n];
      r.nodes[tid] = (int)n;
      deg = (int)min(d, kMany);
      inc = (int)(k > 0 ? min(k, kMany) : kMany);
    }
    for (int off = 1; off < kLinearNodes; off <<= 1) {
      const int d = __shfl_up(deg, off, 64), k = __shfl_up(inc, off, 64);
      if (tid >= off) {
        deg += d;
        inc += k;
      }
    }
    if (tid < nn) {
      r.first[tid + 1] = deg;
      r.rec0[tid + 1] = inc;
    }
    if (tid == 0) r.first[0] = r.rec0[0] = 0;
  }
  __syncthreads();
  const int n = r.rec0[nn];
  if (n > kLinearRecs || r.first[nn] > kClusterSlots) return false;
  for (int t = tid; t < n; t += kBlock) {
    int node = 0;
    while (r.rec0[node + 1] <= t) ++node;
    const int64_t k = m.inc_ptr[r.nodes[node]] + (t - r.rec0[node]);
    const int32_t s = m.inc[k];
    r.elem[t] = s / 4;
    r.info[t] = s % 4;
    r.node[t] = (uint8_t)node;
    *reinterpret_cast<ushort4*>(r.pos + 4 * t) = reinterpret_cast<const ushort4*>(m.posi)[k];
  }
  __syncthreads();
  for (int t = tid; t < n; t += kBlock) {
    const int e = r.elem[t];
    int u = 0;  // found at t at the latest
    for (;; u += 4) {
      const int4 v = *reinterpret_cast<const int4*>(r.elem + u);
      if (v.x == e || v.y == e || v.z == e || v.w == e) {
        u += v.x == e ? 0 : v.y == e ? 1 : v.z == e ? 2 : 3;
        break;
      }
    }
    r.info[t] |= u << 2;
  }
  __syncthreads();
  if (tid < 64) {
    int base = 0;
    for (int t0 = 0; t0 < n; t0 += 64) {
      const int t = t0 + tid;
      const bool is = t < n && (r.info[t] >> 2) == t;
      const unsigned long long b = __ballot(is);
      if (is) r.slot[t] = (uint16_t)(base + __popcll(b & ((1ull << tid) - 1)));
      base += __popcll(b);
    }
    if (tid == 0) r.ne = base;
  }
  __syncthreads();
  return true;
}

// cnt: the visits of every pair of a loaded run of rn nodes, 0 where the pair is
// another run's.  The lanes they take.
__device__ int linear_count(const ClusterMesh& m, const LinearRun& r, int rn, int* cnt, int* total) {
  const int tid = threadIdx.x, n = r.rec0[rn], nb = r.first[rn];
  if (tid == 0) *total = 0;
  for (int s = tid; s < nb; s += kBlock) cnt[s] = 0;
  __syncthreads();
  for (int i = tid; i < 4 * n; i += kBlock) atomicAdd(&cnt[r.first[r.node[i >> 2]] + r.pos[i]], 1);
  __syncthreads();
  int own = 0;
  for (int s = tid; s < nb; s += kBlock) {
    const int c = cnt[s];
    if (!c) continue;
    int node = 0;
    while (r.first[node + 1] <= s) ++node;
    const int64_t ga = r.nodes[node], gb = m.cols[m.row_ptr[4 * ga] + 4 * (s - r.first[node])] / 4;
    if (m.place[gb] < m.place[ga]) cnt[s] = 0;  // the pair is b's run's
    else own += 1 << cluster_log_lanes(c);
  }
  count_lanes(own, total);
  return *total;
}

// parts[g]: the runs (1, 2, 4 or 8) that group g's nodes need to fit; nlanes,
// nelems [8 g + i]: the lanes (whole wavefronts) and elements of its run i, 0
// where there is none.
__global__ __launch_bounds__(kBlock) void linear_split_kernel(ClusterMesh m, int64_t nn, int32_t* parts,
                                                              int32_t* nlanes, int32_t* nelems, int32_t* bad) {
  __shared__ LinearRun r;
  __shared__ int cnt[kClusterSlots], total;
  __shared__ int2 size[kLinearNodes];
  const int64_t lo = (int64_t)blockIdx.x * kLinearNodes, hi = min(lo + kLinearNodes, nn);
  int p = 1;
  for (; p <= kLinearNodes; p *= 2) {
    const int64_t step = kLinearNodes / p;
    bool fits = true;
    int i = 0;
    for (int64_t a = lo; a < hi && fits; a += step, ++i) {
      const int64_t b = min(a + step, hi);
      fits = linear_load(m, a, b, r) && r.ne <= kLinearElems;
      if (!fits) break;
      const int lanes = linear_count(m, r, (int)(b - a), cnt, &total);
      if (threadIdx.x == 0) size[i] = int2{(lanes + 63) / 64 * 64, r.ne};
    }
    if (fits) break;
  }
  __syncthreads();
  const bool fit = p <= kLinearNodes;
  const int64_t step = kLinearNodes / (fit ? p : kLinearNodes);
  const int np = (int)((hi - lo + step - 1) / step), tid = threadIdx.x;
  if (tid < kLinearNodes) {
    nlanes[kLinearNodes * (int64_t)blockIdx.x + tid] = fit && tid < np ? size[tid].x : 0;
    nelems[kLinearNodes * (int64_t)blockIdx.x + tid] = fit && tid < np ? size[tid].y : 0;
  }
  if (tid == 0) {
    parts[blockIdx.x] = np;
    if (!fit) atomicMax(bad, 1);
  }
}

__global__ __launch_bounds__(kBlock) void linear_tables_kernel(ClusterMesh m, int64_t nn, const int32_t* parts,
                                                               const int32_t* nlanes, const int32_t* nelems,
                                                               int4* runs, int2* spans, int32_t* elems,
                                                               ClusterLane* lanes) {
  __shared__ LinearRun r;
  __shared__ int cnt[kClusterSlots], before[kRanks * kGroups], total;
  __shared__ uint16_t at[kClusterSlots], src[4 * kLinearRecs];  // first lane of a pair; a lane's first visit
  __shared__ unsigned long long work[4 * kLinearRecs];          // the visits of every lane
  const int tid = threadIdx.x;
  const int64_t lo = (int64_t)blockIdx.x * kLinearNodes, hi = min(lo + kLinearNodes, nn);
  const int run0 = parts[blockIdx.x], np = parts[blockIdx.x + 1] - run0;
  int64_t step = kLinearNodes;  // np runs came from 1, 2, 4 or 8 equal parts of the group, the last ones empty at the end of the nodes
  while ((hi - lo + step - 1) / step < np) step /= 2;
  for (int p = 0; p < np; ++p) {
    const int64_t a0 = lo + p * step, a1 = min(a0 + step, hi), q = kLinearNodes * (int64_t)blockIdx.x + p;
    const int run = run0 + p, rn = (int)(a1 - a0);
    linear_load(m, a0, a1, r);  // fits: linear_split saw to it
    linear_count(m, r, rn, cnt, &total);
    order_pairs(cnt, r.first[rn], before, at);
    for (int l = tid; l < total; l += kBlock) work[l] = 0;
    __syncthreads();
    const int n = r.rec0[rn], base = nlanes[q], end = nlanes[q + 1], e0 = nelems[q];
    if (tid == 0) {
      runs[run] = int4{(int)a0, (int)a1, e0, r.ne};
      spans[run] = int2{base, end};
    }
    for (int t = tid; t < n; t += kBlock)
      if ((r.info[t] >> 2) == t) elems[e0 + r.slot[t]] = r.elem[t];
    for (int i = tid; i < 4 * n; i += kBlock) {
      const int t = i >> 2, b = i & 3, node = r.node[t], pos = r.pos[i], s = r.first[node] + pos, c = cnt[s];
      if (!c) continue;
      int v = 0;  // visits of the pair before this one
      for (int u = r.rec0[node]; u <= t; ++u) {
        const ushort4 w = *reinterpret_cast<const ushort4*>(r.pos + 4 * u);
        const bool all = u < t;
        v += (w.x == pos && (all || b > 0)) + (w.y == pos && (all || b > 1)) + (w.z == pos && (all || b > 2)) +
             (w.w == pos && all);
      }
      const int lg = cluster_log_lanes(c), lane = at[s] + (v & ((1 << lg) - 1));
      const int code = r.slot[r.info[t] >> 2] | ((r.info[t] & 3) << 9) | (b << 11);
      atomicOr(&work[lane], (unsigned long long)code << (13 * (v >> lg)));
      if (!(v >> lg)) src[lane] = (uint16_t)i;
    }
    __syncthreads();
    for (int l = tid; l < end - base; l += kBlock) {
      ClusterLane o = {0, 0};  // idle lanes: no visits
      if (l < total) {
        const int i = src[l], t = i >> 2, b = i & 3, a = r.info[t] & 3, node = r.node[t], pos = r.pos[i];
        const int s = r.first[node] + pos, lg = cluster_log_lanes(cnt[s]), j = l - at[s];
        const int k = (cnt[s] - j + (1 << lg) - 1) >> lg;  // visits j, j + 2^lg, ..
        const int64_t ga = r.nodes[node], gb = m.cols[m.row_ptr[4 * ga] + 4 * pos] / 4, rb = m.row_ptr[4 * gb];
        const uint64_t pos_t = m.pos[((int64_t)r.elem[t] * 4 + b) * 4 + a];
        o.x = work[l] | ((uint64_t)k << kLaneCount) | ((uint64_t)pos << kLanePos) | ((uint64_t)node << kLaneNode) |
              ((uint64_t)lg << kLaneLog) | kLaneFirst | (ga == gb ? kLaneDiag : 0);
        o.y = (uint64_t)(rb / 16) | ((uint64_t)((m.row_ptr[4 * gb + 1] - rb) / 4) << kLaneDegT) | (pos_t << kLanePosT);
      }
      lanes[base + l] = o;
    }
  }
}

// An element's point state: f_a = F^{-T} grad N_a of its nodes, then with
// dev = dev(b) (neo-Hookean: b = F F^T; J2: the trial elastic b) and the scalars
// the same tangent as the quadratic elements' (top of this file), with C times
// theta for J2 and, where it yields, one more term.  J2's stress is s = theta
// mu dev, theta = 1 - 2 mubar dgam / |s_tr|; along L = e_k (x) f_b, with ed = dev
// f, ee = dev ed, t3 = tr b / 3, nu = mu / |s_tr| and the last Newton iterate's
// derivative alpha d|s_tr| + beta d mubar,
//   ds = theta ds_tr + N kappa_k,  N f_a = nu ed_a,
//   kappa_k = A (2 mu nu (ee_b + t3 ed_b) - 2/3 |s_tr| f_b)_k + B (2 mu / 3) ed_bk,
//   A = 2 mubar (dgam / |s_tr| - alpha),  B = -2 (dgam + mubar beta),
// so K(ai, bk) += ed_ai (q1 ee_b + q2 ed_b + q3 f_b)_k.  All times w dv.
// dev is traceless: its last entry is not kept.
enum : int { lF = 0, lDev = 12, lC = 17, lCT, lPJ, lJ, lBeta, lT, lPi, lKap = lPi + 3, lR1, lQ1, lQ2, lQ3, lPt };
static_assert(lPt == kLinearPoint - 1, "31 of 32 doubles an element");

// Bound by its memory traffic (J2: some 520 bytes an element, 256 of them the
// state; 0.85 ms = 3.2 TB/s on the 5.3 M-tet bar, two waves a SIMD of 204
// registers; held to 168 for three waves it took 0.91).
template <int MODEL>
__global__ __launch_bounds__(256) void linear_points_kernel(AsmArgs a) {
  __shared__ double stage[4][64 * 17];
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x, ne = a.num_elems;
  double o[kLinearPoint];
  o[kLinearPoint - 1] = 0.0;
  if (e < ne) {
    const int4 ec4 = reinterpret_cast<const int4*>(a.conn)[e];
    const int32_t ec[4] = {ec4.x, ec4.y, ec4.z, ec4.w};
    const MatParams mp = a.mats[a.elem_set ? a.elem_set[e] : 0];
    double D[3][4], p = 0.0;
    {
      double U[4][4];
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) U[v][i] = a.x[4 * (int64_t)ec[v] + i];
      p = 0.25 * ((U[0][3] + U[1][3]) + (U[2][3] + U[3][3]));
#pragma unroll
      for (int v = 1; v < 4; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) D[v - 1][i] = U[v][i] - U[0][i];
    }
    double gl[4][3], W, tau;
    {
      double X[4][3];
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int c = 0; c < 3; ++c) X[v][c] = a.coords[3 * (int64_t)ec[v] + c];
      W = dev::tet_gradlambda(X, gl) / 6.0;
      tau = a.stabilization ? dev::stab_tau(X, mp) : 0.0;
    }
    dev::QP qp;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        qp.H[3 * i + j] = D[0][i] * gl[1][j] + D[1][i] * gl[2][j] + D[2][i] * gl[3][j];
        qp.F[3 * i + j] = qp.H[3 * i + j] + (i == j ? 1.0 : 0.0);
      }
      qp.g[j] = D[0][3] * gl[1][j] + D[1][3] * gl[2][j] + D[2][3] * gl[3][j];
    }
    qp.p = p;
    qp.J = dev::det3(qp.F);
    dev::inv3(qp.F, qp.J, qp.Fi);
    const double J = qp.J, iJ = 1.0 / J;
    if constexpr (MODEL == MODEL_NEOHOOKEAN) {
      double b[6];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = i; j < 3; ++j)
          b[sym(i, j)] = qp.F[3 * i] * qp.F[3 * j] + qp.F[3 * i + 1] * qp.F[3 * j + 1] + qp.F[3 * i + 2] * qp.F[3 * j + 2];
      const double third = (b[0] + b[3] + b[5]) / 3.0;
      b[0] -= third;
      b[3] -= third;
      b[5] -= third;
      const double Jm13 = 1.0 / cbrt(J), Jm23 = Jm13 * Jm13;
      if (a.save_state) {
        const double m = mp.mu * (Jm23 * Jm23 * Jm13);
#pragma unroll
        for (int k = 0; k < 9; ++k) a.sigma[k * ne + e] = m * b[sym(k / 3, k % 3)] + (k % 4 == 0 ? p : 0.0);
      }
#pragma unroll
      for (int k = 0; k < 5; ++k) o[lDev + k] = b[k];
      o[lC] = W * (mp.mu * Jm23);
      o[lCT] = o[lC] * third;
      o[lQ1] = o[lQ2] = o[lQ3] = 0.0;
    } else {
      double Fpo[9];
      for (int k = 0; k < 9; ++k) Fpo[k] = a.Fp_old[k * ne + e];
      dev::J2Model m;
      m.init(qp, mp, Fpo, a.eqps_old[e]);
      if (m.failed()) atomicOr(a.status, 1);
      if (a.save_state) {
        a.eqps[e] = m.alpha;
        if (m.plastic) {
          double Fpn[9];
          m.new_Fp(Fpo, Fpn);
          for (int k = 0; k < 9; ++k) a.Fp[k * ne + e] = Fpn[k];
        }
        for (int k = 0; k < 9; ++k) a.sigma[k * ne + e] = m.sig[k];
      }
      const double mu = mp.mu, t3 = m.mubar / mu;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = i; j < 3; ++j)
          if (i < 2) o[lDev + sym(i, j)] = m.str[3 * i + j] / mu;
      double theta = 1.0, q1 = 0.0, q2 = 0.0, q3 = 0.0;
      if (m.plastic) {
        double X, al, bt;
        (void)m.newton(1.0, 0.0, X, al);
        (void)m.newton(0.0, 1.0, X, bt);
        theta = 1.0 - 2.0 * m.mubar * m.dgam / m.smag;
        const double A = 2.0 * m.mubar * (m.dgam / m.smag - al), B = -2.0 * (m.dgam + m.mubar * bt);
        const double nu = mu / m.smag;
        q1 = W * nu * (2.0 * mu * A * nu);
        q2 = W * nu * (2.0 * mu * A * nu * t3 + (2.0 * mu / 3.0) * B);
        q3 = (-2.0 / 3.0) * W * A * mu;
      }
      o[lC] = W * (theta * mu);
      o[lCT] = o[lC] * t3;
      o[lQ1] = q1;
      o[lQ2] = q2;
      o[lQ3] = q3;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        o[lF + 3 * v + k] = qp.Fi[k] * gl[v][0] + qp.Fi[3 + k] * gl[v][1] + qp.Fi[6 + k] * gl[v][2];
#pragma unroll
    for (int k = 0; k < 3; ++k) o[lPi + k] = qp.Fi[k] * qp.g[0] + qp.Fi[3 + k] * qp.g[1] + qp.Fi[6 + k] * qp.g[2];
    o[lPJ] = W * (p * J);
    o[lJ] = W * J;
    o[lBeta] = W * (-0.5 * (J + iJ));
    o[lT] = W * J * tau;
    o[lKap] = W / mp.kappa;
    o[lR1] = W * (p / mp.kappa - 0.5 * (J - iJ));
  }
  // Out through LDS, 16 values a round: eight lanes then store an element's
  // 128 bytes together, where a lane's own 16-byte stores lie 256 bytes apart
  // (5.3 M-tet J2 bar: 0.98 -> 0.85 ms).
  const int lane = threadIdx.x & 63;
  double* w = stage[threadIdx.x >> 6];
  const int64_t e0 = e - lane;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 16; ++k) w[17 * lane + k] = o[16 * h + k];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = 8 * j + (lane >> 3), k = 2 * (lane & 7);
      if (e0 + i < ne)
        *reinterpret_cast<double2*>(a.pt + kLinearPoint * (e0 + i) + 16 * h + k) = double2{w[17 * i + k], w[17 * i + k + 1]};
    }
  }
}

// A pair's sums for linear tets: with plastic points K(ai, bk) and K(bk, ai) differ (vu[3 i + k] = K(bk, ai)).
template <bool PLASTIC>
struct LinearSum : PairSum {
  double vu[PLASTIC ? 9 : 1];
  template <typename F>
  __device__ __forceinline__ void all(F f) {
    each(f);
    if constexpr (PLASTIC)
#pragma unroll
      for (int k = 0; k < 9; ++k) f(vu[k]);
  }
};

template <bool PLASTIC>
__device__ __forceinline__ void linear_visit(const double* p, int la, int lb, bool diag, LinearSum<PLASTIC>& s) {
  double fa[3], fb[3], ha[3], hb[3], dv[6];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    fa[k] = p[lF + 3 * la + k];
    fb[k] = p[lF + 3 * lb + k];
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) dv[k] = p[lDev + k];
  dv[5] = -(dv[0] + dv[3]);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    ha[j] = dv[sym(j, 0)] * fa[0] + dv[sym(j, 1)] * fa[1] + dv[sym(j, 2)] * fa[2];
    hb[j] = dv[sym(j, 0)] * fb[0] + dv[sym(j, 1)] * fb[1] + dv[sym(j, 2)] * fb[2];
  }
  const double d = fa[0] * fb[0] + fa[1] * fb[1] + fa[2] * fb[2];
  {
    const double C = p[lC], CT = p[lCT], PJ = p[lPJ];
    const double hd = ha[0] * fb[0] + ha[1] * fb[1] + ha[2] * fb[2];
    const double m = (-2.0 / 3.0) * C, A = PJ - (2.0 / 3.0) * CT, S = CT - PJ, gg = C * hd + CT * d;
    if (diag) {
#pragma unroll
      for (int i = 0; i < 3; ++i) s.r[i] += C * ha[i] + PJ * fa[i];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double u = m * ha[i] + A * fa[i], v = m * fa[i], w = S * fb[i];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        double t = u * fb[k] + v * hb[k] + w * fa[k];
        if (i == k) t += gg;
        s.uu[3 * i + k] += t;
        if constexpr (PLASTIC) s.vu[3 * i + k] += t;
      }
    }
  }
  pin(s.uu);
  stage_end();
  if constexpr (PLASTIC) {
    const double q1 = p[lQ1], q2 = p[lQ2], q3 = p[lQ3];
    auto extra = [&](const double* h, const double* f, int j) {  // q1 ee + q2 ed + q3 f
      return q1 * (dv[sym(j, 0)] * h[0] + dv[sym(j, 1)] * h[1] + dv[sym(j, 2)] * h[2]) + q2 * h[j] + q3 * f[j];
    };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double xa = extra(ha, fa, k), xb = extra(hb, fb, k);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        s.uu[3 * i + k] += ha[i] * xb;
        s.vu[3 * k + i] += hb[i] * xa;
      }
    }
    pin(s.uu);
    pin(s.vu);
    stage_end();
  }
  constexpr double N = 0.25;
  const double J = p[lJ], be = p[lBeta], t = p[lT];
  const double pi[3] = {p[lPi], p[lPi + 1], p[lPi + 2]};
  const double pa = pi[0] * fa[0] + pi[1] * fa[1] + pi[2] * fa[2];
  const double pb = pi[0] * fb[0] + pi[1] * fb[1] + pi[2] * fb[2];
  const double td = t * d, ta = t * pa, tb = t * pb, jn = J * N, al = be * N + ta, bl = be * N + tb;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    s.ab_c[i] += jn * fa[i];
    s.ba_c[i] += jn * fb[i];
    const double tp = td * pi[i];
    s.ab_r[i] += al * fb[i] - tb * fa[i] - tp;
    s.ba_r[i] += bl * fa[i] - ta * fb[i] - tp;
  }
  s.pp += td + p[lKap] * (N * N);
  if (diag) s.r[3] += p[lR1] * N + ta;
}

// Bound by latency and the occupancy that hides it (blocks stored once, 1.75 GB
// on the 5.3 M-tet J2 bar; states read about three times, each element being in
// three runs; 16 bytes of work list per lane).  There it takes 1.57 ms, and with
// the point pass 2.4 ms, where the element matrices (2 KB a tet) through memory
// and their gather took 9.6; on 162 tets 34 against 41 us, so no size keeps the
// two passes.  Eight vertices a run: about 176 lanes, three waves; sixteen would
// read the states 2.5 instead of 2.9 times but leave two workgroups a CU.  The
// states come in with seven loads in flight a thread (one: 2.6 ms; fourteen
// spill: 3.7), and plastic visits in stages that keep to 168 registers (with
// two waves a SIMD instead 2.2 ms; unstaged, spilling, 4.7).
constexpr int kLinearStride = lPt;  // odd: the elements spread over the LDS banks
constexpr int kLinearThreads = 192;

template <bool PLASTIC, bool TR>
__global__ __launch_bounds__(kLinearThreads, PLASTIC ? 3 : 4) void linear_cluster_kernel(LinearArgs a) {
  __shared__ double pe[kLinearElems * kLinearStride];
  __shared__ int64_t nbase[kLinearNodes];
  __shared__ int32_t nid[kLinearNodes], nlen[kLinearNodes];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int64_t it = 0;; ++it) {
    const int64_t run = run_of(it, a.num_runs, a.xcd_remap);
    if (run < 0) break;
    const int4 r = a.runs[run];
    const int2 sp = a.spans[run];
    if (it > 0) lds_barrier();  // the last run's states are free
    if (tid < r.y - r.x) {  // the run's nodes: CSR base and row length
      const int32_t n = a.nodes[r.x + tid];
      const int64_t b = a.row_ptr[4 * (int64_t)n];
      nid[tid] = n;
      nbase[tid] = b;
      nlen[tid] = (int)(a.row_ptr[4 * (int64_t)n + 1] - b);
    }
    int g = sp.x + 64 * wave;
    ClusterLane e = {0, 0};  // a wave's first lane work is loaded with the states
    if (g < sp.y) e = a.lanes[g + lane];
    // 16 threads copy an element's state, 16 bytes each; seven loads in flight
    constexpr int kStep = kLinearThreads / 16, kBatch = 7;
    static_assert(kLinearElems <= 2 * kStep * kBatch, "two batches hold a run");
    int q = tid;
    asm volatile("" : "+v"(q));  // or fourteen addresses are kept over the runs, and spill
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i0 = q / 16 + h * kStep * kBatch, k = q & 15;
      int32_t id[kBatch];
      double2 v[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) id[j] = i0 + kStep * j < r.w ? a.elems[r.z + i0 + kStep * j] : -1;
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
        if (id[j] >= 0) v[j] = reinterpret_cast<const double2*>(a.pt + (int64_t)kLinearPoint * id[j])[k];
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
        if (id[j] >= 0) {
          double* o = pe + kLinearStride * (i0 + kStep * j) + 2 * k;
          o[0] = v[j].x;
          if (k < 15) o[1] = v[j].y;
        }
    }
    lds_barrier();
    for (; g < sp.y; g += kLinearThreads) {
      if (g >= sp.x + kLinearThreads) e = a.lanes[g + lane];
      const int n = (int)(e.x >> kLaneCount) & 3, lg = (int)(e.x >> kLaneLog) & 7;
      const bool diag = e.x & kLaneDiag;
      LinearSum<PLASTIC> s;
      s.all([](double& v) { v = 0.0; });
      uint64_t code = e.x;
#pragma unroll 1
      for (int v = 0; v < n; ++v, code >>= 13)
        linear_visit<PLASTIC>(pe + kLinearStride * (int)(code & 511), (int)(code >> 9) & 3, (int)(code >> 11) & 3, diag,
                              s);
      const int most = __builtin_amdgcn_readfirstlane(lg);  // the first lane's pair has the most lanes
      if (most > 0) join<0>(lg, s);
      if (most > 1) join<1>(lg, s);
      if (most > 2) join<2>(lg, s);
      if (most > 3) join<3>(lg, s);
      if (most > 4) join<4>(lg, s);
      if (most > 5) join<5>(lg, s);
      const bool mine = n > 0 && !(lane & ((1 << lg) - 1));
      const int nl = (int)(e.x >> kLaneNode) & 31;
      BlockPlace ab = {0, nlen[nl], a.overwrite_vals}, ba = ab;
      if (mine) ab.at = reinterpret_cast<uint64_t>(a.vals + nbase[nl] + 4 * ((int)(e.x >> kLanePos) & 511));
      if (mine && !diag) {
        ba.at = reinterpret_cast<uint64_t>(a.vals + 16 * (int64_t)(e.y & ((uint64_t(1) << kLaneDegT) - 1)) +
                                           4 * (int64_t)(e.y >> kLanePosT));
        ba.len = 4 * ((int)(e.y >> kLaneDegT) & 4095);
      }
      const double* vu = PLASTIC ? s.vu : s.uu;
      put_block(ab, lane & 1, TR ? vu : s.uu, false, TR ? s.ba_r : s.ab_c, TR ? s.ba_c : s.ab_r, s.pp);
      put_block(ba, lane & 1, TR ? s.uu : vu, true, TR ? s.ab_r : s.ba_c, TR ? s.ab_c : s.ba_r, s.pp);
      if (mine && diag) {
        double* o = a.R + 4 * (int64_t)nid[nl];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = (a.overwrite_R ? 0.0 : o[i]) + s.r[i];
        if (a.zero) clear_node(a.zero, nid[nl]);  // at the node table it cost the plastic kernel 2%
      }
    }
  }
}

}  // namespace

// scratch of the sort over n nodes and of scans over up to n + 1 entries
hipError_t cluster_temp_bytes(int64_t nn, size_t* bytes) {
  size_t a = 0, b = 0;
  hipError_t err = hipcub::DeviceRadixSort::SortPairs(nullptr, a, (const int32_t*)nullptr, (int32_t*)nullptr,
                                                      (const int32_t*)nullptr, (int32_t*)nullptr, (int)nn, 0, 31);
  if (err != hipSuccess) return err;
  err = hipcub::DeviceScan::ExclusiveSum(nullptr, b, (const int32_t*)nullptr, (int32_t*)nullptr, (int)(nn + 1));
  *bytes = std::max(a, b);
  return err;
}

namespace {
// nodes: the nodes along the Morton curve; place: its inverse.
hipError_t morton_order(const double* coords, int64_t nn, void* temp, size_t temp_bytes, unsigned long long* box,
                        uint32_t* code, uint32_t* code_sorted, int32_t* place, int32_t* iota, int32_t* nodes,
                        hipStream_t s) {
  hipError_t err = hipMemsetAsync(box, 0xff, 3 * sizeof(*box), s);
  if (err == hipSuccess) err = hipMemsetAsync(box + 3, 0, 3 * sizeof(*box), s);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(cluster_box_kernel, dim3(std::min(grid_for(nn), 256u)), dim3(kBlock), 0, s, coords, nn, box);
  hipLaunchKernelGGL(cluster_morton_kernel, dim3(grid_for(nn)), dim3(kBlock), 0, s, coords, nn, box, code, iota);
  err = hipGetLastError();
  if (err != hipSuccess) return err;
  size_t tb = temp_bytes;
  err = hipcub::DeviceRadixSort::SortPairs(temp, tb, code, code_sorted, iota, nodes, (int)nn, 0, 30, s);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(cluster_place_kernel, dim3(grid_for(nn)), dim3(kBlock), 0, s, nodes, nn, place);
  return hipGetLastError();
}
}  // namespace

hipError_t cluster_order(const int32_t* conn, const double* coords, int64_t ne, int64_t nn, void* temp,
                         size_t temp_bytes, unsigned long long* box, int32_t* keys, int32_t* keys_sorted,
                         int32_t* rank, int32_t* place, int32_t* nodes, int64_t* seg, hipStream_t s) {
  hipError_t err = morton_order(coords, nn, temp, temp_bytes, box, reinterpret_cast<uint32_t*>(keys),
                                reinterpret_cast<uint32_t*>(keys_sorted), rank, place, nodes, s);
  if (err != hipSuccess) return err;
  for (int pass = 0; pass < 3; ++pass)
    hipLaunchKernelGGL(cluster_keys_kernel, dim3(grid_for(pass == 0 ? nn : 6 * ne)), dim3(kBlock), 0, s, conn, ne, nn,
                       pass, rank, keys, place);
  err = hipGetLastError();
  if (err != hipSuccess) return err;
  size_t tb = temp_bytes;
  err = hipcub::DeviceRadixSort::SortPairs(temp, tb, keys, keys_sorted, place, nodes, (int)nn, 0, 31, s);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(cluster_segments_kernel, dim3(grid_for(nn + 1)), dim3(kBlock), 0, s, keys_sorted, nn, seg);
  hipLaunchKernelGGL(cluster_place_kernel, dim3(grid_for(nn)), dim3(kBlock), 0, s, nodes, nn, place);
  return hipGetLastError();
}

hipError_t cluster_count(const ClusterMesh& m, const int64_t* seg, int64_t nn, void* temp, size_t temp_bytes,
                         int32_t* runs, int32_t* more, int32_t* recs, int32_t* most, hipStream_t s) {
  hipLaunchKernelGGL(cluster_count_kernel, dim3(grid_for(64 * (nn + 1))), dim3(kBlock), 0, s, m, seg, nn, runs, more, recs,
                     most);
  hipError_t err = hipGetLastError();
  for (int32_t* v : {runs, more, recs}) {
    if (err != hipSuccess) return err;
    size_t tb = temp_bytes;
    err = hipcub::DeviceScan::ExclusiveSum(temp, tb, v, v, (int)(nn + 1), s);
  }
  return err;
}

hipError_t cluster_totals(const int32_t* a, const int32_t* b, const int32_t* c, const int32_t* d, int4* out,
                          hipStream_t s) {
  hipLaunchKernelGGL(cluster_totals_kernel, dim3(1), dim3(1), 0, s, a, b, c, d, out);
  return hipGetLastError();
}

hipError_t cluster_fill(const ClusterMesh& m, const int64_t* seg, int64_t nn, const int32_t* runs,
                        const int32_t* more, const int32_t* recs, int64_t num_runs, int4* run_tab, int4* chunk_tab,
                        int2* span_tab, uint32_t* elem_tab, int2* rec_tab, hipStream_t s) {
  hipLaunchKernelGGL(cluster_fill_kernel, dim3(grid_for(64 * nn)), dim3(kBlock), 0, s, m, seg, nn, runs, more, recs,
                     num_runs, run_tab, chunk_tab, span_tab, elem_tab, rec_tab);
  return hipGetLastError();
}

hipError_t cluster_lanes(const ClusterMesh& m, int64_t num_runs, int64_t num_chunks, const int4* run_tab,
                         int4* chunk_tab, const int2* span_tab, const uint32_t* elem_tab, const int2* rec_tab,
                         int32_t* nlanes, void* temp, size_t temp_bytes, ClusterLane* lanes, hipStream_t s) {
  if (num_runs == 0) return hipSuccess;
  hipLaunchKernelGGL(cluster_lanes_kernel, dim3((unsigned)num_runs), dim3(kBlock), 0, s, m, run_tab, chunk_tab,
                     span_tab, elem_tab, rec_tab, nlanes, lanes);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || lanes) return err;
  return hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, nlanes, nlanes, (int)(num_chunks + 1), s);
}

hipError_t cluster_conn(int64_t num_chunks, const int4* chunk_tab, const uint32_t* elem_tab, const int32_t* conn,
                        int32_t* chunk_conn, hipStream_t s) {
  hipLaunchKernelGGL(cluster_conn_kernel, dim3(grid_for(num_chunks * kClusterElems * 10)), dim3(kBlock), 0, s,
                     num_chunks, chunk_tab, elem_tab, conn, chunk_conn);
  return hipGetLastError();
}

hipError_t linear_order(const double* coords, int64_t nn, void* temp, size_t temp_bytes, unsigned long long* box,
                        uint32_t* code, uint32_t* code_sorted, int32_t* place, int32_t* nodes, hipStream_t s) {
  // place holds the unsorted ids until the last kernel of the order writes it
  return morton_order(coords, nn, temp, temp_bytes, box, code, code_sorted, place, place, nodes, s);
}

hipError_t linear_split(const ClusterMesh& m, int64_t nn, void* temp, size_t temp_bytes, int32_t* parts,
                        int32_t* nlanes, int32_t* nelems, int32_t* bad, int4* totals, hipStream_t s) {
  const int64_t groups = (nn + kLinearNodes - 1) / kLinearNodes, most = kLinearNodes * groups;
  hipLaunchKernelGGL(linear_split_kernel, dim3((unsigned)groups), dim3(kBlock), 0, s, m, nn, parts, nlanes, nelems,
                     bad);
  hipError_t err = hipGetLastError();
  for (int32_t* v : {parts, nlanes, nelems}) {
    if (err != hipSuccess) return err;
    size_t tb = temp_bytes;
    err = hipcub::DeviceScan::ExclusiveSum(temp, tb, v, v, (int)((v == parts ? groups : most) + 1), s);
  }
  return err != hipSuccess ? err : cluster_totals(parts + groups, nlanes + most, nelems + most, bad, totals, s);
}

hipError_t linear_tables(const ClusterMesh& m, int64_t nn, const int32_t* parts, const int32_t* nlanes,
                         const int32_t* nelems, int4* runs, int2* spans, int32_t* elems, ClusterLane* lanes,
                         hipStream_t s) {
  const int64_t groups = (nn + kLinearNodes - 1) / kLinearNodes;
  hipLaunchKernelGGL(linear_tables_kernel, dim3((unsigned)groups), dim3(kBlock), 0, s, m, nn, parts, nlanes, nelems,
                     runs, spans, elems, lanes);
  return hipGetLastError();
}

hipError_t launch_linear_points(const AsmArgs& a, hipStream_t s) {
  if (a.num_elems == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.num_elems + 255) / 256));
  if (a.model == MODEL_J2) hipLaunchKernelGGL(linear_points_kernel<MODEL_J2>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(linear_points_kernel<MODEL_NEOHOOKEAN>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_linear_cluster(bool transpose, bool plastic, const LinearArgs& a, int blocks, hipStream_t s) {
  if (a.num_runs == 0) return hipSuccess;
  if (blocks <= 0) blocks = (int)std::min<int64_t>((a.num_runs + 7) / 8 * 8, int64_t(1) << 30);  // as launch_cluster
  const dim3 grid(blocks), block(kLinearThreads);
  if (plastic && transpose) hipLaunchKernelGGL((linear_cluster_kernel<true, true>), grid, block, 0, s, a);
  else if (plastic) hipLaunchKernelGGL((linear_cluster_kernel<true, false>), grid, block, 0, s, a);
  else if (transpose) hipLaunchKernelGGL((linear_cluster_kernel<false, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((linear_cluster_kernel<false, false>), grid, block, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_cluster(bool transpose, const ClusterArgs& a, int blocks, hipStream_t s) {
  if (a.num_runs == 0) return hipSuccess;
  // One workgroup per run unless told otherwise (a multiple of 8 for the XCD
  // slabs).  Not a persistent grid: loads and stores share a wait counter, so a
  // workgroup's next run would begin by waiting for all stores of the last one
  // (P2 64^3 cube: 9.5 ms against 6.0).
  if (blocks <= 0) blocks = (int)std::min<int64_t>((a.num_runs + 7) / 8 * 8, int64_t(1) << 30);
  if (transpose) hipLaunchKernelGGL((cluster_kernel<true>), dim3(blocks), dim3(kClusterThreads), 0, s, a);
  else hipLaunchKernelGGL((cluster_kernel<false>), dim3(blocks), dim3(kClusterThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace goal
