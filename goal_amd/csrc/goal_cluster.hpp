// Node clusters of a quadratic mesh: the plan of the one-kernel neo-Hookean
// assembly (goal_cluster.hip).
//
// The nodes are ordered by key -- a vertex's key is its place on a Morton curve
// through the mesh, an edge node's the smaller one of its edge's vertices --
// and each key's nodes are cut into runs, which neighbour each other in space
// as they do in time.  A run is what one workgroup assembles: a vertex and the edge nodes it
// owns share most of their elements (in a regular mesh of six tets per cell,
// 60 incidences over 24 elements), so the point states of 24 elements serve
// 60 x 4 matrix rows.  A run's incidences are cut into chunks whose elements
// fit the kernel's LDS table.
//
// The blocks (a, b) and (b, a) of two nodes share most of their entries, and
// every element that holds b beside a is among a's: the run of the node that
// comes first in the order forms both.  Within a chunk the unit of work is a
// visit: what one element adds to one such pair.  A pair's visits go to 1, 2,
// 4, .. 64 lanes, the fewest with at most three visits each; each lane sums
// its visits in registers and the pair's lanes then add theirs.  Pairs are
// ordered by lanes, then visits, so a wavefront's lanes have equal work.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace goal {

constexpr int kClusterElems = 26;   // elements per chunk
constexpr int kClusterNodes = 32;   // nodes per run
constexpr int kClusterSlots = 512;  // CSR blocks of a run's rows
constexpr uint32_t kClusterOwned = 0x80000000u;  // this chunk writes the element's point states

// What walk_cluster reads: nodes [lo, hi) of the ordered list.
struct ClusterMesh {
  const int32_t* nodes;
  const int64_t* inc_ptr;  // node -> its incidence records
  const int32_t* inc;      // record -> 10 e + local node
  const int64_t* row_ptr;  // CSR rows, four per node
  const uint16_t* posi;    // [records][10] position of each element node in adj(node)
  const uint16_t* pos;     // [elements][10][10] the same by element
  const int32_t* cols;     // CSR columns
  const int32_t* place;    // [nodes] place in the ordered list
};

// Cuts the nodes [lo, hi) into runs and chunks, in order; a wavefront's work (all
// 64 lanes with the same arguments).  Lane s keeps the open chunk's element s, so
// that looking an element up is one ballot; nodes and incidences come in 64 at a
// time.  The sink's calls:
//   run(node_lo)                            a run begins at this place of the list
//   chunk()                                 a chunk begins
//   rec(k, slot, a, node)                   an incidence: record k, element slot, local node, run-local node
//   end_chunk(nelem, elem, own)             its elements, one a lane, and which of them (bits) have their states
//                                           written by this chunk
//   end_run(node_hi, blocks)
//   bare()                                  a node without elements
template <typename Sink>
__device__ inline void walk_cluster(const ClusterMesh& m, int64_t lo, int64_t hi, Sink& out) {
  const int lane = threadIdx.x & 63;
  int32_t mine = -1;  // the open chunk's element in this lane's slot
  uint32_t own = 0;
  int ne = 0, nn = 0;
  int64_t nb = 0;
  bool open_run = false, open_chunk = false;
  for (int64_t i0 = lo; i0 < hi; i0 += 64) {
    int deg_l = 0;
    int64_t k0_l = 0, k1_l = 0;
    if (i0 + lane < hi) {
      const int64_t n = m.nodes[i0 + lane];
      deg_l = (int)((m.row_ptr[4 * n + 1] - m.row_ptr[4 * n]) / 4);
      k0_l = m.inc_ptr[n];
      k1_l = m.inc_ptr[n + 1];
    }
    const int some = hi - i0 < 64 ? (int)(hi - i0) : 64;
    for (int l = 0; l < some; ++l) {
      const int64_t i = i0 + l, k0 = __shfl(k0_l, l, 64), k1 = __shfl(k1_l, l, 64);
      const int deg = __builtin_amdgcn_readlane(deg_l, l);
      if (k0 == k1) out.bare();
      if (open_run && (nn == kClusterNodes || nb + deg > kClusterSlots)) {
        if (open_chunk) out.end_chunk(ne, mine, own);
        open_chunk = false;
        out.end_run(i, nb);
        open_run = false;
      }
      if (!open_run) {
        out.run(i);
        open_run = true;
        nn = 0;
        nb = 0;
      }
      for (int64_t kb = k0; kb < k1; kb += 64) {
        const int32_t inc_l = kb + lane < k1 ? m.inc[kb + lane] : 0;
        const int incs = k1 - kb < 64 ? (int)(k1 - kb) : 64;
        for (int j = 0; j < incs; ++j) {
          const int32_t v = __builtin_amdgcn_readlane(inc_l, j), e = v / 10, a = v % 10;
          int s = 0;
          if (open_chunk) {
            const unsigned long long same = __ballot(lane < ne && mine == e);
            s = same ? __ffsll(same) - 1 : ne;
            if (s == kClusterElems) {
              out.end_chunk(ne, mine, own);
              open_chunk = false;
            }
          }
          if (!open_chunk) {
            out.chunk();
            open_chunk = true;
            ne = s = 0;
            own = 0;
          }
          if (s == ne) {
            if (lane == s) mine = e;
            ++ne;
          }
          if (a == 0) own |= 1u << s;
          out.rec(kb + j, s, a, nn);
        }
      }
      nb += deg;
      ++nn;
    }
  }
  if (open_chunk) out.end_chunk(ne, mine, own);
  if (open_run) out.end_run(hi, nb);
}

// Sinks: the sizes of one key's part, and the tables themselves (written by lane 0).
struct ClusterCount {
  int runs = 0, chunks = 0, recs = 0, most = 0;  // most: blocks of the largest run, kClusterSlots + 1 with a bare node
  __device__ void run(int64_t) { ++runs; }
  __device__ void chunk() { ++chunks; }
  __device__ void rec(int64_t, int, int, int) { ++recs; }
  __device__ void end_chunk(int, int32_t, uint32_t) {}
  __device__ void end_run(int64_t, int64_t nb) { most = nb > most ? (int)nb : most; }
  __device__ void bare() { most = most > kClusterSlots ? most : kClusterSlots + 1; }
};
struct ClusterFill {
  // Chunk r is the first of run r; a run's further chunks follow all runs.
  int4* runs;       // [runs]  node_lo, node_hi (places in the node list), further chunks lo, hi
  int4* chunks;     // [chunks] elements, first and last lane (cluster_lanes), 0
  int2* spans;      // [chunks] its incidences
  uint32_t* elems;  // [chunks][kClusterElems] element | kClusterOwned
  int2* recs;       // [incidences] record, slot | local node << 8 | run-local node << 16
  int r, x, k;      // the next run, further chunk and incidence
  bool writes;      // lane 0
  int c, in_run;
  int4 cur;
  __device__ void run(int64_t node_lo) {
    cur.x = (int)node_lo;
    cur.z = x;
    in_run = 0;
  }
  __device__ void chunk() {
    c = in_run++ ? x++ : r;
    if (writes) spans[c].x = k;
  }
  __device__ void rec(int64_t rk, int s, int a, int node) {
    if (writes) recs[k] = int2{(int)rk, s | (a << 8) | (node << 16)};
    ++k;
  }
  __device__ void end_chunk(int ne, int32_t elem, uint32_t own) {
    const int lane = threadIdx.x & 63;
    if (lane < ne) elems[(int64_t)c * kClusterElems + lane] = (uint32_t)elem | ((own >> lane) & 1u ? kClusterOwned : 0u);
    if (!writes) return;
    spans[c].y = k;
    chunks[c] = int4{ne, 0, 0, 0};
  }
  __device__ void end_run(int64_t node_hi, int64_t) {
    cur.y = (int)node_hi;
    cur.w = x;
    if (writes) runs[r] = cur;
    ++r;
  }
  __device__ void bare() {}
};

// Lanes (as a power of two) of a pair with n visits.
__host__ __device__ inline int cluster_log_lanes(int n) {
  return n <= 3 ? 0 : n <= 6 ? 1 : n <= 12 ? 2 : n <= 24 ? 3 : n <= 48 ? 4 : n <= 96 ? 5 : 6;
}
// Order of the pairs of a chunk: lower first.
__host__ __device__ inline int cluster_rank(int n) { return n == 0 ? 9 : n > 3 ? 6 - cluster_log_lanes(n) : 9 - n; }
__host__ __device__ inline int cluster_lanes_of_rank(int rank) { return rank < 6 ? 64 >> rank : 1; }

// A lane's work.  x: three visits of 13 bits each (element slot 5, local node
// of a 4, of b 4), their number (2 bits), b's position in a's adjacency (9
// bits), a's run-local number (5), log2 of the pair's lanes (3) and two flags.
// y: where block (b, a) goes: b's first block (40 bits), b's degree (12), a's
// position in b's adjacency (12).  The lanes of a pair are neighbours; lane j
// of 2^l takes the pair's visits j, j + 2^l, ...  A chunk has at most
// kClusterElems visits of one pair, so three a lane suffice.
static_assert(kClusterElems <= 32 && kClusterNodes <= 32 && kClusterSlots <= 512 && kClusterElems <= 3 * 16,
              "the fields of a lane's work");
constexpr int kLaneCount = 39, kLanePos = 41, kLaneNode = 50, kLaneLog = 55;
constexpr uint64_t kLaneFirst = uint64_t(1) << 58;  // no earlier chunk adds to this pair
constexpr uint64_t kLaneDiag = uint64_t(1) << 59;   // a = b: one block, and the node's residual
constexpr int kLaneDegT = 40, kLanePosT = 52;
struct alignas(16) ClusterLane {
  uint64_t x, y;
};

// Linear tets with one point (neo-Hookean, J2) go the same way, in two kernels:
// the point states are formed once, 32 doubles an element, and copied to LDS by
// the runs that need them.  Their runs are up to eight vertices that follow
// each other on the Morton curve (in a regular mesh of six tets per cell a
// 2 x 2 x 2 brick: 192 incidences of 120 elements; where the curve and the mesh do
// not line up, up to 156).  A visit's 13 bits are
// element slot 9, local a 2, local b 2.
constexpr int kLinearElems = 160;   // elements per run
constexpr int kLinearNodes = 8;     // vertices per run
constexpr int kLinearRecs = 4 * kLinearElems;  // incidences per run
constexpr int kLinearPoint = 32;    // doubles per element
static_assert(kLinearElems <= 3 * 64 && kLinearElems < 512 && kLinearNodes <= kClusterNodes, "the fields of a lane's work");
struct LinearArgs {
  int64_t num_runs, num_elems;
  const int4* runs;         // node_lo, node_hi, first element of the list, elements
  const int2* spans;        // first and last lane
  const int32_t* elems;
  const ClusterLane* lanes;
  const int32_t* nodes;
  const int64_t* row_ptr;
  const double* pt;         // [elements][kLinearPoint]
  double* R;
  double* vals;
  double* zero;             // [4 nodes] cleared along the way, or null
  int overwrite_R, overwrite_vals, xcd_remap;
};

// One neo-Hookean assembly of a quadratic mesh with four points (ASM_JACOBIAN
// or, transposed, ASM_ADJOINT), FP64.
struct MatParams;
struct AsmArgs;
struct ClusterArgs {
  int64_t num_runs, num_elems;
  const int4* runs;
  const int4* chunks;
  const uint32_t* chunk_elems;
  const int32_t* chunk_conn;  // [chunks][kClusterElems][10] nodes of the chunk's elements
  const ClusterLane* lanes;
  const int32_t* nodes;
  const int64_t* row_ptr;
  const double* coords;
  const double* x;
  const int32_t* elem_set;
  const MatParams* mats;
  double* sigma;
  double* R;
  double* vals;
  double* zero;             // [4 nodes] cleared along the way, or null
  int overwrite_R, overwrite_vals;
  int stabilization, save_state, xcd_remap;
};

// Plan kernels.  box [6]; rank [nn]: places on the curve; keys [nn]: node keys; seg [nn + 1]: starts of each key's part
// of the ordered nodes; place: its inverse; runs/more/recs [nn + 1]: per-key
// numbers of runs, further chunks and incidences, then (scanned) starts; most:
// the largest ClusterCount::most.  cluster_lanes: with lanes null the lanes of
// each chunk, rounded up to whole wavefronts, into nlanes [chunks + 1] (then
// scanned into starts); else the tables.
hipError_t cluster_temp_bytes(int64_t n, size_t* bytes);
hipError_t cluster_order(const int32_t* conn, const double* coords, int64_t ne, int64_t nn, void* temp,
                         size_t temp_bytes, unsigned long long* box, int32_t* keys, int32_t* keys_sorted,
                         int32_t* rank, int32_t* place, int32_t* nodes, int64_t* seg, hipStream_t s);
hipError_t cluster_count(const ClusterMesh& m, const int64_t* seg, int64_t nn, void* temp, size_t temp_bytes,
                         int32_t* runs, int32_t* more, int32_t* recs, int32_t* most, hipStream_t s);
hipError_t cluster_fill(const ClusterMesh& m, const int64_t* seg, int64_t nn, const int32_t* runs,
                        const int32_t* more, const int32_t* recs, int64_t num_runs, int4* run_tab, int4* chunk_tab,
                        int2* span_tab, uint32_t* elem_tab, int2* rec_tab, hipStream_t s);
hipError_t cluster_lanes(const ClusterMesh& m, int64_t num_runs, int64_t num_chunks, const int4* run_tab,
                         int4* chunk_tab, const int2* span_tab, const uint32_t* elem_tab, const int2* rec_tab,
                         int32_t* nlanes, void* temp, size_t temp_bytes, ClusterLane* lanes, hipStream_t s);
hipError_t cluster_conn(int64_t num_chunks, const int4* chunk_tab, const uint32_t* elem_tab, const int32_t* conn,
                        int32_t* chunk_conn, hipStream_t s);
// out: the four values, for one read-back.
hipError_t cluster_totals(const int32_t* a, const int32_t* b, const int32_t* c, const int32_t* d, int4* out,
                          hipStream_t s);
// linear_split: runs per group of kLinearNodes ordered nodes into parts
// [groups + 1], lanes (whole wavefronts) and elements of each run into nlanes
// and nelems [kLinearNodes groups + 1], all scanned into starts; a number above
// zero into *bad (zero before) when a node's incidences do not fit a run; the
// numbers of runs, lanes and elements, and *bad, into *totals.  linear_tables:
// the tables.
hipError_t linear_order(const double* coords, int64_t nn, void* temp, size_t temp_bytes, unsigned long long* box,
                        uint32_t* code, uint32_t* code_sorted, int32_t* place, int32_t* nodes, hipStream_t s);
hipError_t linear_split(const ClusterMesh& m, int64_t nn, void* temp, size_t temp_bytes, int32_t* parts,
                        int32_t* nlanes, int32_t* nelems, int32_t* bad, int4* totals, hipStream_t s);
hipError_t linear_tables(const ClusterMesh& m, int64_t nn, const int32_t* parts, const int32_t* nlanes,
                         const int32_t* nelems, int4* runs, int2* spans, int32_t* elems, ClusterLane* lanes,
                         hipStream_t s);
// Point states of every element (model neo-Hookean or J2; states saved as asked) into a.pt.
hipError_t launch_linear_points(const AsmArgs& a, hipStream_t s);
hipError_t launch_linear_cluster(bool transpose, bool plastic, const LinearArgs& a, int blocks, hipStream_t s);
hipError_t launch_cluster(bool transpose, const ClusterArgs& a, int blocks, hipStream_t s);

}  // namespace goal
