// Neighbourhoods within a geodesic radius and their per-edge geometry, built on
// the GPU from float64 node coordinates.
//
// Membership is the reference's exact rule (discretization/edge_geometry.py:
// 381-387, 492-503): target i and source j are neighbours iff
//   atan2(|p_i x q_j|, clamp(<p_i, q_j>, -1, 1)) <= limit   (limit = r + 1e-10)
// evaluated in float64 with every product rounded on its own and the sums
// taken left to right.  Candidates come from 64-node bounding boxes instead of
// a KD-tree: a wavefront owns 16 consecutive targets and takes the source boxes
// in increasing index, skipping a box only when it lies farther than the chord
// of the limit on some axis (a Euclidean bound, so no neighbour is skipped).
// For unit vectors the computed <p, q> lies within about 1e-15 of cos(angle),
// and the computed geodesic within a few 1e-15 of the angle, so a dot product
// more than 1e-12 above cos(limit) is inside and one more than 1e-12 below is
// outside, whatever atan2 would round to: only pairs in that band take the
// exact test, and the decisions are the exact test's.  A target's neighbours are
// appended in increasing source index, so rows come out target-major,
// source-minor (:701-704) without a sort.
// Two passes: degrees (then an in-place prefix sum into row_ptr, :622-653),
// then the edge list into the rows the caller sized from row_ptr[n].
//
// The per-edge tables (edge_geometry_from_index, :506-619) are one pass per
// edge: log map in the target frame, geodesic distance, Levi-Civita transport
// angle, tangent quadrature weight, polar angle, and both phase tables.
#include <algorithm>

#include "common.hpp"

namespace gm {
namespace {

constexpr int kGeoTile = 64;         // source nodes per bounding box
constexpr int kGeoTargets = 16;      // targets per wavefront
constexpr int kScanThreads = 1024;   // one workgroup turns the degrees into row_ptr
constexpr int kTableThreads = 256;

__device__ __forceinline__ int64_t imin(int64_t x, int64_t y) { return x < y ? x : y; }

// In-wave LDS hand-off: stores before, loads after, with no reordering across it.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double wave_min(double v) {
  for (int o = 32; o; o >>= 1) v = fmin(v, __shfl_xor(v, o, kWave));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
  for (int o = 32; o; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
  return v;
}

// <p, q> with each product rounded and the sum taken left to right.
__device__ __forceinline__ double dot3(const double* p, const double* q) {
#pragma clang fp contract(off)
  return p[0] * q[0] + p[1] * q[1] + p[2] * q[2];
}

// p x q, each product rounded.
__device__ __forceinline__ void cross3(const double* p, const double* q, double* c) {
#pragma clang fp contract(off)
  c[0] = p[1] * q[2] - p[2] * q[1];
  c[1] = p[2] * q[0] - p[0] * q[2];
  c[2] = p[0] * q[1] - p[1] * q[0];
}

__device__ __forceinline__ double norm3(const double* c) {
#pragma clang fp contract(off)
  return sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
}

__device__ __forceinline__ double clamp_unit(double x) { return fmin(fmax(x, -1.0), 1.0); }

// atan2(|p x q|, clamp(<p, q>)), given the unclamped <p, q>.
__device__ __forceinline__ double geodesic(const double* p, const double* q, double dot) {
  double c[3];
  cross3(p, q, c);
  return atan2(norm3(c), clamp_unit(dot));
}

__global__ __launch_bounds__(kGeoTile) void geo_bounds_kernel(const double* __restrict__ nodes, int64_t n,
                                                              double* __restrict__ boxes) {
  const int64_t tile = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t i = imin(tile * kGeoTile + lane, n - 1);  // lanes past the end repeat the last node
  double lo[3], hi[3];
  for (int k = 0; k < 3; ++k) {
    const double x = nodes[3 * i + k];
    lo[k] = wave_min(x);
    hi[k] = wave_max(x);
  }
  if (lane == 0) {
    for (int k = 0; k < 3; ++k) {
      boxes[6 * tile + k] = lo[k];
      boxes[6 * tile + 3 + k] = hi[k];
    }
  }
}

struct WalkArgs {
  const double* targets;
  const double* sources;
  const double* source_boxes;
  int64_t n_targets, n_sources;
  double limit;      // membership: geodesic <= limit
  double cos_floor;  // pairs with <p, q> below this are farther than the limit
  double cos_in;     // pairs with <p, q> at or above this are within the limit
  double reach;      // chord of the limit plus a margin: the box test's distance
  int64_t* row_ptr;  // degree pass: degree of t at row_ptr[t + 1]; edge pass: row offsets (read only)
  int64_t* target_out;
  int64_t* source_out;
  int64_t n_edges;   // edge pass: capacity of target_out / source_out
};

// One wave per kGeoTargets targets.  The wave tests 64 source boxes at a time, a
// box a lane, against its targets' box, then takes each box within reach with a
// source a lane: a target's neighbours among the 64 are one ballot, counted, or
// written behind each other in source order.  With a target a lane and the boxes
// walked one by one, the wave's loop over every box was a chain of scalar loads
// and each lane stored its own row's next element: 256x512 at three rings, 2048
// boxes, 15.7M edges, degrees 0.97 ms and edges 1.45 ms; this form takes 0.22 and
// 0.30 (the edges' 252 MB at 0.85 TB/s; float64 products bound both).  Sixteen
// targets a wave give a small box and 8192 waves.
template <bool kEdges>
__global__ __launch_bounds__(kGeoTile) void geo_walk_kernel(WalkArgs a) {
  __shared__ double pts[kGeoTargets][3];
  const int lane = threadIdx.x, own = lane & (kGeoTargets - 1);
  const int64_t t0 = xcd_block(blockIdx.x, gridDim.x) * kGeoTargets;
  const int nt = (int)imin(kGeoTargets, a.n_targets - t0);
  const int64_t tt = t0 + imin(own, nt - 1);  // lanes past the end repeat the last target
  double tlo[3], thi[3];
  for (int k = 0; k < 3; ++k) {
    const double x = a.targets[3 * tt + k];
    if (lane < kGeoTargets) pts[lane][k] = x;
    tlo[k] = wave_min(x) - a.reach;
    thi[k] = wave_max(x);
  }
  wave_sync();
  int64_t pos = 0, end = 0;  // of target t0 + own: the degree, or the next place and the row's end
  if (kEdges) {
    pos = a.row_ptr[tt];
    end = imin(a.row_ptr[tt + 1], a.n_edges);
  }
  const int64_t source_tiles = (a.n_sources + kGeoTile - 1) / kGeoTile;
  for (int64_t s0 = 0; s0 < source_tiles; s0 += kGeoTile) {
    bool near = s0 + lane < source_tiles;
    const double* box = a.source_boxes + 6 * (near ? s0 + lane : s0);
    for (int k = 0; k < 3; ++k) near &= !(box[k] - a.reach > thi[k]) && !(tlo[k] > box[3 + k]);
    for (uint64_t boxes = __ballot(near); boxes; boxes &= boxes - 1) {
      const int64_t j = (s0 + __ffsll((unsigned long long)boxes) - 1) * kGeoTile + lane;
      const bool live = j < a.n_sources;
      const int64_t jj = live ? j : a.n_sources - 1;
      const double q[3] = {a.sources[3 * jj], a.sources[3 * jj + 1], a.sources[3 * jj + 2]};
      for (int s = 0; s < nt; ++s) {
        const double p[3] = {pts[s][0], pts[s][1], pts[s][2]};
        const double dot = dot3(p, q);
        bool in = live && dot >= a.cos_floor;
        if (in && !(dot >= a.cos_in)) in = geodesic(p, q, dot) <= a.limit;
        const uint64_t hits = __ballot(in);
        if (!hits) continue;
        if (kEdges) {
          const int64_t e = __shfl(pos, s, kWave) + __popcll(hits & ((uint64_t(1) << lane) - 1));
          const int64_t stop = __shfl(end, s, kWave);
          if (in && e < stop) {
            a.target_out[e] = t0 + s;
            a.source_out[e] = j;
          }
        }
        if (own == s) pos += __popcll(hits);
      }
    }
  }
  if (!kEdges && lane < nt) a.row_ptr[t0 + lane + 1] = pos;
}

// row_ptr[1..n] holds the degrees; leaves their inclusive prefix sums there and 0 in row_ptr[0].
// One workgroup, each wave a contiguous sixteenth in steps of 64 coalesced entries: the latency
// of the steps bounds it (131,072 targets: 224 us with a contiguous strip a thread, 101 here).
__global__ __launch_bounds__(kScanThreads) void geo_scan_kernel(int64_t* __restrict__ row_ptr, int64_t n) {
  constexpr int kWaves = kScanThreads / kWave;
  __shared__ int64_t sums[kWaves];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int64_t share = ((n + kWaves - 1) / kWaves + kWave - 1) / kWave * kWave;
  const int64_t lo = 1 + imin(n, wave * share), hi = 1 + imin(n, (wave + 1) * share);
  int64_t s = 0;
#pragma unroll 8
  for (int64_t i = lo + lane; i < hi; i += kWave) s += row_ptr[i];
  for (int o = 32; o; o >>= 1) s += __shfl_xor(s, o, kWave);
  if (lane == 0) sums[wave] = s;
  __syncthreads();
  int64_t run = 0;
  for (int w = 0; w < wave; ++w) run += sums[w];
  for (int64_t i = lo; i < hi; i += kWave) {
    int64_t v = i + lane < hi ? row_ptr[i + lane] : 0;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int64_t below = __shfl_up(v, o, kWave);
      if (lane >= o) v += below;
    }
    if (i + lane < hi) row_ptr[i + lane] = run + v;
    run += __shfl(v, kWave - 1, kWave);
  }
  if (threadIdx.x == 0) row_ptr[0] = 0;
}

struct TableArgs {
  const double* targets;
  const double* target_frames;  // (n_targets, 3, 2): columns e1, e2
  const double* sources;
  const double* source_frames;
  const double* source_quadrature;
  const int64_t* edge_index;    // (2, n_edges): target, source
  int64_t n_edges, n_targets, n_sources;
  int K;
  double* log_coordinates;   // (E, 2)
  double* distances;         // (E)
  double* polar;             // (E)
  double* transport;         // (E)
  double* quadrature;        // (E)
  double* angular_phases;    // (E, K + 1, 2)
  double* transport_phases;  // (E, K + 1, 2)
};

// One edge's tables.  Phase entries go through put(table, k, cos, sin): into the
// workgroup's LDS stage, or straight to HBM when the tables are too wide to stage.
template <class Put>
__device__ __forceinline__ void edge_row(const TableArgs& a, int64_t e, Put put) {
  const int64_t i = a.edge_index[e], j = a.edge_index[a.n_edges + e];
  if (i < 0 || i >= a.n_targets || j < 0 || j >= a.n_sources) {  // an index out of range marks its row
    const double nan = __builtin_nan("");
    reinterpret_cast<double2*>(a.log_coordinates)[e] = make_double2(nan, nan);
    a.distances[e] = a.polar[e] = a.transport[e] = a.quadrature[e] = nan;
    for (int k = 0; k <= a.K; ++k) {
      put(0, k, nan, nan);
      put(1, k, nan, nan);
    }
    return;
  }
  const double p[3] = {a.targets[3 * i], a.targets[3 * i + 1], a.targets[3 * i + 2]};
  const double q[3] = {a.sources[3 * j], a.sources[3 * j + 1], a.sources[3 * j + 2]};
  const double dot = clamp_unit(dot3(p, q));
  double c[3];
  cross3(p, q, c);
  const double d = atan2(norm3(c), dot);
  const double inv_density = d == 0.0 ? 1.0 : d / sin(d);  // r / sin r
  double ambient[3];
  for (int k = 0; k < 3; ++k) ambient[k] = inv_density * (q[k] - dot * p[k]);
  const double* ft = a.target_frames + 6 * i;
  const double* fs = a.source_frames + 6 * j;
  const double l0 = ft[0] * ambient[0] + ft[2] * ambient[1] + ft[4] * ambient[2];
  const double l1 = ft[1] * ambient[0] + ft[3] * ambient[1] + ft[5] * ambient[2];
  // R = I + K + K^2 / (1 + <q, p>), K the cross-product matrix of w = q x p = -(p x q),
  // applied to the source frame's e1; the target frame's components give the angle.
  const double w[3] = {-c[0], -c[1], -c[2]};
  const double u[3] = {fs[0], fs[2], fs[4]};
  double ku[3], kku[3];
  cross3(w, u, ku);
  cross3(w, ku, kku);
  const double inv1 = 1.0 / (1.0 + dot);
  double ru[3];
  for (int k = 0; k < 3; ++k) ru[k] = u[k] + ku[k] + kku[k] * inv1;
  const double t00 = ft[0] * ru[0] + ft[2] * ru[1] + ft[4] * ru[2];
  const double t10 = ft[1] * ru[0] + ft[3] * ru[1] + ft[5] * ru[2];
  const double gamma = atan2(t10, t00);
  const double phi = atan2(l1, l0);
  reinterpret_cast<double2*>(a.log_coordinates)[e] = make_double2(l0, l1);
  a.distances[e] = d;
  a.polar[e] = phi;
  a.transport[e] = gamma;
  a.quadrature[e] = a.source_quadrature[j] * inv_density;
  for (int k = 0; k <= a.K; ++k) {
    double sn, cs;
    sincos(phi * (double)k, &sn, &cs);
    put(0, k, cs, sn);
    sincos(gamma * (double)k, &sn, &cs);
    put(1, k, cs, sn);
  }
}

// Workgroups walk tiles of kTableThreads edges.  With the phase tables staged
// (dynamic LDS of 2 * kTableThreads * (K + 1) double2), a tile's rows of both
// tables, contiguous in HBM, leave in consecutive 16-byte stores.
__global__ __launch_bounds__(kTableThreads) void geo_tables_kernel(TableArgs a, int staged) {
  extern __shared__ double2 stage[];
  const int orders = a.K + 1;
  const int64_t n_tiles = (a.n_edges + kTableThreads - 1) / kTableThreads;
  double2* angular = reinterpret_cast<double2*>(a.angular_phases);
  double2* transport = reinterpret_cast<double2*>(a.transport_phases);
  for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int64_t e0 = tile * kTableThreads;
    const int64_t e = e0 + threadIdx.x;
    const int count = (int)imin(kTableThreads, a.n_edges - e0);
    if (e < a.n_edges) {
      if (staged) {
        double2* row0 = stage + threadIdx.x * orders;
        double2* row1 = stage + (kTableThreads + threadIdx.x) * orders;
        edge_row(a, e, [&](int table, int k, double cs, double sn) {
          (table ? row1 : row0)[k] = make_double2(cs, sn);
        });
      } else {
        edge_row(a, e, [&](int table, int k, double cs, double sn) {
          (table ? transport : angular)[e * orders + k] = make_double2(cs, sn);
        });
      }
    }
    if (staged) {
      __syncthreads();
      const int total = count * orders;
      for (int x = threadIdx.x; x < total; x += kTableThreads) {
        angular[e0 * orders + x] = stage[x];
        transport[e0 * orders + x] = stage[kTableThreads * orders + x];
      }
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(kTableThreads) void geo_distances_kernel(const double* __restrict__ targets,
                                                                      const double* __restrict__ sources,
                                                                      const int64_t* __restrict__ edge_index,
                                                                      int64_t n_edges, int64_t n_targets,
                                                                      int64_t n_sources, double* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * kTableThreads;
  for (int64_t e = (int64_t)blockIdx.x * kTableThreads + threadIdx.x; e < n_edges; e += stride) {
    const int64_t i = edge_index[e], j = edge_index[n_edges + e];
    if (i < 0 || i >= n_targets || j < 0 || j >= n_sources) {
      out[e] = __builtin_nan("");
      continue;
    }
    const double p[3] = {targets[3 * i], targets[3 * i + 1], targets[3 * i + 2]};
    const double q[3] = {sources[3 * j], sources[3 * j + 1], sources[3 * j + 2]};
    out[e] = geodesic(p, q, dot3(p, q));
  }
}

int64_t tiles_of(int64_t n) { return (n + kGeoTile - 1) / kGeoTile; }

unsigned walk_blocks(int64_t n_targets) { return (unsigned)((n_targets + kGeoTargets - 1) / kGeoTargets); }

int64_t table_blocks(int64_t n_edges) {
  return std::max<int64_t>(1, std::min<int64_t>((n_edges + kTableThreads - 1) / kTableThreads, 8192));
}

int prepare_walk(WalkArgs& a, const double* targets, int64_t n_targets, const double* sources, int64_t n_sources,
                 double limit, const double* workspace) {
  GM_REQUIRE(n_targets >= 1 && n_sources >= 1, "the target and source node sets must be non-empty");
  GM_REQUIRE((n_targets + kGeoTargets - 1) / kGeoTargets <= INT32_MAX, "too many target nodes for one launch");
  GM_REQUIRE(targets && sources && workspace && aligned(targets, 8) && aligned(sources, 8) && aligned(workspace, 8),
             "targets, sources and workspace must be 8-byte aligned device pointers");
  GM_REQUIRE(std::isfinite(limit) && limit > 0.0, "the radius limit must be positive and finite");
  a.targets = targets;
  a.sources = sources;
  a.source_boxes = workspace;
  a.n_targets = n_targets;
  a.n_sources = n_sources;
  a.limit = limit;
  const double pi = 3.14159265358979323846;
  // The computed <p, q> of unit vectors is within ~1e-15 of cos(angle) and |d cos| <= |d angle|:
  // 1e-12 on either side of cos(limit) bounds the band where only the exact test decides.
  a.cos_floor = limit >= pi ? -2.0 : std::cos(limit) - 1e-12;
  a.cos_in = limit >= pi ? -2.0 : std::cos(limit) + 1e-12;
  a.reach = (limit >= pi ? 2.0 : 2.0 * std::sin(0.5 * limit)) + 1e-9;
  return GM_OK;
}

}  // namespace
}  // namespace gm

extern "C" int64_t gm_radius_workspace_doubles(int64_t n_targets, int64_t n_sources) {
  (void)n_targets;  // the targets' boxes are the walk's own
  return 6 * gm::tiles_of(n_sources);
}

extern "C" int gm_radius_row_ptr_f64(const double* targets, int64_t n_targets, const double* sources,
                                     int64_t n_sources, double limit, double* workspace, int64_t* row_ptr,
                                     void* stream) {
  gm::WalkArgs a{};
  const int status = gm::prepare_walk(a, targets, n_targets, sources, n_sources, limit, workspace);
  if (status != GM_OK) return status;
  GM_REQUIRE(row_ptr && gm::aligned(row_ptr, 8), "row_ptr must be an 8-byte aligned device pointer");
  a.row_ptr = row_ptr;
  const hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(gm::geo_bounds_kernel, dim3(gm::tiles_of(n_sources)), dim3(gm::kGeoTile), 0, s, sources,
                     n_sources, workspace);
  int rc = gm::check_launch("radius_bounds");
  if (rc != GM_OK) return rc;
  hipLaunchKernelGGL(gm::geo_walk_kernel<false>, dim3(gm::walk_blocks(n_targets)), dim3(gm::kGeoTile), 0, s, a);
  rc = gm::check_launch("radius_degrees");
  if (rc != GM_OK) return rc;
  hipLaunchKernelGGL(gm::geo_scan_kernel, dim3(1), dim3(gm::kScanThreads), 0, s, row_ptr, n_targets);
  return gm::check_launch("radius_row_ptr");
}

extern "C" int gm_radius_edges_f64(const double* targets, int64_t n_targets, const double* sources,
                                   int64_t n_sources, double limit, const double* workspace, const int64_t* row_ptr,
                                   int64_t n_edges, int64_t* edge_index, void* stream) {
  gm::WalkArgs a{};
  const int status = gm::prepare_walk(a, targets, n_targets, sources, n_sources, limit, workspace);
  if (status != GM_OK) return status;
  GM_REQUIRE(row_ptr && gm::aligned(row_ptr, 8), "row_ptr must be an 8-byte aligned device pointer");
  GM_REQUIRE(n_edges >= 0, "n_edges must be non-negative");
  if (n_edges == 0) return GM_OK;
  GM_REQUIRE(edge_index && gm::aligned(edge_index, 8), "edge_index must be an 8-byte aligned device pointer");
  a.row_ptr = const_cast<int64_t*>(row_ptr);
  a.target_out = edge_index;
  a.source_out = edge_index + n_edges;
  a.n_edges = n_edges;
  hipLaunchKernelGGL(gm::geo_walk_kernel<true>, dim3(gm::walk_blocks(n_targets)), dim3(gm::kGeoTile), 0,
                     (hipStream_t)stream, a);
  return gm::check_launch("radius_edges");
}

extern "C" int gm_geodesic_distances_f64(const double* targets, const double* sources, const int64_t* edge_index,
                                         int64_t n_edges, int64_t n_targets, int64_t n_sources, double* distances,
                                         void* stream) {
  GM_REQUIRE(n_edges >= 0 && n_targets >= 0 && n_sources >= 0, "counts must be non-negative");
  if (n_edges == 0) return GM_OK;
  GM_REQUIRE(targets && sources && edge_index && distances, "every pointer must be a device pointer");
  hipLaunchKernelGGL(gm::geo_distances_kernel, dim3(gm::table_blocks(n_edges)), dim3(gm::kTableThreads), 0,
                     (hipStream_t)stream, targets, sources, edge_index, n_edges, n_targets, n_sources, distances);
  return gm::check_launch("geodesic_distances");
}

extern "C" int gm_edge_tables_f64(const double* targets, const double* target_frames, const double* sources,
                                  const double* source_frames, const double* source_quadrature,
                                  const int64_t* edge_index, int64_t n_edges, int64_t n_targets, int64_t n_sources,
                                  int64_t max_frequency, double* log_coordinates, double* distances,
                                  double* polar_angles, double* transport_angles, double* tangent_quadrature,
                                  double* angular_phases, double* transport_phases, void* stream) {
  GM_REQUIRE(n_edges >= 0 && n_targets >= 0 && n_sources >= 0, "counts must be non-negative");
  GM_REQUIRE(max_frequency >= 0 && max_frequency <= 64, "max_frequency must lie in [0, 64]");
  if (n_edges == 0) return GM_OK;
  GM_REQUIRE(targets && target_frames && sources && source_frames && source_quadrature && edge_index,
             "node, frame, quadrature and edge pointers must be device pointers");
  GM_REQUIRE(log_coordinates && distances && polar_angles && transport_angles && tangent_quadrature &&
                 angular_phases && transport_phases,
             "every output must be a device pointer");
  GM_REQUIRE(gm::aligned(log_coordinates, 16) && gm::aligned(angular_phases, 16) && gm::aligned(transport_phases, 16),
             "log_coordinates and the phase tables must be 16-byte aligned");
  gm::TableArgs a{};
  a.targets = targets;
  a.target_frames = target_frames;
  a.sources = sources;
  a.source_frames = source_frames;
  a.source_quadrature = source_quadrature;
  a.edge_index = edge_index;
  a.n_edges = n_edges;
  a.n_targets = n_targets;
  a.n_sources = n_sources;
  a.K = (int)max_frequency;
  a.log_coordinates = log_coordinates;
  a.distances = distances;
  a.polar = polar_angles;
  a.transport = transport_angles;
  a.quadrature = tangent_quadrature;
  a.angular_phases = angular_phases;
  a.transport_phases = transport_phases;
  // Stage the phase tables through LDS while they fit four workgroups per CU.
  const size_t stage_bytes = 2 * gm::kTableThreads * (size_t)(max_frequency + 1) * sizeof(double2);
  const int staged = stage_bytes <= 40 * 1024;
  hipLaunchKernelGGL(gm::geo_tables_kernel, dim3(gm::table_blocks(n_edges)), dim3(gm::kTableThreads),
                     staged ? stage_bytes : 0, (hipStream_t)stream, a, staged);
  return gm::check_launch("edge_tables");
}
