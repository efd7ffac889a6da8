// finder.hip -- candidate pair search on the device.
//
// Reference behaviour (what the result must equal): the quadtree / octree
// finder (src/Quadtree_Intersection_Finder.F90, src/Octree_...F90) returns,
// for every A element, the B elements whose bounding boxes overlap its own
// strictly in every dimension (bboxes_intersect, Quadtree_...F90:411-420) --
// the same set as brute force (src/Intersection_Finder.F90:1032-1050).  The
// R-tree finder uses closed intervals.  Both predicates run here in FP64 on
// exact min/max boxes.
//
// Design: B's element boxes are sorted by the leading 32 bits of the Morton code of their
// centres and grouped into an implicit F-ary hierarchy (node i of level l
// covers children [F*i, F*i+F) of level l-1; level 0 = elements).  Internal
// boxes are exact unions, so pruning with the same predicate never loses a
// pair.  A elements are taken in Morton order, 32 to a wave, which walks the
// union of their depth-first paths; a row is in leaf order.  A count pass
// sizes the CSR rows, a fill pass writes them.
#include <cstring>
#include <utility>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_segmented_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "lsm_geometry.hpp"
#include "lsm_runtime.hpp"

namespace lsm {

constexpr int kFanout = 8;
constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// Mesh staging
// ---------------------------------------------------------------------------

// Elements are simplices (LOC = DIM + 1) or, for the candidate finder only,
// quads / hexahedra (LOC = 2^DIM): those get coordinates, boxes and scale.
// Two meshes of one element type take one launch, A's blocks first.
struct StageJob {
  long ne, nnodes;
  const double* pos;
  const int* enl;
  double *coords, *bbox, *sp, *scale, *planes, *affine;
};
struct StageArgs {
  StageJob job[2];
  long blocks0;  // blocks of job 0
  int* bad;      // set to `serial` where a node index is out of range: a flag
  int serial;    // of an earlier call says nothing, so none has to be cleared
};

template <int DIM, int LOC>
__global__ void __launch_bounds__(kBlock) k_stage(StageArgs args) {
  constexpr bool SIMPLEX = LOC == DIM + 1;
  const bool second = (long)blockIdx.x >= args.blocks0;
  const StageJob& J = args.job[second ? 1 : 0];
  const long ne = J.ne, nnodes = J.nnodes;
  const double* __restrict__ pos = J.pos;
  const int* __restrict__ enl = J.enl;
  double* __restrict__ coords = J.coords;
  double* __restrict__ bbox = J.bbox;
  double* __restrict__ sp = J.sp;
  double* __restrict__ scale = J.scale;
  double* __restrict__ planes = J.planes;
  double* __restrict__ affine = J.affine;
  long e = ((long)blockIdx.x - (second ? args.blocks0 : 0)) * kBlock + threadIdx.x;
  if (e >= ne) return;
  double c[LOC * DIM];
#pragma unroll
  for (int j = 0; j < LOC; j++) {
    long v = enl[e * LOC + j];
    if (v < 0 || v >= nnodes) {
      *args.bad = args.serial;
      v = 0;
    }
#pragma unroll
    for (int d = 0; d < DIM; d++) c[j * DIM + d] = pos[v * DIM + d];
  }
  double sc = 1.0;
#pragma unroll
  for (int k = 0; k < LOC * DIM; k++) {
    coords[e * LOC * DIM + k] = c[k];
    sc = fmax_f(sc, __builtin_fabs(c[k]));
  }
  scale[e] = sc;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    double lo = c[d], hi = c[d];
#pragma unroll
    for (int j = 1; j < LOC; j++) {
      lo = fmin_f(lo, c[j * DIM + d]);
      hi = fmax_f(hi, c[j * DIM + d]);
    }
    bbox[(long)d * ne + e] = lo;
    bbox[(long)(DIM + d) * ne + e] = hi;
  }
  if constexpr (!SIMPLEX) {
    sp[e] = 0.0;
    return;
  } else {
  double m;
  if constexpr (DIM == 2) m = triangle_area(c);
  else m = tet_volume_tet(c);
  sp[e] = fspacing(m);
  if constexpr (DIM == 3) {
   if (planes) {
    Planes P;
    tet_planes(c, P);
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int k = 0; k < 3; k++) planes[e * 16 + 4 * i + k] = P.n[i][k];
      planes[e * 16 + 4 * i + 3] = P.c[i];
    }
   }
  }
  if (affine) {
    // Barycentric coordinates as affine maps: lambda_{1..dim}(x) = Minv (x - v1),
    // lambda_0 = 1 - sum.  Stored as [v1 (dim), Minv (dim x dim, row-major)].
    double* out = affine + e * (DIM + DIM * DIM);
    if constexpr (DIM == 2) {
      double e1x = c[2] - c[0], e1y = c[3] - c[1];
      double e2x = c[4] - c[0], e2y = c[5] - c[1];
      double det = e2y * e1x - (-e2x) * (-e1y);
      out[0] = c[0];
      out[1] = c[1];
      out[2] = e2y / det;
      out[3] = -e2x / det;
      out[4] = -e1y / det;
      out[5] = e1x / det;
    } else {
      double m00 = c[3] - c[0], m01 = c[6] - c[0], m02 = c[9] - c[0];
      double m10 = c[4] - c[1], m11 = c[7] - c[1], m12 = c[10] - c[1];
      double m20 = c[5] - c[2], m21 = c[8] - c[2], m22 = c[11] - c[2];
      double c00 = m11 * m22 - m12 * m21, c01 = m02 * m21 - m01 * m22, c02 = m01 * m12 - m02 * m11;
      double c10 = m12 * m20 - m10 * m22, c11 = m00 * m22 - m02 * m20, c12 = m02 * m10 - m00 * m12;
      double c20 = m10 * m21 - m11 * m20, c21 = m01 * m20 - m00 * m21, c22 = m00 * m11 - m01 * m10;
      double det = m00 * c00 + m01 * c10 + m02 * c20;
      out[0] = c[0];
      out[1] = c[1];
      out[2] = c[2];
      out[3] = c00 / det;
      out[4] = c01 / det;
      out[5] = c02 / det;
      out[6] = c10 / det;
      out[7] = c11 / det;
      out[8] = c12 / det;
      out[9] = c20 / det;
      out[10] = c21 / det;
      out[11] = c22 / det;
    }
  }
  }
}

int* stage_flag(Context& C) { return C.scalars.as<int>(256) + 36; }

// Checks the mesh and allocates its arrays.
static StageJob stage_job(DevMesh& M, int dim, int loc, long nnodes, long ne, const double* positions,
                          const int* enlist, bool need_planes, bool need_affine) {
  LSM_REQUIRE(dim == 2 || dim == 3, LIBSUPERMESH_GPU_ERROR_INVALID, "Invalid dimension");
  const bool simplex = loc == dim + 1;
  LSM_REQUIRE(simplex || loc == (1 << dim), LIBSUPERMESH_GPU_ERROR_INVALID,
              "Unsupported element type: simplices, quads or hexahedra only");
  LSM_REQUIRE(simplex || (!need_planes && !need_affine), LIBSUPERMESH_GPU_ERROR_INVALID,
              "Unsupported element type: clipping and mass take simplices only");
  LSM_REQUIRE(nnodes >= 0 && ne >= 0, LIBSUPERMESH_GPU_ERROR_INVALID, "Negative mesh size");
  LSM_REQUIRE(ne < (1L << 31) && nnodes < (1L << 31), LIBSUPERMESH_GPU_ERROR_OVERFLOW,
              "Mesh larger than 2^31 elements or nodes");
  LSM_REQUIRE(ne == 0 || nnodes > 0, LIBSUPERMESH_GPU_ERROR_INVALID, "No nodes");
  M.dim = dim;
  M.loc = loc;
  M.nnodes = nnodes;
  M.nelements = ne;
  M.ngroups = 0;
  M.enlist_dev = enlist;
  StageJob J;
  J.ne = ne;
  J.nnodes = nnodes;
  J.pos = positions;
  J.enl = enlist;
  J.coords = M.coords.as<double>((size_t)ne * loc * dim);
  J.bbox = M.bbox.as<double>((size_t)ne * 2 * dim);
  J.sp = M.meas_sp.as<double>((size_t)ne);
  J.scale = M.scale.as<double>((size_t)ne);
  J.planes = need_planes && dim == 3 ? M.planes.as<double>((size_t)ne * 16) : nullptr;
  J.affine = need_affine ? M.affine.as<double>((size_t)ne * (dim + dim * dim)) : nullptr;
  return J;
}

static void launch_stage(Context& C, int dim, int loc, const StageJob& a, const StageJob* b) {
  StageArgs args = {};
  args.job[0] = a;
  if (b) args.job[1] = *b;
  args.blocks0 = (a.ne + kBlock - 1) / kBlock;
  args.bad = stage_flag(C);
  args.serial = C.stage_serial;
  const long blocks = args.blocks0 + (b ? (b->ne + kBlock - 1) / kBlock : 0);
  if (blocks == 0) return;
  const dim3 grid((unsigned)blocks), block(kBlock);
  if (dim == 2) {
    if (loc == 3) hipLaunchKernelGGL((k_stage<2, 3>), grid, block, 0, C.stream, args);
    else hipLaunchKernelGGL((k_stage<2, 4>), grid, block, 0, C.stream, args);
  } else {
    if (loc == 4) hipLaunchKernelGGL((k_stage<3, 4>), grid, block, 0, C.stream, args);
    else hipLaunchKernelGGL((k_stage<3, 8>), grid, block, 0, C.stream, args);
  }
  LSM_HIP(hipGetLastError());
}

void stage_mesh(Context& C, DevMesh& M, int dim, int loc, long nnodes, long ne, const double* positions,
                const int* enlist, bool need_planes, bool need_affine) {
  const StageJob J = stage_job(M, dim, loc, nnodes, ne, positions, enlist, need_planes, need_affine);
  C.stage_serial++;
  launch_stage(C, dim, loc, J, nullptr);
  int hbad = 0;
  LSM_HIP(hipMemcpyAsync(&hbad, stage_flag(C), sizeof(int), hipMemcpyDeviceToHost, C.stream));
  LSM_HIP(hipStreamSynchronize(C.stream));
  LSM_REQUIRE(hbad != C.stage_serial, LIBSUPERMESH_GPU_ERROR_INVALID,
              "Invalid node: element-node index out of range");
}

void stage_meshes(Context& C, const libsupermesh_gpu_mesh& a, int loc_a, const libsupermesh_gpu_mesh& b, int loc_b,
                  bool planes_b, bool affine) {
  const StageJob A = stage_job(C.mesh_a, a.dim, loc_a, a.nnodes, a.nelements, a.positions, a.enlist, false, affine);
  const StageJob B = stage_job(C.mesh_b, b.dim, loc_b, b.nnodes, b.nelements, b.positions, b.enlist, planes_b, affine);
  C.stage_serial++;
  if (loc_a == loc_b) {
    launch_stage(C, a.dim, loc_a, A, &B);
  } else {
    launch_stage(C, a.dim, loc_a, A, nullptr);
    launch_stage(C, b.dim, loc_b, B, nullptr);
  }
}

__global__ void __launch_bounds__(kBlock)
k_groups(const long* __restrict__ offsets, int* __restrict__ group) {
  const long g = blockIdx.x;
  for (long e = offsets[g] + threadIdx.x; e < offsets[g + 1]; e += kBlock) group[e] = (int)g;
}

void stage_groups(Context& C, DevMesh& M, long ngroups, const long* offsets) {
  M.ngroups = 0;
  if (ngroups <= 0) return;
  LSM_REQUIRE(ngroups < (1L << 24), LIBSUPERMESH_GPU_ERROR_INVALID, "too many meshes in a batch");
  std::vector<long> h((size_t)ngroups + 1);
  LSM_HIP(hipMemcpyAsync(h.data(), offsets, sizeof(long) * (ngroups + 1), hipMemcpyDeviceToHost,
                         C.stream));
  LSM_HIP(hipStreamSynchronize(C.stream));
  LSM_REQUIRE(h[0] == 0 && h[ngroups] == M.nelements, LIBSUPERMESH_GPU_ERROR_INVALID,
              "batch element offsets must run from 0 to the element count");
  for (long g = 0; g < ngroups; g++)
    LSM_REQUIRE(h[g + 1] >= h[g], LIBSUPERMESH_GPU_ERROR_INVALID, "batch element offsets decrease");
  int* group = M.group.as<int>((size_t)M.nelements);
  hipLaunchKernelGGL(k_groups, dim3((unsigned)ngroups), dim3(kBlock), 0, C.stream, offsets, group);
  LSM_HIP(hipGetLastError());
  M.ngroups = ngroups;
}

// ---------------------------------------------------------------------------
// Morton codes and bounds
// ---------------------------------------------------------------------------

// Bounds of the block's values b (minima, then maxima), in every lane.
template <int DIM, int BLOCK = kBlock>
__device__ __forceinline__ void block_bounds(double* b) {
  __shared__ double red[BLOCK / 64][2 * DIM];
  for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      b[d] = fmin_f(b[d], __shfl_xor(b[d], o, 64));
      b[DIM + d] = fmax_f(b[DIM + d], __shfl_xor(b[DIM + d], o, 64));
    }
  }
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < 2 * DIM; k++) red[threadIdx.x >> 6][k] = b[k];
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < BLOCK / 64; w++) {
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      b[d] = fmin_f(b[d], red[w][d]);
      b[DIM + d] = fmax_f(b[DIM + d], red[w][DIM + d]);
    }
  }
}

// The search's words: [0] longest row, [1] tasks.
static long* search_words(Context& C) { return C.scalars.as<long>(128) + 16; }

// A sort of one mesh's elements by Morton code, or of two meshes' (the
// hierarchy's and the queries') in the same launches.
//
// A least-significant-digit radix sort, four passes of 8 bits: a pass counts
// the digits of every tile of kTile keys, then every tile adds up the counts
// before its own and moves its keys.  The counts of 2^shift tiles are also
// summed, so that a tile reads about 2 sqrt(tiles) rows of 256 counts.  Nine
// launches for both meshes and no block waits for another; the passes of a
// chained scan, where each block waits for the one before, took 30 us each
// for 2 M keys and three launches, and the merge sort below 1 M keys 11 to 21
// launches.
constexpr int kSortItems = 8;
constexpr int kTile = kSortItems * kBlock;
constexpr int kDigits = 256;
constexpr int kSortPasses = 4;
constexpr int kBoundParts = 256;

struct OrderJob {
  long ne;
  const double* bbox;
  const int* group;   // batches: the elements' meshes, above the code's leading bits
  int gbits;
  int nparts;
  double* bounds;     // [nparts][2 DIM]: parts of the centres' bounds
  uint32_t* keys[2];
  int* vals[2];
  int* perm;          // the order
  unsigned* counts;   // [tiles][kDigits]
  unsigned* sums;     // [kSortPasses][groups][kDigits]: counts of 2^shift tiles
  int tiles, groups, shift;
};

struct OrderArgs {
  OrderJob job[2];
  long* words;        // the search's [0] longest row, [1] tasks: cleared here
};

template <int DIM>
__global__ void __launch_bounds__(kBlock) k_center_bounds(OrderArgs args) {
  const OrderJob& J = args.job[blockIdx.y];
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 2) args.words[threadIdx.x] = 0;
  for (long k = (long)blockIdx.x * kBlock + threadIdx.x; k < (long)kSortPasses * J.groups * kDigits;
       k += (long)gridDim.x * kBlock)
    J.sums[k] = 0;
  if ((int)blockIdx.x >= J.nparts) return;
  double b[2 * DIM];
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    b[d] = __builtin_inf();
    b[DIM + d] = -__builtin_inf();
  }
  for (long e = (long)blockIdx.x * kBlock + threadIdx.x; e < J.ne; e += (long)J.nparts * kBlock) {
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      double c = 0.5 * (J.bbox[(long)d * J.ne + e] + J.bbox[(long)(DIM + d) * J.ne + e]);
      b[d] = fmin_f(b[d], c);
      b[DIM + d] = fmax_f(b[DIM + d], c);
    }
  }
  block_bounds<DIM>(b);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < 2 * DIM; k++) J.bounds[blockIdx.x * 2 * DIM + k] = b[k];
  }
}

__device__ __forceinline__ uint64_t spread2(uint64_t x) {  // 32 bits -> even bits
  x &= 0xffffffffULL;
  x = (x | (x << 16)) & 0x0000ffff0000ffffULL;
  x = (x | (x << 8)) & 0x00ff00ff00ff00ffULL;
  x = (x | (x << 4)) & 0x0f0f0f0f0f0f0f0fULL;
  x = (x | (x << 2)) & 0x3333333333333333ULL;
  x = (x | (x << 1)) & 0x5555555555555555ULL;
  return x;
}

__device__ __forceinline__ uint64_t spread3(uint64_t x) {  // 21 bits -> every third bit
  x &= 0x1fffffULL;
  x = (x | (x << 32)) & 0x1f00000000ffffULL;
  x = (x | (x << 16)) & 0x1f0000ff0000ffULL;
  x = (x | (x << 8)) & 0x100f00f00f00f00fULL;
  x = (x | (x << 4)) & 0x10c30c30c30c30c3ULL;
  x = (x | (x << 2)) & 0x1249249249249249ULL;
  return x;
}

// Sort key of element e: its Morton code, or in a batch the mesh id in the
// top gbits bits above the code's leading bits, so that each mesh is one
// contiguous run of the order.  The leading 32 bits (16 per axis in 2D, 10-11
// in 3D, below a batch's mesh id) order the elements finely enough for the
// hierarchy; ties keep element order (the sort is stable), and the candidate
// sets do not depend on the order at all.
template <int DIM>
__device__ __forceinline__ uint32_t morton_key(const OrderJob& J, const double* bounds, long e) {
  constexpr int BITS = DIM == 2 ? 32 : 21;
  const double maxq = (double)((1ULL << BITS) - 1);
  uint64_t code = 0;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    double lo = bounds[d], hi = bounds[DIM + d];
    double c = 0.5 * (J.bbox[(long)d * J.ne + e] + J.bbox[(long)(DIM + d) * J.ne + e]);
    double t = hi > lo ? (c - lo) / (hi - lo) : 0.0;
    t = fmin_f(fmax_f(t, 0.0), 1.0);
    uint64_t q = (uint64_t)(t * maxq);
    code |= (DIM == 2 ? spread2(q) : spread3(q)) << d;
  }
  constexpr int KEYBITS = DIM == 2 ? 64 : 63;
  if (J.group && J.gbits > 0) code = ((uint64_t)J.group[e] << (KEYBITS - J.gbits)) | (code >> J.gbits);
  return (uint32_t)(code >> (KEYBITS - 32));
}

// The block's job and its tile in that job.
__device__ __forceinline__ const OrderJob& tile_job(const OrderArgs& args, int& tile) {
  tile = blockIdx.x;
  if (tile < args.job[0].tiles) return args.job[0];
  tile -= args.job[0].tiles;
  return args.job[1];
}

// A tile's digit counts to its row and to its group's sums.
__device__ __forceinline__ void write_counts(const OrderJob& J, int tile, int pass, unsigned n) {
  J.counts[(long)tile * kDigits + threadIdx.x] = n;
  if (n) atomicAdd(J.sums + ((long)pass * J.groups + (tile >> J.shift)) * kDigits + threadIdx.x, n);
}

// Keys of a tile's elements, and the counts of their lowest digit.  With
// VALS, element ids beside the keys instead, for the other sorts.
template <int DIM, bool VALS>
__global__ void __launch_bounds__(kBlock) k_morton(OrderArgs args) {
  __shared__ unsigned hist[kDigits];
  int tile;
  const OrderJob& J = tile_job(args, tile);
  double b[2 * DIM];
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    b[d] = __builtin_inf();
    b[DIM + d] = -__builtin_inf();
  }
  if ((int)threadIdx.x < J.nparts) {
#pragma unroll
    for (int k = 0; k < 2 * DIM; k++) b[k] = J.bounds[threadIdx.x * 2 * DIM + k];
  }
  hist[threadIdx.x] = 0;
  block_bounds<DIM>(b);  // a barrier
#pragma unroll
  for (int i = 0; i < kSortItems; i++) {
    const long e = (long)tile * kTile + i * kBlock + threadIdx.x;
    if (e >= J.ne) break;
    const uint32_t key = morton_key<DIM>(J, b, e);
    J.keys[0][e] = key;
    if (VALS) J.vals[0][e] = (int)e;
    else atomicAdd(&hist[key & (kDigits - 1)], 1u);
  }
  if (VALS) return;
  __syncthreads();
  write_counts(J, tile, 0, hist[threadIdx.x]);
}

__global__ void __launch_bounds__(kBlock) k_sort_counts(OrderArgs args, int pass) {
  __shared__ unsigned hist[kDigits];
  int tile;
  const OrderJob& J = tile_job(args, tile);
  const uint32_t* __restrict__ keys = J.keys[pass & 1];
  hist[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSortItems; i++) {
    const long e = (long)tile * kTile + i * kBlock + threadIdx.x;
    if (e < J.ne) atomicAdd(&hist[(keys[e] >> (8 * pass)) & (kDigits - 1)], 1u);
  }
  __syncthreads();
  write_counts(J, tile, pass, hist[threadIdx.x]);
}

// Rank of this lane's key among the wave's keys of the same digit d, those of
// earlier calls first; `counts`, the wave's, go on from call to call.
__device__ __forceinline__ int rank_digit(unsigned d, bool live, unsigned* counts) {
  const int lane = threadIdx.x & 63;
  unsigned long long m = __ballot(live);
#pragma unroll
  for (int b = 0; b < 8; b++) {
    const unsigned long long v = __ballot((d >> b) & 1u);
    m &= (d >> b) & 1u ? v : ~v;
  }
  const int lower = __builtin_popcountll(m & ((1ULL << lane) - 1));
  unsigned old = 0;
  if (live && lower == 0) old = atomicAdd(counts + d, (unsigned)__builtin_popcountll(m));
  return (int)__shfl(old, live ? __builtin_ctzll(m) : lane, 64) + lower;
}

// Moves a tile's keys and element ids to their places for one digit.  A wave
// ranks 64 keys at a time among its own (the lanes of equal digit by eight
// ballots), the tile is put in digit order in LDS, and neighbouring lanes
// then write neighbouring places.  The first pass's ids are the indices, the
// last one writes the order alone.
template <int PASS>
__global__ void __launch_bounds__(kBlock) k_sort_move(OrderArgs args) {
  constexpr int kWaves = kBlock / 64;
  constexpr bool kLast = PASS == kSortPasses - 1;
  __shared__ unsigned hist[kWaves][kDigits], place[kDigits], wsum[2][kWaves];
  __shared__ uint32_t skey[kTile];
  __shared__ int sval[kTile];
  int tile;
  const OrderJob& J = tile_job(args, tile);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t* __restrict__ keys = J.keys[PASS & 1];
  const int* __restrict__ vals = J.vals[PASS & 1];
  const long first = (long)tile * kTile;
  const int n = J.ne - first < kTile ? (int)(J.ne - first) : kTile;
#pragma unroll
  for (int w = 0; w < kWaves; w++) hist[w][t] = 0;
  uint32_t key[kSortItems];
  int val[kSortItems], rank[kSortItems];
#pragma unroll
  for (int i = 0; i < kSortItems; i++) {
    const int k = (wave * kSortItems + i) * 64 + lane;
    key[i] = k < n ? keys[first + k] : 0;
    val[i] = PASS == 0 ? (int)(first + k) : (k < n ? vals[first + k] : 0);
  }
  // digit t: its keys in all tiles, and in the tiles before this one
  unsigned all = 0, before = 0;
  {
    const int mine = tile >> J.shift;
    const unsigned* __restrict__ s = J.sums + (long)PASS * J.groups * kDigits + t;
#pragma unroll 8
    for (int g = 0; g < J.groups; g++) {
      const unsigned v = s[(long)g * kDigits];
      all += v;
      before += g < mine ? v : 0u;
    }
    const unsigned* __restrict__ c = J.counts + t;
#pragma unroll 8
    for (int k = mine << J.shift; k < tile; k++) before += c[(long)k * kDigits];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSortItems; i++) {
    rank[i] = rank_digit((key[i] >> (8 * PASS)) & (kDigits - 1), (wave * kSortItems + i) * 64 + lane < n, hist[wave]);
  }
  __syncthreads();
  unsigned mine = 0;  // digit t's keys in this tile; each wave's first place among them
#pragma unroll
  for (int w = 0; w < kWaves; w++) {
    const unsigned c = hist[w][t];
    hist[w][t] = mine;
    mine += c;
  }
  unsigned local = mine, global = all;  // inclusive scans over the digits
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned x = __shfl_up(local, o, 64), y = __shfl_up(global, o, 64);
    if (lane >= o) {
      local += x;
      global += y;
    }
  }
  if (lane == 63) {
    wsum[0][wave] = local;
    wsum[1][wave] = global;
  }
  __syncthreads();
  for (int w = 0; w < wave; w++) {
    local += wsum[0][w];
    global += wsum[1][w];
  }
  local -= mine;  // digit t's first place in the tile
#pragma unroll
  for (int w = 0; w < kWaves; w++) hist[w][t] += local;
  place[t] = global - all + before - local;  // place in the output = this + place in the tile
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kSortItems; i++) {
    if ((wave * kSortItems + i) * 64 + lane < n) {
      const unsigned o = hist[wave][(key[i] >> (8 * PASS)) & (kDigits - 1)] + (unsigned)rank[i];
      skey[o] = key[i];
      sval[o] = val[i];
    }
  }
  __syncthreads();
  int* __restrict__ out = kLast ? J.perm : J.vals[(PASS + 1) & 1];
#pragma unroll
  for (int i = 0; i < kSortItems; i++) {
    const int k = i * kBlock + t;
    if (k >= n) break;
    const unsigned o = place[(skey[k] >> (8 * PASS)) & (kDigits - 1)] + (unsigned)k;
    if (!kLast) J.keys[(PASS + 1) & 1][o] = skey[k];
    out[o] = sval[k];
  }
}

// Elements of a mesh above which the library's sort takes over.  In a pass a tile
// reads 0.4 counts per key at 2^13 elements, 4 at 2^20, 12 at 2^23 and 16 at
// 2^24, which uses up what nine launches for both meshes save: the search of a
// mesh in itself takes 0.20 ms less than with the library's sort at 1 M elements
// (0.75 against 0.95), 0.15 less at 2 M, 0.19 at 4.2 M, 0.09 to 0.18 at 8.4 M,
// and 0.03 ms more at 16.8 M.
constexpr long kOrderMax = 1L << 23;

// ---------------------------------------------------------------------------
// Implicit hierarchy
// ---------------------------------------------------------------------------

struct LevelInfo {
  int levels;
  long count[32];
  long offset[32];
};

static LevelInfo level_info(const DevBVH& H) {
  LevelInfo info;
  info.levels = H.levels;
  for (int l = 0; l < 32; l++) {
    info.count[l] = l < H.levels ? H.count[l] : 0;
    info.offset[l] = l < H.levels ? H.offset[l] : 0;
  }
  return info;
}

// A node's box [lo_0..lo_{dim-1}, hi_0..hi_{dim-1}] and, in batches, its mesh
// range.
template <int DIM>
struct NodeBox {
  double b[2 * DIM];
  int glo, ghi;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      b[d] = __builtin_inf();
      b[DIM + d] = -__builtin_inf();
    }
    glo = 0x7fffffff;
    ghi = -1;
  }
  __device__ __forceinline__ void element(long e, long ne, const double* __restrict__ bbox,
                                          const int* __restrict__ group) {
#pragma unroll
    for (int k = 0; k < 2 * DIM; k++) b[k] = bbox[(long)k * ne + e];
    if (group) glo = ghi = group[e];
  }
  __device__ __forceinline__ void store(const LevelInfo& info, int l, long node, double* __restrict__ boxes,
                                        int* __restrict__ granges) const {
    if (l >= info.levels || node >= info.count[l]) return;
    const long o = info.offset[l] + node;
#pragma unroll
    for (int k = 0; k < 2 * DIM; k++) boxes[o * 2 * DIM + k] = b[k];
    if (granges) {
      granges[2 * o] = glo;
      granges[2 * o + 1] = ghi;
    }
  }
  __device__ __forceinline__ void add(const NodeBox& x) {
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      b[d] = __builtin_fmin(b[d], x.b[d]);
      b[DIM + d] = __builtin_fmax(b[DIM + d], x.b[DIM + d]);
    }
    glo = std::min(glo, x.glo);
    ghi = std::max(ghi, x.ghi);
  }
  // the union with the lanes whose number differs in bit o
  __device__ __forceinline__ void join(int o) {
    NodeBox x;
#pragma unroll
    for (int k = 0; k < 2 * DIM; k++) x.b[k] = __shfl_xor(b[k], o, 64);
    x.glo = __shfl_xor(glo, o, 64);
    x.ghi = __shfl_xor(ghi, o, 64);
    add(x);
  }
};

// Boxes of the three levels above `l0`, and of the elements themselves in
// sorted order if l0 is 0: a wave's 64 nodes have eight parents and one
// grandparent, which come from shuffles, and the block's 512 one node above
// those.  (A launch a level took 5 us each; the nodes were read again.)
constexpr int kLevelBlock = kFanout * kFanout * kFanout;
template <int DIM>
__global__ void __launch_bounds__(kLevelBlock)
k_build_levels(LevelInfo info, int l0, long ne, const double* __restrict__ bbox, const int* __restrict__ perm,
               const int* __restrict__ group, double* __restrict__ boxes, int* __restrict__ granges) {
  __shared__ NodeBox<DIM> top[kFanout];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long i = (long)blockIdx.x * kLevelBlock + threadIdx.x;
  NodeBox<DIM> x;
  x.clear();
  if (i < info.count[l0]) {
    if (l0 == 0) {
      x.element(perm[i], ne, bbox, group);
      x.store(info, 0, i, boxes, granges);
    } else {
      const long o = info.offset[l0] + i;
#pragma unroll
      for (int k = 0; k < 2 * DIM; k++) x.b[k] = boxes[o * 2 * DIM + k];
      if (granges) {
        x.glo = granges[2 * o];
        x.ghi = granges[2 * o + 1];
      }
    }
  }
  for (int o = 1; o < kFanout; o <<= 1) x.join(o);
  if ((lane & 7) == 0) x.store(info, l0 + 1, i / kFanout, boxes, granges);
  for (int o = kFanout; o < 64; o <<= 1) x.join(o);
  if (lane == 0) {
    x.store(info, l0 + 2, i / (kFanout * kFanout), boxes, granges);
    top[wave] = x;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kFanout; w++) x.add(top[w]);
  x.store(info, l0 + 3, blockIdx.x, boxes, granges);
}

// Tiny meshes, a block each: order and, for the first, the hierarchy in one
// launch (five otherwise, each a few microseconds of latency with next to no
// work).  A thread holds a key through the four passes, exchanged in LDS; the
// 64 boxes of a wave give two levels by shuffles, the at most 16 boxes of the
// second level the rest.  With eight keys a thread a block took 73 us for
// 8192 elements: k_rank does those on the whole card.
constexpr int kSmallBlock = 1024;
constexpr long kSmallMax = kSmallBlock;
template <int DIM>
__global__ void __launch_bounds__(kSmallBlock)
k_small_order(OrderArgs args, LevelInfo info, double* __restrict__ boxes, int* __restrict__ granges) {
  constexpr int kWaves = kSmallBlock / 64;
  struct Sort {
    unsigned hist[kWaves][kDigits], wsum[kDigits / 64];
    uint32_t key[kSmallMax];
    int val[kSmallMax];
  };
  __shared__ union {
    Sort sort;
    NodeBox<DIM> top[kWaves];
  } mem;
  const OrderJob& J = args.job[blockIdx.x];
  if (blockIdx.x == 0 && threadIdx.x < 2) args.words[threadIdx.x] = 0;
  const int n = (int)J.ne, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (n == 0) return;
  const bool live = t < n;
  double b[2 * DIM];
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    b[d] = __builtin_inf();
    b[DIM + d] = -__builtin_inf();
  }
  if (live) {
#pragma unroll
    for (int d = 0; d < DIM; d++) b[d] = b[DIM + d] = 0.5 * (J.bbox[d * n + t] + J.bbox[(DIM + d) * n + t]);
  }
  block_bounds<DIM, kSmallBlock>(b);
  uint32_t key = live ? morton_key<DIM>(J, b, t) : 0;
  int val = t;
  for (int pass = 0; pass < kSortPasses; pass++) {
    const int shift = 8 * pass;
#pragma unroll
    for (int k = 0; k < kWaves * kDigits / kSmallBlock; k++) (&mem.sort.hist[0][0])[k * kSmallBlock + t] = 0;
    __syncthreads();
    const int rank = rank_digit((key >> shift) & (kDigits - 1), live, mem.sort.hist[wave]);
    __syncthreads();
    unsigned mine = 0, sum = 0;
    if (t < kDigits) {
#pragma unroll
      for (int w = 0; w < kWaves; w++) {
        const unsigned c = mem.sort.hist[w][t];
        mem.sort.hist[w][t] = mine;
        mine += c;
      }
      sum = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned x = __shfl_up(sum, o, 64);
        if (lane >= o) sum += x;
      }
      if (lane == 63) mem.sort.wsum[wave] = sum;
    }
    __syncthreads();
    if (t < kDigits) {
      for (int w = 0; w < wave; w++) sum += mem.sort.wsum[w];
#pragma unroll
      for (int w = 0; w < kWaves; w++) mem.sort.hist[w][t] += sum - mine;
    }
    __syncthreads();
    if (live) {
      const unsigned o = mem.sort.hist[wave][(key >> shift) & (kDigits - 1)] + (unsigned)rank;
      mem.sort.key[o] = key;
      mem.sort.val[o] = val;
    }
    __syncthreads();
    if (live) {
      key = mem.sort.key[t];
      val = mem.sort.val[t];
    }
  }
  __syncthreads();
  if (live) J.perm[t] = val;
  if (blockIdx.x != 0 || boxes == nullptr) return;
  NodeBox<DIM> x;
  x.clear();
  if (live) {
    x.element(val, n, J.bbox, J.group);
    x.store(info, 0, t, boxes, granges);
  }
  for (int o = 1; o < kFanout; o <<= 1) x.join(o);
  if ((lane & 7) == 0) x.store(info, 1, t / kFanout, boxes, granges);
  for (int o = kFanout; o < 64; o <<= 1) x.join(o);
  if (lane == 0) {
    x.store(info, 2, wave, boxes, granges);
    mem.top[wave] = x;
  }
  __syncthreads();
  if (wave != 0) return;
  x.clear();
  if (lane < kWaves) x = mem.top[lane];
  for (int o = 1; o < kFanout; o <<= 1) x.join(o);
  if ((lane & 7) == 0) x.store(info, 3, lane / kFanout, boxes, granges);
  x.join(kFanout);  // kWaves is two groups
  if (lane == 0) x.store(info, 4, 0, boxes, granges);
}

// The order of a small mesh's keys by counting: an element's place is the
// number of smaller keys, and of equal ones before it.  64 elements to a
// block, a lane each; each wave goes through every sixteenth 64 keys.  n^2
// compares, but one launch on the whole card where the sort's seven wait for
// each other: up to 8192 elements that is the shorter (the sort costs about
// 45 us whatever the size).
constexpr int kRankBlock = 1024;
constexpr long kRankMax = 8192;
__global__ void __launch_bounds__(kRankBlock) k_rank(OrderArgs args, int blocks0) {
  constexpr int kWaves = kRankBlock / 64;
  __shared__ __align__(16) uint32_t keys[kRankMax];
  __shared__ int part[kWaves][64];
  const bool second = (int)blockIdx.x >= blocks0;
  const OrderJob& J = args.job[second ? 1 : 0];
  const int mine = (int)blockIdx.x - (second ? blocks0 : 0);
  const int n = (int)J.ne, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunks = (n + 63) / 64;
  for (int k = threadIdx.x; k < chunks * 64; k += kRankBlock) keys[k] = k < n ? J.keys[0][k] : 0xffffffffu;
  __syncthreads();
  const uint32_t key = keys[mine * 64 + lane];
  int place = 0;
  for (int c = wave; c < chunks; c += kWaves) {
    const uint4* k = reinterpret_cast<const uint4*>(keys + c * 64);
    if (c < mine) {
#pragma unroll
      for (int j = 0; j < 16; j++) {
        const uint4 x = k[j];
        place += (x.x <= key) + (x.y <= key) + (x.z <= key) + (x.w <= key);
      }
    } else if (c > mine) {
#pragma unroll
      for (int j = 0; j < 16; j++) {
        const uint4 x = k[j];
        place += (x.x < key) + (x.y < key) + (x.z < key) + (x.w < key);
      }
    } else {
      for (int j = 0; j < 64; j++) {
        const uint32_t x = keys[c * 64 + j];
        place += x < key || (x == key && j < lane);
      }
    }
  }
  part[wave][lane] = place;
  __syncthreads();
  if (wave != 0 || mine * 64 + lane >= n) return;
  place = 0;
#pragma unroll
  for (int w = 0; w < kWaves; w++) place += part[w][lane];
  J.perm[place] = mine * 64 + lane;
}

// Sorts the elements of M[0], and of M[1] if it is given, by Morton code:
// perm[j] gets the permutation.
// With H (set up but for its boxes), the boxes of its levels over M[0] too.
static void morton_order(Context& C, int n, const DevMesh* const* M, DevBuf* const* perm, const DevBVH* H) {
  OrderArgs args = {};
  args.words = search_words(C);
  size_t total = 0, words = 0;
  bool large = false, small = true, count = true;
  for (int j = 0; j < n; j++) {
    OrderJob& J = args.job[j];
    J.ne = M[j]->nelements;
    J.bbox = static_cast<const double*>(M[j]->bbox.ptr);
    J.group = M[j]->ngroups > 0 ? static_cast<const int*>(M[j]->group.ptr) : nullptr;
    while (J.group && (1L << J.gbits) < M[j]->ngroups) J.gbits++;
    J.nparts = (int)std::min<long>(kBoundParts, (J.ne + kBlock - 1) / kBlock);
    J.tiles = (int)((J.ne + kTile - 1) / kTile);
    while ((1 << (2 * J.shift)) < J.tiles) J.shift++;
    J.groups = (J.tiles + (1 << J.shift) - 1) >> J.shift;
    J.perm = perm[j]->as<int>(J.ne);
    total += (size_t)J.ne;
    words += (size_t)(J.tiles + kSortPasses * J.groups) * kDigits;
    large = large || J.ne > kOrderMax;
    small = small && J.ne <= kSmallMax;
    count = count && J.ne <= kRankMax;
  }
  const bool flat = M[0]->dim == 2;
  const dim3 block(kBlock);
  LevelInfo info = {};
  double* boxes = nullptr;
  int* granges = nullptr;
  if (H) {
    info = level_info(*H);
    boxes = static_cast<double*>(H->boxes.ptr);
    granges = H->grouped ? static_cast<int*>(H->granges.ptr) : nullptr;
  }
  if (small) {
    const dim3 grid((unsigned)n), threads(kSmallBlock);
    if (flat) hipLaunchKernelGGL(k_small_order<2>, grid, threads, 0, C.stream, args, info, boxes, granges);
    else hipLaunchKernelGGL(k_small_order<3>, grid, threads, 0, C.stream, args, info, boxes, granges);
    LSM_HIP(hipGetLastError());
    return;
  }
  double* part = C.partials.as<double>((size_t)n * kBoundParts * 6);
  uint32_t* keys[2] = {C.keys.as<uint32_t>(total), C.keys_alt.as<uint32_t>(total)};
  int* vals[2] = {C.vals.as<int>(total), C.vals_alt.as<int>(total)};
  unsigned* table = large || count ? nullptr : C.sort_tmp.as<unsigned>(words);
  size_t at = 0;
  for (int j = 0; j < n; j++) {
    OrderJob& J = args.job[j];
    J.bounds = part + (size_t)j * kBoundParts * 6;
    for (int k = 0; k < 2; k++) {
      J.keys[k] = keys[k] + at;
      J.vals[k] = vals[k] + at;
    }
    at += (size_t)J.ne;
    if (large || count) {
      J.groups = 0;
      continue;
    }
    J.counts = table;
    J.sums = table + (size_t)J.tiles * kDigits;
    table += (size_t)(J.tiles + kSortPasses * J.groups) * kDigits;
  }
  const dim3 parts((unsigned)std::max(1, std::max(args.job[0].nparts, args.job[1].nparts)), (unsigned)n);
  const dim3 tiles((unsigned)std::max(1, args.job[0].tiles + args.job[1].tiles));
  if (flat) hipLaunchKernelGGL(k_center_bounds<2>, parts, block, 0, C.stream, args);
  else hipLaunchKernelGGL(k_center_bounds<3>, parts, block, 0, C.stream, args);
  if (count) {
    if (flat) hipLaunchKernelGGL((k_morton<2, true>), tiles, block, 0, C.stream, args);
    else hipLaunchKernelGGL((k_morton<3, true>), tiles, block, 0, C.stream, args);
    const int blocks0 = (int)((args.job[0].ne + 63) / 64), blocks1 = (int)((args.job[1].ne + 63) / 64);
    hipLaunchKernelGGL(k_rank, dim3((unsigned)(blocks0 + blocks1)), dim3(kRankBlock), 0, C.stream, args, blocks0);
  } else if (large) {
    if (flat) hipLaunchKernelGGL((k_morton<2, true>), tiles, block, 0, C.stream, args);
    else hipLaunchKernelGGL((k_morton<3, true>), tiles, block, 0, C.stream, args);
    LSM_HIP(hipGetLastError());
    for (int j = 0; j < n; j++) {
      const OrderJob& J = args.job[j];
      if (J.ne == 0) continue;
      size_t bytes = 0;
      LSM_HIP(rocprim::radix_sort_pairs(nullptr, bytes, J.keys[0], J.keys[1], J.vals[0], J.perm, (size_t)J.ne, 0u, 32u,
                                        C.stream));
      void* tmp = C.sort_tmp.get(bytes);
      LSM_HIP(rocprim::radix_sort_pairs(tmp, bytes, J.keys[0], J.keys[1], J.vals[0], J.perm, (size_t)J.ne, 0u, 32u,
                                        C.stream));
    }
  } else {
    if (flat) hipLaunchKernelGGL((k_morton<2, false>), tiles, block, 0, C.stream, args);
    else hipLaunchKernelGGL((k_morton<3, false>), tiles, block, 0, C.stream, args);
    hipLaunchKernelGGL(k_sort_move<0>, tiles, block, 0, C.stream, args);
    hipLaunchKernelGGL(k_sort_counts, tiles, block, 0, C.stream, args, 1);
    hipLaunchKernelGGL(k_sort_move<1>, tiles, block, 0, C.stream, args);
    hipLaunchKernelGGL(k_sort_counts, tiles, block, 0, C.stream, args, 2);
    hipLaunchKernelGGL(k_sort_move<2>, tiles, block, 0, C.stream, args);
    hipLaunchKernelGGL(k_sort_counts, tiles, block, 0, C.stream, args, 3);
    hipLaunchKernelGGL(k_sort_move<3>, tiles, block, 0, C.stream, args);
  }
  for (int l = 0; H && (l == 0 || l + 1 < H->levels); l += 3) {
    const dim3 grid(grid_for(H->count[l], kLevelBlock)), threads(kLevelBlock);
    const OrderJob& J = args.job[0];
    if (flat) hipLaunchKernelGGL(k_build_levels<2>, grid, threads, 0, C.stream, info, l, J.ne, J.bbox, J.perm, J.group, boxes, granges);
    else hipLaunchKernelGGL(k_build_levels<3>, grid, threads, 0, C.stream, info, l, J.ne, J.bbox, J.perm, J.group, boxes, granges);
  }
  LSM_HIP(hipGetLastError());
}

void build_bvh(Context& C, const DevMesh& B, const DevMesh* A) {
  DevBVH& H = C.bvh;
  H.dim = B.dim;
  H.n = B.nelements;
  if (H.n == 0) {
    H.levels = 0;
    return;
  }
  long n = H.n;
  int L = 0;
  long total = 0;
  while (true) {
    H.count[L] = n;
    H.offset[L] = total;
    total += n;
    L++;
    if (n == 1) break;
    n = (n + kFanout - 1) / kFanout;
    LSM_REQUIRE(L < 31, LIBSUPERMESH_GPU_ERROR_OVERFLOW, "hierarchy too deep");
  }
  H.levels = L;
  H.total = total;
  H.grouped = B.ngroups > 0;
  // a walk reads whole groups of children, past the last node too
  H.boxes.as<double>((size_t)(total + kFanout) * 2 * B.dim);
  if (H.grouped) H.granges.as<int>((size_t)(total + kFanout) * 2);
  const DevMesh* meshes[2] = {&B, A};
  DevBuf* orders[2] = {&H.perm, &C.qperm};
  morton_order(C, A ? 2 : 1, meshes, orders, &H);
}

// ---------------------------------------------------------------------------
// Traversal
// ---------------------------------------------------------------------------

// Raises *max to the largest x of the wave; the value read first spares
// nearly all waves the atomic.
__device__ __forceinline__ void raise_max(long* max, int x) {
  for (int o = 32; o > 0; o >>= 1) {
    const int y = __shfl_xor(x, o, 64);
    x = y > x ? y : x;
  }
  if ((threadIdx.x & 63) == 0 && x > *reinterpret_cast<volatile long*>(max)) atomicMax(reinterpret_cast<unsigned long long*>(max), (unsigned long long)x);
}

__global__ void k_clear_words(int n, long* __restrict__ w) {
  if ((int)threadIdx.x < n && blockIdx.x == 0) w[threadIdx.x] = 0;
}

struct SearchArgs {
  long na;
  const int* qperm;     // A's elements in Morton order, kQueries to a wave
  const double* abox;   // [2 DIM][na]
  const int* agroup;    // batches: A's and the nodes' meshes
  const int* granges;
  const double* boxes;
  const int* perm;
  LevelInfo info;
  // tasks: (query wave, node at `level`) pairs; without them, every wave
  // starts at the root
  const int2* tasks;
  const unsigned long long* ntasks;
  unsigned cap;         // tasks that the arrays hold
  int level;
  int* tcount;          // [cap][kQueries]: results of the wave's queries below the task's node, then their prefix sums
  long* row_count;      // [na]
  long* maxrow;
  const long* indptr;
  int* indices;
  int* rows;
};

// A wave tests its queries eight at a time against a node's eight children:
// lane 8 q + c holds child c's box and the queries q of each of the kGroups
// groups of eight.  A node's boxes are then three loads for the wave, one
// compare tests 64 (query, child) pairs, and a query's results lie in
// neighbouring lanes, so that they are written together.
constexpr int kGroups = 4;
constexpr int kQueries = 8 * kGroups;

template <int DIM, bool GROUPED>
struct Queries {
  int a[kGroups], g[kGroups];
  double lo[kGroups][DIM], hi[kGroups][DIM];
  __device__ __forceinline__ Queries(const SearchArgs& s, long wave) {
#pragma unroll
    for (int i = 0; i < kGroups; i++) {
      const long t = wave * kQueries + 8 * i + ((threadIdx.x & 63) >> 3);
      const bool live = t < s.na;
      a[i] = live ? s.qperm[t] : -1;
#pragma unroll
      for (int d = 0; d < DIM; d++) {  // no box overlaps NaN bounds
        lo[i][d] = live ? s.abox[(long)d * s.na + a[i]] : __builtin_nan("");
        hi[i][d] = live ? s.abox[(long)(DIM + d) * s.na + a[i]] : __builtin_nan("");
      }
      g[i] = GROUPED && live ? s.agroup[a[i]] : -1;
    }
  }
};

// Lanes of `start` whose box [lo, hi] (and mesh range) overlaps the query:
// each compare narrows the execution mask that the next one runs under, so
// the conjunction costs no mask arithmetic on the scalar unit, which one walk
// with a scalar `and` per compare was bound by.  `full` is the mask to go on
// with.  Strict: hi > qlo and lo < qhi (Quadtree_...F90:411-420); closed: not
// strict.
template <int DIM, bool CLOSED>
__device__ __forceinline__ unsigned long long overlap_lanes(unsigned long long start, unsigned long long full,
                                                            const double* lo, const double* hi, const double* qlo,
                                                            const double* qhi) {
  unsigned long long m;
  if constexpr (DIM == 2) {
    if constexpr (CLOSED)
      asm volatile("s_mov_b64 exec, %1\n\tv_cmpx_ge_f64 vcc, %3, %4\n\tv_cmpx_le_f64 vcc, %5, %6\n\t"
                   "v_cmpx_ge_f64 vcc, %7, %8\n\tv_cmpx_le_f64 vcc, %9, %10\n\ts_mov_b64 %0, exec\n\ts_mov_b64 exec, %2"
                   : "=&s"(m)
                   : "s"(start), "s"(full), "v"(hi[0]), "v"(qlo[0]), "v"(lo[0]), "v"(qhi[0]), "v"(hi[1]), "v"(qlo[1]),
                     "v"(lo[1]), "v"(qhi[1])
                   : "vcc");
    else
      asm volatile("s_mov_b64 exec, %1\n\tv_cmpx_gt_f64 vcc, %3, %4\n\tv_cmpx_lt_f64 vcc, %5, %6\n\t"
                   "v_cmpx_gt_f64 vcc, %7, %8\n\tv_cmpx_lt_f64 vcc, %9, %10\n\ts_mov_b64 %0, exec\n\ts_mov_b64 exec, %2"
                   : "=&s"(m)
                   : "s"(start), "s"(full), "v"(hi[0]), "v"(qlo[0]), "v"(lo[0]), "v"(qhi[0]), "v"(hi[1]), "v"(qlo[1]),
                     "v"(lo[1]), "v"(qhi[1])
                   : "vcc");
  } else {
    if constexpr (CLOSED)
      asm volatile("s_mov_b64 exec, %1\n\tv_cmpx_ge_f64 vcc, %3, %4\n\tv_cmpx_le_f64 vcc, %5, %6\n\t"
                   "v_cmpx_ge_f64 vcc, %7, %8\n\tv_cmpx_le_f64 vcc, %9, %10\n\tv_cmpx_ge_f64 vcc, %11, %12\n\t"
                   "v_cmpx_le_f64 vcc, %13, %14\n\ts_mov_b64 %0, exec\n\ts_mov_b64 exec, %2"
                   : "=&s"(m)
                   : "s"(start), "s"(full), "v"(hi[0]), "v"(qlo[0]), "v"(lo[0]), "v"(qhi[0]), "v"(hi[1]), "v"(qlo[1]),
                     "v"(lo[1]), "v"(qhi[1]), "v"(hi[2]), "v"(qlo[2]), "v"(lo[2]), "v"(qhi[2])
                   : "vcc");
    else
      asm volatile("s_mov_b64 exec, %1\n\tv_cmpx_gt_f64 vcc, %3, %4\n\tv_cmpx_lt_f64 vcc, %5, %6\n\t"
                   "v_cmpx_gt_f64 vcc, %7, %8\n\tv_cmpx_lt_f64 vcc, %9, %10\n\tv_cmpx_gt_f64 vcc, %11, %12\n\t"
                   "v_cmpx_lt_f64 vcc, %13, %14\n\ts_mov_b64 %0, exec\n\ts_mov_b64 exec, %2"
                   : "=&s"(m)
                   : "s"(start), "s"(full), "v"(hi[0]), "v"(qlo[0]), "v"(lo[0]), "v"(qhi[0]), "v"(hi[1]), "v"(qlo[1]),
                     "v"(lo[1]), "v"(qhi[1]), "v"(hi[2]), "v"(qlo[2]), "v"(lo[2]), "v"(qhi[2])
                   : "vcc");
  }
  return m;
}

// Bit c of the result: some query's byte has bit c.
__device__ __forceinline__ unsigned any_query(const unsigned long long* m) {
  unsigned long long u = 0;
#pragma unroll
  for (int i = 0; i < kGroups; i++) u |= m[i];
  unsigned v = (unsigned)u | (unsigned)(u >> 32);
  v |= v >> 16;
  return (v | v >> 8) & 0xffu;
}

// Visits the nodes below `start` (a node of level `from`, above `to`) whose
// children at level `to` some query overlaps, in index order: hit(first, m)
// with the first child's index and, per group, bit 8 q + c where query q
// overlaps child c.  The wave walks the union of its queries' depth-first
// paths (consecutive queries are close in Morton order, so their paths mostly
// coincide) and keeps, per level, a byte of the children still to visit.  A
// query may be tested against a node whose parent it misses: the boxes are
// exact unions, so it misses that node too.  from == to: start itself, as
// the only child.
template <int DIM, bool CLOSED, bool GROUPED, class Hit>
__device__ __forceinline__ void walk_union(const SearchArgs& s, const Queries<DIM, GROUPED>& Q, int from, long start,
                                           int to, Hit&& hit) {
  const int c = threadIdx.x & 7;
  const unsigned long long full = __ballot(true);
  // level l's first node and node count, in lane l
  const int lane = threadIdx.x & 63;
  const long my_offset = lane < 32 ? s.info.offset[lane & 31] : 0, my_count = lane < 32 ? s.info.count[lane & 31] : 0;
  auto at_level = [](long x, int l) {
    return (long)((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(x >> 32), l) << 32 |
                  (unsigned)__builtin_amdgcn_readlane((int)x, l));
  };
  // the boxes (and mesh ranges) of a node's children, child c in this lane
  struct Boxes {
    double lo[DIM], hi[DIM];
    int2 r;
  };
  auto load = [&](long at, Boxes& x) {
    const long b = (at + c) * 2 * DIM;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      x.lo[d] = s.boxes[b + d];
      x.hi[d] = s.boxes[b + DIM + d];
    }
    if (GROUPED) x.r = *reinterpret_cast<const int2*>(s.granges + 2 * (at + c));
  };
  unsigned long long m[kGroups];
  auto test = [&](const Boxes& x, long n) {  // the first n children
    const unsigned long long in = __ballot(c < n);
#pragma unroll
    for (int i = 0; i < kGroups; i++) {
      // in a batch, only nodes whose mesh range holds A's mesh are visited
      const unsigned long long meshes = GROUPED ? in & __ballot(x.r.x <= Q.g[i] && Q.g[i] <= x.r.y) : in;
      m[i] = overlap_lanes<DIM, CLOSED>(meshes, full, x.lo, x.hi, Q.lo[i], Q.hi[i]);
    }
  };
  Boxes x, y;
  load(at_level(my_offset, from) + start, x);
  test(x, 1);
  if (any_query(m) == 0) return;
  if (from == to) {
    hit(start, m);
    return;
  }
  const long to_offset = at_level(my_offset, to), to_count = at_level(my_count, to);
  if (from == to + 1) {
    load(to_offset + start * kFanout, x);
    test(x, to_count - start * kFanout);
    hit(start * kFanout, m);
    return;
  }
  // levels to + 2 .. from, a byte each (1..8 and 9..16): the children to visit
  unsigned long long ulo = 0, uhi = 0;
  int L = from;
  long node = start;
  while (true) {
    const long first = node * kFanout;
    load(at_level(my_offset, L - 1) + first, x);
    test(x, at_level(my_count, L - 1) - first);
    unsigned u = any_query(m);
    if (L - 1 == to + 1) {
      // the children's children are what is asked for: two nodes' boxes on
      // their way at a time
      while (u) {
        const int k = __builtin_ctz(u);
        u &= u - 1;
        const int k2 = u ? __builtin_ctz(u) : k;
        u &= u - 1u;
        const long f = (first + k) * kFanout, f2 = (first + k2) * kFanout;
        load(to_offset + f, x);
        load(to_offset + f2, y);
        test(x, to_count - f);
        hit(f, m);
        if (k2 == k) break;
        test(y, to_count - f2);
        hit(f2, m);
      }
    } else if (L <= 8) {
      ulo |= (unsigned long long)u << (8 * (L - 1));
    } else {
      uhi |= (unsigned long long)u << (8 * (L - 9));
    }
    // the next node: a child of this one, or of the nearest with one left
    while (true) {
      u = L - 1 == to + 1 ? 0u
                          : (L <= 8 ? (unsigned)(ulo >> (8 * (L - 1))) : (unsigned)(uhi >> (8 * (L - 9)))) & 0xffu;
      if (u || L == from) break;
      node /= kFanout;
      L++;
    }
    if (u == 0) break;
    const int k = __builtin_ctz(u);
    if (L <= 8) ulo &= ~(1ULL << (8 * (L - 1) + k));
    else uhi &= ~(1ULL << (8 * (L - 9) + k));
    node = node * kFanout + k;
    L--;
  }
}

// The wave's index in the grid, as a scalar.
__device__ __forceinline__ long grid_wave() {
  return (long)blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// Splits long walks: for every query wave, the nodes at `level` that its
// queries overlap, one task each.  A wave's tasks are consecutive and in node
// order; first[w] and count[w] say which.
template <int DIM, bool CLOSED, bool GROUPED>
__global__ void __launch_bounds__(kBlock)
k_search_tasks(SearchArgs s, int2* __restrict__ tasks, unsigned long long* __restrict__ ntasks,
               uint2* __restrict__ span) {
  const long w = grid_wave();
  if (w * kQueries >= s.na) return;
  const Queries<DIM, GROUPED> Q(s, w);
  const int top = s.info.levels - 1, lane = threadIdx.x & 63;
  unsigned n = 0;
  walk_union<DIM, CLOSED, GROUPED>(s, Q, top, 0, s.level, [&](long, const unsigned long long* m) {
    n += __builtin_popcount(any_query(m));
  });
  // the first task's place: one beyond the arrays is not written, and all of a
  // total beyond them is unused (the host sees it and calls again with room),
  // so that the places below need no more than 32 bits
  unsigned at = 0;
  if (lane == 0) {
    const unsigned long long first = n ? atomicAdd(ntasks, (unsigned long long)n) : 0;
    at = first < s.cap ? (unsigned)first : s.cap;
    span[w] = make_uint2(at, n);
  }
  at = (unsigned)__builtin_amdgcn_readfirstlane((int)at);
  if (n > s.cap - at) return;
  walk_union<DIM, CLOSED, GROUPED>(s, Q, top, 0, s.level, [&](long first, const unsigned long long* m) {
    const unsigned u = any_query(m);
    if (lane < kFanout && ((u >> lane) & 1u))
      tasks[at + __builtin_popcount(u & ((1u << lane) - 1u))] = make_int2((int)w, (int)first + lane);
    at += __builtin_popcount(u);
  });
}

// The search below every task's node (or the root): counts the results per
// query, or writes them at their places in the CSR arrays.  Two walks instead
// of one into a scratch of fixed row length: a walk is cheaper than writing
// and reading the results once more, and rows of any length take the same
// path.
template <int DIM, bool CLOSED, bool GROUPED, bool FILL>
__global__ void __launch_bounds__(kBlock) k_search(SearchArgs s) {
  const int lane = threadIdx.x & 63, q8 = lane & 56, c = lane & 7;
  const long total = s.tasks ? (long)*s.ntasks : (s.na + kQueries - 1) / kQueries;
  if (s.tasks && total > (long)s.cap) return;
  for (long t = grid_wave(); t < total; t += (long)gridDim.x * (kBlock / 64)) {
    long w = t, node = 0;
    int from = s.info.levels - 1;
    if (s.tasks) {
      const int2 task = s.tasks[t];
      w = __builtin_amdgcn_readfirstlane(task.x);
      node = __builtin_amdgcn_readfirstlane(task.y);
      from = s.level;
    }
    const Queries<DIM, GROUPED> Q(s, w);
    if (FILL) {
      long at[kGroups];
#pragma unroll
      for (int i = 0; i < kGroups; i++) {
        at[i] = Q.a[i] >= 0 ? s.indptr[Q.a[i]] : 0;
        if (s.tasks) at[i] += s.tcount[t * kQueries + 8 * i + (lane >> 3)];
      }
      walk_union<DIM, CLOSED, GROUPED>(s, Q, from, node, 0, [&](long first, const unsigned long long* m) {
        const int b = first + c < s.info.count[0] ? s.perm[first + c] : 0;
#pragma unroll
        for (int i = 0; i < kGroups; i++) {
          if (m[i] == 0) continue;
          const unsigned mine = (unsigned)(m[i] >> q8) & 0xffu;  // this lane's query's results among the children
          if ((mine >> c) & 1u) {
            const long o = at[i] + __builtin_popcount(mine & ((1u << c) - 1u));
            s.indices[o] = b;
            s.rows[o] = Q.a[i];
          }
          at[i] += __builtin_popcount(mine);
        }
      });
    } else {
      int n[kGroups];
#pragma unroll
      for (int i = 0; i < kGroups; i++) n[i] = 0;
      walk_union<DIM, CLOSED, GROUPED>(s, Q, from, node, 0, [&](long, const unsigned long long* m) {
#pragma unroll
        for (int i = 0; i < kGroups; i++) n[i] += __builtin_amdgcn_inverse_ballot_w64(m[i]) ? 1 : 0;
      });
#pragma unroll
      for (int i = 0; i < kGroups; i++) {
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) n[i] += __shfl_xor(n[i], o, 64);
        if (c == 0) {
          if (s.tasks) s.tcount[t * kQueries + 8 * i + (lane >> 3)] = n[i];
          else if (Q.a[i] >= 0) s.row_count[Q.a[i]] = n[i];
        }
        if (!s.tasks) raise_max(s.maxrow, n[i]);
      }
    }
  }
}

// Row lengths from the tasks' counts, which become each task's offset in its
// queries' rows.  A lane per query.
__global__ void __launch_bounds__(kBlock) k_task_rows(SearchArgs s, const uint2* __restrict__ span) {
  const long t = (long)blockIdx.x * kBlock + threadIdx.x;
  if (*s.ntasks > (unsigned long long)s.cap) return;
  long run = 0;
  if (t < s.na) {
    const uint2 sp = span[t / kQueries];
    int* c = s.tcount + (long)sp.x * kQueries + t % kQueries;
    for (unsigned k = 0; k < sp.y; k += 8) {  // eight loads in flight
      int n[8];
#pragma unroll
      for (unsigned j = 0; j < 8; j++) n[j] = k + j < sp.y ? c[(long)(k + j) * kQueries] : 0;
#pragma unroll
      for (unsigned j = 0; j < 8; j++) {
        if (k + j < sp.y) c[(long)(k + j) * kQueries] = (int)run;
        run += n[j];
      }
    }
    s.row_count[s.qperm[t]] = run;
  }
  raise_max(s.maxrow, (int)run);
}

// Sorts each row of at most 256 entries by B id, a wave per row: an entry's
// place is the number of smaller ones (ids are distinct), counted against
// every entry in turn.
__global__ void __launch_bounds__(kBlock)
k_sort_rows(long na, const long* __restrict__ indptr, int* __restrict__ indices) {
  const int lane = threadIdx.x & 63;
  for (long a = grid_wave(); a < na; a += (long)gridDim.x * (kBlock / 64)) {
    const long o = indptr[a];
    const int n = (int)(indptr[a + 1] - o);
    if (n < 2) continue;
    int v[4], place[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = 64 * k + lane < n ? indices[o + 64 * k + lane] : 0x7fffffff;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (64 * k >= n) break;
      const int m = n - 64 * k < 64 ? n - 64 * k : 64;
      for (int j = 0; j < m; j++) {
        const int x = __builtin_amdgcn_readlane(v[k], j);
#pragma unroll
        for (int i = 0; i < 4; i++) place[i] += x < v[i] ? 1 : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (64 * k + lane < n) indices[o + place[k]] = v[k];
  }
}

// The words that the host waits for, in its own memory: [0] the pairs, [1]
// the longest row, [2] the tasks, [3] the staging flag.
__device__ __forceinline__ void publish(long npairs, const long* maxrow, const unsigned long long* ntasks, const int* bad,
                                        long* host) {
  host[0] = npairs;
  host[1] = *maxrow;
  host[2] = ntasks ? (long)*ntasks : 0L;
  host[3] = *bad;
}

__global__ void k_publish(long na, long* __restrict__ indptr, const long* __restrict__ maxrow,
                          const unsigned long long* __restrict__ ntasks, const int* __restrict__ bad,
            long* __restrict__ host) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  indptr[0] = 0;
  publish(indptr[na], maxrow, ntasks, bad, host);
}

// Row offsets of up to kScanMax rows, and the host's words, in one launch of
// one block (three launches with the library's scan).
constexpr int kScanBlock = 1024;
constexpr int kScanItems = 16;
constexpr long kScanMax = (long)kScanBlock * kScanItems;
__global__ void __launch_bounds__(kScanBlock)
k_scan_rows(int na, const long* __restrict__ row_count, long* __restrict__ indptr, const long* __restrict__ maxrow,
            const unsigned long long* __restrict__ ntasks, const int* __restrict__ bad,
            long* __restrict__ host) {
  __shared__ long wsum[kScanBlock / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int items = (na + kScanBlock - 1) / kScanBlock;
  long n[kScanItems], run = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    if (i >= items) break;
    const int k = t * items + i;
    n[i] = k < na ? row_count[k] : 0;
    run += n[i];
  }
  long sum = run;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const long x = __shfl_up(sum, o, 64);
    if (lane >= o) sum += x;
  }
  if (lane == 63) wsum[wave] = sum;
  __syncthreads();
  for (int w = 0; w < wave; w++) sum += wsum[w];
  sum -= run;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    if (i >= items) break;
    const int k = t * items + i;
    if (k >= na) break;
    if (k == 0) indptr[0] = 0;
    sum += n[i];
    indptr[k + 1] = sum;
    if (k == na - 1) publish(sum, maxrow, ntasks, bad, host);
  }
}

// Level of the hierarchy at which walks are cut into tasks, levels - 1 for
// none.  A wave walks its part of the tree by itself, a few microseconds per
// node on an idle card, so a search of few query waves is cut at nodes of 64
// elements.  With more waves the walks hide each other, and the two launches and
// the larger union are only a loss where rows are of like length.  Meshes against
// others of like size, us cut and uncut: triangles, 64 waves 86 and 93, 256 105
// and 113, 576 150 and 151, 1024 167 and 154, 2025 226 and 184, 4096 296 and 197;
// tets, 96 waves 99 and 140, 250 129 and 197, 515 197 and 244, 922 230 and 248,
// 1500 328 and 316, 1997 461 and 322, 6144 943 and 503.  Where one row is long the
// cut is what bounds it, which nothing tells beforehand: a triangle over all of
// 39 000 in 1225 waves 0.35 ms cut and 3.4 uncut, over 58 000 in 1806 0.47 and
// 5.1.  Up to 2048 waves that outweighs what even rows lose.  In a batch, where a
// mesh of a few elements may face one of tens of thousands, always at 512 elements
// (192 uneven mesh pairs: 6.5 ms, 10.8 uncut).  A hierarchy of at most 64 elements
// is walked in less time than the launches that cut it take.
static int task_level(const LevelInfo& info, long waves, bool grouped) {
  const int top = info.levels - 1;
  if (top <= 2) return top;
  return std::min(top, grouped ? 3 : (waves >= 2048 ? top : 2));
}

long find_pairs(Context& C, const DevMesh& A, const DevMesh& B, int finder, int sort_rows, bool ordered) {
  long na = A.nelements;
  long* row_count = C.row_count.as<long>(na + 1);
  long* indptr = C.indptr.as<long>(na + 1);
  volatile long* host = C.hstat + 8;
  if (na == 0 || B.nelements == 0) {
    host[3] = 0;
    LSM_HIP(hipMemsetAsync(indptr, 0, sizeof(long) * (na + 1), C.stream));
    LSM_HIP(hipMemcpyAsync(C.hstat + 11, stage_flag(C), sizeof(int), hipMemcpyDeviceToHost, C.stream));
    LSM_HIP(hipStreamSynchronize(C.stream));
    return 0;
  }
  LSM_REQUIRE(A.dim == B.dim, LIBSUPERMESH_GPU_ERROR_INVALID, "Invalid dimension: meshes differ");
  const DevBVH& H = C.bvh;
  if (!ordered) {
    const DevMesh* mesh = &A;
    DevBuf* order = &C.qperm;
    morton_order(C, 1, &mesh, &order, nullptr);
  }
  LSM_REQUIRE((A.ngroups > 0) == H.grouped && (!H.grouped || A.ngroups == B.ngroups),
              LIBSUPERMESH_GPU_ERROR_INVALID, "batches of A and B hold different mesh counts");
  LSM_REQUIRE(H.levels <= 17, LIBSUPERMESH_GPU_ERROR_OVERFLOW, "hierarchy too deep");
  const bool closed = finder == LIBSUPERMESH_GPU_FINDER_RTREE;
  const long waves = (na + kQueries - 1) / kQueries;
  SearchArgs s = {};
  s.na = na;
  s.qperm = static_cast<const int*>(C.qperm.ptr);
  s.abox = static_cast<const double*>(A.bbox.ptr);
  s.agroup = H.grouped ? static_cast<const int*>(A.group.ptr) : nullptr;
  s.granges = H.grouped ? static_cast<const int*>(H.granges.ptr) : nullptr;
  s.boxes = static_cast<const double*>(H.boxes.ptr);
  s.perm = static_cast<const int*>(H.perm.ptr);
  s.info = level_info(H);
  s.row_count = row_count;
  s.indptr = indptr;
  s.level = task_level(s.info, waves, H.grouped);
  const bool split = s.level < H.levels - 1;
  const dim3 block(kBlock), wave_grid(grid_for(waves, kBlock / 64));
#define LSM_SEARCH(K, ...)                                                                    \
  do {                                                                                        \
    if (A.dim == 2) {                                                                         \
      if (closed) {                                                                           \
        if (H.grouped) hipLaunchKernelGGL((K(2, true, true)), grid, block, 0, C.stream, __VA_ARGS__);   \
        else hipLaunchKernelGGL((K(2, true, false)), grid, block, 0, C.stream, __VA_ARGS__);  \
      } else {                                                                                \
        if (H.grouped) hipLaunchKernelGGL((K(2, false, true)), grid, block, 0, C.stream, __VA_ARGS__);  \
        else hipLaunchKernelGGL((K(2, false, false)), grid, block, 0, C.stream, __VA_ARGS__); \
      }                                                                                       \
    } else {                                                                                  \
      if (closed) {                                                                           \
        if (H.grouped) hipLaunchKernelGGL((K(3, true, true)), grid, block, 0, C.stream, __VA_ARGS__);   \
        else hipLaunchKernelGGL((K(3, true, false)), grid, block, 0, C.stream, __VA_ARGS__);  \
      } else {                                                                                \
        if (H.grouped) hipLaunchKernelGGL((K(3, false, true)), grid, block, 0, C.stream, __VA_ARGS__);  \
        else hipLaunchKernelGGL((K(3, false, false)), grid, block, 0, C.stream, __VA_ARGS__); \
      }                                                                                       \
    }                                                                                         \
    LSM_HIP(hipGetLastError());                                                               \
  } while (0)
#define LSM_TASKS(D, CL, G) k_search_tasks<D, CL, G>
#define LSM_COUNT(D, CL, G) k_search<D, CL, G, false>
#define LSM_FILL(D, CL, G) k_search<D, CL, G, true>
  long* words = search_words(C);  // cleared by the order's first kernel
  s.maxrow = words;
  dim3 grid = wave_grid;
  long room = 16 * waves + 16384;
  while (true) {
    if (split) {
      s.cap = (unsigned)room;
      int2* tasks = C.ftasks.as<int2>(room);
      uint2* span = C.fspan.as<uint2>(waves);
      s.tcount = C.fcount.as<int>((size_t)room * kQueries);
      unsigned long long* ntasks = reinterpret_cast<unsigned long long*>(words + 1);
      s.tasks = nullptr;
      grid = wave_grid;
      LSM_SEARCH(LSM_TASKS, s, tasks, ntasks, span);
      s.tasks = tasks;
      s.ntasks = ntasks;
      grid = dim3(std::min<unsigned>(grid_for(room, kBlock / 64), 8192));
      LSM_SEARCH(LSM_COUNT, s);
      hipLaunchKernelGGL(k_task_rows, dim3(grid_for(na, kBlock)), block, 0, C.stream, s, span);
    } else {
      LSM_SEARCH(LSM_COUNT, s);
    }
    const unsigned long long* ntasks = split ? s.ntasks : nullptr;
    if (na <= kScanMax) {
      hipLaunchKernelGGL(k_scan_rows, dim3(1), dim3(kScanBlock), 0, C.stream, (int)na, row_count, indptr, s.maxrow, ntasks,
                         stage_flag(C), C.hstat + 8);
    } else {
      size_t tmp_bytes = 0;
      LSM_HIP(rocprim::inclusive_scan(nullptr, tmp_bytes, row_count, indptr + 1, (size_t)na,
                                      rocprim::plus<long>(), C.stream));
      void* tmp = C.scan_tmp.get(tmp_bytes);
      LSM_HIP(rocprim::inclusive_scan(tmp, tmp_bytes, row_count, indptr + 1, (size_t)na,
                                      rocprim::plus<long>(), C.stream));
      hipLaunchKernelGGL(k_publish, dim3(1), dim3(64), 0, C.stream, na, indptr, s.maxrow, ntasks, stage_flag(C),
                         C.hstat + 8);
    }
    LSM_HIP(hipGetLastError());
    LSM_HIP(hipStreamSynchronize(C.stream));
    if (!split || host[2] <= room) break;
    LSM_REQUIRE(host[2] < (1L << 31), LIBSUPERMESH_GPU_ERROR_OVERFLOW, "too many search tasks");
    room = host[2] + host[2] / 8;
    hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(64), 0, C.stream, 2, words);
  }
  const long npairs = host[0], maxrow = host[1];
  LSM_REQUIRE(npairs < (1L << 40), LIBSUPERMESH_GPU_ERROR_OVERFLOW, "too many candidate pairs");
  s.indices = C.indices.as<int>(npairs);
  s.rows = C.rows.as<int>(npairs);
  if (npairs > 0) {
    LSM_SEARCH(LSM_FILL, s);
    if (sort_rows) {
      if (maxrow <= 256) {
        hipLaunchKernelGGL(k_sort_rows, dim3(std::min<unsigned>(grid_for(na, kBlock / 64), 65536)), block, 0, C.stream,
                           na, indptr, s.indices);
      } else {
        // long rows (a coarse A element over a fine B mesh): segmented radix
        // sort of the rows, then the sorted copy becomes the indices buffer
        LSM_REQUIRE(npairs < (1L << 32) && na < (1L << 32), LIBSUPERMESH_GPU_ERROR_OVERFLOW,
                    "too many pairs to sort rows");
        int* sorted = C.vals_alt.as<int>(npairs);
        unsigned end_bit = 1;
        while (end_bit < 31 && (1L << end_bit) < B.nelements) end_bit++;
        size_t bytes = 0;
        LSM_HIP(rocprim::segmented_radix_sort_keys(nullptr, bytes, s.indices, sorted, (unsigned)npairs, (unsigned)na,
                                                   indptr, indptr + 1, 0u, end_bit, C.stream));
        void* t3 = C.sort_tmp.get(bytes);
        LSM_HIP(rocprim::segmented_radix_sort_keys(t3, bytes, s.indices, sorted, (unsigned)npairs, (unsigned)na,
                                                   indptr, indptr + 1, 0u, end_bit, C.stream));
        std::swap(C.indices, C.vals_alt);
      }
      LSM_HIP(hipGetLastError());
    }
  }
#undef LSM_SEARCH
#undef LSM_TASKS
#undef LSM_COUNT
#undef LSM_FILL
  return npairs;
}

// indptr over A from the pairs sorted by A id (arow): indptr[r] = the first
// position of row r, indptr[na] = n
__global__ void __launch_bounds__(kBlock)
k_rows_to_indptr(long n, const unsigned* __restrict__ arow, long na, long* __restrict__ indptr) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  const long lo = i == 0 ? 0 : (long)arow[i - 1] + 1;
  const long hi = i == n ? na : (long)arow[i];
  for (long r = lo; r <= hi; r++) indptr[r] = i;
}

long find_pairs_from_b(Context& C, const DevMesh& A, const DevMesh& B, int finder) {
  // B's elements query the hierarchy over A (built by the caller): a CSR over
  // B, in B id order, whose entries are A ids.  The overlap tests are
  // symmetric in the two boxes, so the pair set is the one A's queries find.
  const long npairs = find_pairs(C, B, A, finder, 0, true);
  const long na = A.nelements;
  long* indptr = C.indptr.as<long>(na + 1);
  if (npairs == 0) {
    LSM_HIP(hipMemsetAsync(indptr, 0, sizeof(long) * (na + 1), C.stream));
    return 0;
  }
  LSM_REQUIRE(npairs < (1L << 32), LIBSUPERMESH_GPU_ERROR_OVERFLOW, "too many candidate pairs to regroup");
  unsigned* a_sorted = C.keys_alt.as<unsigned>(npairs);
  int* b_sorted = C.vals_alt.as<int>(npairs);
  const unsigned* a_ids = static_cast<const unsigned*>(C.indices.ptr);
  const int* b_ids = static_cast<const int*>(C.rows.ptr);
  // regrouped by A id with a stable sort: each A row keeps the B id order of
  // the input, ascending
  unsigned end_bit = 1;
  while (end_bit < 31 && (1L << end_bit) < na) end_bit++;
  size_t bytes = 0;
  LSM_HIP(rocprim::radix_sort_pairs(nullptr, bytes, a_ids, a_sorted, b_ids, b_sorted, (size_t)npairs, 0u, end_bit,
                                    C.stream));
  void* tmp = C.sort_tmp.get(bytes);
  LSM_HIP(rocprim::radix_sort_pairs(tmp, bytes, a_ids, a_sorted, b_ids, b_sorted, (size_t)npairs, 0u, end_bit,
                                    C.stream));
  hipLaunchKernelGGL(k_rows_to_indptr, dim3(grid_for(npairs + 1, kBlock)), dim3(kBlock), 0, C.stream, npairs,
                     a_sorted, na, indptr);
  LSM_HIP(hipGetLastError());
  std::swap(C.rows, C.keys_alt);     // the A id of each pair
  std::swap(C.indices, C.vals_alt);  // its B id, ascending within each row
  return npairs;
}

}  // namespace lsm
