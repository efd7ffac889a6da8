// supermesh.hip -- clipping kernels, reductions and P1 x P1 mixed mass.
//
// One candidate pair per lane.  The kernels read element vertex coordinates
// from the element-major arrays staged by finder.hip (48 B per triangle,
// 96 B per tet) and, for tets, B's four planes precomputed once per element
// (get_planes_tet is a pure function of the element, so this is bitwise the
// same as recomputing it per pair).  Per-pair counts and measures are
// bit-identical to the reference's intersect_tris / intersect_tets followed
// by a plain in-order sum of triangle_area / tetrahedron_volume; the global
// sum uses double-double (TwoSum) accumulation in a fixed reduction tree, so
// it is deterministic for a given input.
#include <algorithm>
#include <cstring>


#include "/root/repo/libsupermesh_amd/csrc/lsm_geometry.hpp"
#include "/root/repo/libsupermesh_amd/csrc/lsm_runtime.hpp"

#include "/root/repo/libsupermesh_amd/csrc/tet_quad.hpp"

namespace lsm {

constexpr int kClipBlock = 256;
constexpr int kClipGrid = 2048;  // fixed: the reduction tree depends only on npairs
// The tet triage's blocks: each compacts one contiguous chunk of the pairs
constexpr int kTriageGrid = 16384;

struct Partial {
  double hi, lo;
  long long nonempty, nout;
  long long maxc, pad;
};

__device__ __forceinline__ void two_sum(double a, double b, double& s, double& e) {
  s = a + b;
  double bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

__device__ __forceinline__ void dd_add(double& hi, double& lo, double x) {
  double s, e;
  two_sum(hi, x, s, e);
  hi = s;
  lo = lo + e;
}

__device__ __forceinline__ void dd_merge(double& hi, double& lo, double hi2, double lo2) {
  double s, e;
  two_sum(hi, hi2, s, e);
  hi = s;
  lo = lo + (e + lo2);
}

// Quadrature rules of the reference's mixed-mass tests: Dunavant degree 2 on
// triangles (barycentric (4,1,1)/6, weights 1/3; test_parallel_p1_inner_product_2d.F90:59-68)
// and the 4-point Stroud rule on tets (..._3d.F90:61-80).
__constant__ double kQ2[3][3] = {{4.0 / 6.0, 1.0 / 6.0, 1.0 / 6.0},
                                 {1.0 / 6.0, 4.0 / 6.0, 1.0 / 6.0},
                                 {1.0 / 6.0, 1.0 / 6.0, 4.0 / 6.0}};
#define LSM_QA 5.8541019662496852e-1
#define LSM_QB 1.3819660112501050e-1
__constant__ double kQ3[4][4] = {{LSM_QA, LSM_QB, LSM_QB, LSM_QB},
                                 {LSM_QB, LSM_QA, LSM_QB, LSM_QB},
                                 {LSM_QB, LSM_QB, LSM_QA, LSM_QB},
                                 {LSM_QB, LSM_QB, LSM_QB, LSM_QA}};

template <int DIM>
__device__ __forceinline__ void basis(const double* __restrict__ aff, const double* x, double* f) {
  if constexpr (DIM == 2) {
    double dx = x[0] - aff[0], dy = x[1] - aff[1];
    double f2 = aff[2] * dx;
    f2 = f2 + aff[3] * dy;
    double f3 = aff[4] * dx;
    f3 = f3 + aff[5] * dy;
    f[1] = f2;
    f[2] = f3;
    f[0] = 1.0 - f2 - f3;
  } else {
    double dx = x[0] - aff[0], dy = x[1] - aff[1], dz = x[2] - aff[2];
    double s = 0.0;
#pragma unroll
    for (int r = 0; r < 3; r++) {
      double v = aff[3 + 3 * r] * dx;
      v = v + aff[4 + 3 * r] * dy;
      v = v + aff[5 + 3 * r] * dz;
      f[1 + r] = v;
    }
    s = 1.0 - f[1] - f[2] - f[3];
    f[0] = s;
  }
}

// Adds the element's contributions to blk[LOC][LOC].  2D: the product of two
// P1 functions is quadratic, so the 3-point rule of the reference tests
// (test_parallel_p1_inner_product_2d.F90:59-68) equals the closed form
// int_c f g = |c|/12 (sum_v f_v g_v + (sum_v f_v)(sum_v g_v)) over c's
// vertex values; this evaluates the latter (about half the operations; sums
// may use fused multiply-adds: the mass is compared within 1e-12, not
// bitwise).  3D: the reference's 4-point rule as written.
template <int DIM>
__device__ __forceinline__ void mass_element(const double* el, double meas, const double* affa,
                                             const double* affb, double* blk) {
  if constexpr (DIM == 2) {
    double fa[3][3], fb[3][3];  // [vertex][basis]
#pragma unroll
    for (int v = 0; v < 3; v++) {
      basis<2>(affa, el + 2 * v, fa[v]);
      basis<2>(affb, el + 2 * v, fb[v]);
    }
    const double w = meas * (1.0 / 12.0);
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const double sa = fa[0][i] + fa[1][i] + fa[2][i];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const double sb = fb[0][j] + fb[1][j] + fb[2][j];
        double d = __builtin_fma(fa[0][i], fb[0][j], sa * sb);
        d = __builtin_fma(fa[1][i], fb[1][j], d);
        d = __builtin_fma(fa[2][i], fb[2][j], d);
        blk[i * 3 + j] = __builtin_fma(w, d, blk[i * 3 + j]);
      }
    }
    return;
  }
  constexpr int LOC = DIM + 1;
  constexpr int NQ = DIM == 2 ? 3 : 4;
  const double wq = DIM == 2 ? 1.0 / 3.0 : 0.25;
  const double wm = wq * meas;
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    double x[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      double s = 0.0;
#pragma unroll
      for (int v = 0; v < LOC; v++) s = s + (DIM == 2 ? kQ2[q][v] : kQ3[q][v]) * el[v * DIM + d];
      x[d] = s;
    }
    double fa[LOC], fb[LOC];
    basis<DIM>(affa, x, fa);
    basis<DIM>(affb, x, fb);
#pragma unroll
    for (int i = 0; i < LOC; i++)
#pragma unroll
      for (int j = 0; j < LOC; j++) blk[i * LOC + j] = blk[i * LOC + j] + wm * fa[i] * fb[j];
  }
}

// 2D P1 x P1 mass of a clipped polygon from its moments, the polygon's fan
// triangles accumulated in coordinates d = x - o local to A's first vertex o:
// mom = {int 1, int dx, int dy, int dx^2, int dx dy, int dy^2}.  Per
// triangle (area ar, vertices d_0..d_2; exact for quadratics):
// int dx = ar/3 sum dx_v, int dx dy = ar/12 (sum dx_v dy_v + sum dx_v sum dy_v).
__device__ __forceinline__ void tri_moments(double x0, double y0, double x1, double y1, double x2, double y2,
                                            double ar, double ox, double oy, double* mom) {
  const double a0 = x0 - ox, b0 = y0 - oy, a1 = x1 - ox, b1 = y1 - oy, a2 = x2 - ox, b2 = y2 - oy;
  const double sa = a0 + a1 + a2, sb = b0 + b1 + b2;
  const double w3 = ar * (1.0 / 3.0), w12 = ar * (1.0 / 12.0);
  mom[0] += ar;
  mom[1] += w3 * sa;
  mom[2] += w3 * sb;
  mom[3] += w12 * (a0 * a0 + a1 * a1 + a2 * a2 + sa * sa);
  mom[4] += w12 * (a0 * b0 + a1 * b1 + a2 * b2 + sa * sb);
  mom[5] += w12 * (b0 * b0 + b1 * b1 + b2 * b2 + sb * sb);
}

// blk[i][j] = int phi^A_i phi^B_j over the polygon of moments mom (origin o =
// A's first vertex, where phi^A = (1, 0, 0)): with phi^A_i = alpha_i + g_i.d
// and phi^B_j = beta_j + h_j.d, the integral is alpha_i beta_j I + alpha_i
// h_j.Id + beta_j g_i.Id + g_i^T Idd h_j.  The same integral as summing
// mass_element<2> over the fan, in exact arithmetic.
__device__ __forceinline__ void mass_from_moments(const double* mom, const double* affa, const double* affb,
                                                  double* blk) {
  double g[3][2], h[3][2], beta[3];
  g[1][0] = affa[2];
  g[1][1] = affa[3];
  g[2][0] = affa[4];
  g[2][1] = affa[5];
  g[0][0] = -(g[1][0] + g[2][0]);
  g[0][1] = -(g[1][1] + g[2][1]);
  h[1][0] = affb[2];
  h[1][1] = affb[3];
  h[2][0] = affb[4];
  h[2][1] = affb[5];
  h[0][0] = -(h[1][0] + h[2][0]);
  h[0][1] = -(h[1][1] + h[2][1]);
  const double o[2] = {affa[0], affa[1]};
  basis<2>(affb, o, beta);
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const double hd = h[j][0] * mom[1] + h[j][1] * mom[2];            // h_j . Id
    const double tx = mom[3] * h[j][0] + mom[4] * h[j][1];            // Idd h_j
    const double ty = mom[4] * h[j][0] + mom[5] * h[j][1];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      double v = beta[j] * (g[i][0] * mom[1] + g[i][1] * mom[2]) + (g[i][0] * tx + g[i][1] * ty);
      if (i == 0) v += beta[j] * mom[0] + hd;  // alpha = (1, 0, 0)
      blk[i * 3 + j] = v;
    }
  }
}

struct ClipArgs {
  long npairs;
  const long* npairs_dev;  // when set, the pair count is read here (a recorded graph's count pass)
  const int* rows;
  const int* cols;
  const int* work;    // when non-null: process pairs work[0..nwork)
  const unsigned long long* nwork;
  const double* acoords;
  const double* bcoords;
  const double* asp;
  const double* bsp;
  const double* ascale;
  const double* bscale;
  const double* bplanes;
  const double* aaff;
  const double* baff;
  int* counts;
  double* measure;
  double* blocks;
  const long* offsets;
  double* elements;
  // single pass (predicted budget) clip: per work item budget; each pair's
  // run starts at offsets[p] (the budgets laid end to end)
  const unsigned* budget;  // packed budget levels; this call uses byte bshift / 8
  int bshift;
  // outputs beyond a budget continue in the walking lane's own arena region
  // (no atomics: a lane finishes one pair before the next), elements
  // [arena_base + lane * arena_per_lane, + arena_per_lane); aoff[w] = where
  // work item w's continue.  dropped[w]: 1 the run is split (budget, then
  // arena), 2 the lane's arena ran out (the pair is clipped again)
  long arena_base;
  long arena_per_lane;
  long* aoff;
  unsigned char* dropped;
  unsigned long long* ndropped;  // [0] split runs, [1] pairs clipped again
  // fill pass: when non-null, only items flagged 2 here, each written at
  // aoff[w] (its place in the spill reserve)
  const unsigned char* ovf;
  // tet walks: one work-item counter per XCD share (zeroed before each launch)
  unsigned long long* queue;
  // 2D: pairs whose working polygon outgrew its LDS slots, for the
  // streaming clipper
  int* olist;
  unsigned long long* nolist;
  // mass row slots (2D): the count pass also writes each pair's contributions
  // (B node, value) to the rows of A's nodes, at
  // rbase[a * LOC + li] + (p - indptr[a]) * LOC + j, j = 0..LOC-1 (B's local
  // nodes); an empty pair writes node -1 and no values.  Per-pair blocks
  // only when `blocks` is set.
  const long* rbase;
  const long* indptr;
  const int* enlb;
  int* rkey;
  double* rval;
};

// Output elements are written once and not read again by the pass that
// writes them: streaming (nontemporal) stores keep them from evicting the
// meshes' coordinates and planes that the clippers read from L2 (materialised
// tet 96^3 vs 90^3: the fill walk and the single pass each 6 ms faster).
__device__ __forceinline__ void stream_tri(double* o, double x0, double y0, double x1, double y1, double x2,
                                           double y2) {
  __builtin_nontemporal_store(x0, o);
  __builtin_nontemporal_store(y0, o + 1);
  __builtin_nontemporal_store(x1, o + 2);
  __builtin_nontemporal_store(y1, o + 3);
  __builtin_nontemporal_store(x2, o + 4);
  __builtin_nontemporal_store(y2, o + 5);
}

__device__ __forceinline__ void stream_tet(double* o, const double* t) {
#pragma unroll
  for (int i = 0; i < 12; i++)
o[i]=t[i];

}

// One 16-byte word of a run copy, stored the same way.
__device__ __forceinline__ void stream_word(double2* d, const double2* s) {
  using v2 = double __attribute__((ext_vector_type(2)));
  __builtin_nontemporal_store(*reinterpret_cast<const v2*>(s), reinterpret_cast<v2*>(d));
}

__device__ __forceinline__ long pair_count(const ClipArgs& g) { return g.npairs_dev ? *g.npairs_dev : g.npairs; }

constexpr int kWalkBlock = 128;

// The CDNA4 dispatcher hands consecutive workgroups to its 8 XCDs (each with
// its own L2) in turn: with a grid whose size is a multiple of 8, block b
// runs on XCD b % 8, which takes the share [x * per, (x + 1) * per) of the
// work list.
constexpr int kXcds = 8;

// The walks' waves take work items from queues (counters handing out chunks
// of consecutive items): each XCD's share of the work list is cut into
// kSubQueues contiguous parts, each with its own counter, so the items in
// flight on an XCD stay a few compact windows of the list whose A and B data
// its L2 holds, and no counter takes more than a fraction of the atomics.  A
// wave loads the pairs of a whole chunk at once, one item per lane, and deals
// them to its quads as they finish: the chain of dependent loads (counter,
// work list, pair) is paid once per chunk instead of once per item, and the
// quads of a wave work on neighbouring pairs.  A short list is handed out in
// chunks of a quarter of the items per wave, so that no wave holds work that
// another could do.
constexpr int kSubQueues = 4;
constexpr int kQueues = kXcds * kSubQueues;

struct QuadItems {
  unsigned long long* counter;
  long begin, end;         // this wave's part of the list
  int chunk;               // items per counter increment, at most 64
  int cnt = 0, used = 0;   // items of the current chunk, and how many are dealt
  bool dry = false;        // the part has no further chunk
  int p = 0, a = 0, b = 0, w = 0;  // this lane's item of the chunk: its pair, elements and list index

  __device__ __forceinline__ void init(unsigned long long* queues, long n) {
    const int nx = gridDim.x % kXcds == 0 ? kXcds : 1;
    // every part needs blocks to drain it: a grid with fewer blocks per share
    // than parts keeps one part per share
    const int nsub = (int)(gridDim.x / nx) >= kSubQueues ? kSubQueues : 1;
    const long xcd = blockIdx.x % nx, sub = (blockIdx.x / nx) % nsub;
    const long per = (n + nx - 1) / nx;
    const long b0 = xcd * per, e0 = b0 + per < n ? b0 + per : n;
    const long sper = (e0 - b0 + nsub - 1) / nsub;
    counter = queues + xcd * kSubQueues + sub;
    begin = b0 + sub * sper < e0 ? b0 + sub * sper : e0;
    end = begin + sper < e0 ? begin + sper : e0;
    const long share = n / (4 * (long)gridDim.x * (blockDim.x / 64));
    chunk = share < 1 ? 1 : (share < 64 ? (int)share : 64);
  }

  // The next chunk with an item to do: load(i, p, a, b) gives item i's pair
  // and elements, or false to pass over it.
  template <class Load>
  __device__ __forceinline__ void refill(Load&& load) {
    const int lane = threadIdx.x & 63;
    cnt = used = 0;
    while (cnt == 0 && !dry) {
      unsigned long long got = 0;
      if (lane == 0) got = atomicAdd(counter, (unsigned long long)chunk);
      const long base = begin + (long)((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(got >> 32)) << 32 |
                                       (unsigned)__builtin_amdgcn_readfirstlane((int)got));
      if (base >= end) {
        dry = true;
        break;
      }
      const int n = end - base < chunk ? (int)(end - base) : chunk;
      bool valid = false;
      if (lane < n) {
        w = (int)(base + lane);
        valid = load(base + lane, p, a, b);
      }
      const unsigned long long m = __ballot(valid);
      cnt = __popcll(m);
      if (cnt < n) {  // close the gaps: the k-th valid item to lane k, the others behind
        const int before = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        const int to = (valid ? before : cnt + lane - before) * 4;
        p = __builtin_amdgcn_ds_permute(to, p);
        a = __builtin_amdgcn_ds_permute(to, a);
        b = __builtin_amdgcn_ds_permute(to, b);
        w = __builtin_amdgcn_ds_permute(to, w);
      }
    }
  }

  // Deals an item to each quad that wants one (whole wave; want is the same
  // in a quad's lanes), as far as the chunk and the next one go; true in the
  // quads that got one.
  template <class Load>
  __device__ __forceinline__ bool take(bool want, int& ip, int& ia, int& ib, int& iw, Load&& load) {
    const unsigned long long m = __ballot(want);
    const int n = __popcll(m) >> 2;
    const int rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0)) >> 2;
    bool got = false;
    int before = 0;  // quads served from the chunk that ran out
    for (int pass = 0; pass < 2 && before < n; pass++) {
      if (used == cnt && !dry) refill(load);
      const int left = cnt - used, r = rank - before;
      const bool now = want && r >= 0 && r < left;
      const int src = now ? used + r : 0;
      const int xp = __shfl(p, src, 64), xa = __shfl(a, src, 64), xb = __shfl(b, src, 64), xw = __shfl(w, src, 64);
      ip = now ? xp : ip;
      ia = now ? xa : ia;
      ib = now ? xb : ib;
      iw = now ? xw : iw;
      got = got || now;
      const int served = n - before < left ? n - before : left;
      used += served;
      before += served;
      if (dry) break;
    }
    return got;
  }
};

__global__ void k_zero_queues(unsigned long long* __restrict__ q) {
  if (threadIdx.x < kQueues && blockIdx.x == 0) q[threadIdx.x] = 0;
}

struct TetMoments {
  double m[10];  // 1, x, y, z, xx, xy, xz, yy, yz, zz
  double o[3];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 10; i++) m[i] = 0.0;
  }
  __device__ __forceinline__ void add(const double* t, double vol) {
    double d[4][3], s[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
      for (int v = 0; v < 4; v++) d[v][k] = t[3 * v + k] - o[k];
      s[k] = (d[0][k] + d[1][k]) + (d[2][k] + d[3][k]);
    }
    const double w4 = 0.25 * vol, w20 = 0.05 * vol;
    m[0] += vol;
#pragma unroll
    for (int k = 0; k < 3; k++) m[1 + k] = __builtin_fma(w4, s[k], m[1 + k]);
    int n = 4;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = i; j < 3; j++) {
        double x = s[i] * s[j];
#pragma unroll
        for (int v = 0; v < 4; v++) x = __builtin_fma(d[v][i], d[v][j], x);
        m[n] = __builtin_fma(w20, x, m[n]);
        n++;
      }
  }
  // Row q of the block: int phi^A_q phi^B_j, j = 0..3 (whole quad).
  __device__ __forceinline__ void row(int q, const double* __restrict__ affa, const double* __restrict__ affb,
                                      double* out) {
    double M[10];
#pragma unroll
    for (int i = 0; i < 10; i++) M[i] = quad_sum(m[i]);
    double fa[4], fb[4], ga[3], alpha;
    basis<3>(affa, o, fa);
    basis<3>(affb, o, fb);
    alpha = q == 0 ? fa[0] : (q == 1 ? fa[1] : (q == 2 ? fa[2] : fa[3]));
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double g1 = affa[3 + k], g2 = affa[6 + k], g3 = affa[9 + k];
      ga[k] = q == 0 ? -((g1 + g2) + g3) : (q == 1 ? g1 : (q == 2 ? g2 : g3));
    }
    // int phi^A_q and int phi^A_q d
    const double i0 = alpha * M[0] + (ga[0] * M[1] + ga[1] * M[2] + ga[2] * M[3]);
    const double ix = alpha * M[1] + (ga[0] * M[4] + ga[1] * M[5] + ga[2] * M[6]);
    const double iy = alpha * M[2] + (ga[0] * M[5] + ga[1] * M[7] + ga[2] * M[8]);
    const double iz = alpha * M[3] + (ga[0] * M[6] + ga[1] * M[8] + ga[2] * M[9]);
    double rest = 0.0;
#pragma unroll
    for (int j = 1; j < 4; j++) {
      const double* h = affb + 3 * j;
      const double g = h[0] * ix + h[1] * iy + h[2] * iz;
      out[j] = fb[j] * i0 + g;
      rest += g;
    }
    out[0] = fb[0] * i0 - rest;
  }
};

// MODES: count (FILL and LEARNED false): counts, measures (and mass blocks);
// fill (FILL): writes each pair's counts[p] outputs at offsets[p];
// single pass (LEARNED): the count pass that also writes up to budget[w]
// outputs of work item w at offsets[p] and the rest to the quad's arena.
// BLOCK is a launch shape the count pass can be tuned over.
template <bool MASS, bool FILL, bool LEARNED = false, int BLOCK = kWalkBlock>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(3)))
k_clip_tet_walk(ClipArgs g) {
  __shared__ QuadLds<4> lds[BLOCK / 64];
  __shared__ uint4 table[256];
  for (int i = threadIdx.x; i < 256; i += BLOCK) table[i] = reinterpret_cast<const uint4*>(kSplitTable.e)[i];
  __syncthreads();
  QuadClip<4> W;
  W.init(&lds[threadIdx.x >> 6], table);
  const int q = W.q;
  // blocks go to the XCDs round robin: each XCD takes one contiguous share
  // of the work list, so that its L2 holds one region of A and B
  const long nwork = (long)*g.nwork;
  QuadItems Q;
  Q.init(g.queue, nwork);
  auto load = [&](long i, int& p, int& a, int& b) {
    p = g.work[i];
    a = g.rows[p];
    b = g.cols[p];
    // fill pass: pairs with output, or only those to be clipped again
    return !FILL || (g.counts[p] > 0 && (!g.ovf || g.ovf[i] == 2));
  };
  // The quad's next item, its vertex and plane already on their way: loaded
  // when the one before is begun, so that no quad waits for memory between
  // items (tet 64^3 vs 60^3 count: 13.1 -> 10.2 ms).  The passes that write
  // tets load an item when they begin it: loads and stores complete in order,
  // so a load begun earlier would wait for the stores in between (fill of tet
  // 32^3 vs 29^3: 4.4 ms instead of 2.1).  A list with few items per quad is
  // not dealt ahead.
#ifdef LSM_AH
 constexpr bool AHEAD=true;
#else
  constexpr bool AHEAD = !FILL && !LEARNED;
#endif
  const bool ahead = AHEAD && nwork >= 8L * gridDim.x * (BLOCK / 4);
  bool has_next = false;
  int np = 0, na = 0, nb = 0, nw = 0, ncap = 0;
  long noff = 0;
  double nv[3] = {0.0, 0.0, 0.0}, nP[4] = {0.0, 0.0, 0.0, 0.0}, nsa = 0.0, nsb = 0.0;
  bool active = false;
  long off = 0;
  int p = 0, a = 0, b = 0, w = 0;
  int cap = 0, k = 0;
  // single pass: this quad's arena region, its fill level, and whether the
  // current pair's output outgrew budget and arena
  const long abase =
      LEARNED ? g.arena_base + (((long)blockIdx.x * BLOCK + threadIdx.x) >> 2) * g.arena_per_lane : 0;
  long atop = 0;
  bool lost = false;
  unsigned nsplit = 0, nlost = 0;  // this quad's split runs and pairs to clip again
  double tol = 0.0, m = 0.0;
  TetMoments mom;
  auto start = [&]() {
    p = np;
    a = na;
    b = nb;
    w = nw;
    cap = ncap;
    off = noff;
    tol = 10.0 * fmin_f(nsa, nsb);
    m = 0.0;
    k = 0;
    lost = false;
    if (MASS) mom.clear();
    W.set_plane(q, nP);
    W.begin(nv);
    active = true;
    has_next = false;
  };
  while (true) {
    const bool idle = W.done();
    if (idle && active) {  // the pair is done
      if (LEARNED) {
        const bool any_lost = quad_or(lost ? 1u : 0u) != 0;
        const bool split = k > cap && !any_lost;
        if (q == 0) {
          g.aoff[w] = split ? abase + atop : -1;
          g.dropped[w] = any_lost ? 2 : (split ? 1 : 0);
        }
        if (split) atop += k - cap;
        nsplit += split ? 1u : 0u;
        nlost += any_lost ? 1u : 0u;
      }
      if (!FILL) {
        if (q == 0) {
          g.counts[p] = k;
          g.measure[p] = k == 0 ? 0.0 : m;
        }
        if (MASS) {
          double row[4] = {0.0, 0.0, 0.0, 0.0};
          if (k > 0) mom.row(q, g.aaff + (long)a * 12, g.baff + (long)b * 12, row);
#pragma unroll
          for (int j = 0; j < 4; j++) g.blocks[(long)p * 16 + 4 * q + j] = row[j];
        }
      }
      active = false;
    }
    if (AHEAD && idle && has_next) start();
    const bool want = !has_next && (ahead || !active);
    if (__any(want) && !(Q.dry && Q.used == Q.cnt)) {
      const bool got = Q.take(want, np, na, nb, nw, load);
      if (got) {
        // lane q brings in B's plane q and A's vertex q
#pragma unroll
        for (int i = 0; i < 4; i++) nP[i] = g.bplanes[(long)nb * 16 + 4 * q + i];
#pragma unroll
        for (int i = 0; i < 3; i++) nv[i] = g.acoords[(long)na * 12 + 3 * q + i];
        nsa = g.asp[na];
        nsb = g.bsp[nb];
        if (FILL) {
          ncap = g.counts[np];
          noff = g.ovf ? g.aoff[nw] : g.offsets[np];
        }
        if (LEARNED) {
          ncap = (int)((g.budget[nw] >> g.bshift) & 0xffu);
          noff = g.offsets[np];
        }
        has_next = true;
        if (!AHEAD) start();
      }
    }
    if (!__any(active || has_next)) break;  // the list is dry
    if (!active) continue;
    if (!W.cur) W.pop();
    W.step([&](const double* t, uint32_t lead) {
      const bool keep = ((lead >> q) & 1u) && volume_reaches(t, tol);
      const double vr = keep ? tet_volume_real(t) : 0.0;
      // the reference's order; 0 for the others adds nothing
      m = m + quad_lane<0>(vr);
      m = m + quad_lane<1>(vr);
      m = m + quad_lane<2>(vr);
      const uint32_t kept = quad_or((keep ? 1u : 0u) << q);
      if (MASS) {
        // the origin: the first output's first vertex
        const uint32_t first = lead & -lead;
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const double x0 = quad_lane<0>(t[i]), x1 = quad_lane<1>(t[i]), x2 = quad_lane<2>(t[i]);
          const double x = first == 1u ? x0 : (first == 2u ? x1 : x2);
          mom.o[i] = k == 0 ? x : mom.o[i];
        }
        if (keep) mom.add(t, vr);
      }
      if (FILL || LEARNED) {
        const int at = k + __builtin_popcount(kept & ((1u << q) - 1u));
        if (keep && at < cap) {
          stream_tet(g.elements + (off + at) * 12, t);
        } else if (LEARNED && keep) {
          // beyond the budget: the run continues in this quad's arena
          const long e = atop + (at - cap);
          if (e < g.arena_per_lane) {
            stream_tet(g.elements + (abase + e) * 12, t);
          } else {
            lost = true;
          }
        }
      }
      k += __builtin_popcount(kept);
    });
  }
  if (LEARNED) {
    // one atomic per wave: one per pair on a single counter serialised the
    // single pass (tet 96^3 at budget level 0.9: 7.4 M of them, ~20 ms)
    unsigned long long s = q == 0 ? nsplit : 0u, l = q == 0 ? nlost : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      s += __shfl_xor(s, o, 64);
      l += __shfl_xor(l, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
      if (s) atomicAdd(g.ndropped, s);
      if (l) atomicAdd(g.ndropped + 1, l);
    }
  }
}


template __global__ void k_clip_tet_walk<false,false,false,128>(ClipArgs);
template __global__ void k_clip_tet_walk<false,true,false,128>(ClipArgs);
template __global__ void k_clip_tet_walk<true,false,false,128>(ClipArgs);
template __global__ void k_clip_tet_walk<false,false,true,128>(ClipArgs);}
