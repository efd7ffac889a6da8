// tet_quad.hpp -- the clip of a tetrahedron by NP planes on a quad (four
// consecutive lanes) per pair.
//
// Same tree of tets, same arithmetic and same output order as clip_tet
// (Tetrahedron_Intersection.F90:107-179, 244-436), arranged for a wave:
//
// * A tet is four vertex ids (a byte each) into a pool of vertices in LDS:
//   row 0 holds A's vertices, row r the (up to four) split points of the
//   path's r-th split.  A child is one byte permute of its parent's ids and
//   the new row's, so no coordinates are moved or selected in registers.
// * A vertex's side of every plane is found once, when the vertex is made, and
//   kept as two bits per plane in a code word that travels with the ids (the
//   same permute).  Which plane splits a tet next, or that it is wholly in or
//   out, is then a few integer operations, and tets that a plane keeps whole
//   or drops cost no step.
// * A step splits one tet: the quad's lanes make its four split points (one
//   division each) and its children in parallel, drop the dead children, take
//   the volumes of the children that are outputs already, and leave the rest
//   in a small stack in LDS (a bit per entry says which are pending).
//
// Measured on 222 736 pairs of jittered Kuhn grids (12^3 over 11^3): 4.7
// splits a pair against the 14.5 children that the walk of one lane builds.
#pragma once

#include "lsm_geometry.hpp"

namespace lsm {

// Side of a vertex against a plane: 0 within epsilon of it, 1 inside (d < 0),
// 2 outside (d > 0), 3 none of these (NaN), as the split's case counts them
// (Tetrahedron_Intersection.F90:264-276).
LSM_HD unsigned side_code(double d) {
  return (d > -kEpsilon ? 0u : 1u) | (d < kEpsilon ? 0u : 2u);
}

// How a tet whose vertices have these sides against the splitting plane is
// cut.  child[c]: byte permute (0..3 the parent's vertex, 4..7 a split point)
// giving child c's vertices in the reference's order; splits: byte s holds
// split point s's outside vertex times 8 in bits 3-4 and its inside vertex in
// bits 0-1, and byte 0's bits 5-6 the number of children.
struct alignas(16) SplitCase {
  uint32_t child[3];
  uint32_t splits;
};

constexpr SplitCase split_case(int code) {
  int pos[4] = {0, 0, 0, 0}, neg[4] = {0, 0, 0, 0}, z0 = 0, np = 0, nn = 0, nz = 0;
  for (int v = 0; v < 4; v++) {
    const int s = (code >> (2 * v)) & 3;
    if (s == 0) {
      if (nz == 0) z0 = v;
      nz++;
    }
    if (s == 1) neg[nn++] = v;
    if (s == 2) pos[np++] = v;
  }
  const int p0 = pos[0], p1 = pos[1], n0 = neg[0], n1 = neg[1], n2 = neg[2];
  int src[3][4] = {{0, 1, 2, 3}, {0, 1, 2, 3}, {0, 1, 2, 3}};
  int sp[4] = {0, 0, 0, 0}, sn[4] = {0, 0, 0, 0}, nch = 0, ns = 0;
  if (nn == 0) {
    nch = 0;
  } else if (np == 0) {
    nch = 1;
  } else if (np == 3 || (np == 2 && nn != 2) || (np == 1 && nn == 1)) {
    // +++-, ++-0, +-00: every outside vertex moves to the plane
    for (int i = 0; i < np; i++) {
      sp[i] = pos[i];
      sn[i] = n0;
      src[0][pos[i]] = 4 + i;
    }
    nch = 1;
    ns = np;
  } else if (np == 2) {
    // ++--: split points (p0,n0) (p1,n0) (p0,n1) (p1,n1)
    sp[0] = p0, sn[0] = n0, sp[1] = p1, sn[1] = n0, sp[2] = p0, sn[2] = n1, sp[3] = p1, sn[3] = n1;
    src[0][p0] = 6, src[0][p1] = 5;
    src[1][0] = n1, src[1][1] = 7, src[1][2] = 6, src[1][3] = 5;
    src[2][0] = n0, src[2][1] = 4, src[2][2] = 5, src[2][3] = 6;
    nch = 3;
    ns = 4;
  } else if (nn == 3) {
    // +---: (p0,n0) (p0,n1) (p0,n2)
    sp[0] = p0, sn[0] = n0, sp[1] = p0, sn[1] = n1, sp[2] = p0, sn[2] = n2;
    src[0][p0] = 4;
    src[1][0] = 4, src[1][1] = n1, src[1][2] = n2, src[1][3] = 5;
    src[2][0] = n2, src[2][1] = 5, src[2][2] = 6, src[2][3] = 4;
    nch = 3;
    ns = 3;
  } else {
    // +--0: (p0,n0) (p0,n1)
    sp[0] = p0, sn[0] = n0, sp[1] = p0, sn[1] = n1;
    src[0][p0] = 4;
    src[1][0] = 5, src[1][1] = z0, src[1][2] = n1, src[1][3] = 4;
    nch = 2;
    ns = 2;
  }
  (void)ns;
  SplitCase r = {{0, 0, 0}, 0};
  for (int c = 0; c < 3; c++)
    for (int j = 0; j < 4; j++) r.child[c] |= (uint32_t)src[c][j] << (8 * j);
  for (int s = 0; s < 4; s++) r.splits |= (uint32_t)((sp[s] << 3) | sn[s]) << (8 * s);
  r.splits |= (uint32_t)nch << 5;
  return r;
}

struct SplitTable {
  SplitCase e[256];  // by side_0 + 4 side_1 + 16 side_2 + 64 side_3
};

constexpr SplitTable make_split_table() {
  SplitTable t = {};
  for (int i = 0; i < 256; i++) t.e[i] = split_case(i);
  return t;
}

// Code words of a tet against NP planes: byte v of word w holds vertex v's
// sides of planes 4 w .. 4 w + 3, two bits each, lowest plane first.  Planes
// that a word has beyond NP, and those that the tet is done with, read
// "inside" for all vertices, which asks for nothing.
constexpr int code_words(int np) { return (np + 3) / 4; }

// Per plane (bits 2 j): set where the tet is not kept whole by plane j, and in
// *inside where some vertex lies inside it (clear: the plane drops the tet).
LSM_HD unsigned planes_cut(uint32_t s, unsigned* inside) {
  const uint32_t none = s & (s >> 1) & 0x55555555u;
  uint32_t o = s & ~(none | (none << 1));
  o |= o >> 16;
  o |= o >> 8;
  const unsigned in = o & 0x55u, out = (o >> 1) & 0x55u;
  *inside = in;
  return (0x55u & ~in) | out;
}

#ifdef __HIPCC__
// Index of the split table for plane j (0..3) of code word s.
__device__ __forceinline__ unsigned case_index(uint32_t s, int j) {
  return __builtin_amdgcn_udot4((s >> (2 * j)) & 0x03030303u, 0x40100401u, 0u, false);
}

// Bytes of (lo: selector 0..3, hi: 4..7) picked by the four selector bytes.
__device__ __forceinline__ uint32_t byte_permute(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}
#endif

// s with every vertex inside planes 0..j.
LSM_HD uint32_t done_up_to(uint32_t s, int j) {
  const uint32_t m = ((4u << (2 * j)) - 1u) * 0x01010101u;
  return (s & ~m) | (0x55555555u & m);
}

LSM_HD double plane_distance(const double* pl, const double* v) { return dot3(pl[0], pl[1], pl[2], v[0], v[1], v[2]) - pl[3]; }

// Split point between outside vertex vp (distance dp) and inside vertex vn.
LSM_HD void split_edge(double dp, double dn, const double* vp, const double* vn, double* x) {
  const double invdiff = 1.0 / (dp - dn);
  const double w0 = -dn * invdiff;
  const double w1 = dp * invdiff;
#pragma unroll
  for (int k = 0; k < 3; k++) x[k] = w0 * vp[k] + w1 * vn[k];
}

// tet_volume_tet(t) >= tol without the division by 6 wherever the two sides
// differ by more than its rounding.
LSM_HD bool volume_reaches(const double* t, double tol) {
  const double ax = t[0] - t[9], ay = t[1] - t[10], az = t[2] - t[11];
  const double bx = t[3] - t[9], by = t[4] - t[10], bz = t[5] - t[11];
  const double cx = t[6] - t[9], cy = t[7] - t[10], cz = t[8] - t[11];
  const double c0 = by * cz - bz * cy;
  const double c1 = bz * cx - bx * cz;
  const double c2 = bx * cy - by * cx;
  const double d = __builtin_fabs(dot3(ax, ay, az, c0, c1, c2));
  const double t6 = 6.0 * tol;
  bool keep = d > t6;
  if (__builtin_fabs(d - t6) <= 1e-12 * t6) keep = d / 6.0 >= tol;
  return keep;
}

#ifdef __HIPCC__
// ---------------------------------------------------------------------------
// Device side
// ---------------------------------------------------------------------------

static __device__ const SplitTable kSplitTable = make_split_table();

// Lane I of the quad's value, for all four lanes; and the or over the quad.
template <int I>
__device__ __forceinline__ uint32_t quad_lane(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, I * 0x55, 0xf, 0xf, true);
}
template <int I>
__device__ __forceinline__ double quad_lane(double x) {
  uint64_t b;
  __builtin_memcpy(&b, &x, 8);
  b = (uint64_t)quad_lane<I>((uint32_t)(b >> 32)) << 32 | quad_lane<I>((uint32_t)b);
  __builtin_memcpy(&x, &b, 8);
  return x;
}
__device__ __forceinline__ uint32_t quad_or(uint32_t x) {
  x |= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true);  // lanes 1 0 3 2
  x |= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4e, 0xf, 0xf, true);  // lanes 2 3 0 1
  return x;
}
// The value of the lane whose number differs by X (1 or 2).
template <int X>
__device__ __forceinline__ double quad_xor(double x) {
  constexpr int kPerm = X == 1 ? 0xb1 : 0x4e;
  uint64_t b;
  __builtin_memcpy(&b, &x, 8);
  b = (uint64_t)(uint32_t)__builtin_amdgcn_mov_dpp((int)(b >> 32), kPerm, 0xf, 0xf, true) << 32 |
      (uint32_t)__builtin_amdgcn_mov_dpp((int)b, kPerm, 0xf, 0xf, true);
  __builtin_memcpy(&x, &b, 8);
  return x;
}

// The wave's lanes exchange data through LDS in program order; only the
// compiler has to be kept from moving accesses across.
__device__ __forceinline__ void quad_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of one wave (16 quads).  Vertex ids are row * 16 + column; quads 4 s ..
// 4 s + 3 share pool[s], quad g's columns being 4 (g % 4) .. + 3, so that the
// sixteen lanes of an access cycle, four of each such quad, spread over all
// banks whatever ids they read.
template <int NP>
struct QuadLds {
  static constexpr int kRows = (NP + 1) * 16;
  static constexpr int kWords = 1 + code_words(NP);
  static constexpr int kEntries = 3 * (NP - 1);
  double pool[4][3][kRows];
  double planes[4][NP * 16];
  uint32_t stack[kEntries][kWords][16];
};

// One quad's clip: begin() with a tet, then step() until done().  With REGS the
// planes are kept in registers.
template <int NP, bool REGS = true>
struct QuadClip {
  static constexpr int kRows = QuadLds<NP>::kRows, kWords = QuadLds<NP>::kWords, SW = code_words(NP);
  double* pool;
  double* pl;
  uint32_t* stk;
  const uint4* table;
  int q;            // lane of the quad
  uint32_t T;       // the current tet's vertex ids
  uint32_t S[SW];   // and their sides
  uint32_t pend;    // pending stack entries: four bits a row, child 0 highest, the lowest unused
  int r;            // row of the next split's points
  bool cur;         // T is to be done
  // planes 1..NP-1, which every new vertex is classified against (in LDS they
  // took a fifth of its traffic, which bounds the step beside the VALU)
  double P[REGS ? NP - 1 : 1][4];

  __device__ __forceinline__ void init(QuadLds<NP>* lds, const uint4* tab) {
    const int lane = threadIdx.x & 63, g = lane >> 2;
    pool = &lds->pool[g >> 2][0][(g & 3) * 4];
    pl = &lds->planes[g >> 2][g & 3];
    stk = &lds->stack[0][0][g];
    table = tab;
    q = lane & 3;
    pend = 0;
    cur = false;
  }

  __device__ __forceinline__ bool done() const { return !cur && pend == 0; }

  // Plane j of the quad's pair, by one lane.
  __device__ __forceinline__ void set_plane(int j, const double* p) {
#pragma unroll
    for (int i = 0; i < 4; i++) pl[(4 * j + i) * 4] = p[i];
  }
  __device__ __forceinline__ void get_plane(int j, double* p) const {
#pragma unroll
    for (int i = 0; i < 4; i++) p[i] = pl[(4 * j + i) * 4];
  }

  __device__ __forceinline__ void vertex(uint32_t id, double* v) const {
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] = pool[k * kRows + id];
  }

  // Sides of a vertex against planes 1..NP-1, as code bytes; plane 0 reads
  // side0.
  __device__ __forceinline__ void sides(const double* v, unsigned side0, uint32_t* c) const {
#pragma unroll
    for (int w = 0; w < SW; w++) {
      c[w] = w == 0 ? side0 : 0u;
#pragma unroll
      for (int j = w == 0 ? 1 : 0; j < 4; j++) {
        const int p = 4 * w + j;
        unsigned s = 1u;
        if (p < NP) {
          double pl[4];
          if (!REGS) get_plane(p, pl);
          s = side_code(plane_distance(REGS ? P[REGS && p < NP ? p - 1 : 0] : pl, v));
        }
        c[w] |= s << (2 * j);
      }
    }
  }

  __device__ __forceinline__ void gather_codes(const uint32_t* c, uint32_t* out) const {
#pragma unroll
    for (int w = 0; w < SW; w++) out[w] = quad_or(c[w] << (8 * q));
  }

  // The tet whose vertex q is this lane's v; planes as set before.
  __device__ __forceinline__ void begin(const double* v) {
#pragma unroll
    for (int k = 0; k < 3; k++) pool[k * kRows + q] = v[k];
    quad_fence();
#pragma unroll
    for (int j = 1; j < (REGS ? NP : 1); j++) get_plane(j, P[j - 1]);
    double P0[4];
    get_plane(0, P0);
    uint32_t c[SW];
    sides(v, side_code(plane_distance(P0, v)), c);
    gather_codes(c, S);
    T = 0x03020100u;
    pend = 0;
    r = 1;
    cur = true;
  }

  __device__ __forceinline__ void pop() {
    const int e = 31 - __builtin_clz(pend);
    pend ^= 1u << e;
    r = (e >> 2) + 2;
    const int at = (e - 1 - (e >> 2)) * kWords * 16;
    T = stk[at];
#pragma unroll
    for (int w = 0; w < SW; w++) S[w] = stk[at + (1 + w) * 16];
  }

  // Cuts the current tet by the first plane that cuts it.  Calls leaf(t,
  // lead) with the outputs that come next in the reference's order, one per
  // lane (bit q of lead: this lane's t is one), and keeps the other children.
  template <class Leaf>
  __device__ __forceinline__ void step(Leaf&& leaf) {
    unsigned cut = 0, in = 0;
#pragma unroll
    for (int w = 0; w < SW; w++) {
      unsigned i;
      cut |= planes_cut(S[w], &i) << (8 * w);
      in |= i << (8 * w);
    }
    // no plane left: the tet is an output itself, its own only child
    const int j = cut == 0 ? 0 : __builtin_ctz(cut) >> 1;
    uint4 sc = make_uint4(0x03020100u, 0x03020100u, 0x03020100u, cut == 0 ? 1u << 5 : 0u);
    uint32_t rowS[SW];
#pragma unroll
    for (int w = 0; w < SW; w++) rowS[w] = 0;
    if (cut != 0 && ((in >> (2 * j)) & 1u)) {
      uint32_t sj = S[0];
#pragma unroll
      for (int w = 1; w < SW; w++) sj = (j >> 2) == w ? S[w] : sj;
      sc = table[case_index(sj, j & 3)];
      // this lane's split point
      const uint32_t b = sc.w >> (8 * q);
      double pj[4], vp[3], vn[3], x[3];
      get_plane(j, pj);
      vertex((T >> (b & 24u)) & 255u, vp);
      vertex((T >> ((b << 3) & 24u)) & 255u, vn);
      split_edge(plane_distance(pj, vp), plane_distance(pj, vn), vp, vn, x);
#pragma unroll
      for (int k = 0; k < 3; k++) pool[k * kRows + 16 * r + q] = x[k];
      uint32_t c[SW];
      sides(x, 1u, c);  // any split is by plane 0 or later
      gather_codes(c, rowS);
    }
    quad_fence();
    // the children, one per lane
    const uint32_t sel = q == 0 ? sc.x : (q == 1 ? sc.y : sc.z);
    const uint32_t row = byte_permute(0u, (uint32_t)r << 4, 0u) + 0x03020100u;  // the new points' ids
    const uint32_t ct = byte_permute(row, T, sel);
    uint32_t cs[SW];
    unsigned ccut = 0, cin = 0;
#pragma unroll
    for (int w = 0; w < SW; w++) {
      uint32_t s = byte_permute(rowS[w], S[w], sel);
      if (SW > 1) s = w < (j >> 2) ? 0x55555555u : (w == (j >> 2) ? done_up_to(s, j & 3) : s);
      else s = done_up_to(s, j);
      cs[w] = s;
      unsigned i;
      ccut |= planes_cut(s, &i) << (8 * w);
      cin |= i << (8 * w);
    }
    const bool mine = q < (int)((sc.w >> 5) & 3u);
    const bool whole = ccut == 0;
    const bool cuts = !whole && ((cin >> (__builtin_ctz(ccut | 0x80000000u) & 30)) & 1u);
    // bits 0-3: outputs already, bits 4-7: to be cut further
    const uint32_t kinds = quad_or((mine && whole ? 1u : 0u) << q | (mine && cuts ? 16u : 0u) << q);
    const uint32_t more = kinds >> 4;
    const uint32_t lead = kinds & 15u & ((more & -more) - 1u);  // the outputs before any other child
    if (((kinds & 15u & ~lead) | more) != 0) {
      const bool keep = mine && !((lead >> q) & 1u) && (whole || cuts);
      if (keep) {
        const int at = (3 * r - 1 - q) * kWords * 16;  // row r's entries 3 r - 3 .. 3 r - 1, child 0 last
        stk[at] = ct;
#pragma unroll
        for (int w = 0; w < SW; w++) stk[at + (1 + w) * 16] = cs[w];
      }
      // children 0, 1, 2 at bits 3, 2, 1 of the row's four
      const uint32_t left = (kinds & 15u & ~lead) | more;
      pend |= (__builtin_bitreverse32(left) >> 28) << (4 * r - 4);
    }
    cur = false;
    if (lead) {
      double t[12];
#pragma unroll
      for (int v = 0; v < 4; v++) vertex((ct >> (8 * v)) & 255u, t + 3 * v);
      leaf(t, lead);
    }
    quad_fence();
  }
};
#endif  // __HIPCC__

}  // namespace lsm
