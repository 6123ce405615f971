// The tiled step of meshes built by Cloth::new (springy/cloth.rs:20-113) in the reference's own
// summation order: the work of one TR x TC tile, split into tasks that the waves of one workgroup
// share out between its barriers.
//
//   stage    the states of the tile and a 2-vertex border (bending struts reach two vertices) and
//            the strut constants per row and column, into LDS;
//   tasks    every strut and every face that touches the tile, ONCE, and every tile vertex's six
//            corner weights, into LDS.  A strut's two force vectors (spring, damping) are stored
//            apart, since the reference adds them one after the other; its second end takes exactly
//            their negatives (p_a - p_b = -(p_b - p_a), and every later product carries the sign);
//   finish   each vertex adds its struts in strut-index order and its faces in face-index order
//            (the order of the reference's scatter loops, springy_mesh.rs:533-551, 629-654), then
//            integrates, meets obstacles, restores pins and stores.
//
// Strut order of vertex (r, c) of an R x C grid, and its faces: see grid_kernel in kernels.hip.
//
// Why tasks: a vertex's ten strut ends, two faces and six corner weights are ~1,650 operations, one
// long chain when a single lane takes them.  As tasks the struts are evaluated once (5 a vertex
// instead of 10), few values are live at a time, and twelve waves run struts, faces and corners side
// by side.  The larger tiles (grid_tiled_kernel in grid_tiled.hip) use the staging, the tables and the
// faces of this file and gather the rest per vertex.
#pragma once

#include "kernels.hpp"

#ifndef FP_LDS_CHECK
#define FP_LDS_CHECK(cond) ((void)0)
#endif

namespace fp {
namespace gtile {

// Strut constants of one row or column of the construction grid (Strut::new, springy_mesh.rs:74-90:
// a Cloth::new strut's rest length depends only on the two coordinates' difference): rest length,
// stiffness, damping, and the difference's square (for the shear struts' lengths).
struct KTab {
  float L, k, c, d2;
};

// What a tile's LDS holds of the struts: their constants only (every vertex evaluates its own), or
// their forces too (the 64-vertex tiles).
enum StrutRoom { CONSTANTS, FORCES };

template <int TR, int TC, StrutRoom ROOM>
struct Lds {
  static constexpr int SH = TR + 4, SW = TC + 4;  // staged rows [r0-2, r0+TR+2), columns alike
  static constexpr int QR = TR + 1, QC = TC + 1;  // quads (r', c') with r' in [r0-1, r0+TR), c' alike
  static constexpr int kFaces = 2 * QR * QC - 2;
  static constexpr int NV = TR * TC;
  static_assert(ROOM != FORCES || NV == 64, "forces are kept for 64-vertex tiles");
  // Rows of a wavefront (64 / TC of them) fall on distinct LDS banks (64 of 4 bytes) when rows are an
  // odd multiple of `step` words apart.
  static constexpr int pad(int words) {
    const int step = TC <= 8 ? 8 : TC <= 16 ? 16 : 32;
    int w = words;
    while (w % (2 * step) != step) ++w;
    return w;
  }
  // a staged row holds its six fields one after another (field q of column c at q * SW + c), a strut
  // row its six force components (spring x y z, damping x y z) W words apart, a face row face A's
  // drag + lift and face B's
  static constexpr int W = TC + 2, kSt = pad(6 * SW), kS = pad(6 * W), kF = pad(6 * QC);
  // rows of each class: h (r, c) -> (r, c+1) with c from c0-1 (column c - (c0-1)), v (r, c) -> (r+1, c)
  // with r from r0-1, s (r', c'+1) -> (r'+1, c') of quad (r', c'), bh (r, c) -> (r, c+2) with c from
  // c0-2, bv (r, c) -> (r+2, c) with r from r0-2
  static constexpr int H0 = 0, V0 = H0 + TR, S0 = V0 + TR + 1;
  static constexpr int BH0 = S0 + TR + 1, BV0 = BH0 + TR;
  static constexpr int kRows = ROOM == FORCES ? BV0 + TR + 2 : 1;
  float st[SH][kSt];
  float strut[kRows][kS];
  float face[QR][kF];
  float w[ROOM == FORCES ? 6 : 1][64];  // corner weights of vertex e = lr * TC + lc, in face order
  alignas(16) float atab[kFdlEntries][4];  // corner weights' reduction (fdl_entry)
  KTab th[TC + 1], tv[TR + 1], tbh[TC + 2], tbv[TR + 2];  // by first column / row, as above
  FP_HD float* h(int i, int j) { return at(H0, i, j, TR, TC + 1); }
  FP_HD float* v(int i, int j) { return at(V0, i, j, TR + 1, TC); }
  FP_HD float* s(int i, int j) { return at(S0, i, j, TR + 1, TC + 1); }
  FP_HD float* bh(int i, int j) { return at(BH0, i, j, TR, TC + 2); }
  FP_HD float* bv(int i, int j) { return at(BV0, i, j, TR + 2, TC); }

 private:
  FP_HD float* at(int base, int i, int j, int rows, int cols) {
    FP_LDS_CHECK(i >= 0 && i < rows && j >= 0 && j < cols && base + i < kRows);
    (void)rows; (void)cols;
    return &strut[base + i][j];
  }
};

template <int TR, int TC>
FP_HD bool interior_tile(const ClothView& G, int r0, int c0) {
  return r0 >= 2 && c0 >= 2 && r0 + TR + 2 <= (int)G.rows && c0 + TC + 2 <= (int)G.cols;
}

FP_HD KTab ktab(float d, float kn, float cn) {
  const float L = sqrt_rn(d * d + 0.0f);
  const float inv = rcp_rn(L);
  return KTab{L, inv * kn, inv * cn, d * d};
}

// Stages the tile with NT threads.  Every round's loads are issued, unconditionally, before the first
// LDS store, so that no lane waits for memory twice: a lane past the region's end loads its last entry
// again and on a tile at the grid's edge a lane outside the grid the nearest vertex; only the stores
// are conditional.  Addresses are a workgroup-uniform base (the tile's first vertex, in the grid) and a
// 32-bit byte offset per lane.
template <int NT, int TR, int TC, StrutRoom ROOM>
FP_HD void stage(Lds<TR, TC, ROOM>& L, const StepArgs& A, const ClothView& G, int r0, int c0, bool interior, int tid) {
  using S = Lds<TR, TC, ROOM>;
  constexpr int NS = S::SH * S::SW, RND = (NS + NT - 1) / NT;
  const int R = (int)G.rows, C = (int)G.cols, nthreads = NT;
  const uint32_t g0 = G.base + (uint32_t)(r0 * C + c0);
  float q[RND][6];
#pragma unroll
  for (int k = 0; k < RND; ++k) {
    const int e = tid + k * NT < NS ? tid + k * NT : NS - 1, lr = e / S::SW, lc = e - lr * S::SW;
    int dr = lr - 2, dc = lc - 2;
    if (!interior) {
      dr = r0 + dr < 0 ? -r0 : r0 + dr >= R ? R - 1 - r0 : dr;
      dc = c0 + dc < 0 ? -c0 : c0 + dc >= C ? C - 1 - c0 : dc;
    }
    const int32_t ob = (dr * C + dc) * 4;
    auto at = [&](const float* p) { return *(const float*)((const char*)(p + g0) + ob); };
    q[k][0] = at(A.in.x); q[k][1] = at(A.in.y); q[k][2] = at(A.in.z);
    q[k][3] = at(A.in.vx); q[k][4] = at(A.in.vy); q[k][5] = at(A.in.vz);
  }
  for (int e = tid; e < kFdlEntries; e += nthreads) fdl_entry(e, L.atab[e]);
  // the constant tables, by the workgroup's last threads (the first ones may have a second round of
  // states): columns' struts, rows' struts, columns' bends, rows' bends
  constexpr int N0 = TC + 1, N1 = N0 + TR + 1, N2 = N1 + TC + 2, N3 = N2 + TR + 2;
  for (int e = nthreads - 1 - tid; e < N3; e += nthreads) {
    const bool bend = e >= N1, cols = e < N0 || (bend && e < N2);
    const int j = e - (e >= N2 ? N2 : e >= N1 ? N1 : e >= N0 ? N0 : 0);
    const int first = (cols ? c0 : r0) - (bend ? 2 : 1) + j, second = first + (bend ? 2 : 1);
    const float o = cols ? G.cx : G.cy, p = cols ? G.p0 : G.p1;
    const float d = (((float)first * G.spacing - o) + p) - (((float)second * G.spacing - o) + p);
    const KTab K = ktab(d, bend ? G.bk : G.tk, bend ? G.bc : G.tc);
    (cols ? (bend ? L.tbh : L.th) : (bend ? L.tbv : L.tv))[j] = K;
  }
  // the states last: the tables are formed while they are on their way (32 x 32 vertices: 5.1 -> 4.9 us a
  // step, 256 x 256: 9.4 -> 9.1)
#pragma unroll
  for (int k = 0; k < RND; ++k) {
    const int e = tid + k * NT, lr = e / S::SW, lc = e - lr * S::SW, r = r0 - 2 + lr, c = c0 - 2 + lc;
    if (e < NS && (interior || (r >= 0 && r < R && c >= 0 && c < C))) {
      float* row = &L.st[lr][lc];
#pragma unroll
      for (int f = 0; f < 6; ++f) row[f * S::SW] = q[k][f];
    }
  }
}

template <int TR, int TC, StrutRoom ROOM>
FP_HD f3 pos(const Lds<TR, TC, ROOM>& L, int row, int col) {
  FP_LDS_CHECK(row >= 0 && row < TR + 4 && col >= 0 && col < TC + 4);
  const float* q = &L.st[row][col];
  return f3{q[0], q[TC + 4], q[2 * (TC + 4)]};
}
template <int TR, int TC, StrutRoom ROOM>
FP_HD f3 vel(const Lds<TR, TC, ROOM>& L, int row, int col) {
  FP_LDS_CHECK(row >= 0 && row < TR + 4 && col >= 0 && col < TC + 4);
  const float* q = &L.st[row][col];
  return f3{q[3 * (TC + 4)], q[4 * (TC + 4)], q[5 * (TC + 4)]};
}

// One strut from its first end a to its second b (staged coordinates): the spring and damping force
// on the first end (springy_mesh.rs:535-549).
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void strut(const Lds<TR, TC, ROOM>& L, int ra, int ca, int rb, int cb, float k, float c, float rest, float* out) {
  constexpr int W = Lds<TR, TC, ROOM>::W;
  const f3 d = sub(pos(L, rb, cb), pos(L, ra, ca));
  float len, inv;
  M::sqrt_rcp(dot(d, d), len, inv);
  const f3 u = f3{d.x * inv, d.y * inv, d.z * inv};
  const float s = k * (len - rest);
  const float dd = c * M::dot(sub(vel(L, rb, cb), vel(L, ra, ca)), u);
  out[0] = s * u.x; out[W] = s * u.y; out[2 * W] = s * u.z;
  out[3 * W] = dd * u.x; out[4 * W] = dd * u.y; out[5 * W] = dd * u.z;
}
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void shear_strut(Lds<TR, TC, ROOM>& L, const ClothView& G, int i, int j, int ra, int ca) {
  float rest, inv;
  M::sqrt_rcp(L.th[j].d2 + L.tv[i].d2, rest, inv);
  strut<M>(L, ra, ca, ra + 1, ca - 1, inv * G.sk, inv * G.sc, rest, L.s(i, j));
}

// The struts that vertex (lr, lc) of the tile starts: right, down and down left; right and down bends.
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void own_mesh_struts(Lds<TR, TC, ROOM>& L, const ClothView& G, int lr, int lc) {
  const int a = lr + 2, b = lc + 2;
  const KTab H = L.th[lc + 1], V = L.tv[lr + 1];
  strut<M>(L, a, b, a, b + 1, H.k, H.c, H.L, L.h(lr, lc + 1));
  strut<M>(L, a, b, a + 1, b, V.k, V.c, V.L, L.v(lr + 1, lc));
  shear_strut<M>(L, G, lr + 1, lc, a, b);
}
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void own_bends(Lds<TR, TC, ROOM>& L, int lr, int lc) {
  const int a = lr + 2, b = lc + 2;
  const KTab H = L.tbh[lc + 2], V = L.tbv[lr + 2];
  strut<M>(L, a, b, a, b + 2, H.k, H.c, H.L, L.bh(lr, lc + 2));
  strut<M>(L, a, b, a + 2, b, V.k, V.c, V.L, L.bv(lr + 2, lc));
}

// The struts that reach the tile from outside it: 2 (TR + TC) - 1 mesh struts (column c0-1's row
// struts, row r0-1's column struts, the shear struts of quad row r0-1 and of quad column c0+TC-1) and
// 2 (TR + TC) bends (columns c0-2 and c0-1, rows r0-2 and r0-1).
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void border_mesh_strut(Lds<TR, TC, ROOM>& L, const ClothView& G, int e) {
  if (e < TR + TC) {
    const bool hor = e < TR;
    const int i = hor ? e : e - TR;
    const KTab K = hor ? L.th[0] : L.tv[0];
    const int ra = hor ? i + 2 : 1, ca = hor ? 1 : i + 2;
    strut<M>(L, ra, ca, hor ? ra : ra + 1, hor ? ca + 1 : ca, K.k, K.c, K.L, hor ? L.h(i, 0) : L.v(0, i));
    return;
  }
  e -= TR + TC;
  const int i = e < TC ? 0 : e - TC + 1, j = e < TC ? e + 1 : TC;
  shear_strut<M>(L, G, i, j, i + 1, j + 2);
}
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void border_bend(Lds<TR, TC, ROOM>& L, int e) {
  const bool hor = e < 2 * TR;
  const int q = hor ? e : e - 2 * TR, n = hor ? TR : TC, which = q >= n ? 1 : 0, i = q - which * n;
  const KTab K = hor ? L.tbh[which] : L.tbv[which];
  const int ra = hor ? i + 2 : which, ca = hor ? which : i + 2;
  strut<M>(L, ra, ca, hor ? ra : ra + 2, hor ? ca + 2 : ca, K.k, K.c, K.L, hor ? L.bh(i, which) : L.bv(which, i));
}

// Drag + lift of face f of the tile's 2 QR QC - 2: A(q) = [(r',c'+1), (r'+1,c'), (r',c')] of every quad
// but the first, then B(q) = [(r',c'+1), (r'+1,c'+1), (r'+1,c')] of every quad but the last (those two
// have no corner in the tile; without them a 16x16 tile's 576 faces are nine full wavefronts).
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void face(Lds<TR, TC, ROOM>& L, const StepParams& P, int f) {
  using S = Lds<TR, TC, ROOM>;
  constexpr int NQ = S::QR * S::QC;
  const int which = f >= NQ - 1 ? 1 : 0, q = which ? f - (NQ - 1) : f + 1, i = q / S::QC, j = q - i * S::QC;
  const int a = i + 1, b = j + 1;  // staged corner (r', c')
  const int r1 = a + 1, c1 = b + which, r2 = a + which, c2 = b;
  const f3 F = face_force<M>(pos(L, a, b + 1), pos(L, r1, c1), pos(L, r2, c2), vel(L, a, b + 1), vel(L, r1, c1),
                             vel(L, r2, c2), P);
  float* out = &L.face[i][3 * which * S::QC + j];
  out[0] = F.x; out[S::QC] = F.y; out[2 * S::QC] = F.z;
}

// The two other corners of vertex (lr, lc)'s face number k (its faces in face order: A(r-1,c),
// A(r,c-1), A(r,c), B(r-1,c-1), B(r-1,c), B(r,c-1)): offsets of the next and the previous corner.
FP_HD void corner_ends(int k, int& rn, int& cn, int& rp, int& cp) {
  // next: (-1,0) (1,-1) (0,1) (0,-1) (-1,1) (1,0); previous: (-1,1) (0,-1) (1,0) (-1,0) (0,1) (1,-1)
  rn = k == 0 || k == 4 ? -1 : k == 1 || k == 5 ? 1 : 0;
  cn = k == 1 || k == 3 ? -1 : k == 2 || k == 4 ? 1 : 0;
  rp = k == 0 || k == 3 ? -1 : k == 2 || k == 5 ? 1 : 0;
  cp = k == 1 || k == 5 ? -1 : k == 0 || k == 4 ? 1 : 0;
}
// One corner weight, number k the same for the whole wave.
template <class M, int TR, int TC, StrutRoom ROOM>
FP_HD void corner(Lds<TR, TC, ROOM>& L, int k, int e, int lr, int lc) {
  int rn, cn, rp, cp;
  corner_ends(k, rn, cn, rp, cp);
  const int a = lr + 2, b = lc + 2;
  L.w[k][e] = corner_weight<M, true>(pos(L, a, b), pos(L, a + rn, b + cn), pos(L, a + rp, b + cp), L.atab);
}

// N components, from component q0 on, of vertex (lr, lc)'s force: the reference adds the mesh struts,
// the bends and the faces to what F holds (initial force plus gravity), in this order.
template <int N, bool BORDER, int TR, int TC, StrutRoom ROOM>
struct Summer {
  Lds<TR, TC, ROOM>& L;
  int r, c, lr, lc, q0, R, C;
  using S = Lds<TR, TC, ROOM>;
  FP_HD void plus(float (&F)[N], const float* f) const {
#pragma unroll
    for (int q = 0; q < N; ++q) { F[q] = F[q] + f[(q0 + q) * S::W]; F[q] = F[q] + f[(q0 + q + 3) * S::W]; }
  }
  FP_HD void minus(float (&F)[N], const float* f) const {
#pragma unroll
    for (int q = 0; q < N; ++q) { F[q] = F[q] - f[(q0 + q) * S::W]; F[q] = F[q] - f[(q0 + q + 3) * S::W]; }
  }
  FP_HD bool up() const { return !BORDER || r >= 1; }
  FP_HD bool down() const { return !BORDER || r <= R - 2; }
  FP_HD bool left() const { return !BORDER || c >= 1; }
  FP_HD bool right() const { return !BORDER || c <= C - 2; }
  FP_HD void mesh_struts(float (&F)[N]) const {
    // the last column's upward strut belongs to a bottom-right triangle: after quad (r, c-1)'s
    const bool late = BORDER && c == C - 1 && r >= 1 && r <= R - 2;
    if (up() && right()) minus(F, L.s(lr, lc + 1));
    if (up() && !late) minus(F, L.v(lr, lc));
    if (down() && left()) plus(F, L.s(lr + 1, lc));
    if (left()) minus(F, L.h(lr, lc));
    if (late) minus(F, L.v(lr, lc));
    if (down()) plus(F, L.v(lr + 1, lc));
    if (right()) plus(F, L.h(lr, lc + 1));
  }
  FP_HD void bends(float (&F)[N]) const {
    if (!BORDER || (r >= 2 && c <= C - 3)) minus(F, L.bv(lr, lc));
    if (!BORDER || (c >= 2 && r <= R - 3)) minus(F, L.bh(lr, lc));
    if (!BORDER || (r <= R - 3 && c <= C - 3)) { plus(F, L.bh(lr, lc + 2)); plus(F, L.bv(lr + 2, lc)); }
  }
  FP_HD void faces(float (&F)[N], const float (&w)[6]) const {
    auto add_face = [&](float wk, const float* f) {
#pragma unroll
      for (int q = 0; q < N; ++q) F[q] = F[q] + wk * f[(q0 + q) * S::QC];
    };
    constexpr int B = 3 * S::QC;  // face B's part of a face row
    if (up() && right()) add_face(w[0], &L.face[lr][lc + 1]);
    if (down() && left()) add_face(w[1], &L.face[lr + 1][lc]);
    if (down() && right()) add_face(w[2], &L.face[lr + 1][lc + 1]);
    if (up() && left()) add_face(w[3], &L.face[lr][B + lc]);
    if (up() && right()) add_face(w[4], &L.face[lr][B + lc + 1]);
    if (down() && left()) add_face(w[5], &L.face[lr + 1][B + lc]);
  }
};

}  // namespace gtile
}  // namespace fp
