// LDS-tiled step kernels for meshes built by Cloth::new (springy/cloth.rs:20-113) in the reference's
// summation order, one workgroup per tile: a twelve-wave form for 64-vertex tiles, where a step is one
// tile's chain of dependent work, and a lane per vertex for larger tiles, where it is vector issue
// (the host's rule: tile_rule.hpp).  The per-vertex operations and their order are those of grid_kernel,
// so the EXACT form returns the same bits as the reference.  HBM traffic: the state read once (plus halo
// rows that the L2 serves) and written once.
#include "grid_tile_core.hpp"

namespace fp {

namespace {

using gtile::FORCES;
using gtile::CONSTANTS;

// 64-vertex tiles, twelve waves: two of struts, one of struts reaching in, three of faces, six of
// corners, and then one wave per force component.  Bound by its chain of dependent operations (the
// longest task's ~190 and a component's ~90, against ~1,650 when one lane takes a vertex), the launch
// and the two memory round trips: 4.8 us a step on 64 x 64 vertices, 5.1 on 128 x 128, where a lane per
// vertex took 12.3 (and takes 8.7 now).
template <int MODE>
__global__ void __launch_bounds__(768) grid_tiled_kernel_small(StepArgs A, const ClothView* __restrict__ cloths,
                                                               const TileRange* __restrict__ tiles) {
  using M = ExactMath;
  using S = gtile::Lds<8, 8, FORCES>;
  __shared__ S L;
  __shared__ float s_x[9][64];  // new positions, new velocities, forces
  const TileRange T = tiles[blockIdx.x];
  const ClothView C = cloths[T.mesh];
  const StepParams P = A.params[T.mesh];
  const int r0 = (int)T.r0, c0 = (int)T.c0, tid = (int)threadIdx.x, e = tid & 63, lr = e / 8, lc = e % 8;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = r0 + lr, c = c0 + lc;
  const bool interior = gtile::interior_tile<8, 8>(C, r0, c0);
  const bool mine = wave < 3 && r < (int)C.rows && c < (int)C.cols;  // finishes component `wave` of the vertex
  const uint32_t i = C.base + (uint32_t)(r * (int)C.cols + c);
  const bool pin = mine && pinned(A.pins, i);
  gtile::stage<768>(L, A, C, r0, c0, interior, tid);
  __syncthreads();
  if (wave == 0) gtile::own_mesh_struts<M>(L, C, lr, lc);
  else if (wave == 1) gtile::own_bends<M>(L, lr, lc);
  else if (wave == 2) {
    if (e < 2 * (8 + 8) - 1) gtile::border_mesh_strut<M>(L, C, e);
    else if (e >= 32) gtile::border_bend<M>(L, e - 32);
  } else if (wave < 6) {
    const int f = (wave - 3) * 64 + e;
    if (f < S::kFaces) gtile::face<M>(L, P, f);
  } else {
    gtile::corner<M>(L, wave - 6, e, lr, lc);
  }
  __syncthreads();
  const int q = wave;
  float xn = 0.0f, vn = 0.0f, F[1] = {0.0f}, p = 0.0f, v = 0.0f;
  float* const force = q == 0 ? A.fx : q == 1 ? A.fy : A.fz;
  if (mine) {
    F[0] = (A.force_init ? force[i] : 0.0f) + (q == 0 ? P.gravity.x : q == 1 ? P.gravity.y : P.gravity.z);
    const float w[6] = {L.w[0][e], L.w[1][e], L.w[2][e], L.w[3][e], L.w[4][e], L.w[5][e]};
    auto sum = [&](auto s) {
      s.mesh_struts(F);
      s.bends(F);
      s.faces(F, w);
    };
    if (interior) sum(gtile::Summer<1, false, 8, 8, FORCES>{L, r, c, lr, lc, q, (int)C.rows, (int)C.cols});
    else sum(gtile::Summer<1, true, 8, 8, FORCES>{L, r, c, lr, lc, q, (int)C.rows, (int)C.cols});
    if (pin) F[0] = 0.0f;
    if (MODE == MODE_FORCES) {
      force[i] = F[0];
    } else {
      const float* row = &L.st[lr + 2][lc + 2];
      p = row[q * S::SW];
      v = row[(q + 3) * S::SW];
      integrate1<M>(P, P.mass, p, v, F[0], xn, vn);
      s_x[q][e] = xn;
      s_x[3 + q][e] = vn;
      s_x[6 + q][e] = F[0];
    }
  }
  if (MODE == MODE_FORCES) return;
  if (A.obs.n_faces != 0) {  // each component's wave finds the same hit and keeps its component
    __syncthreads();
    if (mine) {
      const f3 po = gtile::pos(L, lr + 2, lc + 2), pn = f3{s_x[0][e], s_x[1][e], s_x[2][e]};
      const int32_t hit = first_hit(A.obs, po, pn, P.dt_d);
      if (hit >= 0) {
        f3 x = pn, w = f3{s_x[3][e], s_x[4][e], s_x[5][e]};
        collide_response(A.obs.faces[hit], P, P.mass, po, gtile::vel(L, lr + 2, lc + 2),
                         f3{s_x[6][e], s_x[7][e], s_x[8][e]}, x, w);
        xn = q == 0 ? x.x : q == 1 ? x.y : x.z;
        vn = q == 0 ? w.x : q == 1 ? w.y : w.z;
      }
    }
  }
  if (mine) {
    (q == 0 ? A.out.x : q == 1 ? A.out.y : A.out.z)[i] = pin ? p : xn;
    (q == 0 ? A.out.vx : q == 1 ? A.out.vy : A.out.vz)[i] = pin ? v : vn;
    if (A.force_init) force[i] = 0.0f;
  }
}

// One lane per vertex: it evaluates its ten strut ends and six corner weights itself (only the faces
// are shared through LDS).  More operations a vertex than as tasks, but one long run of work between
// two barriers and 21 KB a tile, so seven workgroups a CU keep the vector units busy: the form for
// larger simulations.  Bound by vector issue: 1,640 operations a wave (2,137 before tiles inside the
// grid lost their guards, the shear constants' table, the general square roots, quotients and interval
// selects), 1024 x 1024 vertices in 43.6 us a step where it took 54.7.  Sharing the struts as tasks at
// this tile size was slower: 1,540 operations, but five barriers and 47 KB leave the units idle 30 % of
// the time (49 us).
//
// The compiler would rather load each neighbour once for struts and corners and postpone the sums,
// which takes 158 registers and leaves three waves a SIMD; `settle` makes the tile offset and the
// force so far opaque after every term, so each term is finished before the next begins.
template <class M, int TR, int TC, int MODE, bool BORDER>
__device__ __forceinline__ void gather_vertex(gtile::Lds<TR, TC, CONSTANTS>& L, const StepArgs& A, const StepParams& P,
                                              const ClothView& G, int r, int c, int lr, int lc) {
  using S = gtile::Lds<TR, TC, CONSTANTS>;
  const int R = (int)G.rows, C = (int)G.cols;
  const uint32_t i = G.base + (uint32_t)(r * C + c);
  int own = (lr + 2) * S::kSt + lc + 2;
  auto at = [&](int dr, int dc) { return &L.st[0][0] + own + (dr * S::kSt + dc); };
  auto pos = [&](int dr, int dc) { const float* q = at(dr, dc); return f3{q[0], q[S::SW], q[2 * S::SW]}; };
  auto vel = [&](int dr, int dc) { const float* q = at(dr, dc); return f3{q[3 * S::SW], q[4 * S::SW], q[5 * S::SW]}; };
  const f3 p = pos(0, 0), v = vel(0, 0);
  const float m = P.mass;  // a mesh with unequal masses is not on this kernel
  // MODE_SURROGATE: F collects only the face forces (from zero); gravity and the network's
  // acceleration enter in sur_update
  constexpr bool kStruts = MODE != MODE_SURROGATE;
  f3 F = kStruts && A.force_init ? f3{A.fx[i], A.fy[i], A.fz[i]} : f3{0.0f, 0.0f, 0.0f};
  if (kStruts) F = add(F, P.gravity);
  auto settle = [&] { asm volatile("" : "+v"(own), "+v"(F.x), "+v"(F.y), "+v"(F.z)); };
  auto strut = [&](int dr, int dc, float k, float cc, float rest) {
    strut_accumulate<M>(F, p, v, pos(dr, dc), vel(dr, dc), k, cc, rest);
    settle();
  };
  auto straight = [&](int dr, int dc, const gtile::KTab& K) { strut(dr, dc, K.k, K.c, K.L); };
  auto shear = [&](int dr, int dc, int i2, int j2) {
    float rest, inv;
    M::sqrt_rcp(L.th[j2].d2 + L.tv[i2].d2, rest, inv);
    strut(dr, dc, inv * G.sk, inv * G.sc, rest);
  };
  // struts in strut-index order (see grid_kernel in kernels.hip); quad (r-1, c-1) is number (lr, lc)
  const bool up = !BORDER || r >= 1, down = !BORDER || r <= R - 2, left = !BORDER || c >= 1, right = !BORDER || c <= C - 2;
  const bool late = BORDER && c == C - 1 && r >= 1 && r <= R - 2;  // see Summer::mesh_struts
  if constexpr (kStruts) {
    if (up && right) shear(-1, 1, lr, lc + 1);
    if (up && !late) straight(-1, 0, L.tv[lr]);
    if (down && left) shear(1, -1, lr + 1, lc);
    if (left) straight(0, -1, L.th[lc]);
    if (late) straight(-1, 0, L.tv[lr]);
    if (down) straight(1, 0, L.tv[lr + 1]);
    if (right) straight(0, 1, L.th[lc + 1]);
    if (!BORDER || (r >= 2 && c <= C - 3)) straight(-2, 0, L.tbv[lr]);
    if (!BORDER || (c >= 2 && r <= R - 3)) straight(0, -2, L.tbh[lc]);
    if (!BORDER || (r <= R - 3 && c <= C - 3)) { straight(0, 2, L.tbh[lc + 2]); straight(2, 0, L.tbv[lr + 2]); }
  }
  // faces in face-index order, each this vertex's corner weight times the face's drag + lift
  auto face = [&](int k, const float* f) {
    int rn, cn, rp, cp;
    gtile::corner_ends(k, rn, cn, rp, cp);
    const float w = corner_weight<M, true>(p, pos(rn, cn), pos(rp, cp), L.atab);
    F = add(F, f3{w * f[0], w * f[S::QC], w * f[2 * S::QC]});
    settle();
  };
  constexpr int B = 3 * S::QC;  // face B's part of a face row
  if (up && right) face(0, &L.face[lr][lc + 1]);
  if (down && left) face(1, &L.face[lr + 1][lc]);
  if (down && right) face(2, &L.face[lr + 1][lc + 1]);
  if (up && left) face(3, &L.face[lr][B + lc]);
  if (up && right) face(4, &L.face[lr][B + lc + 1]);
  if (down && left) face(5, &L.face[lr + 1][B + lc]);
  const bool pin = pinned(A.pins, i);
  if (MODE == MODE_SURROGATE) {
    f3 xn = p, vn = v;
    float work = 0.0f;
    if (!pin)
      work = sur_update(P, A.obs, m, p, v, F, f3{0.0f, 0.0f, 0.0f},
                        f3{A.da[3 * (size_t)i], A.da[3 * (size_t)i + 1], A.da[3 * (size_t)i + 2]}, xn, vn);
    A.out.x[i] = xn.x; A.out.y[i] = xn.y; A.out.z[i] = xn.z;
    A.out.vx[i] = vn.x; A.out.vy[i] = vn.y; A.out.vz[i] = vn.z;
    A.work[i] = work;
    return;
  }
  if (pin) F = f3{0.0f, 0.0f, 0.0f};
  if (MODE == MODE_FORCES) {
    A.fx[i] = F.x; A.fy[i] = F.y; A.fz[i] = F.z;
    return;
  }
  f3 xn, vn;
  integrate<M>(P, m, p, v, F, xn, vn);
  const int32_t hit = first_hit(A.obs, p, xn, P.dt_d);
  if (hit >= 0) collide_response(A.obs.faces[hit], P, m, p, v, F, xn, vn);
  if (pin) { xn = p; vn = v; }
  A.out.x[i] = xn.x; A.out.y[i] = xn.y; A.out.z[i] = xn.z;
  A.out.vx[i] = vn.x; A.out.vy[i] = vn.y; A.out.vz[i] = vn.z;
  if (A.force_init) { A.fx[i] = 0.0f; A.fy[i] = 0.0f; A.fz[i] = 0.0f; }
}

template <class M, int TR, int TC, int MODE>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(MODE == MODE_SURROGATE ? 6 : 7, 8)))
grid_tiled_kernel(StepArgs A, const ClothView* __restrict__ cloths, const TileRange* __restrict__ tiles) {
  using S = gtile::Lds<TR, TC, CONSTANTS>;
  __shared__ S L;
  const TileRange T = tiles[blockIdx.x];
  const ClothView C = cloths[T.mesh];
  const StepParams P = A.params[T.mesh];
  const int r0 = (int)T.r0, c0 = (int)T.c0, e = (int)threadIdx.x, lr = e / TC, lc = e - lr * TC;
  const int r = r0 + lr, c = c0 + lc;
  const bool interior = gtile::interior_tile<TR, TC>(C, r0, c0);
  gtile::stage<(int)kBlock>(L, A, C, r0, c0, interior, e);
  __syncthreads();
  for (int f = e; f < S::kFaces; f += kBlock) gtile::face<M>(L, P, f);
  __syncthreads();
  if (e >= S::NV || r >= (int)C.rows || c >= (int)C.cols) return;
  if (interior) gather_vertex<M, TR, TC, MODE, false>(L, A, P, C, r, c, lr, lc);
  else gather_vertex<M, TR, TC, MODE, true>(L, A, P, C, r, c, lr, lc);
}

template <class M, int TR, int TC, int MODE>
hipError_t launch_lanes(const StepArgs& a, const ClothView* cloths, const TileRange* tiles, uint32_t n, hipStream_t s) {
  grid_tiled_kernel<M, TR, TC, MODE><<<dim3(n), dim3(kBlock), 0, s>>>(a, cloths, tiles);
  return hipGetLastError();
}

template <int TR, int TC>
hipError_t launch_shape(const StepArgs& a, const ClothView* cloths, const TileRange* tiles, uint32_t n, int mode,
                        hipStream_t s) {
  if (mode == MODE_STEP) return launch_lanes<ExactMath, TR, TC, MODE_STEP>(a, cloths, tiles, n, s);
  if (mode == MODE_FORCES) return launch_lanes<ExactMath, TR, TC, MODE_FORCES>(a, cloths, tiles, n, s);
  return launch_lanes<FastMath, TR, TC, MODE_SURROGATE>(a, cloths, tiles, n, s);
}

hipError_t launch_small(const StepArgs& a, const ClothView* cloths, const TileRange* tiles, uint32_t n, int mode,
                        hipStream_t s) {
  if (mode == MODE_SURROGATE) return launch_lanes<FastMath, 8, 8, MODE_SURROGATE>(a, cloths, tiles, n, s);
  if (mode == MODE_STEP) grid_tiled_kernel_small<MODE_STEP><<<dim3(n), dim3(768), 0, s>>>(a, cloths, tiles);
  else grid_tiled_kernel_small<MODE_FORCES><<<dim3(n), dim3(768), 0, s>>>(a, cloths, tiles);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_grid_tiled(const StepArgs& a, const ClothView* cloths, const TileRange* tiles, uint32_t n_tiles,
                             int shape, int mode, hipStream_t s) {
  if (n_tiles == 0) return hipSuccess;
  switch (shape) {
    case TILE_15x15: return launch_shape<15, 15>(a, cloths, tiles, n_tiles, mode, s);
    case TILE_7x31: return launch_shape<7, 31>(a, cloths, tiles, n_tiles, mode, s);
    case TILE_16x16: return launch_shape<16, 16>(a, cloths, tiles, n_tiles, mode, s);
    case TILE_8x8: return launch_small(a, cloths, tiles, n_tiles, mode, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fp
