// CPU emulation of the exact tiled grid kernel (feriphys_amd/csrc/grid_tile_core.hpp): each tile's
// staging, tasks and per-vertex sums run on the host in barrier order, every staged index checked and
// the LDS filled with NaN beforehand, so a read of a slot that no task wrote shows in the results.
// Test infrastructure only.  No obstacles.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

#define FP_LDS_CHECK(cond)                                                      \
  do {                                                                          \
    if (!(cond)) {                                                              \
      std::fprintf(stderr, "tile_emul: index check failed: %s\n", #cond);       \
      std::abort();                                                             \
    }                                                                           \
  } while (0)
#include "../../feriphys_amd/csrc/grid_tile_core.hpp"

namespace {

using M = fp::ExactMath;

constexpr int TR = 8, TC = 8;

void run(const fp::StepArgs& A, const fp::ClothView& G, const fp::StepParams& P, int mode) {
  constexpr fp::gtile::StrutRoom ROOM = fp::gtile::FORCES;
  using S = fp::gtile::Lds<TR, TC, ROOM>;
  std::vector<float> Fs(3 * S::NV), ws(6 * S::NV);  // each thread's registers across the barriers
  std::unique_ptr<S> L(new S);
  const float g[3] = {P.gravity.x, P.gravity.y, P.gravity.z};
  float* const force[3] = {A.fx, A.fy, A.fz};
  float* const out[6] = {A.out.x, A.out.y, A.out.z, A.out.vx, A.out.vy, A.out.vz};
  constexpr int threads = 768;
  for (uint32_t t0 = 0; t0 < G.rows; t0 += TR)
    for (uint32_t u0 = 0; u0 < G.cols; u0 += TC) {
      const int r0 = (int)t0, c0 = (int)u0;
      std::memset((void*)L.get(), 0xff, sizeof(S));  // NaN everywhere
      const bool in = fp::gtile::interior_tile<TR, TC>(G, r0, c0);
      for (int t = 0; t < threads; ++t) fp::gtile::stage<threads>(*L, A, G, r0, c0, in, t);
      auto mesh = [&] {
        for (int e = 0; e < S::NV; ++e) fp::gtile::own_mesh_struts<M>(*L, G, e / TC, e % TC);
        for (int e = 0; e < 2 * (TR + TC) - 1; ++e) fp::gtile::border_mesh_strut<M>(*L, G, e);
      };
      auto bends = [&] {
        for (int e = 0; e < S::NV; ++e) fp::gtile::own_bends<M>(*L, e / TC, e % TC);
        for (int e = 0; e < 2 * (TR + TC); ++e) fp::gtile::border_bend<M>(*L, e);
      };
      auto in_grid = [&](int e) { return r0 + e / TC < (int)G.rows && c0 + e % TC < (int)G.cols; };
      // vertex e's sum, one component at a time
      auto sum = [&](int e) {
        const int r = r0 + e / TC, c = c0 + e % TC;
        float w[6];
        for (int k = 0; k < 6; ++k) w[k] = ws[6 * e + k];
        for (int q = 0; q < 3; ++q) {
          float F[1] = {Fs[3 * e + q]};
          auto go = [&](auto s) {
            s.mesh_struts(F);
            s.bends(F);
            s.faces(F, w);
          };
          if (in) go(fp::gtile::Summer<1, false, TR, TC, ROOM>{*L, r, c, e / TC, e % TC, q, (int)G.rows, (int)G.cols});
          else go(fp::gtile::Summer<1, true, TR, TC, ROOM>{*L, r, c, e / TC, e % TC, q, (int)G.rows, (int)G.cols});
          Fs[3 * e + q] = F[0];
        }
      };
      for (int f = 0; f < S::kFaces; ++f) fp::gtile::face<M>(*L, P, f);
      for (int e = 0; e < S::NV; ++e) {
        float w[6];
        for (int k = 0; k < 6; ++k) fp::gtile::corner<M>(*L, k, e, e / TC, e % TC);
        for (int k = 0; k < 6; ++k) w[k] = L->w[k][e];
        for (int k = 0; k < 6; ++k) ws[6 * e + k] = w[k];
        if (!in_grid(e)) continue;
        const uint32_t i = G.base + (uint32_t)((r0 + e / TC) * (int)G.cols + c0 + e % TC);
        for (int q = 0; q < 3; ++q) Fs[3 * e + q] = (A.force_init ? force[q][i] : 0.0f) + g[q];
      }
      mesh();
      bends();
      for (int e = 0; e < S::NV; ++e) {
        if (!in_grid(e)) continue;
        sum(e);
        const int lr = e / TC, lc = e % TC, r = r0 + lr, c = c0 + lc;
        const uint32_t i = G.base + (uint32_t)(r * (int)G.cols + c);
        const bool pin = A.pins && ((A.pins[i >> 5] >> (i & 31u)) & 1u);
        float F[3] = {Fs[3 * e], Fs[3 * e + 1], Fs[3 * e + 2]};
        if (pin) F[0] = F[1] = F[2] = 0.0f;
        if (mode == 1) {
          for (int q = 0; q < 3; ++q) force[q][i] = F[q];
          continue;
        }
        const fp::f3 p = fp::gtile::pos(*L, lr + 2, lc + 2), v = fp::gtile::vel(*L, lr + 2, lc + 2);
        fp::f3 xn, vn;
        fp::integrate1<M>(P, P.mass, p.x, v.x, F[0], xn.x, vn.x);
        fp::integrate1<M>(P, P.mass, p.y, v.y, F[1], xn.y, vn.y);
        fp::integrate1<M>(P, P.mass, p.z, v.z, F[2], xn.z, vn.z);
        if (pin) { xn = p; vn = v; }
        const float nw[6] = {xn.x, xn.y, xn.z, vn.x, vn.y, vn.z};
        for (int q = 0; q < 6; ++q) out[q][i] = nw[q];
        if (A.force_init) for (int q = 0; q < 3; ++q) force[q][i] = 0.0f;
      }
    }
}

}  // namespace

extern "C" {

// The arguments of fast_emul.cpp's emul_fast (there is one tile shape, 8x8).
int emul_fast(uint32_t rows, uint32_t cols, float spacing, const float* position, const float* kc6, const float* state,
              float* out, float* forces, int32_t force_init, const uint32_t* pins, int32_t integration,
              const float* cfg, int32_t mode, int32_t shape) {
  const uint32_t n = rows * cols;
  fp::ClothView G{};
  G.base = 0;
  G.rows = rows;
  G.cols = cols;
  G.spacing = spacing;
  G.cx = (float)cols / 2.0f * spacing;
  G.cy = (float)rows / 2.0f * spacing;
  G.p0 = position[0];
  G.p1 = position[1];
  G.tk = kc6[0]; G.tc = kc6[1]; G.sk = kc6[2]; G.sc = kc6[3]; G.bk = kc6[4]; G.bc = kc6[5];
  fp::StepParams P{};
  P.integration = integration;
  P.dt = cfg[0];
  P.dt_half = cfg[0] * 0.5f;
  P.dt6 = cfg[0] / 6.0f;
  P.dt3 = cfg[0] / 3.0f;
  P.dt_d = cfg[1];
  P.gravity = fp::f3{cfg[2], cfg[3], cfg[4]};
  P.wind = fp::f3{cfg[5], cfg[6], cfg[7]};
  P.neg_drag = -1.0f * cfg[8];
  P.neg_lift = -1.0f * cfg[9];
  P.restitution = cfg[10];
  P.friction = cfg[11];
  P.mass = cfg[12];
  P.uniform_mass = 1;
  // every plane in an allocation of its own, so that an address sanitizer reports any access past
  // a plane's end (one contiguous buffer would hide such a read in the next plane)
  std::vector<std::vector<float>> in(6), o(6, std::vector<float>(n)), f(3);
  for (int k = 0; k < 6; ++k) in[k].assign(state + (size_t)k * n, state + (size_t)(k + 1) * n);
  for (int k = 0; k < 3; ++k) f[k].assign(forces + (size_t)k * n, forces + (size_t)(k + 1) * n);
  std::vector<uint32_t> pin_words;
  if (pins) pin_words.assign(pins, pins + (n + 31) / 32);
  fp::StepArgs A{};
  A.in = fp::SoA{in[0].data(), in[1].data(), in[2].data(), in[3].data(), in[4].data(), in[5].data()};
  A.out = fp::SoA{o[0].data(), o[1].data(), o[2].data(), o[3].data(), o[4].data(), o[5].data()};
  A.fx = f[0].data();
  A.fy = f[1].data();
  A.fz = f[2].data();
  A.pins = pins ? pin_words.data() : nullptr;
  A.force_init = force_init;
  A.obs = fp::ObsView{};
  (void)shape;
  run(A, G, P, mode);
  for (int k = 0; k < 6; ++k) std::copy(o[k].begin(), o[k].end(), out + (size_t)k * n);
  for (int k = 0; k < 3; ++k) std::copy(f[k].begin(), f[k].end(), forces + (size_t)k * n);
  return 0;
}

}  // extern "C"
