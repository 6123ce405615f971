// gfx950 kernels of the learned large-step surrogate: per-vertex features, the fused bf16 MFMA
// inference kernel, the big-step update, step diagnostics and training-sample generation (the
// training kernels are in surrogate_train.hip).
#include "surrogate_device.hpp"

#include <type_traits>

#pragma clang fp contract(fast)

namespace fp {

namespace {

__device__ __forceinline__ void store_state(const SoA& o, uint32_t i, f3 x, f3 v) {
  o.x[i] = x.x; o.y[i] = x.y; o.z[i] = x.z;
  o.vx[i] = v.x; o.vy[i] = v.y; o.vz[i] = v.z;
}

// The 6 features of one slot: strain_scale * strain * d/|d| and (v_nbr - v) * H / L, from the
// neighbour's position q and velocity w; zeros when `has` is false.  Branch-free, so that a caller
// can issue every load of a pass before the first feature is computed.  The short root is exact but for
// d2 < 2^-96, where it may be an ulp off, and for a subnormal d2, |d| < 1.1e-19, where it gives NaN: a caller
// without GENERAL looks for that in its results.
template <bool GENERAL>
__device__ __forceinline__ void slot_feat_from(f3 p, f3 v, f3 q, f3 w, float rest, bool has, FeatParams fp, float* f) {
  const f3 d = sub(q, p);
  const float d2 = d.x * d.x + d.y * d.y + d.z * d.z;
  const float len = GENERAL ? sqrt_rn(d2) : sqrt_in_range(d2);
  const float il = __builtin_amdgcn_rcpf(rest);
  const float st = (has && d2 > 0.0f) ? fp.strain_scale * ((len - rest) * il) * __builtin_amdgcn_rcpf(len) : 0.0f;
  const float hv = has ? fp.H * il : 0.0f;
  f[0] = st * d.x; f[1] = st * d.y; f[2] = st * d.z;
  f[3] = (w.x - v.x) * hv; f[4] = (w.y - v.y) * hv; f[5] = (w.z - v.z) * hv;
}

template <bool GENERAL = true>
__device__ __forceinline__ void slot_feat(const SoA& S, f3 p, f3 v, uint32_t self, SlotEnt e, FeatParams fp,
                                          float* f) {
  const bool has = e.nbr != kNoSlot;
  const uint32_t nb = has ? e.nbr : self;
  slot_feat_from<GENERAL>(p, v, ld3(S.x, S.y, S.z, nb), ld3(S.vx, S.vy, S.vz, nb), has ? e.rest : 1.0f, has, fp, f);
}

__device__ __forceinline__ float unit_open(uint64_t h) { return ((float)(h >> 40) + 0.5f) * (1.0f / 16777216.0f); }

// ---------------------------------------------------------------------------------------------
// Inference: a workgroup takes a contiguous run of units, NT MFMA column tiles of 16 vertices, one
// unit a wave at a time (NT = 2: 16 waves of 32 vertices, 4 waves per SIMD within 128 registers; NT =
// 4: 8 waves of 64).  The units are shared out evenly, so that in the last round every CU has a part
// of its waves busy and not some CUs all of them, and few units are one to a CU.  Bound by the vector
// instructions (768 of a unit's 1,400 are the activation): 330,880 vertices 45.3 us where whole passes
// of 512 vertices a workgroup took 54.0, 1,024 vertices 11.2 (17.1), 1,048,576 vertices 125 (127.5).
// Neurons are the MFMA rows, vertices the columns, so a layer's f32 output tile already holds, per
// lane, 4 consecutive neurons of one vertex; two such tiles form the next layer's 8-element bf16
// operand once the weights' K index is permuted the same way (done when the image is packed).  The
// activations never leave registers; the weights stay in LDS for the whole (persistent) launch.


// One layer, acc = W B + bias then the activation, pipelined by output block: the 16 neurons of
// block mt accumulate (KB MFMAs per column tile, the bias as the accumulators' initial value)
// while the activation of block mt - 1 is evaluated, so that each wave keeps the matrix cores and
// the vector ALUs busy together; two accumulator blocks are live instead of eight.  `out` must not
// alias `B`, which is read until the last block.
template <int KB, int LDW, int NT>
__device__ __forceinline__ void mfma_act_layer(const __bf16* __restrict__ W, const float* __restrict__ bias,
                                               const bf16x8 (&B)[KB][NT], bf16x8 (&out)[4][NT], int col, int g) {
  f32x4 acc[2][NT];
#pragma unroll
  for (int mt = 0; mt <= 8; ++mt) {
    if (mt < 8) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(bias + 16 * mt + 4 * g);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt & 1][nt] = b;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(W + (16 * mt + col) * LDW + kb * 32 + g * 8);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt & 1][nt] = mfma(a, B[kb][nt], acc[mt & 1][nt]);
      }
    }
    if (mt > 0) {
      const int p = mt - 1;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[p >> 1][nt][(p & 1) * 4 + r] = (__bf16)gelu(acc[p & 1][nt][r]);
    }
  }
}

template <int NT>
__global__ void __launch_bounds__(2048 / NT) sur_mlp_kernel(SoA S, const SlotEnt* __restrict__ slots, uint32_t n,
                                                            const uint4* __restrict__ image, FeatParams fp,
                                                            float out_scale, float* __restrict__ da) {
  constexpr int kThreads = 2048 / NT;
  __shared__ uint4 s_img[kImgBytes / 16];
  for (int i = threadIdx.x; i < kImgBytes / 16; i += kThreads) s_img[i] = image[i];
  __syncthreads();
  const char* img = reinterpret_cast<const char*>(s_img);
  const __bf16* W1 = reinterpret_cast<const __bf16*>(img + kImgW1);
  const __bf16* W2 = reinterpret_cast<const __bf16*>(img + kImgW2);
  const __bf16* W3 = reinterpret_cast<const __bf16*>(img + kImgW3);
  const __bf16* W4 = reinterpret_cast<const __bf16*>(img + kImgW4);
  const float* Bias = reinterpret_cast<const float*>(img + kImgB);
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t units = (n + 16 * NT - 1) / (16 * NT);
  const uint32_t u0 = (uint32_t)((uint64_t)blockIdx.x * units / gridDim.x);
  const uint32_t u1 = (uint32_t)((uint64_t)(blockIdx.x + 1) * units / gridDim.x);
  for (uint32_t r0 = u0; r0 < u1; r0 += kThreads / 64) {
    if (r0 + wave >= u1) continue;
    const uint32_t v0 = (r0 + wave) * 16 * NT;
    // One unit; false where its outputs are not all numbers and were not stored.
    const auto unit = [&](auto general) {
      constexpr bool kGeneral = decltype(general)::value;
      // features: lane group g computes slots 3g..3g+2 of its vertex (18 values, then 6 zeros), which
      // are its 8-element K slices of the three 32-wide K blocks of layer 1.  Every load is
      // unconditional (past-the-end columns read vertex n-1, empty slots the vertex itself; both are
      // zeroed), so a pass's loads can all be in flight together.
      bf16x8 B1[3][NT];
      SlotEnt se[NT][3];
      f3 p[NT], v[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const uint32_t iv = v0 + nt * 16 + col;
        const uint32_t i = iv < n ? iv : n - 1;
        const SlotEnt* at = slots + slot_at(i, 3 * g);
        p[nt] = ld3(S.x, S.y, S.z, i);
        v[nt] = ld3(S.vx, S.vy, S.vz, i);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          se[nt][j] = at[64 * j];
          se[nt][j].nbr = iv < n ? se[nt][j].nbr : kNoSlot;
        }
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const uint32_t iv = v0 + nt * 16 + col;
        const uint32_t i = iv < n ? iv : n - 1;
        float f[24];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          slot_feat<kGeneral>(S, p[nt], v[nt], i, se[nt][j], fp, f + 6 * j);
          __builtin_amdgcn_sched_barrier(0x20);  // loads may pass, arithmetic not: slots interleaved spill
        }
#pragma unroll
        for (int k = 18; k < 24; ++k) f[k] = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 3; ++kb)
#pragma unroll
          for (int s = 0; s < 8; ++s) B1[kb][nt][s] = (__bf16)f[kb * 8 + s];
      }
      bf16x8 Bh[4][NT], Bg[4][NT];
      mfma_act_layer<3, kLd1, NT>(W1, Bias, B1, Bh, col, g);
      mfma_act_layer<4, kLd, NT>(W2, Bias + kHid, Bh, Bg, col, g);
      mfma_act_layer<4, kLd, NT>(W3, Bias + 2 * kHid, Bg, Bh, col, g);
      f32x4 o[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) o[nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(W4 + col * kLd + kb * 32 + g * 8);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) o[nt] = mfma(a, Bh[kb][nt], o[nt]);
      }
      if constexpr (!kGeneral) {
        bool number = true;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) number = number && o[nt][0] == o[nt][0];
        if (!__all(number)) return false;
      }
      if (g == 0) {
        const float b0 = Bias[3 * kHid], b1 = Bias[3 * kHid + 1], b2 = Bias[3 * kHid + 2];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const uint32_t i = v0 + nt * 16 + col;
          if (i < n) {
            da[3 * (size_t)i] = out_scale * (o[nt][0] + b0);
            da[3 * (size_t)i + 1] = out_scale * (o[nt][1] + b1);
            da[3 * (size_t)i + 2] = out_scale * (o[nt][2] + b2);
          }
        }
      }
      return true;
    };
    // A strut with a subnormal squared length has NaN for features with the short root, and one NaN
    // feature makes every output of its vertex NaN: only such units (and those whose states are not
    // numbers) are evaluated again, with the general root, and the others pay a compare a tile.
    if (!unit(std::false_type{})) unit(std::true_type{});
  }
}

// ---------------------------------------------------------------------------------------------
// Big-step update: a = (gravity + face forces [+ strut forces]) / m + da; v' = v + H a;
// x' = x + H v'; then the obstacle first-hit test and the reference's collision response over the
// step H, and pinned vertices keep their record.  `work` receives each vertex's face-force work
// F_face . (x' - x), for the energy balance of the diagnostics.
template <bool STRUTS>
__global__ void __launch_bounds__(kBlock) sur_integrate_kernel(StepArgs A, CsrView T, const BlockRange* __restrict__ blocks,
                                                                const float* __restrict__ da, float* __restrict__ work) {
  const BlockRange br = blocks[blockIdx.x];
  const uint32_t i = br.begin + threadIdx.x;
  if (i >= br.end) return;
  const StepParams P = A.params[br.mesh];
  const SoA& S = A.in;
  const f3 p = ld3(S.x, S.y, S.z, i);
  const f3 v = ld3(S.vx, S.vy, S.vz, i);
  if (pinned(A.pins, i)) {
    store_state(A.out, i, p, v);
    work[i] = 0.0f;
    return;
  }
  const float m = P.uniform_mass ? P.mass : A.mass[i];
  f3 Ff = f3{0.0f, 0.0f, 0.0f};
  for (uint32_t e = 0, nf = T.f_cnt[i]; e < nf; ++e) {
    const float4 fc = T.face_c[T.f_first[i] + kSlice * e];
    Ff = add(Ff, f3{fc.x, fc.y, fc.z});
  }
  f3 Fs = f3{0.0f, 0.0f, 0.0f};
  if (STRUTS)
    for (uint32_t e = 0, ns = T.s_cnt[i]; e < ns; ++e) {
      const StrutEnt se = T.s_ent[T.s_first[i] + kSlice * e];
      strut_accumulate<FastMath>(Fs, p, v, ld3(S.x, S.y, S.z, se.nbr), ld3(S.vx, S.vy, S.vz, se.nbr), se.k, se.c,
                                 se.len);
    }
  const f3 d = f3{da[3 * (size_t)i], da[3 * (size_t)i + 1], da[3 * (size_t)i + 2]};
  f3 xn, vn;
  const float w = sur_update(P, A.obs, m, p, v, Ff, Fs, d, xn, vn);
  store_state(A.out, i, xn, vn);
  work[i] = w;
}

// ---------------------------------------------------------------------------------------------
// Diagnostics of a big step over the vertices of `blocks`: the largest change of any strut strain
// (each strut seen from both ends; NaN propagates), energies before and after (kinetic, spring
// with each strut counted half from each end, gravity potential -F_g . x), the face-force work
// subtracted from the energy after.  Bound by the slots' bytes (12 for each of a cloth's ten) and the
// vector instructions (696 a vertex); 330,880 vertices: 17.5 us, 23.7 before the slots were sliced, one
// group of them held at a time and the roots short.
__global__ void __launch_bounds__(kBlock) sur_diag_kernel(SoA I, SoA O, const SlotEnt* __restrict__ slots,
                                                           const float* __restrict__ slot_k,
                                                           const StepParams* __restrict__ params,
                                                           const float* __restrict__ mass, const float* __restrict__ work,
                                                           const BlockRange* __restrict__ blocks,
                                                           const MeshSlots* __restrict__ meshes,
                                                           DiagOut* __restrict__ out) {
  __shared__ float s_ds[kBlock], s_eo[kBlock], s_en[kBlock], s_em[kBlock];
  const BlockRange br = blocks[blockIdx.x];
  const uint32_t iv = br.begin + threadIdx.x;
  const bool valid = iv < br.end;
  const uint32_t i = valid ? iv : br.begin;
  float ds = 0.0f, eo = 0.0f, en = 0.0f, em = 0.0f;
  {
    const StepParams P = params[br.mesh];
    const float m = P.uniform_mass ? P.mass : mass[i];
    const f3 po = ld3(I.x, I.y, I.z, i), pn = ld3(O.x, O.y, O.z, i);
    const f3 vo = ld3(I.vx, I.vy, I.vz, i), vn = ld3(O.vx, O.vy, O.vz, i);
    // five slots at a time (a cloth's vertex has ten): their entries, then their neighbours' positions
    // (empty slots read the vertex itself), so the loads are in flight together
    constexpr int kGroup = 5;
    float so = 0.0f, sn = 0.0f;
    const int n_slots = (int)meshes[br.mesh].n_slots;
#pragma unroll 1
    for (int j0 = 0; j0 < n_slots; j0 += kGroup) {
      SlotEnt e[kGroup];
      float k[kGroup];
#pragma unroll
      for (int j = 0; j < kGroup; ++j) {
        const bool any = j0 + j < kSlots;
        e[j] = slots[slot_at(i, any ? j0 + j : 0)];
        k[j] = slot_k[slot_at(i, any ? j0 + j : 0)];
        if (!any) e[j].nbr = kNoSlot;
      }
      float o2[kGroup], n2[kGroup], lo[kGroup], ln[kGroup];
      uint32_t far = 0;
#pragma unroll
      for (int j = 0; j < kGroup; ++j) {
        const bool has = e[j].nbr != kNoSlot;
        const uint32_t nb = has ? e[j].nbr : i;
        const f3 d_o = sub(ld3(I.x, I.y, I.z, nb), po), d_n = sub(ld3(O.x, O.y, O.z, nb), pn);
        o2[j] = has ? dot(d_o, d_o) : 1.0f;
        n2[j] = has ? dot(d_n, d_n) : 1.0f;
        lo[j] = sqrt_in_range(o2[j]);
        ln[j] = sqrt_in_range(n2[j]);
        far = max(far, max(__float_as_uint(o2[j]) - __float_as_uint(0x1p-96f), __float_as_uint(n2[j]) - __float_as_uint(0x1p-96f)));
      }
      if (far > __float_as_uint(3.40282347e38f) - __float_as_uint(0x1p-96f)) {
#pragma unroll
        for (int j = 0; j < kGroup; ++j) {
          lo[j] = sqrt_rn(o2[j]);
          ln[j] = sqrt_rn(n2[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < kGroup; ++j) {
        const bool has = e[j].nbr != kNoSlot;
        const float r = has ? e[j].rest : 1.0f;
        const float xo = lo[j] - r, xn = ln[j] - r;
        const float d = has ? __builtin_fabsf(xn - xo) * __builtin_amdgcn_rcpf(r) : 0.0f;
        ds = (d > ds || d != d) ? d : ds;
        const float kk = has ? 0.25f * k[j] : 0.0f;
        so += kk * xo * xo;
        sn += kk * xn * xn;
      }
    }
    const float ko = 0.5f * m * dot(vo, vo), kn = 0.5f * m * dot(vn, vn);
    em = ko + so + kn + sn;
    eo = ko + so - dot(P.gravity, po);
    en = kn + sn - dot(P.gravity, pn) - work[i];
    if (!valid) ds = eo = en = em = 0.0f;
  }
  s_ds[threadIdx.x] = ds; s_eo[threadIdx.x] = eo; s_en[threadIdx.x] = en; s_em[threadIdx.x] = em;
  __syncthreads();
  static_assert(kBlock == 256, "four wavefronts");
  // the pairs of a halving tree over the workgroup: two levels from memory, six within a wavefront
  if (threadIdx.x >= 64) return;
  const uint32_t t = threadIdx.x;
  const auto worse = [](float a, float b) { return (b > a || b != b) ? b : a; };
  ds = worse(worse(s_ds[t], s_ds[t + 128]), worse(s_ds[t + 64], s_ds[t + 192]));
  eo = (s_eo[t] + s_eo[t + 128]) + (s_eo[t + 64] + s_eo[t + 192]);
  en = (s_en[t] + s_en[t + 128]) + (s_en[t + 64] + s_en[t + 192]);
  em = (s_em[t] + s_em[t + 128]) + (s_em[t + 64] + s_em[t + 192]);
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) {
    ds = worse(ds, __shfl_down(ds, w));
    eo += __shfl_down(eo, w);
    en += __shfl_down(en, w);
    em += __shfl_down(em, w);
  }
  if (t == 0) out[blockIdx.x] = DiagOut{ds, eo, en, em};
}

// The blocks' diagnostics of one mesh a workgroup.
__global__ void __launch_bounds__(kBlock) sur_mesh_diag_kernel(const DiagOut* __restrict__ part,
                                                                const MeshSlots* __restrict__ meshes,
                                                                MeshDiag* __restrict__ out) {
  __shared__ double s_e[3][kBlock];
  __shared__ float s_ds[kBlock];
  const MeshSlots R = meshes[blockIdx.x];
  const uint32_t t = threadIdx.x;
  double e[3] = {0.0, 0.0, 0.0};
  float ds = 0.0f;
  for (uint32_t b = R.blk_begin + t; b < R.blk_end; b += kBlock) {
    const DiagOut d = part[b];
    ds = (d.max_dstrain > ds || d.max_dstrain != d.max_dstrain) ? d.max_dstrain : ds;
    e[0] += d.e_old;
    e[1] += d.e_new;
    e[2] += d.emech_old;
  }
  s_ds[t] = ds;
  for (int k = 0; k < 3; ++k) s_e[k][t] = e[k];
  __syncthreads();
  for (uint32_t w = kBlock / 2; w > 0; w >>= 1) {
    if (t < w) {
      const float b = s_ds[t + w];
      s_ds[t] = (b > s_ds[t] || b != b) ? b : s_ds[t];
      for (int k = 0; k < 3; ++k) s_e[k][t] += s_e[k][t + w];
    }
    __syncthreads();
  }
  if (t == 0) out[blockIdx.x] = MeshDiag{s_e[0][0], s_e[1][0], s_e[2][0], s_ds[0], 0.0f};
}

// Health of the plain trajectories that feed training: per block, the largest of |v| / vmax and
// strain / smax over its vertices (NaN and infinities count as unhealthy: the result is then +inf).
__global__ void __launch_bounds__(kBlock) sur_health_kernel(SoA S, const SlotEnt* __restrict__ slots,
                                                             const BlockRange* __restrict__ blocks, float vmax,
                                                             float smax, float* __restrict__ out) {
  __shared__ float s_h[kBlock];
  const BlockRange br = blocks[blockIdx.x];
  const uint32_t i = br.begin + threadIdx.x;
  float h = 0.0f;
  if (i < br.end) {
    const f3 p = ld3(S.x, S.y, S.z, i), v = ld3(S.vx, S.vy, S.vz, i);
    h = __builtin_sqrtf(dot(v, v)) / vmax;
    for (int j = 0; j < kSlots; ++j) {
      const SlotEnt e = slots[slot_at(i, j)];
      if (e.nbr == kNoSlot) continue;
      const f3 d = sub(ld3(S.x, S.y, S.z, e.nbr), p);
      h = fmaxf(h, __builtin_fabsf(__builtin_sqrtf(dot(d, d)) - e.rest) / (e.rest * smax));
    }
    if (!(h <= 3.0e38f)) h = __builtin_inff();
  }
  s_h[threadIdx.x] = h;
  __syncthreads();
  for (int w = kBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s_h[threadIdx.x] = fmaxf(s_h[threadIdx.x], s_h[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = s_h[0];
}

__global__ void __launch_bounds__(kBlock) sur_features_kernel(SoA S, const SlotEnt* __restrict__ slots,
                                                               const uint32_t* __restrict__ ids, uint32_t n,
                                                               FeatParams fp, float* __restrict__ out) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= n) return;
  const uint32_t i = ids[j];
  const f3 p = ld3(S.x, S.y, S.z, i), v = ld3(S.vx, S.vy, S.vz, i);
  for (int s = 0; s < kSlots; ++s) slot_feat(S, p, v, i, slots[slot_at(i, s)], fp, out + (size_t)j * kFeat + 6 * s);
}

__global__ void __launch_bounds__(kBlock) sur_noise_kernel(Pos3 prev, Pos3 cur, SoA o, const uint32_t* __restrict__ pins,
                                                            uint32_t n, float H, float sigma, uint64_t seed) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float e[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  if (sigma > 0.0f && !pinned(pins, i)) {
    for (int k = 0; k < 3; ++k) {
      const uint64_t h = mix64(seed ^ mix64(((uint64_t)i << 3) | (uint64_t)k));
      const float r = sigma * sqrtf(-2.0f * logf(unit_open(h))), th = 6.283185307179586f * unit_open(mix64(h));
      e[2 * k] = r * cosf(th);
      e[2 * k + 1] = r * sinf(th);
    }
  }
  const float xb = cur.x[i] + e[0], yb = cur.y[i] + e[1], zb = cur.z[i] + e[2];
  const float xp = prev.x[i] + e[3], yp = prev.y[i] + e[4], zp = prev.z[i] + e[5];
  const float iH = 1.0f / H;
  o.x[i] = xb; o.y[i] = yb; o.z[i] = zb;
  o.vx[i] = (xb - xp) * iH; o.vy[i] = (yb - yp) * iH; o.vz[i] = (zb - zp) * iH;
}

template <bool STRUTS>
__global__ void __launch_bounds__(kBlock) sur_samples_kernel(StepArgs A, CsrView T, const uint32_t* __restrict__ ids,
                                                              const uint32_t* __restrict__ mesh_of, uint32_t n, Pos3 nx,
                                                              const SlotEnt* __restrict__ slots, FeatParams fp,
                                                              float out_scale, __bf16* __restrict__ X,
                                                              float* __restrict__ Tg) {
  const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= n) return;
  const uint32_t i = ids[j];
  const StepParams P = A.params[mesh_of[i]];
  const SoA& S = A.in;
  const f3 p = ld3(S.x, S.y, S.z, i), v = ld3(S.vx, S.vy, S.vz, i);
  float f[kFeat];
  bool ok = true;
  for (int s = 0; s < kSlots; ++s) slot_feat(S, p, v, i, slots[slot_at(i, s)], fp, f + 6 * s);
  for (int c = 0; c < kFeat; ++c) ok = ok && __builtin_isfinite(f[c]);
  const float m = P.uniform_mass ? P.mass : A.mass[i];
  f3 F = P.gravity;
  for (uint32_t e = 0, nf = T.f_cnt[i]; e < nf; ++e) {
    const float4 fc = T.face_c[T.f_first[i] + kSlice * e];
    F = add(F, f3{fc.x, fc.y, fc.z});
  }
  if (STRUTS)
    for (uint32_t e = 0, ns = T.s_cnt[i]; e < ns; ++e) {
      const StrutEnt se = T.s_ent[T.s_first[i] + kSlice * e];
      strut_accumulate<FastMath>(F, p, v, ld3(S.x, S.y, S.z, se.nbr), ld3(S.vx, S.vy, S.vz, se.nbr), se.k, se.c, se.len);
    }
  const float H = fp.H, iH = 1.0f / H, iH2 = iH * iH, im = 1.0f / m, is = 1.0f / out_scale;
  float t[3] = {((nx.x[i] - p.x) * iH2 - v.x * iH - F.x * im) * is, ((nx.y[i] - p.y) * iH2 - v.y * iH - F.y * im) * is,
                ((nx.z[i] - p.z) * iH2 - v.z * iH - F.z * im) * is};
  for (int c = 0; c < 3; ++c) ok = ok && __builtin_isfinite(t[c]);
  // a non-finite sample (from a trajectory the health check has not yet dropped) becomes a zero row
  for (int c = 0; c < kFeat; ++c) X[(size_t)j * kFeat + c] = (__bf16)(ok ? f[c] : 0.0f);
  for (int c = 0; c < 3; ++c) Tg[3 * (size_t)j + c] = ok ? t[c] : 0.0f;
}

__global__ void __launch_bounds__(kBlock) to_bf16_kernel(const float* __restrict__ in, __bf16* __restrict__ out, long n) {
  const long i = (long)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) out[i] = (__bf16)in[i];
}

inline unsigned blocks_for(long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

hipError_t launch_sur_mlp(const SoA& st, const SlotEnt* slots, uint32_t n, const void* image, FeatParams fp,
                          float out_scale, float* da, int grid, int variant, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const uint32_t units = (n + 16 * variant - 1) / (16 * variant);
  const dim3 g((uint32_t)grid < units ? (uint32_t)grid : units);
  if (variant == 4)
    hipLaunchKernelGGL(sur_mlp_kernel<4>, g, dim3(512), 0, s, st, slots, n, reinterpret_cast<const uint4*>(image), fp,
                       out_scale, da);
  else
    hipLaunchKernelGGL(sur_mlp_kernel<2>, g, dim3(1024), 0, s, st, slots, n, reinterpret_cast<const uint4*>(image), fp,
                       out_scale, da);
  return hipGetLastError();
}

hipError_t launch_sur_integrate(const StepArgs& a, const CsrView& t, const BlockRange* blocks, uint32_t n_blocks,
                                const float* da, float* work, bool struts, hipStream_t s) {
  if (n_blocks == 0) return hipSuccess;
  if (struts)
    hipLaunchKernelGGL(sur_integrate_kernel<true>, dim3(n_blocks), dim3(kBlock), 0, s, a, t, blocks, da, work);
  else
    hipLaunchKernelGGL(sur_integrate_kernel<false>, dim3(n_blocks), dim3(kBlock), 0, s, a, t, blocks, da, work);
  return hipGetLastError();
}

hipError_t launch_sur_diag(const SoA& in, const SoA& out, const SlotEnt* slots, const float* slot_k,
                           const StepParams* params, const float* mass, const float* work, const BlockRange* blocks,
                           uint32_t n_blocks, const MeshSlots* meshes, uint32_t n_meshes, DiagOut* diag,
                           MeshDiag* per_mesh, hipStream_t s) {
  if (n_blocks)
    hipLaunchKernelGGL(sur_diag_kernel, dim3(n_blocks), dim3(kBlock), 0, s, in, out, slots, slot_k, params, mass, work,
                       blocks, meshes, diag);
  if (n_meshes) hipLaunchKernelGGL(sur_mesh_diag_kernel, dim3(n_meshes), dim3(kBlock), 0, s, diag, meshes, per_mesh);
  return hipGetLastError();
}

hipError_t launch_sur_health(const SoA& st, const SlotEnt* slots, const BlockRange* blocks, uint32_t n_blocks,
                             float vmax, float smax, float* out, hipStream_t s) {
  if (n_blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(sur_health_kernel, dim3(n_blocks), dim3(kBlock), 0, s, st, slots, blocks, vmax, smax, out);
  return hipGetLastError();
}

hipError_t launch_sur_features(const SoA& st, const SlotEnt* slots, const uint32_t* ids, uint32_t n, FeatParams fp,
                               float* out, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(sur_features_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, st, slots, ids, n, fp, out);
  return hipGetLastError();
}

hipError_t launch_sur_noise(Pos3 prev, Pos3 cur, SoA noisy, const uint32_t* pins, uint32_t n, float H, float sigma,
                            uint64_t seed, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(sur_noise_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, prev, cur, noisy, pins, n, H, sigma,
                     seed);
  return hipGetLastError();
}

hipError_t launch_sur_samples(const StepArgs& a, const CsrView& t, const uint32_t* ids, const uint32_t* mesh_of,
                              uint32_t n, Pos3 next, const SlotEnt* slots, FeatParams fp, float out_scale, bool struts,
                              __bf16* X, float* T, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (struts)
    hipLaunchKernelGGL(sur_samples_kernel<true>, dim3(blocks_for(n)), dim3(kBlock), 0, s, a, t, ids, mesh_of, n, next,
                       slots, fp, out_scale, X, T);
  else
    hipLaunchKernelGGL(sur_samples_kernel<false>, dim3(blocks_for(n)), dim3(kBlock), 0, s, a, t, ids, mesh_of, n, next,
                       slots, fp, out_scale, X, T);
  return hipGetLastError();
}

hipError_t launch_to_bf16(const float* in, __bf16* out, long n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n)), dim3(kBlock), 0, s, in, out, n);
  return hipGetLastError();
}

}  // namespace fp
