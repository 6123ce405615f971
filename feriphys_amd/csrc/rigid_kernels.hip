// The rigid-body step (rigidbody/simulation.rs:26-52) for a batch of unit cubes, one thread per
// body, in the reference's operation order (no FMA contraction; correctly rounded division and
// square root):
//   accumulate_forces / accumulate_torques (rigidbody.rs:322-328);
//   State::rk4_step or euler_step over the body's 29-float record (state.rs:75-106), whose
//     derivative (rigidbody.rs:94-157) is (p / m, 0.5 (0, w) q, F, tau, 0...) with
//     w = (R I0^-1 R^T) L and R = Matrix3::from(q);
//   normalize_rotation (:29-31);
//   update_state (:257-319): each of the cube's 8 vertices, old and new world positions, the first
//     obstacle face its segment crosses (CollidableMesh::get_collided_face_from_list), and the
//     reference's impulse response on the new state;
//   clear_forces / clear_torques (:330-336).
// cgmath's quaternion and matrix operations are restated below with their component order.
#include "rigid.hpp"

namespace fp {

namespace {

struct Q {
  float s;
  f3 v;
};
// Quaternion * Quaternion (Hamilton product), each component summed left to right.
__device__ __forceinline__ Q qmul(Q a, Q b) {
  return Q{a.s * b.s - a.v.x * b.v.x - a.v.y * b.v.y - a.v.z * b.v.z,
           f3{a.s * b.v.x + a.v.x * b.s + a.v.y * b.v.z - a.v.z * b.v.y,
              a.s * b.v.y + a.v.y * b.s + a.v.z * b.v.x - a.v.x * b.v.z,
              a.s * b.v.z + a.v.z * b.s + a.v.x * b.v.y - a.v.y * b.v.x}};
}
struct M3 {
  f3 c[3];  // columns
};
__device__ __forceinline__ f3 row(const M3& m, int i) {
  return i == 0 ? f3{m.c[0].x, m.c[1].x, m.c[2].x} : i == 1 ? f3{m.c[0].y, m.c[1].y, m.c[2].y}
                                                             : f3{m.c[0].z, m.c[1].z, m.c[2].z};
}
// Matrix3 * Vector3: row(i) . v
__device__ __forceinline__ f3 mv(const M3& m, f3 v) { return f3{dot(row(m, 0), v), dot(row(m, 1), v), dot(row(m, 2), v)}; }
__device__ __forceinline__ M3 mm(const M3& a, const M3& b) { return M3{{mv(a, b.c[0]), mv(a, b.c[1]), mv(a, b.c[2])}}; }
__device__ __forceinline__ M3 tr(const M3& m) { return M3{{row(m, 0), row(m, 1), row(m, 2)}}; }
// Matrix3::from(Quaternion)
__device__ __forceinline__ M3 from_quat(Q q) {
  const float x2 = q.v.x + q.v.x, y2 = q.v.y + q.v.y, z2 = q.v.z + q.v.z;
  const float xx2 = x2 * q.v.x, xy2 = x2 * q.v.y, xz2 = x2 * q.v.z;
  const float yy2 = y2 * q.v.y, yz2 = y2 * q.v.z, zz2 = z2 * q.v.z;
  const float sy2 = y2 * q.s, sz2 = z2 * q.s, sx2 = x2 * q.s;
  return M3{{f3{1.0f - yy2 - zz2, xy2 + sz2, xz2 - sy2}, f3{xy2 - sz2, 1.0f - xx2 - zz2, yz2 + sx2},
             f3{xz2 + sy2, yz2 - sx2, 1.0f - xx2 - yy2}}};
}
// State::get_moment_of_inertia_inverted (rigidbody.rs:33-36): (R I0^-1) R^T
__device__ __forceinline__ M3 inertia_inv(Q q, const M3& I0) {
  const M3 R = from_quat(q);
  return mm(mm(R, I0), tr(R));
}

// The fields of a record that a step changes; the mass and I0^-1 stay, force and torque are cleared.
struct Body {
  f3 x;
  Q q;
  f3 p, l;  // linear and angular momentum
};
// Stateful::derivative (rigidbody.rs:94-157) of those fields; the momenta's are force and torque.
__device__ __forceinline__ void derivative(const Body& S, float m, const M3& I0, f3& dx, Q& dq, M3& I, f3& w) {
  dx = ExactMath::div3(S.p, m);  // linear_momentum / mass
  I = inertia_inv(S.q, I0);
  w = mv(I, S.l);
  dq = qmul(Q{0.5f * 0.0f, f3{0.5f * w.x, 0.5f * w.y, 0.5f * w.z}}, S.q);
}
// Makes values opaque where they stand: the compiler otherwise interleaves the four stages (the momenta's
// slopes, and so every stage's division, are known from the start) and holds 210 registers.
__device__ __forceinline__ void settle(f3& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z)); }
__device__ __forceinline__ void settle(Q& q) { asm volatile("" : "+v"(q.s), "+v"(q.v.x), "+v"(q.v.y), "+v"(q.v.z)); }
__device__ __forceinline__ void settle(Body& b) { settle(b.x); settle(b.q); settle(b.p); settle(b.l); }
// From the second stage on a -0 in the mass or the inertia has become +0 (every field advances by its
// slope, and theirs is 0); formed anew per stage, not held.
__device__ __forceinline__ void derivative_later(const Body& S, float m, M3 I0, f3& dx, Q& dq) {
  for (int c = 0; c < 3; ++c) {
    settle(I0.c[c]);
    I0.c[c] = add(I0.c[c], f3{0.0f, 0.0f, 0.0f});
  }
  M3 I;
  f3 w;
  derivative(S, m + 0.0f, I0, dx, dq, I, w);
}
// a + s b, per component, as the reference's vec_add and scale round it
__device__ __forceinline__ f3 axpy(f3 a, float s, f3 b) { return f3{a.x + b.x * s, a.y + b.y * s, a.z + b.z * s}; }
__device__ __forceinline__ Q axpy(Q a, float s, Q b) { return Q{a.s + b.s * s, axpy(a.v, s, b.v)}; }

// The world offsets of the cube's corners, R c with c = (+-1/2, +-1/2, +-1/2): with a = R / 2 (exact),
// row by row (+-a0 +- a1) +- a2, where negation is exact but for a zero's sign: corner k is +-(s or d) +- a2
// with s = a0 + a1 and d = a0 - a1.
struct Corners {
  f3 s, d, a;
};
// An offset that cancels to zero is +0 in the reference and may be -0 here, which a position of -0 would
// let through into the corner, and from there into the side of a plane: corners are formed at x + 0.
__device__ __forceinline__ f3 at_plus_zero(f3 x) { return add(x, f3{0.0f, 0.0f, 0.0f}); }
__device__ __forceinline__ Corners corners_of(const M3& R) {
  const f3 a0 = smul(0.5f, R.c[0]), a1 = smul(0.5f, R.c[1]);
  return Corners{add(a0, a1), sub(a0, a1), smul(0.5f, R.c[2])};
}
// Corner k of kCubeCorner's order at body position x (of at_plus_zero): the offsets are -(s - a), d + a,
// s + a, -(d - a), -(s + a), d - a, s - a, -(d + a).
__device__ __forceinline__ f3 corner_at(const Corners& C, f3 x, int k) {
  const f3 b = k % 2 == 0 ? C.s : C.d;
  const bool minus = k == 0 || k == 3 || k == 5 || k == 6, negative = k == 0 || k == 3 || k == 4 || k == 7;
  const f3 v = minus ? sub(b, C.a) : add(b, C.a);
  return negative ? sub(x, v) : add(v, x);
}
// The same for a corner number of each lane's own, by selects and sign flips (b - a is b + (-a), x - v is
// (-v) + x).
__device__ __forceinline__ f3 corner_of_lane(const Corners& C, f3 x, uint32_t k) {
  const bool even = (k & 1u) == 0u;
  const uint32_t minus = (0x69u >> k & 1u) << 31, negative = (0x99u >> k & 1u) << 31;
  auto flip = [](float v, uint32_t sign) { return __uint_as_float(__float_as_uint(v) ^ sign); };
  auto one = [&](float s, float d, float a, float xc) { return flip((even ? s : d) + flip(a, minus), negative) + xc; };
  return f3{one(C.s.x, C.d.x, C.a.x, x.x), one(C.s.y, C.d.y, C.a.y, x.y), one(C.s.z, C.d.z, C.a.z, x.z)};
}

// The same as the reference writes it, (r0 c0 + r1 c1) + r2 c2 per row and then + x: for a pose that is not a
// number, where the sign of a NaN decides on which side of a plane the corner is, and the flips above would
// turn it.  Opaque, so that nothing of it is shared with the usual form (171 registers, two waves a SIMD).
__device__ __forceinline__ f3 corner_as_written(Q q, f3 x, uint32_t k) {
  f3 c = f3{0x66u >> k & 1u ? 0.5f : -0.5f, 0xccu >> k & 1u ? 0.5f : -0.5f, k < 4u ? 0.5f : -0.5f};
  settle(q);
  settle(c);
  const M3 R = from_quat(q);
  return add(mv(R, c), x);
}

// Obstacle face f (the same for the whole wave): never written while a kernel runs, so read through the
// constant address space, which puts it in scalar registers.
__device__ __forceinline__ ObsFace uniform_face(const ObsView& O, uint32_t f) {
  const auto* F = (const __attribute__((address_space(4))) ObsFace*)(O.faces + f);
  ObsFace q;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    q.v0[c] = F->v0[c];
    q.v1[c] = F->v1[c];
    q.v2[c] = F->v2[c];
    q.n[c] = F->n[c];
  }
  q.axis = F->axis;
  return q;
}

// Few faces: on which side of each face's plane the eight corners of a pose are, the first test of
// face_hit as it computes it: bit 8 f + k is the sign of corner k's distance from face f.
static_assert(kScanFaces * 8 <= 64, "a bit for each face and corner");
__device__ __forceinline__ uint64_t corner_sides(const ObsView& O, const Corners& C, f3 x) {
  uint64_t sides = 0;
  x = at_plus_zero(x);
  for (uint32_t f = 0; f < O.n_faces; f += 2) {  // two at a time, so that each corner is formed half as often
    // (of an odd number the last one twice)
    const ObsFace F = uniform_face(O, f), G = uniform_face(O, f + 1 < O.n_faces ? f + 1 : f);
    const f3 v0 = f3{F.v0[0], F.v0[1], F.v0[2]}, n = f3{F.n[0], F.n[1], F.n[2]};
    const f3 w0 = f3{G.v0[0], G.v0[1], G.v0[2]}, o = f3{G.n[0], G.n[1], G.n[2]};
    uint32_t side = 0, other = 0;
#pragma unroll
    for (int k = 7; k >= 0; --k) {
      if (k % 2 == 1) settle(x);  // the corners' positions formed as they are needed, not held in 24 registers
      const f3 c = corner_at(C, x, k);
      side = __builtin_amdgcn_alignbit(side, __float_as_uint(dot(sub(c, v0), n)), 31);
      other = __builtin_amdgcn_alignbit(other, __float_as_uint(dot(sub(c, w0), o)), 31);
    }
    sides |= (uint64_t)(side | other << 8) << (8 * f);
  }
  return sides;
}
// The grids: whether any corner can meet an obstacle between the two poses, by the box around all the
// corners against the faces' box.
__device__ __forceinline__ bool near_box(const ObsView& O, const Corners& Co, f3 xo, const Corners& Cn, f3 xn) {
  if (O.n_always != 0) return true;
  // a corner's offset is at most max(|s|, |d|) + |a| in each row
  auto meets = [&](float s0, float d0, float a0, float x0, float s1, float d1, float a1, float x1, float lo, float hi) {
    const float e0 = fmaxf(fabsf(s0), fabsf(d0)) + fabsf(a0), e1 = fmaxf(fabsf(s1), fabsf(d1)) + fabsf(a1);
    // 2 margin: the corners' own test grows by one; the other covers the rounding of these sums (the
    // margin is at least 1e-4 of the largest obstacle coordinate)
    return !(fminf(x0 - e0, x1 - e1) - 2.0f * O.margin > hi) && !(fmaxf(x0 + e0, x1 + e1) + 2.0f * O.margin < lo);
  };
  return meets(Co.s.x, Co.d.x, Co.a.x, xo.x, Cn.s.x, Cn.d.x, Cn.a.x, xn.x, O.box_lo[0], O.box_hi[0]) &&
         meets(Co.s.y, Co.d.y, Co.a.y, xo.y, Cn.s.y, Cn.d.y, Cn.a.y, xn.y, O.box_lo[1], O.box_hi[1]) &&
         meets(Co.s.z, Co.d.z, Co.a.z, xo.z, Cn.s.z, Cn.d.z, Cn.a.z, xn.z, O.box_lo[2], O.box_hi[2]);
}

// The face that a segment hits first (first_hit), and the face itself.
template <bool GRID>
__device__ __forceinline__ bool hit_face(const ObsView& O, f3 op, f3 np, float dt_d, f3& n, f3& v0) {
  if constexpr (!GRID) {
    for (uint32_t f = 0; f < O.n_faces; ++f) {
      const ObsFace F = uniform_face(O, f);
      if (face_hit(F, op, np, dt_d)) {
        n = f3{F.n[0], F.n[1], F.n[2]};
        v0 = f3{F.v0[0], F.v0[1], F.v0[2]};
        return true;
      }
    }
    return false;
  } else {
    const int32_t hit = first_hit(O, op, np, dt_d);
    if (hit < 0) return false;
    const ObsFace& F = O.faces[hit];
    n = f3{F.n[0], F.n[1], F.n[2]};
    v0 = f3{F.v0[0], F.v0[1], F.v0[2]};
    return true;
  }
}

// What a step forms of its poses early and needs again only where a corner hits, in the lane's own words of
// LDS: the old pose's world inertia, angular velocity and velocity, and the corners of both poses (the new
// one's are the next step's old ones).  Held in registers it would cost a third wave a SIMD; formed again
// it was 260 operations a step with a hit.  The clobbers keep it from staying in registers all the same.
struct Kept {
  float4 (*at)[kBlock];
  __device__ float4& word(int k) const { return at[k][threadIdx.x]; }
  __device__ void pose(const M3& I, f3 w, f3 vel) const {
    word(0) = make_float4(I.c[0].x, I.c[0].y, I.c[0].z, w.x);
    word(1) = make_float4(I.c[1].x, I.c[1].y, I.c[1].z, w.y);
    word(2) = make_float4(I.c[2].x, I.c[2].y, I.c[2].z, w.z);
    word(3) = make_float4(vel.x, vel.y, vel.z, 0.0f);
  }
  __device__ void get_pose(M3& I, f3& w, f3& vel) const {
    asm volatile("" ::: "memory");
    const float4 a = word(0), b = word(1), c = word(2), d = word(3);
    I = M3{{f3{a.x, a.y, a.z}, f3{b.x, b.y, b.z}, f3{c.x, c.y, c.z}}};
    w = f3{a.w, b.w, c.w};
    vel = f3{d.x, d.y, d.z};
  }
  __device__ void corners(uint32_t which, const Corners& C) const {
    word(4 + 3 * which) = make_float4(C.s.x, C.s.y, C.s.z, 0.0f);
    word(5 + 3 * which) = make_float4(C.d.x, C.d.y, C.d.z, 0.0f);
    word(6 + 3 * which) = make_float4(C.a.x, C.a.y, C.a.z, 0.0f);
  }
  __device__ Corners get_corners(uint32_t which) const {
    asm volatile("" ::: "memory");
    const float4 s = word(4 + 3 * which), d = word(5 + 3 * which), a = word(6 + 3 * which);
    return Corners{f3{s.x, s.y, s.z}, f3{d.x, d.y, d.z}, f3{a.x, a.y, a.z}};
  }
};

// `steps` steps of every body, one thread per body, the record in registers from the first to the last
// (bodies do not interact) and stored in place: the 13 fields that change, and the others only where
// they hold something else than what the reference leaves there.  Bound by vector issue (~1,250
// operations a body-step in free fall): 1,048,576 cubes 27.6 us a step falling and 39.2 lying on a floor,
// where a launch per step, the record through memory each time and eight obstacle searches a body took
// 71 and 74 (30.4 and 42.7 before the corners' sides and the old pose's values were carried); 131,072
// cubes 4.4 and 7.2 (15.4 and 18.3); below ~20,000, one wave's chain, 3.1 and 5.2.
template <bool GRID>
__global__ void __launch_bounds__(kBlock) rigid_step_kernel(float* __restrict__ rec, uint32_t n, uint32_t pitch,
                                                             RigidParams P, ObsView O, uint32_t steps) {
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
  __shared__ float4 s_kept[10][kBlock];
  const Kept keep{s_kept};
  if (b >= n) return;
  // one coalesced wavefront access: a uniform base per field and a 32-bit byte offset per lane
  auto field = [&](int k) -> float& { return *(float*)((char*)(rec + (size_t)k * pitch) + b * 4u); };
  Body S{f3{field(0), field(1), field(2)}, Q{field(6), f3{field(3), field(4), field(5)}},
         f3{field(7), field(8), field(9)}, f3{field(10), field(11), field(12)}};
  float m = field(13);
  M3 I{{f3{field(14), field(15), field(16)}, f3{field(17), field(18), field(19)}, f3{field(20), field(21), field(22)}}};
  f3 F = f3{field(23), field(24), field(25)}, tau = f3{field(26), field(27), field(28)};
  // cleared at the end of every step: stored only where the record holds something else
  auto bits = [](f3 v) { return __float_as_uint(v.x) | __float_as_uint(v.y) | __float_as_uint(v.z); };
  if (steps != 0 && (bits(F) | bits(tau)) != 0u)
    for (int k = 23; k < kRigidRecord; ++k) field(k) = 0.0f;
  const float h = P.dt;
  // the sides on which a step's last pose left the corners are the next step's old ones
  uint64_t sides = 0;
  if (steps != 0 && O.n_faces != 0) {
    const Corners C = corners_of(from_quat(S.q));
    keep.corners(0, C);
    if (!GRID) sides = corner_sides(O, C, S.x);
  }
  for (uint32_t step = 0; step < steps; ++step) {
    // accumulate_forces, accumulate_torques
    F = add(F, P.gravity);
    tau = add(tau, P.torque);
    Body T;
    f3 dx;
    Q dq;
    {
      M3 I_old;
      f3 w;
      derivative(S, m, I, dx, dq, I_old, w);
      keep.pose(I_old, w, dx);
    }
    const f3 z = f3{0.0f, 0.0f, 0.0f};
    if (P.integration == FP_EULER) {  // S + S' h (state.rs:75-83)
      T = Body{axpy(S.x, h, dx), axpy(S.q, h, dq), axpy(S.p, h, F), axpy(S.l, h, tau)};
    } else {  // state.rs:86-106, delta accumulated left to right
      const float hh = h * 0.5f, h6 = h / 6.0f, h3 = h / 3.0f;
      f3 ax = smul(h6, dx);
      Q aq = Q{h6 * dq.s, smul(h6, dq.v)};
      T = Body{axpy(S.x, hh, dx), axpy(S.q, hh, dq), axpy(S.p, hh, F), axpy(S.l, hh, tau)};
      settle(T); settle(ax); settle(aq);
      derivative_later(T, m, I, dx, dq);
      ax = axpy(ax, h3, dx);
      aq = axpy(aq, h3, dq);
      T = Body{axpy(S.x, hh, dx), axpy(S.q, hh, dq), axpy(S.p, hh, add(F, z)), axpy(S.l, hh, add(tau, z))};
      settle(T); settle(ax); settle(aq);
      derivative_later(T, m, I, dx, dq);
      ax = axpy(ax, h3, dx);
      aq = axpy(aq, h3, dq);
      T = Body{axpy(S.x, h, dx), axpy(S.q, h, dq), axpy(S.p, h, add(F, z)), axpy(S.l, h, add(tau, z))};
      settle(T); settle(ax); settle(aq);
      derivative_later(T, m, I, dx, dq);
      ax = axpy(ax, h6, dx);
      aq = axpy(aq, h6, dq);
      const f3 F2 = add(F, z), tau2 = add(tau, z);
      const f3 ap = axpy(axpy(axpy(smul(h6, F), h3, F2), h3, F2), h6, F2);
      const f3 al = axpy(axpy(axpy(smul(h6, tau), h3, tau2), h3, tau2), h6, tau2);
      T = Body{add(S.x, ax), Q{S.q.s + aq.s, add(S.q.v, aq.v)}, add(S.p, ap), add(S.l, al)};
      settle(T);
    }
    // normalize_rotation: q * (1 / sqrt(s s + v . v)).  A step is odd where that is out of the short forms'
    // range (the test is theirs): every step whose new rotation is NaN is, and so every one whose old was.
    bool odd;
    {
      const float n2 = T.q.s * T.q.s + dot(T.q.v, T.q.v);
      odd = !(n2 >= 0x1p-96f && n2 <= 0x1p96f);
      float root, inv;
      sqrt_rcp_rn(n2, root, inv);
      T.q = Q{T.q.s * inv, f3{T.q.v.x * inv, T.q.v.y * inv, T.q.v.z * inv}};
    }
    // update_state: the cube's vertices against the obstacles
    if (O.n_faces != 0) {
      // the corners (bit k: corner k) that can meet an obstacle: with few faces, those that change sides
      // of some face's plane; with the grids, all or none
      uint32_t near = 0;
      const uint32_t was = step & 1u, is = was ^ 1u;
      {
        const Corners C = corners_of(from_quat(T.q));
        keep.corners(is, C);
        if constexpr (GRID) {
          near = near_box(O, keep.get_corners(was), S.x, C, T.x) ? 0xffu : 0u;
        } else {
          const uint64_t now = corner_sides(O, C, T.x);
          uint64_t crossed = now ^ sides;
          sides = now;
          crossed |= crossed >> 32;
          near = (uint32_t)crossed | (uint32_t)crossed >> 16;
          near = (near | near >> 8) & 0xffu;
        }
      }
      if (odd) near = 0xffu;  // the sides of a NaN's corners say nothing
      if (near != 0) {
        const Corners Co = keep.get_corners(was), Cn = keep.get_corners(is);
        const f3 x_new = T.x;
        // what the response needs of the old pose: once for the few-face scenes, whose marked corners mostly
        // hit, and per hit with the grids, where the search needs the registers
        M3 I_old;
        f3 vel, w;
        if (!GRID) keep.get_pose(I_old, w, vel);
        bool moved = false;
        // each lane its own marked corners in ascending order: as many rounds as the body with the most
        // has, not eight
        while (near != 0) {
          const uint32_t k = (uint32_t)__builtin_ctz(near);
          near &= near - 1u;
          f3 op, np;
          if (__builtin_expect(odd, 0)) {
            op = corner_as_written(S.q, S.x, k);
            np = corner_as_written(T.q, x_new, k);
          } else {
            op = corner_of_lane(Co, at_plus_zero(S.x), k);
            np = corner_of_lane(Cn, at_plus_zero(x_new), k);
          }
          f3 nrm, v0;
          if (!hit_face<GRID>(O, op, np, P.dt_d, nrm, v0)) continue;
          if (GRID) keep.get_pose(I_old, w, vel);
          const float od = dot(sub(op, v0), nrm), nd = dot(sub(np, v0), nrm);
          const f3 r = sub(op, S.x);
          const float frac = od / (od - nd);
          const f3 cv = add(vel, cross(w, r));
          const f3 cp = add(op, smul(P.dt * frac, cv));
          const float vn = dot(cv, nrm);
          const float j = (-(1.0f + P.restitution) * vn) / (1.0f / m + dot(nrm, mv(I_old, cross(cross(r, nrm), r))));
          const f3 imp = smul(j, nrm);
          T.x = add(sub(cp, r), smul(0.0001f * 2.0f, nrm));  // consts::EPSILON * 2.0
          T.p = add(T.p, imp);  // apply_impulse (:38-41)
          T.l = add(T.l, cross(r, imp));
          moved = true;
        }
        if (!GRID && moved) sides = corner_sides(O, Cn, T.x);
      }
    }
    S = T;
    // clear_forces, clear_torques
    F = tau = f3{0.0f, 0.0f, 0.0f};
    if (step == 0) {  // a -0 of the record among the constant fields becomes +0
      auto plus = [&](int k, float& v) {
        const float w = v + 0.0f;
        if (__float_as_uint(v) != __float_as_uint(w)) field(k) = w;
        v = w;
      };
      plus(13, m);
      for (int c = 0; c < 3; ++c) {
        plus(14 + 3 * c, I.c[c].x);
        plus(15 + 3 * c, I.c[c].y);
        plus(16 + 3 * c, I.c[c].z);
      }
    }
  }
  field(0) = S.x.x; field(1) = S.x.y; field(2) = S.x.z;
  field(3) = S.q.v.x; field(4) = S.q.v.y; field(5) = S.q.v.z; field(6) = S.q.s;
  field(7) = S.p.x; field(8) = S.p.y; field(9) = S.p.z;
  field(10) = S.l.x; field(11) = S.l.y; field(12) = S.l.z;
}

// Field-major device records <-> the caller's 29-float records, body after body.
__global__ void __launch_bounds__(kBlock) rigid_pack_kernel(const float* __restrict__ in, uint32_t n, uint32_t pitch,
                                                             float* __restrict__ out) {
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
  if (b >= n) return;
#pragma unroll
  for (int k = 0; k < kRigidRecord; ++k) out[(size_t)kRigidRecord * b + k] = in[(size_t)k * pitch + b];
}
__global__ void __launch_bounds__(kBlock) rigid_unpack_kernel(const float* __restrict__ in, uint32_t n, uint32_t pitch,
                                                               float* __restrict__ out) {
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
  if (b >= n) return;
#pragma unroll
  for (int k = 0; k < kRigidRecord; ++k) out[(size_t)k * pitch + b] = in[(size_t)kRigidRecord * b + k];
}

}  // namespace

hipError_t launch_rigid_records(const float* in, float* out, uint32_t n, uint32_t pitch, bool pack, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (pitch < n) return hipErrorInvalidValue;
  const dim3 g((n + kBlock - 1) / kBlock), b(kBlock);
  if (pack) rigid_pack_kernel<<<g, b, 0, s>>>(in, n, pitch, out);
  else rigid_unpack_kernel<<<g, b, 0, s>>>(in, n, pitch, out);
  return hipGetLastError();
}

hipError_t launch_rigid_steps(float* rec, uint32_t n, uint32_t pitch, const RigidParams& p, const ObsView& obs,
                              uint32_t steps, hipStream_t s) {
  if (n == 0 || steps == 0) return hipSuccess;
  if (pitch < n) return hipErrorInvalidValue;
  constexpr uint32_t kMost = 1u << 28;  // bodies a launch: the kernel's byte offsets are 32 bits
  for (uint32_t first = 0; first < n; first += kMost) {
    const uint32_t count = n - first < kMost ? n - first : kMost;
    const dim3 g((count + kBlock - 1) / kBlock), b(kBlock);
    if (obs.use_grid) rigid_step_kernel<true><<<g, b, 0, s>>>(rec + first, count, pitch, p, obs, steps);
    else rigid_step_kernel<false><<<g, b, 0, s>>>(rec + first, count, pitch, p, obs, steps);
    if (n - first <= kMost) break;
  }
  return hipGetLastError();
}

}  // namespace fp
