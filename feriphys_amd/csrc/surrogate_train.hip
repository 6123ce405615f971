// gfx950 training kernels of the learned surrogate (surrogate.hpp): a step is three launches.
//
//   train_chain_kernel    the whole per-row chain.  A wave owns 16 batch rows: it gathers their
//                         features, runs the four layers, the error, and the error back to every
//                         layer's pre-activations, with the activations in registers and LDS.
//   train_weights_kernel  weight and bias gradients, products over the batch rows: each workgroup
//                         one layer and one slice of the batch.
//   train_update_kernel   sums the slices, Adam, the bf16 copies the next step reads.
//
// What bounds them: the work of a step is 254 kFLOP and ~2 KB of workspace traffic per row (4.2
// GFLOP, 34 MB at 16,384 rows), so a step is a chain of latencies (row gather, weight staging, seven
// dependent layers) rather than a rate.  The layer-by-layer form this replaces launched 22 kernels a
// step, wrote every f32 pre-activation to HBM and formed each weight gradient in four workgroups
// that walked the whole batch: a call that sets the parameters, takes 8 steps of 16,384 rows and reads
// the parameters back took 65.3 ms, and takes 0.43 ms in this form.  (The chain kernel itself took 30 us
// while its weights were staged a load at a time and the workgroup waited at every layer, and 21.6 now.  The
// weight kernel reads the 32 MB workspace in 15 us; four blocks in flight instead of one did not change it.)
//
// Each MFMA accumulates the same 32-wide K blocks in the same order from zero, biases are added
// afterwards and activations are rounded to bf16 where they always were, so every per-row value
// keeps its bits; only the sums over the batch have another order (64 slices of f32 sums).
#include "surrogate_device.hpp"

#pragma clang fp contract(fast)

namespace fp {

namespace {

// LDS of the chain kernel: the forward weights as in the inference image (natural K order), later
// overlaid by the transposed W3 and W2; each wave's activations [16 rows][kLd]; its output errors.
constexpr int kImgFwd = kImgB;               // W1, W2, W3, W4 of the image layout, no biases
constexpr int kActBytes = 16 * kLd * 2;
static_assert(2 * kHid * kLd * 2 <= kImgW4, "the transposed W3 and W2 leave W4 in place");

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u32x2 pack4(const __bf16 (&h)[4]) {
  u32x2 q;
  q[0] = (uint32_t)__builtin_bit_cast(uint16_t, h[0]) | (uint32_t)__builtin_bit_cast(uint16_t, h[1]) << 16;
  q[1] = (uint32_t)__builtin_bit_cast(uint16_t, h[2]) | (uint32_t)__builtin_bit_cast(uint16_t, h[3]) << 16;
  return q;
}

// `ROWS` rows of K bf16 (16-byte units) on their way to LDS rows of LD elements, zero up to KPAD: every
// load of a thread is issued by `load`, before the first is waited for by `store` (a load, its wait and
// its LDS write in turn cost the latency 24 times).
template <int K, int KPAD, int LD, int ROWS, int THREADS>
struct Staged {
  static constexpr int kU = KPAD / 8, kRounds = (ROWS * kU + THREADS - 1) / THREADS;
  uint4 q[kRounds];
  __device__ __forceinline__ void load(const __bf16* __restrict__ src, int rows) {
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
      const int e = threadIdx.x + j * THREADS, r = e / kU, u = e - r * kU;
      q[j] = make_uint4(0, 0, 0, 0);
      if (r < rows && u < K / 8) q[j] = *reinterpret_cast<const uint4*>(src + r * K + 8 * u);
    }
  }
  __device__ __forceinline__ void store(__bf16* dst) const {
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
      const int e = threadIdx.x + j * THREADS, r = e / kU, u = e - r * kU;
      if (ROWS * kU % THREADS == 0 || r < ROWS) *reinterpret_cast<uint4*>(dst + r * LD + 8 * u) = q[j];
    }
  }
};

// Between a wave's LDS writes and its own reads of them (its activations are its own: no other wave waits).
__device__ __forceinline__ void own_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int WAVES>
__global__ void __launch_bounds__(64 * WAVES) train_chain_kernel(TrainBatch A) {
  constexpr int kThreads = 64 * WAVES;
  __shared__ uint4 s_img[kImgFwd / 16];
  __shared__ uint4 s_act[WAVES][kActBytes / 16];
  __shared__ __bf16 s_dy[WAVES][16][4];
  __shared__ float s_loss[WAVES];
  __shared__ float s_bias[3][kHid];
  char* img = reinterpret_cast<char*>(s_img);
  __bf16 *W1 = reinterpret_cast<__bf16*>(img + kImgW1), *W2 = reinterpret_cast<__bf16*>(img + kImgW2),
         *W3 = reinterpret_cast<__bf16*>(img + kImgW3), *W4 = reinterpret_cast<__bf16*>(img + kImgW4);
  __bf16 *W3t = reinterpret_cast<__bf16*>(img), *W2t = W3t + kHid * kLd;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
  __bf16* act = reinterpret_cast<__bf16*>(s_act[wave]);
  const int row0 = (blockIdx.x * WAVES + wave) * 16;  // the wave's first batch row
  const int myrow = row0 + col;
  // operand rows: lane (col, g) holds batch row `col`; products' rows: lane holds rows 4g .. 4g+3
  uint64_t src = 0;
  if (myrow < A.rows) src = A.count ? mix64(A.seed ^ mix64((uint64_t)myrow)) % A.count : (uint64_t)myrow;
  auto features = [&](bf16x8(&xf)[3]) {
#pragma unroll
    for (int kb = 0; kb < 3; ++kb) {
      uint4 q = make_uint4(0, 0, 0, 0);
      const int u = 4 * kb + g;
      if (myrow < A.rows && u < kFeat / 8) q = *reinterpret_cast<const uint4*>(A.X + src * kFeat + 8 * u);
      xf[kb] = __builtin_bit_cast(bf16x8, q);
    }
  };
  bf16x8 xf[3];
  features(xf);
  {
    Staged<kFeat, 96, kLd1, kHid, kThreads> w1;
    Staged<kHid, kHid, kLd, kHid, kThreads> w2, w3;
    Staged<kHid, kHid, kLd, 16, kThreads> w4;
    w1.load(A.wb + kOffW1, kHid);
    w2.load(A.wb + kOffW2, kHid);
    w3.load(A.wb + kOffW3, kHid);
    w4.load(A.wb + kOffW4, kOut);
    for (int k = threadIdx.x; k < 3 * kHid; k += kThreads) {
      const int l = k / kHid, n = k - l * kHid;
      s_bias[l][n] = A.P[(l == 0 ? kOffB1 : l == 1 ? kOffB2 : kOffB3) + n];
    }
    w1.store(W1);
    w2.store(W2);
    w3.store(W3);
    w4.store(W4);
  }
  // the targets of the lane's output rows (the eight-wave form has no registers to hold them)
  auto target_of = [&](int r) {
    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)src, 4 * g + r, 64),
                   hi = (uint32_t)__shfl((int)(uint32_t)(src >> 32), 4 * g + r, 64);
    const uint64_t from = (uint64_t)hi << 32 | lo;
    return row0 + 4 * g + r < A.rows && col < kOut ? A.T[from * kOut + col] : 0.0f;
  };
  float target[4];
  if constexpr (WAVES == 4)
#pragma unroll
    for (int r = 0; r < 4; ++r) target[r] = target_of(r);

  const size_t pitch = (size_t)A.pitch;
  // the lane's four values of an operand row to the workspace (the grid covers the pitch); rows past
  // the batch are stored as zero
  // (a uniform base and a 32-bit byte offset per lane: 16 rows of the pitch are below 4 GB)
  const uint32_t put_at = 2u * ((uint32_t)col * (uint32_t)A.pitch + (uint32_t)(row0 + 4 * g));
  auto put = [&](int operand_rows, const __bf16(&h)[4]) {
    __bf16 v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = row0 + 4 * g + r < A.rows ? h[r] : (__bf16)0.0f;
    *reinterpret_cast<u32x2*>(reinterpret_cast<char*>(A.tr + (size_t)operand_rows * pitch) + put_at) = pack4(v);
  };
  f32x4 z1[8], z2[8], z3[8];
  bf16x8 hf[4];
  // activations of one layer from its pre-activations: to LDS (row-major, the next operand) and to
  // the workspace (transposed)
  auto activate = [&](f32x4(&z)[8], const float (&bias)[kHid], int tr_row) {
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      const float b = bias[16 * mt + col];
      __bf16 h[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        z[mt][r] = z[mt][r] + b;
        h[r] = (__bf16)gelu(z[mt][r]);
        act[(4 * g + r) * kLd + 16 * mt + col] = h[r];
      }
      put(tr_row + 16 * mt, h);
    }
  };
  auto fragments = [&]() {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) hf[kb] = *reinterpret_cast<const bf16x8*>(act + col * kLd + kb * 32 + 8 * g);
  };
  auto layer = [&](const __bf16* W, f32x4(&z)[8]) {
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        acc = mfma(hf[kb], *reinterpret_cast<const bf16x8*>(W + (16 * mt + col) * kLd + kb * 32 + 8 * g), acc);
      z[mt] = acc;
    }
  };
  // the features, transposed
#pragma unroll
  for (int kb = 0; kb < 3; ++kb) *reinterpret_cast<bf16x8*>(act + col * kLd + kb * 32 + 8 * g) = xf[kb];
  own_lds();
#pragma unroll
  for (int mt = 0; mt < 5; ++mt) {
    __bf16 x[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = act[(4 * g + r) * kLd + 16 * mt + col];
    put(kTrX + 16 * mt, x);
  }
  own_lds();
  __syncthreads();  // the weights are staged
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < 3; ++kb)
      acc = mfma(xf[kb], *reinterpret_cast<const bf16x8*>(W1 + (16 * mt + col) * kLd1 + kb * 32 + 8 * g), acc);
    z1[mt] = acc;
  }
  activate(z1, s_bias[0], kTrH1);
  own_lds();
  fragments();
  own_lds();
  layer(W2, z2);
  activate(z2, s_bias[1], kTrH2);
  own_lds();
  fragments();
  own_lds();
  layer(W3, z3);
  activate(z3, s_bias[2], kTrH3);
  own_lds();
  fragments();
  f32x4 y = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
    y = mfma(hf[kb], *reinterpret_cast<const bf16x8*>(W4 + col * kLd + kb * 32 + 8 * g), y);
  // mean squared error: dY = 2 (y - t) / (3 rows)
  float e2 = 0.0f;
  {
    const float b4 = col < kOut ? A.P[kOffB4 + col] : 0.0f;
    if constexpr (WAVES != 4)
#pragma unroll
      for (int r = 0; r < 4; ++r) target[r] = target_of(r);
    __bf16 d4[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 4 * g + r;
      d4[r] = (__bf16)0.0f;
      if (row < A.rows && col < kOut) {
        const float v = y[r] + b4;
        if (A.Y) A.Y[(size_t)row * kOut + col] = v;
        const float d = v - target[r];
        e2 += d * d;
        d4[r] = (__bf16)(2.0f * d / (3.0f * (float)A.rows));
      }
      if (col < 4) s_dy[wave][4 * g + r][col] = d4[r];
    }
    put(kTrY, d4);  // rows 3..15 of the operand are zero
  }
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) e2 += __shfl_xor(e2, w, 64);
  if (lane == 0) s_loss[wave] = e2;
  __syncthreads();  // every wave is done with the forward weights
  {
    Staged<kHid, kHid, kLd, kHid, kThreads> w3t, w2t;
    w3t.load(A.wbt + kHid * kHid, kHid);
    w2t.load(A.wbt, kHid);
    w3t.store(W3t);
    w2t.store(W2t);
  }
  if (threadIdx.x == 0) {
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) s += s_loss[w];
    A.loss_part[blockIdx.x] = s;
  }
  // dH3 = dY W4 (K = 3, padded with zeros)
  bf16x8 dyf;
#pragma unroll
  for (int s = 0; s < 8; ++s) dyf[s] = (g == 0 && s < kOut) ? s_dy[wave][col][s] : (__bf16)0.0f;
  f32x4 dh[8];
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    bf16x8 w;
#pragma unroll
    for (int s = 0; s < 8; ++s) w[s] = (g == 0 && s < kOut) ? W4[s * kLd + 16 * mt + col] : (__bf16)0.0f;
    dh[mt] = mfma(dyf, w, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
  }
  // dZ = bf16(dH * gelu'(Z)): to LDS as the next operand (unless it is the last) and to the workspace
  auto backward = [&](const f32x4(&z)[8], int tr_row, bool next) {
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      __bf16 d[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        d[r] = (__bf16)(dh[mt][r] * gelu_grad(z[mt][r]));
        if (next) act[(4 * g + r) * kLd + 16 * mt + col] = d[r];
      }
      put(tr_row + 16 * mt, d);
    }
  };
  backward(z3, kTrZ3, true);
  __syncthreads();  // the transposed weights are staged
  fragments();
  own_lds();
  layer(W3t, dh);
  backward(z2, kTrZ2, true);
  own_lds();
  fragments();
  own_lds();
  layer(W2t, dh);
  backward(z1, kTrZ1, false);
}

// One layer's gradient over one slice of the batch: dW[n][k] = sum over rows of dZ[n] H[k], and
// db[n] from a column of ones.  Four waves of 32 output rows by all columns; the operands are read
// straight from the transposed workspace (16 consecutive bytes a lane, 64-byte segments, shared by
// the waves through the L1).  Layer 4 has one 16-row tile: its waves split the columns.
template <int NT>
__device__ __forceinline__ void layer_grad(const __bf16* __restrict__ Z, const __bf16* __restrict__ H, size_t pitch,
                                           int k0, int k1, int kin, float* __restrict__ dW, float* __restrict__ db) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
  f32x4 acc[2][NT], accb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accb[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
  bf16x8 ones;
#pragma unroll
  for (int s = 0; s < 8; ++s) ones[s] = (__bf16)1.0f;
  const __bf16* za = Z + (size_t)(32 * wave + col) * pitch + 8 * g;
  const __bf16* hb = H + (size_t)col * pitch + 8 * g;
  bf16x8 na[2], nb[NT];  // the next block's operands, in flight while this one multiplies
  auto fetch = [&](int k) {
#pragma unroll
    for (int i = 0; i < 2; ++i) na[i] = *reinterpret_cast<const bf16x8*>(za + (size_t)(16 * i) * pitch + k);
#pragma unroll
    for (int j = 0; j < NT; ++j) nb[j] = *reinterpret_cast<const bf16x8*>(hb + (size_t)(16 * j) * pitch + k);
  };
  if (k0 < k1) fetch(k0);
  for (int k = k0; k < k1; k += 32) {
    bf16x8 a[2], b[NT];
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = na[i];
#pragma unroll
    for (int j = 0; j < NT; ++j) b[j] = nb[j];
    if (k + 32 < k1) fetch(k + 32);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      accb[i] = mfma(a[i], ones, accb[i]);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = mfma(a[i], b[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 32 * wave + 16 * i + 4 * g + r;
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if (16 * j + col < kin) dW[n * kin + 16 * j + col] = acc[i][j][r];
      if (col == 0) db[n] = accb[i][r];
    }
}

__global__ void __launch_bounds__(256) train_weights_kernel(const __bf16* __restrict__ tr, int pitch_, int slice_rows,
                                                            float* __restrict__ part) {
  const size_t pitch = (size_t)pitch_;
  const int k0 = blockIdx.y * slice_rows, k1 = min(k0 + slice_rows, pitch_);
  float* out = part + (size_t)blockIdx.y * kParams;
  switch (blockIdx.x) {
    case 0: layer_grad<8>(tr + kTrZ3 * pitch, tr + kTrH2 * pitch, pitch, k0, k1, kHid, out + kOffW3, out + kOffB3); return;
    case 1: layer_grad<8>(tr + kTrZ2 * pitch, tr + kTrH1 * pitch, pitch, k0, k1, kHid, out + kOffW2, out + kOffB2); return;
    case 2: layer_grad<5>(tr + kTrZ1 * pitch, tr + kTrX * pitch, pitch, k0, k1, kFeat, out + kOffW1, out + kOffB1); return;
    default: break;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
  f32x4 acc[2], accb = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  acc[0] = acc[1] = accb;
  bf16x8 ones;
#pragma unroll
  for (int s = 0; s < 8; ++s) ones[s] = (__bf16)1.0f;
  const __bf16* za = tr + (size_t)(kTrY + col) * pitch + 8 * g;
  const __bf16* hb = tr + (size_t)(kTrH3 + 32 * wave + col) * pitch + 8 * g;
  for (int k = k0; k < k1; k += 32) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(za + k);
    accb = mfma(a, ones, accb);
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[j] = mfma(a, *reinterpret_cast<const bf16x8*>(hb + (size_t)(16 * j) * pitch + k), acc[j]);
  }
  if (g == 0) {
#pragma unroll
    for (int r = 0; r < kOut; ++r) {
#pragma unroll
      for (int j = 0; j < 2; ++j) out[kOffW4 + r * kHid + 32 * wave + 16 * j + col] = acc[j][r];
      if (col == 0 && wave == 0) out[kOffB4 + r] = accb[r];
    }
  }
}

// bf16 copies of parameter i: natural order, and for W2 and W3 the transpose.
__device__ __forceinline__ void put_weight(int i, float p, __bf16* __restrict__ wb, __bf16* __restrict__ wbt) {
  const __bf16 h = (__bf16)p;
  wb[i] = h;
  const int j2 = i - kOffW2, j3 = i - kOffW3;
  if (j2 >= 0 && j2 < kHid * kHid) wbt[(j2 % kHid) * kHid + j2 / kHid] = h;
  else if (j3 >= 0 && j3 < kHid * kHid) wbt[kHid * kHid + (j3 % kHid) * kHid + j3 / kHid] = h;
}

// One thread per parameter (the last workgroup: the loss).
__global__ void __launch_bounds__(kBlock) train_update_kernel(const float* __restrict__ part, int slices,
                                                              float* __restrict__ g, const float* __restrict__ loss_part,
                                                              int n_loss, float scale, float* __restrict__ loss,
                                                              AdamArgs A, __bf16* __restrict__ wb,
                                                              __bf16* __restrict__ wbt) {
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ float s[kBlock];
    float acc = 0.0f;
    for (int k = threadIdx.x; k < n_loss; k += kBlock) acc += loss_part[k];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = s[0] * scale;
    return;
  }
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= kParams) return;
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  int k = 0;
  for (; k + 16 <= slices; k += 16) {
    float v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = part[(size_t)(k + q) * kParams + i];
#pragma unroll
    for (int q = 0; q < 16; ++q) s[q & 3] += v[q];
  }
  for (; k < slices; ++k) s[k & 3] += part[(size_t)k * kParams + i];
  const float gi = (s[0] + s[1]) + (s[2] + s[3]);
  g[i] = gi;
  if (A.p == nullptr) return;
  const float mi = A.b1 * A.m[i] + (1.0f - A.b1) * gi;
  const float vi = A.b2 * A.v[i] + (1.0f - A.b2) * gi * gi;
  A.m[i] = mi;
  A.v[i] = vi;
  const float p = A.p[i] - A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
  A.p[i] = p;
  put_weight(i, p, wb, wbt);
}

__global__ void __launch_bounds__(kBlock) weights_bf16_kernel(const float* __restrict__ p, __bf16* __restrict__ wb,
                                                              __bf16* __restrict__ wbt) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < kParams) put_weight(i, p[i], wb, wbt);
}

constexpr int kParamBlocks = (kParams + (int)kBlock - 1) / (int)kBlock;

}  // namespace

hipError_t launch_train_chain(const TrainBatch& b, hipStream_t s) {
  if (b.rows <= 0 || b.pitch < b.rows || b.pitch % kTrainTile != 0) return hipErrorInvalidValue;
  // four waves (64 rows) a workgroup until that gives every CU one, then eight, so that a CU's one
  // resident workgroup (the weights take its LDS) has two waves per SIMD
  if (train_waves(b.pitch) == 4) train_chain_kernel<4><<<dim3(train_groups(b.pitch)), dim3(256), 0, s>>>(b);
  else train_chain_kernel<8><<<dim3(train_groups(b.pitch)), dim3(512), 0, s>>>(b);
  return hipGetLastError();
}

hipError_t launch_train_weights(const __bf16* tr, int pitch, float* part, hipStream_t s) {
  if (pitch <= 0 || pitch % kTrainTile != 0) return hipErrorInvalidValue;
  const int n = train_slices(pitch);
  const int rows = ((pitch + n - 1) / n + 31) / 32 * 32;  // n slices of this many rows cover the pitch
  train_weights_kernel<<<dim3(4, n), dim3(256), 0, s>>>(tr, pitch, rows, part);
  return hipGetLastError();
}

hipError_t launch_train_update(const float* part, int slices, float* g, const float* loss_part, int n_loss,
                               float scale, float* loss, const AdamArgs& a, __bf16* wb, __bf16* wbt, hipStream_t s) {
  train_update_kernel<<<dim3(kParamBlocks + 1), dim3(kBlock), 0, s>>>(part, slices, g, loss_part, n_loss, scale, loss,
                                                                      a, wb, wbt);
  return hipGetLastError();
}

hipError_t launch_train_weights_bf16(const float* p, __bf16* wb, __bf16* wbt, hipStream_t s) {
  weights_bf16_kernel<<<dim3(kParamBlocks), dim3(kBlock), 0, s>>>(p, wb, wbt);
  return hipGetLastError();
}

}  // namespace fp
