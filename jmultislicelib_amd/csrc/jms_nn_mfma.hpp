// jms_nn_mfma.hpp -- the surrogate's 3x3 convolutions as implicit GEMMs on
// the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16: bf16 operands, FP32
// accumulation), included by jms_nn.hip.
//
// Images are staged in LDS in a channels-last layout with a one-pixel zero
// border, so that the 8 bf16 values of an MFMA operand fragment -- 8
// consecutive channels at one (pixel, tap) -- are one aligned 16-byte LDS read
// and the padding needs no bounds checks.  The GEMM K index of the forward and
// data-gradient products runs over (tap, 8-channel group), of the weight
// gradients over the output pixels (transposed LDS reads).  Weights come as A
// fragments in their own order.
//
// MFMA 16x16x32 operand layout (lane l of 64, g = l / 16): A fragment = row
// l % 16, K elements 8g .. 8g+7; B fragment = column l % 16, the same K
// elements; result = rows 4g .. 4g+3 of column l % 16.
#pragma once

namespace nnmfma {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int CH = 32;  // output (and hidden) channels of every convolution

__device__ __forceinline__ f32x4 mfma(const u16x8& a, const u16x8& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                0, 0);
}

__device__ __forceinline__ uint16_t f2bf_rne(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// ---------------------------------------------------------------------------
// Weights in fragment order.  A fragments of conv l: tile mt (output channels
// 16 mt ..), K step ks, lane (g, r), element j = w[16 mt + r][ci][tap] with
// K group kg = 4 ks + g = tap * CI/8 + ci/8, ci % 8 = j; one 16-byte load per
// lane and fragment.  Dense 1 is transposed to [input / 8][output][input % 8],
// so that the lanes of a wavefront (outputs) load 1 KiB at once.  The copies
// are written by the kernels that round the parameters to bf16.
// ---------------------------------------------------------------------------
constexpr int conv_ks(int ci) { return (9 * ci / 8 + 3) / 4; }
constexpr int frag_off(int l) { return l == 0 ? 0 : (2 * conv_ks(8) + (l - 1) * 2 * conv_ks(CH)) * 512; }
constexpr int PACK_D1 = frag_off(4);             // dense 1 after the four convolutions
// A fragments of the data gradients: tile mt (input channels 16 mt ..), tap,
// lane (g, r), element j = w[8 g + j][16 mt + r][tap]
constexpr int PACK_B = PACK_D1 + 64 * 512;
constexpr int PACK_SIZE = PACK_B + 3 * 2 * 9 * 512;  // bf16 elements
__device__ __forceinline__ int conv_pack_b(int l, int co, int ci, int tap) {
  return PACK_B + ((((l - 1) * 2 + (ci >> 4)) * 9 + tap) * 64 + 16 * (co >> 3) + (ci & 15)) * 8 + (co & 7);
}
__device__ __forceinline__ int conv_pack(int l, int ci_n, int co, int ci, int tap) {
  const int kg = tap * (ci_n / 8) + ci / 8, ks = kg >> 2, g = kg & 3;
  return frag_off(l) + (((co >> 4) * conv_ks(ci_n) + ks) * 64 + 16 * g + (co & 15)) * 8 + (ci & 7);
}

// four bf16 (round to nearest even) of relu(acc + b)
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t cvt2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ uint2 relu4(const f32x4& acc, const f32x4& b) {
  return make_uint2(cvt2(fmaxf(acc[0] + b[0], 0.f), fmaxf(acc[1] + b[1], 0.f)),
                    cvt2(fmaxf(acc[2] + b[2], 0.f), fmaxf(acc[3] + b[3], 0.f)));
}
__device__ __forceinline__ f32x4 ld4(const float* p) { return f32x4{p[0], p[1], p[2], p[3]}; }
// channels-last LDS images of 32 channels: the four 16-byte groups of a pixel
// at column x (padded) are rotated by x / 4, so that 16 neighbouring pixels
// written 8 bytes each, or 8 pixels two apart read 16 bytes each, fall on
// distinct banks
__device__ __forceinline__ int swz(int x, int group) { return 8 * (group ^ ((x >> 2) & 3)); }

__device__ __forceinline__ u16x8 ldfrag(const uint16_t* p) { return *reinterpret_cast<const u16x8*>(p); }

// The four convolutions of one sample after the other, one block of 8
// wavefronts per CU: y = relu(b + conv(x)) four times, every intermediate in
// LDS (channels last, one-pixel zero border), so that a sample costs one read
// of its 16 KiB window and one write of its 512 features.  What bounds it: the
// 16-byte B-fragment reads from LDS and the MFMAs of the first two layers
// (672 of 762 per sample).  The A fragments of the first three layers stay in
// registers over all samples of the block, those of the last in LDS (138 KiB
// in all).  The next window is loaded while this one is worked on.
// KEEP (training): the intermediates also go to memory, channels last.
// 16384 windows: 258 us (690 TFLOP/s);
// four launches per 2048 windows, each with its own staging, took 1720 us.
// grid: min(n, CUs); feat[n][512] in channel-major order; idx (or nullptr):
// sample s is window idx[s]
constexpr int NET_THREADS = 512;
template <bool KEEP>
__global__ __launch_bounds__(NET_THREADS) void k_net_fwd(const uint16_t* __restrict__ x,
                                                         const int* __restrict__ idx,
                                                         const uint16_t* __restrict__ wp,
                                                         const float* __restrict__ b0, const float* __restrict__ b1,
                                                         const float* __restrict__ b2, const float* __restrict__ b3,
                                                         int n, uint16_t* __restrict__ feat, uint16_t* __restrict__ y1,
                                                         uint16_t* __restrict__ y2, uint16_t* __restrict__ y3) {
  constexpr int P0 = 34, P2 = 18, P3 = 10;  // padded edges: input and conv 1 output, conv 2, conv 3 output
  __shared__ __align__(16) uint16_t s_x[P0 * P0 * 8];
  __shared__ __align__(16) uint16_t s_1[P0 * P0 * CH];
  __shared__ __align__(16) uint16_t s_2[P2 * P2 * CH];
  __shared__ __align__(16) uint16_t s_3[P3 * P3 * CH];
  __shared__ __align__(16) uint16_t s_w[2 * 9 * 512];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto zero = [&](uint16_t* p, int cnt) {
    for (int i = tid; i < cnt / 8; i += NET_THREADS) reinterpret_cast<u16x8*>(p)[i] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  };
  zero(s_x, P0 * P0 * 8);
  zero(s_1, P0 * P0 * CH);
  zero(s_2, P2 * P2 * CH);
  zero(s_3, P3 * P3 * CH);
  for (int i = tid; i < 2 * 9 * 64; i += NET_THREADS)
    reinterpret_cast<u16x8*>(s_w)[i] = ldfrag(wp + frag_off(3) + i * 8);
  u16x8 a0[2][3], a1[2][9], a2[9];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
    for (int ks = 0; ks < 3; ++ks) a0[mt][ks] = ldfrag(wp + ((mt * 3 + ks) * 64 + lane) * 8);
#pragma unroll
    for (int ks = 0; ks < 9; ++ks) a1[mt][ks] = ldfrag(wp + frag_off(1) + ((mt * 9 + ks) * 64 + lane) * 8);
  }
  const int mt2 = wv & 1;  // the channel tile of this wavefront in conv 3
#pragma unroll
  for (int ks = 0; ks < 9; ++ks) a2[ks] = ldfrag(wp + frag_off(2) + ((mt2 * 9 + ks) * 64 + lane) * 8);
  const f32x4 c00 = ld4(b0 + 4 * g), c01 = ld4(b0 + 16 + 4 * g), c10 = ld4(b1 + 4 * g), c11 = ld4(b1 + 16 + 4 * g);
  const f32x4 c2 = ld4(b2 + 16 * mt2 + 4 * g), c3 = ld4(b3 + 16 * (wv & 1) + 4 * g);
  const int half = 4 * (g & 1);  // this lane's four channels in their 16-byte group
  // LDS offset of this lane's tap in the K steps of conv 1 (one tap per K
  // group; the groups past the ninth tap read the zero border pixel 0)
  const int tap0[3] = {((g / 3) * P0 + g % 3) * 8, (((4 + g) / 3) * P0 + (4 + g) % 3) * 8, (2 * P0 + 2) * 8};
  // pixels 2 tid, 2 tid + 1 of the eight input planes
  uint32_t in[8];
  auto load_in = [&](int sample) {
    const long long w = idx ? idx[sample] : sample;
    const uint32_t* xn = reinterpret_cast<const uint32_t*>(x + w * (8 * 1024)) + tid;
#pragma unroll
    for (int c = 0; c < 8; ++c) in[c] = xn[c * 512];
  };
  int sample = blockIdx.x;
  if (sample < n) load_in(sample);
  __syncthreads();
  for (; sample < n; sample += gridDim.x) {
    {  // the window into LDS, eight channels of a pixel together
      const int p = 2 * tid, iy = p >> 5, ix = p & 31;
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        lo[c] = (in[2 * c] & 0xffffu) | (in[2 * c + 1] << 16);
        hi[c] = (in[2 * c] >> 16) | (in[2 * c + 1] & 0xffff0000u);
      }
      uint4* d = reinterpret_cast<uint4*>(&s_x[((iy + 1) * P0 + ix + 1) * 8]);
      d[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      d[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    }
    __syncthreads();
    if (sample + (int)gridDim.x < n) load_in(sample + gridDim.x);
    // conv 1: 64 groups of 16 pixels, both channel tiles per wavefront
#pragma unroll 4
    for (int k = 0; k < 8; ++k) {
      const int p = (wv + 8 * k) * 16 + r, oy = p >> 5, ox = p & 31;
      const int xp = (oy * P0 + ox) * 8;
      f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 3; ++ks) {
        const u16x8 bf = ldfrag(s_x + (ks < 2 || g == 0 ? xp + tap0[ks] : 0));
        acc0 = mfma(a0[0][ks], bf, acc0);
        acc1 = mfma(a0[1][ks], bf, acc1);
      }
      uint16_t* d = s_1 + ((oy + 1) * P0 + ox + 1) * CH + half;
      const uint2 o0 = relu4(acc0, c00), o1 = relu4(acc1, c01);
      *reinterpret_cast<uint2*>(d + swz(ox + 1, g >> 1)) = o0;
      *reinterpret_cast<uint2*>(d + swz(ox + 1, 2 + (g >> 1))) = o1;
      if constexpr (KEEP) {
        uint16_t* yn = y1 + ((long long)sample * 1024 + p) * CH + 4 * g;
        *reinterpret_cast<uint2*>(yn) = o0;
        *reinterpret_cast<uint2*>(yn + 16) = o1;
      }
    }
    __syncthreads();
    // conv 2: 16 groups
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int p = (wv + 8 * k) * 16 + r, oy = p >> 4, ox = p & 15;
      const uint16_t* xp = s_1 + (2 * oy * P0 + 2 * ox) * CH;
      const int sx[3] = {swz(2 * ox, g), swz(2 * ox + 1, g) + CH, swz(2 * ox + 2, g) + 2 * CH};
      f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const u16x8 bf = ldfrag(xp + sx[t % 3] + (t / 3) * P0 * CH);
        acc0 = mfma(a1[0][t], bf, acc0);
        acc1 = mfma(a1[1][t], bf, acc1);
      }
      uint16_t* d = s_2 + ((oy + 1) * P2 + ox + 1) * CH + half;
      const uint2 o0 = relu4(acc0, c10), o1 = relu4(acc1, c11);
      *reinterpret_cast<uint2*>(d + swz(ox + 1, g >> 1)) = o0;
      *reinterpret_cast<uint2*>(d + swz(ox + 1, 2 + (g >> 1))) = o1;
      if constexpr (KEEP) {
        uint16_t* yn = y2 + ((long long)sample * 256 + p) * CH + 4 * g;
        *reinterpret_cast<uint2*>(yn) = o0;
        *reinterpret_cast<uint2*>(yn + 16) = o1;
      }
    }
    __syncthreads();
    {  // conv 3: 4 groups x 2 channel tiles, one per wavefront
      const int p = (wv >> 1) * 16 + r, oy = p >> 3, ox = p & 7;
      const uint16_t* xp = s_2 + (2 * oy * P2 + 2 * ox) * CH;
      const int sx[3] = {swz(2 * ox, g), swz(2 * ox + 1, g) + CH, swz(2 * ox + 2, g) + 2 * CH};
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 9; ++t) acc = mfma(a2[t], ldfrag(xp + sx[t % 3] + (t / 3) * P2 * CH), acc);
      const uint2 o = relu4(acc, c2);
      uint16_t* d = s_3 + ((oy + 1) * P3 + ox + 1) * CH + half;
      *reinterpret_cast<uint2*>(d + swz(ox + 1, 2 * mt2 + (g >> 1))) = o;
      if constexpr (KEEP)
        *reinterpret_cast<uint2*>(y3 + ((long long)sample * 64 + p) * CH + 16 * mt2 + 4 * g) = o;
    }
    __syncthreads();
    if (wv < 2) {  // conv 4: 16 pixels x 2 channel tiles
      const int mt = wv, oy = r >> 2, ox = r & 3;
      const uint16_t* xp = s_3 + (2 * oy * P3 + 2 * ox) * CH;
      const int sx[3] = {swz(2 * ox, g), swz(2 * ox + 1, g) + CH, swz(2 * ox + 2, g) + 2 * CH};
      const uint16_t* wl = s_w + (mt * 9 * 64 + lane) * 8;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 9; ++t) acc = mfma(ldfrag(wl + t * 512), ldfrag(xp + sx[t % 3] + (t / 3) * P3 * CH), acc);
      const uint2 o = relu4(acc, c3);
      uint16_t* f = feat + (long long)sample * 512 + (16 * mt + 4 * g) * 16 + r;
      f[0] = (uint16_t)o.x;
      f[16] = (uint16_t)(o.x >> 16);
      f[32] = (uint16_t)o.y;
      f[48] = (uint16_t)(o.y >> 16);
    }
  }
}

// The dense head: h = relu(b1 + W1 f) (512 -> 64, bf16), out = b2 + W2 h
// (64 -> 3), the products summed in the order of the inputs.  A wavefront's
// lanes are the 64 hidden units of NS samples: the features are uniform and
// come through scalar loads, the weights are in LDS once per block.
// grid: ceil(n / (16 NS)), block: 1024
template <int NS>
__global__ __launch_bounds__(1024) void k_head(const uint16_t* __restrict__ feat, const uint16_t* __restrict__ w1t,
                                               const float* __restrict__ b1, const uint16_t* __restrict__ w2,
                                               const float* __restrict__ b2, int n, float* __restrict__ out) {
  __shared__ uint4 s_w[64 * 64];
  __shared__ uint16_t s_h[16][NS][64];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int i = threadIdx.x; i < 64 * 64; i += 1024) s_w[i] = reinterpret_cast<const uint4*>(w1t)[i];
  const int s0 = (blockIdx.x * 16 + wv) * NS;
  const uint4* f[NS];
  float acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    f[s] = reinterpret_cast<const uint4*>(feat) + (long long)(s0 + s < n ? s0 + s : n - 1) * 64;
    acc[s] = b1[lane];
  }
  __syncthreads();
#pragma unroll 2
  for (int k = 0; k < 64; ++k) {
    const uint4 w4 = s_w[k * 64 + lane];
    const uint32_t wa[4] = {w4.x, w4.y, w4.z, w4.w};
    float wf[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wf[2 * j] = __uint_as_float(wa[j] << 16);
      wf[2 * j + 1] = __uint_as_float(wa[j] & 0xFFFF0000u);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint4 f4 = f[s][k];
      const uint32_t fa[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[s] = fmaf(__uint_as_float(fa[j] << 16), wf[2 * j], acc[s]);
        acc[s] = fmaf(__uint_as_float(fa[j] & 0xFFFF0000u), wf[2 * j + 1], acc[s]);
      }
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    s_h[wv][s][lane] = f2bf_rne(fmaxf(acc[s], 0.f));
  }
  __syncthreads();
  if (lane < 3 * NS) {
    const int s = lane / 3, d = lane % 3;
    float y = b2[d];
#pragma unroll 4
    for (int k = 0; k < 64; ++k)
      y = fmaf(__uint_as_float((uint32_t)s_h[wv][s][k] << 16), __uint_as_float((uint32_t)w2[d * 64 + k] << 16), y);
    if (s0 + s < n) out[(long long)(s0 + s) * 3 + d] = y;
  }
}

// ---------------------------------------------------------------------------
// training
// ---------------------------------------------------------------------------
// Head of a training batch, one wavefront per sample (four per block): the
// forward of k_head, the loss mean(((y - t) / scale)^2) with its gradient,
// and what follows from it per sample: gh [n][64] (hidden units), df [n][512]
// (features, masked by their relu); hid [n][64] the hidden units themselves,
// dy [n][4] the output gradient and the sum of squared residuals.
// grid: ceil(n / 4), block: 256
__global__ __launch_bounds__(256) void k_head_train(const uint16_t* __restrict__ feat, const uint16_t* __restrict__ w1t,
                                                    const float* __restrict__ b1, const uint16_t* __restrict__ w2,
                                                    const float* __restrict__ b2, const float* __restrict__ T,
                                                    const int* __restrict__ idx, const float* __restrict__ scale, int n,
                                                    float* __restrict__ gh, float* __restrict__ df,
                                                    float* __restrict__ hid, float* __restrict__ dyo) {
  __shared__ uint4 s_w[64 * 64];
  __shared__ float s_h[4][64], s_gh[4][64], s_dy[4][4], s_w2[3 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // weights [k / 8][(unit + k / 8) mod 64]: read along the units (forward) or
  // along the inputs (backward), the lanes fall on distinct banks
  auto wat = [](int k8, int u) { return k8 * 64 + ((u + k8) & 63); };
  for (int i = tid; i < 64 * 64; i += 256) s_w[wat(i >> 6, i & 63)] = reinterpret_cast<const uint4*>(w1t)[i];
  if (tid < 3 * 64) s_w2[tid] = __uint_as_float((uint32_t)w2[tid] << 16);
  const int s = blockIdx.x * 4 + wv;
  const bool valid = s < n;
  const long long sm = valid ? s : n - 1;
  const uint4* f = reinterpret_cast<const uint4*>(feat) + sm * 64;
  const uint4 fl = f[lane];  // features 8 lane .., for the mask at the end
  const int d3 = lane < 3 ? lane : 0;
  const float tv = T[(idx ? idx[sm] : sm) * 3 + d3], sc = scale[d3], b2v = b2[d3];
  float acc = b1[lane];
  __syncthreads();
#pragma unroll 4
  for (int k = 0; k < 64; ++k) {
    const uint4 w4 = s_w[wat(k, lane)], f4 = f[k];
    const uint32_t wa[4] = {w4.x, w4.y, w4.z, w4.w}, fa[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc = fmaf(__uint_as_float(fa[j] << 16), __uint_as_float(wa[j] << 16), acc);
      acc = fmaf(__uint_as_float(fa[j] & 0xFFFF0000u), __uint_as_float(wa[j] & 0xFFFF0000u), acc);
    }
  }
  const float h = __uint_as_float((uint32_t)f2bf_rne(fmaxf(acc, 0.f)) << 16);
  s_h[wv][lane] = h;
  if (valid) hid[(long long)s * 64 + lane] = h;
  __syncthreads();
  if (lane < 4) {
    float l = 0.f;  // squared residual of output `lane`; their sum in lane 3
    if (lane < 3) {
      float y = b2v;
#pragma unroll 16
      for (int k = 0; k < 64; ++k) y = fmaf(s_h[wv][k], s_w2[lane * 64 + k], y);
      const float rs = (y - tv) / sc;
      s_dy[wv][lane] = 2.f * rs / sc / (float)(n * 3);
      l = rs * rs;
    }
    l += __shfl_xor(l, 1, 64);
    l += __shfl_xor(l, 2, 64);
    if (lane == 3) s_dy[wv][3] = l;
    if (valid) dyo[(long long)s * 4 + lane] = s_dy[wv][lane];
  }
  __syncthreads();
  float gv = 0.f;
  if (h > 0.f) {
#pragma unroll
    for (int d = 0; d < 3; ++d) gv = fmaf(s_dy[wv][d], s_w2[d * 64 + lane], gv);
  }
  s_gh[wv][lane] = gv;
  if (valid) gh[(long long)s * 64 + lane] = gv;
  __syncthreads();
  // features: lane k8 holds inputs 8 k8 .., the units summed in their order
  // (it decides the bf16 rounding of the gradient, which training follows)
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < 64; ++k) {
    const uint4 w4 = s_w[wat(lane, k)];
    const uint32_t wa[4] = {w4.x, w4.y, w4.z, w4.w};
    const float gu = s_gh[wv][k];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[2 * j] = fmaf(gu, __uint_as_float(wa[j] << 16), o[2 * j]);
      o[2 * j + 1] = fmaf(gu, __uint_as_float(wa[j] & 0xFFFF0000u), o[2 * j + 1]);
    }
  }
  if (valid) {
    const uint32_t fa[4] = {fl.x, fl.y, fl.z, fl.w};  // relu: a feature is zero or positive
    float4* d = reinterpret_cast<float4*>(df + (long long)s * 512 + 8 * lane);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!(__uint_as_float(fa[j] << 16) > 0.f)) o[2 * j] = 0.f;
      if (!(__uint_as_float(fa[j] & 0xFFFF0000u) > 0.f)) o[2 * j + 1] = 0.f;
    }
    d[0] = make_float4(o[0], o[1], o[2], o[3]);
    d[1] = make_float4(o[4], o[5], o[6], o[7]);
  }
}

// Sums over the samples of a batch are made in shares, each in sample order,
// then over the shares: short chains, and the same rounding in every run.
__device__ __forceinline__ int share_begin(int n, int y, int shares) { return (int)((long long)n * y / shares); }

// 16-bit transposed LDS read: of the 16 lanes of a group, lane i points to
// four columns (4 (i % 4) ..) of row i / 4; lane c receives column c of the
// four rows.  Two of them make an operand fragment whose K elements are rows
// (pixels) of a channels-last image.
typedef short v4s __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u16x8 ldtr(const uint16_t* p0, const uint16_t* p1) {
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)p0);
  const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)p1);
  return __builtin_bit_cast(u16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Weight gradient of a stride-2 convolution: rows co, columns 16 input
// channels (half h) of tap t, K the output pixels.  d: output gradient image
// (edge HOUT, row pitch PD), in: input image (row pitch PI, one-pixel
// border), both channels last.  Wavefront wv holds column tiles ct = wv + 8 j
// = 2 t + h, j = 0..2, ct < 18, and adds them to dw [ct][channel tile][lane]
// (add: a later sample of the block).
template <int HOUT, int PD, int PI>
__device__ __forceinline__ void wgrad(const uint16_t* d, const uint16_t* in, int wv, int g, int r, bool add,
                                      float* __restrict__ dw) {
  constexpr int KS = (HOUT * HOUT + 31) / 32;
  const int cg = (r & 3) >> 1, half = 4 * (r & 1);
  f32x4 acc[3][2];
#pragma unroll
  for (int j = 0; j < 3; ++j) acc[j][0] = acc[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int ks = 0; ks < KS; ++ks) {
    const int p0 = ks * 32 + 8 * g + (r >> 2), p1 = p0 + 4;
    const bool ok = HOUT * HOUT >= 32 || g < 2;  // 16 pixels fill half a K step
    const int y0 = ok ? p0 / HOUT : 0, x0 = p0 % HOUT, y1 = ok ? p1 / HOUT : 0, x1 = p1 % HOUT;
    u16x8 a[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      a[mt] = ldtr(d + (y0 * PD + x0) * CH + swz(x0, 2 * mt + cg) + half,
                   d + (y1 * PD + x1) * CH + swz(x1, 2 * mt + cg) + half);
      if (!ok) a[mt] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int ct = wv + 8 * j;
      if (ct >= 18) break;  // uniform in the wavefront
      const int t = ct >> 1, h = ct & 1, ky = t / 3, kx = t % 3;
      const int c0 = 2 * x0 + kx, c1 = 2 * x1 + kx;
      const u16x8 b = ldtr(in + ((2 * y0 + ky) * PI + c0) * CH + swz(c0, 2 * h + cg) + half,
                           in + ((2 * y1 + ky) * PI + c1) * CH + swz(c1, 2 * h + cg) + half);
      acc[j][0] = mfma(a[0], b, acc[j][0]);
      acc[j][1] = mfma(a[1], b, acc[j][1]);
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int ct = wv + 8 * j;
    if (ct >= 18) break;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      f32x4* q = reinterpret_cast<f32x4*>(dw) + (2 * ct + mt) * 64 + 16 * g + r;
      *q = add ? *q + acc[j][mt] : acc[j][mt];
    }
  }
}

// The gradient sums of a block of k_net_bwd: conv 1 (five column tiles of two
// taps x 8 input channels), convs 2..4 (18 column tiles each), every tile
// [channel tile][lane][4] as the accumulators hold it (16-byte stores), then
// the four biases.
constexpr int part_off(int l) { return l == 0 ? 0 : 5 * 512 + (l - 1) * 18 * 512; }
constexpr int PART_B = part_off(4), PART = PART_B + 4 * CH;
// the parameter at position j < PART_B of the sums: conv l, output channel,
// input channel, tap (9: none)
struct PartIdx {
  int l, co, ci, tap;
};
__device__ __forceinline__ PartIdx part_index(int j) {
  PartIdx q;
  q.l = j < part_off(1) ? 0 : 1 + (j - part_off(1)) / (18 * 512);
  const int e = j - part_off(q.l), ct = e >> 9, lane = (e >> 2) & 63, r = lane & 15;
  q.co = 16 * ((e >> 8) & 1) + 4 * (lane >> 4) + (e & 3);
  q.ci = q.l == 0 ? r & 7 : 16 * (ct & 1) + r;
  q.tap = q.l == 0 ? 2 * ct + (r >> 3) : ct >> 1;
  return q;
}

// Data gradient of a stride-2 convolution for the 16 input pixels of this
// wavefront's lanes: (2 m + PY, 2 mx + PX), one pair (m, mx) per lane r.
// Only the taps of the pixel's parity contribute: ky = 1 on even rows, 0 and
// 2 on odd ones.  d: output gradient image (row pitch PD, zero beyond its
// edge), w: A fragments [mt][tap].  Result: rows input channels 16 mt + 4 g + i.
template <int PY, int PX, int PD, int MT0, int NMT>
__device__ __forceinline__ void dgrad(const uint16_t* d, const uint16_t* w, int m, int mx, int g, int lane,
                                      f32x4 (&acc)[NMT]) {
#pragma unroll
  for (int mt = 0; mt < NMT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a <= PY; ++a)
#pragma unroll
    for (int b = 0; b <= PX; ++b) {
      const int ky = PY ? 2 * a : 1, kx = PX ? 2 * b : 1;
      const int oy = m + (PY && a == 0 ? 1 : 0), ox = mx + (PX && b == 0 ? 1 : 0);
      const u16x8 bf = ldfrag(d + (oy * PD + ox) * CH + swz(ox, g));
#pragma unroll
      for (int mt = 0; mt < NMT; ++mt)
        acc[mt] = mfma(ldfrag(w + (((MT0 + mt) * 9 + ky * 3 + kx) * 64 + lane) * 8), bf, acc[mt]);
    }
}

// relu mask of four channels (bf16 activations, zero or positive) on a
// gradient, its bias sum, and the bf16 image of it
__device__ __forceinline__ uint2 mask4(f32x4& v, uint2 a, f32x4& bias) {
  if (!(__uint_as_float(a.x << 16) > 0.f)) v[0] = 0.f;
  if (!(__uint_as_float(a.x & 0xFFFF0000u) > 0.f)) v[1] = 0.f;
  if (!(__uint_as_float(a.y << 16) > 0.f)) v[2] = 0.f;
  if (!(__uint_as_float(a.y & 0xFFFF0000u) > 0.f)) v[3] = 0.f;
  bias += v;
  return make_uint2(cvt2(v[0], v[1]), cvt2(v[2], v[3]));
}

// Backward of the four convolutions, sample by sample, one block of 8
// wavefronts per CU: from the gradient of the features down to the first
// layer, every gradient image in LDS (bf16, channels last), the weight
// gradients summed over the block's samples in its part of memory, the bias
// gradients from the unrounded FP32 values.  The gradient of conv 1's output
// takes the place of its activations once conv 2's weight gradient has read
// them (142 KiB in all).  Bound by the LDS reads of the fragments and, at one
// sample per block, by loading its activations (102 KiB).
// x, idx: input windows; y1..y3 (channels last) and df from the forward pass
// and the head; part[block][PART]: the block's sums.  grid: min(n, CUs)
__global__ __launch_bounds__(NET_THREADS) void k_net_bwd(const uint16_t* __restrict__ x, const int* __restrict__ idx,
                                                         const uint16_t* __restrict__ wp,
                                                         const uint16_t* __restrict__ y1,
                                                         const uint16_t* __restrict__ y2,
                                                         const uint16_t* __restrict__ y3,
                                                         const float* __restrict__ df, int n,
                                                         float* __restrict__ part) {
  constexpr int P0 = 34, P2 = 18, P3 = 10, D2 = 17, D3 = 9, D4 = 5;
  __shared__ __align__(16) uint16_t s_x[P0 * P0 * 8];
  __shared__ __align__(16) uint16_t s_1[P0 * P0 * CH];
  __shared__ __align__(16) uint16_t s_2[P2 * P2 * CH];
  __shared__ __align__(16) uint16_t s_3[P3 * P3 * CH];
  __shared__ __align__(16) uint16_t s_d2[D2 * D2 * CH];
  __shared__ __align__(16) uint16_t s_d3[D3 * D3 * CH];
  __shared__ __align__(16) uint16_t s_d4[D4 * D4 * CH];
  const int tid = threadIdx.x, lane = tid & 63;
  int g = lane >> 4, r = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto zero = [&](uint16_t* p, int cnt) {
    for (int i = tid; i < cnt / 8; i += NET_THREADS) reinterpret_cast<u16x8*>(p)[i] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  };
  zero(s_x, P0 * P0 * 8);
  zero(s_1, P0 * P0 * CH);
  zero(s_2, P2 * P2 * CH);
  zero(s_3, P3 * P3 * CH);
  zero(s_d2, D2 * D2 * CH);
  zero(s_d3, D3 * D3 * CH);
  zero(s_d4, D4 * D4 * CH);
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  f32x4 bs1[2] = {z4, z4}, bs2[2] = {z4, z4}, bs3 = z4;
  float bs4 = 0.f;
  float* out = part + (long long)blockIdx.x * PART;
  __syncthreads();
  for (int sample = blockIdx.x; sample < n; sample += gridDim.x) {
    const bool add = sample != (int)blockIdx.x;
    // hidden from the optimiser: weight fragments and the many offsets derived
    // from the lane are formed where they are used instead of being kept (and
    // spilled) over the samples
    const uint16_t* wb = wp + PACK_B;
    __asm__ volatile("" : "+s"(wb));
    __asm__ volatile("" : "+s"(out));
    __asm__ volatile("" : "+v"(r), "+v"(g));
    // ---- the sample's images into LDS
    const long long win = idx ? idx[sample] : sample;
    {
      const uint32_t* xn = reinterpret_cast<const uint32_t*>(x + win * (8 * 1024)) + tid;
      uint32_t in[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) in[c] = xn[c * 512];
      u16x8 t1[8], t2[2];
      const u16x8* a1 = reinterpret_cast<const u16x8*>(y1) + (long long)sample * 4096;
      const u16x8* a2 = reinterpret_cast<const u16x8*>(y2) + (long long)sample * 1024;
#pragma unroll
      for (int k = 0; k < 8; ++k) t1[k] = a1[tid + 512 * k];
#pragma unroll
      for (int k = 0; k < 2; ++k) t2[k] = a2[tid + 512 * k];
      const uint2 t3 = reinterpret_cast<const uint2*>(y3)[(long long)sample * 512 + tid];
      const float d = df[(long long)sample * 512 + tid];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int e = tid + 512 * k, p = e >> 2, q = e & 3, iy = p >> 5, ix = p & 31;
        *reinterpret_cast<u16x8*>(s_1 + ((iy + 1) * P0 + ix + 1) * CH + swz(ix + 1, q)) = t1[k];
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = tid + 512 * k, p = e >> 2, q = e & 3, iy = p >> 4, ix = p & 15;
        *reinterpret_cast<u16x8*>(s_2 + ((iy + 1) * P2 + ix + 1) * CH + swz(ix + 1, q)) = t2[k];
      }
      {
        const int p = tid >> 3, q = tid & 7, iy = p >> 3, ix = p & 7;
        *reinterpret_cast<uint2*>(s_3 + ((iy + 1) * P3 + ix + 1) * CH + swz(ix + 1, q >> 1) + 4 * (q & 1)) = t3;
      }
      {
        const int p = 2 * tid, iy = p >> 5, ix = p & 31;
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          lo[c] = (in[2 * c] & 0xffffu) | (in[2 * c + 1] << 16);
          hi[c] = (in[2 * c] >> 16) | (in[2 * c + 1] & 0xffff0000u);
        }
        uint4* dst = reinterpret_cast<uint4*>(&s_x[((iy + 1) * P0 + ix + 1) * 8]);
        dst[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        dst[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      }
      {  // feature gradient: thread = channel (tid / 16), pixel (tid % 16)
        const int co = tid >> 4, p = tid & 15, oy = p >> 2, ox = p & 3;
        s_d4[(oy * D4 + ox) * CH + swz(ox, co >> 3) + (co & 7)] = f2bf_rne(d);
        bs4 += d;
      }
    }
    __syncthreads();
    // ---- conv 4: weight gradient, and the data gradient of one parity class
    // and channel tile per wavefront
    wgrad<4, D4, P3>(s_d4, s_3, wv, g, r, add, out + part_off(3));
    {
      const int mt = wv & 1, cls = wv >> 1, py = cls >> 1, px = cls & 1, m = r >> 2, mx = r & 3;
      const uint16_t* w = wb + (2 * 2 + mt) * 9 * 512;
      f32x4 acc[1];
      if (cls == 0) dgrad<0, 0, D4, 0, 1>(s_d4, w, m, mx, g, lane, acc);
      else if (cls == 1) dgrad<0, 1, D4, 0, 1>(s_d4, w, m, mx, g, lane, acc);
      else if (cls == 2) dgrad<1, 0, D4, 0, 1>(s_d4, w, m, mx, g, lane, acc);
      else dgrad<1, 1, D4, 0, 1>(s_d4, w, m, mx, g, lane, acc);
      const int iy = 2 * m + py, ix = 2 * mx + px, c = 4 * (g & 1), q = 2 * mt + (g >> 1);
      const uint2 a = *reinterpret_cast<const uint2*>(s_3 + ((iy + 1) * P3 + ix + 1) * CH + swz(ix + 1, q) + c);
      *reinterpret_cast<uint2*>(s_d3 + (iy * D3 + ix) * CH + swz(ix, q) + c) = mask4(acc[0], a, bs3);
    }
    __syncthreads();
    // ---- conv 3: 64 pixels per parity class, two groups of 16 per wavefront
    wgrad<8, D3, P2>(s_d3, s_2, wv, g, r, add, out + part_off(2));
    auto down3 = [&](auto PYX, int k) {  // group k (16 pixels) of a class
      constexpr int py = decltype(PYX)::value >> 1, px = decltype(PYX)::value & 1;
      const int p = k * 16 + r, m = p >> 3, mx = p & 7, iy = 2 * m + py, ix = 2 * mx + px;
      f32x4 acc[2];
      dgrad<py, px, D3, 0, 2>(s_d3, wb + 2 * 9 * 512, m, mx, g, lane, acc);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int c = 4 * (g & 1), q = 2 * mt + (g >> 1);
        const uint2 a = *reinterpret_cast<const uint2*>(s_2 + ((iy + 1) * P2 + ix + 1) * CH + swz(ix + 1, q) + c);
        *reinterpret_cast<uint2*>(s_d2 + (iy * D2 + ix) * CH + swz(ix, q) + c) = mask4(acc[mt], a, bs2[mt]);
      }
    };
    if (wv < 4) {
      down3(std::integral_constant<int, 0>{}, wv);
      down3(std::integral_constant<int, 3>{}, wv);
    } else {
      down3(std::integral_constant<int, 1>{}, wv - 4);
      down3(std::integral_constant<int, 2>{}, wv - 4);
    }
    __syncthreads();
    // ---- conv 2: the weight gradient reads the activations that the data
    // gradient then replaces
    wgrad<16, D2, P0>(s_d2, s_1, wv, g, r, add, out + part_off(1));
    __syncthreads();
    auto down2 = [&](auto PYX) {
      constexpr int py = decltype(PYX)::value >> 1, px = decltype(PYX)::value & 1;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int p = (wv + 8 * k) * 16 + r, m = p >> 4, mx = p & 15, iy = 2 * m + py, ix = 2 * mx + px;
        f32x4 acc[2];
        dgrad<py, px, D2, 0, 2>(s_d2, wb, m, mx, g, lane, acc);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          uint2* a = reinterpret_cast<uint2*>(s_1 + ((iy + 1) * P0 + ix + 1) * CH +
                                              swz(ix + 1, 2 * mt + (g >> 1)) + 4 * (g & 1));
          *a = mask4(acc[mt], *a, bs1[mt]);
        }
      }
    };
    down2(std::integral_constant<int, 0>{});
    down2(std::integral_constant<int, 1>{});
    down2(std::integral_constant<int, 2>{});
    down2(std::integral_constant<int, 3>{});
    __syncthreads();
    // ---- conv 1: weight gradient, wavefront wv < 5 the columns of taps 2 wv,
    // 2 wv + 1 (8 channels each; the tenth tap is not written out), K the 32
    // image rows
    if (wv < 5) {
      const int cg = (r & 3) >> 1, half = 4 * (r & 1), x0 = 8 * g + (r >> 2), x1 = x0 + 4;
      const int t = 2 * wv + cg < 9 ? 2 * wv + cg : 8, o = ((t / 3) * P0 + t % 3) * 8 + half;
      f32x4 acc[2] = {z4, z4};
#pragma unroll 4
      for (int oy = 0; oy < 32; ++oy) {
        const u16x8 b = ldtr(s_x + oy * P0 * 8 + o + x0 * 8, s_x + oy * P0 * 8 + o + x1 * 8);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          acc[mt] = mfma(ldtr(s_1 + ((oy + 1) * P0 + x0 + 1) * CH + swz(x0 + 1, 2 * mt + cg) + half,
                              s_1 + ((oy + 1) * P0 + x1 + 1) * CH + swz(x1 + 1, 2 * mt + cg) + half),
                         b, acc[mt]);
      }
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        f32x4* q = reinterpret_cast<f32x4*>(out) + (2 * wv + mt) * 64 + lane;
        *q = add ? *q + acc[mt] : acc[mt];
      }
    }
    __syncthreads();
  }
  // biases: over the 16 pixels of a fragment, then the wavefronts
  float* rb = reinterpret_cast<float*>(s_2);  // [8][80]: 32 of conv 1, 32 of conv 2, 16 of conv 3
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        bs1[mt][i] += __shfl_xor(bs1[mt][i], o, 64);
        bs2[mt][i] += __shfl_xor(bs2[mt][i], o, 64);
      }
      bs3[i] += __shfl_xor(bs3[i], o, 64);
    }
    bs4 += __shfl_xor(bs4, o, 64);
  }
  if (r == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        rb[wv * 80 + 16 * mt + 4 * g + i] = bs1[mt][i];
        rb[wv * 80 + 32 + 16 * mt + 4 * g + i] = bs2[mt][i];
      }
      rb[wv * 80 + 64 + 4 * g + i] = bs3[i];
    }
    out[PART_B + 3 * CH + (tid >> 4)] = bs4;
  }
  __syncthreads();
  if (tid < 96) {
    const int l = tid >> 5, c = tid & 31;  // bias c of conv l + 1
    float v = 0.f;
    for (int w = 0; w < 8; ++w) {
      if (l == 2) v += (w & 1) == (c >> 4) ? rb[w * 80 + 64 + (c & 15)] : 0.f;
      else v += rb[w * 80 + 32 * l + c];
    }
    out[PART_B + tid] = v;
  }
}

}  // namespace nnmfma
