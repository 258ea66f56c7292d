// jms_nn_mfma.hpp -- the surrogate's 3x3 convolutions as implicit GEMMs on
// the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16: bf16 operands, FP32
// accumulation), included by jms_nn.hip.
//
// One block of 256 threads (4 wavefronts) per sample.  The layer input (or,
// for the data gradient, the output gradient) is staged once into LDS in a
// channels-last layout with a one-pixel zero border, so that the 8 bf16
// values of an MFMA operand fragment -- 8 consecutive channels at one
// (pixel, tap) -- are one aligned 16-byte LDS read and the padding needs no
// bounds checks.  The GEMM K index runs over (tap, 8-channel group); weights
// are loaded once per wavefront into registers as A fragments.
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
constexpr int PACK_SIZE = PACK_D1 + 64 * 512;    // bf16 elements
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
// grid: min(n, CUs); feat[n][512] in channel-major order
constexpr int NET_THREADS = 512;
template <bool KEEP>
__global__ __launch_bounds__(NET_THREADS) void k_net_fwd(const uint16_t* __restrict__ x,
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
  auto load_in = [&](long long sample) {
    const uint32_t* xn = reinterpret_cast<const uint32_t*>(x + sample * (8 * 1024)) + tid;
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
// grid: ceil(n / (16 NS)), block: 1024; hid (training) [n][64]
template <int NS>
__global__ __launch_bounds__(1024) void k_head(const uint16_t* __restrict__ feat, const uint16_t* __restrict__ w1t,
                                               const float* __restrict__ b1, const uint16_t* __restrict__ w2,
                                               const float* __restrict__ b2, int n, uint16_t* __restrict__ hid,
                                               float* __restrict__ out) {
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
    const uint16_t h = f2bf_rne(fmaxf(acc[s], 0.f));
    s_h[wv][s][lane] = h;
    if (hid && s0 + s < n) hid[(long long)(s0 + s) * 64 + lane] = h;
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

// y[n][co][oy][ox] = relu(b[co] + sum_{ci,ky,kx} x[n][ci][oy*S+ky-1][ox*S+kx-1] w[co][ci][ky][kx])
// grid: one block per sample
template <int S, int CI, int HIN>
__global__ __launch_bounds__(256) void k_conv_fwd(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                  const float* __restrict__ b, uint16_t* __restrict__ y) {
  constexpr int HP = HIN + 2, HOUT = HIN / S, NPIX = HOUT * HOUT;
  constexpr int KG = 9 * CI / 8;          // K groups of 8 (tap, channel group)
  constexpr int KS = (KG + 3) / 4;        // K steps of 32
  constexpr int CG = CI / 8;
  __shared__ __align__(16) uint16_t xs[HP * HP * CI];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, r = lane & 15;
  const long long n = blockIdx.x;
  // zero the whole staging area (border included), then the interior
  for (int i = tid; i < HP * HP * CI / 2; i += 256) reinterpret_cast<uint32_t*>(xs)[i] = 0u;
  __syncthreads();
  const uint16_t* xn = x + n * CI * HIN * HIN;
  for (int i = tid; i < CI * HIN * HIN; i += 256) {
    const int c = i / (HIN * HIN), p = i % (HIN * HIN), iy = p / HIN, ix = p % HIN;
    xs[((iy + 1) * HP + ix + 1) * CI + c] = xn[i];
  }
  // A fragments: w[co][ci0+j][tap] for co = mt*16 + r
  u16x8 af[2][KS];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kg = ks * 4 + g;
      const int co = mt * 16 + r;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        uint16_t v = 0;
        if (kg < KG) {
          const int t = kg / CG, ci = (kg % CG) * 8 + j;
          v = w[(co * CI + ci) * 9 + t];
        }
        af[mt][ks][j] = v;
      }
    }
  __syncthreads();
  uint16_t* yn = y + n * CH * NPIX;
  for (int gi = wv; gi < NPIX / 16; gi += 4) {
    const int p = gi * 16 + r, oy = p / HOUT, ox = p % HOUT;
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kg = ks * 4 + g;
      u16x8 bf = {0, 0, 0, 0, 0, 0, 0, 0};
      if (kg < KG) {
        const int t = kg / CG, c0 = (kg % CG) * 8, ky = t / 3, kx = t % 3;
        bf = *reinterpret_cast<const u16x8*>(&xs[((oy * S + ky) * HP + ox * S + kx) * CI + c0]);
      }
      acc0 = mfma(af[0][ks], bf, acc0);
      acc1 = mfma(af[1][ks], bf, acc1);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int co0 = 4 * g + i, co1 = 16 + 4 * g + i;
      yn[co0 * NPIX + p] = f2bf_rne(fmaxf(acc0[i] + b[co0], 0.f));
      yn[co1 * NPIX + p] = f2bf_rne(fmaxf(acc1[i] + b[co1], 0.f));
    }
  }
}

// dx[n][ci][iy][ix] = [a[n][ci][iy][ix] > 0] * sum_{co,ky,kx} dy[n][co][oy][ox] w[co][ci][ky][kx]
// over iy = oy*S + ky - 1, ix = ox*S + kx - 1 (CI = CH); dy is rounded to
// bf16 as it is staged.  grid: one block per sample
template <int S, int HIN>
__global__ __launch_bounds__(256) void k_conv_bwd_data(const float* __restrict__ dy, const uint16_t* __restrict__ w,
                                                       const uint16_t* __restrict__ a, float* __restrict__ dx) {
  constexpr int CI = CH, HOUT = HIN / S, HP = HOUT + 2, NPIN = HIN * HIN, NPOUT = HOUT * HOUT;
  constexpr int KS = 9;  // 36 K groups (tap, 8-channel group of co) in steps of 4
  __shared__ __align__(16) uint16_t gs[HP * HP * CH];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, r = lane & 15;
  const long long n = blockIdx.x;
  for (int i = tid; i < HP * HP * CH / 2; i += 256) reinterpret_cast<uint32_t*>(gs)[i] = 0u;
  __syncthreads();
  const float* dyn = dy + n * CH * NPOUT;
  for (int i = tid; i < CH * NPOUT; i += 256) {
    const int c = i / NPOUT, p = i % NPOUT, oy = p / HOUT, ox = p % HOUT;
    gs[((oy + 1) * HP + ox + 1) * CH + c] = f2bf_rne(dyn[i]);
  }
  // A fragments: w[co0+j][ci][tap] for ci = mt*16 + r
  u16x8 af[2][KS];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kg = ks * 4 + g, t = kg / 4, co0 = (kg % 4) * 8, ci = mt * 16 + r;
#pragma unroll
      for (int j = 0; j < 8; ++j) af[mt][ks][j] = w[((co0 + j) * CI + ci) * 9 + t];
    }
  __syncthreads();
  const uint16_t* an = a + n * CI * NPIN;
  float* dxn = dx + n * CI * NPIN;
  for (int gi = wv; gi < NPIN / 16; gi += 4) {
    const int p = gi * 16 + r, iy = p / HIN, ix = p % HIN;
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kg = ks * 4 + g, t = kg / 4, co0 = (kg % 4) * 8, ky = t / 3, kx = t % 3;
      const int ty = iy + 1 - ky, tx = ix + 1 - kx;  // in [-1, HIN]
      int slot = 0;                                   // the zero border pixel (0, 0)
      if (S == 1 || ((ty & 1) == 0 && (tx & 1) == 0)) {
        const int oy = (S == 1) ? ty : (ty >> 1), ox = (S == 1) ? tx : (tx >> 1);  // in [-1, HOUT]
        slot = (oy + 1) * HP + ox + 1;
      }
      const u16x8 bf = *reinterpret_cast<const u16x8*>(&gs[slot * CH + co0]);
      acc0 = mfma(af[0][ks], bf, acc0);
      acc1 = mfma(af[1][ks], bf, acc1);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ci0 = 4 * g + i, ci1 = 16 + 4 * g + i;
      const long long o0 = (long long)ci0 * NPIN + p, o1 = (long long)ci1 * NPIN + p;
      dxn[o0] = (__uint_as_float((uint32_t)an[o0] << 16) > 0.f) ? acc0[i] : 0.f;
      dxn[o1] = (__uint_as_float((uint32_t)an[o1] << 16) > 0.f) ? acc1[i] : 0.f;
    }
  }
}

// per-sample partial weight gradient:
//   part[n][co][ci][tap] = sum_{oy,ox} dy[n][co][oy][ox] x[n][ci][oy*S+ky-1][ox*S+kx-1]
// (dy rounded to bf16).  The GEMM: rows co, columns c = ci*9 + tap, K the
// sample's output pixels.  grid: one block per sample
template <int S, int CI, int HIN>
__global__ __launch_bounds__(256) void k_conv_bwd_w(const float* __restrict__ dy, const uint16_t* __restrict__ x,
                                                    float* __restrict__ part) {
  constexpr int HP = HIN + 2, HOUT = HIN / S, NPOUT = HOUT * HOUT;
  constexpr int NCOL = CI * 9, NT = (NCOL + 15) / 16;  // column tiles
  constexpr int KS = (NPOUT + 31) / 32;                // K steps over the output pixels
  constexpr int NPAD = KS * 32;
  __shared__ __align__(16) uint16_t xs[CI * HP * HP];  // [ci][HP][HP], zero border
  __shared__ __align__(16) uint16_t gs[CH * NPAD];     // [co][p], bf16, zero beyond NPOUT
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, r = lane & 15;
  const long long n = blockIdx.x;
  for (int i = tid; i < CI * HP * HP / 2; i += 256) reinterpret_cast<uint32_t*>(xs)[i] = 0u;
  for (int i = tid; i < CH * NPAD / 2; i += 256) reinterpret_cast<uint32_t*>(gs)[i] = 0u;
  __syncthreads();
  const uint16_t* xn = x + n * CI * HIN * HIN;
  for (int i = tid; i < CI * HIN * HIN; i += 256) {
    const int c = i / (HIN * HIN), p = i % (HIN * HIN), iy = p / HIN, ix = p % HIN;
    xs[(c * HP + iy + 1) * HP + ix + 1] = xn[i];
  }
  const float* dyn = dy + n * CH * NPOUT;
  for (int i = tid; i < CH * NPOUT; i += 256) gs[(i / NPOUT) * NPAD + i % NPOUT] = f2bf_rne(dyn[i]);
  __syncthreads();
  float* pn = part + n * CH * NCOL;
  for (int nt = wv; nt < NT; nt += 4) {
    const int c = nt * 16 + r;  // this lane's column
    const bool cok = c < NCOL;
    const int ci = cok ? c / 9 : 0, t = cok ? c % 9 : 0, ky = t / 3, kx = t % 3;
    const uint16_t* xc = xs + ci * HP * HP;
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < KS; ++ks) {
      const int k0 = ks * 32 + 8 * g;  // first output pixel of this lane's K elements
      const u16x8 a0 = *reinterpret_cast<const u16x8*>(&gs[r * NPAD + k0]);
      const u16x8 a1 = *reinterpret_cast<const u16x8*>(&gs[(16 + r) * NPAD + k0]);
      u16x8 bf;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int p = k0 + j;
        uint16_t v = 0;
        if (cok && p < NPOUT) {
          const int oy = p / HOUT, ox = p % HOUT;
          v = xc[(oy * S + ky) * HP + ox * S + kx];
        }
        bf[j] = v;
      }
      acc0 = mfma(a0, bf, acc0);
      acc1 = mfma(a1, bf, acc1);
    }
    if (cok) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pn[(4 * g + i) * NCOL + c] = acc0[i];
        pn[(16 + 4 * g + i) * NCOL + c] = acc1[i];
      }
    }
  }
}

// dw[i] += sum over this block's share of the samples of part[n][i] (i <
// cnt); dw is cleared first.  grid: (ceil(cnt / 256), shares)
__global__ __launch_bounds__(256) void k_reduce_parts(const float* __restrict__ part, int nsamp, int cnt,
                                                      float* __restrict__ dw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  const int k0 = (int)((long long)nsamp * blockIdx.y / gridDim.y);
  const int k1 = (int)((long long)nsamp * (blockIdx.y + 1) / gridDim.y);
  float s = 0.f;
  for (int k = k0; k < k1; ++k) s += part[(long long)k * cnt + i];
  atomicAdd(&dw[i], s);
}

// db[co] += sum over this block's share of the samples of dy[n][co][p];
// db is cleared first.  grid: (CH, shares)
__global__ __launch_bounds__(256) void k_bias_grad(const float* __restrict__ dy, int nsamp, int npix,
                                                   float* __restrict__ db) {
  const int co = blockIdx.x;
  const int k0 = (int)((long long)nsamp * blockIdx.y / gridDim.y);
  const int k1 = (int)((long long)nsamp * (blockIdx.y + 1) / gridDim.y);
  float s = 0.f;
  for (int k = k0; k < k1; ++k) {
    const float* d = dy + ((long long)k * CH + co) * npix;
    for (int p = threadIdx.x; p < npix; p += 256) s += d[p];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  __shared__ float red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(&db[co], red[0] + red[1] + red[2] + red[3]);
}

}  // namespace nnmfma
