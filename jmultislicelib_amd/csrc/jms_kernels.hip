// jms_kernels.hip -- size dispatch of the line-length templated kernels and
// the small non-templated kernels (readout combine, incident-wave offset,
// accumulation).
#include <hip/hip_runtime.h>
#include <mutex>
#include <vector>
#include <cstdint>
#include "jms_fft_device.hpp"
#include "jms_kernels.h"
#include "jms_sizes.h"
#include "jms_cfg.hpp"

namespace jms {

template <int N>
hipError_t launch_row_pass_n(int ny, int nwave, float2* wave, long long wave_stride,
                             const float2* pgr, long long slc_off, long long npg,
                             const int* var_tab, int var_ld, int jslc, const float2* twx,
                             const RowChanHost& rc, int mode, bool panel, const BandHost& bd, Shape shape,
                             hipStream_t st);
template <int N>
hipError_t launch_col_pass_n(int nwave, bool init, bool exit_, const ColArgsHost& h,
                             hipStream_t st);
template <int N>
hipError_t launch_row_fft_n(int ny, int nbatch, float2* data, long long stride, int dir,
                            const float2* twx, hipStream_t st);
template <int N>
hipError_t launch_col_fft_n(int nx, int nbatch, float2* data, long long stride, int dir,
                            const float2* twy, hipStream_t st);
template <int N>
hipError_t launch_row_pass_grp_n(int ny, int nwave, long long wave_stride, long long npg, const float2* twx,
                                 const GrpArgs& ga, bool panel, const BandHost& bd, hipStream_t st);
template <int N>
hipError_t launch_col_pass_grp_n(int nx, int nwave, bool init, bool exit_, bool detect, long long part_dstride,
                                 const float2* twy, const GrpArgs& ga, bool panel, const BandHost& bd,
                                 hipStream_t st);
template <int NX>
void band_row_n(int x0, int x1, int tile, BandHost& b);
template <int NX, int NY>
hipError_t launch_loop_n(int nwave, const LoopArgs& a, bool band, hipStream_t st);
template <int NY>
bool band_col_n(int y0, int y1);

// frequency index of position i on an n-point grid in FFT order
// (JMultiSlice.cpp:1699-1712)
__device__ __forceinline__ int fidx(int i, int n) {
  const int h = (n - (n & 1)) >> 1;
  return ((i + h) % n) - h;
}

// ---------------------------------------------------------------------------
// combine partial detector sums of a batch into per-position results:
//   out[(p0+p), idet, d] (+)= sum_r weight[r] * sum_tile partial[(p*npass+r), idet, d, tile]
// mirror (or nullptr): the same values in host memory, for a caller that reads
// them right after the run
// ---------------------------------------------------------------------------
__global__ void k_combine(const float* __restrict__ partial, int ntiles, int ndet, int ndetslc,
                          int npos, int npass, const float* __restrict__ weights,
                          float* __restrict__ out, int accumulate, float* __restrict__ mirror) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int per = ndetslc * ndet;
  if (i >= npos * per) return;
  const int p = i / per, r0 = i % per;  // r0 = idet*ndet + d
  double acc = 0.0;
  for (int r = 0; r < npass; ++r) {
    const float* src = partial + ((long long)(p * npass + r) * per + r0) * ntiles;
    double s = 0.0;
    for (int k = 0; k < ntiles; ++k) s += (double)src[k];
    acc += (double)weights[r] * s;
  }
  const float r = accumulate ? (float)((double)out[i] + acc) : (float)acc;
  out[i] = r;
  if (mirror) mirror[i] = r;
}

__global__ void k_zero_partial(float* __restrict__ partial, long long part_w, long long off, int len) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < len) partial[blockIdx.y * part_w + off + k] = 0.f;
}

// psi_out = psi0 * exp(-i [2 pi (kx dx + ky dy + k^2 fz) + cppl]) in Fourier space
// (OffsetIncomingWave GPU branch, JMultiSlice.cpp:2036-2077; ArrayOps.cu:390-422),
// with an optional cyclic beam-tilt shift of psi0 by (ish0, ish1) pixels
// (CShift2dKernel, ArrayOps.cu:340-352).
__global__ void k_offset_wave(float2* __restrict__ out, const float2* __restrict__ in, int nx,
                              int ny, float kscx, float kscy, float dx, float dy, float fz,
                              const float* __restrict__ cppl, int ish0, int ish1) {
  const long long n = (long long)nx * ny;
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int i = (int)(idx % nx), j = (int)(idx / nx);
  const float kx = (float)fidx(i, nx) * kscx, ky = (float)fidx(j, ny) * kscy;
  const float ksqr = kx * kx + ky * ky;
  float chi = -6.28318531f * (dx * kx + dy * ky + fz * ksqr);
  if (cppl) chi -= cppl[idx];
  float sn, cs;
  sincosf(chi, &sn, &cs);
  int i0 = i - ish0, j0 = j - ish1;
  i0 %= nx; if (i0 < 0) i0 += nx;
  j0 %= ny; if (j0 < 0) j0 += ny;
  out[idx] = cmul(in[(long long)i0 + (long long)j0 * nx], make_float2(cs, sn));
}

// ---------------------------------------------------------------------------
// probe in Fourier space on the device: the aperture of ApertureFunctionA
// (JProbeGen.cpp:471-505) times exp(-i chi) with the axial aberration phase
// of AberrationFunction (JProbeGen.cpp:508-571), then normalised to unit
// intensity (CalculateProbeWaveFourier, JProbeGen.cpp:707-777).
// ---------------------------------------------------------------------------
__device__ float probe_chi(float qx, float qy, const ProbeArgsHost& a) {
  const float wx = qx * a.wl, wy = qy * a.wl;
  const float w = sqrtf(wx * wx + wy * wy);
  float px[9], py[9], pw[9];
  px[0] = py[0] = pw[0] = 1.f;
#pragma unroll
  for (int i = 1; i < 9; ++i) { px[i] = px[i - 1] * wx; py[i] = py[i - 1] * wy; pw[i] = pw[i - 1] * w; }
  const float re_il[4] = {1.f, 0.f, -1.f, 0.f};
  float sum = 0.f;
  for (int k = 0; k < a.nab; ++k) {
    const float cx = a.coeff[2 * k], cy = a.coeff[2 * k + 1];
    if (cx * cx + cy * cy > 1.0e-15f) {
      const int m = a.mn[2 * k], n = a.mn[2 * k + 1];
      float term = 0.f;
      for (int l = 0; l <= n; ++l) {
        float c = 0.f;
        c = c + re_il[l & 3] * cx;
        c = c + re_il[(l + 3) & 3] * cy;
        term = term + c * (float)a.binom[n + 9 * l] * px[n - l] * py[l];
      }
      sum = sum + term * pw[m - n] / (float)m;
    }
  }
  return sum * (6.28318530717958648f / a.wl);
}

__global__ void k_probe(float2* __restrict__ out, double* __restrict__ partial, ProbeArgsHost a) {
  __shared__ double red[256];
  const long long n = (long long)a.nx * a.ny;
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double pw = 0.0;
  if (idx < n) {
    const int i = (int)(idx % a.nx), j = (int)(idx / a.nx);
    const float qx = (float)fidx(i, a.nx) / a.ax, qy = (float)fidx(j, a.ny) / a.ay;
    float amp = 0.f;
    if (a.qlim > 0.f && a.open) {
      const float dqx = (qx - a.btx) - a.qlcx, dqy = (qy - a.bty) - a.qlcy;
      const float ux = ((1.f - a.a1x) * dqx - a.a1y * dqy) * a.radet;
      const float uy = (-a.a1y * dqx + (1.f + a.a1x) * dqy) * a.radet;
      const float dqm = sqrtf(ux * ux + uy * uy);
      const float dqs = fabsf(a.qrs * a.qlim);
      if (dqm <= 0.f) amp = 1.f;
      else if (dqs > 0.f) amp = (1.f - tanhf(3.14159265358979324f * (dqm - a.qlim) / dqs)) * 0.5f;
      else if (dqm < a.qlim) amp = 1.f;
    }
    float2 v = make_float2(0.f, 0.f);
    if (amp > 1.0e-6f) {
      const float chi = a.nab > 0 ? probe_chi(qx, qy, a) : 0.f;
      float sn, cs;
      sincosf(chi, &sn, &cs);
      v = make_float2(amp * cs, -amp * sn);
      pw = (double)(amp * amp);
    }
    out[idx] = v;
  }
  red[threadIdx.x] = pw;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_probe_scale(float2* __restrict__ out, const double* __restrict__ partial, int nblk,
                              long long n) {
  __shared__ double red[256];
  double s = 0.0;
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) s += partial[b];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  const float fsca = 1.f / sqrtf((float)red[0]);
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < n) {
    float2 v = out[idx];
    v.x *= fsca;
    v.y *= fsca;
    out[idx] = v;
  }
}

// ---------------------------------------------------------------------------
// phase gratings of the Gaussian projected-potential model on the device
// (the host generator jms_gaussian_phase_grating, evaluated per pixel): each
// pixel adds amp * exp(-r^2 / (2 s^2)) of every atom image within the cut-off
// in the host's order (atoms ascending; per atom, pixel rows then columns of
// the unwrapped range), in double, then t = exp(i sig_int V).
// grid: (ceil(nx/16), ceil(ny/16), nvar), block: 16 x 16
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_gauss_gratings(float2* __restrict__ out, int nx, int ny, double hx,
                                                        double hy, double rc2, double inv2s2, double sig_int,
                                                        const GaussAtom* __restrict__ atoms,
                                                        const int* __restrict__ off, const int* __restrict__ idx) {
  const int px = blockIdx.x * 16 + threadIdx.x, py = blockIdx.y * 16 + threadIdx.y;
  const int v = blockIdx.z;
  const int ntx = (nx + 15) / 16, nty = (ny + 15) / 16, ntiles = ntx * nty;
  const int t = blockIdx.y * ntx + blockIdx.x;
  const int* o = off + (long long)v * (ntiles + 1);
  const int a0 = o[t], a1 = o[t + 1];
  if (px >= nx || py >= ny) return;
  double pot = 0.0;
  for (int k = a0; k < a1; ++k) {
    const GaussAtom at = atoms[idx[k]];
    // unwrapped rows j = py + m ny and columns i = px + l nx inside the range
    int j = at.j0 + (((py - at.j0) % ny) + ny) % ny;
    for (; j <= at.j1; j += ny) {
      const double dy = j * hy - at.ya;
      const double dy2 = dy * dy;
      if (dy2 > rc2) continue;
      int i = at.i0 + (((px - at.i0) % nx) + nx) % nx;
      for (; i <= at.i1; i += nx) {
        const double dx = i * hx - at.xa;
        const double r2 = dx * dx + dy2;
        if (r2 > rc2) continue;
        pot += at.amp * exp(-r2 * inv2s2);
      }
    }
  }
  const double ph = sig_int * pot;
  out[(long long)v * nx * ny + (long long)py * nx + px] = make_float2((float)cos(ph), (float)sin(ph));
}

// ---------------------------------------------------------------------------
// phase gratings from projected atomic form factors (CalculatePhasegratingGPU,
// JEElaSca.cpp:978-1159; AddFormFactor2dKernel / PotToPgrKernel,
// scapot.cu:29-41,80-89).  Spatial frequencies in FFT order [1/nm],
// q = fidx(i) * (1 / a) (InitHelper, JEElaSca.cpp:529-541); every product
// and sum that decides an aperture edge is rounded as written, so that the
// edge pixels do not depend on contraction.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float ff_freq(int i, int n, float itog) { return __fmul_rn((float)fidx(i, n), itog); }
__device__ __forceinline__ float ff_gmag(float qx, float qy) {
  return __fsqrt_rn(__fadd_rn(__fmul_rn(qx, qx), __fmul_rn(qy, qy)));
}

// Fourier-space projected potential of atom set v (atoms off[v] .. off[v+1],
// grouped by type, ascending atom order inside a type):
//   pot(q) = sum_t ff_t(q) ap(q) sum_{atoms of t} occ exp(-2 pi i (x qx + y qy))
// ap(q) = 1/2 - 1/2 tanh(30 (|q|/kmax - 0.9)) with the potential band limit,
// else 1 (JEElaSca.cpp:592-595).  The phase factor is one of x times one of y,
// so the sum over the atoms of a type is a product of two thin matrices: a
// block of (16 P)^2 pixels takes kFFChunk atoms at a time, computes their
// factors once per column and row (the phase in turns in double, reduced, sine
// and cosine in double, rounded: the product is then no further from exact
// than one float sine and cosine of the whole phase) and adds outer products,
// P x P pixels a thread from 2 P values in LDS.  Bound by the float FMAs (four
// per atom and pixel) where one sine and cosine per atom and pixel was: 8
// variants of 512^2, 160 atoms each, 364 -> 99 us on MI355X (34 of them the FMAs
// at 80 TFLOP/s; with float sines and cosines 94; in tiles of 32 or 48 pixels
// 125 and 150, as the factors are computed more often).
// Every thread walks the same list, so the type switches are uniform.
// grid: (ceil(nx / 16 P), ceil(ny / 16 P), nvar), block: 256
constexpr int kFFChunk = 32;
template <int P>
__global__ __launch_bounds__(256) void k_ff_sum(float2* __restrict__ out, const float2* __restrict__ ff,
                                                const FFAtom* __restrict__ atoms, const int* __restrict__ off,
                                                int nx, int ny, float itogx, float itogy, float kmax,
                                                int bwl_pot) {
  constexpr int TILE = 16 * P;
  __shared__ float2 s_x[kFFChunk][TILE], s_y[kFFChunk][TILE];
  __shared__ int s_type[kFFChunk];
  const long long n = (long long)nx * ny;
  const int v = blockIdx.z, tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int x0 = blockIdx.x * TILE, y0 = blockIdx.y * TILE;
  float2 pot[P][P], s[P][P];
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int i = 0; i < P; ++i) pot[j][i] = s[j][i] = make_float2(0.f, 0.f);
  int cur = -1;  // type of the running sums s
  auto flush = [&]() {
#pragma unroll
    for (int j = 0; j < P; ++j)
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int x = x0 + tx + 16 * i, y = y0 + ty + 16 * j;
        if (x < nx && y < ny) {
          float ap = 1.f;
          if (bwl_pot)
            ap = 0.5f - 0.5f * tanhf((ff_gmag(ff_freq(x, nx, itogx), ff_freq(y, ny, itogy)) / kmax - 0.9f) * 30.f);
          const float2 f = ff[(long long)cur * n + (long long)y * nx + x], z = s[j][i];
          pot[j][i].x += ap * (f.x * z.x - f.y * z.y);
          pot[j][i].y += ap * (f.x * z.y + f.y * z.x);
        }
        s[j][i] = make_float2(0.f, 0.f);
      }
  };
  const int a1 = off[v + 1];
  for (int c0 = off[v]; c0 < a1; c0 += kFFChunk) {
    const int m = (a1 - c0 < kFFChunk) ? (a1 - c0) : kFFChunk;
    __syncthreads();  // the previous chunk's reads are done
    for (int e = threadIdx.x; e < m * 2 * TILE; e += 256) {
      const int k = e / (2 * TILE), r = e % (2 * TILE), c = r % TILE;
      const FFAtom at = atoms[c0 + k];
      const bool isx = r < TILE;
      const float q = isx ? ff_freq(min(x0 + c, nx - 1), nx, itogx) : ff_freq(min(y0 + c, ny - 1), ny, itogy);
      double ud = (double)(isx ? at.x : at.y) * (double)q;
      ud -= rint(ud);
      double sn, cs;
      sincospi(2.0 * ud, &sn, &cs);
      const double o = isx ? 1.0 : (double)at.occ;
      (isx ? s_x : s_y)[k][c] = make_float2((float)(o * cs), (float)(-o * sn));
    }
    if ((int)threadIdx.x < m) s_type[threadIdx.x] = atoms[c0 + threadIdx.x].type;
    __syncthreads();
    for (int k = 0; k < m; ++k) {
      if (s_type[k] != cur) {
        if (cur >= 0) flush();
        cur = s_type[k];
      }
      float2 ex[P], ey[P];
#pragma unroll
      for (int i = 0; i < P; ++i) {
        ex[i] = s_x[k][tx + 16 * i];
        ey[i] = s_y[k][ty + 16 * i];
      }
#pragma unroll
      for (int j = 0; j < P; ++j)
#pragma unroll
        for (int i = 0; i < P; ++i) {
          s[j][i].x = fmaf(ey[j].x, ex[i].x, fmaf(-ey[j].y, ex[i].y, s[j][i].x));
          s[j][i].y = fmaf(ey[j].x, ex[i].y, fmaf(ey[j].y, ex[i].x, s[j][i].y));
        }
    }
  }
  if (cur >= 0) flush();
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int x = x0 + tx + 16 * i, y = y0 + ty + 16 * j;
      if (x < nx && y < ny) out[(long long)v * n + (long long)y * nx + x] = pot[j][i];
    }
}

// a <- exp(i sg sc a): real-space potential (complex: the imaginary part
// absorbs) to transmission function, exp(-sg Im V) (cos sg Re V, sin sg Re V)
// with V = sc a (JEElaSca.cpp:1129-1141; PotToPgrKernel)
__global__ void k_pot_pgr(float2* __restrict__ a, long long n, float sc, float sg) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float2 p = a[i];
  const float vr = p.x * sc, vi = p.y * sc;
  const float m = expf(-sg * vi);
  float sn, cs;
  sincosf(sg * vr, &sn, &cs);
  a[i] = make_float2(m * cs, m * sn);
}

// a(q) <- a(q) * (|q| > kthr ? 0 : ftrn) on nvar Fourier-space gratings
// (phase-grating band limit, JEElaSca.cpp:597-604 with ftrn = 1/(nx ny))
__global__ void k_pgr_aperture(float2* __restrict__ a, int nx, int ny, long long total, float itogx,
                               float itogy, float kthr, float ftrn) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const long long p = i % ((long long)nx * ny);
  const int ix = (int)(p % nx), iy = (int)(p / nx);
  const float w = (ff_gmag(ff_freq(ix, nx, itogx), ff_freq(iy, ny, itogy)) > kthr) ? 0.f : ftrn;
  float2 z = a[i];
  z.x *= w;
  z.y *= w;
  a[i] = z;
}

// dst += w * src (complex), n items
__global__ void k_axpy_c(float2* __restrict__ dst, const float2* __restrict__ src, long long n, float w) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float2 s = src[i];
  float2 d = dst[i];
  d.x += w * s.x;
  d.y += w * s.y;
  dst[i] = d;
}

// ---------------------------------------------------------------------------
// dispatch over the compiled line lengths
// ---------------------------------------------------------------------------
bool size_supported(int n) {
  switch (n) {
#define JMS_CASE(N) case N: return true;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return false;
  }
}

int row_tiles(int nx, int ny) {
  switch (nx) {
#define JMS_CASE(N) case N: return (ny + Cfg<N>::LPB - 1) / Cfg<N>::LPB;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return 0;
  }
}

template <int N>
static constexpr int tile_width(Tile tile) {
  return tile == Tile::Small ? Lat<N>::CC : tile == Tile::Wide ? Wide<N>::CC : Cfg<N>::CC;
}
int col_tiles(int ny, int nx, Tile tile) {
  switch (ny) {
#define JMS_CASE(N) case N: return (nx + tile_width<N>(tile) - 1) / tile_width<N>(tile);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return 0;
  }
}

template <int NY>
static bool band_loop_col_n(int y0, int y1) {
  using BS = BandSlots<NY, radix_at<typename Cfg<NY>::PC, true>(0)>;
  return BS::G0_MAX >= BS::G1_MIN || (y0 <= BS::G0_MAX && y1 >= BS::G1_MIN);
}
BandHost band_of(int nx, int ny, int gx0, int gx1, int gy0, int gy1, Tile tl) {
  BandHost b;
  int tile = 0;
  switch (ny) {
#define JMS_CASE(N) case N: tile = tile_width<N>(tl); b.rows = band_col_n<N>(gy0, gy1); break;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return b;
  }
  switch (nx) {
#define JMS_CASE(N) case N: band_row_n<N>(gx0, gx1, tile, b); break;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
  }
  return b;
}

bool lat_ok(int nx, int ny, int nwave) {
  // the long-column kernel has one shape; its launches fill the device
  const bool wl = ny != 1024 && ny != 2048;
  // a pair of passes in this shape / in Cfg's, us: 512^2 1 wave 10.8 / 13.2,
  // 4 waves 17.0 / 16.2; 256^2 8 waves 12.4 / 12.7, 16 waves 16.8 / 15.3;
  // 128^2 16 waves 8.8 / 9.3, 32 waves 11.8 / 11.0 (tiles: 32, 16, 8)
  return wl && nwave * col_tiles(ny, nx, Tile::Own) < 128;
}

// The slice loop in one launch takes one block per wave and CU (two at 64^2)
// and is bound by arithmetic; two launches per slice are bound by latency for
// few waves and by memory for many.  The measured lines (jms_loop_impl.hpp): a
// wave of up to 4096 points is always faster in one launch; up to 9216 points
// from about 32 waves on; up to 16384 points from about 112 waves on, as long
// as the last round of 256 blocks is mostly full, and not beyond 1024 waves.
bool loop_ok(int nx, int ny, int nwave) {
  auto edge = [](int n) { return n == 64 || n == 96 || n == 128; };
  if (!edge(nx) || !edge(ny)) return false;
  const int n = nx * ny;
  if (n <= 64 * 64) return true;
  if (n <= 96 * 96) return nwave >= 32;
  constexpr int kCUs = 256;
  const int rounds = (nwave + kCUs - 1) / kCUs;
  return nwave >= 112 && nwave <= 4 * kCUs && (rounds == 1 || nwave * 20 >= rounds * kCUs * 17);
}
BandHost loop_band(int nx, int ny, int gx0, int gx1, int gy0, int gy1) {
  BandHost b;
  switch (nx) {
    case 64: band_row_n<64>(gx0, gx1, 1, b); break;
    case 96: band_row_n<96>(gx0, gx1, 1, b); break;
    case 128: band_row_n<128>(gx0, gx1, 1, b); break;
  }
  // the kernels' band has dead rows too; where the column plan has no slot
  // that is dead, that asks for nothing
  switch (ny) {
    case 64: b.rows = band_loop_col_n<64>(gy0, gy1); break;
    case 96: b.rows = band_loop_col_n<96>(gy0, gy1); break;
    case 128: b.rows = band_loop_col_n<128>(gy0, gy1); break;
  }
  return b;
}
hipError_t launch_loop(int nx, int ny, int nwave, const LoopArgs& a, bool band, hipStream_t st) {
  switch (nx * 1000 + ny) {
#define JMS_LOOP(NX, NY) case NX * 1000 + NY: return launch_loop_n<NX, NY>(nwave, a, band, st);
    JMS_LOOP(64, 64) JMS_LOOP(64, 96) JMS_LOOP(64, 128) JMS_LOOP(96, 64) JMS_LOOP(96, 96) JMS_LOOP(96, 128)
    JMS_LOOP(128, 64) JMS_LOOP(128, 96) JMS_LOOP(128, 128)
#undef JMS_LOOP
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_row_pass(int nx, int ny, int nwave, float2* wave, long long wave_stride,
                           const float2* pgr, long long slc_off, long long npg, const int* var_tab,
                           int var_ld, int jslc, const float2* twx, const RowChanHost& rc, int mode,
                           bool panel, const BandHost& bd, Shape shape, hipStream_t st) {
  switch (nx) {
#define JMS_CASE(N)                                                                         \
  case N:                                                                                   \
    return launch_row_pass_n<N>(ny, nwave, wave, wave_stride, pgr, slc_off, npg, var_tab, \
                                var_ld, jslc, twx, rc, mode, panel, bd, shape, st);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_col_pass(int ny, int nwave, bool init, bool exit_, const ColArgsHost& a,
                           hipStream_t st) {
  switch (ny) {
#define JMS_CASE(N) case N: return launch_col_pass_n<N>(nwave, init, exit_, a, st);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
}

bool panel_ok(int nx, int ny) {
  bool rx = false, cy = false;
  switch (nx) {
#define JMS_CASE(N) case N: rx = Cfg<N>::PANEL; break;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return false;
  }
  switch (ny) {
#define JMS_CASE(N) case N: cy = Cfg<N>::PANEL; break;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return false;
  }
  return rx && cy;
}

bool grp_supported(int nx, int ny) {
  if (!size_supported(nx)) return false;
  switch (ny) {
#define JMS_CASE(N) case N: return Cfg<N>::WL || Cfg<N>::XL;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return false;
  }
}

hipError_t launch_row_pass_grp(int nx, int ny, int nwave, long long wave_stride, long long npg,
                               const float2* twx, const GrpArgs& ga, bool panel, const BandHost& bd,
                               hipStream_t st) {
  switch (nx) {
#define JMS_CASE(N) case N: return launch_row_pass_grp_n<N>(ny, nwave, wave_stride, npg, twx, ga, panel, bd, st);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_col_pass_grp(int nx, int ny, int nwave, bool init, bool exit_, bool detect,
                               long long part_dstride, const float2* twy, const GrpArgs& ga,
                               bool panel, const BandHost& bd, hipStream_t st) {
  switch (ny) {
#define JMS_CASE(N) \
  case N: return launch_col_pass_grp_n<N>(nx, nwave, init, exit_, detect, part_dstride, twy, ga, panel, bd, st);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_col_fft(int nx, int ny, int nbatch, float2* data, int dir, const float2* twy,
                          hipStream_t st) {
  const long long stride = (long long)nx * ny;
  switch (ny) {
#define JMS_CASE(N) case N: return launch_col_fft_n<N>(nx, nbatch, data, stride, dir, twy, st);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_fft2d(int nx, int ny, int nbatch, float2* data, int dir, const float2* twx,
                        const float2* twy, hipStream_t st) {
  const long long stride = (long long)nx * ny;
  hipError_t e = hipErrorInvalidValue;
  switch (nx) {
#define JMS_CASE(N) case N: e = launch_row_fft_n<N>(ny, nbatch, data, stride, dir, twx, st); break;
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
  if (e != hipSuccess) return e;
  switch (ny) {
#define JMS_CASE(N) case N: return launch_col_fft_n<N>(nx, nbatch, data, stride, dir, twy, st);
    JMS_SIZES(JMS_CASE)
#undef JMS_CASE
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_combine(const float* partial, int ntiles, int ndet, int ndetslc, int npos,
                          int npass, const float* weights, float* out, int accumulate, float* mirror,
                          hipStream_t st) {
  const int total = npos * ndetslc * ndet;
  if (total <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_combine, dim3((total + 255) / 256), dim3(256), 0, st, partial, ntiles, ndet,
                     ndetslc, npos, npass, weights, out, accumulate, mirror);
  return hipGetLastError();
}

hipError_t launch_zero_partial(float* partial, long long part_w, long long off, int len, int nwave,
                               hipStream_t st) {
  if (len <= 0 || nwave <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_partial, dim3((len + 255) / 256, nwave), dim3(256), 0, st, partial, part_w, off, len);
  return hipGetLastError();
}

hipError_t launch_offset_wave(float2* out, const float2* in, int nx, int ny, float kscx,
                              float kscy, float dx, float dy, float fz, const float* cppl,
                              int ish0, int ish1, hipStream_t st) {
  const long long n = (long long)nx * ny;
  hipLaunchKernelGGL(k_offset_wave, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, out, in,
                     nx, ny, kscx, kscy, dx, dy, fz, cppl, ish0, ish1);
  return hipGetLastError();
}

hipError_t launch_gauss_gratings(float2* out, int nx, int ny, int nvar, double hx, double hy,
                                 double rc2, double inv2s2, double sig_int, const GaussAtom* atoms,
                                 const int* off, const int* idx, hipStream_t st) {
  dim3 g((nx + 15) / 16, (ny + 15) / 16, nvar), b(16, 16);
  hipLaunchKernelGGL(k_gauss_gratings, g, b, 0, st, out, nx, ny, hx, hy, rc2, inv2s2, sig_int, atoms, off,
                     idx);
  return hipGetLastError();
}

hipError_t launch_ff_gratings(float2* out, int nx, int ny, int nvar, const float2* ff, const FFAtom* atoms,
                              const int* off, float itogx, float itogy, float kmax, int bwl_pot, float sc,
                              float sg, int bwl_pgr, float kthr, float ftrn, const float2* twx,
                              const float2* twy, hipStream_t st) {
  const long long n = (long long)nx * ny, total = n * nvar;
  // tiles of 64 x 64 pixels where they give every CU two blocks, else of 32 x 32
  auto sum = [&](auto kern, int tile) {
    hipLaunchKernelGGL(kern, dim3((nx + tile - 1) / tile, (ny + tile - 1) / tile, nvar), dim3(256), 0, st, out, ff,
                       atoms, off, nx, ny, itogx, itogy, kmax, bwl_pot);
  };
  if ((long long)((nx + 63) / 64) * ((ny + 63) / 64) * nvar >= 512) sum(k_ff_sum<4>, 64);
  else sum(k_ff_sum<2>, 32);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = launch_fft2d(nx, ny, nvar, out, +1, twx, twy, st);
  if (e != hipSuccess) return e;
  const dim3 g((unsigned)((total + 255) / 256)), b(256);
  hipLaunchKernelGGL(k_pot_pgr, g, b, 0, st, out, total, sc, sg);
  e = hipGetLastError();
  if (e != hipSuccess || !bwl_pgr) return e;
  e = launch_fft2d(nx, ny, nvar, out, -1, twx, twy, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_pgr_aperture, g, b, 0, st, out, nx, ny, total, itogx, itogy, kthr, ftrn);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_fft2d(nx, ny, nvar, out, +1, twx, twy, st);
}

hipError_t launch_probe(float2* out, double* partial, const ProbeArgsHost& a, hipStream_t st) {
  const long long n = (long long)a.nx * a.ny;
  const unsigned nblk = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(k_probe, dim3(nblk), dim3(256), 0, st, out, partial, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_probe_scale, dim3(nblk), dim3(256), 0, st, out, (const double*)partial, (int)nblk, n);
  return hipGetLastError();
}

hipError_t launch_axpy_c(float2* dst, const float2* src, long long n, float w, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_axpy_c, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dst, src, n, w);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Scratch of the allocation-free batch entry (jms_hip_run_batch_noalloc):
// the readout partial sums of one batch.  A file-scope device array, so each
// GPU the library runs on holds its own copy until the process ends; host
// code must use the address scratch_address() resolves for the current
// device, never the array's name.
// ---------------------------------------------------------------------------
static __device__ __align__(256) float scratch[kScratchFloats];

hipError_t scratch_address(int device, float** out) {
  static std::mutex mu;
  static std::vector<float*> addr;  // per device, resolved once
  std::lock_guard<std::mutex> lock(mu);
  if (device < 0) return hipErrorInvalidDevice;
  if ((int)addr.size() <= device) addr.resize(device + 1, nullptr);
  if (!addr[device]) {
    int cur = -1;
    hipError_t err = hipGetDevice(&cur);
    if (err == hipSuccess && cur != device) err = hipSetDevice(device);
    float* p = nullptr;
    if (err == hipSuccess) err = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
    if (cur >= 0 && cur != device) (void)hipSetDevice(cur);
    if (err != hipSuccess) return err;
    addr[device] = p;
  }
  *out = addr[device];
  return hipSuccess;
}

}  // namespace jms
