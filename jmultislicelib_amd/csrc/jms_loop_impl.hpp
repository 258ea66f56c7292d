// jms_loop_impl.hpp -- the whole slice loop of a small wave in one launch
// (gfx950): one block per wave, the wave in LDS from the incident wave to the
// exit plane.
//
// A 128^2 wave (128 KiB) fits the 160 KiB of a CU, so the wave does not leave it
// between the passes, and the launches of a pass, their fill and drain, are gone.
// Per slice a block reads its grating and the propagator (from L2).  The work is
// that of the two passes (jms_kernels_impl.hpp): rows inverse, * grating, forward;
// columns forward, * propagator, readout, inverse; the same plans and twiddles.
// Lines are transformed in place, by 4 or 8 threads each, inside a
// wavefront; two barriers per slice.
// What bounds it: the vector instructions and LDS exchanges of one wave per CU,
// and, where the columns have 128 points, spilled registers: a block of 1024
// threads gets 128 VGPRs a thread, too few for 16 values of a column beside their
// propagator or grating and the transform, so 86-107 of them (348-432 bytes a
// lane) go through scratch memory.  128 x 96: 16 (with a band) and 35; the other
// grids: none.
#pragma once
#include "jms_kernels_impl.hpp"

namespace jms {

// threads per line and LDS row pitch: a pitch of 8 mod 32 complex slots puts
// 8 threads x 4 lines (rows or columns) on distinct banks
template <int N>
constexpr int loop_threads() { return N >= 64 ? 8 : 4; }
constexpr int loop_pitch(int nx) { return nx + ((40 - nx % 32) % 32); }
template <int NX, int NY>
constexpr int loop_block() {
  const int r = NY * loop_threads<NX>(), c = NX * loop_threads<NY>();
  return ((r > c ? r : c) + 63) / 64 * 64;
}
template <int PITCH>
struct LoopRow : LdsPos<0, 24> {
  __device__ static __forceinline__ int idx(int line, int e) { return line * PITCH + e; }
};
template <int PITCH>
struct LoopCol {
  static constexpr bool AFFINE = true, FLAT = true;
  static constexpr int PAD = 24;
  __device__ static __forceinline__ int idx(int line, int e) { return e * PITCH + line; }
  static constexpr int step(int d) { return d * PITCH; }
};

// BAND: columns [gx0, gx1) and the dead row slots are zero in every
// propagator and the columns in the source: their LDS columns stay zero and
// are not transformed.  The source may hold anything in the dead rows: the
// incident plane's readout and the first transform take them all.
// The same loop in two launches per slice / here, us per slice on MI355X:
// 64^2 with 1, 64, 256, 1024 waves 6.7 / 4.8, 8.0 / 4.9, 14.8 / 5.2, 25 / 16.8;
// 96^2 with 1, 64, 256, 1024 waves 8.2 / 10.5, 14.8 / 10.8, 26.6 / 11.6,
// 57 / 43.7; 128^2 with 1, 64, 128, 256, 512, 1024, 2048 waves 7.4 / 20.5,
// 16.3 / 21.0, 25.2 / 21.2, 31.6 / 21.8, 48 / 42, 86 / 84, 165 / 167.
// grid: nwave; block: loop_block
template <int NX, int NY, bool BAND>
__global__ __launch_bounds__((loop_block<NX, NY>())) void k_loop(LoopArgs a) {
  using CX = Cfg<NX>;
  using CY = Cfg<NY>;
  using PX = typename CX::P;
  using PY = typename CY::PC;
  constexpr int TX = loop_threads<NX>(), TY = loop_threads<NY>(), BS = loop_block<NX, NY>();
  constexpr int PITCH = loop_pitch(NX);
  using LX = LoopRow<PITCH>;
  using LY = LoopCol<PITCH>;
  constexpr int RX = regs_needed<NX, TX, PX>(), RY = regs_needed<NY, TY, PY>();
  using X0 = IOMap<NX, TX, PX, false>;
  using X1 = IOMap<NX, TX, PX, true>;
  using Y0 = IOMap<NY, TY, PY, false>;
  using Y1 = IOMap<NY, TY, PY, true>;
  using BX = BandSlots<NX, radix_at<PX, false>(0)>;
  using BY = BandSlots<NY, radix_at<PY, true>(0)>;
  constexpr auto dead_x = [](int q) { return BAND && BX::dead(q); };
  constexpr auto dead_y = [](int q) { return BAND && BY::dead(q); };
  __shared__ float2 s_w[NY * PITCH];
  __shared__ float2 s_tx[NX], s_ty[NY];
  __shared__ float s_red[16 * kMaxDet];
  const int tid = threadIdx.x;
  const long long w = blockIdx.x;
  for (int e = tid; e < NX; e += BS) s_tx[e] = a.twx[e];
  for (int e = tid; e < NY; e += BS) s_ty[e] = a.twy[e];
  // rows: thread tx of row; columns: thread ty of the cl-th live column x
  int row = tid / TX, tx = tid % TX, ty = tid % TY;
  const int cl = tid / TY;
  const int gap = BAND ? a.gx1 - a.gx0 : 0;
  int x = BAND && cl >= a.gx0 ? cl + gap : cl;
  const bool row_on = row < NY, col_on = cl < NX - gap;
  if constexpr (BAND) {
    for (int i = tid; i < NY * gap; i += BS) s_w[(i / gap) * PITCH + a.gx0 + i % gap] = make_float2(0.f, 0.f);
  }
  auto each_y1 = [&](auto&& f) {  // slots of the transformed column: f(slot, ky, q)
    static_for<0, Y1::NB>([&](auto I) {
      constexpr int i = decltype(I)::value;
      const int b = ty + i * TY;
      if (Y1::FULL || b < Y1::NBF)
        static_for<0, Y1::R0>([&](auto Q) { f(ic<i * Y1::R0 + decltype(Q)::value>{}, b + decltype(Q)::value * Y1::NBF, Q); });
    });
  };
  float2 v[RX > RY ? RX : RY];
  float2 (&vx)[RX] = reinterpret_cast<float2 (&)[RX]>(v);
  float2 (&vy)[RY] = reinterpret_cast<float2 (&)[RY]>(v);
  // readout of plane p from the columns in registers; INC: the incident wave,
  // which no propagator has made zero in the dead rows
  auto readout = [&](int p, auto INC) {
    const long long off = a.pl[p].part_off;
    if (off < 0) return;  // uniform
    float acc[kMaxDet];
#pragma unroll
    for (int d = 0; d < kMaxDet; ++d) acc[d] = 0.f;
    if (col_on) {
      const int xs = wrap_sub(x, a.dsx, NX);  // de-scan: pixel i is weighted with det(i - d)
      for (int d = 0; d < a.ndet && d < kMaxDet; ++d) {
        const float* dw = a.detw_t + (long long)d * NX * NY + xs * NY;
        float s0 = 0.f, s1 = 0.f;  // two chains: eight terms each, as in a thread of the passes
        each_y1([&](auto K, int ky, auto Q) {
          if constexpr (!decltype(INC)::value && dead_y(decltype(Q)::value)) return;
          const float2 z = vy[decltype(K)::value];
          (decltype(K)::value & 1 ? s1 : s0) += (z.x * z.x + z.y * z.y) * dw[wrap_sub(ky, a.dsy, NY)];
        });
#pragma unroll
        for (int dd = 0; dd < kMaxDet; ++dd)
          if (dd == d) acc[dd] += s0 + s1;
      }
    }
    // one tile holds the whole sum: the wavefronts' parts are added in double, as
    // k_combine adds the tiles of the passes
    block_reduce_det<double>(acc, a.ndet, s_red, a.partial + w * a.part_wstride + off, 1);
  };
  auto down = [&]() {  // inverse column transform, back into LDS
    LineFFT<NY, TY, +1, PY, true, LY, RY, CY::TWR>::run(vy, s_w, x, s_ty, ty, SyncWave{});
    SyncWave{}();
    static_for<0, Y0::NB>([&](auto I) {
      constexpr int i = decltype(I)::value;
      const int b = ty + i * TY;
      if (Y0::FULL || b < Y0::NBF)
        static_for<0, Y0::R0>([&](auto Q) {
          constexpr int q = decltype(Q)::value;
          s_w[LY::idx(x, b + q * Y0::NBF)] = vy[i * Y0::R0 + q];
        });
    });
  };
  // incident wave: source times the phase plate of the position
  if (col_on) {
    float dx = 0.f, dy = 0.f, fz = 0.f;
    const bool pp = a.ppar != nullptr;
    if (pp) {
      const float4 q4 = a.ppar[w];
      dx = q4.x; dy = q4.y; fz = q4.z;
    }
    const float2* src = a.src + w * a.src_stride + x;
    const float kx = (float)fidx(x, NX) * a.kscx;
    each_y1([&](auto K, int ky, auto) {
      float2 z = src[ky * NX];
      if (pp) {
        const float kyf = (float)fidx(ky, NY) * a.kscy;
        const float ksqr = kx * kx + kyf * kyf;
        float chi = -6.28318531f * (dx * kx + dy * kyf + fz * ksqr);
        if (a.cppl_t) chi -= a.cppl_t[x * NY + ky];
        float sn, cs;
        sincosf(chi, &sn, &cs);
        z = cmul(z, make_float2(cs, sn));
      }
      vy[decltype(K)::value] = z;
    });
  }
  __syncthreads();  // tables and zeros in place
  readout(a.islc0, std::true_type{});
  if (col_on) down();
  const int* var = a.var + w * a.var_ld;
#pragma unroll 1
  for (int j = a.islc0; j < a.nslc; ++j) {
    // hidden from the optimiser: the many offsets derived from the thread are
    // formed where they are used instead of being kept over the slices (they
    // would add to the spills)
    __asm__ volatile("" : "+v"(row), "+v"(tx), "+v"(x), "+v"(ty));
    __syncthreads();
    // ---- rows
    if (row_on) {
      float2 tg[RX];
      const float2* g = a.pgr + a.pl[j].slc_off + (long long)var[j] * (NX * NY) + row * NX;
      static_for<0, X1::NB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const int b = tx + i * TX;
        if (X1::FULL || b < X1::NBF)
          static_for<0, X1::R0>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            tg[i * X1::R0 + q] = g[b + q * X1::NBF];
          });
      });
      static_for<0, X0::NB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const int b = tx + i * TX;
        if (X0::FULL || b < X0::NBF)
          static_for<0, X0::R0>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            if constexpr (dead_x(q)) vx[i * X0::R0 + q] = make_float2(0.f, 0.f);
            else vx[i * X0::R0 + q] = s_w[LX::idx(row, b + q * X0::NBF)];
          });
      });
      SyncWave{}();
      LineFFT<NX, TX, +1, PX, false, LX, RX, CX::TWR_ROW>::run(vx, s_w, row, s_tx, tx, SyncWave{});
      static_for<0, X1::NB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const int b = tx + i * TX;
        if (X1::FULL || b < X1::NBF)
          static_for<0, X1::R0>([&](auto Q) {
            constexpr int k = i * X1::R0 + decltype(Q)::value;
            vx[k] = cmul(vx[k], tg[k]);
          });
      });
      SyncWave{}();
      LineFFT<NX, TX, -1, PX, true, LX, RX, CX::TWR_ROW>::run(vx, s_w, row, s_tx, tx, SyncWave{});
      SyncWave{}();
      static_for<0, X0::NB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const int b = tx + i * TX;
        if (X0::FULL || b < X0::NBF)
          static_for<0, X0::R0>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            const int e = b + q * X0::NBF;
            if constexpr (dead_x(q)) return;
            // the exchanges used the whole line: the gap goes back to zero
            // where it is read again
            float2 z = vx[i * X0::R0 + q];
            if constexpr (BAND && BX::part(q)) {
              if (e >= a.gx0 && e < a.gx1) z = make_float2(0.f, 0.f);
            }
            s_w[LX::idx(row, e)] = z;
          });
      });
    }
    __syncthreads();
    // ---- columns
    if (col_on) {
      float2 pv[RY];
      const float2* pro = (const float2*)a.pl[j].pro_t + x * NY;
      each_y1([&](auto K, int ky, auto Q) {
        if constexpr (!dead_y(decltype(Q)::value)) pv[decltype(K)::value] = pro[ky];
      });
      static_for<0, Y0::NB>([&](auto I) {
        constexpr int i = decltype(I)::value;
        const int b = ty + i * TY;
        if (Y0::FULL || b < Y0::NBF)
          static_for<0, Y0::R0>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            vy[i * Y0::R0 + q] = s_w[LY::idx(x, b + q * Y0::NBF)];
          });
      });
      SyncWave{}();
      LineFFT<NY, TY, -1, PY, false, LY, RY, CY::TWR>::run(vy, s_w, x, s_ty, ty, SyncWave{});
      each_y1([&](auto K, int, auto Q) {
        constexpr int k = decltype(K)::value;
        if constexpr (dead_y(decltype(Q)::value)) vy[k] = make_float2(0.f, 0.f);
        else vy[k] = cmul(vy[k], pv[k]);
      });
    }
    readout(j + 1, std::false_type{});
    if (j + 1 < a.nslc && col_on) {
      SyncWave{}();
      down();
    }
  }
  if (a.wave) {  // psi(k) of the exit plane
    float2* o = a.wave + w * a.wave_stride;
    float2 zero = make_float2(0.f, 0.f);  // the dead rows
    if constexpr (BAND) {
      bool some = !col_on;
      each_y1([&](auto K, int, auto Q) {
        if constexpr (!dead_y(decltype(Q)::value)) some |= is_finite(vy[decltype(K)::value]);
      });
      if (!some) zero = not_a_number();
    }
    if (col_on)
      each_y1([&](auto K, int ky, auto Q) {
        if constexpr (dead_y(decltype(Q)::value)) o[ky * NX + x] = zero;
        else o[ky * NX + x] = vy[decltype(K)::value];
      });
    if constexpr (BAND) {
      if (__syncthreads_or(cl == 0 && zero.x != 0.f)) zero = not_a_number();
      else zero = make_float2(0.f, 0.f);
      for (int i = tid; i < NY * gap; i += BS) o[(i / gap) * NX + a.gx0 + i % gap] = zero;
    }
  }
}

template <int NX, int NY>
hipError_t launch_loop_n(int nwave, const LoopArgs& a, bool band, hipStream_t st) {
  const dim3 g(nwave), b(loop_block<NX, NY>());
  if (band) hipLaunchKernelGGL((k_loop<NX, NY, true>), g, b, 0, st, a);
  else hipLaunchKernelGGL((k_loop<NX, NY, false>), g, b, 0, st, a);
  return hipGetLastError();
}

}  // namespace jms
