// qs_slab.hip -- whole multislice runs of small windows in one launch.
//
// A window of 64 or 128 points per side fits one CU: its band-compact state (128 x 85 complex,
// 87 KB) and the exchange slots of the transforms share the 160 KB of LDS.  One block then
// takes one probe through every slice of a run (runMulsSTEM's loop, stem3/stemlib.cpp:
// 2403-2482): row IFFT, transmit and row FFT of all rows, a block barrier, column FFT,
// propagation, detector sums and column IFFT of all band columns, a block barrier.  The wave
// never leaves the CU between slices and no launch separates the sweeps; only the
// transmission rows are read from memory, the next step's while the current one is
// transformed.  The sweeps of qs_sweep.hpp take two dependent launches of 4.5 us (one probe of
// 128^2) to 12 us (128 probes) each per slice; here a slice takes 12 us for up to 256 probes,
// bounded by the CU's vector instructions and LDS accesses (about 9 us and 7 us of them).
// A scan of 256 probes of 128^2 over 20 slices: 630 -> 300 us (the rule of its use, with both
// sides: slab_run in qs_capi.cpp).
#include <hip/hip_runtime.h>

#include "qs_sweep.hpp"

namespace qs {

template <int NX, int NY> struct SlabCfg {
  static constexpr int BLK = NX * NY <= 64 * 64 ? 512 : 1024, WAVES = BLK / 64;
  static constexpr int TX = NX / Plan<NX>::E, WX = 64 / TX, TY = NY / Plan<NY>::E, WY = 64 / TY;
  // float2 of exchange slots per wavefront
  static constexpr int SLOT = WX * lds_slot<NX>() > WY * lds_slot<NY>() ? WX * lds_slot<NX>() : WY * lds_slot<NY>();
  static_assert(NX % (WAVES * WY) == 0, "whole rounds of rows");
  // odd row pitch of the state: a column's rows on distinct banks
  static constexpr int pitch(int kc) { return kc | 1; }
  static size_t lds(int kc) { return sizeof(float2) * ((size_t)NX * pitch(kc) + WAVES * SLOT); }
};

template <int NX, int NY>
__global__ __launch_bounds__((SlabCfg<NX, NY>::BLK)) void k_slab(SlabArgs A) {
  const SweepArgs& a = A.f;
  using C = SlabCfg<NX, NY>;
  constexpr int EX = Plan<NX>::E, TX = C::TX, WX = C::WX, EY = Plan<NY>::E, TY = C::TY, WY = C::WY;
  constexpr int WAVES = C::WAVES, BLK = C::BLK, ROUNDS = NX / (WAVES * WY);
  constexpr int GX = gap_mask<NX>(), GY = gap_mask<NY>();
  extern __shared__ float2 st[];  // [NX][PC] state, then the wavefronts' slots
  __shared__ float red[WAVES][kMaxDet + 1];
  const int PC = C::pitch(a.kc);
  const int lane = threadIdx.x & 63, wv = wave_uniform(threadIdx.x >> 6);
  const int tx = lane % TX, subx = lane / TX, ty = lane % TY, suby = lane / TY;
  float2* const slots = st + NX * PC + wv * C::SLOT;
  float2* const slotx = slots + subx * lds_slot<NX>();
  float2* const sloty = slots + suby * lds_slot<NY>();
  const int p = blockIdx.x;
  Twiddles<NY> twy;
  twy.init(a.twy, ty);
  Twiddles<NX> twx0;  // (one set of registers for both axes of a square window)
  if constexpr (NX != NY) twx0.init(a.twx, tx);
  const Twiddles<NX>& twx = [&]() -> const Twiddles<NX>& {
    if constexpr (NX == NY) return twy;
    else return twx0;
  }();
  // state column of the lane's row elements, -1 outside the band
  const int gap = a.ny - a.band_b - a.band_a - 1;
  int col[EY];
#pragma unroll
  for (int m = 0; m < EY; m++) {
    const int iy = ty + TY * m;
    col[m] = (unsigned)(iy - a.band_a - 1) < (unsigned)gap ? -1 : (iy > a.band_a ? iy - gap : iy);
  }
  float2* const gst = a.state + (size_t)p * NX * a.kcp;
  if (A.start) {
    for (int i = threadIdx.x; i < NX * a.kcp; i += BLK) {
      const int x = i / a.kcp, c = i - x * a.kcp;
      if (c < a.kc) st[x * PC + c] = gst[i];
    }
  }
  const int2 ip = a.ipos[p];
  const float2* tr = a.trans + (a.cfg ? (long long)a.cfg[p] * a.cfg_stride : 0LL) +
                     (size_t)(wv * WY + suby + ip.x) * a.potNy + ip.y + ty;
  float2 nt[EY];  // the next step's transmission row
  auto fetch = [&](int s, int r) {
    const float2* q = tr + (long long)s * A.slice_elems + (size_t)r * (WAVES * WY) * a.potNy;
#pragma unroll
    for (int m = 0; m < EY; m++) nt[m] = q[TY * m];
  };
  fetch(0, 0);
  if (A.start) __syncthreads();
  for (int s = 0; s < A.nslice; s++) {
    const bool last = s == A.nslice - 1;
#pragma unroll 1
    for (int r = 0; r < ROUNDS; r++) {
      const int x = r * (WAVES * WY) + wv * WY + suby;
      float2* const row = st + x * PC;
      float2 v[EY], t[EY];
#pragma unroll
      for (int m = 0; m < EY; m++) t[m] = nt[m];
      if (r + 1 < ROUNDS) fetch(s, r + 1);
      else if (!last) fetch(s + 1, 0);
      if (s == 0 && !A.start) {
#pragma unroll
        for (int m = 0; m < EY; m++) v[m] = a.probe[(size_t)x * NY + ty + TY * m];
      } else {
#pragma unroll
        for (int m = 0; m < EY; m++) {
          v[m] = make_float2(0.f, 0.f);
          if (!((GY >> m) & 1) && col[m] >= 0) v[m] = row[col[m]];
        }
        fft_wave<NY, +1, kSwz<NY>, GY>(v, sloty, twy, ty);
      }
#pragma unroll
      for (int m = 0; m < EY; m++) v[m] = cmul(v[m], t[m]);
      fft_wave<NY, -1, kSwz<NY>, 0, ~GY>(v, sloty, twy, ty);
#pragma unroll
      for (int m = 0; m < EY; m++)
        if (!((GY >> m) & 1) && col[m] >= 0) row[col[m]] = v[m];
    }
    __syncthreads();
    const int bin = A.bin[s];
    const bool rec = bin >= 0 || (last && A.total);
    if (rec && lane <= kMaxDet) red[wv][lane] = 0.f;
    for (int c0 = wv * WX; c0 < a.kc; c0 += WAVES * WX) {
      // surplus transforms of the last wavefront repeat the last column and store nothing
      const int c = min(c0 + subx, a.kc - 1);
      const bool own = c0 + subx < a.kc;
      const int iy = c <= a.band_a ? c : c - (a.band_a + 1) + (a.ny - a.band_b);
      float2 v[EX];
#pragma unroll
      for (int m = 0; m < EX; m++) v[m] = st[(tx + TX * m) * PC + c];
      fft_wave<NX, -1, kSwz<NX>, 0, ~GX>(v, slotx, twx, tx);
      const float ky2 = a.ky2[iy];
      const float2 py = a.py[iy];
#pragma unroll
      for (int m = 0; m < EX; m++) {
        const float kx2 = a.kx2[tx + TX * m];
        const bool in = !((GX >> m) & 1) && kx2 < a.k2max && (kx2 + ky2) < a.k2max;
        v[m] = in ? cmul(cmul(v[m], py), a.px[tx + TX * m]) : make_float2(0.f, 0.f);
      }
      if (rec) {  // this wavefront's sums (collectIntensity, stemlib.cpp:2576-2687)
        auto add = [&](float q, int d) {
          q = wave_sum(own ? q : 0.f);
          if (lane == 0) red[wv][d] += q;
        };
        float n2[EX], total = 0.f;
#pragma unroll
        for (int m = 0; m < EX; m++) {
          n2[m] = cnorm(v[m]);
          total += n2[m];
        }
        add(total, kMaxDet);
#pragma unroll 1
        for (int d = 0; d < (bin >= 0 ? a.ndet : 0); d++) {
          const float k2y = a.ky2[(iy - a.det_sy[d]) & (a.ny - 1)], lo = a.det_k2in[d], hi = a.det_k2out[d];
          float q = 0.f;
#pragma unroll
          for (int m = 0; m < EX; m++) {
            const float k2 = a.kx2[(tx + TX * m - a.det_sx[d]) & (a.nx - 1)] + k2y;
            q += (k2 >= lo && k2 <= hi) ? n2[m] : 0.f;
          }
          add(q, d);
        }
      }
      if (last && a.diff && own) {  // fftshifted |Psi|^2/sqrt(nx*ny) of the unnormalised Psi
        float* dp = a.diff + (size_t)p * NX * NY + (iy + NY / 2) % NY;
#pragma unroll
        for (int m = 0; m < EX; m++) dp[(size_t)((tx + TX * m + NX / 2) % NX) * NY] = cnorm(v[m]) * a.diff_scale;
      }
      fft_wave<NX, +1, kSwz<NX>, GX>(v, slotx, twx, tx);
      if (own) {
#pragma unroll
        for (int m = 0; m < EX; m++) st[(tx + TX * m) * PC + c] = v[m];
      }
    }
    __syncthreads();
    if (rec && threadIdx.x <= a.ndet) {
      const int d = threadIdx.x < a.ndet ? threadIdx.x : kMaxDet;
      double q = 0;
      for (int w = 0; w < WAVES; w++) q += red[w][d];
      if (d < kMaxDet) {
        if (bin >= 0) A.det[((size_t)bin * a.ndet + d) * a.nprobe + p] = (float)(q * A.escale);
      } else if (last && A.total) {
        A.total[p] = (float)q;
      }
    }
  }
  // the state for a continuing call, and the exit waves
  for (int i = threadIdx.x; i < NX * a.kcp; i += BLK) {
    const int x = i / a.kcp, c = i - x * a.kcp;
    gst[i] = c < a.kc ? st[x * PC + c] : make_float2(0.f, 0.f);
  }
  if (a.out_wave) {
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
      const int x = r * (WAVES * WY) + wv * WY + suby;
      float2 v[EY];
#pragma unroll
      for (int m = 0; m < EY; m++) {
        v[m] = make_float2(0.f, 0.f);
        if (!((GY >> m) & 1) && col[m] >= 0) v[m] = st[x * PC + col[m]];
      }
      fft_wave<NY, +1, kSwz<NY>, GY>(v, sloty, twy, ty);
      float2* dst = a.out_wave + ((size_t)p * NX + x) * NY + ty;
#pragma unroll
      for (int m = 0; m < EY; m++) dst[TY * m] = v[m];
    }
  }
}

// LDS of a CU, and what a block holds besides the state and the slots (red).
constexpr size_t kLds = 163840;
template <int NX, int NY>
static constexpr size_t static_lds() { return sizeof(float) * SlabCfg<NX, NY>::WAVES * (kMaxDet + 1); }
template <int NX, int NY>
static bool fits(int kc) { return SlabCfg<NX, NY>::lds(kc) + static_lds<NX, NY>() <= kLds; }
template <int NX, int NY>
static hipError_t allow() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_slab<NX, NY>), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)(kLds - static_lds<NX, NY>()));
}
template <int NX, int NY>
static hipError_t launch(const SlabArgs& a, hipStream_t st) {
  using C = SlabCfg<NX, NY>;
  hipLaunchKernelGGL((k_slab<NX, NY>), dim3((unsigned)a.f.nprobe), dim3(C::BLK), C::lds(a.f.kc), st, a);
  return hipSuccess;
}

#define QS_SLAB(F, ...)                                              \
  if (nx == 64 && ny == 64) return F<64, 64>(__VA_ARGS__);           \
  if (nx == 64 && ny == 128) return F<64, 128>(__VA_ARGS__);         \
  if (nx == 128 && ny == 64) return F<128, 64>(__VA_ARGS__);         \
  if (nx == 128 && ny == 128) return F<128, 128>(__VA_ARGS__);
bool slab_fits(int nx, int ny, int kc) {
  QS_SLAB(fits, kc)
  return false;
}
hipError_t launch_slab(const SlabArgs& a, hipStream_t st) {
  const int nx = a.f.nx, ny = a.f.ny;
  QS_SLAB(launch, a, st)
  return hipErrorInvalidValue;
}
#undef QS_SLAB
hipError_t set_slab_lds() {
  hipError_t e = allow<64, 64>(), r;
  if ((r = allow<64, 128>()) != hipSuccess) e = r;
  if ((r = allow<128, 64>()) != hipSuccess) e = r;
  if ((r = allow<128, 128>()) != hipSuccess) e = r;
  return e;
}

}  // namespace qs
