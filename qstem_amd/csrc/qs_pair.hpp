// qs_pair.hpp -- wavefront-resident mixed-radix sweeps with two-pass plans.
//
// A length N = R0 R1 (R0 <= R1 <= 32) is transformed in two register passes with one
// exchange through LDS.  R1 lanes of one wavefront own the transform: pass one is R1
// butterflies of radix R0, pass two R0 butterflies of radix R1, so the lanes need not hold
// equally many values and every length with such a pair of radices has a plan (the plans of
// qs_mix.hpp need one number of values per lane that all radices divide).  Two layouts
// alternate: in L0 lane j < R1 holds elements j + k R1 (k < R0), in L1 lane j < R0 holds
// j + k R0 (k < R1).  A transform whose first radix is R0 takes L0 to L1, one whose first
// radix is R1 takes L1 to L0: the row sweep loads and stores the state in L0 and multiplies
// by the transmission row in L1, the column sweep propagates in L1.  64/R1 transforms share
// a wavefront (rows next to each other); lanes without an element of a pass repeat the last
// lane's (same inputs, same LDS words written, nothing stored).  State layout
// ([probe][x][ny], in-band ky columns only), modes and outputs are those of k_gen_rows and
// k_gen_cols (runMulsSTEM's slice step, stem3/stemlib.cpp:2405-2443).
#pragma once
#include <hip/hip_runtime.h>

#include "qs_dft.hpp"
#include "qs_fft.hpp"
#include "qs_internal.hpp"

namespace qs {

// The pair of N: most transforms per wavefront (the smallest larger radix).
constexpr bool pair_radix(int r) {
  constexpr int set[] = {8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 24, 25, 27, 28, 30, 32};
  for (int s : set)
    if (s == r) return true;
  return false;
}
constexpr int pair_r1(int n) {
  for (int r = 8; r <= 32; r++)
    if (n % r == 0 && pair_radix(r) && pair_radix(n / r) && n / r <= r) return r;
  return 0;
}
// float2 per transform slot: both exchanges (rows of one odd pitch) and the natural order,
// on a bank offset that spreads the slots that the column staging writes together
constexpr int pair_slot(int n, int r0, int r1) {
  int ld = n;
  if (r0 * (r1 | 1) > ld) ld = r0 * (r1 | 1);
  if (r1 * (r0 | 1) > ld) ld = r1 * (r0 | 1);
  const int want = 64 / r1 >= 4 ? 1 : 4;
  while (ld % 32 != want) ld++;
  return ld;
}
template <int N>
struct Pair {
  static constexpr int R1 = pair_r1(N), R0 = N / R1, S = 64 / R1, LD = pair_slot(N, R0, R1);
  static constexpr int WAVES = 4, CPB = WAVES * S;
  // wavefronts per SIMD: the values of the larger radix and its butterfly take the registers
  static constexpr int OCC = R1 <= 21 ? 4 : (R1 <= 25 ? 3 : 2);
  // log-free check that register slot k of L1 (elements j + k R0) lies inside the 2/3 band's
  // gap (N/3, N - N/3) for every lane, and the same for L0
  static constexpr bool gap1(int k) { return R0 * k > N / 3 && R0 * k + R0 - 1 < N - N / 3; }
  static constexpr bool gap0(int k) { return R1 * k > N / 3 && R1 * k + R1 - 1 < N - N / 3; }
};

// Radices of the pairs that qs_dft.hpp does not name.
template <int R, int DIR>
__device__ __forceinline__ void pair_dft(float2* a) {
  if constexpr (R == 27) dft_2stage<3, 9, DIR>(a);
  else if constexpr (R == 32) dft_2stage<2, 16, DIR>(a);
  else dft_any<R, DIR>(a);
}

// Length RA RB transform: v[k] = element t + k RB (lanes t < RB) in, element t + k RA (lanes
// t < RA) out.  tw: W_N^m, m < N.
template <int RA, int RB, int DIR>
__device__ __forceinline__ void pair_fft(float2* v, float2* slot, const float2* __restrict__ tw, int t) {
  constexpr int PB = RB | 1;  // odd: consecutive lanes' rows of the second pass on distinct banks
  pair_dft<RA, DIR>(v);
  const int ta = min(t, RB - 1), tb = min(t, RA - 1);
  wave_lds_sync();  // the slot's earlier reads are done
#pragma unroll
  for (int k = 0; k < RA; k++) slot[k * PB + ta] = v[k];
  wave_lds_sync();
#pragma unroll
  for (int k = 0; k < RB; k++) v[k] = slot[tb * PB + k];
  // opaque per call: the twiddle loads are neither hoisted out of the callers' loops nor
  // shared between transforms (registers held)
  int e = tb;
  asm volatile("" : "+v"(e));
  // w^k loaded for k < 4 and k a multiple of 4, the others as w^(k & ~3) w^(k & 3)
  float2 pw[RB];
#pragma unroll
  for (int k = 1; k < RB; k++)
    if (k < 4 || (k & 3) == 0) pw[k] = tw[k * e];
#pragma unroll
  for (int k = 5; k < RB; k++)
    if (k & 3) pw[k] = cmul(pw[k & ~3], pw[k & 3]);
#pragma unroll
  for (int k = 1; k < RB; k++) v[k] = DIR < 0 ? cmul(v[k], pw[k]) : cmulc(v[k], pw[k]);
  pair_dft<RB, DIR>(v);
}

// Buffer-resource access (MUBUF): a per-lane byte offset; an offset past the resource
// (kPairOut) reads zero and stores nothing.
constexpr unsigned kPairOut = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pair_rsrc(const void* base, long bytes) {
  const int n = bytes < 0x7fffffffL ? (int)bytes : 0x7fffffff;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, n, 0x00020000);
}
__device__ __forceinline__ float2 pair_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ void pair_store(float2 v, __amdgpu_buffer_rsrc_t r, unsigned off) {
  using U2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0u, 0, 0));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, off, 0, 0);
}

// Rows (length ny = N): a wavefront advances S adjacent rows (row = probe * nx + x) in each
// of a.rpb steps.  Modes as k_gen_rows: 0 probe input, 1 state input (y-IFFT first), 2 exit
// (y-IFFT into a.exitw, no transmit).
template <int N>
__global__ __launch_bounds__(64 * Pair<N>::WAVES) __attribute__((amdgpu_waves_per_eu(Pair<N>::OCC))) void k_pair_rows(GenRowArgs a) {
  using P = Pair<N>;
  constexpr int R0 = P::R0, R1 = P::R1, S = P::S;
  __shared__ float2 lds[P::WAVES * S * P::LD];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = min(lane / R1, S - 1), t = lane - sub * R1;
  const bool act = lane < S * R1;
  float2* slot = lds + (wv * S + sub) * P::LD;
  const int nrows = a.nprobe * a.nx;
  const int base = (blockIdx.x * P::WAVES + wv) * (S * a.rpb);
  if (base >= nrows) return;  // whole wavefronts, and no block barriers below
  const int t0 = min(t, R1 - 1), t1 = min(t, R0 - 1);
  unsigned band = 0;  // bit k: element t0 + k R1 is a ky column inside the band
#pragma unroll
  for (int k = 0; k < R0; k++) band |= (!P::gap0(k) && a.ky2[t0 + R1 * k] < a.k2max ? 1u : 0u) << k;
  // the launch's state from this wavefront's first row on; rows past the last are out of range
  const auto rs = pair_rsrc(a.state + ((size_t)a.probe0 * a.nx + base) * N, (long)(nrows - base) * N * 8);
  for (int i = 0; i < a.rpb; i++) {
    const int r0 = base + i * S + sub, r = min(r0, nrows - 1);
    const int p = r / a.nx, x = r - p * a.nx, pg = a.probe0 + p;
    const unsigned off = (unsigned)((i * S + sub) * N + t0) * 8u;
    float2 v[R1];
    if (a.mode == 0) {
#pragma unroll
      for (int k = 0; k < R0; k++) v[k] = a.probe[(size_t)x * N + t0 + R1 * k];
    } else {
#pragma unroll
      for (int k = 0; k < R0; k++)
        v[k] = P::gap0(k) ? make_float2(0.f, 0.f) : pair_load(rs, (band >> k) & 1 ? off + 8u * R1 * k : kPairOut);
    }
    if (a.mode != 0) {
      pair_fft<R0, R1, +1>(v, slot, a.tw, t);
      if (a.mode == 2) {
        if (act && t < R0 && r0 < nrows) {
          float2* dst = a.exitw + ((size_t)pg * a.nx + x) * N + t;
#pragma unroll
          for (int k = 0; k < R1; k++) dst[R0 * k] = v[k];
        }
        continue;
      }
    } else {  // probe rows come in L0: their L1 order through the slot
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < R0; k++) slot[t0 + R1 * k] = v[k];
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < R1; k++) v[k] = slot[t1 + R0 * k];
    }
    // transmit (stemlib.cpp:2880-2887): the window's row, loaded after the IFFT (its
    // registers are not held through the transform)
    const int2 ip = a.ipos[pg];
    const float2* trow = a.trans + (a.cfg ? (long long)a.cfg[pg] * a.cfg_stride : 0LL) +
                         (size_t)(x + ip.x) * a.potNy + ip.y + t1;
#pragma unroll
    for (int k = 0; k < R1; k++) v[k] = cmul(v[k], trow[R0 * k]);
    pair_fft<R1, R0, -1>(v, slot, a.tw, t);
    const unsigned own = act && t < R1 ? off : kPairOut;
#pragma unroll
    for (int k = 0; k < R0; k++)
      if (!P::gap0(k)) pair_store(v[k], rs, (band >> k) & 1 ? own + 8u * R1 * k : kPairOut);
  }
}

// Columns (length nx = N): as k_mix_cols (qs_mix.hpp): block b of probe p has transform slots
// ci = CPB b .. CPB b + CPB - 1 and slot ci takes band column a.tiles[ci] (a.tc of them,
// ascending); the columns are staged through the slots by CPB consecutive lanes per state
// row, and blocks of kPairGroup consecutive b run on one XCD back to back, where they share
// the rows' 128-byte lines that their columns split.  x-FFT, propagator, band limit, detector
// sums into partial[p][b][kMaxDet + 1] and the diffraction pattern, x-IFFT.
constexpr int kPairGroup = 4;
template <int N>
__global__ __launch_bounds__(64 * Pair<N>::WAVES) __attribute__((amdgpu_waves_per_eu(Pair<N>::OCC))) void k_pair_cols(GenColArgs a) {
  using P = Pair<N>;
  constexpr int R0 = P::R0, R1 = P::R1, S = P::S, LD = P::LD, CPB = P::CPB;
  __shared__ float2 lds[P::WAVES * S * LD];
  __shared__ float red[kMaxDet + 1];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int sub = min(lane / R1, S - 1), t = lane - sub * R1;
  const bool act = lane < S * R1;
  float2* slot = lds + (wv * S + sub) * LD;
  // logical block: groups of kPairGroup consecutive ones per XCD (the last partial round of
  // 8 kPairGroup blocks keeps the dispatch order)
  const int nblk = (int)gridDim.x, blk = (int)blockIdx.x;
  int lb = blk;
  if (blk < (nblk / (8 * kPairGroup)) * (8 * kPairGroup)) {
    const int xcd = blk & 7, slot8 = blk >> 3;
    lb = (slot8 / kPairGroup) * (8 * kPairGroup) + xcd * kPairGroup + slot8 % kPairGroup;
  }
  const int nb = (a.tc + CPB - 1) / CPB;  // blocks per probe
  const int p = lb / nb, b = lb - p * nb, ny = a.ny;
  const int ci = (b * P::WAVES + wv) * S + sub;
  const bool ok = act && ci < a.tc;
  const int ky = a.tiles[min(ci, a.tc - 1)];
  // this probe's state; element x of column ky at byte (x ny + ky) 8 (below 2^31: nx, ny <= 2048)
  const auto rs = pair_rsrc(a.state + (size_t)(a.probe0 + p) * N * ny, (long)N * ny * 8);
  // staging: lane (sc, sx) moves block column sc (slot sc) of rows sx + SR i
  constexpr int SR = 64 * P::WAVES / CPB;
  const int sc = threadIdx.x % CPB, sx = threadIdx.x / CPB;
  const int sci = b * CPB + sc;
  const bool sok = sx < SR && sci < a.tc;
  const unsigned soff = sok ? (unsigned)(sx * ny + a.tiles[sci]) * 8u : 0u, sstep = (unsigned)(SR * ny) * 8u;
  float2* const sslot = lds + sc * LD;
  if (threadIdx.x <= kMaxDet) red[threadIdx.x] = 0.f;
  if (sok) {
#pragma unroll 8
    for (int i = 0; i * SR + sx < N; i++) sslot[sx + SR * i] = pair_load(rs, soff + i * sstep);
  }
  __syncthreads();
  const int t0 = min(t, R1 - 1), t1 = min(t, R0 - 1);
  float2 v[R1];
#pragma unroll
  for (int k = 0; k < R0; k++) v[k] = slot[t0 + R1 * k];
  pair_fft<R0, R1, -1>(v, slot, a.tw, t);
  const float2 pyk = a.py[ky];
  const float ky2 = a.ky2[ky];
#pragma unroll
  for (int k = 0; k < R1; k++) {
    if (P::gap1(k)) {
      v[k] = make_float2(0.f, 0.f);
      continue;
    }
    const int kx = t1 + R0 * k;
    const float kx2 = a.kx2[kx];
    const bool in = kx2 < a.k2max && (kx2 + ky2) < a.k2max;
    v[k] = in ? cmul(cmul(v[k], pyk), a.px[kx]) : make_float2(0.f, 0.f);
  }
  const bool own = ok && t < R0;  // lanes that hold elements of their own in L1
  if (a.diff && own) {
#pragma unroll
    for (int k = 0; k < R1; k++) {
      const int hx = t1 + R0 * k + N / 2, hy = ky + ny / 2;
      a.diff[((size_t)(a.probe0 + p) * N + (hx >= N ? hx - N : hx)) * ny + (hy >= ny ? hy - ny : hy)] =
          cnorm(v[k]) * a.diff_scale;
    }
  }
  if (a.rec) {  // sum by sum: one in a register at a time
    auto add = [&](float s, int d) {
      for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (lane == 0) atomicAdd(&red[d], s);
    };
    float total = 0.f;
#pragma unroll
    for (int k = 0; k < R1; k++) total += P::gap1(k) ? 0.f : cnorm(v[k]);
    add(own ? total : 0.f, kMaxDet);
#pragma unroll 1
    for (int d = 0; d < a.ndet; d++) {
      int sy = ky - a.det_sy[d];
      sy += sy < 0 ? ny : 0;
      const float k2y = a.ky2[sy], lo = a.det_k2in[d], hi = a.det_k2out[d];
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < R1; k++) {
        if (P::gap1(k)) continue;
        int sx2 = t1 + R0 * k - a.det_sx[d];
        sx2 += sx2 < 0 ? N : 0;
        const float k2 = a.kx2[sx2] + k2y;
        s += (k2 >= lo && k2 <= hi) ? cnorm(v[k]) : 0.f;
      }
      add(own ? s : 0.f, d);
    }
  }
  pair_fft<R1, R0, +1>(v, slot, a.tw, t);
  wave_lds_sync();  // the transform's last reads of its slot are done
#pragma unroll
  for (int k = 0; k < R0; k++) slot[t0 + R1 * k] = v[k];
  __syncthreads();
  if (a.rec && threadIdx.x <= kMaxDet) a.partial[((size_t)p * nb + b) * (kMaxDet + 1) + threadIdx.x] = red[threadIdx.x];
  if (sok) {
#pragma unroll 8
    for (int i = 0; i * SR + sx < N; i++) pair_store(sslot[sx + SR * i], rs, soff + i * sstep);
  }
}

template <int N>
void launch_pair_rows_t(const GenRowArgs& a, hipStream_t st) {
  using P = Pair<N>;
  const long nrows = (long)a.nprobe * a.nx, per = (long)P::WAVES * P::S * a.rpb;
  hipLaunchKernelGGL(k_pair_rows<N>, dim3((unsigned)((nrows + per - 1) / per)), dim3(64 * P::WAVES), 0, st, a);
}

template <int N>
void launch_pair_cols_t(const GenColArgs& a, int nblocks, hipStream_t st) {
  hipLaunchKernelGGL(k_pair_cols<N>, dim3((unsigned)(nblocks * a.nprobe)), dim3(64 * Pair<N>::WAVES), 0, st, a);
}

}  // namespace qs
