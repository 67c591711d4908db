// qs_sweep.hpp -- templated multislice sweep kernels and their launchers.
//
// Wave state layout in HBM between slices: state[p][x][c], complex64, where
// p is the probe, x the real-space row (0..nx-1) and c indexes only the ky
// columns that survive the 2/3 band limit of propagate_slow
// (stem3/stemlib.cpp:2831-2849); everything outside that band is zero after
// propagation, so it is neither stored nor transformed.  At nx = 4096 a 128-byte line holds
// four columns of four rows instead of sixteen of one (row_off, col_off).
//
// One slice = two fused sweeps:
//   sweep A (per row x):     row IFFT (finishes slice s-1) -> transmit t_s
//                            (stemlib.cpp:2867-2888) -> row FFT (starts slice s)
//   sweep B (per ky column): column FFT (finishes the forward 2D FFT) ->
//                            propagate + band limit (:2760-2850) -> detector
//                            annuli (:2576-2687) -> column IFFT
// The 1/(nx*ny) of fft_normalize (:2890-2906) is folded into the propagator.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "qs_fft.hpp"
#include "qs_internal.hpp"

namespace qs {

constexpr int kBlock = 256;
// Threads per block of the row-type kernels for transform length N: 256, or
// the transform's own thread count when larger (one transform per block).
template <int N> constexpr int row_block() { return (N / Plan<N>::E) > kBlock ? N / Plan<N>::E : kBlock; }


// ============================================================================
// Buffer-resource (MUBUF) access with hardware range checking: a load at an
// offset at or past the resource's byte size returns zero and a store there is
// dropped.  kOut is past every resource built here (sizes stay below 2^31).
using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr unsigned kOut = 0x80000000u;

__device__ __forceinline__ rsrc_t make_rsrc(const void* base, long bytes) {
  const int n = bytes < 0x7fffffffL ? (int)bytes : 0x7fffffff;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, n, 0x00020000);
}
__device__ __forceinline__ float2 buf_load_c64(rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ void buf_store_c64(float2 v, rsrc_t r, unsigned off) {
  using U2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0u, 0, 0));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, off, 0, 0);
}
// 16-byte store with the whole offset in the VGPR offset and a zero soffset.  A MUBUF
// store of more than 8 bytes reads its data VGPRs after issue, and the compiler puts
// wait states before a later VALU write of those VGPRs only when the soffset is not an
// SGPR; with an SGPR soffset it scheduled such writes directly after the store, and on
// gfx950 the store then sometimes wrote the new values (LDS addresses in place of the
// wave data, a few elements per launch, differing between runs).
__device__ __forceinline__ void buf_store_f4(float4 v, rsrc_t r, unsigned off) {
  using U4 = decltype(__builtin_amdgcn_raw_buffer_load_b128(r, 0u, 0, 0));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, v), r, off, 0, 0);
}

// Byte offsets inside a band-compact state of rows of kcp columns whose 128-byte lines hold
// 1 << lb columns of 16 >> lb rows (col_line): row x at row_off(x), column c of it at
// col_off(c) more.  For x0 and x of which one is a multiple of a power of two above the
// other, row_off(x0 + x) = row_off(x0) + row_off(x).
__device__ __forceinline__ unsigned col_off(int c, int lb) {
  return ((unsigned)(c >> lb) << 7) + ((unsigned)(c & ((1 << lb) - 1)) << 3);
}
__device__ __forceinline__ unsigned row_off(int x, int lb, int kcp) {
  const int rb = 4 - lb;
  return ((unsigned)(x >> rb) * (unsigned)kcp << (rb + 3)) + ((unsigned)(x & ((1 << rb) - 1)) << (lb + 3));
}

// Byte offset of ky column iy inside a band-compact row, or kOut when iy lies in
// the zero gap (band_a, ny-band_b) between the two halves of the band;
// gap = ny - band_b - band_a - 1.
__device__ __forceinline__ unsigned band_off(int iy, int band_a, int gap, int lb) {
  const int c = iy > band_a ? iy - gap : iy;
  return (unsigned)(iy - band_a - 1) < (unsigned)gap ? kOut : col_off(c, lb);
}

__device__ __forceinline__ int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Work item of block `blk` of nblk such that work items gs*j ... gs*j+gs-1 (gs a power of two:
// those that share 128-byte lines of the state) run back to back on the same XCD: blocks are
// dispatched round-robin over the 8 XCDs, each with its own L2, so blocks b, b+8, ...,
// b+8*(gs-1) share an L2.  The last partial group of 8*gs blocks keeps the identity mapping.
__device__ __forceinline__ int xcd_group_block(int blk, int nblk, int gs) {
  if (blk >= (nblk & ~(8 * gs - 1))) return blk;
  const int xcd = blk & 7, slot = blk >> 3;
  return (slot / gs) * (8 * gs) + xcd * gs + (slot % gs);
}

// ============================================================================
// sin and cos of a phase x (|x| well below 2^16 rad): Cody-Waite reduction by
// pi/2 in two FMA steps (pi/2 = H + L, H = float(pi/2); x - kH is exact under the
// fused multiply-add), then the Taylor series of sin and cos on |r| <= pi/4 to
// degrees 9 and 10 (truncation below 2e-9) and the quadrant k mod 4.
__device__ __forceinline__ void sincos_phase(float x, float& s, float& c) {
  const float k = rintf(x * 0.63661977236758134f);  // 2/pi
  float r = fmaf(-k, 1.57079637050628662f, x);       // H
  r = fmaf(-k, -4.37113900018624283e-8f, r);         // L = pi/2 - H
  const float r2 = r * r;
  const float ps = r + r * r2 * fmaf(r2, fmaf(r2, fmaf(r2, 1.0f / 362880.0f, -1.0f / 5040.0f), 1.0f / 120.0f),
                                     -1.0f / 6.0f);
  const float pc = fmaf(r2, fmaf(r2, fmaf(r2, fmaf(r2, fmaf(r2, -1.0f / 3628800.0f, 1.0f / 40320.0f),
                                                   -1.0f / 720.0f), 1.0f / 24.0f), -0.5f), 1.0f);
  const int q = (int)k & 3;
  const float s0 = (q & 1) ? pc : ps, c0 = (q & 1) ? ps : pc;
  s = (q & 2) ? -s0 : s0;
  c = ((q + 1) & 2) ? -c0 : c0;
}

// Columns per tile of the column sweeps at length N, and log2 of the columns that a
// 128-byte line of the state holds (its other rows: 16 >> col_line): at 4096, where a tile
// is two columns, 32 bytes of four rows, so that a column block's access touches a quarter
// of the lines (per slice of one wave: columns 108 -> 78 us, reverse columns 114 -> 85 us; the
// row sweeps, whose wavefronts then touch 32-byte pieces, 59 -> 78 us; a gradient of one
// 4096^2 wave 8.0 -> 7.2 ms for 12 slices, the forward pass alone unchanged).
template <int N> constexpr int col_tc() { return N == 512 ? 16 : (N <= 1024 ? 8 : (N == 2048 ? 4 : 2)); }
template <int N> constexpr int col_line() { return N == 4096 ? 2 : 4; }

// Largest band-compact row pitch (complex values) at length N: the 2/3 band keeps at
// most 2 floor(N/3) + 1 columns, padded to whole column tiles and then to 16.
template <int N>
constexpr int band_pitch_max() {
  constexpr int tc = col_tc<N>();
  constexpr int kc = 2 * (N / 3) + 1;
  return ((kc + tc - 1) / tc * tc + 15) / 16 * 16;
}

// Sweep A: rows.
// mode 0: input is the shared real-space probe (first slice of a fresh run)
// mode 1: input is the band-compact state (a.state_in if set, else a.state); row IFFT first
// mode 2: exit: row IFFT of the state, write the real-space wave, no transmit
// mode 3: input is a full real-space row of each probe (a.probe + probe*nx*NY);
//         row FFT only, no transmit (first sweep of a band limit)
// mode 4: as mode 2, but the row g is not stored: dL/dV = sigma Im(g conj(u)),
//         u = exp(i sigma V), is written to a.gv (last sweep of the band-limited
//         potential gradient)
// A unit (a wavefront, or the block for block-wide transforms) advances TPW rows (TPW = 64/T
// transforms side by side) in each of a.rw steps; the units of a team (the block's
// wavefronts, or as many blocks on one XCD as a 128-byte line of the state has rows) take
// adjacent rows of one probe in the same step, so that a line's rows are read and written
// at about the same time by one L2.  A team's rows divide nx: probe, window offset and row
// bases are wave-uniform scalars.  Twiddles and band offsets are set up once per unit; all
// loads of a step are issued before its first transform.
template <int NY> __device__ __host__ constexpr int row_team(int lb) {
  return NY / Plan<NY>::E <= 64 ? row_block<NY>() / 64 : 16 >> lb;
}
template <int NY, int MODE, bool COPY = MODE == 1 && NY <= 512>
__global__ __launch_bounds__(row_block<NY>(), Plan<NY>::E <= 8 && NY / Plan<NY>::E <= 64 ? 4 : (NY == 4096 && MODE >= 3 ? 3 : 1)) void k_sweep_rows(SweepArgs a) {
  constexpr int E = Plan<NY>::E;
  constexpr int T = NY / E;
  constexpr int BLK = row_block<NY>();
  static_assert(T <= 64 || T == BLK, "a transform is a wavefront part or the whole block");
  constexpr int TPW = T <= 64 ? 64 / T : 1;   // transforms side by side per unit
  constexpr int SPB = BLK / T;       // transform slots per block
  constexpr bool BOFF = E <= 16;     // keep the band offsets in registers
  constexpr int GAP = gap_mask<NY>();  // slots in the band gap: never loaded, stored or computed
  __shared__ float2 lds[SPB * lds_slot<NY>()];
  const int lane = T <= 64 ? (threadIdx.x & 63) : threadIdx.x;
  const int sub = lane / T;
  const int t = lane % T;
  const int lb = COPY ? 4 : a.lb;
  const int tu = row_team<NY>(lb);  // units per team
  const int item = T <= 64 ? blockIdx.x : xcd_group_block(blockIdx.x, gridDim.x, tu);
  const int unit = T <= 64 ? (threadIdx.x >> 6) : item % tu;
  const int team0 = (T <= 64 ? item : item / tu) * (tu * TPW * a.rw);
  const int row0 = wave_uniform(team0 + unit * TPW);
  if (row0 >= a.nprobe * a.nx) return;  // whole teams only (a team's rows divide nx)
  const int p = row0 / a.nx;
  const int x0 = row0 - p * a.nx;    // first row of the unit; step i: x0 + i * rstep + sub
  const int rstep = tu * TPW;
  const int pg = a.probe0 + p;       // global probe index (ipos, state)
  float2* slot = lds + (threadIdx.x / T) * lds_slot<NY>();
  const size_t sprobe = (size_t)pg * a.nx * a.kcp;
  const long sbytes = (long)a.nx * a.kcp * 8;
  const rsrc_t rs = make_rsrc(a.state + sprobe, sbytes);
  // loads from a.state_in when given (the state of slice s-1 kept elsewhere)
  const rsrc_t rsi = a.state_in ? make_rsrc(a.state_in + sprobe, sbytes) : rs;
  const int gap = NY - a.band_b - a.band_a - 1;
  // per-lane byte offset of element m within a step's rows (kOut outside the band);
  // step i adds the wave-uniform offset of its first row as the scalar offset
  const unsigned subo = row_off(sub, lb, a.kcp);
  unsigned boff[BOFF ? E : 1];
  auto bo = [&](int m) -> unsigned {
    const unsigned o = band_off(t + T * m, a.band_a, gap, lb);
    return o == kOut ? kOut : o + subo;
  };
  auto step_off = [&](int i) -> unsigned { return wave_uniform(row_off(x0 + i * rstep, lb, a.kcp)); };
  if constexpr (BOFF) {
#pragma unroll
    for (int m = 0; m < E; m++) boff[m] = bo(m);
  }
  // MODE 1 up to 512: the state rows of the next step are copied straight into this
  // wavefront's LDS staging area (buffer loads with an LDS destination, no registers)
  // while the current step is transformed; only the first step waits for its state.
  // A step's TPW band rows hold at most 384 complex values (three 1 KB copies): the
  // band keeps at most 2 floor(NY/3) + 1 columns, padded to whole tiles and 16.  (COPY
  // needs lines of one row, whose bytes are contiguous; other layouts load into registers.)
  constexpr bool DMA = COPY;
  constexpr int kStg = 384;
  static_assert(!DMA || TPW * band_pitch_max<NY>() <= kStg, "a step's band rows exceed the staging area");
  __shared__ float2 stg[DMA ? (BLK / 64) * kStg : 1];
  float2* const wstg = stg + (DMA ? wave_uniform(threadIdx.x >> 6) * kStg : 0);
  auto prefetch = [&](int i) {
    if constexpr (DMA) {
      // the whole offset in the VGPR offset, so that the resource's range check covers
      // it: the copy's tail past the last row reads zeros, and past the chunk's last
      // step (kOut) nothing is read
      const unsigned vo = (i < a.rw ? step_off(i) : kOut) + 16u * lane;
#pragma unroll
      for (int j = 0; j < 3; j++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsi, (__attribute__((address_space(3))) void*)(wstg + 128 * j), 16,
                                                 vo + 1024u * j, 0, 0, 0);
    }
  };
  int2 ip = make_int2(0, 0);
  const float2* trc = a.trans;  // this probe's configuration, slice s
  if constexpr (MODE <= 1) {
    ip = a.ipos[pg];
    if (a.cfg) trc += (size_t)a.cfg[pg] * (size_t)a.cfg_stride;
  }
  const float2* tr0 = trc + (size_t)(x0 + ip.x) * a.potNy + ip.y;

  auto load = [&](int i, float2* dv, float2* dt) {
    const int xr = i * rstep + sub;  // row relative to x0
    if constexpr (MODE <= 1) {
      const float2* tr = tr0 + (size_t)xr * a.potNy;
#pragma unroll
      for (int m = 0; m < E; m++) dt[m] = tr[t + T * m];
    }
    if constexpr (MODE == 0 || MODE == 3) {
      const float2* src = a.probe + ((MODE == 3 ? (size_t)pg * a.nx : (size_t)0) + x0 + xr) * NY;
#pragma unroll
      for (int m = 0; m < E; m++) dv[m] = src[t + T * m];
    } else if constexpr (DMA) {
#pragma unroll
      for (int m = 0; m < E; m++) {
        if ((GAP >> m) & 1) {
          dv[m] = make_float2(0.f, 0.f);
          continue;
        }
        const unsigned o = BOFF ? boff[m] : bo(m);
        const float2 w = wstg[min(o >> 3, (unsigned)kStg - 1u)];  // index kept inside the area
        dv[m] = o == kOut ? make_float2(0.f, 0.f) : w;
      }
    } else {
      const unsigned so = step_off(i);
#pragma unroll
      for (int m = 0; m < E; m++) {
        if ((GAP >> m) & 1) dv[m] = make_float2(0.f, 0.f);  // inside the band gap for every thread
        else dv[m] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rsi, BOFF ? boff[m] : bo(m), so, 0));
      }
    }
  };
  Twiddles<NY> tw;
  tw.init(a.twy, t);
  // one step: finish row i (v: state or probe row, tv: its transmission row)
  auto step = [&](int i, float2* v, const float2* tv) {
    if constexpr (MODE == 1 || MODE == 2 || MODE == 4) fft_wave<NY, +1, kSwz<NY>, GAP>(v, slot, tw, t);
    const int xr = i * rstep + sub;
    if constexpr (MODE == 2) {
      float2* dst = a.out_wave + ((size_t)pg * a.nx + x0 + xr) * NY;
#pragma unroll
      for (int m = 0; m < E; m++) dst[t + T * m] = v[m];
    } else if constexpr (MODE == 4) {
      const size_t r = ((size_t)pg * a.nx + x0 + xr) * NY;
      const float* vp = a.vpot + r;
      float* gp = a.gv + r;
#pragma unroll
      for (int m = 0; m < E; m++) {
        float sn, cs;
        sincos_phase(vp[t + T * m] * a.gv_sigma, sn, cs);
        gp[t + T * m] = a.gv_sigma * (v[m].y * cs - v[m].x * sn);
      }
    } else {
      if constexpr (MODE <= 1) {
#pragma unroll
        for (int m = 0; m < E; m++) v[m] = cmul(v[m], tv[m]);
      }
      fft_wave<NY, -1, kSwz<NY>, 0, ~GAP>(v, slot, tw, t);
      const unsigned so = step_off(i);
      using U2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(rs, 0u, 0, 0));
#pragma unroll
      for (int m = 0; m < E; m++)
        if (!((GAP >> m) & 1))
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v[m]), rs, BOFF ? boff[m] : bo(m), so, 0);
    }
  };
  // one register set: at 4 wavefronts per SIMD the other wavefronts cover the
  // load latency (measured equal to a two-set software pipeline at 3 per SIMD); at
  // 512 the state rows come through the LDS copies (the transmission rows of the next
  // step in registers as well measured slower: 121 VGPRs)
  float2 va[E], ta[E];
  prefetch(0);
  for (int i = 0; i < a.rw; i++) {
    load(i, va, ta);
    if constexpr (DMA) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wavefront's staging reads are done
      prefetch(i + 1);  // unconditional: one path into the step, so its waits count these copies
    }
    step(i, va, ta);
  }
  // vmcnt(0): the last (empty) copy has landed before the workgroup's LDS can be released
  if constexpr (DMA) __builtin_amdgcn_s_waitcnt(0x0F70);
}

// ============================================================================
// Sum over the 64 lanes of a wavefront (result valid in every lane).
__device__ __forceinline__ float wave_sum(float s) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  return s;
}

// ============================================================================
// Sweep B up to 2048: tiles staged through LDS, a wavefront (2048: the block) or part of one
// per column, no block barriers between a wavefront's passes.  At 512 a tile is 16 columns =
// one whole 128-byte line of every state row, staged by a 512-thread block.  (k_sweep_cols
// below at these lengths: one 256^2 probe 7.0 instead of 5.3 us, 64 of them 11.9 instead of
// 11.2; 64 of 512^2, beside another stream's row sweeps, 81 instead of 68; a 2048^2 scan of 8
// probes 2.7-2.9 instead of 2.6 ms; 1024 equal.)
template <int NX> struct TileCfg {
  using P = Plan<NX>;
  static constexpr int TC = col_tc<NX>();
  static constexpr int BLK = NX == 512 ? 512 : row_block<NX>();
  // tiles grouped on one XCD: those sharing a 128-byte line (16 columns); pairs
  // of whole-line tiles at 512 (measured faster than no grouping)
  static constexpr int GS = TC >= 16 ? 2 : 16 / TC;
  // column slots use the PAD layout (registers are the scarcer resource here);
  // float2 per LDS column, rounded so the tile staging is at most 2-way
  static constexpr int STRIDE = ((lds_slot<NX, false>() + 31) / 32) * 32 + 2;
};
template <int NX> constexpr bool col_staged() { return NX <= 2048; }
// the reverse column sweep has the staged kernel, the direct one (k_adj_cols), or both
template <int NX> constexpr bool adj_col_staged() { return NX <= 2048; }
template <int NX> constexpr bool adj_col_direct() { return NX <= 256 || NX == 4096; }

// Tile staging between the row-major state (TC contiguous complex per row) and
// the column-major LDS tile (PAD layout); 16-byte accesses (two columns per
// thread).  Thread (c, x0) moves columns c, c+1 of rows x0 + XS*i: one buffer
// offset and one LDS base per thread, the row step as the scalar offset and
// as immediate LDS offsets (XS is a multiple of 16 and x0 < XS, so
// lidx(x0 + XS*i) = lidx(x0) + XS*i + XS*i/16).  Global loads are issued in
// batches of up to 8 per thread before their LDS writes.
template <int NX>
struct TileStage {
  using C = TileCfg<NX>;
  static constexpr int TC = C::TC, ST = C::STRIDE, BLK = C::BLK, H = TC / 2;
  static constexpr int IT = H * NX / BLK, IB = IT < 8 ? IT : 8, XS = BLK / H;
  static_assert(H * NX % BLK == 0 && BLK % H == 0 && IT % IB == 0 && XS % 16 == 0,
                "tile staging assumes whole rounds");
  static constexpr int lstep(int i) { return XS * i + XS * i / 16; }
  rsrc_t rs;          // the probe's band-compact state
  unsigned voff;      // byte offset of (row x0, column c) relative to the tile's first column
  int lbase;          // LDS index of (column c, row x0)
  unsigned rstep;     // bytes per XS rows
  __device__ __forceinline__ TileStage(const float2* pstate, int nx, int kcp) {
    const int c = 2 * (threadIdx.x % H), x0 = threadIdx.x / H;
    rs = make_rsrc(pstate, (long)nx * kcp * 8);
    voff = (unsigned)(x0 * kcp + c) * 8u;
    lbase = c * ST + lidx<NX, false>(x0);
    rstep = (unsigned)(XS * kcp) * 8u;
  }
  __device__ __forceinline__ void in(float2* tile, int c0) const {
    const unsigned co = (unsigned)c0 * 8u;
#pragma unroll
    for (int i0 = 0; i0 < IT; i0 += IB) {
      if (i0 > 0) __builtin_amdgcn_sched_barrier(0);  // keep the batches apart (registers)
      float4 q[IB];
#pragma unroll
      for (int i = 0; i < IB; i++)
        q[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff + co, (i0 + i) * rstep, 0));
#pragma unroll
      for (int i = 0; i < IB; i++) {
        tile[lbase + lstep(i0 + i)] = make_float2(q[i].x, q[i].y);
        tile[lbase + ST + lstep(i0 + i)] = make_float2(q[i].z, q[i].w);
      }
    }
  }
  __device__ __forceinline__ void out(const float2* tile, int c0) const {
    const unsigned co = (unsigned)c0 * 8u;
#pragma unroll
    for (int i0 = 0; i0 < IT; i0 += IB) {
      if (i0 > 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = i0; i < i0 + IB; i++) {
        const float2 u = tile[lbase + lstep(i)], w = tile[lbase + ST + lstep(i)];
        buf_store_f4(make_float4(u.x, u.y, w.x, w.y), rs, voff + co + i * rstep);
      }
    }
  }
};

// collectIntensity's sums of one wavefront's pixels (rows t + T m of column iy, value v(m)),
// added to the block's red: detector d sums |Psi|^2 over pixels whose (shift-corrected) k^2
// lies in [k2in, k2out], red[kMaxDet] the total.  Detector by detector: one sum in a
// register at a time (17 of them cost a third of the wavefronts in flight; 137 -> 99 us for 64 probes of 512^2).
template <int NX, class C, class V>
__device__ __forceinline__ void detector_sums(const SweepArgs& a, float* red, int iy, int t, V v) {
  constexpr int E = C::P::E, T = NX / E;
  float n2[E], total = 0.f;
#pragma unroll
  for (int m = 0; m < E; m++) {
    n2[m] = cnorm(v(m));
    total += n2[m];
  }
  total = wave_sum(total);
  if ((threadIdx.x & 63) == 0) atomicAdd(&red[kMaxDet], total);
#pragma unroll 1
  for (int d = 0; d < a.ndet; d++) {
    const int sx = a.det_sx[d];
    const float k2y = a.ky2[(iy - a.det_sy[d]) & (a.ny - 1)];
    const float lo = a.det_k2in[d], hi = a.det_k2out[d];
    float s = 0.f;
#pragma unroll
    for (int m = 0; m < E; m++) {
      const float k2 = a.kx2[(t + T * m - sx) & (a.nx - 1)] + k2y;
      s += (k2 >= lo && k2 <= hi) ? n2[m] : 0.f;
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) atomicAdd(&red[d], s);
  }
}

// Forward column sweep on staged tiles.  A block advances a.tpb consecutive tiles of one probe.
template <int NX, bool REC, bool DIFF>
__global__ __launch_bounds__(TileCfg<NX>::BLK) void k_tile_cols(SweepArgs a) {
  constexpr int E = Plan<NX>::E;
  constexpr int T = NX / E;
  constexpr int TC = TileCfg<NX>::TC;
  constexpr int ST = TileCfg<NX>::STRIDE;
  constexpr int G = TileCfg<NX>::BLK / T;  // transforms in flight per block
  constexpr int ROUNDS = (TC + G - 1) / G;
  constexpr bool PXR = E <= 8;   // per-thread propagator factors and k^2 kept in registers
  constexpr int GAP = gap_mask<NX>();  // kx slots in the band gap: zero after the propagator
  extern __shared__ float2 tile[];  // TC * ST
  __shared__ float red[kMaxDet + 1];

  const int bpp = (a.ntiles + a.tpb - 1) / a.tpb;  // blocks per probe
  const int b = xcd_group_block(blockIdx.x, gridDim.x, TileCfg<NX>::GS);
  const int p = b / bpp;
  const int tile_first = (b % bpp) * a.tpb;
  const int tile_end = min(tile_first + a.tpb, a.ntiles);
  const int pg = a.probe0 + p;
  const TileStage<NX> stage(a.state + (size_t)pg * a.nx * a.kcp, a.nx, a.kcp);

  // one transform per wavefront when T == 64: the column is wave-uniform
  const int slot_id = T == 64 ? wave_uniform(threadIdx.x >> 6) : threadIdx.x / T;
  const int t = threadIdx.x % T;
  Twiddles<NX> tw;
  tw.init(a.twx, t);
  // per-thread propagator factors and k^2 (independent of the column)
  float2 pxr[PXR ? E : 1];
  float kx2r[PXR ? E : 1];
  if constexpr (PXR) {
#pragma unroll
    for (int m = 0; m < E; m++) {
      pxr[m] = a.px[t + T * m];
      kx2r[m] = a.kx2[t + T * m];
    }
  }
  auto kx2_of = [&](int m) -> float { return PXR ? kx2r[m] : a.kx2[t + T * m]; };
  auto px_of = [&](int m) -> float2 { return PXR ? pxr[m] : a.px[t + T * m]; };
  for (int tl = tile_first; tl < tile_end; tl++) {
    if (tl > tile_first) __syncthreads();  // previous tile's LDS reads (stage-out, red) are done
    stage.in(tile, tl * TC);
    if constexpr (REC) {
      if (threadIdx.x <= kMaxDet) red[threadIdx.x] = 0.f;
    }
    __syncthreads();
    const int c0 = tl * TC;
#pragma unroll 1
    for (int r = 0; r < ROUNDS; r++) {
      const int cl = r * G + slot_id;
      if (cl >= TC) break;  // only when G does not divide TC (uniform per transform)
      float2* col = tile + cl * ST;
      const int c = c0 + cl;
      const int iy = c <= a.band_a ? c : (c < a.kc ? c - (a.band_a + 1) + (a.ny - a.band_b) : -1);
      float2 v[E];
#pragma unroll
      for (int m = 0; m < E; m++) v[m] = col[lidx<NX, false>(t + T * m)];
      fft_wave<NX, -1, false, 0, ~GAP>(v, col, tw, t);
      // propagate: P = px[ix]*py[iy] (1/(nx*ny) folded into px), zero outside k2max
      if (iy >= 0) {
        const float ky2 = a.ky2[iy];
        const float2 py = a.py[iy];
#pragma unroll
        for (int m = 0; m < E; m++) {
          if ((GAP >> m) & 1) {  // kx in the band gap for every thread
            v[m] = make_float2(0.f, 0.f);
            continue;
          }
          const float kx2 = kx2_of(m);
          if (kx2 < a.k2max && (kx2 + ky2) < a.k2max) v[m] = cmul(cmul(v[m], py), px_of(m));
          else v[m] = make_float2(0.f, 0.f);
        }
        if constexpr (DIFF) {  // fftshifted |Psi|^2/sqrt(nx*ny) of the unnormalised Psi
          float* dp = a.diff + (size_t)pg * a.nx * a.ny;
          const int sy = (iy + a.ny / 2) % a.ny;
#pragma unroll
          for (int m = 0; m < E; m++) {
            const int ix = t + T * m;
            dp[(size_t)((ix + a.nx / 2) % a.nx) * a.ny + sy] = cnorm(v[m]) * a.diff_scale;
          }
        }
      } else {
#pragma unroll
        for (int m = 0; m < E; m++) v[m] = make_float2(0.f, 0.f);
      }
      // outside the branch: up to 256 a wavefront holds several columns, whose lanes the sums
      // gather (padding columns hold zeros)
      if constexpr (REC) detector_sums<NX, TileCfg<NX>>(a, red, max(iy, 0), t, [&](int m) { return v[m]; });
      fft_wave<NX, +1, false, GAP, -1>(v, col, tw, t);
      xform_sync<NX>();
#pragma unroll
      for (int m = 0; m < E; m++) col[lidx<NX, false>(t + T * m)] = v[m];
    }
    __syncthreads();
    stage.out(tile, c0);
    if constexpr (REC) {
      if (threadIdx.x <= kMaxDet) a.partial[((size_t)p * a.ntiles + tl) * (kMaxDet + 1) + threadIdx.x] = red[threadIdx.x];
    }
  }
}

// ============================================================================
// Sweep B at 4096, and the reverse column sweep there and, of many probes, up to 256 (reverse
// sweeps of 1024 probes of 256^2: 178 us staged, 137 here; with the loss, 432 and 315).
//
// A block transforms TC adjacent columns of one probe, T threads per column with E values
// each: thread (t, c), c fastest, holds rows t + T m of column c.  Its loads and stores are
// then whole TC-column pieces of the state's rows straight to and from the transform's
// registers (128 bytes per row at TC = 16), with no staging pass through LDS; only the
// exchanges between the radix passes go through it, at pos(x) TC + c.  A column's threads
// lie in several wavefronts, so the exchanges use block barriers, which the CU's other
// blocks cover.
template <int N> struct ColPlan : Plan<N> {};
// two passes (one exchange) where E = 16 allows it
template <> struct ColPlan<64>   { static constexpr int E = 8,  NP = 2, R0 = 8,  R1 = 8,  R2 = 1, R3 = 1; };
template <> struct ColPlan<128>  { static constexpr int E = 16, NP = 2, R0 = 16, R1 = 8,  R2 = 1, R3 = 1; };
template <> struct ColPlan<256>  { static constexpr int E = 16, NP = 2, R0 = 16, R1 = 16, R2 = 1, R3 = 1; };

template <int NX> struct ColCfg {
  using P = ColPlan<NX>;
  static constexpr int TC = NX <= 256 ? 16 : col_tc<NX>();  // whole 128-byte lines up to 256
  static constexpr int T = NX / P::E;
  static constexpr int BLK = T * TC;
  // tiles that share the state's 128-byte lines, kept on one XCD
  static constexpr int GS = (1 << col_line<NX>()) / TC > 1 ? (1 << col_line<NX>()) / TC : 1;
  // one row of padding every R0: the first pass writes rows R0 j + k of consecutive j, all
  // later accesses consecutive rows; both then fall on distinct banks
  static __device__ __forceinline__ int pos(int x) { return (x + x / P::R0) * TC; }
  static constexpr int LDS = (NX + NX / P::R0) * TC;  // float2
};

// Column blocks of a probe (its a.ntiles tiles are col_tc columns each).
template <int NX>
__host__ __device__ __forceinline__ int col_blocks(const SweepArgs& a) {
  return (a.ntiles * col_tc<NX>() + ColCfg<NX>::TC - 1) / ColCfg<NX>::TC;
}

// Wavefronts per SIMD of the column sweeps: two 512-thread blocks per CU at 4096; with the loss
// up to 256 one wavefront more for 28 bytes of scratch (320 probes, us without / with the cap:
// 128^2 28 / 23, 256^2 106 / 101).
template <int NX> constexpr int col_waves() { return ColPlan<NX>::E > 8 ? 4 : 1; }

// Slots m of the column plan inside the 2/3 band's gap for every thread (gap_mask).
template <int NX>
constexpr int col_gap() {
  constexpr int E = ColPlan<NX>::E, T = NX / E, A = NX / 3;
  int m = 0;
  for (int j = 0; j < E; j++)
    if (T * j > A && T * j + T - 1 < NX - A) m |= 1 << j;
  return m;
}

// Constants of the twiddled passes.  Two-pass plans hold those of their one twiddled pass in
// registers for every transform of the block (per launch of 320 probes of 256^2 48 us, read
// where they are used 51).  At 4096 they are read from the table where they are used: held
// across both transforms of a column they spill (128 registers), and with the powers of w
// alone held and the others multiplied out a pass takes 40 instructions more (one 4096^2 wave
// 13.5 against 13.3 ms here, its gradient 13.8 against 13.5).
template <int N>
struct ColTwiddles {
  using P = ColPlan<N>;
  static constexpr bool HELD = P::NP == 2;
  static constexpr int T = N / P::E;
  const float2* __restrict__ tab;
  float2 w[HELD ? P::E / 2 : 1];
  template <int R, int NS>
  static __device__ __forceinline__ int index(int t, int b) { return (t + T * b) % NS * (N / (NS * R)); }
  __device__ __forceinline__ void init(const float2* __restrict__ tw, int t) {
    tab = tw;
    if constexpr (HELD) {
#pragma unroll
      for (int b = 0; b < P::E / P::R1; b++) tw_load<N, P::R1>(w + b * (P::R1 / 2), tw, index<P::R1, P::R0>(t, b));
    }
  }
  template <int R, int NS>
  __device__ __forceinline__ void get(float2* c, int t, int b) const {
    if constexpr (HELD) {
#pragma unroll
      for (int i = 0; i < R / 2; i++) c[i] = w[b * (R / 2) + i];
    } else {
      int m = index<R, NS>(t, b);
      asm volatile("" : "+v"(m));  // opaque: loaded here, not hoisted and held across transforms
      tw_load<N, R>(c, tab, m);
    }
  }
};

template <int N, int R, int NS, int DIR, bool FIRST, bool LAST, int ZIN = 0, int NEED = -1>
__device__ __forceinline__ void col_pass(float2* v, float2* tile, const ColTwiddles<N>& tw, int t) {
  using C = ColCfg<N>;
  constexpr int E = C::P::E, T = C::T, NB = E / R;
  float2 a[NB][R];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int k = 0; k < R; k++) {
      if constexpr (FIRST) a[b][k] = v[b + k * NB];
      else a[b][k] = tile[C::pos(t + T * b + k * (N / R))];
    }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    if constexpr (FIRST) {
      if constexpr (NB == 1) dft<R, DIR, ZIN>(a[b]);
      else dft<R, DIR>(a[b]);
    } else {
      float2 c[R / 2];
      tw.template get<R, NS>(c, t, b);
      dft_tw<R, DIR, LAST && NB == 1 ? NEED : -1>(a[b], c);
    }
  }
  if constexpr (LAST) {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int k = 0; k < R; k++) v[b + k * NB] = a[b][k];
  } else {
    __syncthreads();  // all earlier reads of the tile precede these writes
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int j = t + T * b;
      const int base = (j / NS) * NS * R + (j % NS);
#pragma unroll
      for (int k = 0; k < R; k++) tile[C::pos(base + k * NS)] = a[b][k];
    }
    __syncthreads();
  }
}

// Length-N transform of the block's columns; tile: the block's LDS at this thread's column.
template <int N, int DIR, int ZIN = 0, int NEED = -1>
__device__ __forceinline__ void col_fft(float2* v, float2* tile, const ColTwiddles<N>& tw, int t) {
  using P = ColPlan<N>;
  constexpr int S1 = P::R0, S2 = P::R0 * P::R1;
  col_pass<N, P::R0, 1, DIR, true, false, ZIN>(v, tile, tw, t);
  if constexpr (P::NP == 2) {
    col_pass<N, P::R1, S1, DIR, false, true, 0, NEED>(v, tile, tw, t);
  } else {
    static_assert(P::NP == 3, "two or three passes");
    col_pass<N, P::R1, S1, DIR, false, false>(v, tile, tw, t);
    col_pass<N, P::R2, S2, DIR, false, true, 0, NEED>(v, tile, tw, t);
  }
}

// One thread's part of a column block: its column and row, transform constants and the
// state's addressing, and the propagator P = px py (1/(nx ny) folded into px) of its rows,
// zero outside k2max.  With E = 8, P is kept in registers for every probe of the block;
// with E = 16 those would cost half the wavefronts, and a bit per row and py are kept.
template <int NX>
struct ColThread {
  using C = ColCfg<NX>;
  static constexpr int E = C::P::E, T = C::T, GAP = col_gap<NX>();
  static constexpr bool PREG = E <= 8;
  int c, t, iy;  // tile column, transform thread, ky index (-1: padding column)
  unsigned voff, rstep;
  float2 P[PREG ? E : 1];
  unsigned inside = 0;  // bit m: row t + T m lies inside the band
  float2 py;
  const float2* px;
  ColTwiddles<NX> tw;
  __device__ __forceinline__ ColThread(const SweepArgs& a, int c0) {
    c = threadIdx.x % C::TC;
    t = threadIdx.x / C::TC;
    const int col = c0 + c;
    iy = col <= a.band_a ? col : (col < a.kc ? col - (a.band_a + 1) + (a.ny - a.band_b) : -1);
    constexpr int LB = col_line<NX>();
    static_assert(T % (16 >> LB) == 0, "rows t + T m lie in the same row of their lines");
    voff = row_off(t, LB, a.kcp) + col_off(col, LB);
    rstep = (unsigned)(T * a.kcp) * 8u;
    tw.init(a.twx, t);
    const float ky2 = a.ky2[max(iy, 0)];
    py = a.py[max(iy, 0)];
    px = a.px + t;
#pragma unroll
    for (int m = 0; m < E; m++) {
      if ((GAP >> m) & 1) continue;
      const float kx2 = a.kx2[t + T * m];
      const bool in = iy >= 0 && kx2 < a.k2max && (kx2 + ky2) < a.k2max;
      inside |= in ? 1u << m : 0u;
      if constexpr (PREG) {
        const float2 p = cmul(px[T * m], py);
        P[m] = in ? p : make_float2(0.f, 0.f);
      }
    }
  }
  // v P (CONJ: v conj(P)) at row m
  template <bool CONJ>
  __device__ __forceinline__ float2 prop(float2 v, int m) const {
    if ((GAP >> m) & 1) return make_float2(0.f, 0.f);
    if constexpr (PREG) return CONJ ? cmulc(v, P[m]) : cmul(v, P[m]);
    const float2 p = cmul(px[T * m], py);
    const float2 r = CONJ ? cmulc(v, p) : cmul(v, p);
    return (inside >> m) & 1 ? r : make_float2(0.f, 0.f);
  }
  __device__ __forceinline__ void load(float2* v, rsrc_t rs) const {
#pragma unroll
    for (int m = 0; m < E; m++) v[m] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, m * rstep, 0));
  }
  __device__ __forceinline__ void store(const float2* v, rsrc_t rs) const {
    using U2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(rs, 0u, 0, 0));
#pragma unroll
    for (int m = 0; m < E; m++) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v[m]), rs, voff, m * rstep, 0);
  }
};

// Forward column sweep: column FFT, propagate, detector sums (REC) and diffraction pattern
// (DIFF), column IFFT.  A block advances one tile of a.tpb consecutive probes; tiles that
// share 128-byte state lines run on one XCD at about the same time, so the line is fetched
// from HBM once and the others hit L2.
template <int NX, bool REC, bool DIFF>
__global__ __launch_bounds__(ColCfg<NX>::BLK, col_waves<NX>()) void k_sweep_cols(SweepArgs a) {
  using C = ColCfg<NX>;
  using W = ColThread<NX>;
  constexpr int E = W::E, T = W::T, GAP = W::GAP;
  extern __shared__ float2 tile[];  // C::LDS
  __shared__ float red[kMaxDet + 1];
  const int item = xcd_group_block(blockIdx.x, gridDim.x, C::GS);
  const int tl = item % a.ntiles;
  const int p0 = item / a.ntiles * a.tpb, p1 = min(p0 + a.tpb, a.nprobe);
  const W w(a, tl * C::TC);
  float2* const col = tile + w.c;
  for (int p = p0; p < p1; p++) {
    const int pg = a.probe0 + p;
    const rsrc_t rs = make_rsrc(a.state + (size_t)pg * a.nx * a.kcp, (long)a.nx * a.kcp * 8);
    float2 v[E];
    w.load(v, rs);
    if constexpr (REC) {
      if (threadIdx.x <= kMaxDet) red[threadIdx.x] = 0.f;
    }
    col_fft<NX, -1, 0, ~GAP>(v, col, w.tw, w.t);
#pragma unroll
    for (int m = 0; m < E; m++) v[m] = w.template prop<false>(v[m], m);
    // (the exchanges' barriers lie between the clearing of red, the additions and its reading;
    // padding columns hold zeros)
    if constexpr (REC) detector_sums<NX, C>(a, red, max(w.iy, 0), w.t, [&](int m) { return v[m]; });
    if constexpr (DIFF) {  // fftshifted |Psi|^2/sqrt(nx*ny) of the unnormalised Psi
      if (w.iy >= 0) {
        float* dp = a.diff + (size_t)pg * a.nx * a.ny + (w.iy + a.ny / 2) % a.ny;
#pragma unroll
        for (int m = 0; m < E; m++) dp[(size_t)((w.t + T * m + a.nx / 2) % a.nx) * a.ny] = cnorm(v[m]) * a.diff_scale;
      }
    }
    col_fft<NX, +1, GAP, -1>(v, col, w.tw, w.t);
    w.store(v, rs);
    if constexpr (REC) {
      if (threadIdx.x <= kMaxDet) a.partial[((size_t)p * a.ntiles + tl) * (kMaxDet + 1) + threadIdx.x] = red[threadIdx.x];
      __syncthreads();  // red is read before the next probe clears it
    }
  }
}

// ============================================================================
// Generic batched row transforms of length L (power of two), full rows.
template <int L, int DIR>
__global__ __launch_bounds__(row_block<L>()) void k_rows_fft(float2* __restrict__ data, long nrows,
                                                             const float2* __restrict__ tw, float scale) {
  constexpr int E = Plan<L>::E;
  constexpr int T = L / E;
  constexpr int RPB = row_block<L>() / T;
  __shared__ float2 lds[RPB * lds_slot<L>()];
  const int slot_id = threadIdx.x / T, t = threadIdx.x % T;
  const long row = (long)blockIdx.x * RPB + slot_id;
  if (row >= nrows) return;
  float2* r = data + row * L;
  float2 v[E];
#pragma unroll
  for (int m = 0; m < E; m++) v[m] = r[t + T * m];
  Twiddles<L> twc;
  twc.init(tw, t);
  fft_wave<L, DIR>(v, lds + slot_id * lds_slot<L>(), twc, t);
#pragma unroll
  for (int m = 0; m < E; m++) r[t + T * m] = cscale(v[m], scale);
}

// Bluestein transform of rows of length n through a length-M power-of-two FFT.
// chirp[k] = exp(DIR*i*pi*k^2/n); vhat = FFT_M of the wrapped conj(chirp).
template <int M>
__global__ __launch_bounds__(row_block<M>()) void k_rows_bluestein(float2* __restrict__ data, long nrows, int n,
                                                           const float2* __restrict__ chirp,
                                                           const float2* __restrict__ vhat,
                                                           const float2* __restrict__ tw, float scale) {
  constexpr int E = Plan<M>::E;
  constexpr int T = M / E;
  constexpr int RPB = row_block<M>() / T;
  __shared__ float2 lds[RPB * lds_slot<M>()];
  const int slot_id = threadIdx.x / T, t = threadIdx.x % T;
  const long row = (long)blockIdx.x * RPB + slot_id;
  if (row >= nrows) return;
  float2* r = data + row * n;
  float2* slot = lds + slot_id * lds_slot<M>();
  float2 v[E];
#pragma unroll
  for (int m = 0; m < E; m++) {
    const int k = t + T * m;
    v[m] = k < n ? cmul(r[k], chirp[k]) : make_float2(0.f, 0.f);
  }
  Twiddles<M> twc;
  twc.init(tw, t);
  fft_wave<M, -1>(v, slot, twc, t);
#pragma unroll
  for (int m = 0; m < E; m++) v[m] = cmul(v[m], vhat[t + T * m]);
  fft_wave<M, +1>(v, slot, twc, t);
  const float s = scale / (float)M;
#pragma unroll
  for (int m = 0; m < E; m++) {
    const int k = t + T * m;
    if (k < n) r[k] = cscale(cmul(v[m], chirp[k]), s);
  }
}


// ============================================================================
// Launch templates, instantiated per size in qs_sizes.hip.
// Steps per unit (a wavefront, or the block for block-wide transforms): enough
// units to fill every CU several times over, each looping over up to a.rw
// steps (a power of two such that a team's rows divide nx).
template <int N>
void launch_rows_mode(const SweepArgs& a0, int mode, hipStream_t st) {
  constexpr int T = N / Plan<N>::E;
  constexpr int TPW = T <= 64 ? 64 / T : 1;
  constexpr int UPB = T <= 64 ? row_block<N>() / 64 : 1;
  SweepArgs a = a0;
  const int tu = row_team<N>(a.lb);
  const long rows = (long)a.nprobe * a.nx;
  const int max_rw = a.rw > 0 ? a.rw : 4;  // caller's cap (0: default, measured best at 512^2)
  const long target_units = 256L * 8 * UPB;
  int rw = 1;
  while (rw < max_rw && rows / ((long)TPW * rw * 2) >= target_units && a.nx % (TPW * tu * rw * 2) == 0) rw *= 2;
  a.rw = rw;
  const dim3 grid((unsigned)(rows / ((long)TPW * rw) / UPB));  // nx >= 64 is a multiple of every team's rows
  if (mode == 0) hipLaunchKernelGGL((k_sweep_rows<N, 0>), grid, dim3(row_block<N>()), 0, st, a);
  else if (mode == 1) {
    if (a.lb == 4) hipLaunchKernelGGL((k_sweep_rows<N, 1>), grid, dim3(row_block<N>()), 0, st, a);
    else hipLaunchKernelGGL((k_sweep_rows<N, 1, false>), grid, dim3(row_block<N>()), 0, st, a);
  }
  else if (mode == 2) hipLaunchKernelGGL((k_sweep_rows<N, 2>), grid, dim3(row_block<N>()), 0, st, a);
  else if (mode == 3) hipLaunchKernelGGL((k_sweep_rows<N, 3>), grid, dim3(row_block<N>()), 0, st, a);
  else hipLaunchKernelGGL((k_sweep_rows<N, 4>), grid, dim3(row_block<N>()), 0, st, a);
}

template <int N, bool STAGED>
constexpr int col_lds_bytes_t() {
  if constexpr (STAGED) return (int)sizeof(float2) * TileCfg<N>::TC * TileCfg<N>::STRIDE;
  else return (int)sizeof(float2) * ColCfg<N>::LDS;
}

// Probes per block of the direct column kernels: as many as leave two blocks for every place
// on the chip, at most 4 (the block's propagator and constants are set up once for all of them).
template <int N>
int col_probes(const SweepArgs& a) {
  constexpr long by_lds = 163840 / col_lds_bytes_t<N, false>(), by_threads = 2048 / ColCfg<N>::BLK;
  constexpr long places = 256 * (by_lds < by_threads ? by_lds : by_threads);
  return (int)std::max<long>(1, std::min<long>(4, (long)a.nprobe * col_blocks<N>(a) / (2 * places)));
}

// Column kernel of length N: staged tiles or k_sweep_cols.
template <int N, bool REC, bool DIFF>
constexpr auto col_kernel() {
  if constexpr (col_staged<N>()) return &k_tile_cols<N, REC, DIFF>;
  else return &k_sweep_cols<N, REC, DIFF>;
}

template <int N>
void launch_cols_t(const SweepArgs& a0, bool rec, bool diff, hipStream_t st) {
  SweepArgs a = a0;
  dim3 grid, block;
  if constexpr (col_staged<N>()) {  // tiles per block: 1 unless set (more only lengthen its serial phases)
    a.tpb = std::max(1, a0.tpb);
    grid = dim3((unsigned)(a.nprobe * ((a.ntiles + a.tpb - 1) / a.tpb)));
    block = dim3(TileCfg<N>::BLK);
  } else {
    a.tpb = a0.tpb > 0 ? a0.tpb : col_probes<N>(a0);
    grid = dim3((unsigned)((a.nprobe + a.tpb - 1) / a.tpb * col_blocks<N>(a)));
    block = dim3(ColCfg<N>::BLK);
  }
  constexpr int lds = col_lds_bytes_t<N, col_staged<N>()>();
  if (rec && diff) hipLaunchKernelGGL((col_kernel<N, true, true>()), grid, block, lds, st, a);
  else if (rec) hipLaunchKernelGGL((col_kernel<N, true, false>()), grid, block, lds, st, a);
  else if (diff) hipLaunchKernelGGL((col_kernel<N, false, true>()), grid, block, lds, st, a);
  else hipLaunchKernelGGL((col_kernel<N, false, false>()), grid, block, lds, st, a);
}

template <int N>
hipError_t set_col_lds_t() {
  const void* kernels[] = {reinterpret_cast<const void*>(col_kernel<N, false, false>()),
                           reinterpret_cast<const void*>(col_kernel<N, false, true>()),
                           reinterpret_cast<const void*>(col_kernel<N, true, false>()),
                           reinterpret_cast<const void*>(col_kernel<N, true, true>())};
  for (const void* k : kernels) {
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             col_lds_bytes_t<N, col_staged<N>()>());
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int L, int DIR>
void rows_fft_t(float2* d, long nrows, const float2* tw, float scale, hipStream_t st) {
  constexpr int RPB = row_block<L>() / (L / Plan<L>::E);
  hipLaunchKernelGGL((k_rows_fft<L, DIR>), dim3((unsigned)((nrows + RPB - 1) / RPB)), dim3(row_block<L>()), 0, st, d, nrows, tw,
                     scale);
}

template <int M>
void blue_t(float2* d, long nrows, int n, const float2* chirp, const float2* vhat, const float2* tw, float scale,
            hipStream_t st) {
  constexpr int RPB = row_block<M>() / (M / Plan<M>::E);
  hipLaunchKernelGGL((k_rows_bluestein<M>), dim3((unsigned)((nrows + RPB - 1) / RPB)), dim3(row_block<M>()), 0, st, d, nrows, n,
                     chirp, vhat, tw, scale);
}


// ============================================================================
// Adjoint sweeps (reverse mode of the two forward sweeps).
//
// Column sweep (slice s, reverse):  g_Phi = colFFT(g_X)  [last slice: 4 (I - T) Phi,
// Phi = colFFT(X_{S-1})/nx, I = |Phi|^2]  ->  g_Psi = conj(P) g_Phi  ->  g_R = colIFFT(g_Psi).
template <int NX, bool LAST>
__global__ __launch_bounds__(ColCfg<NX>::BLK, col_waves<NX>()) void k_adj_cols(AdjArgs A) {
  const SweepArgs& a = A.f;
  using C = ColCfg<NX>;
  using W = ColThread<NX>;
  constexpr int E = W::E, T = W::T, GAP = W::GAP;
  extern __shared__ float2 tile[];  // C::LDS
  __shared__ float red;
  const int item = xcd_group_block(blockIdx.x, gridDim.x, C::GS);
  const int nt = col_blocks<NX>(a), tl = item % nt;
  const int p0 = item / nt * a.tpb, p1 = min(p0 + a.tpb, a.nprobe);
  const W w(a, tl * C::TC);
  float2* const col = tile + w.c;
  for (int p = p0; p < p1; p++) {
    const int pg = a.probe0 + p;
    const size_t off = (size_t)pg * a.nx * a.kcp;
    const long bytes = (long)a.nx * a.kcp * 8;
    float2 v[E];
    w.load(v, make_rsrc((LAST ? A.xprev : A.gx) + off, bytes));
    if constexpr (LAST) {
      if (threadIdx.x == 0) red = 0.f;
    }
    col_fft<NX, -1, 0, ~GAP>(v, col, w.tw, w.t);
    float lsum = 0.f;
    const float inx = 1.0f / (float)a.nx;
#pragma unroll
    for (int m = 0; m < E; m++) {
      if ((GAP >> m) & 1) {
        v[m] = make_float2(0.f, 0.f);
        if (!LAST) continue;
      }
      float2 g = v[m];
      if constexpr (LAST) {
        if (w.iy >= 0) {
          const float2 phi = (w.inside >> m) & 1 ? cscale(g, inx) : make_float2(0.f, 0.f);
          const float d = cnorm(phi) - A.target[((size_t)pg * a.nx + w.t + T * m) * a.ny + w.iy];
          lsum += d * d;
          g = cscale(phi, 4.0f * d);
        }
      }
      v[m] = w.template prop<true>(g, m);
    }
    if constexpr (LAST) {  // one LDS addition per wavefront; red is cleared and read across the exchanges' barriers
      lsum = wave_sum(lsum);
      if ((threadIdx.x & 63) == 0) atomicAdd(&red, lsum);
    }
    col_fft<NX, +1, GAP, -1>(v, col, w.tw, w.t);
    w.store(v, make_rsrc(A.gx + off, bytes));
    if constexpr (LAST) {
      constexpr int R = C::TC / col_tc<NX>();  // tiles of the partial sums' layout per block
      const int i = tl * R + threadIdx.x;
      if (threadIdx.x < R && i < a.ntiles) A.loss_partial[(size_t)p * a.ntiles + i] = threadIdx.x == 0 ? red : 0.f;
      __syncthreads();
    }
  }
}

// k_adj_cols on staged tiles.
template <int NX, bool LAST>
__global__ __launch_bounds__(TileCfg<NX>::BLK) void k_tile_adj_cols(AdjArgs A) {
  const SweepArgs& a = A.f;
  constexpr int E = Plan<NX>::E;
  constexpr int T = NX / E;
  constexpr int TC = TileCfg<NX>::TC;
  constexpr int ST = TileCfg<NX>::STRIDE;
  constexpr int G = TileCfg<NX>::BLK / T;
  constexpr int ROUNDS = (TC + G - 1) / G;
  extern __shared__ float2 tile[];
  __shared__ float red;
  const int b = xcd_group_block(blockIdx.x, gridDim.x, TileCfg<NX>::GS);
  const int p = b / a.ntiles;
  const int tile_id = b % a.ntiles;
  const int pg = a.probe0 + p;
  const int c0 = tile_id * TC;
  const size_t off = (size_t)pg * a.nx * a.kcp;
  if (threadIdx.x == 0) red = 0.f;
  TileStage<NX>((LAST ? A.xprev : A.gx) + off, a.nx, a.kcp).in(tile, c0);
  __syncthreads();
  const int slot_id = threadIdx.x / T;
  const int t = threadIdx.x % T;
  Twiddles<NX> tw;
  tw.init(a.twx, t);
  float lsum = 0.f;
#pragma unroll 1
  for (int r = 0; r < ROUNDS; r++) {
    const int cl = r * G + slot_id;
    if (cl >= TC) break;
    float2* col = tile + cl * ST;
    const int c = c0 + cl;
    const int iy = c <= a.band_a ? c : (c < a.kc ? c - (a.band_a + 1) + (a.ny - a.band_b) : -1);
    float2 v[E];
#pragma unroll
    for (int m = 0; m < E; m++) v[m] = col[lidx<NX, false>(t + T * m)];
    fft_wave<NX, -1, false, 0, -1>(v, col, tw, t);
    if (iy >= 0) {
      const float ky2 = a.ky2[iy];
      const float2 py = a.py[iy];
      const float inx = 1.0f / (float)a.nx;
#pragma unroll
      for (int m = 0; m < E; m++) {
        const int ix = t + T * m;
        const float kx2 = a.kx2[ix];
        const bool in = kx2 < a.k2max && (kx2 + ky2) < a.k2max;
        float2 g;
        if constexpr (LAST) {
          const float2 phi = in ? cscale(v[m], inx) : make_float2(0.f, 0.f);
          const float d = cnorm(phi) - A.target[((size_t)pg * a.nx + ix) * a.ny + iy];
          lsum += d * d;
          g = cscale(phi, 4.0f * d);
        } else {
          g = v[m];
        }
        v[m] = in ? cmulc(cmulc(g, py), a.px[ix]) : make_float2(0.f, 0.f);
      }
    } else {
#pragma unroll
      for (int m = 0; m < E; m++) v[m] = make_float2(0.f, 0.f);
    }
    fft_wave<NX, +1, false, 0, -1>(v, col, tw, t);
    xform_sync<NX>();
#pragma unroll
    for (int m = 0; m < E; m++) col[lidx<NX, false>(t + T * m)] = v[m];
  }
  if constexpr (LAST) atomicAdd(&red, lsum);
  __syncthreads();
  TileStage<NX>(A.gx + off, a.nx, a.kcp).out(tile, c0);
  if constexpr (LAST) {
    if (threadIdx.x == 0) A.loss_partial[(size_t)p * a.ntiles + tile_id] = red;
  }
}

// Row sweep (slice s, reverse) of a single probe:  g_a = rowIFFT(g_R);  psi_s =
// rowIFFT(X_{s-1}) (or the probe);  g_t += conj(psi_s) g_a;  g_psi = conj(t_s) g_a;
// g_X_{s-1} = rowFFT(g_psi) (s > 0) or g_psi -> gprobe (s = 0).  BLF (the window is the
// whole slice): the row of g_t is complete here, so its row FFT, band-compact in the
// potential grid's band, goes to A.blstate (the band limit's first pass) instead of the
// row to A.gT.
template <int NY, bool FIRST, bool BLF>
__global__ __launch_bounds__(row_block<NY>()) void k_adj_rows(AdjArgs A) {
  const SweepArgs& a = A.f;
  constexpr int E = Plan<NY>::E;
  constexpr int T = NY / E;
  constexpr int RPB = row_block<NY>() / T;
  __shared__ float2 lds[RPB * lds_slot<NY>()];
  const int slot_id = threadIdx.x / T;
  const int t = threadIdx.x % T;
  // one probe; block-wide transforms: a line's rows on one XCD at the same time
  const int blk = RPB > 1 ? blockIdx.x : xcd_group_block(blockIdx.x, gridDim.x, 16 >> a.lb);
  const int x = blk * RPB + slot_id;
  if (x >= a.nx) return;
  const int pg = a.probe0;
  float2* slot = lds + slot_id * lds_slot<NY>();
  Twiddles<NY> tw;
  tw.init(a.twy, t);
  // band columns through buffer resources: offsets in the band gap are kOut, so
  // their loads return 0 and their stores are dropped (no per-element branches)
  const int gap = NY - a.band_b - a.band_a - 1;
  const size_t poff = (size_t)pg * a.nx * a.kcp;
  const long pbytes = (long)a.nx * a.kcp * 8;
  const rsrc_t rg = make_rsrc(A.gx + poff, pbytes);
  const unsigned xo = row_off(x, a.lb, a.kcp);
  unsigned bo[E];
#pragma unroll
  for (int m = 0; m < E; m++) {
    const unsigned o = band_off(t + T * m, a.band_a, gap, a.lb);
    bo[m] = o == kOut ? kOut : o + xo;
  }
  float2 g[E], w[E];
#pragma unroll
  for (int m = 0; m < E; m++) g[m] = buf_load_c64(rg, bo[m]);
  fft_wave<NY, +1>(g, slot, tw, t);
  if constexpr (FIRST) {
    const float2* pr = a.probe + (size_t)x * NY;
#pragma unroll
    for (int m = 0; m < E; m++) w[m] = pr[t + T * m];
  } else {
    const rsrc_t rx = make_rsrc(A.xprev + poff, pbytes);
#pragma unroll
    for (int m = 0; m < E; m++) w[m] = buf_load_c64(rx, bo[m]);
    fft_wave<NY, +1>(w, slot, tw, t);
  }
  const int2 ip = a.ipos[pg];
  const float2* tr = a.trans + (size_t)(x + ip.x) * a.potNy + ip.y;
  float* gt = BLF ? nullptr : A.gT + 2 * ((size_t)(x + ip.x) * a.potNy + ip.y);  // BLF: no dL/dt buffer
#pragma unroll
  for (int m = 0; m < E; m++) {
    const int iy = t + T * m;
    const float2 gtv = cmulc(g[m], w[m]);  // conj(psi) * g_a
    if constexpr (BLF) {
      w[m] = gtv;  // kept for the row FFT below
    } else if (A.single_writer == 2) {  // the window is the whole slice: this is the pixel's only term
      *reinterpret_cast<float2*>(gt + 2 * iy) = gtv;
    } else {  // one probe per launch: each transmission pixel has one writer
      float2* p2 = reinterpret_cast<float2*>(gt + 2 * iy);
      const float2 o = *p2;
      *p2 = make_float2(o.x + gtv.x, o.y + gtv.y);
    }
    g[m] = cmulc(g[m], tr[iy]);  // conj(t) * g_a
  }
  if constexpr (BLF) {
    // the band limit's first pass (k_sweep_rows mode 3) on the row x of g_t: row FFT,
    // band columns of the potential grid stored (offsets in its band gap are kOut)
    fft_wave<NY, -1>(w, slot, tw, t);
    const rsrc_t rb = make_rsrc(A.blstate, (long)a.nx * A.bl_kcp * 8);  // (the window is the whole slice: x is its row)
    const unsigned bxo = row_off(x, a.lb, A.bl_kcp);
#pragma unroll
    for (int m = 0; m < E; m++) {
      const unsigned o = band_off(t + T * m, A.bl_band_a, A.bl_gap, a.lb);
      buf_store_c64(w[m], rb, o == kOut ? kOut : o + bxo);
    }
  }
  if constexpr (FIRST) {
    float* gp = A.gprobe + 2 * (size_t)x * NY;
#pragma unroll
    for (int m = 0; m < E; m++) {
      atomicAdd(gp + 2 * (t + T * m), g[m].x);
      atomicAdd(gp + 2 * (t + T * m) + 1, g[m].y);
    }
  } else {
    fft_wave<NY, -1>(g, slot, tw, t);
#pragma unroll
    for (int m = 0; m < E; m++) buf_store_c64(g[m], rg, bo[m]);
  }
}

// The same sweep for several probes, whose windows overlap in the slice.  A block owns a
// group of TPW consecutive transmission rows (the rows that the transforms of one wavefront
// work on side by side) and a chunk of the probes that read them.  Each wavefront takes a
// contiguous run of the chunk, one probe at a time (its row bases are scalars), and sums
// dL/dt of the rows in an LDS area of its own by plain loads and stores; at the end the
// block adds the areas and issues one global atomic pair per touched pixel.  With one
// global atomic pair per pixel and probe the sweep was bound by the atomics (134 M float
// atomics per slice for 1024 probes of 256^2 in 384^2: 1346 us; with the sums as LDS float
// atomics 1143 us; now 372 us, of which the 1.1 GB of state take 206 us at copy rate).  In the first slice a wavefront sums
// g_psi of neighbouring probes with the same x offset in registers before the atomics on
// gprobe.
template <int N> constexpr int adj_tpw() { return N / Plan<N>::E <= 64 ? 64 / (N / Plan<N>::E) : 1; }
template <int N> constexpr int adj_units() { return N / Plan<N>::E <= 64 ? row_block<N>() / 64 : 1; }
// Widest span of a chunk's windows that is summed in LDS (48 KB per block); wider ones add
// straight to A.gT.
template <int N> constexpr int adj_acc_max() { return 6144 / (adj_tpw<N>() * adj_units<N>()); }

template <int NY, bool FIRST>
__global__ __launch_bounds__(row_block<NY>()) void k_adj_rows_acc(AdjArgs A) {
  const SweepArgs& a = A.f;
  constexpr int E = Plan<NY>::E;
  constexpr int T = NY / E;
  constexpr int BLK = row_block<NY>();
  constexpr int TPW = adj_tpw<NY>();
  constexpr int GAP = gap_mask<NY>();  // slots in the band gap: never loaded, stored or computed
  constexpr int UPB = adj_units<NY>();  // units (wavefronts, or the block) per block
  __shared__ float2 lds[(BLK / T) * lds_slot<NY>()];
  __shared__ int yspan[2];
  extern __shared__ float2 acc[];  // [UPB][TPW][span]
  // the groups that share a line of the state (x0 of a probe moves them against the lines,
  // so only most of them) take the same chunk on one XCD at the same time
  const int ls = 16 >> a.lb;
  const int item = xcd_group_block(blockIdx.x, gridDim.x, ls);
  const int group = item / ls / A.nchunk * ls + item % ls, chunk = item / ls % A.nchunk;
  const int X0 = group * TPW;
  if (X0 >= A.potNx) return;
  const int2 range = A.xrange[group];
  const int lo = range.x + chunk * A.chunk, hi = min(range.y, lo + A.chunk);
  if (lo >= hi) return;  // whole blocks
  if (threadIdx.x == 0) {
    yspan[0] = 0x7fffffff;
    yspan[1] = 0;
  }
  __syncthreads();
  for (int i = lo + threadIdx.x; i < hi; i += BLK) {
    const int y = a.ipos[A.order[i]].y;
    atomicMin(&yspan[0], y);
    atomicMax(&yspan[1], y + NY);
  }
  __syncthreads();
  const int ylo = wave_uniform(yspan[0]), span = wave_uniform(yspan[1]) - ylo;
  const bool in_lds = span <= adj_acc_max<NY>();
  if (in_lds) {
    for (int i = threadIdx.x; i < UPB * TPW * span; i += BLK) acc[i] = make_float2(0.f, 0.f);
  }
  __syncthreads();
  const int lane = T <= 64 ? (threadIdx.x & 63) : threadIdx.x;
  const int unit = T <= 64 ? wave_uniform(threadIdx.x >> 6) : 0;
  const int sub = lane / T, t = lane % T;
  float2* slot = lds + (threadIdx.x / T) * lds_slot<NY>();
  Twiddles<NY> tw;
  tw.init(a.twy, t);
  // band columns through buffer resources, as in k_adj_rows
  const int gap = NY - a.band_b - a.band_a - 1;
  unsigned bo[E];
#pragma unroll
  for (int m = 0; m < E; m++) bo[m] = band_off(t + T * m, a.band_a, gap, a.lb);
  const int X = X0 + sub;
  const float2* const trow = a.trans + (size_t)min(X, A.potNx - 1) * a.potNy + t;
  float* const grow = A.gT + 2 * ((size_t)min(X, A.potNx - 1) * a.potNy + t);
  float2* const accr = acc + (unit * TPW + sub) * span + t;
  const int per = (hi - lo + UPB - 1) / UPB;  // probes of this unit
  const int i1 = min(hi, lo + (unit + 1) * per);
  float2 gsum[FIRST ? E : 1];
  if constexpr (FIRST) {
#pragma unroll
    for (int m = 0; m < E; m++) gsum[m] = make_float2(0.f, 0.f);
  }
  for (int i = lo + unit * per; i < i1; i++) {
    const int p = A.order[i];
    const int2 ip = a.ipos[p];
    const int x0 = X0 - ip.x;  // window row of sub 0; rows outside [0, nx) read zeros and store nothing
    const bool row = x0 + sub >= 0 && x0 + sub < a.nx;
    const size_t poff = (size_t)p * a.nx * a.kcp;
    const long pbytes = (long)a.nx * a.kcp * 8;
    const rsrc_t rg = make_rsrc(A.gx + poff, pbytes);
    const unsigned ro = row_off(x0 + sub, a.lb, a.kcp);
    auto off = [&](int m) -> unsigned { return bo[m] == kOut || !row ? kOut : bo[m] + ro; };
    float2 g[E], w[E];
#pragma unroll
    for (int m = 0; m < E; m++) g[m] = (GAP >> m) & 1 ? make_float2(0.f, 0.f) : buf_load_c64(rg, off(m));
    if constexpr (FIRST) {
      const float2* pr = a.probe + (size_t)(row ? x0 + sub : 0) * NY + t;
#pragma unroll
      for (int m = 0; m < E; m++) w[m] = row ? pr[T * m] : make_float2(0.f, 0.f);
    } else {
      const rsrc_t rx = make_rsrc(A.xprev + poff, pbytes);
#pragma unroll
      for (int m = 0; m < E; m++) w[m] = (GAP >> m) & 1 ? make_float2(0.f, 0.f) : buf_load_c64(rx, off(m));
    }
    fft_wave<NY, +1, kSwz<NY>, GAP>(g, slot, tw, t);
    if constexpr (!FIRST) fft_wave<NY, +1, kSwz<NY>, GAP>(w, slot, tw, t);
    const float2* tr = trow + ip.y;
#pragma unroll
    for (int m = 0; m < E; m++) {
      const float2 gtv = cmulc(g[m], w[m]);  // conj(psi) * g_a
      if (in_lds) {  // the unit's own area (block-wide transforms: ordered by their barriers)
        float2* const q = accr + (ip.y - ylo) + T * m;
        *q = cadd(*q, gtv);
      } else if (row) {
        atomicAdd(grow + 2 * (ip.y + T * m), gtv.x);
        atomicAdd(grow + 2 * (ip.y + T * m) + 1, gtv.y);
      }
      g[m] = cmulc(g[m], tr[T * m]);  // conj(t) * g_a
    }
    if constexpr (FIRST) {
#pragma unroll
      for (int m = 0; m < E; m++) gsum[m] = cadd(gsum[m], g[m]);
      if (i + 1 == i1 || a.ipos[A.order[i + 1]].x != ip.x) {  // the unit's next row is another row of gprobe
        if (row) {
          float* gp = A.gprobe + 2 * ((size_t)(x0 + sub) * NY + t);
#pragma unroll
          for (int m = 0; m < E; m++) {
            atomicAdd(gp + 2 * T * m, gsum[m].x);
            atomicAdd(gp + 2 * T * m + 1, gsum[m].y);
          }
        }
#pragma unroll
        for (int m = 0; m < E; m++) gsum[m] = make_float2(0.f, 0.f);
      }
    } else {
      fft_wave<NY, -1, kSwz<NY>, 0, ~GAP>(g, slot, tw, t);
#pragma unroll
      for (int m = 0; m < E; m++)
        if (!((GAP >> m) & 1)) buf_store_c64(g[m], rg, off(m));
    }
  }
  __syncthreads();
  if (in_lds) {
#pragma unroll 1
    for (int r = 0; r < TPW && X0 + r < A.potNx; r++) {
      float* const gr = A.gT + 2 * ((size_t)(X0 + r) * a.potNy + ylo);
      for (int i = threadIdx.x; i < span; i += BLK) {
        float2 sum = acc[r * span + i];
#pragma unroll
        for (int u = 1; u < UPB; u++) sum = cadd(sum, acc[(u * TPW + r) * span + i]);
        atomicAdd(gr + 2 * i, sum.x);
        atomicAdd(gr + 2 * i + 1, sum.y);
      }
    }
  }
}

template <int N>
void launch_adj_rows_acc_t(const AdjArgs& a, bool first, hipStream_t st) {
  constexpr int TPW = adj_tpw<N>();
  const int ls = 16 >> a.f.lb, groups = (a.potNx + TPW - 1) / TPW;  // adj_row_shape's rows per group
  const dim3 grid((unsigned)((groups + ls - 1) / ls * ls * a.nchunk));
  const size_t lds = sizeof(float2) * TPW * adj_units<N>() * (a.f.potNy < adj_acc_max<N>() ? a.f.potNy : adj_acc_max<N>());
  if (first) hipLaunchKernelGGL((k_adj_rows_acc<N, true>), grid, dim3(row_block<N>()), lds, st, a);
  else hipLaunchKernelGGL((k_adj_rows_acc<N, false>), grid, dim3(row_block<N>()), lds, st, a);
}

template <int N>
void launch_adj_rows_t(const AdjArgs& a, bool first, hipStream_t st) {
  if (!a.single_writer) return launch_adj_rows_acc_t<N>(a, first, st);
  constexpr int T = N / Plan<N>::E;
  constexpr int RPB = row_block<N>() / T;
  const long rows = (long)a.f.nprobe * a.f.nx;
  dim3 grid((unsigned)((rows + RPB - 1) / RPB));
  if (a.blstate) {
    if (first) hipLaunchKernelGGL((k_adj_rows<N, true, true>), grid, dim3(row_block<N>()), 0, st, a);
    else hipLaunchKernelGGL((k_adj_rows<N, false, true>), grid, dim3(row_block<N>()), 0, st, a);
  } else {
    if (first) hipLaunchKernelGGL((k_adj_rows<N, true, false>), grid, dim3(row_block<N>()), 0, st, a);
    else hipLaunchKernelGGL((k_adj_rows<N, false, false>), grid, dim3(row_block<N>()), 0, st, a);
  }
}

// Up to 256 the direct reverse kernel has a longer serial chain (block barriers in every
// exchange) and half as many blocks: from three blocks per CU on it is the faster one, with the
// loss, whose target reads it spreads over whole lines, from two (at 64 always).  Staged /
// direct, us: 256 points, 40 probes 12.1 / 13.5, 60 13.6 / 15.0, 80 17.9 / 16.9; with the loss
// 30 14.3 / 15.9, 40 16.8 / 16.6, 60 25.7 / 18.8; 128 points, 40 probes 7.4 / 8.0, 120 12.4 /
// 13.0, 320 19.4 / 16.0; with the loss 60 12.1 / 13.9, 120 20.7 / 15.6; 64 points, 160 probes
// 5.6 / 6.1, 640 12.3 / 11.4; with the loss 2 7.9 / 6.8, 640 19.3 / 12.8.
template <int N>
bool adj_cols_staged_run(const SweepArgs& a, bool last) {
  if constexpr (!adj_col_direct<N>()) return true;
  if constexpr (!adj_col_staged<N>()) return false;
  return (long)a.nprobe * col_blocks<N>(a) < (last ? (N == 64 ? 0 : 512) : 768);
}

template <int N>
void launch_adj_cols_t(const AdjArgs& a0, bool last, hipStream_t st) {
  AdjArgs a = a0;
  if (adj_cols_staged_run<N>(a.f, last)) {
    if constexpr (adj_col_staged<N>()) {
      const dim3 grid((unsigned)(a.f.nprobe * a.f.ntiles)), block(TileCfg<N>::BLK);
      constexpr int lds = col_lds_bytes_t<N, true>();
      if (last) hipLaunchKernelGGL((k_tile_adj_cols<N, true>), grid, block, lds, st, a);
      else hipLaunchKernelGGL((k_tile_adj_cols<N, false>), grid, block, lds, st, a);
    }
  } else if constexpr (adj_col_direct<N>()) {
    a.f.tpb = col_probes<N>(a.f);
    const dim3 grid((unsigned)((a.f.nprobe + a.f.tpb - 1) / a.f.tpb * col_blocks<N>(a.f))), block(ColCfg<N>::BLK);
    constexpr int lds = col_lds_bytes_t<N, false>();
    if (last) hipLaunchKernelGGL((k_adj_cols<N, true>), grid, block, lds, st, a);
    else hipLaunchKernelGGL((k_adj_cols<N, false>), grid, block, lds, st, a);
  }
}

template <int N>
hipError_t set_adj_lds_t() {
  hipError_t e = hipSuccess;
  auto allow = [&](const void* kernel, int bytes) {
    if (e == hipSuccess) e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  };
  if constexpr (adj_col_staged<N>()) {
    allow(reinterpret_cast<const void*>(&k_tile_adj_cols<N, true>), col_lds_bytes_t<N, true>());
    allow(reinterpret_cast<const void*>(&k_tile_adj_cols<N, false>), col_lds_bytes_t<N, true>());
  }
  if constexpr (adj_col_direct<N>()) {
    allow(reinterpret_cast<const void*>(&k_adj_cols<N, true>), col_lds_bytes_t<N, false>());
    allow(reinterpret_cast<const void*>(&k_adj_cols<N, false>), col_lds_bytes_t<N, false>());
  }
  const int acc = (int)sizeof(float2) * adj_tpw<N>() * adj_units<N>() * adj_acc_max<N>();
  allow(reinterpret_cast<const void*>(&k_adj_rows_acc<N, true>), acc);
  allow(reinterpret_cast<const void*>(&k_adj_rows_acc<N, false>), acc);
  return e;
}

}  // namespace qs
