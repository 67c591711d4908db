// qs_fft.hpp -- wavefront-resident Stockham FFT building blocks for gfx950.
//
// A length-N transform is owned by T = N/E consecutive threads: lanes of one
// 64-wide wavefront up to N = 1024, a whole 256-thread block beyond; each
// thread holds E complex values in registers.  In the natural layout thread t
// holds elements t + T*m, m = 0..E-1, which is also the layout coalesced
// global loads and stores produce, so the first pass takes its input straight
// from registers and the last pass leaves its output there.  Between passes
// the values are exchanged through a per-transform LDS slot.
//
// Pass structure (Stockham autosort): for radix R and span Ns, butterfly
// j = t + T*b (b < E/R) reads x[j + k*N/R], applies twiddles
// W_{Ns R}^{k (j mod Ns)} and writes y_k to out[(j/Ns)*Ns*R + j%Ns + k*Ns].
// Directions follow FFTW/QSTEM: DIR = -1 forward, +1 backward, both
// unnormalised (libs/data_containers.cpp:50-51).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace qs {

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {  // a * conj(b)
  return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__device__ __forceinline__ float cnorm(float2 a) { return a.x * a.x + a.y * a.y; }
// multiply by -i (DIR=-1) or +i (DIR=+1)
template <int DIR>
__device__ __forceinline__ float2 mul_i(float2 a) {
  return DIR < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

// ---- in-register DFTs ------------------------------------------------------
template <int DIR>
__device__ __forceinline__ void dft2(float2& a, float2& b) {
  float2 t = a;
  a = cadd(t, b);
  b = csub(t, b);
}

template <int DIR>
__device__ __forceinline__ void dft4(float2& a0, float2& a1, float2& a2, float2& a3) {
  float2 t0 = cadd(a0, a2), t1 = csub(a0, a2);
  float2 t2 = cadd(a1, a3), t3 = mul_i<DIR>(csub(a1, a3));
  a0 = cadd(t0, t2);
  a2 = csub(t0, t2);
  a1 = cadd(t1, t3);
  a3 = csub(t1, t3);
}

// dft4 with inputs known to be zero (bit j of Z: input j is zero); the
// additions with a zero operand are left out.
__device__ __forceinline__ float2 cneg(float2 a) { return make_float2(-a.x, -a.y); }
template <int DIR, int Z>
__device__ __forceinline__ void dft4z(float2& a0, float2& a1, float2& a2, float2& a3) {
  if constexpr (Z == 0) {
    dft4<DIR>(a0, a1, a2, a3);
  } else {
    float2 t0, t1, t2, t3;
    if constexpr ((Z & 4) != 0) { t0 = a0; t1 = a0; }
    else if constexpr ((Z & 1) != 0) { t0 = a2; t1 = cneg(a2); }
    else { t0 = cadd(a0, a2); t1 = csub(a0, a2); }
    if constexpr ((Z & 8) != 0) { t2 = a1; t3 = mul_i<DIR>(a1); }
    else if constexpr ((Z & 2) != 0) { t2 = a3; t3 = mul_i<DIR>(cneg(a3)); }
    else { t2 = cadd(a1, a3); t3 = mul_i<DIR>(csub(a1, a3)); }
    a0 = cadd(t0, t2);
    a2 = csub(t0, t2);
    a1 = cadd(t1, t3);
    a3 = csub(t1, t3);
  }
}

// W8^k for k = 1,3 with sign DIR: e^{DIR*i*pi*k/4}
template <int DIR>
__device__ __forceinline__ float2 w8_1(float2 a) {  // a * e^{DIR i pi/4}
  const float h = 0.70710678118654752440f;
  return DIR < 0 ? make_float2((a.x + a.y) * h, (a.y - a.x) * h) : make_float2((a.x - a.y) * h, (a.y + a.x) * h);
}
template <int DIR>
__device__ __forceinline__ float2 w8_3(float2 a) {  // a * e^{DIR i 3pi/4}
  const float h = 0.70710678118654752440f;
  return DIR < 0 ? make_float2((a.y - a.x) * h, -(a.x + a.y) * h) : make_float2(-(a.x + a.y) * h, (a.x - a.y) * h);
}

// Z: bit j set when input j is zero; O: bit k set when output k is needed
// (the others are left unspecified).
template <int DIR, int Z = 0, int O = 0xff>
__device__ __forceinline__ void dft8(float2* a) {
  // decimation in time: even/odd halves, then combine with W8^k
  constexpr int ZE = ((Z >> 0) & 1) | (((Z >> 2) & 1) << 1) | (((Z >> 4) & 1) << 2) | (((Z >> 6) & 1) << 3);
  constexpr int ZO = ((Z >> 1) & 1) | (((Z >> 3) & 1) << 1) | (((Z >> 5) & 1) << 2) | (((Z >> 7) & 1) << 3);
  float2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6];
  float2 o0 = a[1], o1 = a[3], o2 = a[5], o3 = a[7];
  dft4z<DIR, ZE>(e0, e1, e2, e3);
  dft4z<DIR, ZO>(o0, o1, o2, o3);
  o1 = w8_1<DIR>(o1);
  o2 = mul_i<DIR>(o2);
  o3 = w8_3<DIR>(o3);
  if constexpr ((O & 0x01) != 0) a[0] = cadd(e0, o0);
  if constexpr ((O & 0x10) != 0) a[4] = csub(e0, o0);
  if constexpr ((O & 0x02) != 0) a[1] = cadd(e1, o1);
  if constexpr ((O & 0x20) != 0) a[5] = csub(e1, o1);
  if constexpr ((O & 0x04) != 0) a[2] = cadd(e2, o2);
  if constexpr ((O & 0x40) != 0) a[6] = csub(e2, o2);
  if constexpr ((O & 0x08) != 0) a[3] = cadd(e3, o3);
  if constexpr ((O & 0x80) != 0) a[7] = csub(e3, o3);
}

// cos and sin of pi/8, and the next larger float of the cosine: the nearest one loses 2.9e-8
// of the modulus, the next gains 2.7e-8, and what every transform loses adds up over a run.
// The transforms below (BAL) use the next one often enough to balance the losses at pi/8 and
// pi/4.
constexpr float kCos16 = 0.92387953251128675613f, kCos16Up = 0x1.d906bep-1f, kSin16 = 0.38268343236508977173f;

template <int DIR, int Z = 0, bool BAL = true>
__device__ __forceinline__ void dft16(float2* a) {
  // 16 = 4 x 4: columns of stride 4, twiddles W16^{n1 k2}, rows of length 4
  const float c1 = kCos16, cu = BAL ? kCos16Up : kCos16, s1 = kSin16;
  const float h = 0.70710678118654752440f;
  float2 b[16];
  auto colz = [](int n1) constexpr {
    return ((Z >> n1) & 1) | (((Z >> (n1 + 4)) & 1) << 1) | (((Z >> (n1 + 8)) & 1) << 2) | (((Z >> (n1 + 12)) & 1) << 3);
  };
  auto col = [&](auto n1c) {
    constexpr int n1 = decltype(n1c)::value;
    float2 x0 = a[n1], x1 = a[n1 + 4], x2 = a[n1 + 8], x3 = a[n1 + 12];
    dft4z<DIR, colz(n1)>(x0, x1, x2, x3);
    b[n1 * 4 + 0] = x0; b[n1 * 4 + 1] = x1; b[n1 * 4 + 2] = x2; b[n1 * 4 + 3] = x3;
  };
  col(std::integral_constant<int, 0>{});
  col(std::integral_constant<int, 1>{});
  col(std::integral_constant<int, 2>{});
  col(std::integral_constant<int, 3>{});
  // twiddle b[n1*4+k2] *= W16^{n1*k2}
  const float sg = (float)DIR;
  const float2 w1 = make_float2(c1, sg * s1), w2 = make_float2(h, sg * h), w3 = make_float2(s1, sg * cu);
  const float2 w6 = make_float2(-h, sg * h), w9 = make_float2(-cu, -sg * s1);
  b[1 * 4 + 1] = cmul(b[5], w1);
  b[1 * 4 + 2] = cmul(b[6], w2);
  b[1 * 4 + 3] = cmul(b[7], w3);
  b[2 * 4 + 1] = cmul(b[9], w2);
  b[2 * 4 + 2] = mul_i<DIR>(b[10]);
  b[2 * 4 + 3] = cmul(b[11], w6);
  b[3 * 4 + 1] = cmul(b[13], w3);
  b[3 * 4 + 2] = cmul(b[14], w6);
  b[3 * 4 + 3] = cmul(b[15], w9);
#pragma unroll
  for (int k2 = 0; k2 < 4; k2++) {
    float2 x0 = b[k2], x1 = b[4 + k2], x2 = b[8 + k2], x3 = b[12 + k2];
    dft4<DIR>(x0, x1, x2, x3);
    a[k2] = x0; a[k2 + 4] = x1; a[k2 + 8] = x2; a[k2 + 12] = x3;
  }
}

// Z, O: zero inputs and needed outputs (dft8 prunes both, dft16 the inputs).
template <int R, int DIR, int Z = 0, int O = -1, bool BAL = true>
__device__ __forceinline__ void dft(float2* a) {
  if constexpr (R == 2) dft2<DIR>(a[0], a[1]);
  else if constexpr (R == 4) dft4z<DIR, Z & 15>(a[0], a[1], a[2], a[3]);
  else if constexpr (R == 8) dft8<DIR, Z & 0xff, O & 0xff>(a);
  else if constexpr (R == 16) dft16<DIR, Z & 0xffff, BAL>(a);
}

// ---- radix plans -------------------------------------------------------------
// E: values per thread; T = N/E threads per transform (one wavefront up to
// N = 1024, the whole 256-thread block for 2048 and 4096); NP passes of radix
// R0..R3 (each divides E).  At 4096, {8,8,8,8} over 512 threads (about half
// the registers per thread, twice the waves per CU) measured slower than
// {16,16,16} over 256: forward rows by 27 %, reverse columns by 57 %, forward
// columns 3 % faster.
template <int N> struct Plan;
template <> struct Plan<64>   { static constexpr int E = 4,  NP = 3, R0 = 4,  R1 = 4,  R2 = 4,  R3 = 1; };
template <> struct Plan<128>  { static constexpr int E = 8,  NP = 3, R0 = 8,  R1 = 8,  R2 = 2,  R3 = 1; };
template <> struct Plan<256>  { static constexpr int E = 8,  NP = 3, R0 = 8,  R1 = 8,  R2 = 4,  R3 = 1; };
template <> struct Plan<512>  { static constexpr int E = 8,  NP = 3, R0 = 8,  R1 = 8,  R2 = 8,  R3 = 1; };
template <> struct Plan<1024> { static constexpr int E = 16, NP = 3, R0 = 16, R1 = 8,  R2 = 8,  R3 = 1; };
template <> struct Plan<2048> { static constexpr int E = 8,  NP = 4, R0 = 8,  R1 = 8,  R2 = 8,  R3 = 4; };
template <> struct Plan<4096> { static constexpr int E = 16, NP = 3, R0 = 16, R1 = 16, R2 = 16, R3 = 1; };

// LDS placement of element i of a length-N transform, in one of two layouts.
// On gfx950 a ds_read_b64 serves 32 lanes at a time over 32 eight-byte bank
// pairs and a ds_write_b64 16 lanes over 16.
//  SWZ (default up to N = 512): the low four index bits are XORed with a
//    function of bits 4.. (i ^ f_N(i >> 4)); every read and write pattern of
//    fft_wave below then hits distinct bank pairs (sizes 64 and 128 also need
//    the slot strides of lds_slot, as several transforms share a wavefront).
//    The write addresses are no longer immediate offsets from one base, so
//    the compiler keeps one address register per access.
//  PAD: one float2 of padding every 16 (i + (i >> 4)): immediate offsets from
//    a per-thread base, at a residual 1.3-1.6-way conflict rate; used beyond
//    512 and wherever registers are the scarcer resource.
template <int N> constexpr bool kSwz = N <= 512;
template <int N, bool SWZ = kSwz<N>>
__device__ __forceinline__ int lidx(int i) {
  if constexpr (!SWZ) {
    return i + (i >> 4);
  } else {
    const int j = i >> 4;
    int f;
    if constexpr (N == 64) f = ((j & 1) ? 9 : 0) ^ (((j ^ (j >> 1)) & 1) ? 6 : 0);
    else f = (j & 7) | (((j >> 2) & 1) << 3);
    return i ^ f;
  }
}
template <int N, bool SWZ = kSwz<N>>
constexpr int lds_slot() { return SWZ ? (N == 64 ? 80 : (N == 128 ? 144 : N)) : N + N / 16; }

// Orders this lane's LDS reads before later LDS writes of other lanes of the
// same wavefront and vice versa (all lanes of a transform live in one wave).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS ordering between the threads of one length-N transform: a wavefront
// barrier when the transform lives in one wavefront, else a block barrier
// (the block is the transform; every thread of it reaches every call).
template <int N>
__device__ __forceinline__ void xform_sync() {
  if constexpr (N / Plan<N>::E <= 64) wave_lds_sync();
  else __syncthreads();
}

// ---- twiddled butterflies ------------------------------------------------------
// A radix-R butterfly of inputs a_k with twiddles w^k evaluates A(z) = sum_k a_k z^k at
// z = w W_R^q, q < R.  Splitting z^(R/2) = +-c at every level makes it log2(R) stages of
// radix-2 butterflies u = a + c b, v = a - c b with the twiddle and the rotation in c.  With
// c = cos (1 + i tan) each takes six fused multiply-adds: b (1 + i tan) in two, and its
// product with the cosine added to and subtracted from a in four: 72 instead of 84
// instructions for R = 8, 192 instead of 228 for R = 16.  (v = 2a - u from u = a + c b also
// takes six, but carries the rounding of u into v: where |u| is much larger than |v|, as for
// a wave with a large mean, a 4096-point transform's rms error was 30% larger.)  The node of
// size R' at offset q0 (points q0 + (R/R') k) splits with c = w^(R'/2) W_R^(q0 R'/2); odd
// halves differ from their even siblings by a quarter turn, so R/2 constants serve all nodes:
//   R = 2: w;  4: w^2, w;  8: w^4, w^2, w, w W_8;
//   16: w^8, w^4, w^2, w^2 W_8, w, w W_8, w W_16, w W_16^3.

// u = a + c b -> a, v = a - c b -> b, with c = (cos, tan) conjugated for DIR > 0 and a quarter
// turn in the direction of the transform for ROT.  NU, NV: outputs needed.
template <int DIR, bool ROT, bool NU = true, bool NV = true>
__device__ __forceinline__ void bf_tw(float2& a, float2& b, float2 c) {
  const float t = DIR < 0 ? c.y : -c.y;
  float2 y = make_float2(fmaf(-t, b.y, b.x), fmaf(t, b.x, b.y));
  if constexpr (ROT) y = mul_i<DIR>(y);
  const float2 x = a;
  if constexpr (NU) a = make_float2(fmaf(c.x, y.x, x.x), fmaf(c.x, y.y, x.y));
  if constexpr (NV) b = make_float2(fmaf(-c.x, y.x, x.x), fmaf(-c.x, y.y, x.y));
}

// Exponents of constant i: w^tw_pow W_R^tw_rot.
template <int R> constexpr int tw_pow(int i) {
  if (R == 2) return 1;
  if (R == 4) return i == 0 ? 2 : 1;
  if (R == 8) return i == 0 ? 4 : (i == 1 ? 2 : 1);
  return i == 0 ? 8 : (i == 1 ? 4 : (i < 4 ? 2 : 1));
}
template <int R> constexpr int tw_rot(int i) {
  if (R == 8) return i == 3 ? 1 : 0;
  if (R == 16) return i == 3 ? 2 : (i == 5 ? 2 : (i == 6 ? 1 : (i == 7 ? 3 : 0)));
  return 0;
}
// Constant (and quarter turn) of the node of size S at offset q0 of a radix-R butterfly.
template <int R> constexpr int tw_index(int S, int q0) {
  const int rot = q0 * (S / 2) % (R / 4 > 0 ? R / 4 : 1);  // without the quarter turn
  for (int i = 0; i < R / 2; i++)
    if (tw_pow<R>(i) == S / 2 && tw_rot<R>(i) == rot) return i;
  return -1;
}
template <int R> constexpr bool tw_quarter(int S, int q0) { return R >= 4 && q0 * (S / 2) >= R / 4; }

// The node of size S at offset q0, its inputs in a[0], a[1], ..; y[q] receives the outputs.
template <int R, int S, int Q0, int DIR, int NEED>
__device__ __forceinline__ void node_tw(float2* a, float2* y, const float2* c) {
  constexpr int I = tw_index<R>(S, Q0);
  static_assert(I >= 0, "no constant for this node");
  constexpr bool ROT = tw_quarter<R>(S, Q0);
  constexpr int q1 = Q0 + R / 2;
  constexpr bool NU = S > 2 || ((NEED >> Q0) & 1) != 0, NV = S > 2 || ((NEED >> q1) & 1) != 0;
#pragma unroll
  for (int j = 0; j < S / 2; j++) bf_tw<DIR, ROT, NU, NV>(a[j], a[j + S / 2], c[I]);
  if constexpr (S == 2) {
    y[Q0] = a[0];
    y[q1] = a[1];
  } else {
    node_tw<R, S / 2, Q0, DIR, NEED>(a, y, c);
    node_tw<R, S / 2, Q0 + R / S, DIR, NEED>(a + S / 2, y, c);
  }
}
template <int R, int DIR, int NEED = -1>
__device__ __forceinline__ void dft_tw(float2* a, const float2* c) {
  float2 y[R];
  node_tw<R, R, 0, DIR, NEED>(a, y, c);
#pragma unroll
  for (int q = 0; q < R; q++) a[q] = y[q];
}

// The R/2 constants of a butterfly whose twiddle is w = W_N^m, from the table of W_N^m as
// (cos, tan) pairs.
template <int N, int R>
__device__ __forceinline__ void tw_load(float2* c, const float2* __restrict__ tw, int m) {
#pragma unroll
  for (int i = 0; i < R / 2; i++) c[i] = tw[tw_pow<R>(i) * m + tw_rot<R>(i) * (N / R)];
}

// Per-thread constants of the twiddled passes, read once from the table and kept in registers
// (8 to 16 complex values) for every transform the thread performs.  Computing the twiddles in
// the pass instead (sines and cosines by series, 25 instructions each) was half of the
// 4096-point row sweep's instructions.
template <int N>
struct Twiddles {
  using P = Plan<N>;
  static constexpr int T = N / P::E;
  static constexpr int NS1 = P::R0, NS2 = P::R0 * P::R1, NS3 = P::R0 * P::R1 * P::R2;
  // butterflies of a pass share their constants when T is a multiple of the span
  static constexpr int B1 = T % NS1 == 0 ? 1 : P::E / P::R1;
  static constexpr int B2 = P::NP < 3 ? 0 : (T % NS2 == 0 ? 1 : P::E / P::R2);
  static constexpr int B3 = P::NP < 4 ? 0 : (T % NS3 == 0 ? 1 : P::E / P::R3);
  float2 w1[B1 * (P::R1 / 2)], w2[B2 > 0 ? B2 * (P::R2 / 2) : 1], w3[B3 > 0 ? B3 * (P::R3 / 2) : 1];
  template <int R, int NS, int B>
  static __device__ __forceinline__ void load(float2* w, const float2* __restrict__ tw, int t) {
#pragma unroll
    for (int b = 0; b < B; b++) tw_load<N, R>(w + b * (R / 2), tw, (t + T * b) % NS * (N / (NS * R)));
  }
  __device__ __forceinline__ void init(const float2* __restrict__ tw, int t) {
    load<P::R1, NS1, B1>(w1, tw, t);
    if constexpr (P::NP >= 3) load<P::R2, NS2, B2>(w2, tw, t);
    if constexpr (P::NP >= 4) load<P::R3, NS3, B3>(w3, tw, t);
  }
};

// One Stockham pass.  FIRST: input from registers (natural layout), no twiddles.  LAST:
// output to registers (natural layout).  Otherwise through the LDS slot.
// w: the pass's constants (Twiddles), B sets of them over the thread's butterflies.
// ZIN (first pass) / NEED (last pass): masks over the natural-layout register
// slots m (element t + T*m) that are zero on input / needed on output; used when
// one butterfly covers all E slots (R == E), ignored otherwise.
template <int N, int R, int NS, int DIR, bool FIRST, bool LAST, bool SWZ, int B, int ZIN = 0, int NEED = -1>
__device__ __forceinline__ void stockham_pass(float2* v, float2* slot, const float2* w, int t) {
  constexpr int E = Plan<N>::E;
  constexpr int T = N / E;
  constexpr int NB = E / R;
  float2 a[NB][R];
  if constexpr (FIRST) {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int k = 0; k < R; k++) a[b][k] = v[b + k * NB];
  } else {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int k = 0; k < R; k++) a[b][k] = slot[lidx<N, SWZ>(t + T * b + k * (N / R))];
  }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    if constexpr (FIRST) {
      if constexpr (NB == 1) dft<R, DIR, ZIN>(a[b]);
      else dft<R, DIR>(a[b]);
    } else {
      dft_tw<R, DIR, LAST && NB == 1 ? NEED : -1>(a[b], w + (B > 1 ? b * (R / 2) : 0));
    }
  }
  if constexpr (LAST) {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int k = 0; k < R; k++) v[b + k * NB] = a[b][k];
  } else {
    xform_sync<N>();  // all earlier reads of the slot precede these writes
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int j = t + T * b;
      const int base = (j / NS) * NS * R + (j % NS);
#pragma unroll
      for (int k = 0; k < R; k++) slot[lidx<N, SWZ>(base + k * NS)] = a[b][k];
    }
    xform_sync<N>();
  }
}

// Register slots m (element t + T*m) that lie, for every thread, strictly
// inside the gap (N/3, N - N/3) of the 2/3 band limit of propagate_slow
// (stem3/stemlib.cpp:2815-2849): the band keeps |index| <= floor(N/3) on each
// axis, so these slots are zero in k-space after the propagator.
template <int N>
constexpr int gap_mask() {
  constexpr int E = Plan<N>::E, T = N / E, A = N / 3;
  int m = 0;
  for (int j = 0; j < E && j < 31; j++)
    if (T * j > A && T * j + T - 1 < N - A) m |= 1 << j;
  return m;
}

// Full length-N transform of the thread-distributed vector v (natural layout
// in and out).  slot: this transform's LDS region of lds_slot<N, SWZ>() float2.
// ZIN: slots known to be zero on input; NEED: slots needed on output.
template <int N, int DIR, bool SWZ = kSwz<N>, int ZIN = 0, int NEED = -1>
__device__ __forceinline__ void fft_wave(float2* v, float2* slot, const Twiddles<N>& tw, int t) {
  using P = Plan<N>;
  using W = Twiddles<N>;
  constexpr int S1 = P::R0;
  constexpr int S2 = P::R0 * P::R1;
  stockham_pass<N, P::R0, 1, DIR, true, false, SWZ, 1, ZIN>(v, slot, nullptr, t);
  stockham_pass<N, P::R1, S1, DIR, false, false, SWZ, W::B1>(v, slot, tw.w1, t);
  if constexpr (P::NP == 3) {
    stockham_pass<N, P::R2, S2, DIR, false, true, SWZ, W::B2, 0, NEED>(v, slot, tw.w2, t);
  } else {
    stockham_pass<N, P::R2, S2, DIR, false, false, SWZ, W::B2>(v, slot, tw.w2, t);
    stockham_pass<N, P::R3, S2 * P::R2, DIR, false, true, SWZ, W::B3, 0, NEED>(v, slot, tw.w3, t);
  }
}

}  // namespace qs
