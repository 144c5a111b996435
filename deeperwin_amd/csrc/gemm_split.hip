// FP32 GEMMs of the Laplacian pass's derivative channels on 16-bit MFMA with FP32 sums.
//
// Two forms.  BF16 parts: an FP32 operand is the exact sum of three BF16 numbers (x = h + m + l: h = bf16(x),
// m = bf16(x - h), l = x - h - m; 8 + 8 + 8 significant bits, m up to 2^-8 |x|, l up to 2^-17 |x|), so a product is the sum
// of nine BF16 products; three (m l and l m, up to 2^-25 |a b|, and l l) are left out.  FP16 parts: x = h + m with 11 + 11
// bits, m up to 2^-11 |x|, and a rest up to 2^-23 |x|; three products (m m, up to 2^-22 |a b|, left out).  It needs operands
// near the top of FP16's range, so a row block (one electron's channels) and each column of the weights are scaled by powers
// of two, and an element keeps those bits down to 2^-17 of its block's or column's largest (below that its absolute error is
// 2^-39 of the largest).  A single product is thus less exact than FP32's (whose products the FP32 MFMA does not round); sums
// are not: a 32-wide K slice rounds the accumulator six or three times, where the FP32 MFMA (16x16x4) rounds it at least
// eight times, and over 320 products of random operands that leaves 1.3e-7 (BF16) and 1.2e-7 (FP16) of the norm against
// 1.6e-7 for FP32.
// The 16-bit MFMA runs at 16 times the FP32 rate: 6 / 16 and 3 / 16 of the FP32 form's time.
//
// FP16 parts are taken where the largest magnitudes are known: the layer's kernel leaves the maxima of what it writes,
// and the columns of other kernels (pair features, the last slices) are looked at while they wait in registers.
// Layer 0 (K of a few features) and the mean product, bound by memory, use BF16 parts.
//
// Measured against 64 bits (E_loc of 48 to 2048 walkers, 4 to 60 electrons, both models): the same relative error as the
// FP32 form to a few per cent (5e-7 to 6e-5 of the norm, 9e-7 to 8e-4 for the median of unequilibrated walkers: set by the
// value channel), between the two 1e-7 to 2e-6 of the norm, a quarter of that error or less.
//
// Only derivative channels (tangents, Laplacian) come from here.  The value channel of the pass (the first row
// of an electron) keeps the FP32 MFMA of the value pass: log|psi|, the orbital matrices and their inverses
// amplify its rounding by the walker's conditioning, the derivative channels enter E_loc linearly.
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace dwmi {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

// ------------------------------------------------------------------------------------------------
// Operand parts
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {  // v_cvt_pk_bf16_f32 (nearest even)
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, v2bf));
}
__device__ __forceinline__ float lo_f(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_f(unsigned u) { return __uint_as_float(u & 0xFFFF0000u); }

// v * f, rounded: a part's rest is not fused with it.
__device__ __forceinline__ v4f scaled(v4f v, float f) {
#pragma clang fp contract(off)
  return v4f{v[0] * f, v[1] * f, v[2] * f, v[3] * f};
}

// Four floats -> the three parts of each, packed in 8 bytes per part.
__device__ __forceinline__ void split4(v4f x, uint2 (&p)[3]) {
  const unsigned h0 = pack_bf16(x[0], x[1]), h1 = pack_bf16(x[2], x[3]);
  const float r0 = x[0] - lo_f(h0), r1 = x[1] - hi_f(h0), r2 = x[2] - lo_f(h1), r3 = x[3] - hi_f(h1);
  const unsigned m0 = pack_bf16(r0, r1), m1 = pack_bf16(r2, r3);
  p[0] = uint2{h0, h1};
  p[1] = uint2{m0, m1};
  p[2] = uint2{pack_bf16(r0 - lo_f(m0), r1 - hi_f(m0)), pack_bf16(r2 - lo_f(m1), r3 - hi_f(m1))};
}

// Four floats -> two FP16 parts of each (x = h + m + rest, |rest| below 2^-23 of |x| for |x| >= 2^-2).
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split4h(v4f x, uint2 (&p)[2]) {
  const v2h h0 = __builtin_convertvector(v2f{x[0], x[1]}, v2h), h1 = __builtin_convertvector(v2f{x[2], x[3]}, v2h);
  const v2h m0 = __builtin_convertvector(v2f{x[0] - (float)h0[0], x[1] - (float)h0[1]}, v2h);
  const v2h m1 = __builtin_convertvector(v2f{x[2] - (float)h1[0], x[3] - (float)h1[1]}, v2h);
  p[0] = uint2{__builtin_bit_cast(unsigned, h0), __builtin_bit_cast(unsigned, h1)};
  p[1] = uint2{__builtin_bit_cast(unsigned, m0), __builtin_bit_cast(unsigned, m1)};
}

// Weights Bt [rows, ldb] (row = output column, K contiguous) in the order the MFMA lanes read them:
// P[((slice * ncb + cb) * 3 + part) * 64 + lane] = 8 BF16 of column 16 cb + lane % 16, k = 32 slice +
// 8 (lane / 16) + 0..7.  Columns at or past `cols` are zero.
__global__ __launch_bounds__(256) void k_split_pack(const float* __restrict__ Bt, int ldb, int cols, int ncb,
                                                    int slices, uint4* __restrict__ P) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= slices * ncb * 64) return;
  const int lane = t & 63, cb = (t >> 6) % ncb, sl = (t >> 6) / ncb;
  const int col = cb * 16 + (lane & 15), k = sl * 32 + (lane >> 4) * 8;
  v4f a = {0.f, 0.f, 0.f, 0.f}, b = a;
  if (col < cols) {
    a = *(const v4f*)(Bt + (long)col * ldb + k);
    b = *(const v4f*)(Bt + (long)col * ldb + k + 4);
  }
  uint2 pa[3], pb[3];
  split4(a, pa);
  split4(b, pb);
#pragma unroll
  for (int p = 0; p < 3; ++p)
    P[((long)(sl * ncb + cb) * 3 + p) * 64 + lane] = uint4{pa[p].x, pa[p].y, pb[p].x, pb[p].y};
}

size_t split_pack_bytes(int cols, int K) { return (size_t)(K / 32) * (dw_pad(cols, 256) / 16) * 3 * 64 * 16; }

void launch_split_pack(const float* Bt, int ldb, int cols, int K, void* out, hipStream_t s) {
  const int ncb = dw_pad(cols, 256) / 16, slices = K / 32;
  hipLaunchKernelGGL(k_split_pack, dim3((slices * ncb * 64 + 255) / 256), dim3(256), 0, s, Bt, ldb, cols, ncb, slices,
                     (uint4*)out);
}

// The same order with two FP16 parts of W times a power of two per output column: P16[((slice * ncb + cb) * 2 + part) * 64 +
// lane], then the columns' shifts (16 ncb of them).
__global__ __launch_bounds__(256) void k_split_pack16(const float* __restrict__ Bt, int ldb, int cols, int ncb,
                                                      int slices, uint4* __restrict__ P) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= slices * ncb * 64) return;
  const int lane = t & 63, cb = (t >> 6) % ncb, sl = (t >> 6) / ncb;
  const int col = cb * 16 + (lane & 15), k = sl * 32 + (lane >> 4) * 8;
  v4f a = {0.f, 0.f, 0.f, 0.f}, b = a;
  if (col < cols) {
    a = *(const v4f*)(Bt + (long)col * ldb + k);
    b = *(const v4f*)(Bt + (long)col * ldb + k + 4);
  }
  const float scale = ldexpf(1.f, ((const int*)(P + (long)slices * ncb * 128))[col]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    a[j] *= scale;
    b[j] *= scale;
  }
  uint2 pa[2], pb[2];
  split4h(a, pa);
  split4h(b, pb);
#pragma unroll
  for (int p = 0; p < 2; ++p)
    P[((long)(sl * ncb + cb) * 2 + p) * 64 + lane] = uint4{pa[p].x, pa[p].y, pb[p].x, pb[p].y};
}

size_t split_pack16_bytes(int cols, int K) {
  return (size_t)(K / 32) * (dw_pad(cols, 256) / 16) * 2 * 64 * 16 + (size_t)dw_pad(cols, 256) * sizeof(int);
}
int* split_pack16_shifts(void* P16, int cols, int K) {
  return (int*)((uint4*)P16 + (size_t)(K / 32) * (dw_pad(cols, 256) / 16) * 128);
}

void launch_split_pack16(const float* Bt, int ldb, int cols, int K, void* out, hipStream_t s) {
  const int ncb = dw_pad(cols, 256) / 16, slices = K / 32;
  hipLaunchKernelGGL(k_split_pack16, dim3((slices * ncb * 64 + 255) / 256), dim3(256), 0, s, Bt, ldb, cols, ncb, slices,
                     (uint4*)out);
}

// Power of two that brings a block of largest magnitude `m` under 2^15.  Bounded so that the units of the accumulators
// (this plus a weight column's shift of -19 .. 60, orbitals 74) and their inverse stay in range.
__device__ __forceinline__ int split_shift(float m) {
  const int e = (int)((__float_as_uint(m) >> 23) & 255u) - 127;
  return min(40, max(-100, 14 - e));
}

__device__ __forceinline__ int tile_of(int bid, int total) {
  // workgroups are dealt round-robin to 8 XCDs; each XCD gets a contiguous range of tiles
  const int per = (total + 7) / 8;
  return (bid & 7) * per + (bid >> 3);
}

// ------------------------------------------------------------------------------------------------
// Main loop of one 256-thread workgroup: acc = A[row0 .. row0 + 16 RB) B[:, 64 NQ columns], wave w owning
// the 16 NQ columns from block cb0.  A slices of 32 are split while they are staged into LDS (two buffers,
// one barrier per slice), in lane order (part, row block, lane), so every LDS access is 16 consecutive bytes
// per lane; a wave's B parts come from L2 straight into registers, one slice ahead.
// ------------------------------------------------------------------------------------------------
// One product of row block i with the NQ column blocks (parts PA of a, PB of b).
#define DW_SPLIT_MFMA(PA, PB) \
  _Pragma("unroll") for (int q = 0; q < NQ; ++q) acc[i][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16( \
      (v8bf)a[PA], (v8bf)b[q][PB], acc[i][q], 0, 0, 0);
#define DW_SPLIT_MFMA16(PA, PB) \
  _Pragma("unroll") for (int q = 0; q < NQ; ++q) acc[i][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16( \
      __builtin_bit_cast(v8h, a[PA]), __builtin_bit_cast(v8h, b[q][PB]), acc[i][q], 0, 0, 0);

template <int RB, int PARTS>
struct SplitLds {
  uint4 a[2][PARTS][RB][64];
};

// Weights of a split GEMM in lane order: three BF16 parts of W, or two FP16 parts of its scaled columns (and their shifts).
struct SplitB {
  const uint4* P;
  int ncb, slices;
  __device__ __forceinline__ int shift(int col) const { return ((const int*)(P + (long)slices * ncb * 128))[col]; }
};

// Unit u of a slice: row u / 128 * 16 + u % 16 (row block u / 128), quad of 4 k (u / 16) % 8.
template <int RB>
struct SplitUnits {
  static constexpr int AU = RB * 128, AIT = (AU + 255) / 256;
  const float* ap[AIT];
  __device__ __forceinline__ SplitUnits(const float* A, long row0, long rows, long lda) {
#pragma unroll
    for (int it = 0; it < AIT; ++it) {
      const int u = threadIdx.x + 256 * it;
      long gr = row0 + (u >> 7) * 16 + (u & 15);
      if (gr > rows - 1) gr = rows - 1;
      ap[it] = A + gr * lda + ((u >> 4) & 7) * 4;
    }
  }
  __device__ __forceinline__ bool in(int it) const { return AU % 256 == 0 || (int)threadIdx.x + 256 * it < AU; }
  __device__ __forceinline__ void load(int s, v4f (&ra)[AIT]) const {
#pragma unroll
    for (int it = 0; it < AIT; ++it)
      if (in(it)) ra[it] = *(const v4f*)(ap[it] + s * 32);
  }
  static __device__ __forceinline__ int block(int it) { return ((int)threadIdx.x + 256 * it) >> 7; }
};

template <int NQ, int PARTS>
__device__ __forceinline__ void split_bload(const SplitB& W, int s, int cb0, v8s (&d)[NQ][PARTS]) {
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int p = 0; p < PARTS; ++p)
      d[q][p] = *(const v8s*)&W.P[((long)(s * W.ncb + cb0 + q) * PARTS + p) * 64 + (threadIdx.x & 63)];
}

// BF16 parts: any K.
template <int RB, int NQ>
__device__ __forceinline__ void split_main(const SplitUnits<RB>& U, const SplitB& W, int cb0, SplitLds<RB, 3>& lds,
                                           v4f (&acc)[RB][NQ]) {
  constexpr int AIT = SplitUnits<RB>::AIT;
  const int tid = threadIdx.x, lane = tid & 63, slices = W.slices;
  v4f ra[AIT];
  auto sstore = [&](int buf) {
#pragma unroll
    for (int it = 0; it < AIT; ++it)
      if (U.in(it)) {
        const int u = tid + 256 * it, quad = (u >> 4) & 7;
        uint2 p[3];
        split4(ra[it], p);
#pragma unroll
        for (int k = 0; k < 3; ++k) *((uint2*)&lds.a[buf][k][u >> 7][(quad >> 1) * 16 + (u & 15)] + (quad & 1)) = p[k];
      }
  };
  v8s b[NQ][3], bn[NQ][3];
  auto slice = [&](int s, v8s (&b)[NQ][3], v8s (&bn)[NQ][3]) {
    const int buf = s & 1;
    __syncthreads();  // slice s is in lds.a[buf]; every read of lds.a[buf ^ 1] (slice s - 1) is done
    if (s + 1 < slices) split_bload<NQ, 3>(W, s + 1, cb0, bn);
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      v8s a[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p] = *(const v8s*)&lds.a[buf][p][i][lane];
      DW_SPLIT_MFMA(2, 0)
      DW_SPLIT_MFMA(0, 2)
      DW_SPLIT_MFMA(1, 1)
      DW_SPLIT_MFMA(1, 0)
      DW_SPLIT_MFMA(0, 1)
      DW_SPLIT_MFMA(0, 0)
      if (i == RB / 2 && s + 1 < slices) {  // the next slice, loaded a slice ago
        sstore(buf ^ 1);
        if (s + 2 < slices) U.load(s + 2, ra);
      }
    }
  };
  U.load(0, ra);
  split_bload<NQ, 3>(W, 0, cb0, b);
  sstore(0);
  if (slices > 1) U.load(1, ra);
  int s = 0;
  for (; s + 1 < slices; s += 2) {
    slice(s, b, bn);
    slice(s + 1, bn, b);
  }
  if (s < slices) slice(s, b, bn);
}

// FP16 parts of rows scaled by sc[] (a power of two per row block): an even number of slices, taken in the order
// slices - tail, .., slices - 1, 0, 1, ..; the first two are already in ra0 and ra1.  Rows are loaded two slices ahead.
template <int RB, int NQ>
__device__ __forceinline__ void split_main16(const SplitUnits<RB>& U, const SplitB& W, int tail,
                                             v4f (&ra0)[SplitUnits<RB>::AIT], v4f (&ra1)[SplitUnits<RB>::AIT],
                                             const float (&sc)[SplitUnits<RB>::AIT], int cb0, SplitLds<RB, 2>& lds,
                                             v4f (&acc)[RB][NQ]) {
  constexpr int AIT = SplitUnits<RB>::AIT;
  const int tid = threadIdx.x, lane = tid & 63, slices = W.slices;
  auto at = [&](int t) { return t < tail ? slices - tail + t : t - tail; };
  auto sstore = [&](int buf, v4f (&ra)[AIT]) {
#pragma unroll
    for (int it = 0; it < AIT; ++it)
      if (U.in(it)) {
        const int u = tid + 256 * it, quad = (u >> 4) & 7;
        v4f x = ra[it];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] *= sc[it];
        uint2 p[2];
        split4h(x, p);
#pragma unroll
        for (int k = 0; k < 2; ++k) *((uint2*)&lds.a[buf][k][u >> 7][(quad >> 1) * 16 + (u & 15)] + (quad & 1)) = p[k];
      }
  };
  v8s b[NQ][2], bn[NQ][2];
  auto slice = [&](int t, v8s (&b)[NQ][2], v8s (&bn)[NQ][2], v4f (&ra)[AIT]) {
    const int buf = t & 1;
    __syncthreads();  // slice t is in lds.a[buf]; every read of lds.a[buf ^ 1] (slice t - 1) is done
    if (t + 1 < slices) split_bload<NQ, 2>(W, at(t + 1), cb0, bn);
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      v8s a[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) a[p] = *(const v8s*)&lds.a[buf][p][i][lane];
      DW_SPLIT_MFMA16(1, 0)
      DW_SPLIT_MFMA16(0, 1)
      DW_SPLIT_MFMA16(0, 0)
      if (i == RB / 2 && t + 1 < slices) {  // slice t + 1, loaded two slices ago
        sstore(buf ^ 1, ra);
        if (t + 3 < slices) U.load(at(t + 3), ra);
      }
    }
  };
  split_bload<NQ, 2>(W, at(0), cb0, b);
  sstore(0, ra0);
  if (slices > 2) U.load(at(2), ra0);
  for (int t = 0; t < slices; t += 2) {
    slice(t, b, bn, ra1);
    slice(t + 1, bn, b, ra0);
  }
}

// Scales of a tile's row blocks (16 rows of one electron each, rbe blocks an electron): from the per-wave maxima that
// the producer of A left (np per electron, ms apart) and, for the `tail` slices it did not write, from the rows
// themselves (the first slices read; C channels an electron).  sM: RB words; eA gets the shifts; returns with sc[] set and the LDS words
// readable by all.
template <int RB>
__device__ __forceinline__ void tile_scales(const SplitUnits<RB>& U, const float* __restrict__ amax, int np, int ms, int tail,
                                            const v4f (&ra0)[SplitUnits<RB>::AIT],
                                            const v4f (&ra1)[SplitUnits<RB>::AIT], long block0, long blocks, int rbe, int C,
                                            unsigned* sM, int* eA, float (&sc)[SplitUnits<RB>::AIT]) {
  constexpr int AIT = SplitUnits<RB>::AIT;
  const int tid = threadIdx.x;
  if (tid < RB) {
    const long el = min(block0 + tid, blocks - 1) / rbe;
    float m = 0.f;
    for (int p = 0; p < np; ++p) m = fmaxf(m, amax[el * ms + p]);
    sM[tid] = __float_as_uint(m);
  }
  __syncthreads();
  if (tail > 0) {  // uniform
#pragma unroll
    for (int it = 0; it < AIT; ++it) {
      float m = 0.f;
      const int ch = (int)((block0 + U.block(it)) % rbe) * 16 + (tid & 15);
      if (U.in(it) && ch > 0 && ch < C) {  // derivative channels only: the rows of padding channels hold anything
#pragma unroll
        for (int j = 0; j < 4; ++j) m = fmaxf(m, fabsf(ra0[it][j]));
        if (tail > 1) {
#pragma unroll
          for (int j = 0; j < 4; ++j) m = fmaxf(m, fabsf(ra1[it][j]));
        }
      }
      // a wave's 64 units of one step lie in one row block; blocks of an electron share the scale
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
      if ((tid & 63) == 0 && U.in(it)) {
        const int e0 = (int)((block0 + U.block(it)) / rbe * rbe - block0);
        for (int k = max(e0, 0); k < min(e0 + rbe, RB); ++k) atomicMax(&sM[k], __float_as_uint(m));
      }
    }
    __syncthreads();
  }
  if (tid < RB) eA[tid] = split_shift(__uint_as_float(sM[tid]));
#pragma unroll
  for (int it = 0; it < AIT; ++it)
    sc[it] = ldexpf(1.f, split_shift(__uint_as_float(sM[min(U.block(it), RB - 1)])));
}

// ------------------------------------------------------------------------------------------------
// C[M, N] = A[M, K] B (no epilogue): the orbital GEMMs of the Laplacian pass.  688,128 x 256 x 224: 783 us with
// FP32 MFMA on 128-row tiles, 480 us with BF16 parts, 349 us here with one scale for all weights; a scale per column takes
// 1 to 2 % more (365 -> 371 us there, 1,064,960 x 256 x 416 1,090 -> 1,117; with its loads before the main loop 1,181).
// ------------------------------------------------------------------------------------------------
template <int RB, int NQ>
__global__ __launch_bounds__(256, 2) void k_split_gemm(const float* __restrict__ A, int lda, SplitB W,
                                                       const float* __restrict__ amax, int np, int ms, int rbe,
                                                       float* __restrict__ Cm, int ldc, int M, int N, int tilesN,
                                                       int tilesTotal) {
  constexpr int AIT = SplitUnits<RB>::AIT;
  __shared__ SplitLds<RB, 2> lds;
  __shared__ unsigned sM[RB];
  __shared__ int eA[RB];
  const int tile = tile_of(blockIdx.x, tilesTotal);
  if (tile >= tilesTotal) return;  // uniform over the workgroup, before any barrier
  const long row0 = (long)(tile / tilesN) * (16 * RB);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int cb0 = (tile % tilesN) * (4 * NQ) + wv * NQ;
  const SplitUnits<RB> U(A, row0, M, lda);
  v4f ra0[AIT], ra1[AIT];
  float sc[AIT];
  U.load(0, ra0);
  U.load(1, ra1);
  tile_scales<RB>(U, amax, np, ms, 0, ra0, ra1, row0 >> 4, M >> 4, rbe, 0, sM, eA, sc);
  v4f acc[RB][NQ];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
  split_main16<RB, NQ>(U, W, 0, ra0, ra1, sc, cb0, lds, acc);
  float wi[NQ];  // 2^-shift of this lane's columns
#pragma unroll
  for (int q = 0; q < NQ; ++q) wi[q] = ldexpf(1.f, -W.shift((cb0 + q) * 16 + (lane & 15)));
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const float ai = ldexpf(1.f, -eA[i]);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int c = (cb0 + q) * 16 + (lane & 15);
      const float inv = ai * wi[q];
      if (c < N) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const long r = row0 + i * 16 + 4 * (lane >> 4) + j;
          if (r < M) Cm[r * ldc + c] = acc[i][q][j] * inv;
        }
      }
    }
  }
}

void split_gemm(const float* A, int lda, const void* P16, const float* amax, int np, int ms, int rbe, float* C,
                int ldc, int M, int N, int K, int tile, hipStream_t s) {
  if (M <= 0 || N <= 0) return;
  const SplitB W{(const uint4*)P16, dw_pad(N, 256) / 16, K / 32};
  const long big = ((long)(M + 95) / 96) * ((N + 255) / 256);
  if (tile < 0 ? big >= 512 : tile > 0) {
    const int tilesN = (N + 255) / 256, total = (M + 95) / 96 * tilesN;
    hipLaunchKernelGGL((k_split_gemm<6, 4>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, A, lda, W, amax, np, ms, rbe, C,
                       ldc, M, N, tilesN, total);
  } else {
    const int tilesN = (N + 127) / 128, total = (M + 47) / 48 * tilesN;
    hipLaunchKernelGGL((k_split_gemm<3, 2>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, A, lda, W, amax, np, ms, rbe, C,
                       ldc, M, N, tilesN, total);
  }
}

// ------------------------------------------------------------------------------------------------
// 1-el embedding GEMM of the Laplacian pass with the tanh forward-Laplacian rule.  A workgroup owns E whole
// electrons (RBE row blocks of 16 channels each) and 64 NQ columns; `out` already holds the value channel y_0
// (row 0 of each electron).  Per column: z_ch = (X W)_ch + V[walker, ch], y_k = t' z_k (k = 1 .. 3n),
// y_lap = t' z_lap + t'' sum_k z_k^2.  The rule runs on the accumulators: a column's
// channels lie in the four 16-lane groups (4 consecutive channels each), so the sum over the tangents is two
// lane exchanges and the stores are 64-byte row segments, four rows at a time.  Padding channels are left
// unwritten: rows are independent and nothing reads those of a padding channel.
//
// 1,376,256 rows (2048 walkers of 14 electrons) x 320 x 256: 2000 us with FP32 MFMA, 1240 us with BF16 parts, 980 us
// with FP16 parts and rows loaded two slices ahead (1050 us with one slice).  Reading X and writing the output take 610
// us at the card's rates (6.4 TB/s reads alone, 4.1 TB/s writes alone); matrix cores are busy for a third of the cycles
// (with BF16 parts for half of them, at 2.0 GHz: the card lowers its clock from 2.4).  26 electrons (1.7 M rows): 3600,
// 1960, 1540 us; 42 electrons (1.0 M rows): 1930, 990, 905 us.
// ------------------------------------------------------------------------------------------------
template <int RBE, int E, int NQ, bool HALF>
__global__ __launch_bounds__(256, 2) void k_split_lap(const float* __restrict__ X, int ldx, SplitB W,
                                                      const float* __restrict__ amax, int np, int tail,
                                                      const float* __restrict__ V, int ldv, float* __restrict__ out,
                                                      int ldo, float* __restrict__ omax, int permute, Shape sh,
                                                      int tilesN, int tilesTotal) {
  constexpr int RB = RBE * E, AIT = SplitUnits<RB>::AIT;
  __shared__ SplitLds<RB, HALF ? 2 : 3> lds;
  __shared__ unsigned sM[HALF ? RB : 1];
  __shared__ int eA[HALF ? RB : 1];
  const int tile = tile_of(blockIdx.x, tilesTotal);
  if (tile >= tilesTotal) return;  // uniform over the workgroup, before any barrier
  const int n = sh.n, C = sh.C, Cp = sh.Cp;
  const long n_el = (long)sh.B * n;
  const long g0 = (long)(tile / tilesN) * E;  // first electron
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g4 = lane >> 4;
  const int cb0 = (tile % tilesN) * (4 * NQ) + wv * NQ;
  const int dn = n - sh.u;
  const int col = cb0 * 16 + (lane & 15);
  const SplitUnits<RB> U(X, g0 * Cp, n_el * Cp, ldx);
  v4f ra0[HALF ? AIT : 1], ra1[HALF ? AIT : 1];
  float sc[HALF ? AIT : 1];
  int shifts[NQ];  // of this lane's columns
  if constexpr (HALF) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) shifts[q] = W.shift(col + 16 * q);
    const int first = tail > 0 ? W.slices - tail : 0;
    U.load(first, ra0);
    U.load(tail == 1 ? 0 : first + 1, ra1);
  }
  // the accumulators start from V (in their units): its loads run beside the first slices'
  v4f acc[RB][NQ];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const long g = min(g0 + e, n_el - 1);
    const float* Vp = V + (g / n * Cp + 4 * g4) * (long)ldv + col;
#pragma unroll
    for (int kb = 0; kb < RBE; ++kb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[e * RBE + kb][q][j] = Vp[(long)(kb * 16 + j) * ldv + 16 * q];
  }
  if constexpr (HALF) {
    tile_scales<RB>(U, amax, np, sh.W1 >> 5, tail, ra0, ra1, g0 * RBE, n_el * RBE, RBE, C, sM, eA, sc);
    __syncthreads();  // eA
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const float unit = ldexpf(1.f, eA[i]);
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const float u = unit * ldexpf(1.f, shifts[q]);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][q][j] *= u;
      }
    }
    split_main16<RB, NQ>(U, W, tail, ra0, ra1, sc, cb0, lds, acc);
  } else {
    split_main<RB, NQ>(U, W, cb0, lds, acc);
  }

#pragma unroll
  for (int e = 0; e < E; ++e) {
    const long g = g0 + e;
    if (g >= n_el) break;  // uniform
    const long b = g / n;
    const int i = (int)(g - b * n);
    long ob = g * Cp;
    if (permute) ob = (i < sh.u) ? (b * sh.u + i) * Cp : (long)sh.B * sh.u * Cp + (b * dn + (i - sh.u)) * Cp;
    float* op = out + (ob + 4 * g4) * ldo + col;
    const float* vp = out + ob * ldo + col;
    float inv[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      inv[q] = HALF ? ldexpf(1.f, -eA[HALF ? e * RBE : 0]) * ldexpf(1.f, -shifts[q]) : 1.f;
    float d1[NQ], d2[NQ], S[NQ], zl[NQ], mx = 0.f;  // mx: largest |y| of the derivative channels
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const float th = vp[16 * q];
      d1[q] = 1.f - th * th;
      d2[q] = -2.f * th * d1[q];
      S[q] = 0.f;
      zl[q] = 0.f;
    }
#pragma unroll
    for (int kb = 0; kb < RBE; ++kb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int ch = kb * 16 + 4 * g4 + j;
        const bool tan = ch >= 1 && ch < C - 1;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const float z = acc[e * RBE + kb][q][j] * inv[q];
          S[q] += tan ? z * z : 0.f;
          if (ch == C - 1) zl[q] = z;
          if (tan) {
            const float y = d1[q] * z;
            mx = fmaxf(mx, fabsf(y));
            op[(long)(kb * 16 + j) * ldo + 16 * q] = y;
          }
        }
      }
    }
    const int cl = C - 1 - (RBE - 1) * 16;  // the Laplacian's row in the last block
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      float s = S[q] + __shfl_xor(S[q], 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (g4 == (cl >> 2)) {
        const float y = d1[q] * zl[q] + d2[q] * s;
        mx = fmaxf(mx, fabsf(y));
        out[(ob + C - 1) * ldo + col + 16 * q] = y;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) omax[ob / Cp * (sh.W1 >> 5) + cb0 / NQ] = mx;
  }
}

int split_lap(const float* X, int ldx, const void* P, int K, const float* amax, int np, int tail,
              const float* V, int ldv, float* out, int ldo, float* omax, int permute, const Shape& sh, int E_max,
              int cols, hipStream_t s) {
  const int RBE = sh.Cp / 16;
  const SplitB W{(const uint4*)P, dw_pad(sh.W1, 256) / 16, K / 32};
  const long n_el = (long)sh.B * sh.n;
#define DW_SPLIT_LAP(R, EE, Q)                                                                                        \
  do {                                                                                                                \
    const int tilesN = sh.W1 / (64 * Q);                                                                              \
    const long total = (n_el + EE - 1) / EE * tilesN;                                                                 \
    const dim3 grid((unsigned)((total + 7) / 8 * 8));                                                                 \
    if (amax)                                                                                                         \
      hipLaunchKernelGGL((k_split_lap<R, EE, Q, true>), grid, dim3(256), 0, s, X, ldx, W, amax, np, tail, V, ldv, out, \
                         ldo, omax, permute, sh, tilesN, (int)total);                                                 \
    else                                                                                                              \
      hipLaunchKernelGGL((k_split_lap<R, EE, Q, false>), grid, dim3(256), 0, s, X, ldx, W, amax, np, tail, V, ldv,     \
                         out, ldo, omax, permute, sh, tilesN, (int)total);                                            \
    return sh.W1 / (16 * Q);                                                                                          \
  } while (0)
  // full tiles (96 rows or one electron, 256 columns: A read and split once) where they give two workgroups to
  // every CU; otherwise fewer electrons and 128 columns, which fill the chip from half as many rows.  More than
  // 96 rows per electron take 128 columns so that the accumulators stay in registers.  The choice does not change
  // results.
  const int EF = RBE <= 6 ? 6 / RBE : 1;
  bool big = sh.W1 % 256 == 0 && RBE <= 6 && (n_el + EF - 1) / EF * (sh.W1 / 256) >= 512;
  if (cols == 128 || (E_max > 0 && E_max < EF)) big = false;
  if (cols == 256 && sh.W1 % 256 == 0 && RBE <= 6 && (E_max <= 0 || E_max >= EF)) big = true;
  switch (RBE * 2 + (big ? 1 : 0)) {
    case 3: DW_SPLIT_LAP(1, 6, 4);
    case 5: DW_SPLIT_LAP(2, 3, 4);
    case 7: DW_SPLIT_LAP(3, 2, 4);
    case 9: DW_SPLIT_LAP(4, 1, 4);
    case 11: DW_SPLIT_LAP(5, 1, 4);
    case 13: DW_SPLIT_LAP(6, 1, 4);
    case 2: DW_SPLIT_LAP(1, 2, 2);
    case 4: DW_SPLIT_LAP(2, 1, 2);
    case 6: DW_SPLIT_LAP(3, 1, 2);
    case 8: DW_SPLIT_LAP(4, 1, 2);
    case 10: DW_SPLIT_LAP(5, 1, 2);
    case 12: DW_SPLIT_LAP(6, 1, 2);
    case 14: DW_SPLIT_LAP(7, 1, 2);
    case 16: DW_SPLIT_LAP(8, 1, 2);
    case 18: DW_SPLIT_LAP(9, 1, 2);
    case 20: DW_SPLIT_LAP(10, 1, 2);
    case 22: DW_SPLIT_LAP(11, 1, 2);
    case 24: DW_SPLIT_LAP(12, 1, 2);
    default: return 0;
  }
#undef DW_SPLIT_LAP
}

// ------------------------------------------------------------------------------------------------
// Per-walker term of a 1-el layer for the derivative channels, spin means fused in:
//   V[r, o] = sum_k MU[r, k] Wmu[o, k],  r = b Cp + ch,
//   MU[r, k] = mean over the electrons of spin s(k) of X[(b n + i) Cp + ch, k - s Kh]   (electrons in order, FP32).
// A workgroup forms the means of 48 rows x 128 k at a time and splits them straight into LDS (37 KB: four workgroups
// per CU, whose load and MFMA phases overlap); the weights' parts come from L2.  Bound by the read of X's h columns
// (1.41 GB for 2048 walkers of 14 electrons: 364 us = 3.9 TB/s against 471 us with FP32 MFMA; 26 electrons, 1024
// walkers: 575 -> 461 us).  Smaller batches form their means in k_spin_mean (split_mean says where).
//
// NP = 2 is the BF16x3 form: the first two parts and three products, every row (the value channel and its bias too), 64
// rows.  Its sums are k_gemm_bf16's (v_mfma_f32_32x32x16_bf16 over 16 k at a time, low x high, high x low, high x high), so
// results are bit-equal to the separate kernels (k_spin_mean and that GEMM), which small batches keep (launch_mean).
// ------------------------------------------------------------------------------------------------
template <int NP>
__global__ __launch_bounds__(256, NP == 2 ? 4 : 1) void k_split_mean(const float* __restrict__ X, int Kx, int Kh,
                                                    const uint4* __restrict__ P, int ncb, int Km,
                                                    const float* __restrict__ bias, float* __restrict__ V, int ldv,
                                                    Shape sh, int tilesN, int total) {
  constexpr int RB = NP == 2 ? 4 : 3, CS = 4, NQ = 4;  // row blocks, 32-wide slices per chunk, 16-column blocks of a wave
  __shared__ uint4 lds[CS][NP][RB][64];
  const int tile = tile_of(blockIdx.x, total);
  if (tile >= total) return;  // uniform over the workgroup, before any barrier
  const long rows = (long)sh.B * sh.Cp, r0 = (long)(tile / tilesN) * (16 * RB);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int cb0 = (tile % tilesN) * (4 * NQ) + wv * NQ;
  const int n = sh.n, u = sh.u, Cp = sh.Cp;
  const long xstride = (long)Cp * Kx;  // one electron further
  v4f acc[NP == 3 ? RB : 1][NQ];
  v16f acc2[NP == 2 ? 2 : 1][NP == 2 ? 2 : 1];  // 32 x 32 blocks
  if constexpr (NP == 3) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc2[i][q][j] = 0.f;
  }
  for (int kc = 0; kc < Km; kc += 32 * CS) {
    const int ns = min(CS, (Km - kc) >> 5);
    __syncthreads();  // the previous chunk's reads are done
    // consecutive lanes take consecutive quads of a row (coalesced); 4 quads a slice-row group
    auto put = [&](int rr, int qd, v4f v, float inv) {
      uint2 p[3];
      split4(scaled(v, inv), p);
      const int quad = qd & 7;
#pragma unroll
      for (int m = 0; m < NP; ++m)
        *((uint2*)&lds[qd >> 3][m][rr >> 4][(quad >> 1) * 16 + (rr & 15)] + (quad & 1)) = p[m];
    };
    const int units = 16 * RB * 8 * ns;
    for (int t = tid; t < units; t += 256) {
      const int rr = t / (8 * ns), qd = t - rr * (8 * ns);
      const long r = r0 + rr;
      const int k = kc + 4 * qd;
      v4f v = {0.f, 0.f, 0.f, 0.f};
      float inv = 0.f;
      if (r < rows && k < 2 * Kh) {
        const long b = div_idx(r, Cp);
        const int ch = (int)(r - b * Cp);
        const int s = k >= Kh ? 1 : 0;
        const int i0 = s ? u : 0, i1 = s ? n : u;
        const float* xp = X + ((b * n + i0) * Cp + ch) * (long)Kx + (k - s * Kh);
#pragma unroll 8
        for (int i = i0; i < i1; ++i, xp += xstride) {
          const v4f x = *(const v4f*)xp;
          v[0] += x[0];
          v[1] += x[1];
          v[2] += x[2];
          v[3] += x[3];
        }
        inv = 1.f / (float)(i1 - i0);
      }
      put(rr, qd, v, inv);
    }
    __syncthreads();
    for (int s = 0; s < ns; ++s) {
      if constexpr (NP == 3) {
        v8s b[NQ][NP];
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
          for (int m = 0; m < NP; ++m)
            b[q][m] = *(const v8s*)&P[((long)(((kc >> 5) + s) * ncb + cb0 + q) * 3 + m) * 64 + lane];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          v8s a[NP];
#pragma unroll
          for (int m = 0; m < NP; ++m) a[m] = *(const v8s*)&lds[s][m][i][lane];
          DW_SPLIT_MFMA(2, 0)
          DW_SPLIT_MFMA(0, 2)
          DW_SPLIT_MFMA(1, 1)
          DW_SPLIT_MFMA(1, 0)
          DW_SPLIT_MFMA(0, 1)
          DW_SPLIT_MFMA(0, 0)
        }
      } else {
        // lane l of a 32 x 32 x 16 block: row or column l % 32 (of two 16-blocks), k = 16 h + 8 (l / 32) + 0..7
        const int blk = (lane >> 4) & 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int at = (lane & 15) + 16 * (2 * h + (lane >> 5));
          v8s a[2][2], b[2][2];
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
              a[q][m] = *(const v8s*)&lds[s][m][2 * q + blk][at];
              b[q][m] = *(const v8s*)&P[((long)(((kc >> 5) + s) * ncb + cb0 + 2 * q + blk) * 3 + m) * 64 + at];
            }
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              acc2[i][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16((v8bf)a[i][1], (v8bf)b[q][0], acc2[i][q], 0, 0, 0);
              acc2[i][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16((v8bf)a[i][0], (v8bf)b[q][1], acc2[i][q], 0, 0, 0);
              acc2[i][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16((v8bf)a[i][0], (v8bf)b[q][0], acc2[i][q], 0, 0, 0);
            }
        }
      }
    }
  }
  if constexpr (NP == 3) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const long r = r0 + i * 16 + 4 * (lane >> 4) + j;
          if (r < rows) V[r * ldv + (cb0 + q) * 16 + (lane & 15)] = acc[i][q][j];
        }
  } else {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = cb0 * 16 + 32 * q + (lane & 31);
      const float bc = bias[c];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const long r = r0 + 32 * i + 8 * (j >> 2) + 4 * (lane >> 5) + (j & 3);
          if (r < rows) {
            float v = acc2[i][q][j];
            if ((unsigned)r % (unsigned)Cp == 0) v += bc;
            V[r * ldv + c] = v;
          }
        }
    }
  }
}

// The product alone, from means that k_spin_mean has formed: C[M, 64 NQ tilesN columns] = A[M, K] B in BF16 parts, the sums of
// k_split_mean.
template <int RB, int NQ>
__global__ __launch_bounds__(256) void k_split_gemm_mu(const float* __restrict__ A, int lda, SplitB W, float* __restrict__ C,
                                                       int ldc, int M, int tilesN, int total) {
  __shared__ SplitLds<RB, 3> lds;
  const int tile = tile_of(blockIdx.x, total);
  if (tile >= total) return;  // uniform over the workgroup, before any barrier
  const long row0 = (long)(tile / tilesN) * (16 * RB);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int cb0 = (tile % tilesN) * (4 * NQ) + wv * NQ;
  const SplitUnits<RB> U(A, row0, M, lda);
  v4f acc[RB][NQ];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[i][q] = v4f{0.f, 0.f, 0.f, 0.f};
  split_main<RB, NQ>(U, W, cb0, lds, acc);
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const long r = row0 + i * 16 + 4 * (lane >> 4) + j;
        if (r < M) C[r * ldc + (cb0 + q) * 16 + (lane & 15)] = acc[i][q][j];
      }
}

template <int RB, int NQ>
static void mu_launch(const float* MU, const void* P, int Km, float* V, int ldv, const Shape& sh, hipStream_t s) {
  const SplitB W{(const uint4*)P, dw_pad(sh.W1, 256) / 16, Km / 32};
  const int M = sh.B * sh.Cp, tilesN = sh.W1 / (64 * NQ), total = (M + 16 * RB - 1) / (16 * RB) * tilesN;
  hipLaunchKernelGGL((k_split_gemm_mu<RB, NQ>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, MU, Km, W, V, ldv, M, tilesN,
                     total);
}

// The smallest tiles whose workgroups come to about four per CU: 16 or 32 rows x 64 columns, then 48 or 96 x 128.
void split_mean_product(const float* MU, int Km, const void* P, float* V, int ldv, const Shape& sh, hipStream_t s) {
  const long M = (long)sh.B * sh.Cp;
  if ((M + 15) / 16 * (sh.W1 / 64) <= 1024)
    mu_launch<1, 1>(MU, P, Km, V, ldv, sh, s);
  else if ((M + 31) / 32 * (sh.W1 / 64) <= 1024)
    mu_launch<2, 1>(MU, P, Km, V, ldv, sh, s);
  else if ((M + 47) / 48 * (sh.W1 / 128) <= 768)
    mu_launch<3, 2>(MU, P, Km, V, ldv, sh, s);
  else
    mu_launch<6, 2>(MU, P, Km, V, ldv, sh, s);
}

// 256 columns a workgroup (X read once) where that gives two workgroups to every CU; below that its few workgroups form
// their means one after another, and two kernels win.  E_loc fused / apart, us: 14 electrons 473 / 317 (10 walkers), 765 / 619
// (125), 2,096 / 1,780 (500), 3,297 / 3,372 (1,000: fused); 4 electrons 291 / 259 (93), 1,338 / 1,395 (3,000: fused); 42
// electrons 1,160 / 994 (11); width 512, 14 electrons 877 / 542 (10), 4,182 / 4,118 (500: fused); other widths have 64-column
// workgroups only (width 384, 14 electrons, 500 walkers 4,143 / 3,320).
bool split_mean(const float* X, int Kx, int Kh, const void* P, int Km, float* V, int ldv, const Shape& sh, hipStream_t s) {
  const long tilesM = ((long)sh.B * sh.Cp + 47) / 48;
  if (sh.W1 % 256 != 0 || tilesM * (sh.W1 / 256) < 512) return false;
  const int tilesN = sh.W1 / 256, total = (int)(tilesM * tilesN);
  hipLaunchKernelGGL((k_split_mean<3>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, X, Kx, Kh, (const uint4*)P,
                     dw_pad(sh.W1, 256) / 16, Km, (const float*)nullptr, V, ldv, sh, tilesN, total);
  return true;
}

// From 600 tiles of 64 rows up the fused kernel keeps every CU busy; below, its few workgroups form their means one
// after another and the two separate kernels win.  E_loc, separate / fused: 14 electrons 510 / 702 us (85 walkers, 64
// tiles), 1,939 / 2,052 (583, 438), 2,794 / 2,766 (833, 625), 3,306 / 3,236 (1,000, 750), 4,384 / 4,225 (1,365, 1,024); 8
// electrons 1,184 / 1,262 (438 tiles), 1,739 / 1,705 (625).  From 20 electrons (longer sums to form a mean, which the fused
// kernel does not store) from 400 tiles: 20 electrons 2,622 / 2,595 (375), 3,504 / 3,436 (512); 26 electrons 1,287 / 1,460
// (128), 3,813 / 3,779 (438), 5,350 / 5,189 (625); 42 electrons 4,000 / 3,999 (256), 7,476 / 7,366 (512).
bool mean_bf16x3(const float* X, int Kx, int Kh, const void* P, int Km, const float* bias, float* V, int ldv, const Shape& sh,
                 hipStream_t s) {
  const long tilesM = ((long)sh.B * sh.Cp + 63) / 64;
  if (sh.W1 % 256 != 0 || tilesM * (sh.W1 / 256) < (sh.n >= 20 ? 400 : 600)) return false;
  const int tilesN = sh.W1 / 256, total = (int)(tilesM * tilesN);
  hipLaunchKernelGGL((k_split_mean<2>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, X, Kx, Kh, (const uint4*)P,
                     dw_pad(sh.W1, 256) / 16, Km, bias, V, ldv, sh, tilesN, total);
  return true;
}

}  // namespace dwmi
