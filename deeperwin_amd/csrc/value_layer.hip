// One launch per 1-el layer of the value channel (FP32): spin means, their product with the mean blocks of W,
// the per-electron GEMM, V, tanh and the spin-major order of the last layer; and one launch for both orbital
// GEMMs.  The rows of whole walkers stay in LDS, so the means need no launch and no second read; the weights
// come from L2 straight into registers, several slices ahead, so the main loop has no barrier.
//
// Every sum runs in the order of the separate kernels (k_spin_mean; k_gemm_f32's 16-wide K slices in order, MFMA
// step s of lane group g taking k = 4 g + s; the K parts of the mean product added in order), so results are
// bit-equal to them.
//
// Small batches were bound by latency: three launches a layer, 20 short K slices with two barriers each and a load
// to wait for.  256 LiH walkers (1,024 rows x 320 x 256): 30 us a layer in three launches, 10 us here; both orbital
// GEMMs 17 us in two launches, 4.2 us in one.  Larger batches take all layers in one launch, whole walkers and all
// columns per workgroup (k_value_net below).
#include "common.h"
#include "kernels.h"
#include <algorithm>

namespace dwmi {

// Weights in the order the MFMA lanes read them: P[(cb * S + slice) * 64 + lane] = column 16 cb + lane % 16,
// k = 16 slice + 4 (lane / 16) + 0..3, so a wave reads one contiguous run (rows of Bt, 2 KB apart in the mean
// product, would all come from one or two L2 channels).  Columns at or past `cols` are zero.
__global__ __launch_bounds__(256) void k_lane_pack(const float* __restrict__ Bt, int ldb, int cols, int ncb, int S,
                                                   v4f* __restrict__ P) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= ncb * S * 64) return;
  const int lane = t & 63, sl = (t >> 6) % S, cb = (t >> 6) / S;
  const int col = cb * 16 + (lane & 15);
  v4f v = {0.f, 0.f, 0.f, 0.f};
  if (col < cols) v = *(const v4f*)(Bt + (long)col * ldb + sl * 16 + (lane >> 4) * 4);
  P[t] = v;
}

size_t lane_pack_bytes(int cols, int K) { return (size_t)dw_pad(cols, 64) * K * 4; }

void launch_lane_pack(const float* Bt, int ldb, int cols, int K, void* out, hipStream_t s) {
  const int ncb = dw_pad(cols, 64) / 16, S = K / 16;
  hipLaunchKernelGGL(k_lane_pack, dim3((ncb * S * 64 + 255) / 256), dim3(256), 0, s, Bt, ldb, cols, ncb, S, (v4f*)out);
}

constexpr int MAXS = 20;  // 16-wide K slices of the per-electron and orbital GEMMs

// Rows in LDS, 16 bytes per (row, quad of 4 k): slice-major, then row block, lane group and row, the 16 rows of
// a quad rotated by the quad's number so that a fragment read (16 rows of a quad) and a walk along the quads of
// one row both cover all banks.
template <int RB>
__device__ __forceinline__ int slot(int row, int quad) {
  return (((quad >> 2) * RB + (row >> 4)) * 4 + (quad & 3)) * 16 + ((row + quad) & 15);
}

// Division of small non-negative numbers (products below 2^32 / d, exact there) by a multiplication.
struct FastDiv {
  unsigned d, m;
};
static inline FastDiv fast_div(int d) { return FastDiv{(unsigned)d, (unsigned)((0x100000000ull + d - 1) / d)}; }
__device__ __forceinline__ int operator/(int x, FastDiv f) { return f.d == 1 ? x : (int)__umulhi((unsigned)x, f.m); }

// 16 RB rows x 4 KQ columns from global rows row_of(local row) into LDS.
template <int RB, int NT, typename F>
__device__ __forceinline__ void stage_rows(v4f* As, int KQ, FastDiv fq, F row_ptr) {
  constexpr int AHEAD = (RB * 16 * MAXS * 4 + NT - 1) / NT > 8 ? 8 : (RB * 16 * MAXS * 4 + NT - 1) / NT;
  const int units = RB * 16 * KQ;
  for (int u0 = threadIdx.x; u0 < units; u0 += NT * AHEAD) {
    v4f v[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int u = min(u0 + a * NT, units - 1), t = u >> 4;
      const int rb = t / fq;
      v[a] = *(const v4f*)(row_ptr(rb * 16 + (u & 15)) + (t - rb * KQ) * 4);
    }
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      const int u = u0 + a * NT, t = u >> 4;
      const int rb = t / fq;
      if (u < units) As[slot<RB>(rb * 16 + (u & 15), t - rb * KQ)] = v[a];
    }
  }
}

// acc[rb] += rows (LDS) x 16 weight columns, K = 16 S <= 16 MAXS, the wave's weights already in registers.
__device__ __forceinline__ void load_weights(const v4f* __restrict__ bp, int S, v4f (&b)[MAXS]) {
#pragma unroll
  for (int j = 0; j < MAXS; ++j)
    if (j < S) b[j] = bp[64 * j];
}
template <int RB>
__device__ __forceinline__ void wave_gemm(const v4f* As, const v4f (&b)[MAXS], int S, v4f (&acc)[RB]) {
  const int lane = threadIdx.x & 63, g = lane >> 4, cl = lane & 15;
  v4f a[2][RB];  // the next slice's rows are read before this slice's products
  auto rows = [&](int s, v4f (&d)[RB]) {
#pragma unroll
    for (int i = 0; i < RB; ++i) d[i] = As[((s * RB + i) * 4 + g) * 16 + ((cl + 4 * s + g) & 15)];
  };
  rows(0, a[0]);
#pragma unroll
  for (int s = 0; s < MAXS; s += 2) {
    if (s < S) {  // uniform; S is even
      rows(s + 1, a[1]);
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < RB; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0][i][st], b[s][st], acc[i], 0, 0, 0);
      if (s + 2 < MAXS) rows(min(s + 2, S - 1), a[0]);
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < RB; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1][i][st], b[s + 1][st], acc[i], 0, 0, 0);
    }
  }
}

struct ValueLayer {
  const float* X;  // row (b n + i) at X + (b n + i) * ldx: [h (Kh) | ...], K columns
  long ldx;
  const v4f *W, *Wmu;           // lane order (launch_lane_pack): K and Km wide
  const float* bias;            // [W1]
  float* out;                   // row (b n + i), or spin-major, at out + row * ldo
  long ldo;
  int K, Kh, Km, vs, permute, B, n, u, W1, rw;
  FastDiv fq, fm, fn;  // by K / 4, Km / 4, n
};

// ------------------------------------------------------------------------------------------------
// rw whole walkers (rw n <= 16 RB rows) x 64 columns per workgroup of 12 waves: waves 0-3 own 16 columns each of
// the per-electron GEMM, waves 4-11 half of the K parts each of the mean product for 16 columns.  Every wave loads
// its weights before the rows are staged.
// ------------------------------------------------------------------------------------------------
template <int RB>
__global__ __launch_bounds__(768) void k_value_layer(ValueLayer p) {
  extern __shared__ __align__(16) float smem[];
  constexpr int NT = 768;
  v4f* const As = (v4f*)smem;                     // 16 RB rows x K
  const int pitch = p.Km + 4;
  float* const Ms = smem + 16 * RB * p.K;         // spin means, rw x (Km + 4)
  float* const Vs = Ms + p.rw * pitch;            // parts of V, vs x rw x 64
  const int tilesN = p.W1 / 64;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, cl = lane & 15;
  const int b0 = blockIdx.x / tilesN * p.rw;
  const int c0 = (blockIdx.x % tilesN) * 64;
  const int rw = min(p.rw, p.B - b0), n = p.n, rows = rw * n;
  const bool mean_wave = wv >= 4;
  const int cb = mean_wave ? (wv - 4) >> 1 : wv, half = (wv - 4) & 1;
  const int c = c0 + cb * 16 + cl;
  // mean product: parts [q0, q0 + nq) of vs, Sp slices each (vs = 1: the first half-wave has them all)
  const int Sp = (p.Km >> 4) / p.vs, nq = p.vs == 4 ? 2 : 1, q0 = p.vs == 4 ? 2 * half : half;
  const int Sw = mean_wave ? (p.vs == 1 && half ? 0 : nq * Sp) : p.K >> 4;  // slices of this wave
  v4f b[MAXS];
  const int cbg = (c0 >> 4) + cb;
  const v4f* bp = lane + (mean_wave ? p.Wmu + 64 * (cbg * (p.Km >> 4) + q0 * Sp) : p.W + 64 * (cbg * (p.K >> 4)));
  load_weights(bp, Sw, b);
  const float* Xb = p.X + (long)b0 * n * p.ldx;
  stage_rows<RB, NT>(As, p.K >> 2, p.fq, [&](int r) { return Xb + min(r, rows - 1) * p.ldx; });
  __syncthreads();
  v4f acc[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
  if (mean_wave) {
    const int Kh4 = p.Kh >> 2, Km4 = p.Km >> 2;
    for (int t = tid - 256; t < rw * Km4; t += NT - 256) {  // spin means: electrons in order, then 1 / n_s
      const int w = t / p.fm, f = t - w * Km4;
      v4f v = {0.f, 0.f, 0.f, 0.f};
      if (f < 2 * Kh4) {
        const int s = f >= Kh4 ? 1 : 0;
        const int quad = f - s * Kh4, i0 = s ? p.u : 0, i1 = s ? n : p.u;
#pragma unroll 4
        for (int i = i0; i < i1; ++i) {
          const v4f x = As[slot<RB>(w * n + i, quad)];
          v[0] += x[0];
          v[1] += x[1];
          v[2] += x[2];
          v[3] += x[3];
        }
        const float inv = 1.f / (float)(i1 - i0);
        v[0] *= inv;
        v[1] *= inv;
        v[2] *= inv;
        v[3] *= inv;
      }
      *(v4f*)(Ms + w * pitch + 4 * f) = v;
    }
  } else {
    wave_gemm<RB>(As, b, Sw, acc);
  }
  __syncthreads();
  if (mean_wave && Sw > 0) {
    const float* ap = Ms + min(cl, rw - 1) * pitch + 16 * q0 * Sp + 4 * g;
    v4f v0 = {0.f, 0.f, 0.f, 0.f}, v1 = v0;
    if (nq == 2) {  // two parts of 8 slices, interleaved
      v4f a0[8], a1[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        a0[t] = *(const v4f*)(ap + 16 * t);
        a1[t] = *(const v4f*)(ap + 16 * (8 + t));
      }
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          v0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[t][st], b[t][st], v0, 0, 0, 0);
          v1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[t][st], b[8 + t][st], v1, 0, 0, 0);
        }
    } else {
      v4f a0 = *(const v4f*)ap, a1;
#pragma unroll
      for (int t = 0; t < MAXS; ++t)
        if (t < Sw) {  // uniform
          a1 = *(const v4f*)(ap + 16 * min(t + 1, Sw - 1));
#pragma unroll
          for (int st = 0; st < 4; ++st) v0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[st], b[t][st], v0, 0, 0, 0);
          a0 = a1;
        }
      for (int t = MAXS; t < Sw; ++t) {
        const v4f at = *(const v4f*)(ap + 16 * t), bt = bp[64 * t];
#pragma unroll
        for (int st = 0; st < 4; ++st) v0 = __builtin_amdgcn_mfma_f32_16x16x4f32(at[st], bt[st], v0, 0, 0, 0);
      }
    }
    const float bias = q0 == 0 ? p.bias[c] : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (4 * g + e < rw) {
        float* vp = Vs + (q0 * p.rw + 4 * g + e) * 64 + cb * 16 + cl;
        vp[0] = q0 == 0 ? v0[e] + bias : v0[e];
        if (nq == 2) vp[p.rw * 64] = v1[e];
      }
  }
  __syncthreads();
  if (mean_wave) return;
  const int dn = n - p.u;
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = i * 16 + 4 * g + e;
      if (r < rows) {
        const int w = r / p.fn, el = r - w * n;
        const float* vp = Vs + w * 64 + cb * 16 + cl;
        float v = vp[0];
        for (int q = 1; q < p.vs; ++q) v += vp[q * p.rw * 64];
        const float y = tanh_fast(acc[i][e] + v);
        const long bb = b0 + w;
        long orow = bb * n + el;
        if (p.permute) orow = (el < p.u) ? bb * p.u + el : (long)p.B * p.u + bb * dn + (el - p.u);
        p.out[orow * p.ldo + c] = y;
      }
    }
}

// ------------------------------------------------------------------------------------------------
// Orbital GEMMs of both spins: rows [0, up_rows) of H times Wo_up, the rest times Wo_dn.  C[M, N], 16 RB rows x
// 64 columns per workgroup.
// ------------------------------------------------------------------------------------------------
template <int RB>
__global__ __launch_bounds__(256) void k_value_orb(const float* __restrict__ H, long ldh, int K,
                                                   const v4f* __restrict__ W_up, const v4f* __restrict__ W_dn,
                                                   float* __restrict__ O, long ldo, int up_rows, int dn_rows, int N,
                                                   int tilesN, int tiles_up, FastDiv fq) {
  extern __shared__ __align__(16) float smem[];
  v4f* const As = (v4f*)smem;
  int tm = blockIdx.x / tilesN;
  const int c0 = (blockIdx.x % tilesN) * 64;
  const bool dn = tm >= tiles_up;  // uniform
  if (dn) tm -= tiles_up;
  const int row0 = tm * 16 * RB, M = dn ? dn_rows : up_rows;
  const long base = dn ? up_rows : 0;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, cl = lane & 15;
  const int c = c0 + wv * 16 + cl;
  v4f b[MAXS];
  load_weights((dn ? W_dn : W_up) + 64 * (((c0 >> 4) + wv) * (K >> 4)) + lane, K >> 4, b);
  stage_rows<RB, 256>(As, K >> 2, fq, [&](int r) { return H + (base + min(row0 + r, M - 1)) * ldh; });
  __syncthreads();
  v4f acc[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
  wave_gemm<RB>(As, b, K >> 4, acc);
  if (c < N) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = row0 + i * 16 + 4 * g + e;
        if (r < M) O[(base + r) * ldo + c] = acc[i][e];
      }
  }
}

// ------------------------------------------------------------------------------------------------
// Whole layers of 256 columns for rw walkers (rw n <= 16 RB rows) per workgroup of 16 waves, wave w owning columns
// [16 w, 16 w + 16) of the per-electron GEMM and of the mean product.  The activations stay in LDS from layer to
// layer; the mean product's slices run between the per-electron GEMM's, so both weights stream from L2 at an even rate
// two slices ahead; a layer has three barriers.
// What bounds it: FP32 MFMA (28,672 rows x 320 x 256 with 2,048 x 512 x 256: 37 us at the matrix rate), then the phases
// without products (means, tanh, barriers: about 12 us).  28,672 rows (2,048 N2 walkers), per layer of three: 72 us in
// three launches (means, mean product, per-electron GEMM), 55 here.
// ------------------------------------------------------------------------------------------------
struct NetLayer {
  const float* X;  // row (b n + i): [h (Kt, filled here for l > 0) | pair columns]
  long ldx;
  const v4f *W, *Wmu;
  const float* bias;
  float* out;  // may be null for l < L - 1
  long ldo;
  int K, Km, Kh, vs;
  FastDiv fm;  // by Km / 4
};
struct ValueNet {
  NetLayer l[DW_MAX_LAYERS];
  int L, permute, B, n, u, rw, mu_off;  // mu_off: floats of the row area
  FastDiv fq, fn;                       // by K / 4 of the first layer, n
};

template <int RB>
__global__ __launch_bounds__(1024) void k_value_net(ValueNet p) {
  extern __shared__ __align__(16) float smem[];
  constexpr int NT = 1024, TL = (RB * 16 * 16 + NT - 1) / NT;
  v4f* const As = (v4f*)smem;
  float* const Ms = smem + p.mu_off;  // spin means, rw x (Km + 4); after the products each wave's V, rw x 16
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, cl = lane & 15;
  const int b0 = blockIdx.x * p.rw;
  const int rw = min(p.rw, p.B - b0), n = p.n, rows = rw * n, dn = n - p.u;
  const int c = wv * 16 + cl;
  {
    const float* Xb = p.l[0].X + (long)b0 * n * p.l[0].ldx;
    const long ldx = p.l[0].ldx;
    stage_rows<RB, NT>(As, p.l[0].K >> 2, p.fq, [&](int r) { return Xb + min(r, rows - 1) * ldx; });
  }
#pragma unroll 1
  for (int l = 0; l < p.L; ++l) {
    const NetLayer& q = p.l[l];
    const int S = q.K >> 4, SV = q.Km >> 4, Sp = SV / q.vs, pitch = q.Km + 4;
    const v4f* bp = q.W + (long)wv * S * 64 + lane;
    const v4f* mp = q.Wmu + (long)wv * SV * 64 + lane;
    v4f b0v = bp[0], b1v = bp[64 * min(1, S - 1)];
    v4f m0 = mp[0], m1 = mp[64 * min(1, SV - 1)];
    // the next layer's pair columns, written to LDS when this layer's products are done
    v4f tl[TL];
    const bool more = l + 1 < p.L;
    if (more) {
      const NetLayer& nx = p.l[l + 1];
      const int tq = (nx.K - 256) >> 2;  // quads of pair columns (at most 16)
#pragma unroll
      for (int t = 0; t < TL; ++t) {
        const int idx = tid + t * NT, row = idx >> 4, quad = idx & 15;
        if (quad < tq && row < RB * 16)
          tl[t] = *(const v4f*)(nx.X + ((long)b0 * n + min(row, rows - 1)) * nx.ldx + 256 + quad * 4);
      }
    }
    const float bias = q.bias[c];
    __syncthreads();  // rows of this layer complete
    const int Kh4 = q.Kh >> 2, Km4 = q.Km >> 2;
    for (int t = tid; t < rw * Km4; t += NT) {  // spin means: electrons in order, then 1 / n_s
      const int w = t / q.fm, f = t - w * Km4;
      v4f v = {0.f, 0.f, 0.f, 0.f};
      if (f < 2 * Kh4) {
        const int sp = f >= Kh4 ? 1 : 0;
        const int quad = f - sp * Kh4, i0 = sp ? p.u : 0, i1 = sp ? n : p.u;
#pragma unroll 4
        for (int i = i0; i < i1; ++i) {
          const v4f x = As[slot<RB>(w * n + i, quad)];
          v[0] += x[0];
          v[1] += x[1];
          v[2] += x[2];
          v[3] += x[3];
        }
        const float inv = 1.f / (float)(i1 - i0);
        v[0] *= inv;
        v[1] *= inv;
        v[2] *= inv;
        v[3] *= inv;
      }
      *(v4f*)(Ms + w * pitch + 4 * f) = v;
    }
    __syncthreads();
    v4f acc[RB], va = {0.f, 0.f, 0.f, 0.f}, vsum = va;
#pragma unroll
    for (int i = 0; i < RB; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
    const float* ap = Ms + min(cl, rw - 1) * pitch + 4 * g;
    int j = 0, jp = 0;  // mean product: next slice, its number inside its part
    bool first = true;
    auto mean_slice = [&](const v4f& b) {
      const v4f a = *(const v4f*)(ap + 16 * j);
#pragma unroll
      for (int st = 0; st < 4; ++st) va = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st], b[st], va, 0, 0, 0);
      ++j;
      if (++jp == Sp) {  // uniform: parts added in order, the bias on the first
#pragma unroll
        for (int e = 0; e < 4; ++e) vsum[e] = first ? va[e] + bias : vsum[e] + va[e];
        va = v4f{0.f, 0.f, 0.f, 0.f};
        first = false;
        jp = 0;
      }
    };
#pragma unroll 1
    for (int s = 0; s < S; ++s) {
      v4f a[RB];
#pragma unroll
      for (int i = 0; i < RB; ++i) a[i] = As[((s * RB + i) * 4 + g) * 16 + ((cl + 4 * s + g) & 15)];
      const v4f bc = b0v;
      b0v = b1v;
      b1v = bp[64 * min(s + 2, S - 1)];
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < RB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][st], bc[st], acc[i], 0, 0, 0);
      if (j < SV) {  // two slices of the mean product (uniform)
        const v4f c0 = m0, c1 = m1;
        m0 = mp[64 * min(j + 2, SV - 1)];
        m1 = mp[64 * min(j + 3, SV - 1)];
        mean_slice(c0);
        if (j < SV) mean_slice(c1);
      }
    }
    while (j < SV) {
      const v4f c0 = m0;
      m0 = m1;
      m1 = mp[64 * min(j + 2, SV - 1)];
      mean_slice(c0);
    }
    __syncthreads();  // every wave is done with the rows and the means
    float* const Vs = Ms + wv * rw * 16;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (4 * g + e < rw) Vs[(4 * g + e) * 16 + cl] = vsum[e];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float* const out = q.out;
    const bool perm = p.permute && !more;
    int g4 = 4 * g;  // opaque: the outputs' addresses are formed here, not kept in registers over the layers
    asm volatile("" : "+v"(g4));
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = i * 16 + g4 + e;
        const int w = min(r / p.fn, rw - 1);
        const float y = tanh_fast(acc[i][e] + Vs[w * 16 + cl]);
        if (more) smem[slot<RB>(r, c >> 2) * 4 + (c & 3)] = y;
        if (out && r < rows) {
          const int el = r - w * n;
          const long bb = b0 + w;
          long orow = bb * n + el;
          if (perm) orow = (el < p.u) ? bb * p.u + el : (long)p.B * p.u + bb * dn + (el - p.u);
          out[orow * q.ldo + c] = y;
        }
      }
    if (more) {
      const int tq = (p.l[l + 1].K - 256) >> 2;
#pragma unroll
      for (int t = 0; t < TL; ++t) {
        const int idx = tid + t * NT, row = idx >> 4, quad = idx & 15;
        if (quad < tq && row < RB * 16) As[slot<RB>(row, 64 + quad)] = tl[t];
      }
    }
  }
}

template <int RB>
static void launch_net(const ValueNet& p, size_t shm, hipStream_t s) {
  if (shm > 65536)
    (void)hipFuncSetAttribute((const void*)k_value_net<RB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
  hipLaunchKernelGGL((k_value_net<RB>), dim3((unsigned)((p.B + p.rw - 1) / p.rw)), dim3(1024), shm, s, p);
}

// A layer of RB row blocks takes about 5.5 RB + 15 us a round of 256 workgroups, at any batch; the separate kernels about
// 18 + 0.0025 us a row.  Measured per layer of three, separate / here: 14 electrons 37.6 / 27 (512 walkers), 54 / 38
// (1,000), 72 / 55 (2,048), 121 / 97 (3,000); 4 electrons 101 / 75 (8,192); 42 electrons 38 / 31 (192), 66 / 50 (512);
// 60 electrons 47 / 37 (200) but 105 / 111 (600: one walker a workgroup, whose mean product fills one MFMA row of 16).
bool value_net(const ValueNetLayer* layers, int L, int permute, int B, int n, int u, int W1, hipStream_t s) {
  if (W1 != 256 || L < 1 || L > DW_MAX_LAYERS || B < 1) return false;
  ValueNet p{};
  int Kmax = 0, Kmm = 256;
  for (int l = 0; l < L; ++l) {
    const ValueNetLayer& a = layers[l];
    if (a.K % 16 || a.K < 16 || a.K > 16 * MAXS || a.Km % (16 * a.vs) || a.Km < 16 || a.Kh % 4 || a.ldx % 4) return false;
    if (l > 0 && (a.Kh != 256 || a.Kt != 256 || a.K < 256 || a.K > 320)) return false;
    Kmax = a.K > Kmax ? a.K : Kmax;
    Kmm = a.Km > Kmm ? a.Km : Kmm;
    p.l[l] = NetLayer{a.X, a.ldx, (const v4f*)a.W, (const v4f*)a.Wmu, a.bias, a.out, a.ldo, a.K, a.Km, a.Kh, a.vs,
                      fast_div(a.Km / 4)};
  }
  p.L = L;
  p.permute = permute;
  p.B = B;
  p.n = n;
  p.u = u;
  p.fq = fast_div(layers[0].K / 4);
  p.fn = fast_div(n);
  double cost = 18.0 + 0.0025 * (double)B * n;
  int best = 0, best_rw = 0;
  for (int RB = 1; RB <= 7; ++RB) {
    const int rw = std::min(std::min(16 * RB / n, 16), B);
    if (rw < 1 || ((size_t)16 * RB * Kmax + (size_t)rw * (Kmm + 4)) * 4 > 160 * 1024) continue;
    const double t = (((B + rw - 1) / rw + 255) / 256) * (5.5 * RB + 15.0);
    if (t < cost) {
      cost = t;
      best = RB;
      best_rw = rw;
    }
  }
  if (!best) return false;
  p.rw = best_rw;
  p.mu_off = 16 * best * Kmax;
  const size_t shm = ((size_t)p.mu_off + (size_t)p.rw * (Kmm + 4)) * 4;
  switch (best) {
    case 1: launch_net<1>(p, shm, s); break;
    case 2: launch_net<2>(p, shm, s); break;
    case 3: launch_net<3>(p, shm, s); break;
    case 4: launch_net<4>(p, shm, s); break;
    case 5: launch_net<5>(p, shm, s); break;
    case 6: launch_net<6>(p, shm, s); break;
    default: launch_net<7>(p, shm, s); break;
  }
  return true;
}

template <int RB>
static bool launch_layer(ValueLayer p, hipStream_t s) {
  p.rw = 16 * RB / p.n;
  // what the kernel's registers hold: 20 slices of W, 16 of W_mu per wave and part (vs = 1 reads the rest as it goes)
  if (p.K > 16 * MAXS || p.K % 32 || p.Km > 512 || p.Km % (16 * p.vs) || p.Kh % 4 || p.ldx % 4) return false;
  if (p.vs == 4 && p.Km != 512) return false;
  if (p.rw > 16) p.rw = 16;
  if (p.rw > p.B) p.rw = p.B;
  const size_t shm = ((size_t)16 * RB * p.K + (size_t)p.rw * (p.Km + 4) + (size_t)p.vs * p.rw * 64) * 4;
  if (shm > 160 * 1024) return false;
  if (shm > 65536)
    (void)hipFuncSetAttribute((const void*)k_value_layer<RB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
  const unsigned grid = (unsigned)((p.B + p.rw - 1) / p.rw * (p.W1 / 64));
  hipLaunchKernelGGL((k_value_layer<RB>), dim3(grid), dim3(768), shm, s, p);
  return true;
}

// The smallest row tile whose workgroups fit the 256 CUs in one round.  One round takes 9 to 24 us by height (10 at
// 16 rows, 13, 16, 19, 24 at 80), the separate kernels (means, mean product, per-electron GEMM) 27 to 35 us there: 1.2
// to 3.4 times faster at 3 to 60 electrons.  With a second round (24 us or more at 32 rows) they win: every workgroup
// reads its 64 columns of both weights again, and the mean product fills 16 MFMA rows with one to five walkers.
bool value_layer(const float* X, long ldx, int K, int Kh, const void* W, const void* Wmu, int Km, const float* bias,
                 int vs, float* out, long ldo, int permute, int B, int n, int u, int W1, hipStream_t s) {
  const ValueLayer p{X, ldx, (const v4f*)W, (const v4f*)Wmu, bias, out, ldo, K, Kh, Km, vs, permute, B, n, u, W1, 1,
                     fast_div(K / 4), fast_div(Km / 4), fast_div(n)};
  for (int RB = 1; RB <= 5; ++RB) {
    const int rw = 16 * RB / n < 16 ? 16 * RB / n : 16;
    if (rw < 1 || (long)(B + rw - 1) / rw * (W1 / 64) > 256) continue;
    switch (RB) {
      case 1: return launch_layer<1>(p, s);
      case 2: return launch_layer<2>(p, s);
      case 3: return launch_layer<3>(p, s);
      case 4: return launch_layer<4>(p, s);
      default: return launch_layer<5>(p, s);
    }
  }
  return false;
}

// Up to 2048 workgroups of 16 rows: 4 to 18 us, against 17 us and more for two launches of k_gemm_f32 (25 us at 9,000
// rows x 416 columns, where both meet).
bool value_orbitals(const float* H, long ldh, int K, const void* W_up, const void* W_dn, float* O, long ldo,
                    int up_rows, int dn_rows, int N, hipStream_t s) {
  const int tilesN = (N + 63) / 64, tu = (up_rows + 15) / 16, td = (dn_rows + 15) / 16;
  if (K > 16 * MAXS || K % 32 || (long)(tu + td) * tilesN > 2048) return false;
  hipLaunchKernelGGL((k_value_orb<1>), dim3((tu + td) * tilesN), dim3(256), (size_t)16 * K * 4, s, H, ldh, K,
                     (const v4f*)W_up, (const v4f*)W_dn, O, ldo, up_rows, dn_rows, N, tilesN, tu, fast_div(K / 4));
  return true;
}

}  // namespace dwmi
