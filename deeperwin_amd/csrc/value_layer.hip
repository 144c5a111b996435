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
// GEMMs 17 us in two launches, 4.2 us in one.
#include "common.h"
#include "kernels.h"

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
