// Embedding of the dpe4 model (configuration.py:875-891, 422-441, 666-674; ferminet_embedding.py:97-188,
// 196-267): FermiNet iterations whose 1-el input is [h, mean_up h, mean_dn h, e_ee, e_ei] with
//   e_ee[i] = sum_j w_{s(i,j)}(p_l[i, j]) * hm_l[j],  hm_l = tanh(h W_map + b)      (SchNet-style, self pair in)
//   e_ei[i] = sum_I q_l[i, I] * tanh(h_ion W + b)[I],  h_ion = table[Z_I - Z_min]
// where p_l is the same/diff-spin pair stream (started from |r_j - r_i| alone) and q_l the el-ion stream
// (started from [|r_i - R_I|, r_i - R_I]), each taking one residual tanh layer between iterations, and
// w_same / w_diff one tanh layer applied to p_l.
//
// Every quantity carries the forward-mode Laplacian channels of the pass.  A pair quantity depends on
// d = r_j - r_i only and keeps 5 channels [value, d/dd_x, d/dd_y, d/dd_z, total Laplacian over all 3n
// coordinates] (d/dr_j = +grad, d/dr_i = -grad, so each |grad_c|^2 enters the Laplacian twice); an el-ion
// quantity depends on r_i only and keeps [value, d/dr_i (3), Laplacian in r_i].  The electron rows of X_l
// carry the pass's C = 3n+2 channels (value, 1 + 3e + c, Laplacian) padded to Cp rows.
//
// Kernels: k_dpe4_pairs_mfma (pair stream and the mapped w_l for every iteration, stored per pair; k_dpe4_pairs and
// k_dpe4_pairs_value in the FP64 form), k_dpe4_elion (el-ion stream and e_ei of every iteration, written into X_l),
// k_dpe4_hmap (hm = tanh rule of X_l[:, h] W_map; the other forms take the library's GEMM and k_dpe4_tanh),
// k_dpe4_conv and k_dpe4_conv_lap (e_ee into X_l).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "common.h"
#include "kernels.h"

namespace dwmi {

namespace {

constexpr int EMB = 32;  // emb_dim = width of the pair and el-ion streams

__device__ __forceinline__ float sqrt_t(float x) { return sqrtf(x); }
__device__ __forceinline__ double sqrt_t(double x) { return sqrt(x); }
__device__ __forceinline__ float tanh_t(float x) { return tanh_fast(x); }
__device__ __forceinline__ double tanh_t(double x) { return tanh(x); }

// y = tanh(z) in NCH channels; lap_factor 2 for pair quantities (both electrons see the gradient), 1 for
// el-ion quantities.
template <int NCH, typename T>
__device__ __forceinline__ void tanh_channels(const T z[NCH], T y[NCH], T lap_factor) {
  const T t = tanh_t(z[0]);
  y[0] = t;
  if constexpr (NCH > 1) {
    const T d1 = T(1) - t * t, d2 = T(-2) * t * d1;
    y[1] = d1 * z[1];
    y[2] = d1 * z[2];
    y[3] = d1 * z[3];
    y[4] = d1 * z[4] + d2 * lap_factor * (z[1] * z[1] + z[2] * z[2] + z[3] * z[3]);
  }
}

// ------------------------------------------------------------------------------------------------------
// Pair streams of the FP64 form, Laplacian pass.  One workgroup per (walker, 8 electrons i); thread (il, f) walks the
// partners j in order.
// Weight sets q = 0 .. L-1 are the maps w_same/w_diff of iteration q, q = L .. 2L-2 the stream layers
// h_same/h_diff of iteration q - L; each [2 (same, diff)][32 k][32 f] (rows k >= fan-in zero) with biases
// [2][32].  Output: wm[l][b][i][j][ch][f].
// ------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void k_dpe4_pairs(const float* __restrict__ r, const T* __restrict__ Wp,
                                                    const T* __restrict__ bp, T* __restrict__ wm, Shape sh) {
  constexpr int NCH = 5;
  extern __shared__ unsigned char smem_raw[];
  const int L = sh.L, n = sh.n, u = sh.u;
  T* xs = (T*)smem_raw;  // [8][NCH][32]
  const T *gW = Wp, *gB = bp;  // read through the caches

  const int groups = (n + 7) >> 3;
  const long b = blockIdx.x / groups;
  const int il = threadIdx.x >> 5, f = threadIdx.x & 31;
  const int i = (int)(blockIdx.x % groups) * 8 + il;
  const bool active = i < n;
  const float* rb = r + b * n * 3;
  const T rix = active ? (T)rb[i * 3 + 0] : T(0), riy = active ? (T)rb[i * 3 + 1] : T(0),
          riz = active ? (T)rb[i * 3 + 2] : T(0);
  const T rs2 = (T)0.70710678118654752440;
  const long per_l = (long)sh.B * n * n * NCH * EMB;
  T* xrow = xs + (size_t)il * NCH * EMB;

  for (int j = 0; j < n; ++j) {
    const int s = ((i < u) == (j < u)) ? 0 : 1;
    T x[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) x[c] = T(0);
    if (active && j != i && f == 0) {
      const T dx = (T)rb[j * 3 + 0] - rix, dy = (T)rb[j * 3 + 1] - riy, dz = (T)rb[j * 3 + 2] - riz;
      const T rho = sqrt_t(dx * dx + dy * dy + dz * dz);
      x[0] = rho;
      x[1] = dx / rho;
      x[2] = dy / rho;
      x[3] = dz / rho;
      x[4] = T(4) / rho;  // 2 / rho from each of the two electrons
    }
    T* out = wm + ((((long)b * n + (active ? i : 0)) * n + j) * NCH) * EMB + f;
    for (int l = 0; l < L; ++l) {
      const int kin = (l == 0) ? 1 : EMB;
      __syncthreads();  // the weight tiles are loaded / the previous reads of xs are done
#pragma unroll
      for (int c = 0; c < NCH; ++c) xrow[c * EMB + f] = x[c];
      __syncthreads();
      const T* Wm = gW + ((size_t)l * 2 + s) * EMB * EMB;
      T zm[NCH], zh[NCH];
      zm[0] = gB[(l * 2 + s) * EMB + f];
#pragma unroll
      for (int c = 1; c < NCH; ++c) zm[c] = T(0);
      const bool stream = l < L - 1;
      const T* Wh = gW + ((size_t)(L + l) * 2 + s) * EMB * EMB;
      zh[0] = stream ? gB[((L + l) * 2 + s) * EMB + f] : T(0);
#pragma unroll
      for (int c = 1; c < NCH; ++c) zh[c] = T(0);
      for (int k = 0; k < kin; ++k) {
        const T wmk = Wm[k * EMB + f];
        const T whk = stream ? Wh[k * EMB + f] : T(0);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
          const T xv = xrow[c * EMB + k];
          zm[c] += xv * wmk;
          zh[c] += xv * whk;
        }
      }
      T y[NCH];
      tanh_channels<NCH, T>(zm, y, T(2));
      if (active) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) out[(long)l * per_l + c * EMB] = y[c];
      }
      if (stream) {
        tanh_channels<NCH, T>(zh, y, T(2));
        if (kin == EMB) {
#pragma unroll
          for (int c = 0; c < NCH; ++c) y[c] = (x[c] + y[c]) * rs2;
        }
#pragma unroll
        for (int c = 0; c < NCH; ++c) x[c] = y[c];
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------------
// El-ion stream and its convolution.  k_dpe4_him forms h_ion_map of every iteration, him[l][I][f] (zero
// beyond the iteration's width g_l; NaN for a Z outside the embedding table).  k_dpe4_elion: one workgroup
// per (walker, 8 electrons i); thread (il, f) walks the ions.  Stream layer l: Wei[l][32 k][32 f] (rows
// k >= fan-in zero).  e_ei of iteration l goes to the columns tail[l] + EMB + f (f < g_l) of X_l for every
// channel row.
// ------------------------------------------------------------------------------------------------------
template <typename T>
struct ElIonOut {
  T* X[MAXL_DPE4];
  int Kx[MAXL_DPE4];
  int tail[MAXL_DPE4];  // first column of [e_ee | e_ei] in X_l
};

template <typename T>
__global__ __launch_bounds__(256) void k_dpe4_him(const float* __restrict__ Z, const T* __restrict__ table,
                                                  const T* __restrict__ Whim, const T* __restrict__ bhim, int n_types,
                                                  int z_min, T* __restrict__ him, int L, int I) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= L * I * EMB) return;
  const int l = q / (I * EMB), ion = (q / EMB) % I, f = q % EMB;
  const int g = (l == 0) ? 4 : EMB;
  T v = T(0);
  if (f < g) {
    const int idx = (int)lrintf(Z[ion]) - z_min;
    if (idx < 0 || idx >= n_types) {
      v = (T)NAN;  // a charge outside the embedding table: the walkers' results become NaN (flagged)
    } else {
      T z = bhim[l * EMB + f];
      for (int k = 0; k < EMB; ++k) z += table[idx * EMB + k] * Whim[((size_t)l * EMB + k) * EMB + f];
      v = tanh_t(z);
    }
  }
  him[q] = v;
}

template <bool LAP, typename T>
__global__ __launch_bounds__(256) void k_dpe4_elion(const float* __restrict__ r, const float* __restrict__ R,
                                                    const T* __restrict__ Wei, const T* __restrict__ bei,
                                                    const T* __restrict__ him, ElIonOut<T> out, Shape sh) {
  constexpr int NCH = LAP ? 5 : 1;
  __shared__ T xs[8 * NCH * EMB];
  const int L = sh.L, I = sh.I, n = sh.n, C = sh.C, Cp = sh.Cp;

  const int groups = (n + 7) >> 3;
  const long b = blockIdx.x / groups;
  const int il = threadIdx.x >> 5, f = threadIdx.x & 31;
  const int i = (int)(blockIdx.x % groups) * 8 + il;
  const bool active = i < n;
  const long bi = b * n + (active ? i : 0);
  const T rs2 = (T)0.70710678118654752440;
  T* xrow = xs + (size_t)il * NCH * EMB;
  T acc[MAXL_DPE4][NCH];
#pragma unroll
  for (int l = 0; l < MAXL_DPE4; ++l)
#pragma unroll
    for (int c = 0; c < NCH; ++c) acc[l][c] = T(0);
  const float* ri = r + bi * 3;

  for (int ion = 0; ion < I; ++ion) {
    T x[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) x[c] = T(0);
    if (active && f < 4) {
      const T d[3] = {(T)ri[0] - (T)R[ion * 3 + 0], (T)ri[1] - (T)R[ion * 3 + 1], (T)ri[2] - (T)R[ion * 3 + 2]};
      const T rho = sqrt_t(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
      if (f == 0) {
        x[0] = rho;
        if constexpr (LAP) {
          x[1] = d[0] / rho;
          x[2] = d[1] / rho;
          x[3] = d[2] / rho;
          x[4] = T(2) / rho;
        }
      } else {
        x[0] = d[f - 1];
        if constexpr (LAP) x[f] = T(1);
      }
    }
#pragma unroll
    for (int l = 0; l < MAXL_DPE4; ++l) {
      if (l >= L) break;
      __syncthreads();  // the previous reads of xs are done
      const T hv = him[((size_t)l * I + ion) * EMB + f];
#pragma unroll
      for (int c = 0; c < NCH; ++c) acc[l][c] += x[c] * hv;
      if (l == L - 1) break;
      const int kin = (l == 0) ? 4 : EMB;
#pragma unroll
      for (int c = 0; c < NCH; ++c) xrow[c * EMB + f] = x[c];
      __syncthreads();
      const T* W = Wei + (size_t)l * EMB * EMB;
      T z[NCH];
      z[0] = bei[l * EMB + f];
#pragma unroll
      for (int c = 1; c < NCH; ++c) z[c] = T(0);
      for (int k = 0; k < kin; ++k) {
        const T w = W[k * EMB + f];
#pragma unroll
        for (int c = 0; c < NCH; ++c) z[c] += xrow[c * EMB + k] * w;
      }
      T y[NCH];
      tanh_channels<NCH, T>(z, y, T(1));
      if (kin == EMB) {
#pragma unroll
        for (int c = 0; c < NCH; ++c) y[c] = (x[c] + y[c]) * rs2;
      }
#pragma unroll
      for (int c = 0; c < NCH; ++c) x[c] = y[c];
    }
  }
  if (!active) return;
#pragma unroll
  for (int l = 0; l < MAXL_DPE4; ++l) {
    if (l >= L) break;
    const int g = (l == 0) ? 4 : EMB;
    if (f >= g) continue;
    T* col = out.X[l] + bi * Cp * (long)out.Kx[l] + out.tail[l] + EMB + f;
    col[0] = acc[l][0];
    if constexpr (LAP) {
      for (int ch = 1; ch < C - 1; ++ch) {
        const int k = ch - 1, e = k / 3, c = k - 3 * e;
        col[(long)ch * out.Kx[l]] = (e == i) ? acc[l][1 + c] : T(0);
      }
      col[(long)(C - 1) * out.Kx[l]] = acc[l][4];
    }
    for (int ch = LAP ? C : 1; ch < Cp; ++ch) col[(long)ch * out.Kx[l]] = T(0);
  }
}

// ------------------------------------------------------------------------------------------------------
// hm = tanh(z + b) with the forward-Laplacian rule over an electron's channel rows of z = X_l[:, h] W_map.
// One thread per (electron row, f).
// ------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void k_dpe4_tanh(T* __restrict__ hm, const T* __restrict__ bias, Shape sh) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)sh.B * sh.n * EMB) return;
  const long bi = t / EMB;
  const int f = (int)(t % EMB);
  T* p = hm + bi * sh.Cp * EMB + f;
  const T th = tanh_t(p[0] + bias[f]);
  p[0] = th;
  if (sh.C == 1) return;
  const T d1 = T(1) - th * th;
  T sq = T(0);
  for (int ch = 1; ch < sh.C - 1; ++ch) {
    const T z = p[(long)ch * EMB];
    sq += z * z;
    p[(long)ch * EMB] = d1 * z;
  }
  p[(long)(sh.C - 1) * EMB] = d1 * p[(long)(sh.C - 1) * EMB] - T(2) * th * d1 * sq;
  for (int ch = sh.C; ch < sh.Cp; ++ch) p[(long)ch * EMB] = T(0);
}

// ------------------------------------------------------------------------------------------------------
// h_map of one iteration (FP32): hm = tanh rule of X_l[:, h] W_map + b, 32 columns, in one pass over X.  MB blocks of
// 16 rows per wave, whole electrons per workgroup in the Laplacian pass; the rows go from memory to the A operand 32
// columns at a time, one step ahead, W_map sits in LDS in lane order.  Slices and step order (k = 4 g + s) are
// k_gemm_f32's and the rule's sums run over the channels in order: bit-equal to that GEMM and a pass over its result.
// What bounds it: reading X.  688,128 rows x 256 (1,024 walkers of 14): 255 us in a 64 x 64-tile GEMM (half its columns
// idle) + 37 us for the rule, 185 us here.
// ------------------------------------------------------------------------------------------------------
template <bool LAP, int MB>
__global__ __launch_bounds__(256) void k_dpe4_hmap(const float* __restrict__ X, int ldx, const float* __restrict__ Wt,
                                                   int K, const float* __restrict__ bias, float* __restrict__ hm,
                                                   long units, int per_wg, int C, int Cp) {
  // unit: an electron (LAP, Cp rows) or a row; per_wg units per workgroup, at most 64 MB rows
  constexpr int PITCH = EMB + 1;
  extern __shared__ __align__(16) float sm[];
  v4f* const sB = (v4f*)sm;  // [slice][nb][lane]
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, cl = lane & 15;
  const int S = K >> 4;
  for (int q = tid; q < S * 128; q += 256) {
    const int l = q & 63, nb = (q >> 6) & 1, sl = q >> 7;
    sB[q] = *(const v4f*)(Wt + (long)(16 * nb + (l & 15)) * K + 16 * sl + 4 * (l >> 4));
  }
  const long u0 = (long)blockIdx.x * per_wg;
  const int nu = (int)(units - u0 < per_wg ? units - u0 : per_wg);
  const int rpu = LAP ? Cp : 1, rows = nu * rpu;
  const float* Xb = X + u0 * rpu * ldx + 4 * g;
  const float* xp[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) xp[m] = Xb + (long)min((wv * MB + m) * 16 + cl, rows - 1) * ldx;
  v4f a[2][MB], nx[2][MB];
  auto load = [&](int sl, v4f(&d)[2][MB]) {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) d[h][m] = *(const v4f*)(xp[m] + 16 * min(sl + h, S - 1));
  };
  v4f acc[MB][2];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) acc[m][nb] = v4f{0.f, 0.f, 0.f, 0.f};
  load(0, nx);
  __syncthreads();
  for (int sl = 0; sl < S; sl += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MB; ++m) a[h][m] = nx[h][m];
    load(sl + 2, nx);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (sl + h < S) {  // uniform
        const v4f b0 = sB[(sl + h) * 128 + lane], b1 = sB[(sl + h) * 128 + 64 + lane];
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            acc[m][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][m][st], b0[st], acc[m][0], 0, 0, 0);
            acc[m][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][m][st], b1[st], acc[m][1], 0, 0, 0);
          }
      }
  }
  float* out = hm + u0 * rpu * EMB;
  if constexpr (!LAP) {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = (wv * MB + m) * 16 + 4 * g + e, f = 16 * nb + cl;
          if (row < rows) out[(long)row * EMB + f] = tanh_t(acc[m][nb][e] + bias[f]);
        }
  } else {
    __syncthreads();  // W_map has been read: its space holds the rows
    float* const sZ = sm;
    float* const sR = sm + 64 * MB * PITCH;  // [unit][f]: value, sum of squares
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) sZ[((wv * MB + m) * 16 + 4 * g + e) * PITCH + 16 * nb + cl] = acc[m][nb][e];
    __syncthreads();
    for (int q = tid; q < nu * EMB; q += 256) {
      const int f = q & 31;
      const float* p = sZ + (q >> 5) * Cp * PITCH + f;
      float sq = 0.f;
      for (int ch = 1; ch < C - 1; ++ch) {
        const float z = p[ch * PITCH];
        sq += z * z;
      }
      sR[2 * q] = tanh_t(p[0] + bias[f]);
      sR[2 * q + 1] = sq;
    }
    __syncthreads();
    for (int e = 0; e < nu; ++e)
      for (int q = tid; q < Cp * EMB; q += 256) {
        const int ch = q >> 5, f = q & 31;
        const float z = sZ[(e * Cp + ch) * PITCH + f];
        const float th = sR[2 * (e * EMB + f)], sq = sR[2 * (e * EMB + f) + 1];
        const float d1 = 1.f - th * th;
        float y = 0.f;
        if (ch == 0)
          y = th;
        else if (ch < C - 1)
          y = d1 * z;
        else if (ch == C - 1)
          y = d1 * z - 2.f * th * d1 * sq;
        out[(long)e * Cp * EMB + q] = y;
      }
  }
}

// ------------------------------------------------------------------------------------------------------
// Value pass: e_ee[i][f] = sum_j w[i, j][f] hm[j][f].  One workgroup per walker, the walker's hm in LDS.
// ------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void k_dpe4_conv(const T* __restrict__ wm, const T* __restrict__ hm,
                                                   T* __restrict__ X, int Kx, int col0, Shape sh) {
  extern __shared__ unsigned char smem_raw[];
  T* hs = (T*)smem_raw;  // [n][32]
  const int n = sh.n;
  const long b = blockIdx.x;
  for (int q = threadIdx.x; q < n * EMB; q += 256) hs[q] = hm[b * n * EMB + q];
  __syncthreads();
  const int il = threadIdx.x >> 5, f = threadIdx.x & 31;
  for (int i = il; i < n; i += 8) {
    T acc = T(0);
    const T* w = wm + (b * n + i) * n * EMB + f;
    for (int j = 0; j < n; ++j) acc += w[(long)j * EMB] * hs[j * EMB + f];
    X[(b * n + i) * Kx + col0 + f] = acc;
  }
}

// ------------------------------------------------------------------------------------------------------
// Laplacian pass: e_ee[i][ch][f] = sum_j w[i, j][f] hm[j][ch][f] plus the pair derivatives:
//   tangent row (e, c):  + (delta_{e j} - delta_{e i}) g_c[i, j] hm[j][0]
//   Laplacian row:       + L_w[i, j] hm[j][0] + 2 sum_c g_c[i, j] (hm[j][(j, c)] - hm[j][(i, c)])
// (g = d w / d d, L_w the pair's total Laplacian; the self pair's w is constant).  A workgroup takes a walker,
// w of NI electrons i at a time in LDS (all blocks of NI in turn, or one) and a part of the channel rows (conv_launch says
// how many); a thread owns (channel row, f) and NI electrons i, so every element of hm is read once per NI and the row's own
// e is fixed: its derivative terms are NI products at j = e, and one chain of its own for i = e.  The Laplacian row takes a
// group of 32 lanes per electron i.  Terms are added in order of j, whatever the split.
// What bounds it: memory, w and hm read two to three times (the derivative terms' rows no longer in L2), e_ee written.
// 1,024 walkers of 14 (48 rows): 269 us with a thread per (i, f) and 16
// channel rows testing each row against (i, j), 196 us here.
// ------------------------------------------------------------------------------------------------------
template <int NI, typename T>
__global__ __launch_bounds__(512) void k_dpe4_conv_lap(const T* __restrict__ wm, const T* __restrict__ hm,
                                                       T* __restrict__ X, int Kx, int col0, Shape sh, int iblocks,
                                                       int parts) {
  extern __shared__ unsigned char smem_raw[];
  T* ws = (T*)smem_raw;  // [NI][n][32]: w of electrons i0 .. i0 + NI - 1
  const int n = sh.n, C = sh.C, Cp = sh.Cp;
  // workgroup: walker, block of electrons (iblocks = 1: all of them in turn), part of the channel rows
  const int part = (int)(blockIdx.x % (unsigned)parts), rest = (int)(blockIdx.x / (unsigned)parts);
  const int ib = rest % iblocks;
  const long b = rest / iblocks;
  const int grp = threadIdx.x >> 5, f = threadIdx.x & 31;
  const T* hb = hm + b * n * Cp * EMB + f;
  const T* wb = wm + b * n * n * 5 * EMB + f;
  const long hj = (long)Cp * EMB;
  for (int i0 = ib * NI; i0 < n; i0 += iblocks * NI) {
    if (i0 > ib * NI) __syncthreads();
    for (int p = grp; p < NI * n; p += 16)
      ws[p * EMB + f] = i0 * n + p < n * n ? wb[(long)(i0 * n + p) * 5 * EMB] : T(0);
    __syncthreads();
    const T* wf = ws + f;
    for (int ch = part * 16 + grp; ch < Cp; ch += parts * 16) {
      if (ch == C - 1) continue;
      T acc[NI], own = T(0);
#pragma unroll
      for (int k = 0; k < NI; ++k) acc[k] = T(0);
      const int e = ch >= 1 && ch < C ? (ch - 1) / 3 : -1, c = ch - 1 - 3 * e;
      const bool mine = e >= i0 && e < i0 + NI;  // row e = i belongs to this block
      if (ch < C) {
        T h = hb[(long)ch * EMB];
        for (int j = 0; j < n; ++j) {
          const T hn = hb[min(j + 1, n - 1) * hj + (long)ch * EMB];
#pragma unroll
          for (int k = 0; k < NI; ++k) acc[k] += wf[(k * n + j) * EMB] * h;
          if (mine) {
            own += wf[((e - i0) * n + j) * EMB] * h;
            if (j != e) own -= wb[((long)(e * n + j) * 5 + 1 + c) * EMB] * hb[j * hj];
          }
          if (j == e) {
            const T h0 = hb[j * hj];
#pragma unroll
            for (int k = 0; k < NI; ++k)
              if (i0 + k < n) acc[k] += wb[((long)((i0 + k) * n + j) * 5 + 1 + c) * EMB] * h0;
          }
          h = hn;
        }
      }
      T* out = X + ((b * n + i0) * Cp + ch) * Kx + col0 + f;
#pragma unroll
      for (int k = 0; k < NI; ++k)
        if (i0 + k < n) out[(long)k * Cp * Kx] = i0 + k == e ? own : acc[k];
    }
    const int i = i0 + grp;
    if (part == parts - 1 && grp < NI && i < n) {
      T acc = T(0);
#pragma unroll 2
      for (int j = 0; j < n; ++j) {
        const T* w = wb + (long)(i * n + j) * 5 * EMB;
        const T* hg = hb + j * hj;
        acc += wf[(grp * n + j) * EMB] * hg[(long)(C - 1) * EMB];
        if (j != i) {
          T v = w[4 * EMB] * hg[0];
#pragma unroll
          for (int c = 0; c < 3; ++c)
            v += T(2) * w[(1 + c) * EMB] * (hg[(long)(1 + 3 * j + c) * EMB] - hg[(long)(1 + 3 * i + c) * EMB]);
          acc += v;
        }
      }
      X[((b * n + i) * Cp + C - 1) * Kx + col0 + f] = acc;
    }
  }
}

// ------------------------------------------------------------------------------------------------------
// Value pass of the pair streams (FP64 form): one lane per pair.  The pairs of one spin relation (s = 0 same, 1 diff)
// are enumerated walker by walker (same: up-up then down-down; diff: up-down then down-up) and the blocks
// of each relation are contiguous, so a wavefront's weights are uniform (scalar loads).  Each lane keeps
// its pair's 32 features in registers and writes w_l[b][i][j][f] as 16-byte vectors.
// ------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void k_dpe4_pairs_value(const float* __restrict__ r, const T* __restrict__ Wp,
                                                          const T* __restrict__ bp, T* __restrict__ wm, Shape sh,
                                                          int blocks_same) {
  const int n = sh.n, u = sh.u, d = sh.n - sh.u, L = sh.L;
  const int s = (int)blockIdx.x >= blocks_same ? 1 : 0;
  const long P = s == 0 ? (long)u * u + (long)d * d : 2L * u * d;  // pairs of this relation per walker
  const long t = (long)(blockIdx.x - (s ? blocks_same : 0)) * blockDim.x + threadIdx.x;
  if (t >= (long)sh.B * P) return;
  const long b = t / P;
  const int q = (int)(t - b * P);
  int i, j;
  if (s == 0) {
    if (q < u * u) {
      i = q / u;
      j = q - i * u;
    } else {
      const int q2 = q - u * u;
      i = u + q2 / d;
      j = u + q2 % d;
    }
  } else {
    if (q < u * d) {
      i = q / d;
      j = u + q % d;
    } else {
      const int q2 = q - u * d;
      i = u + q2 / u;
      j = q2 % u;
    }
  }
  const float* rb = r + b * n * 3;
  T x[EMB];
#pragma unroll
  for (int k = 0; k < EMB; ++k) x[k] = T(0);
  if (i != j) {
    const T dx = (T)rb[j * 3 + 0] - (T)rb[i * 3 + 0], dy = (T)rb[j * 3 + 1] - (T)rb[i * 3 + 1],
            dz = (T)rb[j * 3 + 2] - (T)rb[i * 3 + 2];
    x[0] = sqrt_t(dx * dx + dy * dy + dz * dz);
  }
  const long per_l = (long)sh.B * n * n * EMB;
  T* out = wm + ((long)(b * n + i) * n + j) * EMB;
  const T rs2 = (T)0.70710678118654752440;
  for (int l = 0; l < L; ++l) {
    const T* Wm = Wp + ((size_t)l * 2 + s) * EMB * EMB;
    const T* Bm = bp + ((size_t)l * 2 + s) * EMB;
    // the map w_l
#pragma unroll
    for (int f0 = 0; f0 < EMB; f0 += 4) {
      T y4[4];
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int fo = f0 + q4;
        T z = Bm[fo];
        if (l == 0) {
          z += Wm[fo] * x[0];
        } else {
#pragma unroll
          for (int k = 0; k < EMB; ++k) z += Wm[k * EMB + fo] * x[k];
        }
        y4[q4] = tanh_t(z);
      }
      *(double2*)(out + l * per_l + f0) = make_double2(y4[0], y4[1]);
      *(double2*)(out + l * per_l + f0 + 2) = make_double2(y4[2], y4[3]);
    }
    if (l == L - 1) break;
    // the stream layer h_same / h_diff (residual from the second iteration on)
    const T* Wh = Wp + ((size_t)(L + l) * 2 + s) * EMB * EMB;
    const T* Bh = bp + ((size_t)(L + l) * 2 + s) * EMB;
    T y[EMB];
#pragma unroll
    for (int fo = 0; fo < EMB; ++fo) {
      T z = Bh[fo];
      if (l == 0) {
        z += Wh[fo] * x[0];
      } else {
#pragma unroll
        for (int k = 0; k < EMB; ++k) z += Wh[k * EMB + fo] * x[k];
      }
      y[fo] = tanh_t(z);
    }
#pragma unroll
    for (int k = 0; k < EMB; ++k) x[k] = (l == 0) ? y[k] : (x[k] + y[k]) * rs2;
  }
}

// ------------------------------------------------------------------------------------------------------
// Pair streams in FP32, value (NCH = 1) and Laplacian (NCH = 5) passes: 16 pairs of one spin relation per wavefront
// and step, on FP32 MFMA.  Weights are the A operand (rows = output features), the pairs the columns of B, so a pair
// stays in its lane column (pair = lane % 16) and the four lane groups share its 32 features.  Step t of a product
// takes k = 4 t + g; a stream layer's output rows are ordered so that group g holds features 4 t + g, register t: the
// next product's B operand, with no exchange.  A map's rows keep their order (16 nb + 4 g + e): 16-byte stores.
// v_mfma_f32_16x16x4_f32 adds its four products to C as fmaf in order of k, so every sum is the chain
// z = b; z = fmaf(x_k, w_k, z), k ascending, of a kernel without MFMA; the residual's sum is rounded by itself
// (residual() below), so the rest is too.
// Pairs of a relation are enumerated walker by walker (same: up-up then down-down; diff: up-down then down-up).
// What bounds it: stores and tanh.  200,704 pairs (1,024 walkers of 14), 4 iterations, Laplacian: 762 us with a
// thread per (electron, feature) reading x from LDS, 166 us here; value, 144,500 pairs (500 walkers of 17): 69 us
// with a lane per pair, 31 us here.
// ------------------------------------------------------------------------------------------------------
// (x + y) / sqrt 2.  y is the product t' z for a tangent: the compiler would fuse it into the sum, and every energy (and
// with it the FP64 loss) would change by a rounding against the kernels that keep x and y apart.
__device__ __forceinline__ float residual(float x, float y) {
#pragma clang fp contract(off)
  return (x + y) * (float)0.70710678118654752440;
}

template <int NCH>
__global__ __launch_bounds__(256, 4) void k_dpe4_pairs_mfma(const float* __restrict__ r, const float* __restrict__ Wp,
                                                         const float* __restrict__ bp, float* __restrict__ wm, Shape sh,
                                                         int blocks_same) {
  extern __shared__ __align__(16) float sw[];
  const int n = sh.n, u = sh.u, d = sh.n - sh.u, L = sh.L, NS = 2 * L - 1;
  const int s = (int)blockIdx.x >= blocks_same ? 1 : 0;
  const int blk = (int)blockIdx.x - (s ? blocks_same : 0), nblk = s ? (int)gridDim.x - blocks_same : blocks_same;
  const int lane = threadIdx.x & 63, g = lane >> 4, cl = lane & 15;
  // [set][nb][t quad][lane] v4f: row of block nb in this lane's position, k = 4 t + g; then [set][nb][g] v4f of biases
  v4f* const sW = (v4f*)sw;
  v4f* const sB = sW + NS * 2 * 2 * 64;
  for (int q = threadIdx.x; q < NS * 256; q += 256) {
    const int set = q >> 8, nb = (q >> 7) & 1, tq = (q >> 6) & 1, l = q & 63, row = l & 15;
    const int f = set < L ? 16 * nb + row : 16 * nb + 4 * (row & 3) + (row >> 2);
    const float* W = Wp + ((size_t)set * 2 + s) * EMB * EMB + f;
    v4f v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = W[(4 * (4 * tq + e) + (l >> 4)) * EMB];
    sW[q] = v;
  }
  for (int q = threadIdx.x; q < NS * 8; q += 256) {
    const int set = q >> 3, nb = (q >> 2) & 1, gg = q & 3;
    v4f v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = bp[((size_t)set * 2 + s) * EMB + 16 * nb + (set < L ? 4 * gg + e : 4 * e + gg)];
    sB[q] = v;
  }
  __syncthreads();
  const int P = s == 0 ? u * u + d * d : 2 * u * d;  // pairs of this relation per walker
  const long total = (long)sh.B * P;
  const long per_l = (long)sh.B * n * n * NCH * EMB;
  for (long t0 = ((long)blk * 4 + (threadIdx.x >> 6)) * 16; t0 < total; t0 += (long)nblk * 64) {
    const bool ok = t0 + cl < total;
    const long t = ok ? t0 + cl : total - 1;
    const long b = div_idx(t, P);
    const int q = (int)(t - b * P);
    int i, j;
    if (s == 0) {
      if (q < u * u) {
        i = q / u;
        j = q - i * u;
      } else {
        const int q2 = q - u * u;
        i = u + q2 / d;
        j = u + q2 % d;
      }
    } else {
      if (q < u * d) {
        i = q / d;
        j = u + q % d;
      } else {
        const int q2 = q - u * d;
        i = u + q2 / u;
        j = q2 % u;
      }
    }
    float x0[NCH];  // the first iteration's input, one feature
#pragma unroll
    for (int c = 0; c < NCH; ++c) x0[c] = 0.f;
    if (i != j) {
      const float* rb = r + b * n * 3;
      const float dx = rb[j * 3 + 0] - rb[i * 3 + 0], dy = rb[j * 3 + 1] - rb[i * 3 + 1],
                  dz = rb[j * 3 + 2] - rb[i * 3 + 2];
      const float rho = sqrt_t(dx * dx + dy * dy + dz * dz);
      x0[0] = rho;
      if constexpr (NCH == 5) {
        x0[1] = dx / rho;
        x0[2] = dy / rho;
        x0[3] = dz / rho;
        x0[4] = 4.f / rho;
      }
    }
    float x[NCH][8];
    float* out = wm + ((b * n + i) * n + j) * NCH * EMB + 4 * g;
    // rows of one set times the pairs' features (iteration 0: one feature, k = 0, whose weights group 0 holds)
    auto product = [&](int set, int l, v4f(&z)[NCH][2]) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        z[0][nb] = sB[set * 8 + nb * 4 + g];
#pragma unroll
        for (int c = 1; c < NCH; ++c) z[c][nb] = v4f{0.f, 0.f, 0.f, 0.f};
      }
      if (l == 0) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w = sW[(set * 2 + nb) * 128 + 4 * g + e][0];  // row 4 g + e, k = 0
#pragma unroll
            for (int c = 0; c < NCH; ++c) z[c][nb][e] += x0[c] * w;
          }
        return;
      }
#pragma unroll
      for (int tq = 0; tq < 2; ++tq)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          const v4f w = sW[((set * 2 + nb) * 2 + tq) * 64 + lane];
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < NCH; ++c)
              z[c][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[c][4 * tq + e], z[c][nb], 0, 0, 0);
        }
    };
#pragma unroll 1
    for (int l = 0; l < L; ++l) {
      v4f z[NCH][2];
      product(l, l, z);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        v4f o[NCH];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float zz[NCH], y[NCH];
#pragma unroll
          for (int c = 0; c < NCH; ++c) zz[c] = z[c][nb][e];
          tanh_channels<NCH, float>(zz, y, 2.f);
#pragma unroll
          for (int c = 0; c < NCH; ++c) o[c][e] = y[c];
        }
        if (ok)
#pragma unroll
          for (int c = 0; c < NCH; ++c) *(v4f*)(out + l * per_l + c * EMB + 16 * nb) = o[c];
      }
      if (l == L - 1) break;
      product(L + l, l, z);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float zz[NCH], y[NCH];
#pragma unroll
          for (int c = 0; c < NCH; ++c) zz[c] = z[c][nb][e];
          tanh_channels<NCH, float>(zz, y, 2.f);
#pragma unroll
          for (int c = 0; c < NCH; ++c) x[c][4 * nb + e] = l == 0 ? y[c] : residual(x[c][4 * nb + e], y[c]);
        }
    }
  }
}

}  // namespace

template <typename T>
void launch_dpe4_pairs(const float* r, const T* Wp, const T* bp, T* wm, const Shape& sh, hipStream_t s) {
  if constexpr (sizeof(T) == 4) {
    // each relation's workgroups in proportion to its pairs, at most four per CU in all (the weights of a relation are
    // staged once per workgroup)
    const long u = sh.u, d = sh.n - sh.u;
    const long gs = (sh.B * (u * u + d * d) + 63) / 64, gd = (sh.B * 2 * u * d + 63) / 64, all = gs + gd;
    const long cap = all < 1024 ? all : 1024;
    const int bs = (int)((gs * cap + all - 1) / all), bd = (int)((gd * cap + all - 1) / all);
    const size_t smem = (size_t)(2 * sh.L - 1) * (256 + 8) * 16;
    if (sh.C == 1)
      hipLaunchKernelGGL(k_dpe4_pairs_mfma<1>, dim3(bs + bd), dim3(256), smem, s, r, Wp, bp, wm, sh, bs);
    else
      hipLaunchKernelGGL(k_dpe4_pairs_mfma<5>, dim3(bs + bd), dim3(256), smem, s, r, Wp, bp, wm, sh, bs);
    return;
  } else {
  if (sh.C == 1) {  // lane per pair, wave-uniform weights
    const long u = sh.u, d = sh.n - sh.u;
    const int blocks_same = (int)((sh.B * (u * u + d * d) + 255) / 256);
    const int blocks_diff = (int)((sh.B * 2 * u * d + 255) / 256);
    hipLaunchKernelGGL(k_dpe4_pairs_value<T>, dim3(blocks_same + blocks_diff), dim3(256), 0, s, r, Wp, bp, wm, sh,
                       blocks_same);
    return;
  }
  const unsigned grid = (unsigned)(sh.B * ((sh.n + 7) / 8));
  const size_t smem = (size_t)8 * 5 * EMB * sizeof(T);
  hipLaunchKernelGGL((k_dpe4_pairs<T>), dim3(grid), dim3(256), smem, s, r, Wp, bp, wm, sh);
  }
}

template <typename T>
void launch_dpe4_elion(const float* r, const float* R, const float* Z, const T* Wei, const T* bei, const T* Whim,
                       const T* bhim, const T* table, int n_types, int z_min, T* him, T* const* X, const int* Kx,
                       const int* tail, const Shape& sh, hipStream_t s) {
  const int total = sh.L * sh.I * EMB;
  hipLaunchKernelGGL(k_dpe4_him<T>, dim3((total + 255) / 256), dim3(256), 0, s, Z, table, Whim, bhim, n_types, z_min,
                     him, sh.L, sh.I);
  ElIonOut<T> o{};
  for (int l = 0; l < sh.L; ++l) {
    o.X[l] = X[l];
    o.Kx[l] = Kx[l];
    o.tail[l] = tail[l];
  }
  const unsigned grid = (unsigned)(sh.B * ((sh.n + 7) / 8));
  if (sh.C > 1)
    hipLaunchKernelGGL((k_dpe4_elion<true, T>), dim3(grid), dim3(256), 0, s, r, R, Wei, bei, him, o, sh);
  else
    hipLaunchKernelGGL((k_dpe4_elion<false, T>), dim3(grid), dim3(256), 0, s, r, R, Wei, bei, him, o, sh);
}

template <typename T>
void launch_dpe4_tanh(T* hm, const T* bias, const Shape& sh, hipStream_t s) {
  const long total = (long)sh.B * sh.n * EMB;
  hipLaunchKernelGGL(k_dpe4_tanh<T>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, hm, bias, sh);
}

bool launch_dpe4_hmap(const float* X, int ldx, const float* Wt, int K, const float* bias, float* hm, const Shape& sh,
                      hipStream_t s) {
  if (K % 16 || K < 16 || K > 512 || ldx % 4) return false;
  const size_t wb = (size_t)K * 128;
  if (sh.C == 1) {
    const long rows = (long)sh.B * sh.n;
    hipLaunchKernelGGL((k_dpe4_hmap<false, 1>), dim3((unsigned)((rows + 63) / 64)), dim3(256), wb, s, X, ldx, Wt, K, bias,
                       hm, rows, 64, 1, 1);
    return true;
  }
  if (sh.Cp > 192) return false;
  const int per = 192 / sh.Cp;
  const long units = (long)sh.B * sh.n;
  const size_t zb = ((size_t)192 * (EMB + 1) + (size_t)per * EMB * 2) * 4;
  hipLaunchKernelGGL((k_dpe4_hmap<true, 3>), dim3((unsigned)((units + per - 1) / per)), dim3(256), wb > zb ? wb : zb, s,
                     X, ldx, Wt, K, bias, hm, units, per, sh.C, sh.Cp);
  return true;
}

template <typename T, int NI>
static void conv_launch(const T* wm, const T* hm, T* X, int Kx, int col0, const Shape& sh, hipStream_t s) {
  // Up to 512 workgroups are made of a small batch, whose threads otherwise walk the blocks of electrons and their channel
  // rows one after another, waiting for memory at every j; more than two blocks are separate at any batch (hm stays in L2).
  // E_loc (1 determinant) with a workgroup per walker / as chosen, us: 42 electrons 3,968 / 1,255 (1 walker), 7,424 / 3,552
  // (64), 14,061 / 11,231 (256); 26 electrons 1,723 / 889 (16), 7,777 / 7,465 (512); 20 electrons 1,528 / 1,125 (64), 4,903
  // (512; 5,038 with two blocks); 14 electrons 741 / 654 (16), 1,611 / 1,527 (256), 2,630 (512; 2,747 with two parts); FP64, 42
  // electrons 9,536 / 4,015 (16).
  const int blocks = (sh.n + NI - 1) / NI;
  const long most = 512;
  const int ib = blocks > 2 || (long)sh.B * blocks <= most ? blocks : 1;
  const int parts = (int)std::max<long>(1, std::min<long>((sh.Cp + 15) / 16, most / ((long)sh.B * ib)));
  hipLaunchKernelGGL((k_dpe4_conv_lap<NI, T>), dim3((unsigned)(sh.B * ib * parts)), dim3(512),
                     (size_t)NI * sh.n * EMB * sizeof(T), s, wm, hm, X, Kx, col0, sh, ib, parts);
}

template <typename T>
void launch_dpe4_conv(const T* wm, const T* hm, T* X, int Kx, int col0, const Shape& sh, hipStream_t s) {
  if (sh.C == 1) {
    hipLaunchKernelGGL(k_dpe4_conv<T>, dim3((unsigned)sh.B), dim3(256), (size_t)sh.n * EMB * sizeof(T), s, wm, hm, X, Kx,
                       col0, sh);
    return;
  }
  // electrons per block: w of a block stays within 48 KB of LDS (three workgroups per CU), 64 KB for 4 electrons
  const size_t row_bytes = (size_t)sh.n * EMB * sizeof(T);
  if (row_bytes * 16 <= 48 * 1024)
    conv_launch<T, 16>(wm, hm, X, Kx, col0, sh, s);
  else if (row_bytes * 8 <= 48 * 1024)
    conv_launch<T, 8>(wm, hm, X, Kx, col0, sh, s);
  else
    conv_launch<T, 4>(wm, hm, X, Kx, col0, sh, s);
}

#define DPE4_INST(T)                                                                                               \
  template void launch_dpe4_pairs<T>(const float*, const T*, const T*, T*, const Shape&, hipStream_t);             \
  template void launch_dpe4_elion<T>(const float*, const float*, const float*, const T*, const T*, const T*,       \
                                     const T*, const T*, int, int, T*, T* const*, const int*, const int*,          \
                                     const Shape&, hipStream_t);                                                   \
  template void launch_dpe4_tanh<T>(T*, const T*, const Shape&, hipStream_t);                                      \
  template void launch_dpe4_conv<T>(const T*, const T*, T*, int, int, const Shape&, hipStream_t);
DPE4_INST(float)
DPE4_INST(double)

}  // namespace dwmi
