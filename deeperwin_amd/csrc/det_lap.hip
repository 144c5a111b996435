// Laplacian-mode determinants (FP64), in two launches: log|det|, sign and M^-1 per matrix,
// then the channel passes
//   Y_k = M^-1 dM_k,  g_k = tr Y_k,  q_k = tr(Y_k^2),  Lap log|det| = tr(M^-1 Lap M) - sum_k q_k.
// Both read the orbitals O and apply the envelope themselves, so the product envelope x orbitals (3 n + 2 matrices per
// determinant) is never stored.
//
// 16,384 matrices of 26 (1024 walkers): 4.17 ms for the determinants and 1.99 ms for the stored product before, 0.84 ms
// (inverses) + 2.08 ms (channels) here; 1,536 matrices of 42: 4.06 + 0.75 ms before, 0.55 + 1.04 ms here; 32,768
// matrices of 14: 1.14 ms (one wavefront per matrix) before, 0.08 + 0.43 ms here.  Above 16 electrons the channel
// passes run at half the FP64 matrix rate, padding to 16 x 16 blocks counted (1.06 and 0.54 ms at 78 TFLOP/s).
#include <utility>

#include "common.h"
#include "det_common.h"
#include "kernels.h"

namespace dwmi {

// Value-channel element (i, column of this lane) of matrix (b, d): envelope x orbital, in TA as the channels are.
template <typename TA>
__device__ __forceinline__ double value_at(const OrbSrc<TA>& src, const Shape& sh, long b, int i, int oc) {
  TA env, g0, g1, g2, le;
  envelope_at<TA, true>(src.kappa, src.wenv, src.r, src.R, sh, b, i, oc, env, g0, g1, g2, le);
  return (double)(env * src.O[orb_row(sh, b, i) * src.ldo + oc]);
}

// Lane P of every 16-lane row to all lanes of that row (DPP row_newbcast).
template <int P>
__device__ __forceinline__ int row_bcast(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + P, 0xF, 0xF, true);
}
template <int P>
__device__ __forceinline__ double row_bcast(double v) {
  return __hiloint2double(row_bcast<P>(__double2hiint(v)), row_bcast<P>(__double2loint(v)));
}
// n <= 16: four matrices per wavefront, one per 16-lane row, a lane per column; entries are broadcast inside a row by
// DPP, so all four eliminate at once (a matrix per wavefront kept 14 of 64 lanes busy: 32,768 matrices of 14 took 358
// us, 83 us here).  The operations and their order are lu_columns'.
template <typename TA>
__global__ __launch_bounds__(256) void k_det_inv16(OrbSrc<TA> src, Shape sh, double* __restrict__ Minv,
                                                   double* __restrict__ ld, double* __restrict__ sd,
                                                   float* __restrict__ dcond, long nmat) {
  constexpr int N = 16;
  const int lane = threadIdx.x & 63, c = lane & 15, n = sh.n;
  long bd = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  const bool valid = bd < nmat;
  if (!valid) bd = nmat - 1;  // whole waves stay in the lane exchanges; results are not stored
  const long b = bd / sh.D;
  const int dcol = (int)(bd - b * sh.D) * n;
  const bool act = c < n;
  double col[N];
  int perm[N];
  double csum = 0.0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    col[i] = (act && i < n) ? value_at<TA>(src, sh, b, i, dcol + c) : 0.0;
    csum += fabs(col[i]);
    perm[i] = i;
  }
  auto row_max = [](double v) {
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
  };
  const double normA = row_max(csum);
  double mydiag = 1.0;
  bool sing = false;
  int swaps = 0;
  unroll_seq(
      [&](auto PP) {
        constexpr int p = PP;
        if (p < n) {  // uniform
          double best = -1.0;
          int bidx = p;
#pragma unroll
          for (int i = p; i < N; ++i) {
            const double a = fabs(col[i]);
            const bool take = i < n && a > best;
            best = take ? a : best;
            bidx = take ? i : bidx;
          }
          const int piv = row_bcast<p>(bidx);
          if (!(row_bcast<p>(best) > 0.0)) sing = true;
          swaps += piv != p ? 1 : 0;
          const double old = col[p];
          const int oldp = perm[p];
#pragma unroll
          for (int i = p + 1; i < N; ++i) {
            const bool sw = i == piv;
            col[p] = sw ? col[i] : col[p];
            perm[p] = sw ? perm[i] : perm[p];
            col[i] = sw ? old : col[i];
            perm[i] = sw ? oldp : perm[i];
          }
          if (c == p) mydiag = col[p];
          const double rp = 1.0 / row_bcast<p>(col[p]);
#pragma unroll
          for (int i = p + 1; i < N; ++i) {
            const double l = col[i] * rp;
            if (c == p) col[i] = l;
            const double li = row_bcast<p>(col[i]);
            if (c > p) col[i] -= li * col[p];
          }
        }
      },
      std::make_integer_sequence<int, N>{});
  double lg = act ? log(fabs(mydiag)) : 0.0;
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) lg += __shfl_xor(lg, o, 64);
  const unsigned long long neg = __ballot(act && mydiag < 0.0);
  const int nneg = __popc((unsigned)(neg >> (lane & 48)) & 0xFFFFu) + swaps;
  double x[N];  // column c of the inverse: L y = P e_c, then U x = y
  unroll_seq(
      [&](auto PP) {
        constexpr int p = PP;
        double y = (p < n && perm[p] == c) ? 1.0 : 0.0;
        if (p < n)
          unroll_seq([&](auto QQ) { y -= row_bcast<int(QQ)>(col[p]) * x[int(QQ)]; }, std::make_integer_sequence<int, p>{});
        x[p] = y;
      },
      std::make_integer_sequence<int, N>{});
  unroll_seq(
      [&](auto PP) {
        constexpr int p = N - 1 - int(PP);
        if (p < n) {
          double y = x[p];
          unroll_seq(
              [&](auto QQ) {
                constexpr int q = p + 1 + int(QQ);
                if (q < n) y -= row_bcast<q>(col[p]) * x[q];
              },
              std::make_integer_sequence<int, N - 1 - p>{});
          x[p] = y / row_bcast<p>(col[p]);
        }
      },
      std::make_integer_sequence<int, N>{});
  double isum = 0.0;
#pragma unroll
  for (int a = 0; a < N; ++a) {
    isum += act ? fabs(x[a]) : 0.0;
    if (act && a < n && valid) Minv[bd * n * n + a * n + c] = x[a];
  }
  const double normMi = row_max(isum);
  if (c == 0 && valid) {
    ld[bd] = sing ? -INFINITY : lg;
    sd[bd] = sing ? 0.0 : ((nneg & 1) ? -1.0 : 1.0);
    dcond[bd] = (float)(normA * normMi);
  }
}

// 16 < n <= 32: one matrix per wavefront, a lane per column, LU and inverse in registers.  Minv [matrix][n][n].
template <int NMAX, typename TA>
__global__ __launch_bounds__(256) void k_det_inv(OrbSrc<TA> src, Shape sh, double* __restrict__ Minv,
                                                 double* __restrict__ ld, double* __restrict__ sd,
                                                 float* __restrict__ dcond, long nmat) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n = sh.n;
  const long bd = (long)blockIdx.x * 4 + wv;
  if (bd >= nmat) return;  // uniform over the wave; no barriers
  const long b = bd / sh.D;
  const int dcol = (int)(bd - b * sh.D) * n;
  const bool act = lane < n;
  double col[NMAX];
  int perm[NMAX];
  double csum = 0.0;
#pragma unroll
  for (int i = 0; i < NMAX; ++i) {
    col[i] = (act && i < n) ? value_at<TA>(src, sh, b, i, dcol + lane) : 0.0;
    csum += fabs(col[i]);
  }
  const double normA = wave_max_d(csum);
  double mydiag = 1.0;
  bool sing = false;
  const int swaps = lu_columns<NMAX>(col, perm, mydiag, sing, n, lane);
  double logabs, sgn;
  finish_slogdet<NMAX>(mydiag, swaps, sing, n, lane, logabs, sgn);
  double x[NMAX];  // column `lane` of the inverse: L y = P e_lane, then U x = y
#pragma unroll
  for (int p = 0; p < NMAX; ++p) {
    if (p < n) {
      double y = (perm[p] == lane) ? 1.0 : 0.0;
#pragma unroll
      for (int q = 0; q < p; ++q) y -= readlane_d(col[p], q) * x[q];
      x[p] = y;
    } else {
      x[p] = 0.0;
    }
  }
#pragma unroll
  for (int p = NMAX - 1; p >= 0; --p) {
    if (p < n) {
      double y = x[p];
#pragma unroll
      for (int q = p + 1; q < NMAX; ++q)
        if (q < n) y -= readlane_d(col[p], q) * x[q];
      x[p] = y / readlane_d(col[p], p);
    }
  }
  double isum = 0.0;
#pragma unroll
  for (int a = 0; a < NMAX; ++a) {
    isum += act ? fabs(x[a]) : 0.0;
    if (act && a < n) Minv[bd * n * n + a * n + lane] = x[a];
  }
  const double normMi = wave_max_d(isum);
  if (lane == 0) {
    ld[bd] = logabs;
    sd[bd] = sgn;
    dcond[bd] = (float)(normA * normMi);
  }
}

// 32 < n <= 63: one matrix per 64-thread workgroup, a lane per column, matrix and inverse in LDS (pitch n + 1).
// Column-parallel elimination and substitution: a step reads one broadcast and one own element and four partial sums
// run side by side, so a matrix is about n^2 pipelined LDS steps (a workgroup of 256 threads with barriers per
// elimination step and 42 busy lanes in the substitution took most of 4.1 ms per 1536 matrices of 42).
template <typename TA>
__global__ __launch_bounds__(64) void k_det_inv_lds(OrbSrc<TA> src, Shape sh, double* __restrict__ Minv,
                                                    double* __restrict__ ld, double* __restrict__ sd,
                                                    float* __restrict__ dcond) {
  extern __shared__ double sm[];
  const int n = sh.n, P = n + 1, j = threadIdx.x;
  double* T = sm;          // LU factors
  double* X = T + n * P;   // inverse
  int* perm = (int*)(X + n * P);
  const long bd = blockIdx.x, b = bd / sh.D;
  const int dcol = (int)(bd - b * sh.D) * n;
  const bool act = j < n;
  double csum = 0.0;
  if (act) {
    for (int i = 0; i < n; ++i) {
      const double v = value_at<TA>(src, sh, b, i, dcol + j);
      T[i * P + j] = v;
      csum += fabs(v);
    }
    perm[j] = j;
  }
  const double normA = wave_max_d(csum);
  __syncthreads();
  int swaps = 0;
  bool sing = false;
  for (int p = 0; p < n; ++p) {
    // pivot: lane i holds row i of column p; largest |a|, lowest row on ties
    double best = (act && j >= p) ? fabs(T[j * P + p]) : -1.0;
    int bidx = j;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bidx, o, 64);
      if (ob > best || (ob == best && oi < bidx)) {
        best = ob;
        bidx = oi;
      }
    }
    const int piv = __builtin_amdgcn_readfirstlane(bidx);
    if (!(best > 0.0)) sing = true;
    if (piv != p) {  // uniform; a NaN column keeps every lane's own index, where lane 0's is taken
      ++swaps;
      if (act) {
        const double t = T[p * P + j];
        T[p * P + j] = T[piv * P + j];
        T[piv * P + j] = t;
      }
      if (j == 0) {
        const int tp = perm[p];
        perm[p] = perm[piv];
        perm[piv] = tp;
      }
    }
    __syncthreads();
    const double rp = 1.0 / T[p * P + p];
    if (act && j > p) T[j * P + p] *= rp;  // multiplier of row j
    __syncthreads();
    if (act && j > p) {
      const double u = T[p * P + j];
#pragma unroll 8
      for (int i = p + 1; i < n; ++i) T[i * P + j] -= T[i * P + p] * u;
    }
    __syncthreads();
  }
  const double up = act ? T[j * P + j] : 1.0;
  const double lsum = wave_sum_d(act ? log(fabs(up)) : 0.0);
  const int nneg = __popcll(__ballot(act && up < 0.0)) + swaps;
  double isum = 0.0;
  if (act) {
    for (int p = 0; p < n; ++p) {
      double y0 = (perm[p] == j) ? 1.0 : 0.0, y1 = 0.0, y2 = 0.0, y3 = 0.0;
      int q = 0;
#pragma unroll 2
      for (; q + 4 <= p; q += 4) {
        y0 -= T[p * P + q] * X[q * P + j];
        y1 -= T[p * P + q + 1] * X[(q + 1) * P + j];
        y2 -= T[p * P + q + 2] * X[(q + 2) * P + j];
        y3 -= T[p * P + q + 3] * X[(q + 3) * P + j];
      }
      for (; q < p; ++q) y0 -= T[p * P + q] * X[q * P + j];
      X[p * P + j] = (y0 + y1) + (y2 + y3);
    }
    for (int p = n - 1; p >= 0; --p) {
      double y0 = X[p * P + j], y1 = 0.0, y2 = 0.0, y3 = 0.0;
      int q = p + 1;
#pragma unroll 2
      for (; q + 4 <= n; q += 4) {
        y0 -= T[p * P + q] * X[q * P + j];
        y1 -= T[p * P + q + 1] * X[(q + 1) * P + j];
        y2 -= T[p * P + q + 2] * X[(q + 2) * P + j];
        y3 -= T[p * P + q + 3] * X[(q + 3) * P + j];
      }
      for (; q < n; ++q) y0 -= T[p * P + q] * X[q * P + j];
      const double x = ((y0 + y1) + (y2 + y3)) / T[p * P + p];
      X[p * P + j] = x;
      isum += fabs(x);
      Minv[bd * n * n + p * n + j] = x;
    }
  }
  const double normMi = wave_max_d(isum);
  if (j == 0) {
    ld[bd] = sing ? -INFINITY : lsum;
    sd[bd] = sing ? 0.0 : ((nneg & 1) ? -1.0 : 1.0);
    dcond[bd] = (float)(normA * normMi);
  }
}

// ------------------------------------------------------------------------------------------------
// Channel passes, one matrix per workgroup of 4 waves, wave w taking channels w, w + 4, ...  NB = ceil(n / 16)
// blocks of 16 per side on v_mfma_f64_16x16x4f64: lane l (g = l / 16, c = l % 16) holds M^-1[16 I + c][16 K + g + 4 q]
// as A operand (registers for NB = 2) and dM_k[16 K + g + 4 q][16 J + c] as B operand, read from O with the envelope
// applied (tables of the envelope and of the own-electron terms in LDS); the next channel's O is loaded before this
// channel's products.  tr(Y^2) = sum_IJ Y_IJ o (Y_JI)^T: a block is transposed through a wave-private LDS tile instead
// of being computed a second time as (dM^T M^-T), so a channel is NB^3 x 4 MFMAs of 64 cycles, half of what two
// products take; tr Y comes from the diagonal the same tile holds.
// ------------------------------------------------------------------------------------------------
template <int NB, typename TA>
__global__ __launch_bounds__(256, NB == 1 ? 6 : NB == 4 ? 1 : (NB == 2 && sizeof(TA) == 4 ? 3 : 2)) void k_det_chan(OrbSrc<TA> src, Shape sh,
                                                                               const double* __restrict__ Minv,
                                                                               double* __restrict__ g,
                                                                               double* __restrict__ lapd, int nmat) {
  extern __shared__ double sm[];
  constexpr int NP = 16 * NB, PM = NP + 1;
  const int n = sh.n, nd = 3 * n, C = sh.C;
  double* sM = sm;                        // M^-1, NP x PM, zero outside n x n
  double* sT = sM + NP * PM;              // transposition tiles, 4 x 16 x 17
  double* sD = sT + 4 * 16 * 17;          // diagonals of Y_k, nd x 16
  double* red = sD + nd * 16;             // 32
  TA* sE = (TA*)(red + 32);               // envelope, NP x NP, zero outside
  // own-electron terms g_c bf0, 3 x NP x NP; FP64 orbitals of more than 48 electrons have no room for them and form
  // the channel's row again (4 x NP)
  constexpr bool TABLE = NB < 4 || sizeof(TA) == 4;
  TA* sG = sE + NP * NP;
  const int per = (nmat + 7) / 8;         // the determinants of a walker share rows of O: keep them on one XCD
  const int bd = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (bd >= nmat) return;  // uniform over the workgroup, before any barrier
  const long b = bd / sh.D;
  const int dcol = (int)(bd - b * sh.D) * n;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, gq = lane >> 4, cl = lane & 15;

  for (int e = tid; e < NP * NP; e += 256) {
    const int i = e / NP, c = e - (e / NP) * NP;
    sM[i * PM + c] = (i < n && c < n) ? Minv[(long)bd * n * n + i * n + c] : 0.0;
  }
  __syncthreads();
  double tp = 0.0;  // tr(M^-1 Lap M)
  for (int e = tid; e < NP * NP; e += 256) {
    const int i = e / NP, c = e - (e / NP) * NP;
    TA env = TA(0), b0 = TA(0), b1 = TA(0), b2 = TA(0);
    if (i < n && c < n) {
      TA g0, g1, g2, le;
      envelope_at<TA, true>(src.kappa, src.wenv, src.r, src.R, sh, b, i, dcol + c, env, g0, g1, g2, le);
      const TA* Oi = src.O + orb_row(sh, b, i) * src.ldo + dcol + c;
      const TA bf0 = Oi[0];
      const TA t0 = Oi[(long)(1 + 3 * i) * src.ldo];
      const TA t1 = Oi[(long)(2 + 3 * i) * src.ldo];
      const TA t2 = Oi[(long)(3 + 3 * i) * src.ldo];
      b0 = g0 * bf0;
      b1 = g1 * bf0;
      b2 = g2 * bf0;
      const TA lp = le * bf0 + env * Oi[(long)(C - 1) * src.ldo] + TA(2) * (g0 * t0 + g1 * t1 + g2 * t2);
      tp += sM[c * PM + i] * (double)lp;
    }
    sE[e] = env;
    if constexpr (TABLE) {
      sG[e] = b0;
      sG[NP * NP + e] = b1;
      sG[2 * NP * NP + e] = b2;
    }
  }
  __syncthreads();

  constexpr bool REG = NB <= 2;
  double mi[REG ? NB : 1][REG ? NB : 1][4];
  if constexpr (REG) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = 0; K < NB; ++K)
#pragma unroll
        for (int q = 0; q < 4; ++q) mi[I][K][q] = sM[(I * 16 + cl) * PM + K * 16 + gq + 4 * q];
  }
  auto mia = [&](int I, int K, int q) -> double {
    if constexpr (REG)
      return mi[I][K][q];
    else
      return sM[(I * 16 + cl) * PM + K * 16 + gq + 4 * q];
  };
  // O rows of this lane: electron rr at row base (up or down block) + rr Cp
  const long stride = (long)sh.Cp * src.ldo;
  const TA* const base_u = src.O + b * sh.u * stride + dcol;
  const TA* const base_d = src.O + ((long)sh.B * sh.u + b * (n - sh.u) - sh.u) * stride + dcol;
  TA nxt[NB][NB][4];
  auto load = [&](int k) {
    const long choff = (long)(1 + k) * src.ldo;
#pragma unroll
    for (int K = 0; K < NB; ++K)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rr = K * 16 + gq + 4 * q;
        const TA* row = (rr < sh.u ? base_u : base_d) + rr * stride + choff;
#pragma unroll
        for (int J = 0; J < NB; ++J) {
          const int cc = J * 16 + cl;
          nxt[K][J][q] = (rr < n && cc < n) ? row[cc] : TA(0);
        }
      }
  };
  double* T = sT + wv * 16 * 17;
  double qacc = 0.0;
  constexpr bool AHEAD = sizeof(TA) == 4;  // FP64 orbitals: no registers for a second channel
  if (AHEAD && wv < nd) load(wv);
  for (int k = wv; k < nd; k += 4) {
    const int kr = k / 3, kc = k - 3 * kr;  // the channel's electron and axis
    double dm[NB][NB][4];
    if (!AHEAD) load(k);
    if constexpr (!TABLE) {
      TA own = TA(0);
      if (lane < n) {
        TA env, g0, g1, g2, le;
        envelope_at<TA, true>(src.kappa, src.wenv, src.r, src.R, sh, b, kr, dcol + lane, env, g0, g1, g2, le);
        own = (kc == 0 ? g0 : kc == 1 ? g1 : g2) * src.O[orb_row(sh, b, kr) * src.ldo + dcol + lane];
      }
      sG[wv * NP + lane] = own;  // NP == 64; read by this wave only, in order
    }
#pragma unroll
    for (int K = 0; K < NB; ++K)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rr = K * 16 + gq + 4 * q;
        const TA* er = sE + rr * NP + cl;
        const TA* gr = (TABLE ? sG + (kc * NP + rr) * NP : sG + wv * NP) + cl;
#pragma unroll
        for (int J = 0; J < NB; ++J) {
          const TA own = rr == kr ? gr[16 * J] : TA(0);
          dm[K][J][q] = (double)fma(er[16 * J], nxt[K][J][q], own);
        }
      }
    if (AHEAD && k + 4 < nd) load(k + 4);
    __builtin_amdgcn_sched_barrier(0);  // the products follow one block pair at a time (register budget)
    double gp = 0.0;
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int J = I; J < NB; ++J) {
        v4d y = {0.0, 0.0, 0.0, 0.0}, z = y;
#pragma unroll
        for (int K = 0; K < NB; ++K)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            y = __builtin_amdgcn_mfma_f64_16x16x4f64(mia(I, K, q), dm[K][J][q], y, 0, 0, 0);
            if (J > I) z = __builtin_amdgcn_mfma_f64_16x16x4f64(mia(J, K, q), dm[K][I][q], z, 0, 0, 0);
          }
        if (J == I) z = y;
        // lane l, element e: row 4 e + g, column c of the block (LDS accesses of one wave stay in order)
#pragma unroll
        for (int e = 0; e < 4; ++e) T[(4 * e + gq) * 17 + cl] = z[e];
        double s = 0.0;
#pragma unroll
        for (int e = 0; e < 4; ++e) s += y[e] * T[cl * 17 + 4 * e + gq];
        qacc += J > I ? 2.0 * s : s;
        if (J == I) gp += T[cl * 18];
        __builtin_amdgcn_sched_barrier(0);
      }
    if (lane < 16) sD[k * 16 + lane] = gp;
  }
  qacc = block_sum_d(qacc, red);
  tp = block_sum_d(tp, red + 16);
  __syncthreads();
  for (int k = tid; k < nd; k += 256) {
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < 16; ++c) s += sD[k * 16 + c];
    g[(long)bd * nd + k] = s;
  }
  if (tid == 0) lapd[bd] = tp - qacc;
}

template <int NB, typename TA>
static void launch_chan(const OrbSrc<TA>& src, const Shape& sh, const double* Minv, double* g, double* lapd,
                        hipStream_t s) {
  constexpr int NP = 16 * NB;
  const size_t shm = (size_t)(NP * (NP + 1) + 4 * 16 * 17 + 3 * sh.n * 16 + 32) * sizeof(double) +
                     ((size_t)NP * NP + (NB < 4 || sizeof(TA) == 4 ? 3 * NP * NP : 4 * NP)) * sizeof(TA);
  if (shm > 65536)
    (void)hipFuncSetAttribute((const void*)k_det_chan<NB, TA>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
  const int nmat = sh.B * sh.D;
  hipLaunchKernelGGL((k_det_chan<NB, TA>), dim3((nmat + 7) / 8 * 8), dim3(256), shm, s, src, sh, Minv, g, lapd, nmat);
}

template <typename TA>
void launch_det_lap(const OrbSrc<TA>& src, double* Minv, double* ld, double* sd, double* g, double* lapd,
                          float* dcond, const Shape& sh, hipStream_t s) {
  const int n = sh.n;
  const long nmat = (long)sh.B * sh.D;
  if (n <= 16) {
    hipLaunchKernelGGL((k_det_inv16<TA>), dim3((unsigned)((nmat + 15) / 16)), dim3(256), 0, s, src, sh, Minv, ld, sd,
                       dcond, nmat);
  } else if (n <= 32) {
    hipLaunchKernelGGL((k_det_inv<32, TA>), dim3((unsigned)((nmat + 3) / 4)), dim3(256), 0, s, src, sh, Minv, ld, sd,
                       dcond, nmat);
  } else {
    const size_t shm = (size_t)2 * n * (n + 1) * sizeof(double) + 64 * sizeof(int);
    if (shm > 65536)
      (void)hipFuncSetAttribute((const void*)k_det_inv_lds<TA>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    hipLaunchKernelGGL((k_det_inv_lds<TA>), dim3((unsigned)nmat), dim3(64), shm, s, src, sh, Minv, ld, sd, dcond);
  }
  switch ((n + 15) / 16) {
    case 1: launch_chan<1, TA>(src, sh, Minv, g, lapd, s); break;
    case 2: launch_chan<2, TA>(src, sh, Minv, g, lapd, s); break;
    case 3: launch_chan<3, TA>(src, sh, Minv, g, lapd, s); break;
    default: launch_chan<4, TA>(src, sh, Minv, g, lapd, s); break;
  }
}
template void launch_det_lap<float>(const OrbSrc<float>&, double*, double*, double*, double*, double*, float*,
                                          const Shape&, hipStream_t);
template void launch_det_lap<double>(const OrbSrc<double>&, double*, double*, double*, double*, double*, float*,
                                           const Shape&, hipStream_t);

}  // namespace dwmi
