// Laplacian-mode determinants (FP64), in two launches: log|det|, sign and M^-1 per matrix,
// then the channel passes
//   Y_k = M^-1 dM_k,  g_k = tr Y_k,  q_k = tr(Y_k^2),  Lap log|det| = tr(M^-1 Lap M) - sum_k q_k.
// Both read the orbitals O and apply the envelope themselves, so the product envelope x orbitals (3 n + 2 matrices per
// determinant) is never stored.
//
// 16,384 matrices of 26 (1024 walkers): 4.17 ms for the determinants and 1.99 ms for the stored product before, 0.73 ms
// (inverses) + 2.06 ms (channels; 2.30 in the old order of sums) here; 3,072 matrices of 42: 0.70 + 1.94 (2.13) ms; 32,768
// matrices of 14: 1.14 ms (one wavefront per matrix) before, 0.13 + 0.50 (0.60) ms here.  Above 16 electrons the channel
// passes run at half the FP64 matrix rate, padding to 16 x 16 blocks counted.
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
// Sums over the wavefront's lanes, in every lane; lanes paired as in wave_sum_d (xor 32, 16, 8, 4, 2, 1), without LDS.
// After xor 8 the 16 lanes of a row hold 8 values twice, so a rotation by 4 meets the lane that xor 4 does; and so on.
template <int CTRL>
__device__ __forceinline__ double row_ror(double v) {
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + CTRL, 0xF, 0xF, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ double row_sum_dpp(double v) {
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += row_ror<2>(v);
  v += row_ror<1>(v);
  return v;
}
// v_permlane32_swap(a, b): the low halves of a and b, and their high halves; the sum of the two holds a's sum over xor 32
// in the low half and b's in the high one.  v_permlane16_swap does the same for neighbouring rows of 16.
__device__ __forceinline__ double fold32(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ __forceinline__ double wave_sum_dpp(double v) {
  v = fold32(v, v);
  return row_sum_dpp(fold16(v, v));
}
// Four sums at once: rows of 16 lanes get v0's, v2's, v1's and v3's.
__device__ __forceinline__ double wave_sums_dpp(double v0, double v1, double v2, double v3) {
  return row_sum_dpp(fold16(fold32(v0, v1), fold32(v2, v3)));
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
// Column-parallel elimination and substitution: a step reads one broadcast and one own element (eight steps' reads in
// flight) and every element is one chain, in the order of a row-by-row elimination, so a matrix is about n^2 pipelined LDS
// steps.  3,072 matrices of 42: 0.70 ms (a workgroup of 256 threads, with barriers per elimination step and 42 busy lanes in
// the substitution, took several times that).
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
    if (act && j > p) T[j * P + p] /= T[p * P + p];  // multiplier of row j
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
      double y = (perm[p] == j) ? 1.0 : 0.0;
#pragma unroll 8
      for (int q = 0; q < p; ++q) y -= T[p * P + q] * X[q * P + j];
      X[p * P + j] = y;
    }
    for (int p = n - 1; p >= 0; --p) {
      double y = X[p * P + j];
#pragma unroll 8
      for (int q = p + 1; q < n; ++q) y -= T[p * P + q] * X[q * P + j];
      X[p * P + j] = y / T[p * P + p];
    }
#pragma unroll 4
    for (int p = 0; p < n; ++p) {
      const double x = X[p * P + j];
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
// as A operand (registers for NB <= 2) and dM_k[16 K + g + 4 q][16 J + c] as B operand, read from O with the envelope
// applied (tables of the envelope and of the own-electron terms in LDS); the next channel's O is loaded before this
// channel's products.  tr(Y^2) = sum_IJ Y_IJ o (Y_JI)^T: blocks are transposed through wave-private LDS tiles instead
// of being computed a second time as (dM^T M^-T), so a channel is NB^3 x 4 MFMAs of 64 cycles, half of what two
// products take.
//
// KEEP, order of the sums (an ill-conditioned walker's E_loc, and with it the FP64 loss, turns a rounding here into a last
// bit; the loss and every form that was there before the split one keep it): lane l of block (I, J) forms
// s_IJ = sum_e Y_IJ[4 e + g][c] Y_JI[c][4 e + g]; a chain per lane (NB <= 2) or
// per lane and J (NB > 2) adds them channel by channel, (I, J) in order, then the lanes meet.  The channels of a round
// lie in different waves, so they leave their s_IJ in LDS and every wave continues a part of the chains: a barrier or two
// a round of 4 channels (16 for NB = 1, whose channels are short).  tr Y is one chain of the operands' products per lane.
// Otherwise (energies of the split form, whose channels are rounded in another way already) each wave adds up its own
// channels, off-diagonal pairs once and doubled, tr Y from the diagonal that the transposition tile holds: 16,384 matrices of
// 26 2.06 ms against 2.30, 3,072 of 42 1.94 against 2.13, 32,768 of 14 0.50 against 0.60.
// ------------------------------------------------------------------------------------------------
template <int NB, bool KEEP>
constexpr int chan_region() {  // doubles of LDS per wave: transposition tiles, behind or over them the s_IJ of a round
  return !KEEP ? 16 * 17 : NB == 1 ? 16 * 17 + 4 * 64 : NB == 2 ? 16 * 17 + 2 * 4 * 64 : NB * NB * 64;
}

template <int NB, typename TA, bool KEEP>
__global__ __launch_bounds__(256, NB == 1 ? 6 : NB == 4 ? 1 : (NB == 2 && sizeof(TA) == 4 ? 3 : 2)) void k_det_chan(OrbSrc<TA> src, Shape sh,
                                                                               const double* __restrict__ Minv,
                                                                               double* __restrict__ g,
                                                                               double* __restrict__ lapd, int nmat) {
  extern __shared__ double sm[];
  constexpr int NP = 16 * NB, PM = NP + 1, REGION = chan_region<NB, KEEP>(), RC = NB == 1 && KEEP ? 4 : 1, NT = NB * NB;
  constexpr bool TWO = NB == 2;  // two buffers of s_IJ: one barrier a round
  const int n = sh.n, nd = 3 * n, C = sh.C;
  double* sM = sm;                        // M^-1, NP x PM, zero outside n x n
  double* sT = sM + NP * PM;              // 4 x REGION; before the rounds the Laplacian channel, n rows of NP
  double* red = sT + 4 * REGION;          // 32
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

  TA* const sL = (TA*)sT;
  double tp = 0.0;  // tr(M^-1 Lap M); KEEP: a row of M^-1 per lane, or elements 256 apart per thread
  for (int e = tid; e < NP * NP; e += 256) {
    const int i = e / NP, c = e - (e / NP) * NP;
    sM[i * PM + c] = (i < n && c < n) ? Minv[(long)bd * n * n + i * n + c] : 0.0;
  }
  if constexpr (!KEEP) __syncthreads();
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
      if constexpr (KEEP)
        sL[e] = lp;
      else
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
  if constexpr (KEEP && NB <= 2) {
    if (tid < n)
      for (int e = 0; e < n; ++e) tp += sM[tid * PM + e] * (double)sL[e * NP + tid];
  } else if constexpr (KEEP) {
    for (int e = tid; e < n * n; e += 256) {
      const int a = e / n, q = e - (e / n) * n;
      tp += sM[a * PM + q] * (double)sL[q * NP + a];
    }
  }
  if constexpr (KEEP) __syncthreads();  // sL has been read

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
  double* const T = sT + wv * REGION;
  // s_IJ of channel c of a wave's round: 64 lanes at this place in its region
  constexpr int S0 = NB <= 2 ? 16 * 17 : 0;
  int buf = 0;
  constexpr bool AHEAD = sizeof(TA) == 4;  // FP64 orbitals: no registers for a second channel
  double qacc = 0.0;  // KEEP: NB <= 2, chain of lane 16 wv + lane (lanes 0 to 15); NB > 2, chain of (J = wv, lane)
  if (AHEAD && wv < nd) load(wv);
  for (int k0 = 0; k0 < nd; k0 += 4 * RC) {  // every wave takes every round (KEEP's barriers)
    double gp[4];  // NB > 2: tr Y's chains
    gp[3] = 0.0;
#pragma unroll
    for (int rc = 0; rc < RC; ++rc) {
      const int k = k0 + 4 * rc + wv;
      if (k >= nd) break;  // uniform over the wave
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
      double st[NT], t = 0.0;  // t: tr Y, the operands' products over (I, K, q); above 32 electrons a chain for each I
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int J = I; J < NB; ++J) {
          v4d y = {0.0, 0.0, 0.0, 0.0}, z = y;
          if (KEEP && NB > 2 && J == I) t = 0.0;
#pragma unroll
          for (int K = 0; K < NB; ++K)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              y = __builtin_amdgcn_mfma_f64_16x16x4f64(mia(I, K, q), dm[K][J][q], y, 0, 0, 0);
              if (J > I) z = __builtin_amdgcn_mfma_f64_16x16x4f64(mia(J, K, q), dm[K][I][q], z, 0, 0, 0);
              if (KEEP && J == I) t += mia(I, K, q) * dm[K][I][q];
            }
          if constexpr (KEEP && NB > 2)
            if (J == I) gp[I] = t;
          // lane l, element e: row 4 e + g, column c of the block (LDS accesses of one wave stay in order)
          auto against = [&](double* tile, const v4d& a, const v4d& other) {
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[(4 * e + gq) * 17 + cl] = other[e];
            v4d w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = tile[cl * 17 + 4 * e + gq];
            return a[0] * w[0] + a[1] * w[1] + a[2] * w[2] + a[3] * w[3];
          };
          if constexpr (!KEEP) {
            if (J == I) {
              qacc += against(T, y, y);
              t += T[cl * 18];
            } else {
              qacc += 2.0 * against(T, y, z);
            }
          } else if (J == I) {
            st[I * NB + I] = against(T, y, y);
          } else {
            st[I * NB + J] = against(T, y, z);
            st[J * NB + I] = against(T + (NB > 2 ? 16 * 17 : 0), z, y);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      if constexpr (!KEEP) {
        const double g_k = row_sum_dpp(t);
        if (lane == 0) g[(long)bd * nd + k] = g_k;
        continue;
      }
#pragma unroll
      for (int x = 0; x < NT; ++x) T[S0 + buf + (rc * NT + x) * 64 + lane] = st[x];  // over the tiles (NB > 2), now read
      if constexpr (NB <= 2) {
        const double s = wave_sum_dpp(t);
        if (lane == 0) g[(long)bd * nd + k] = s;
      } else {
        const double s = wave_sums_dpp(gp[0], gp[1], gp[2], gp[3]);
        const double s0 = readlane_d(s, 0), s1 = readlane_d(s, 32), s2 = readlane_d(s, 16), s3 = readlane_d(s, 48);
        if (lane == 0) g[(long)bd * nd + k] = ((s0 + s1) + s2) + s3;
      }
    }
    if constexpr (!KEEP) continue;
    __syncthreads();  // every wave's s_IJ of the round are in LDS
    const int nc = min(4 * RC, nd - k0);
    if constexpr (NB <= 2) {
      if (lane < 16)
        for (int c = 0; c < nc; ++c) {
          const double* p = sT + (c & 3) * REGION + S0 + buf + (c >> 2) * NT * 64 + 16 * wv + lane;
#pragma unroll
          for (int x = 0; x < NT; ++x) qacc += p[64 * x];
        }
    } else if (wv < NB) {
      for (int c = 0; c < nc; ++c) {
        const double* p = sT + c * REGION + wv * 64 + lane;
#pragma unroll
        for (int I = 0; I < NB; ++I) qacc += p[I * NB * 64];
      }
    }
    if constexpr (TWO)
      buf ^= NT * 64;
    else
      __syncthreads();  // and have been read
  }
  if constexpr (KEEP && NB <= 2) {  // the 64 chains to the lanes of wave 0
    if (lane < 16) sT[16 * wv + lane] = qacc;
    __syncthreads();
    if (wv == 0) {
      const double q = wave_sum_d(sT[lane]);
      tp = wave_sum_d(tp);
      if (lane == 0) lapd[bd] = tp - q;
    }
  } else {
    qacc = block_sum_d(qacc, red);
    tp = block_sum_d(tp, red + 16);
    if (tid == 0) lapd[bd] = tp - qacc;
  }
}

template <int NB, typename TA, bool KEEP>
static void launch_chan(const OrbSrc<TA>& src, const Shape& sh, const double* Minv, double* g, double* lapd,
                        hipStream_t s) {
  constexpr int NP = 16 * NB;
  const size_t shm = (size_t)(NP * (NP + 1) + 4 * chan_region<NB, KEEP>() + 32) * sizeof(double) +
                     ((size_t)NP * NP + (NB < 4 || sizeof(TA) == 4 ? 3 * NP * NP : 4 * NP)) * sizeof(TA);
  if (shm > 65536)
    (void)hipFuncSetAttribute((const void*)k_det_chan<NB, TA, KEEP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
  const int nmat = sh.B * sh.D;
  hipLaunchKernelGGL((k_det_chan<NB, TA, KEEP>), dim3((nmat + 7) / 8 * 8), dim3(256), shm, s, src, sh, Minv, g, lapd, nmat);
}

template <typename TA, bool KEEP>
static void dispatch_chan(const OrbSrc<TA>& src, const Shape& sh, const double* Minv, double* g, double* lapd, hipStream_t s) {
  switch ((sh.n + 15) / 16) {
    case 1: launch_chan<1, TA, KEEP>(src, sh, Minv, g, lapd, s); break;
    case 2: launch_chan<2, TA, KEEP>(src, sh, Minv, g, lapd, s); break;
    case 3: launch_chan<3, TA, KEEP>(src, sh, Minv, g, lapd, s); break;
    default: launch_chan<4, TA, KEEP>(src, sh, Minv, g, lapd, s); break;
  }
}

template <typename TA>
void launch_det_lap(const OrbSrc<TA>& src, double* Minv, double* ld, double* sd, double* g, double* lapd,
                          float* dcond, const Shape& sh, bool keep_order, hipStream_t s) {
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
  if constexpr (sizeof(TA) == 4) {
    if (!keep_order) {
      dispatch_chan<TA, false>(src, sh, Minv, g, lapd, s);
      return;
    }
  }
  dispatch_chan<TA, true>(src, sh, Minv, g, lapd, s);
}
template void launch_det_lap<float>(const OrbSrc<float>&, double*, double*, double*, double*, double*, float*,
                                          const Shape&, bool, hipStream_t);
template void launch_det_lap<double>(const OrbSrc<double>&, double*, double*, double*, double*, double*, float*,
                                           const Shape&, bool, hipStream_t);

}  // namespace dwmi
