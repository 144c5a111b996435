// FP64 GEMM  C[M, N] = epi(A[M, K] * Bt[N, K]^T)  on v_mfma_f64_16x16x4f64 (the FP64 form of every pass).
#include "common.h"
#include "gemm_epi.h"
#include "kernels.h"

namespace dwmi {

// ------------------------------------------------------------------------------------------------
// Tile (32 WM) x (32 WN) per 256-thread workgroup; 4 waves in 2 x 2, each wave owns WM x WN blocks of 16 x 16.
// Both operand slices (16 k) are staged in LDS, two buffers and one barrier per slice; MFMA step s of lane group
// g = lane / 16 takes k = 4 s + g, so that an element is one chain over k ascending, as a VALU kernel forms it (in another
// order ill-conditioned walkers' E_loc differ in the last bit, 1 of 500 at 42 electrons).  Element k of a row lies at
// 4 (k % 4) + k / 4: a lane reads its operands of a slice as two 16-byte vectors per block (row pitch 18 doubles: the 16
// rows of a read start 4 banks apart).  A block's step takes the matrix
// core 64 cycles and needs 16 bytes per lane from LDS for WM + WN blocks of operands, so the matrix core bounds
// it (a VALU tile of 4 x 4 per thread waited on LDS: 64 bytes per 16 multiply-adds).  172,032 x 320 x 256 (256
// walkers of 14 electrons, Laplacian pass): 1160 us with the VALU tile, 533 us with this (53 TFLOP/s; 60 without
// the V epilogue; the card's large FP64 product reaches 68).
// ------------------------------------------------------------------------------------------------
template <int FLAGS, int WM, int WN>
__global__ __launch_bounds__(256) void k_gemm_f64(const double* __restrict__ A, int lda, const double* __restrict__ Bt,
                                                  int ldb, double* __restrict__ Cm, int ldc, int M, int N, int K,
                                                  int tilesN, int tilesTotal, GemmEpiD ep) {
  constexpr int BM = 32 * WM, BN = 32 * WN, BK = 16, PITCH = BK + 2;
  constexpr int AIT = BM * 8 / 256, BIT = BN * 8 / 256;  // double2 per thread and slice
  __shared__ __align__(16) double As[2][BM][PITCH];
  __shared__ __align__(16) double Bs[2][BN][PITCH];
  const int tile = tile_index(blockIdx.x, tilesTotal);
  if (tile >= tilesTotal) return;  // uniform over the workgroup, before any barrier
  const long row0 = (long)(tile / tilesN) * BM;
  const int col0 = (tile % tilesN) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid >> 1, wn = wid & 1, g = lane >> 4, cl = lane & 15;

  v4d acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  typedef double v2d __attribute__((ext_vector_type(2)));
  v2d ra[AIT], rb[BIT];
  auto gload = [&](int k0) {
#pragma unroll
    for (int it = 0; it < AIT; ++it) {
      const int idx = tid + 256 * it;
      long gr = row0 + (idx >> 3);
      if (gr > M - 1) gr = M - 1;
      ra[it] = *(const v2d*)(A + gr * lda + k0 + (idx & 7) * 2);
    }
#pragma unroll
    for (int it = 0; it < BIT; ++it) {
      const int idx = tid + 256 * it;
      rb[it] = *(const v2d*)(Bt + (long)(col0 + (idx >> 3)) * ldb + k0 + (idx & 7) * 2);
    }
  };
  const int at = 8 * (tid & 1) + ((tid & 7) >> 1);  // place of k = 2 (tid % 8); k + 1 lies 4 further
  auto sstore = [&](int buf) {
#pragma unroll
    for (int it = 0; it < AIT; ++it) {
      As[buf][(tid + 256 * it) >> 3][at] = ra[it][0];
      As[buf][(tid + 256 * it) >> 3][at + 4] = ra[it][1];
    }
#pragma unroll
    for (int it = 0; it < BIT; ++it) {
      Bs[buf][(tid + 256 * it) >> 3][at] = rb[it][0];
      Bs[buf][(tid + 256 * it) >> 3][at + 4] = rb[it][1];
    }
  };

  const int S = K / BK;
  gload(0);
  sstore(0);
  if (S > 1) gload(BK);
  for (int sl = 0; sl < S; ++sl) {
    const int buf = sl & 1;
    __syncthreads();  // slice sl is staged, and every read of the other buffer (slice sl - 1) is done
    v2d b[WN][2];
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) b[j][h] = *(const v2d*)&Bs[buf][wn * 16 * WN + j * 16 + cl][4 * g + 2 * h];
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      v2d a[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) a[h] = *(const v2d*)&As[buf][wm * 16 * WM + i * 16 + cl][4 * g + 2 * h];
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int j = 0; j < WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[st >> 1][st & 1], b[j][st >> 1][st & 1], acc[i][j], 0, 0, 0);
      if (i == 0 && sl + 1 < S) {
        sstore(buf ^ 1);
        if (sl + 2 < S) gload((sl + 2) * BK);
      }
    }
  }
  // result layout of the FP64 block: lane l, element e holds row 4 e + l / 16, column l % 16
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = (int)row0 + wm * 16 * WM + i * 16 + 4 * e + g;
        const int c = col0 + wn * 16 * WN + j * 16 + cl;
        if (r < M && c < N) epi_store<FLAGS, double>(acc[i][j][e], r, c, Cm, ldc, ep);
      }
}

template <int FLAGS, int WM, int WN>
static void launch_f64(const double* A, int lda, const double* Bt, int ldb, double* C, int ldc, int M, int N, int K,
                       const GemmEpiD& ep, hipStream_t s) {
  const int tilesN = (N + 32 * WN - 1) / (32 * WN), total = (M + 32 * WM - 1) / (32 * WM) * tilesN;
  hipLaunchKernelGGL((k_gemm_f64<FLAGS, WM, WN>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, A, lda, Bt, ldb, C, ldc,
                     M, N, K, tilesN, total, ep);
}

template <int FLAGS>
static void dispatch_f64(const double* A, int lda, const double* Bt, int ldb, double* C, int ldc, int M, int N, int K,
                         const GemmEpiD& ep, hipStream_t s) {
  // 64 x 64 tiles once they give every CU two workgroups, 32 x 32 below that (latency: more workgroups).
  // 172,032 x 320 x 256: 468 us with 64 x 64, 565 with 128 x 64, 587 with 128 x 128; 3,584 x 320 x 256: 19.9 us
  // with 64 x 64, 17.3 with 32 x 32.
  if (((long)M + 63) / 64 * ((N + 63) / 64) >= 512)
    launch_f64<FLAGS, 2, 2>(A, lda, Bt, ldb, C, ldc, M, N, K, ep, s);
  else
    launch_f64<FLAGS, 1, 1>(A, lda, Bt, ldb, C, ldc, M, N, K, ep, s);
}

void gemm_f64(const double* A, int lda, const double* Bt, int ldb, double* C, int ldc, int M, int N, int K,
              const GemmEpiD& ep, hipStream_t s) {
  if (M <= 0 || N <= 0) return;
  // the passes' epilogues: none (orbitals, gradients), bias (spin-mean part), V (pre-activations of the Laplacian
  // pass); the rest is tested at run time inside epi_store
  const int flags = (ep.bias ? EPI_BIAS : 0) | (ep.V ? EPI_V : 0) | (ep.act_tanh ? EPI_TANH : 0) |
                    (ep.permute ? EPI_PERM : 0);
  switch (flags) {
    case 0: dispatch_f64<0>(A, lda, Bt, ldb, C, ldc, M, N, K, ep, s); break;
    case EPI_BIAS: dispatch_f64<EPI_BIAS>(A, lda, Bt, ldb, C, ldc, M, N, K, ep, s); break;
    case EPI_V: dispatch_f64<EPI_V>(A, lda, Bt, ldb, C, ldc, M, N, K, ep, s); break;
    default: dispatch_f64<EPI_BIAS | EPI_V | EPI_TANH | EPI_PERM>(A, lda, Bt, ldb, C, ldc, M, N, K, ep, s); break;
  }
}

}  // namespace dwmi
