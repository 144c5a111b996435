// Launchers of the dwmi device kernels (definitions in gemm.hip and wf_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dwmi {

// Epilogue of the batched-row GEMM  C[M, N] = A[M, K] * Bt[N, K]^T.
template <typename T>
struct GemmEpiT {
  const T* bias = nullptr;      // + bias[col] on rows with row % C == 0 (value channel)
  const T* V = nullptr;         // + V[((row / nC) * C + row % C) * ldv + col]   (per-walker broadcast)
  int ldv = 0;
  int C = 1;                    // channels per electron
  int nC = 1;                   // n_el * C
  int act_tanh = 0;             // y = tanh(.)  (value-only forward)
  int permute = 0;              // output rows go to spin-major order (up block, then down block)
  int n = 0, u = 0, B = 0;      // shape for `permute`
  int vsplit = 1;               // V is the sum of vsplit partial buffers V + s * vstride
  long vstride = 0;
  int tile = -1;                // FP32 tile: -1 = heuristic, 0 = 64x64, 1 = 64x128, 2 = 128x128,
                                // 4 = 112x256 (N = 256, no split-K; else 64x64)
  int ksplit = 1;               // split K over ksplit partial outputs C + s * cstride (bias on s = 0 only)
  long cstride = 0;
};
using GemmEpi = GemmEpiT<float>;
using GemmEpiD = GemmEpiT<double>;

enum GemmPrec { GEMM_F32 = 0, GEMM_BF16X3 = 1, GEMM_BF16 = 2, GEMM_F64 = 3 };

// Operands: A row-major [M, lda] fp32, Bt row-major [>= pad128(N), ldb] fp32 (rows beyond N are zero),
// K a multiple of 32, lda/ldb multiples of 4.  For the BF16 forms, `Bhi`/`Blo` are the pre-split BF16
// weights with the same layout as Bt.
void gemm(GemmPrec prec, const float* A, int lda, const float* Bt, const uint16_t* Bhi, const uint16_t* Blo,
          int ldb, float* C, int ldc, int M, int N, int K, const GemmEpi& ep, hipStream_t s);

// FP64 form (FP64 MFMA, gemm_f64.hip).  Same operand conventions; K a multiple of 16.
void gemm_f64(const double* A, int lda, const double* Bt, int ldb, double* C, int ldc, int M, int N, int K,
              const GemmEpiD& ep, hipStream_t s);

// B walkers, n electrons (u up), I ions, D dets, C channels per electron (1, or 3 n + 2 in the
// Laplacian pass) stored in Cp rows (C, or pad16(C) in the Laplacian pass), widths W1 / W2, L iterations.
struct Shape {
  int B, n, u, I, D, C, Cp, W1, W2, L;
};

// Fused 1-el GEMM + tanh forward-Laplacian rule of the Laplacian pass (rows: Cp per electron).
// E_override > 0 sets the electrons per workgroup (E * Cp / 16 <= 12); 0 picks lap_electrons_per_tile:
// FP32 min(4, 192 / Cp), BF16 forms 96 / Cp (at least 1).
// cols = 256 asks for 256-column tiles (FP32 form, E * Cp <= 96); otherwise 128.  Bt: FP32 (and gemm_value16) in lane
// order (launch_lane_pack), BF16 forms the parts of launch_split_pack; K a multiple of 32.
void gemm_lap(GemmPrec prec, const float* X, int ldx, const float* Bt, int K,
              const float* V, int ldv, float* out, int ldo, int permute, const Shape& sh, int E_override, int cols,
              hipStream_t s);
int lap_electrons_per_tile(int Cp, GemmPrec prec);

// FP32 GEMMs on 16-bit MFMA with both operands split into three BF16 or two FP16 parts (gemm_split.hip).  P: weights
// Bt [rows, K] (row = output column, columns at or past `cols` zero) packed by launch_split_pack into
// split_pack_bytes(cols, K) bytes; K a multiple of 32.
size_t split_pack_bytes(int cols, int K);
void launch_split_pack(const float* Bt, int ldb, int cols, int K, void* out, hipStream_t s);
// The same weights as two FP16 parts of each column times 2^shift (K columns from Bt, split_pack16_bytes(cols, K) bytes); the
// columns' shifts are put at split_pack16_shifts before.
size_t split_pack16_bytes(int cols, int K);
int* split_pack16_shifts(void* P16, int cols, int K);
void launch_split_pack16(const float* Bt, int ldb, int cols, int K, void* out, hipStream_t s);
// C[M, N] = A[M, K] B for rows of electrons (16 rbe rows each), K a multiple of 64, B in FP16 parts.  amax: np per-wave
// maxima of each electron's A rows, ms apart.  tile: -1 chosen by size, 0 = 48 x 128, 1 or 2 = 96 x 256 (results do not
// depend on it).
void split_gemm(const float* A, int lda, const void* P16, const float* amax, int np, int ms, int rbe, float* C,
                int ldc, int M, int N, int K, int tile, hipStream_t s);
// V[(b Cp + ch), o] of the derivative channels: spin means of X's first Kh columns times W_mu (no bias), from three BF16 parts
// of each (FP32 accuracy); false, launching nothing, where the batch is too small to gain against launch_spin_mean and
// split_mean_product (V = MU times W_mu, the same sums).
bool split_mean(const float* X, int Kx, int Kh, const void* P, int Km, float* V, int ldv, const Shape& sh, hipStream_t s);
void split_mean_product(const float* MU, int Km, const void* P, float* V, int ldv, const Shape& sh, hipStream_t s);
// The same for the BF16x3 form, all channels and the bias, bit-equal to launch_spin_mean and its GEMM; false, launching
// nothing, where the batch is too small to gain.
bool mean_bf16x3(const float* X, int Kx, int Kh, const void* P, int Km, const float* bias, float* V, int ldv, const Shape& sh,
                 hipStream_t s);
// 1-el GEMM and tanh forward-Laplacian rule of the derivative channels; `out` holds the value channel already.  With
// amax (np maxima per electron, W1 / 32 apart, covering all but the last `tail` <= 2 slices of 32 columns; K a multiple of 64)
// P is in FP16 parts, without it in BF16 parts.  omax (W1 / 32 places per electron, in the order of out's rows) receives the maxima
// of the derivative channels written, one per wave: returns their number per electron (0: shape not supported).  E_max
// > 0 / cols = 128 ask for the smaller tiles (results do not depend on them).
int split_lap(const float* X, int ldx, const void* P, int K, const float* amax, int np, int tail,
              const float* V, int ldv, float* out, int ldo, float* omax, int permute, const Shape& sh, int E_max,
              int cols, hipStream_t s);

// One-launch value layers and orbital GEMMs for small batches (value_layer.hip), bit-equal to the separate kernels.
// Weights in lane order (launch_lane_pack: Bt [rows >= cols, K] into lane_pack_bytes(cols, K) bytes, K a multiple of
// 32).  value_layer: out = tanh(X W + V), V = the vs K parts of (spin means of the first Kh columns) W_mu plus bias,
// added in order; rows of X ldx apart, of out ldo apart.  All return false, launching nothing, where the batch is too
// large to gain (the rules stand beside them).
size_t lane_pack_bytes(int cols, int K);
void launch_lane_pack(const float* Bt, int ldb, int cols, int K, void* out, hipStream_t s);
bool value_layer(const float* X, long ldx, int K, int Kh, const void* W, const void* Wmu, int Km, const float* bias,
                 int vs, float* out, long ldo, int permute, int B, int n, int u, int W1, hipStream_t s);
// value_net: L consecutive value layers in one launch (W1 = 256; layers after the first take their first Kt = 256
// columns from the one before and the rest from X); out may be null for all but the last layer, the only one that
// `permute` applies to.
struct ValueNetLayer {
  const float* X;
  long ldx;
  const void *W, *Wmu;
  const float* bias;
  float* out;
  long ldo;
  int K, Km, Kh, Kt, vs;
};
constexpr int DW_MAX_LAYERS = 8;
bool value_net(const ValueNetLayer* layers, int L, int permute, int B, int n, int u, int W1, hipStream_t s);
bool value_orbitals(const float* H, long ldh, int K, const void* W_up, const void* W_dn, float* O, long ldo,
                    int up_rows, int dn_rows, int N, hipStream_t s);

// Value-pass 1-el GEMM on the Laplacian GEMM's 16x16 MFMA main loop (FP32): out = tanh(X W + V[walker]),
// V summed over vsplit parts vstride apart; permute sends rows to spin-major order.
void gemm_value16(const float* X, int ldx, const float* Bt, int K, const float* V, int ldv, int vsplit, long vstride,
                  float* out, int ldo, int permute, const Shape& sh, hipStream_t s);

// Laplacian-pass per-walker GEMM with the spin means of X's h columns formed in LDS (FP32):
// V[r, o] = sum_k MU[r, k] Wmu[o, k] + bias[o] on value-channel rows, equal to launch_spin_mean followed by
// the bias-only gemm on MU.  Returns false, launching nothing, unless W1 == 256, Km >= 256, Km % 16 == 0 and
// Kh, Kx are multiples of 4 (C > 1).
bool gemm_mean_lap(const float* X, int Kx, int Kh, const float* Wmu, int Km, const float* bias, float* V, int ldv,
                   const Shape& sh, hipStream_t s);

// Layer-0 input rows: the el-ion features in columns [0, 4 I); the columns [tail0, tail0 + tailw) are left
// to the 2-el kernels for the real channel rows; every other column and padding row is zero.  With normals
// (and the device chain record), the rows are those of the Gaussian proposal r + stepsize * normals, which is
// also written to r_out.
template <typename T>
void launch_features0(const float* r, const float* R, T* X0, int Kx0, int tail0, int tailw, const Shape& sh,
                      hipStream_t s, const float* normals = nullptr, const void* chain = nullptr,
                      float* r_out = nullptr);
template <typename T>
void launch_twoel(const float* r, T* const* X, const int* Kx, const int* Kh, const T* W2e, const T* b2e,
                  const Shape& sh, hipStream_t s);
template <typename T>
void launch_spin_mean(const T* X, int Kx, int Kh, T* MU, int Km, const Shape& sh, hipStream_t s);
template <typename T>
void launch_tanh_rule(const T* Z, T* out, int ldo, int permute, const Shape& sh, hipStream_t s);
template <typename T>
void launch_envelope(const T* O, int ldo, const float* r, const float* R, const T* kappa, const T* wenv, T* A,
                     const Shape& sh, hipStream_t s);
// Orbitals and envelope parameters as the determinant kernels read them when they apply the envelope
// themselves (det_reads_orbitals): O holds spin-major rows (Cp per electron, ldo columns).
template <typename T>
struct OrbSrc {
  const T* O;
  int ldo;
  const float* r;
  const float* R;
  const T* kappa;
  const T* wenv;
};
// True when the determinant kernels for n electrons and C channels apply the envelope while reading O
// (no envelope launch, no stored product); otherwise launch_envelope fills A first.
inline bool det_reads_orbitals(int n, int C) { return C > 1 || n <= 32; }
// Doubles of inverse matrices that launch_det needs as scratch (`minv`): the Laplacian pass.
inline size_t det_inverse_elems(long matrices, int n, int C) {
  return C > 1 ? (size_t)matrices * n * n : 0;
}
// Outputs of the value-pass combine (launch_combine's, C == 1) when launch_det runs it itself.
struct CombineValue {
  float* out_lp;
  float* out_phase;
  uint32_t* out_flags;
  float* out_kappa;
  float cond_thr;
  int fuse;  // set by launch_det
};
// Returns true when it also ran the value-pass combine for `combine` (value pass, n <= 32, D dividing the
// determinants per workgroup); the caller then skips launch_combine.
template <typename TA>
bool launch_det(const TA* A, const OrbSrc<TA>& src, double* minv, double* ld, double* sd, double* g, double* lapd, float* dcond,
                const Shape& sh, hipStream_t s, const CombineValue* combine = nullptr, bool keep_order = true);
// Its part for the Laplacian pass (det_lap.hip, which says what keep_order keeps).
template <typename TA>
void launch_det_lap(const OrbSrc<TA>& src, double* minv, double* ld, double* sd, double* g, double* lapd,
                          float* dcond, const Shape& sh, bool keep_order, hipStream_t s);
void launch_combine(const double* ld, const double* sd, const double* g, const double* lapd, const float* dcond,
                    float cond_thr, const float* r, const float* R, const float* Z, float* out_lp, float* out_phase,
                    float* out_eloc, uint32_t* out_flags, float* out_kappa, const Shape& sh, hipStream_t s);

void launch_fill_i32(int32_t* p, int32_t v, int count, hipStream_t s);
// JAX threefry streams (threefry.hip)
void launch_threefry_split(const uint32_t* key, int num, uint32_t* out, hipStream_t s);
void launch_threefry_normal(const uint32_t* key, long count, float* out, hipStream_t s);
void launch_threefry_mcmc(const uint32_t* keys_in, uint32_t* keys_out, int B, int n, int n_steps, float* normals,
                          float* uniforms, hipStream_t s);
// out[0] = nanmean(e[0:n]), out[1] = nanmean(|e - out[0]|^2), FP64, deterministic order.
void launch_energy_moments(const float* e, int n, double* out, hipStream_t s);
// Clipped-energy statistics and per-walker gradient weights (optimization/loss_function.py:12-110); one
// workgroup.  A median center needs n <= clip_max_walkers().
int clip_max_walkers();
void launch_clip_energies(const float* e, int n, int tanh_clip, int median, int mae, double clip_by,
                          int from_previous, const double* state_in, float* weights, float* eclip, double* stats,
                          hipStream_t s);
// ---- dpe4 embedding (csrc/dpe4.hip) ----
constexpr int MAXL_DPE4 = 4;  // iterations
// Pair streams: wm[l][b][i][j][ch][f] (ch: value, d/dd (3), total Laplacian in the Laplacian pass).
// Wp [2L-1][2][32][32], bp [2L-1][2][32]: the maps of iterations 0..L-1, then the stream layers.
template <typename T>
void launch_dpe4_pairs(const float* r, const T* Wp, const T* bp, T* wm, const Shape& sh, hipStream_t s);
// El-ion stream: e_ei of every iteration into X[l] columns tail[l] + 32 ...; him: scratch [L][I][32].
template <typename T>
void launch_dpe4_elion(const float* r, const float* R, const float* Z, const T* Wei, const T* bei, const T* Whim,
                       const T* bhim, const T* table, int n_types, int z_min, T* him, T* const* X, const int* Kx,
                       const int* tail, const Shape& sh, hipStream_t s);
// hm [B n Cp][32] = tanh rule of (hm + bias) over each electron's channel rows, in place.
// h_map with its tanh rule in one launch (FP32; Wt [32, K], rows = output columns); false, launching nothing, for shapes
// it does not take (K a multiple of 16 up to 512, Cp <= 192).
bool launch_dpe4_hmap(const float* X, int ldx, const float* Wt, int K, const float* bias, float* hm, const Shape& sh,
                      hipStream_t s);
template <typename T>
void launch_dpe4_tanh(T* hm, const T* bias, const Shape& sh, hipStream_t s);
// e_ee of one iteration from wm (that iteration's slice) and hm into X columns col0 .. col0 + 31.
template <typename T>
void launch_dpe4_conv(const T* wm, const T* hm, T* X, int Kx, int col0, const Shape& sh, hipStream_t s);

void launch_gather_walkers(const float* r, const int32_t* idx, int count, int n, float* out, hipStream_t s);
void launch_scatter_values(const float* v, const int32_t* idx, int count, float* out, hipStream_t s);
void launch_propose(const float* r, const float* normals, const void* chain, float* r_prop, int count, hipStream_t s);
// Local-stepsize (kind DW_PROPOSAL_LOCAL) and approximate-Langevin (DW_PROPOSAL_LANGEVIN) proposals
// (mcmc.py:218-236, 255-284): r_prop [B, n, 3] and the per-walker log proposal ratio logq [B].  n <= 64.
void launch_propose_scaled(int kind, const float* r, const float* normals, const void* chain, const float* R,
                           const float* Z, int I, float r_min, float r_max, float lscale, float* r_prop, float* logq,
                           int B, int n, hipStream_t s);
// One-electron moves (DW_PROPOSAL_NORMAL_ONE_EL / DW_PROPOSAL_LOCAL_ONE_EL, mcmc.py:183-192, 239-252): electron
// step_nr mod n moves by xi [B, 3]; logq [B] written by the local form only.
void launch_propose_one_el(int kind, const float* r, const float* xi, const void* chain, const float* R, int I,
                           float r_min, float r_max, float* r_prop, float* logq, int B, int n, hipStream_t s);
// logq (may be null for a symmetric proposal) is added to the exponent: accept iff exp(lp' - lp + logq) > u.
// The step's accepted walkers are added to *acc_count; the last workgroup (by *ticket, which must be zero
// on entry) then updates the chain record: step_nr, acc_rate and, every `interval` steps, the stepsize from
// the previous acc_rate, clipped to [lo, hi]; out_acc (may be null) receives the step's acceptance.
void launch_accept(float* r, const float* r_prop, float* lp, const float* lp_prop, const float* logq,
                   const float* uniforms, int32_t* age, int max_age, int32_t* acc_count, uint32_t* flags, int B,
                   int n, void* chain, int32_t* ticket, float* out_acc, int interval, float target, float lo,
                   float hi, hipStream_t s);

}  // namespace dwmi
