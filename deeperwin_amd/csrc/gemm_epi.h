// Epilogue and tile order shared by the FP32, BF16 and FP64 GEMMs.
#pragma once
#include "common.h"
#include "kernels.h"

namespace dwmi {

enum { EPI_BIAS = 1, EPI_V = 2, EPI_TANH = 4, EPI_PERM = 8 };

__device__ __forceinline__ float act_tanh(float v) { return tanh_fast(v); }
__device__ __forceinline__ double act_tanh(double v) { return tanh(v); }

// Epilogue of one element at row r = (b * n + i) * C + ch, column c.  Index math in 32 bits (M < 2^31).
template <int FLAGS, typename T>
__device__ __forceinline__ void epi_store(T v, int r, int c, T* __restrict__ Cm, int ldc, const GemmEpiT<T>& ep) {
  int bi = r, ch = 0;
  if ((FLAGS & (EPI_BIAS | EPI_V | EPI_PERM)) && ep.C > 1) {
    bi = r / ep.C;
    ch = r - bi * ep.C;
  }
  if ((FLAGS & EPI_BIAS) && ep.bias) {
    if (ch == 0) v += ep.bias[c];
  }
  int b = 0;
  if ((FLAGS & (EPI_V | EPI_PERM)) && (ep.V || ep.permute)) b = bi / ep.n;
  if ((FLAGS & EPI_V) && ep.V) {
    const T* Vp = ep.V + ((long)b * ep.C + ch) * ep.ldv + c;
    T vs = Vp[0];
    for (int q = 1; q < ep.vsplit; ++q) vs += Vp[q * ep.vstride];
    v += vs;
  }
  if ((FLAGS & EPI_TANH) && ep.act_tanh) v = act_tanh(v);
  long orow = r;
  if ((FLAGS & EPI_PERM) && ep.permute) {
    const int i = bi - b * ep.n, dn = ep.n - ep.u;
    orow = (i < ep.u) ? ((long)b * ep.u + i) * ep.C + ch
                      : (long)ep.B * ep.u * ep.C + ((long)b * dn + (i - ep.u)) * ep.C + ch;
  }
  Cm[orow * ldc + c] = v;
}

__device__ __forceinline__ int tile_index(int bid, int total) {
  // XCD-aware: workgroups are dealt round-robin to 8 XCDs; give each XCD a contiguous tile range.
  const int per = (total + 7) / 8;
  return (bid & 7) * per + (bid >> 3);
}

}  // namespace dwmi
