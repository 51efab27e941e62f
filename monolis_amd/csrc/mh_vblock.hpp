// diag_V preconditioner apply as a row op (one thread per block row), used
// standalone and inside the CG / BiCGSTAB drivers for variable block sizes.
#pragma once

#include "mh_internal.hpp"
#include "mh_kernels.hpp"

namespace mh {

// dst = M_V^-1 src (src/prec/diag/diag_V.f90:177-204): per block row, forward
// substitution with the unit-lower factor, then backward substitution with
// the reciprocal pivots.  With DOT, also the partial (src, dst) and, in
// finalize, CG's rho = (r, z) and beta = rho / rho_prev (0 when `first`),
// CG.f90:71-84, or with `first` = 2 GropCG's gamma = (r, u).
// Block rows go in 256-thread workgroups (kVPrecBS sets the row kernels' size;
// the op does its own loads): 85,184 block rows in 1024-thread ones reached 84 of
// 256 CUs.  Blocks of up to kVPrecRegs rows run with every factor loaded up front
// into registers; as loops over the block's size the working vector was indexed
// dynamically, in scratch memory, and each factor waited for (24.8 -> 7.3 us with
// blocks of 1, 2, 3 and 6; both orders of arithmetic are the same).
constexpr int kVPrecBS = 4;
constexpr int kVPrecRegs = 6;

template <typename T, bool DOT>
struct OpVPrec {
  static constexpr int KCLASS = 2;  // kClsPrec: applies the preconditioner
  using VT = T;
  static constexpr int BS = kVPrecBS;
  static constexpr int NV = DOT ? 1 : 0;
  const T* __restrict__ src;
  T* __restrict__ dst;
  const int* __restrict__ list;
  const int* __restrict__ dof_index;
  const long long* __restrict__ doff;
  const T* __restrict__ D;
  KState* st;  // null for a standalone apply
  int first;
  int maxb;  // largest block
  __device__ bool skip() const { return st != nullptr && st->done != 0; }
  __device__ void begin() {}
  __device__ void row(int i, bool valid, double (&part)[1], const WaveRows<T, kVPrecBS>&) const {
    if (!valid) return;
    const int nd = list[i];
    const int o = dof_index[i];
    const T* L = D + doff[i];
    if (maxb <= kVPrecRegs) {
      constexpr int M = kVPrecRegs;
      T l[M][M], v[M], t[M];
#pragma unroll
      for (int j = 0; j < M; ++j) {
        v[j] = j < nd ? src[o + j] : (T)0;
#pragma unroll
        for (int k = 0; k < M; ++k) l[j][k] = j < nd && k < nd ? L[nd * j + k] : (T)0;
      }
#pragma unroll
      for (int j = 0; j < M; ++j) {
        t[j] = v[j];
#pragma unroll
        for (int k = 0; k < j; ++k) t[j] = j < nd ? t[j] - l[j][k] * t[k] : t[j];
      }
#pragma unroll
      for (int j = M - 1; j >= 0; --j) {
#pragma unroll
        for (int k = M - 1; k > j; --k) t[j] = k < nd ? t[j] - l[j][k] * t[k] : t[j];
        t[j] = l[j][j] * t[j];
      }
#pragma unroll
      for (int j = 0; j < M; ++j)
        if (j < nd) {
          dst[o + j] = t[j];
          if constexpr (DOT) part[0] += (double)v[j] * (double)t[j];
        }
      return;
    }
    T t[kMaxVBlock];
    for (int j = 0; j < nd; ++j) t[j] = src[o + j];
    for (int j = 1; j < nd; ++j)
      for (int k = 0; k < j; ++k) t[j] = t[j] - L[nd * j + k] * t[k];
    for (int j = nd - 1; j >= 0; --j) {
      for (int k = nd - 1; k > j; --k) t[j] = t[j] - L[nd * j + k] * t[k];
      t[j] = L[(nd + 1) * j] * t[j];
    }
    for (int j = 0; j < nd; ++j) {
      dst[o + j] = t[j];
      if constexpr (DOT) part[0] += (double)src[o + j] * (double)t[j];
    }
  }
  __device__ void finalize(const double (&tot)[1]) const {
    if constexpr (DOT) {
      if (first == 2) {
        st->gamma = tot[0];
        return;
      }
      const double rho = tot[0];
      st->beta = first ? 0.0 : rho / st->rho;
      st->rho = rho;
    }
  }
};

}  // namespace mh
