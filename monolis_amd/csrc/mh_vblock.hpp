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
// FP64 block rows go in 256-thread workgroups (kVPrecBS sets the row kernels' size
// by the bytes of that many values; the op does its own loads): 85,184 block rows
// in 1024-thread ones, which FP32 keeps, reached 84 of 256 CUs.  Blocks of up to kVPrecRegs rows run with every factor loaded up front
// into registers; as loops over the block's size the working vector was indexed
// dynamically, in scratch memory, and each factor waited for (24.8 -> 7.3 us with
// blocks of 1, 2, 3 and 6; both orders of arithmetic are the same).
constexpr int kVPrecBS = 4;
constexpr int kVPrecRegs = 6;

// One block row's factors in registers (nd <= kVPrecRegs rows, zeros beyond).
template <typename T>
struct VBlockRegs {
  static constexpr int M = kVPrecRegs;
  T l[M][M];
  __device__ __forceinline__ void load(const T* __restrict__ L, int nd) {
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
      for (int k = 0; k < M; ++k) l[j][k] = j < nd && k < nd ? L[nd * j + k] : (T)0;
  }
  __device__ __forceinline__ void solve(int nd, T (&t)[M]) const {
#pragma unroll
    for (int j = 1; j < M; ++j)
#pragma unroll
      for (int k = 0; k < j; ++k) t[j] = j < nd ? t[j] - l[j][k] * t[k] : t[j];
#pragma unroll
    for (int j = M - 1; j >= 0; --j) {
#pragma unroll
      for (int k = M - 1; k > j; --k) t[j] = k < nd ? t[j] - l[j][k] * t[k] : t[j];
      t[j] = l[j][j] * t[j];
    }
  }
};

// CG step with variable blocks of up to kVPrecRegs rows in one pass: alpha from
// the SpMV's partials, x += alpha p, r -= alpha q, z = M_V^-1 r, partials (r, r),
// (r, z) (CG.f90:86-100, diag_V.f90:177-204).  A workgroup takes kVUpdBlocks
// block rows, so its rows are one contiguous range: the vectors are read and
// written coalesced, r passes through LDS to the thread that solves its block and
// z back.  Bound by launch and latency at these sizes (277,000 rows: 40 MB in
// one launch against 7.6 + 7.3 us for the update and the preconditioner alone;
// CG on 44^3 coupled nodes 6.0 -> 5.2 ms).
constexpr int kVUpdBlocks = kBlock;
template <typename T>
__global__ void __launch_bounds__(kBlock) k_v_cg_update(int nb, T* __restrict__ x, T* __restrict__ r,
                                                        T* __restrict__ z, const T* __restrict__ p,
                                                        const T* __restrict__ q, const int* __restrict__ list,
                                                        const int* __restrict__ dof_index,
                                                        const long long* __restrict__ doff,
                                                        const T* __restrict__ D, KState* st, int it,
                                                        const double* __restrict__ pre, int npre,
                                                        double* __restrict__ partials) {
  if (st->done) return;
  __shared__ T rl[kVUpdBlocks * kVPrecRegs];
  const int b0 = blockIdx.x * kVUpdBlocks, i = b0 + (int)threadIdx.x;
  const int last = (b0 + kVUpdBlocks < nb ? b0 + kVUpdBlocks : nb) - 1;
  const int o0 = dof_index[b0], o1 = dof_index[last] + list[last];
  // the block's factors are in flight during the sums and the update
  const int ic = i < nb ? i : nb - 1;
  const int nd = i < nb ? list[ic] : 0, o = dof_index[ic] - o0;
  VBlockRegs<T> f;
  f.load(D + doff[ic], nd);
  double tot[1];
  sum_partials<1>(pre, npre, tot);
  const double ad = st->rhok[it & 1] / tot[0];  // CG.f90:87-88
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->pq = tot[0];
    st->alpha = ad;
  }
  const T alpha = (T)ad;
  double part[2] = {0.0, 0.0};
#pragma unroll 3
  for (int e = o0 + (int)threadIdx.x; e < o1; e += kBlock) {
    const T xv = x[e], pv = p[e], rv0 = r[e], qv = q[e];
    st_stream(x + e, fma(alpha, pv, xv));           // X = alpha*P + X  (CG.f90:89)
    const T rv = fma(-alpha, qv, rv0);              // R = -alpha*Q + R (CG.f90:94)
    st_stream(r + e, rv);
    rl[e - o0] = rv;
    part[0] += (double)rv * (double)rv;
  }
  __syncthreads();
  if (nd > 0) {
    T v[kVPrecRegs], t[kVPrecRegs];
#pragma unroll
    for (int j = 0; j < kVPrecRegs; ++j) v[j] = t[j] = j < nd ? rl[o + j] : (T)0;
    f.solve(nd, t);
#pragma unroll
    for (int j = 0; j < kVPrecRegs; ++j)
      if (j < nd) {
        rl[o + j] = t[j];
        part[1] += (double)v[j] * (double)t[j];
      }
  }
  __syncthreads();
  for (int e = o0 + (int)threadIdx.x; e < o1; e += kBlock) st_stream(z + e, rl[e - o0]);
  block_sum<2>(part);
  store_partials<2>(part, partials, blockIdx.x);
}

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
      VBlockRegs<T> f;
      f.load(L, nd);
      T v[kVPrecRegs], t[kVPrecRegs];
#pragma unroll
      for (int j = 0; j < kVPrecRegs; ++j) v[j] = t[j] = j < nd ? src[o + j] : (T)0;
      f.solve(nd, t);
#pragma unroll
      for (int j = 0; j < kVPrecRegs; ++j)
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
