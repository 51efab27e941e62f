// Device-side matrix assembly, the GPU counterpart of monolis's host assembly:
//   * the nonzero pattern of a simple mesh (monolis_get_nonzero_pattern_by_simple_mesh_R,
//     src/matrix/spmat_nzpattern.f90:15-49, with the nodal graph of
//     spmat_nzpattern_util.f90:13-58): element nodes radix-sorted by node, then
//     each row's columns sorted and made unique on chip;
//   * batched element matrices (monolis_add_matrix_to_sparse_matrix_main_R,
//     src/matrix/spmat_handler_util.f90:398-497): the node pairs of all
//     elements grouped by block row (by block position for elements that list a
//     node twice, very long rows or few elements) in element order, then every block
//     component summed left to right onto its current value, so the result equals
//     one add-matrix call per element in element order, bit for bit;
//   * Dirichlet conditions (monolis_set_Dirichlet_bc_main_R,
//     src/matrix/spmat_handler_util.f90:604-677) for a whole list in one pass;
//   * value and pattern read-back in monolis's layout.
// The value kernels are shared by real and complex matrices (complex element
// matrices: monolis_add_matrix_to_sparse_matrix_main_C, spmat_handler_util.f90:
// 501-600, the same loop on complex(kdouble); complex conditions:
// monolis_set_Dirichlet_bc_main_C, :681-749, whose B update multiplies two
// complex numbers as (ar*br - ai*bi, ar*bi + ai*br) without contraction).
#include <algorithm>
#include <cstdlib>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "mh_assembly.hpp"
#include "mh_launch.hpp"

namespace mh {

namespace {

int grid_for(long long n) {
  const long long g = (n + kBlock - 1) / kBlock;
  return (int)(g > 0 ? g : 1);
}

int bits_for(unsigned long long v) {
  int b = 1;
  while (b < 64 && (v >> b) != 0) ++b;
  return b;
}

// Device copy of a host array (device pointers are used in place).
template <typename T>
int stage(const T* src, size_t count, DevArray<T>& tmp, const T** out, hipStream_t s) {
  if (count == 0 || is_device_pointer(src)) {
    *out = src;
    return 0;
  }
  MH_TRY(tmp.alloc(count));
  MH_TRY(upload(tmp.p, src, count * sizeof(T), s));
  *out = tmp.p;
  return 0;
}

int read_flag(const int* d, int* h, hipStream_t s) {
  MH_HIP(hipMemcpyAsync(h, d, sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  return 0;
}

__global__ void k_check_range(long long m, const int* __restrict__ v, int hi, int* __restrict__ bad) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (long long)gridDim.x * blockDim.x) {
    const int x = v[i];
    if (x < 0 || x >= hi) atomicOr(bad, 1);
  }
}

// keys of every ordered node pair (a != c) of every element, then the diagonal
// (pattern builds with a node of more than kRowCand candidate columns)
__global__ void k_mesh_keys(int n_node, int n_base, int n_elem, const int* __restrict__ elem,
                            unsigned long long* __restrict__ keys) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = (long long)n_base * (n_base - 1);
  const long long npair = (long long)n_elem * per;
  if (t < npair) {
    const long long e = t / per;
    const int q = (int)(t % per);
    const int a = q / (n_base - 1);
    int c = q % (n_base - 1);
    if (c >= a) ++c;
    keys[t] = ((unsigned long long)elem[e * n_base + a] << 32) | (unsigned)elem[e * n_base + c];
  } else if (t < npair + n_node) {
    const unsigned i = (unsigned)(t - npair);
    keys[t] = ((unsigned long long)i << 32) | i;
  }
}

// index[r] = first key of row r, item = column + 1 (keys sorted and unique)
__global__ void k_pattern_csr(int n_node, int nz, const unsigned long long* __restrict__ keys,
                              int* __restrict__ index, int* __restrict__ item) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t <= n_node) {
    const unsigned long long target = (unsigned long long)t << 32;
    int lo = 0, hi = nz;
    while (lo < hi) {
      const int mid = lo + (hi - lo) / 2;
      if (keys[mid] < target) lo = mid + 1;
      else hi = mid;
    }
    index[t] = lo;
  }
  if (t < nz) item[t] = (int)(keys[t] & 0xffffffffull) + 1;
}

// ---- node -> (element, local node) adjacency ----------------------------------
// Pattern and element assembly are organised by block row: a row's elements are
// found once (2.1 M 32-bit keys sorted for 262,144 hexahedra, about 0.1 ms)
// instead of sorting every node pair (16.8 M 64-bit keys, 0.8 ms for the pattern
// and 0.9 ms for the element pairs), and the pairs themselves are only formed on
// chip (pattern rows: 0.21 ms).
__global__ void k_adj_keys(long long m, const int* __restrict__ elem, unsigned* __restrict__ keys,
                           int* __restrict__ ids) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m) return;
  keys[t] = (unsigned)elem[t];
  ids[t] = (int)t;
}

// start[r] = first sorted entry of row r, start[n] = m
__global__ void k_adj_start(int n, int m, const unsigned* __restrict__ keys, int* __restrict__ start) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r > n) return;
  int lo = 0, hi = m;
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if (keys[mid] < (unsigned)r) lo = mid + 1;
    else hi = mid;
  }
  start[r] = lo;
}

// Columns of one block row per wavefront: the nodes of the row's elements (at
// most kRowCand, else `over`), sorted by a bitonic network in the wavefront's
// LDS and made unique.  The list goes to tmp at start[r]*n_base + r, its length
// to cnt[r].  Rows without an element keep their diagonal alone.
constexpr int kRowCand = 512;
__global__ void __launch_bounds__(kBlock) k_pattern_rows(int n, int n_base, const int* __restrict__ start,
                                                         const int* __restrict__ ids, const int* __restrict__ elem,
                                                         int* __restrict__ tmp, int* __restrict__ cnt,
                                                         int* __restrict__ over) {
  __shared__ int lds[kWpb][kRowCand];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int r = blockIdx.x * kWpb + w;
  if (r >= n) return;  // no workgroup barrier below
  int* v = lds[w];
  const int j0 = start[r];
  const long long cand = (long long)(start[r + 1] - j0) * n_base;
  if (cand > kRowCand) {
    if (lane == 0) {
      cnt[r] = 0;
      atomicOr(over, 1);
    }
    return;
  }
  const int C = cand > 0 ? (int)cand : 1;
  int P = 2;
  while (P < C) P <<= 1;
  for (int i = lane; i < P; i += kWave) {
    int c = 0x7fffffff;  // past the end: sorts last
    if (i < cand) {
      const int pid = ids[j0 + i / n_base];
      c = elem[(size_t)(pid / n_base) * n_base + i % n_base];
    } else if (i == 0) {
      c = r;
    }
    v[i] = c;
  }
  wave_sync();
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = lane; i < P / 2; i += kWave) {
        const int a = ((i & ~(j - 1)) << 1) | (i & (j - 1)), b = a | j;
        const int x = v[a], y = v[b];
        const bool up = (a & k) == 0;
        v[a] = (x < y) == up ? x : y;
        v[b] = (x < y) == up ? y : x;
      }
      wave_sync();
    }
  int* out = tmp + (size_t)j0 * n_base + r;
  int m = 0;
  for (int i0 = 0; i0 < C; i0 += kWave) {
    const int i = i0 + lane;
    const bool keep = i < C && (i == 0 || v[i] != v[i - 1]);
    const unsigned long long mask = __ballot(keep);
    if (keep) out[m + __popcll(mask & ((1ull << lane) - 1))] = v[i];
    m += __popcll(mask);
  }
  if (lane == 0) cnt[r] = m;
}

// item of row r from its unique list (one wavefront per row)
__global__ void __launch_bounds__(kBlock) k_pattern_copy(int n, int n_base, const int* __restrict__ start,
                                                         const int* __restrict__ tmp, const int* __restrict__ index,
                                                         int* __restrict__ item) {
  const int lane = threadIdx.x & (kWave - 1);
  const int r = blockIdx.x * kWpb + (int)(threadIdx.x / kWave);
  if (r >= n) return;
  const int* src = tmp + (size_t)start[r] * n_base + r;
  const int j0 = index[r], m = index[r + 1] - j0;
  for (int i = lane; i < m; i += kWave) item[j0 + i] = src[i] + 1;
}

// flags[0]: a node id outside [0, hi); flags[1]: an element that lists a node twice
// (n_base^2 / 2 comparisons per element; elements of more than kDupNodes nodes
// are not compared and flagged)
constexpr int kDupNodes = 64;
__global__ void k_check_elems(int n_elem, int n_base, const int* __restrict__ elem, int hi, int* __restrict__ flags) {
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n_elem;
       e += (long long)gridDim.x * blockDim.x) {
    const int* q = elem + (size_t)e * n_base;
    bool bad = false, dup = n_base > kDupNodes;
    for (int a = 0; a < n_base; ++a) {
      const int x = q[a];
      bad |= x < 0 || x >= hi;
      for (int c = 0; !dup && c < a; ++c) dup = q[c] == x;
    }
    if (bad) atomicOr(flags, 1);
    if (dup) atomicOr(flags + 1, 1);
  }
}

// Block position of (row, col) in the CSR, -1 when absent (item sorted per row).
__device__ __forceinline__ int find_block(const int* __restrict__ rowptr, const int* __restrict__ item, int row,
                                          int col) {
  int lo = rowptr[row];
  const int end = rowptr[row + 1];
  int hi = end;
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if (item[mid] < col + 1) lo = mid + 1;
    else hi = mid;
  }
  return (lo < end && item[lo] == col + 1) ? lo : -1;
}

// One thread per (element, a, c) node pair: key = block position of
// (elem[a], elem[c]) or `none` (sorted last) when the block is absent; value =
// the pair id e*n_base^2 + a*n_base + c.  A stable sort by key keeps the pairs
// of one block in element order.
__global__ void k_elem_targets(int ne, int n_base, const int* __restrict__ elem, const int* __restrict__ rowptr,
                               const int* __restrict__ item, unsigned long long* __restrict__ keys,
                               int* __restrict__ ids, int* __restrict__ bad, unsigned long long none) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long per = (long long)n_base * n_base;
  if (t >= (long long)ne * per) return;
  const int e = (int)(t / per);
  const int q = (int)(t % per);
  const int a = q / n_base, c = q % n_base;
  const int blk = find_block(rowptr, item, elem[(size_t)e * n_base + a], elem[(size_t)e * n_base + c]);
  if (blk < 0) atomicOr(bad, 1);
  keys[t] = blk >= 0 ? (unsigned long long)blk : none;
  ids[t] = (int)t;
}

// Slot (block position inside its row) of every (sorted adjacency entry, c):
// pos[j*n_base + c] of column elem[e][c] in row keys[j].
__global__ void k_elem_pos(long long m, int n_base, const unsigned* __restrict__ keys, const int* __restrict__ ids,
                           const int* __restrict__ elem, const int* __restrict__ rowptr,
                           const int* __restrict__ item, unsigned short* __restrict__ pos, int* __restrict__ bad) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m * n_base) return;
  const int j = (int)(t / n_base), c = (int)(t % n_base);
  const int r = (int)keys[j];
  const int blk = find_block(rowptr, item, r, elem[(size_t)(ids[j] / n_base) * n_base + c]);
  if (blk < 0) atomicOr(bad, 1);
  pos[t] = (unsigned short)(blk >= 0 ? blk - rowptr[r] : 0);
}

// Element assembly by block row.  A workgroup keeps the stored values of RW
// consecutive block rows in LDS (rows of `stride` values); each wavefront takes
// its rows' adjacency entries in element order and adds the entry's strip of Ke
// -- the b rows of the element matrix that belong to node a are n_base*b*b
// consecutive values -- component by component.  Every component is summed in
// element order onto its stored value, so the result equals one add-matrix call
// per element bit for bit; an element lists a node at most once here, so the
// lanes of one strip never meet.  Ke is read once, in contiguous strips, J of
// them in flight per wavefront; the SELL values are read and written once, RW
// rows side by side (16 bytes per row and pair).
// Bound by HBM: 262,144 hexahedra x 3 DOF move 1.21 GB of Ke and 2 x 0.53 GB of
// values in 0.54 ms, 4.2 TB/s (4.39 ms as one thread per block component, which
// gathered its 8 contributions one by one).  NCH: 64-lane pieces of a strip held in registers (0: any length, one
// strip at a time).
template <typename V, int RW, int NCH>
__global__ void __launch_bounds__(kBlock) k_elem_rows(int n, int n_base, int b, const int* __restrict__ start,
                                                      const int* __restrict__ ids,
                                                      const unsigned short* __restrict__ pos,
                                                      const V* __restrict__ Ke, const int* __restrict__ rowptr,
                                                      const int* __restrict__ slice_ptr, V* __restrict__ val,
                                                      int stride) {
  extern __shared__ double elem_lds[];
  V* acc = reinterpret_cast<V*>(elem_lds);
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int bb = b * b;
  const int r0 = blockIdx.x * RW;  // RW divides the slice height: one slice
  const size_t slot0 = (size_t)slice_ptr[r0 / kWave];
  // stored values <-> LDS; consecutive threads take consecutive rows
  constexpr int PW = sell_paired<V>() ? 2 : 1;  // values per access
  const int units = (bb + PW - 1) / PW;
  const int maxlen = stride / bb;
  const int rr = threadIdx.x % RW, row = r0 + rr;
  const int len = row < n && start[row + 1] > start[row] ? rowptr[row + 1] - rowptr[row] : 0;
  const int rlane = row % kWave;
  auto exchange = [&](auto&& f) {
    for (int i = threadIdx.x / RW; i < maxlen * units; i += kBlock / RW) {
      const int k = i / units, e = (i % units) * PW;
      if (k < len) f(val + (slot0 + k) * (size_t)bb * kWave + sell_vofs<V>(e, bb, rlane), acc + rr * stride + k * bb + e,
                     e + PW <= bb);
    }
  };
  exchange([&](const V* g, V* l, bool full) {
    if constexpr (PW == 2) {
      if (full) {
        const d2v t = *(const d2v*)g;
        l[0] = t.x;
        l[1] = t.y;
        return;
      }
    }
    l[0] = *g;
  });
  __syncthreads();
  const long long S = (long long)n_base * bb;  // values per strip
  constexpr int NC = NCH > 0 ? NCH : 1;
  constexpr int J = NCH == 1 ? 8 : NCH == 2 ? 8 : NCH > 2 ? 4 : 1;
  const int nb = n_base * b;
  int cc[NC], off[NC];
  if constexpr (NCH > 0) {
#pragma unroll
    for (int h = 0; h < NC; ++h) {
      const int t = h * kWave + lane, k1 = t / nb, q = t % nb;
      cc[h] = t < S ? q / b : -1;
      off[h] = k1 * b + q % b;
    }
  }
  for (int q = w; q < RW; q += kWpb) {
    const int r = r0 + q;
    if (r >= n) break;
    const int j0 = start[r], j1 = start[r + 1];
    V* a = acc + q * stride;
    if constexpr (NCH > 0) {
      for (int j = j0; j < j1; j += J) {
        V v[J][NC];
        int p[J][NC];
#pragma unroll
        for (int u = 0; u < J; ++u) {
          const int ju = j + u < j1 ? j + u : j1 - 1;
          const V* strip = Ke + (long long)ids[ju] * S;
#pragma unroll
          for (int h = 0; h < NC; ++h) {
            const int t = h * kWave + lane;
            v[u][h] = ld_val<true>(strip + (cc[h] >= 0 ? t : 0));
            p[u][h] = pos[(long long)ju * n_base + (cc[h] >= 0 ? cc[h] : 0)];
          }
        }
#pragma unroll
        for (int u = 0; u < J; ++u) {
          if (j + u < j1) {
#pragma unroll
            for (int h = 0; h < NC; ++h)
              if (cc[h] >= 0) {
                V* d = a + p[u][h] * bb + off[h];
                *d = *d + v[u][h];
              }
          }
          wave_sync();
        }
      }
    } else {
      for (int j = j0; j < j1; ++j) {
        const V* strip = Ke + (long long)ids[j] * S;
        for (int t = lane; t < S; t += kWave) {
          const int k1 = t / nb, x = t % nb;
          V* d = a + pos[(long long)j * n_base + x / b] * bb + k1 * b + x % b;
          *d = *d + ld_val<true>(strip + t);
        }
        wave_sync();
      }
    }
  }
  __syncthreads();
  exchange([&](V* g, const V* l, bool full) {
    if constexpr (PW == 2) {
      if (full) {
        d2v t;
        t.x = l[0];
        t.y = l[1];
        *(d2v*)g = t;
        return;
      }
    }
    *g = l[0];
  });
}

// SELL position of block `blk`, component e (row found by bisection).
template <typename V>
__device__ __forceinline__ size_t sell_pos(int blk, int e, int bb, int n, const int* __restrict__ rowptr,
                                           const int* __restrict__ slice_ptr) {
  int lo = 0, hi = n - 1;  // first row r with rowptr[r + 1] > blk
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if (rowptr[mid + 1] > blk) hi = mid;
    else lo = mid + 1;
  }
  const int r = lo;
  const size_t slot = (size_t)slice_ptr[r / kWave] + (size_t)(blk - rowptr[r]);
  return sell_vpos<V>(slot, e, bb, r % kWave);
}

// Thread (i, component): at the head i of each run of equal block keys, adds
// the component of every pair in the run, in order, onto the stored value.
template <typename V>
__global__ void k_elem_accumulate(long long m, const unsigned long long* __restrict__ keys,
                                  const int* __restrict__ ids, const V* __restrict__ Ke, int n_base, int b,
                                  int n, const int* __restrict__ rowptr, const int* __restrict__ slice_ptr,
                                  V* __restrict__ val, unsigned long long none) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int bb = b * b;
  if (t >= m * bb) return;
  const long long i = t / bb;
  const int ee = (int)(t % bb);
  const unsigned long long key = keys[i];
  if (key == none || (i > 0 && keys[i - 1] == key)) return;
  const int k1 = ee / b, k2 = ee % b;
  const long long per = (long long)n_base * n_base;
  const long long nzm = (long long)n_base * b;
  const size_t pos = sell_pos<V>((int)key, ee, bb, n, rowptr, slice_ptr);
  V acc = val[pos];
  for (long long j = i; j < m && keys[j] == key; ++j) {
    const long long pid = ids[j];
    const long long e = pid / per;
    const int q = (int)(pid % per);
    const int a = q / n_base, c = q % n_base;
    acc = acc + Ke[e * nzm * nzm + (long long)(a * b + k1) * nzm + (c * b + k2)];
  }
  val[pos] = acc;
}

template <typename V>
__global__ void k_bc_mark(int nbc, const int* __restrict__ node, const int* __restrict__ dof,
                          const V* __restrict__ v, int b, int* __restrict__ isbc, V* __restrict__ bcval,
                          int* __restrict__ nodebc, int* __restrict__ dup) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nbc) return;
  const int d = node[i] * b + dof[i];
  nodebc[node[i]] = 1;
  if (atomicAdd(&isbc[d], 1) != 0) atomicOr(dup, 1);
  bcval[d] = v[i];
}

__global__ void k_bc_check_diag(int nbc, const int* __restrict__ node, const int* __restrict__ rowptr,
                                const int* __restrict__ item, int* __restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nbc) return;
  if (find_block(rowptr, item, node[i], node[i]) < 0) atomicOr(bad, 1);
}

// val * A of a condition column, as monolis multiplies (no fused multiply-add).
__device__ __forceinline__ double bc_prod(double v, double a) {
#pragma clang fp contract(off)
  return v * a;
}
__device__ __forceinline__ zd bc_prod(zd v, zd a) {
#pragma clang fp contract(off)
  return zd(v.re * a.re - v.im * a.im, v.re * a.im + v.im * a.re);
}

// A workgroup per slice, one thread per block row: rows of condition DOFs become
// unit rows with rhs = val; other rows move val * A(r, c) of condition columns to
// the right-hand side (blocks in column order, then component order) and zero
// them.  nodebc flags the nodes with a condition: the four wavefronts look over a
// slice's column ids together, and most rows, coupling to none, end there (12,675
// conditions on 274,625 rows of 27 blocks: 134 -> 83 us).
template <typename V>
__global__ void __launch_bounds__(kBlock) k_bc_apply(int n, int b, const int* __restrict__ slice_ptr,
                                                     const int* __restrict__ rowptr, const int* __restrict__ col,
                                                     V* __restrict__ val, const int* __restrict__ isbc,
                                                     const int* __restrict__ nodebc, const V* __restrict__ bcval,
                                                     V* __restrict__ rhs) {
#pragma clang fp contract(off)
  __shared__ int flag[kWpb][kWave];
  const int s = blockIdx.x, lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int r = s * kWave + lane;
  const int k0 = slice_ptr[s];
  const int len = r < n ? rowptr[r + 1] - rowptr[r] : 0;
  const int bb = b * b;
  int any = r < n ? nodebc[r] : 0;
#pragma unroll 4
  for (int k = w; k < len; k += kWpb) any |= nodebc[col[((size_t)k0 + k) * kWave + lane]];
  flag[w][lane] = any;
  __syncthreads();
  if (w != 0) return;
#pragma unroll
  for (int u = 1; u < kWpb; ++u) any |= flag[u][lane];
  if (!any) return;
  for (int k1 = 0; k1 < b; ++k1) {
    const bool rowbc = isbc[r * b + k1] != 0;
    V acc = rhs[(size_t)r * b + k1];
    for (int k = 0; k < len; ++k) {
      const size_t slot = (size_t)k0 + k;
      const int c = col[slot * kWave + lane];
      for (int k2 = 0; k2 < b; ++k2) {
        const bool colbc = isbc[c * b + k2] != 0;
        const size_t pos = sell_vpos<V>(slot, k1 * b + k2, bb, lane);
        if (colbc && !rowbc) {
          const V t = bc_prod(bcval[c * b + k2], val[pos]);
          acc = acc - t;  // B(n) = B(n) - val*A(m)  (spmat_handler_util.f90:636, :723)
        }
        if (rowbc || colbc) val[pos] = V((rowbc && c == r && k1 == k2) ? 1.0 : 0.0);
      }
    }
    rhs[(size_t)r * b + k1] = rowbc ? bcval[r * b + k1] : acc;
  }
}

// ---- variable block sizes (monolis n_dof = -1): values in monolis's layout,
// block (i, j) at index2[e] with n_i x n_j row-major components ----------------
// Element e's matrix is (sum_a n(elem[e][a]))^2 row-major; sz[e] is its size.
__global__ void k_v_elem_sizes(int ne, int n_base, const int* __restrict__ elem, const int* __restrict__ list,
                               long long* __restrict__ sz) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ne) return;
  long long d = 0;
  for (int a = 0; a < n_base; ++a) d += list[elem[(size_t)e * n_base + a]];
  sz[e] = d * d;
}

// Block row of block position blk (bisection over the block CSR offsets).
__device__ __forceinline__ int block_row(int blk, int n, const int* __restrict__ index) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = lo + (hi - lo) / 2;
    if (index[mid + 1] > blk) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}

// k_elem_accumulate for variable blocks: thread (i, component k1*maxb + k2) at
// the head i of a run of equal block keys adds that component of every pair in
// the run, in order, onto monolis's A (entry (k1, k2) of block (r, c) at
// index2[blk] + n_c*k1 + k2; element entry (off_a + k1, off_c + k2), off_a the
// sum of the block sizes of the element's nodes before a).
template <typename V>
__global__ void k_v_elem_accumulate(long long m, const unsigned long long* __restrict__ keys,
                                    const int* __restrict__ ids, const V* __restrict__ Ke,
                                    const long long* __restrict__ koff, const int* __restrict__ elem, int n_base,
                                    int maxb, int n, const int* __restrict__ list, const int* __restrict__ index,
                                    const int* __restrict__ item, const int* __restrict__ index2, V* __restrict__ A,
                                    unsigned long long none) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int mm = maxb * maxb;
  if (t >= m * mm) return;
  const long long i = t / mm;
  const int comp = (int)(t % mm);
  const unsigned long long key = keys[i];
  if (key == none || (i > 0 && keys[i - 1] == key)) return;
  const int blk = (int)key;
  const int r = block_row(blk, n, index), c = item[blk] - 1;
  const int n1 = list[r], n2 = list[c];
  const int k1 = comp / maxb, k2 = comp % maxb;
  if (k1 >= n1 || k2 >= n2) return;
  const long long pos = (long long)index2[blk] + (long long)n2 * k1 + k2;
  const long long per = (long long)n_base * n_base;
  V acc = A[pos];
  for (long long j = i; j < m && keys[j] == key; ++j) {
    const long long pid = ids[j];
    const long long e = pid / per;
    const int q = (int)(pid % per);
    const int a = q / n_base, cc = q % n_base;
    long long S = 0, ro = 0, co = 0;
    for (int u = 0; u < n_base; ++u) {
      const int d = list[elem[e * n_base + u]];
      if (u < a) ro += d;
      if (u < cc) co += d;
      S += d;
    }
    acc = acc + Ke[koff[e] + (ro + k1) * S + co + k2];
  }
  A[pos] = acc;
}

template <typename V>
__global__ void k_v_bc_mark(int nbc, const int* __restrict__ node, const int* __restrict__ dof,
                            const V* __restrict__ v, const int* __restrict__ dof_index, const int* __restrict__ list,
                            int* __restrict__ isbc, V* __restrict__ bcval, int* __restrict__ flags) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nbc) return;
  if (dof[i] >= list[node[i]]) {  // monolis_stop_by_submatrix_access
    atomicOr(flags + 2, 1);
    return;
  }
  const int d = dof_index[node[i]] + dof[i];
  if (atomicAdd(&isbc[d], 1) != 0) atomicOr(flags + 1, 1);
  bcval[d] = v[i];
}

// k_bc_apply on monolis's variable-block layout (one thread per block row).
template <typename V>
__global__ void k_v_bc_apply(int n, const int* __restrict__ list, const int* __restrict__ dof_index,
                             const int* __restrict__ index, const int* __restrict__ item,
                             const int* __restrict__ index2, V* __restrict__ A, const int* __restrict__ isbc,
                             const V* __restrict__ bcval, V* __restrict__ rhs) {
#pragma clang fp contract(off)
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int n1 = list[r];
  for (int k1 = 0; k1 < n1; ++k1) {
    const int d = dof_index[r] + k1;
    const bool rowbc = isbc[d] != 0;
    V acc = rhs[d];
    for (int e = index[r]; e < index[r + 1]; ++e) {
      const int c = item[e] - 1;
      const int n2 = list[c];
      for (int k2 = 0; k2 < n2; ++k2) {
        const int dc = dof_index[c] + k2;
        const bool colbc = isbc[dc] != 0;
        const long long pos = (long long)index2[e] + (long long)n2 * k1 + k2;
        if (colbc && !rowbc) {
          const V t = bc_prod(bcval[dc], A[pos]);
          acc = acc - t;
        }
        if (rowbc || colbc) A[pos] = V((rowbc && c == r && k1 == k2) ? 1.0 : 0.0);
      }
    }
    rhs[d] = rowbc ? bcval[d] : acc;
  }
}

int require_assemblable(const Matrix& M, const char* what, bool cplx) {
  if (M.vb || M.is_complex != cplx) {
    set_error("%s: %s fixed-block matrices only", what, cplx ? "complex" : "real");
    return -2;
  }
  if (M.np != M.n) {
    set_error("%s: square local matrices only (n == np)", what);
    return -2;
  }
  return 0;
}

void mark_values_changed(Matrix* M) {
  M->diag_ready = M->diag32_ready = M->diagz_ready = false;
  M->val32_ready = false;  // the FP32 copy is rebuilt on its next use
  M->transpose_stale = true;
}

template <typename V>
DevArray<V>& vb_values(VBlock& Vb);
template <>
DevArray<double>& vb_values<double>(VBlock& Vb) {
  return Vb.A64;
}
template <>
DevArray<zd>& vb_values<zd>(VBlock& Vb) {
  return Vb.Az;
}

// Re-expands a variable-block matrix from its kept monolis-layout values.
int vb_reexpand(Matrix* M, const double* A, hipStream_t s) { return matrix_set_values_vblock(M, A, s); }
int vb_reexpand(Matrix* M, const zd* A, hipStream_t s) { return matrix_set_values_vblock_complex(M, A, s); }

int require_vblock(const Matrix& M, const char* what, bool cplx) {
  if (!M.vb || M.is_complex != cplx) {
    set_error("%s: %s matrices only", what, cplx ? "complex" : "real");
    return -2;
  }
  if (M.vb->npb != M.vb->nb) {
    set_error("%s: square local matrices only (n == np)", what);
    return -2;
  }
  return 0;
}

template <typename V>
V* values_of(Matrix* M);
template <>
double* values_of<double>(Matrix* M) {
  return M->val64.p;
}
template <>
zd* values_of<zd>(Matrix* M) {
  return M->valz.p;
}

// Entries e*n_base + a of `elem` sorted by node (stable: element order kept),
// and the first entry of every node.
struct Adjacency {
  DevArray<unsigned> keys;  // node of entry j
  DevArray<int> ids;        // e*n_base + a of entry j
  DevArray<int> start;      // n + 1
  int build(int n, int m, const int* elem, hipStream_t s) {
    DevArray<unsigned> k0;
    DevArray<int> i0;
    MH_TRY(keys.alloc((size_t)m));
    MH_TRY(ids.alloc((size_t)m));
    MH_TRY(start.alloc((size_t)n + 1));
    if (m > 0) {
      MH_TRY(k0.alloc((size_t)m));
      MH_TRY(i0.alloc((size_t)m));
      k_adj_keys<<<grid_for(m), kBlock, 0, s>>>(m, elem, k0.p, i0.p);
      MH_HIP(hipGetLastError());
      const int end_bit = bits_for((unsigned long long)n);
      size_t bytes = 0;
      MH_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k0.p, keys.p, i0.p, ids.p, m, 0, end_bit, s));
      DevArray<unsigned char> tmp;
      MH_TRY(tmp.alloc(bytes));
      MH_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, k0.p, keys.p, i0.p, ids.p, m, 0, end_bit, s));
      k_adj_start<<<grid_for((long long)n + 1), kBlock, 0, s>>>(n, m, keys.p, start.p);
      MH_HIP(hipGetLastError());
      MH_HIP(hipStreamSynchronize(s));  // k0, i0 and tmp are released on return
    } else {
      MH_HIP(hipMemsetAsync(start.p, 0, sizeof(int) * ((size_t)n + 1), s));
    }
    return 0;
  }
};

// Launch of k_elem_rows for one chunk of elements; RW rows of LDS per workgroup.
template <typename V, int RW>
int launch_elem_rows_rw(const Matrix& M, int n_base, const Adjacency& adj, const unsigned short* pos, const V* Ke,
                        V* val, hipStream_t s) {
  const int b = M.b, stride = M.max_width * b * b;
  const size_t lds = (size_t)RW * stride * sizeof(V);
  const int grid = (M.n + RW - 1) / RW;
  const long long S = (long long)n_base * b * b;
#define MH_ELEM_ROWS(NCH)                                                                                       \
  k_elem_rows<V, RW, NCH><<<grid, kBlock, lds, s>>>(M.n, n_base, b, adj.start.p, adj.ids.p, pos, Ke, M.rowptr.p, \
                                                    M.slice_ptr.p, val, stride)
  if (S <= kWave) MH_ELEM_ROWS(1);
  else if (S <= 2 * kWave) MH_ELEM_ROWS(2);
  else if (S <= 4 * kWave && sizeof(V) == 8) MH_ELEM_ROWS(4);
  else MH_ELEM_ROWS(0);
#undef MH_ELEM_ROWS
  MH_HIP(hipGetLastError());
  return 0;
}

// LDS a workgroup of k_elem_rows may take: what every device grants without an attribute.
constexpr size_t kElemLds = (size_t)64 << 10;

template <typename V>
bool elem_rows_fit(const Matrix& M, int n_base) {
  return M.max_width < 65536 && (size_t)4 * M.max_width * M.b * M.b * sizeof(V) <= kElemLds &&
         (long long)n_base * M.b * M.b < (1LL << 30);
}

// Whether a call of n_elem elements is worth a pass over every block row: the pass
// and the adjacency cost the same however few rows the elements touch.  us of a
// call by rows / by sorted pairs, device inputs, consecutive hexahedra, 3 DOF:
// 4,913 nodes: 64 elements 98 / 85, 1,024 135 / 122, 2,048 123 / 149, 4,096 145 /
// 209; 274,625 nodes: 64 147 / 85, 2,048 171 / 149, 4,096 194 / 212, 65,536 389 /
// 1,334 (scattered elements: 4,096 314 / 223, 16,384 489 / 554): a node pair per
// block row, and 2^16 of them.  Rows too long for 16 of them in a workgroup's LDS
// cost more to pass over (20-node elements, 3 DOF, 274,625 nodes: 64 elements 429
// / 127, 4,096 592 / 615, scattered 1,653 / 742, 16,384 866 / 2,200): eight pairs.
template <typename V>
bool elem_rows_pay(const Matrix& M, long long pairs) {
  const bool short_rows = (size_t)16 * M.max_width * M.b * M.b * sizeof(V) <= kElemLds;
  return pairs >= std::max(1LL << 16, (long long)M.n * (short_rows ? 1 : 8));
}

template <typename V>
int launch_elem_rows(const Matrix& M, int n_base, const Adjacency& adj, const unsigned short* pos, const V* Ke, V* val,
                     hipStream_t s) {
  // 16 rows: 256-byte accesses of the stored values, about 32 KB of LDS for 27
  // blocks of 3 x 3 (five workgroups per CU)
  const size_t per_row = (size_t)M.max_width * M.b * M.b * sizeof(V);
  if (16 * per_row <= kElemLds) return launch_elem_rows_rw<V, 16>(M, n_base, adj, pos, Ke, val, s);
  if (8 * per_row <= kElemLds) return launch_elem_rows_rw<V, 8>(M, n_base, adj, pos, Ke, val, s);
  return launch_elem_rows_rw<V, 4>(M, n_base, adj, pos, Ke, val, s);
}

}  // namespace

int pattern_by_simple_mesh(int n_node, int n_base, int n_elem, const int* elem, DevArray<int>& index,
                           DevArray<int>& item, int* nz_out, hipStream_t s) {
  if (n_node < 1 || n_base < 1 || n_elem < 0) {
    set_error("invalid mesh sizes n_node=%d n_base=%d n_elem=%d", n_node, n_base, n_elem);
    return -2;
  }
  const long long nelem_ids = (long long)n_elem * n_base;
  const long long npair = (long long)n_elem * n_base * (n_base - 1);
  const long long K = npair + n_node;
  if (K >= (1LL << 31)) {
    set_error("mesh too large for one pattern build (%lld node pairs)", K);
    return -2;
  }
  DevArray<int> etmp;
  const int* de = nullptr;
  MH_TRY(stage(elem, (size_t)nelem_ids, etmp, &de, s));
  DevArray<int> flag;  // [0] node id out of range, [1] a row with too many candidate columns
  MH_TRY(flag.alloc(2));
  MH_HIP(hipMemsetAsync(flag.p, 0, 2 * sizeof(int), s));
  if (nelem_ids > 0) {
    k_check_range<<<std::min(grid_for(nelem_ids), 65536), kBlock, 0, s>>>(nelem_ids, de, n_node, flag.p);
    MH_HIP(hipGetLastError());
  }
  int bad = 0;
  MH_TRY(read_flag(flag.p, &bad, s));
  if (bad) {
    set_error("element connectivity holds a node id outside 0..%d", n_node - 1);
    return -2;
  }
  {
    Adjacency adj;
    MH_TRY(adj.build(n_node, (int)nelem_ids, de, s));
    DevArray<int> tmp, cnt;
    MH_TRY(tmp.alloc((size_t)nelem_ids * n_base + n_node));
    MH_TRY(cnt.alloc((size_t)n_node + 1));
    MH_TRY(index.alloc((size_t)n_node + 1));
    MH_HIP(hipMemsetAsync(cnt.p + n_node, 0, sizeof(int), s));
    const int grid = (n_node + kWpb - 1) / kWpb;
    k_pattern_rows<<<grid, kBlock, 0, s>>>(n_node, n_base, adj.start.p, adj.ids.p, de, tmp.p, cnt.p, flag.p + 1);
    MH_HIP(hipGetLastError());
    size_t scan_bytes = 0;
    MH_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, cnt.p, index.p, n_node + 1, s));
    DevArray<unsigned char> scan_tmp;
    MH_TRY(scan_tmp.alloc(scan_bytes));
    MH_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp.p, scan_bytes, cnt.p, index.p, n_node + 1, s));
    int nz = 0;
    MH_HIP(hipMemcpyAsync(&bad, flag.p + 1, sizeof(int), hipMemcpyDeviceToHost, s));
    MH_TRY(read_flag(index.p + n_node, &nz, s));
    if (!bad) {
      MH_TRY(item.alloc((size_t)nz));
      k_pattern_copy<<<grid, kBlock, 0, s>>>(n_node, n_base, adj.start.p, tmp.p, index.p, item.p);
      MH_HIP(hipGetLastError());
      MH_HIP(hipStreamSynchronize(s));
      *nz_out = nz;
      return 0;
    }
  }
  // a hub node with more than kRowCand candidates: sort every pair of the mesh
  DevArray<unsigned long long> k0, k1;
  MH_TRY(k0.alloc((size_t)K));
  MH_TRY(k1.alloc((size_t)K));
  k_mesh_keys<<<grid_for(K), kBlock, 0, s>>>(n_node, n_base, n_elem, de, k0.p);
  MH_HIP(hipGetLastError());
  const int end_bit = 32 + bits_for((unsigned long long)n_node);
  size_t tmp_bytes = 0, tmp2 = 0;
  MH_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tmp_bytes, k0.p, k1.p, (int)K, 0, end_bit, s));
  MH_HIP(hipcub::DeviceSelect::Unique(nullptr, tmp2, k1.p, k0.p, flag.p, (int)K, s));
  DevArray<unsigned char> tmp;
  MH_TRY(tmp.alloc(std::max(tmp_bytes, tmp2)));
  MH_HIP(hipcub::DeviceRadixSort::SortKeys(tmp.p, tmp_bytes, k0.p, k1.p, (int)K, 0, end_bit, s));
  MH_HIP(hipcub::DeviceSelect::Unique(tmp.p, tmp2, k1.p, k0.p, flag.p, (int)K, s));
  int nz = 0;
  MH_TRY(read_flag(flag.p, &nz, s));
  MH_TRY(index.alloc((size_t)n_node + 1));
  MH_TRY(item.alloc((size_t)nz));
  k_pattern_csr<<<grid_for(std::max<long long>(nz, (long long)n_node + 1)), kBlock, 0, s>>>(n_node, nz, k0.p,
                                                                                            index.p, item.p);
  MH_HIP(hipGetLastError());
  MH_HIP(hipStreamSynchronize(s));
  *nz_out = nz;
  return 0;
}

template <typename V>
static int add_elements_T(Matrix* M, int n_elem, int n_base, const int* elem, const V* Ke, hipStream_t s) {
  MH_TRY(require_assemblable(*M, "element assembly", sizeof(V) == sizeof(zd)));
  if (n_elem < 0 || n_base < 1) {
    set_error("invalid element sizes n_elem=%d n_base=%d", n_elem, n_base);
    return -2;
  }
  if (n_elem == 0 || M->n == 0) return 0;
  const int b = M->b, bb = b * b;
  const long long nzm = (long long)n_base * b;
  const long long per_elem = nzm * nzm;       // values per element matrix
  const long long pairs_elem = (long long)n_base * n_base;
  if (per_elem > (1LL << 30)) {
    set_error("element matrix too large (%lld entries)", per_elem);
    return -2;
  }
  // node pairs per chunk: bounded temporaries, element order kept across chunks
  // (MONOLIS_HIP_ASSEMBLY_CHUNK_PAIRS overrides the 2^24 default)
  long long max_pairs = 1LL << 24;
  if (const char* env = getenv("MONOLIS_HIP_ASSEMBLY_CHUNK_PAIRS")) {
    const long long v = atoll(env);
    if (v > 0) max_pairs = v;
  }
  const int chunk = (int)std::max<long long>(1, std::min<long long>(n_elem, max_pairs / pairs_elem));
  DevArray<int> etmp;
  const int* de = nullptr;
  MH_TRY(stage(elem, (size_t)n_elem * n_base, etmp, &de, s));
  DevArray<int> flag;  // [0] node id out of range / absent block, [1] an element that lists a node twice
  MH_TRY(flag.alloc(2));
  MH_HIP(hipMemsetAsync(flag.p, 0, 2 * sizeof(int), s));
  k_check_elems<<<std::min(grid_for(n_elem), 65536), kBlock, 0, s>>>(n_elem, n_base, de, M->n, flag.p);
  MH_HIP(hipGetLastError());
  int chk[2] = {0, 0};
  MH_HIP(hipMemcpyAsync(chk, flag.p, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (chk[0]) {
    set_error("element connectivity holds a node id outside 0..%d", M->n - 1);
    return -2;
  }
  // By block row when no element lists a node twice, four rows fit in a
  // workgroup's LDS and the elements are enough; otherwise by sorted node pairs.
  const bool by_rows = !chk[1] && elem_rows_fit<V>(*M, n_base) && elem_rows_pay<V>(*M, n_elem * pairs_elem);
  int bad = 0;
  const bool ke_dev = is_device_pointer(Ke);
  const long long cap = (long long)chunk * pairs_elem;
  DevArray<unsigned long long> k0, k1;
  DevArray<int> i0, i1;
  DevArray<unsigned short> pos;
  DevArray<unsigned char> tmp;
  DevArray<V> kt;
  if (!ke_dev) MH_TRY(kt.alloc((size_t)chunk * per_elem));
  // keys are block positions < nz; `none` (an absent block) sorts last
  const int end_bit = bits_for((unsigned long long)M->nz) + 1;
  const unsigned long long none = 1ull << (end_bit - 1);
  size_t tmp_bytes = 0;
  if (by_rows) {
    MH_TRY(pos.alloc((size_t)cap));
  } else {
    MH_TRY(k0.alloc((size_t)cap));
    MH_TRY(k1.alloc((size_t)cap));
    MH_TRY(i0.alloc((size_t)cap));
    MH_TRY(i1.alloc((size_t)cap));
    MH_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, k0.p, k1.p, i0.p, i1.p, (int)cap, 0, end_bit, s));
    MH_TRY(tmp.alloc(tmp_bytes));
  }
  for (int e0 = 0; e0 < n_elem; e0 += chunk) {
    const int ne = std::min(chunk, n_elem - e0);
    const long long m = (long long)ne * pairs_elem;
    const int* ec = de + (size_t)e0 * n_base;
    const V* kc = nullptr;
    if (ke_dev) {
      kc = Ke + (size_t)e0 * per_elem;
    } else {
      MH_TRY(upload(kt.p, Ke + (size_t)e0 * per_elem, (size_t)ne * per_elem * sizeof(V), s));
      kc = kt.p;
    }
    Adjacency adj;
    if (by_rows) {
      MH_TRY(adj.build(M->n, ne * n_base, ec, s));
      k_elem_pos<<<grid_for(m), kBlock, 0, s>>>((long long)ne * n_base, n_base, adj.keys.p, adj.ids.p, ec, M->rowptr.p,
                                                M->csr_item.p, pos.p, flag.p);
    } else {
      k_elem_targets<<<grid_for(m), kBlock, 0, s>>>(ne, n_base, ec, M->rowptr.p, M->csr_item.p, k0.p, i0.p, flag.p,
                                                    none);
    }
    MH_HIP(hipGetLastError());
    MH_TRY(read_flag(flag.p, &bad, s));
    if (bad) {
      // monolis stops here (monolis_stop_by_matrix_assemble); earlier chunks stay added
      set_error("element %d..%d couples nodes whose block is not in the nonzero pattern", e0, e0 + ne - 1);
      mark_values_changed(M);
      return -2;
    }
    if (by_rows) {
      MH_TRY(launch_elem_rows<V>(*M, n_base, adj, pos.p, kc, values_of<V>(M), s));
      MH_HIP(hipStreamSynchronize(s));  // adj is rebuilt for the next chunk
    } else {
      size_t tb = tmp_bytes;
      MH_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, k0.p, k1.p, i0.p, i1.p, (int)m, 0, end_bit, s));
      k_elem_accumulate<V><<<grid_for(m * bb), kBlock, 0, s>>>(m, k1.p, i1.p, kc, n_base, b, M->n, M->rowptr.p,
                                                                M->slice_ptr.p, values_of<V>(M), none);
      MH_HIP(hipGetLastError());
    }
  }
  MH_HIP(hipStreamSynchronize(s));
  mark_values_changed(M);
  return 0;
}

// Element assembly on a variable-block matrix: monolis's layout values kept in
// the VBlock are updated (sorted node pairs, sums in element order, as for fixed
// blocks), then the scalar expansion and the diag_V factors are rebuilt.
template <typename V>
static int add_elements_V_T(Matrix* M, int n_elem, int n_base, const int* elem, const V* Ke, hipStream_t s) {
  MH_TRY(require_vblock(*M, "element assembly", sizeof(V) == sizeof(zd)));
  VBlock& Vb = *M->vb;
  if (n_elem < 0 || n_base < 1) {
    set_error("invalid element sizes n_elem=%d n_base=%d", n_elem, n_base);
    return -2;
  }
  if (n_elem == 0 || Vb.nb == 0) return 0;
  const int n = Vb.nb;
  const long long pairs_elem = (long long)n_base * n_base;
  long long max_pairs = 1LL << 24;
  if (const char* env = getenv("MONOLIS_HIP_ASSEMBLY_CHUNK_PAIRS")) {
    const long long v = atoll(env);
    if (v > 0) max_pairs = v;
  }
  const int chunk = (int)std::max<long long>(1, std::min<long long>(n_elem, max_pairs / pairs_elem));
  DevArray<int> etmp;
  const int* de = nullptr;
  MH_TRY(stage(elem, (size_t)n_elem * n_base, etmp, &de, s));
  DevArray<int> flag;
  MH_TRY(flag.alloc(1));
  MH_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), s));
  k_check_range<<<std::min(grid_for((long long)n_elem * n_base), 65536), kBlock, 0, s>>>((long long)n_elem * n_base,
                                                                                        de, n, flag.p);
  MH_HIP(hipGetLastError());
  int bad = 0;
  MH_TRY(read_flag(flag.p, &bad, s));
  if (bad) {
    set_error("element connectivity holds a node id outside 0..%d", n - 1);
    return -2;
  }
  // element offsets into Ke: exclusive sum of (sum of the nodes' block sizes)^2
  DevArray<long long> sz, koff;
  MH_TRY(sz.alloc((size_t)n_elem + 1));
  MH_TRY(koff.alloc((size_t)n_elem + 1));
  MH_HIP(hipMemsetAsync(sz.p + n_elem, 0, sizeof(long long), s));
  k_v_elem_sizes<<<grid_for(n_elem), kBlock, 0, s>>>(n_elem, n_base, de, Vb.list.p, sz.p);
  MH_HIP(hipGetLastError());
  size_t scan_bytes = 0;
  MH_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, sz.p, koff.p, n_elem + 1, s));
  DevArray<unsigned char> scan_tmp;
  MH_TRY(scan_tmp.alloc(scan_bytes ? scan_bytes : 1));
  MH_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp.p, scan_bytes, sz.p, koff.p, n_elem + 1, s));
  long long total = 0;
  MH_HIP(hipMemcpyAsync(&total, koff.p + n_elem, sizeof(long long), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  DevArray<V> kt;
  const V* dk = Ke;
  if (!is_device_pointer(Ke)) {
    MH_TRY(kt.alloc((size_t)total + 1));
    MH_TRY(upload(kt.p, Ke, (size_t)total * sizeof(V), s));
    dk = kt.p;
  }
  const long long cap = (long long)chunk * pairs_elem;
  DevArray<unsigned long long> k0, k1;
  DevArray<int> i0, i1;
  MH_TRY(k0.alloc((size_t)cap));
  MH_TRY(k1.alloc((size_t)cap));
  MH_TRY(i0.alloc((size_t)cap));
  MH_TRY(i1.alloc((size_t)cap));
  const int end_bit = bits_for((unsigned long long)Vb.nzb) + 1;
  const unsigned long long none = 1ull << (end_bit - 1);
  size_t tmp_bytes = 0;
  MH_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, k0.p, k1.p, i0.p, i1.p, (int)cap, 0, end_bit, s));
  DevArray<unsigned char> tmp;
  MH_TRY(tmp.alloc(tmp_bytes ? tmp_bytes : 1));
  V* A = vb_values<V>(Vb).p;
  const int mm = Vb.maxb * Vb.maxb;
  for (int e0 = 0; e0 < n_elem; e0 += chunk) {
    const int ne = std::min(chunk, n_elem - e0);
    const long long m = (long long)ne * pairs_elem;
    k_elem_targets<<<grid_for(m), kBlock, 0, s>>>(ne, n_base, de + (size_t)e0 * n_base, Vb.index.p, Vb.item.p, k0.p,
                                                   i0.p, flag.p, none);
    MH_HIP(hipGetLastError());
    MH_TRY(read_flag(flag.p, &bad, s));
    if (bad) {
      set_error("element %d..%d couples nodes whose block is not in the nonzero pattern", e0, e0 + ne - 1);
      MH_TRY(vb_reexpand(M, A, s));  // earlier chunks stay added, as monolis stops there
      mark_values_changed(M);
      return -2;
    }
    size_t tb = tmp_bytes;
    MH_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, k0.p, k1.p, i0.p, i1.p, (int)m, 0, end_bit, s));
    k_v_elem_accumulate<V><<<grid_for(m * mm), kBlock, 0, s>>>(m, k1.p, i1.p, dk, koff.p + e0,
                                                                de + (size_t)e0 * n_base, n_base, Vb.maxb, n,
                                                                Vb.list.p, Vb.index.p, Vb.item.p, Vb.index2.p, A,
                                                                none);
    MH_HIP(hipGetLastError());
  }
  MH_TRY(vb_reexpand(M, A, s));
  mark_values_changed(M);
  return 0;
}

int matrix_add_elements(Matrix* M, int n_elem, int n_base, const int* elem, const double* Ke, hipStream_t s) {
  if (M->vb) return add_elements_V_T<double>(M, n_elem, n_base, elem, Ke, s);
  return add_elements_T<double>(M, n_elem, n_base, elem, Ke, s);
}
int matrix_add_elements_C(Matrix* M, int n_elem, int n_base, const int* elem, const zd* Ke, hipStream_t s) {
  if (M->vb) return add_elements_V_T<zd>(M, n_elem, n_base, elem, Ke, s);
  return add_elements_T<zd>(M, n_elem, n_base, elem, Ke, s);
}

template <typename V>
static int dirichlet_T(Matrix* M, V* rhs, int n_bc, const int* node, const int* dof, const V* val, hipStream_t s) {
  MH_TRY(require_assemblable(*M, "Dirichlet conditions", sizeof(V) == sizeof(zd)));
  if (n_bc < 0) {
    set_error("negative number of conditions");
    return -2;
  }
  if (n_bc == 0 || M->n == 0) return 0;
  const int b = M->b;
  DevArray<int> nt, dt;
  DevArray<V> vt;
  const int *dn = nullptr, *dd = nullptr;
  const V* dv = nullptr;
  MH_TRY(stage(node, (size_t)n_bc, nt, &dn, s));
  MH_TRY(stage(dof, (size_t)n_bc, dt, &dd, s));
  MH_TRY(stage(val, (size_t)n_bc, vt, &dv, s));
  DevArray<int> flag;
  MH_TRY(flag.alloc(2));
  MH_HIP(hipMemsetAsync(flag.p, 0, 2 * sizeof(int), s));
  k_check_range<<<std::min(grid_for(n_bc), 65536), kBlock, 0, s>>>(n_bc, dn, M->n, flag.p);
  k_check_range<<<std::min(grid_for(n_bc), 65536), kBlock, 0, s>>>(n_bc, dd, b, flag.p + 1);
  MH_HIP(hipGetLastError());
  int bad[2] = {0, 0};
  MH_HIP(hipMemcpyAsync(bad, flag.p, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (bad[0] || bad[1]) {
    set_error("Dirichlet condition outside the matrix (%s)", bad[0] ? "node id" : "DOF index");
    return -2;
  }
  MH_HIP(hipMemsetAsync(flag.p, 0, 2 * sizeof(int), s));
  k_bc_check_diag<<<grid_for(n_bc), kBlock, 0, s>>>(n_bc, dn, M->rowptr.p, M->csr_item.p, flag.p);
  MH_HIP(hipGetLastError());
  DevArray<int> isbc;  // per DOF, then per node
  DevArray<V> bcval;
  const size_t m = (size_t)M->n * b;
  MH_TRY(isbc.alloc(m + (size_t)M->n));
  MH_TRY(bcval.alloc(m));
  int* nodebc = isbc.p + m;
  MH_HIP(hipMemsetAsync(isbc.p, 0, (m + (size_t)M->n) * sizeof(int), s));
  k_bc_mark<V><<<grid_for(n_bc), kBlock, 0, s>>>(n_bc, dn, dd, dv, b, isbc.p, bcval.p, nodebc, flag.p + 1);
  MH_HIP(hipGetLastError());
  MH_HIP(hipMemcpyAsync(bad, flag.p, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (bad[0]) {
    // monolis stops (monolis_stop_by_set_DBC)
    set_error("Dirichlet condition on a node without a diagonal block");
    return -2;
  }
  if (bad[1]) {
    set_error("the same DOF is listed twice among the Dirichlet conditions");
    return -2;
  }
  DevArray<V> rtmp;
  V* dr = rhs;
  const bool rhs_dev = is_device_pointer(rhs);
  if (!rhs_dev) {
    MH_TRY(rtmp.alloc(m));
    MH_TRY(upload(rtmp.p, rhs, m * sizeof(V), s));
    dr = rtmp.p;
  }
  k_bc_apply<V><<<(M->n + kWave - 1) / kWave, kBlock, 0, s>>>(M->n, b, M->slice_ptr.p, M->rowptr.p, M->col.p, values_of<V>(M),
                                                  isbc.p, nodebc, bcval.p, dr);
  MH_HIP(hipGetLastError());
  if (!rhs_dev) MH_HIP(hipMemcpyAsync(rhs, dr, m * sizeof(V), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  mark_values_changed(M);
  return 0;
}

// Dirichlet conditions on a variable-block matrix (monolis's layout values kept
// in the VBlock, then the expansion and the diag_V factors are rebuilt).
template <typename V>
static int dirichlet_V_T(Matrix* M, V* rhs, int n_bc, const int* node, const int* dof, const V* val, hipStream_t s) {
  MH_TRY(require_vblock(*M, "Dirichlet conditions", sizeof(V) == sizeof(zd)));
  VBlock& Vb = *M->vb;
  if (n_bc < 0) {
    set_error("negative number of conditions");
    return -2;
  }
  if (n_bc == 0 || Vb.nb == 0) return 0;
  DevArray<int> nt, dt;
  DevArray<V> vt;
  const int *dn = nullptr, *dd = nullptr;
  const V* dv = nullptr;
  MH_TRY(stage(node, (size_t)n_bc, nt, &dn, s));
  MH_TRY(stage(dof, (size_t)n_bc, dt, &dd, s));
  MH_TRY(stage(val, (size_t)n_bc, vt, &dv, s));
  DevArray<int> flag;
  MH_TRY(flag.alloc(3));
  MH_HIP(hipMemsetAsync(flag.p, 0, 3 * sizeof(int), s));
  k_check_range<<<std::min(grid_for(n_bc), 65536), kBlock, 0, s>>>(n_bc, dn, Vb.nb, flag.p);
  k_check_range<<<std::min(grid_for(n_bc), 65536), kBlock, 0, s>>>(n_bc, dd, Vb.maxb, flag.p + 1);
  MH_HIP(hipGetLastError());
  int bad[3] = {0, 0, 0};
  MH_HIP(hipMemcpyAsync(bad, flag.p, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (bad[0] || bad[1]) {
    set_error("Dirichlet condition outside the matrix (%s)", bad[0] ? "node id" : "DOF index");
    return -2;
  }
  MH_HIP(hipMemsetAsync(flag.p, 0, 3 * sizeof(int), s));
  k_bc_check_diag<<<grid_for(n_bc), kBlock, 0, s>>>(n_bc, dn, Vb.index.p, Vb.item.p, flag.p);
  MH_HIP(hipGetLastError());
  const size_t m = (size_t)M->n;  // scalar rows = DOFs
  DevArray<int> isbc;
  DevArray<V> bcval;
  MH_TRY(isbc.alloc(m));
  MH_TRY(bcval.alloc(m));
  MH_HIP(hipMemsetAsync(isbc.p, 0, m * sizeof(int), s));
  k_v_bc_mark<V><<<grid_for(n_bc), kBlock, 0, s>>>(n_bc, dn, dd, dv, Vb.dof_index.p, Vb.list.p, isbc.p, bcval.p,
                                                   flag.p);
  MH_HIP(hipGetLastError());
  MH_HIP(hipMemcpyAsync(bad, flag.p, 3 * sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (bad[0]) {
    set_error("Dirichlet condition on a node without a diagonal block");
    return -2;
  }
  if (bad[2]) {  // monolis_stop_by_submatrix_access
    set_error("Dirichlet condition on a DOF beyond its node's block size");
    return -2;
  }
  if (bad[1]) {
    set_error("the same DOF is listed twice among the Dirichlet conditions");
    return -2;
  }
  DevArray<V> rtmp;
  V* dr = rhs;
  const bool rhs_dev = is_device_pointer(rhs);
  if (!rhs_dev) {
    MH_TRY(rtmp.alloc(m));
    MH_TRY(upload(rtmp.p, rhs, m * sizeof(V), s));
    dr = rtmp.p;
  }
  V* A = vb_values<V>(Vb).p;
  k_v_bc_apply<V><<<grid_for(Vb.nb), kBlock, 0, s>>>(Vb.nb, Vb.list.p, Vb.dof_index.p, Vb.index.p, Vb.item.p,
                                                     Vb.index2.p, A, isbc.p, bcval.p, dr);
  MH_HIP(hipGetLastError());
  if (!rhs_dev) MH_HIP(hipMemcpyAsync(rhs, dr, m * sizeof(V), hipMemcpyDeviceToHost, s));
  MH_TRY(vb_reexpand(M, A, s));
  mark_values_changed(M);
  return 0;
}

int matrix_dirichlet(Matrix* M, double* rhs, int n_bc, const int* node, const int* dof, const double* val,
                     hipStream_t s) {
  if (M->vb) return dirichlet_V_T<double>(M, rhs, n_bc, node, dof, val, s);
  return dirichlet_T<double>(M, rhs, n_bc, node, dof, val, s);
}
int matrix_dirichlet_C(Matrix* M, zd* rhs, int n_bc, const int* node, const int* dof, const zd* val, hipStream_t s) {
  if (M->vb) return dirichlet_V_T<zd>(M, rhs, n_bc, node, dof, val, s);
  return dirichlet_T<zd>(M, rhs, n_bc, node, dof, val, s);
}

template <typename V>
static int get_values_T(const Matrix& M, V* A, hipStream_t s) {
  if (M.vb && M.is_complex == (sizeof(V) == sizeof(zd))) {  // monolis's layout, kept in the VBlock
    const size_t nv = (size_t)M.vb->nzs;
    if (nv) MH_HIP(hipMemcpyAsync(A, vb_values<V>(*M.vb).p, nv * sizeof(V), hipMemcpyDefault, s));
    MH_HIP(hipStreamSynchronize(s));
    return 0;
  }
  if (M.vb || M.is_complex != (sizeof(V) == sizeof(zd))) {
    set_error("value read-back: %s fixed-block matrices only", sizeof(V) == sizeof(zd) ? "complex" : "real");
    return -2;
  }
  const size_t nv = (size_t)M.nz * M.b * M.b;
  if (nv == 0) return 0;
  DevArray<V> tmp;
  V* dA = A;
  const bool dev = is_device_pointer(A);
  if (!dev) {
    MH_TRY(tmp.alloc(nv));
    dA = tmp.p;
    if (M.n < M.np) MH_HIP(hipMemsetAsync(dA, 0, nv * sizeof(V), s));
  }
  if (M.n > 0) {
    MH_TRY(launch_sell_gather(M, values_of<V>(const_cast<Matrix*>(&M)), dA, s));
  }
  if (!dev) MH_HIP(hipMemcpyAsync(A, dA, nv * sizeof(V), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  return 0;
}

int matrix_get_values(const Matrix& M, double* A, hipStream_t s) { return get_values_T<double>(M, A, s); }
int matrix_get_values_C(const Matrix& M, zd* A, hipStream_t s) { return get_values_T<zd>(M, A, s); }

int matrix_get_pattern(const Matrix& M, int* index, int* item, hipStream_t s) {
  if (M.vb) {  // the block pattern, not the scalar expansion's
    const VBlock& V = *M.vb;
    if (index) MH_HIP(hipMemcpyAsync(index, V.index.p, sizeof(int) * ((size_t)V.npb + 1), hipMemcpyDefault, s));
    if (item && V.nzb > 0) MH_HIP(hipMemcpyAsync(item, V.item.p, sizeof(int) * (size_t)V.nzb, hipMemcpyDefault, s));
    MH_HIP(hipStreamSynchronize(s));
    return 0;
  }
  if (index) MH_HIP(hipMemcpyAsync(index, M.rowptr.p, sizeof(int) * ((size_t)M.np + 1), hipMemcpyDefault, s));
  if (item && M.nz > 0) MH_HIP(hipMemcpyAsync(item, M.csr_item.p, sizeof(int) * (size_t)M.nz, hipMemcpyDefault, s));
  MH_HIP(hipStreamSynchronize(s));
  return 0;
}

}  // namespace mh
