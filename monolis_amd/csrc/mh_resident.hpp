// On-chip CG: a scalar system solved by one workgroup, or by a team of them,
// whose vectors never leave the CUs.
//
// A member owns a contiguous range of the system's 64-row slices, at most
// RP * 8 of them.  p of its rows and of the rows it couples to (its halo) lives
// in LDS; x, r and q / z live in registers, RP rows per thread.  An iteration
// then streams only the matrix -- 8 bytes of value and 2 bytes of LDS index per
// entry -- and the preconditioner's 8 bytes per row: about 80 bytes per row of a
// 7-point system against 190 with the vectors in memory.  512 Poisson systems of
// 10^3..40^3 rows: 51.1 -> 17.6 ms, 1.377e9 row-iterations at 78 G/s (6.3 TB/s of
// those bytes): bound by the matrix stream.  A single 32^3 system: 1.93 -> 0.77
// ms (17.7 -> 7.0 us per iteration, three launches before): bound by the two
// exchanges and the halo loads, about 1 us each, and the sums' serial chains.
//
// Team members exchange two things, through agent-scope stores and loads that
// bypass the XCD's L2 (no cache write-back or invalidation): the partial sums of
// the two reductions of an iteration, and z of the rows some other member
// reads.  Every member updates its copy of a halo row's p as its owner does,
// p = z + beta p, so p itself is never exchanged.
//
// Members of at most kResRowsSmall * 512 rows of up to 8 entries also keep their
// part of the matrix in registers (MR): an iteration then touches no memory but
// the exchange.
#pragma once

#include <memory>
#include <vector>

#include "mh_internal.hpp"
#include "mh_kernels.hpp"
#include "mh_resident_plan.hpp"

namespace mh {

constexpr int kResLds = 20320;              // doubles of LDS for p (158.75 KB of the CU's 160)
constexpr int kResSpinMax = 1 << 24;        // polls of one team wait at most (a bound that needs no clock)
constexpr int kResIterRR = 200;             // residual replacement (CG.f90:91-95)

struct ResMember {
  int sys, rank, T, team;
  int slice0, nsl;      // own slices
  int row0, nown;       // first own row (global) and own rows
  int sysrow0, sysslice0, sysrows;
  int halo_off, halo_cap, nhalo;
  int w8;               // no own slice is wider than 8 slots
  int pad;
};

struct ResView {
  int nmem;
  const ResMember* mem;
  const int* slice_ptr;   // SELL slot offsets
  const int* g_ptr;       // per slice: first group of 8 LDS indices
  const double* val;      // SELL values, one plane per slot
  const uint4* lcol;      // per group and lane: 8 16-bit LDS indices
  const unsigned char* expf;  // per slice: some other member reads a row of it
  const double* dinv;     // diagonal preconditioner per row
  const int* halo;        // global rows, per member
  int* ctl;               // [0] next member, [1] abort flag
  unsigned long long* part;  // per team: 2 alternating sets x kResTeamMax x 4 tagged halves of two sums
  long long limit;        // wall-clock ticks one wait may last
  int* sticky;            // set with the abort flag, cleared only by the host
};

// Per-system results.
struct BatchOut {
  int* iters;
  double* resid;
  int* status;   // 0 converged, 1 not converged, 2 zero rhs, 3 a team wait gave up
};

struct ResArgs {
  const double* b;
  double* x;
  double* z;       // exported z (written for exported slices only)
  double* p;       // p and x during a residual replacement
  double* xe;
  BatchOut out;
  double* hist;    // residual history of the only system, or null
  long long* ticks;  // timed solves of one system: wall-clock ticks of the products, of the
                     // update and preconditioner passes, and of the whole solve
  int max_iter;
  double tol;
  int init_x, precond;
};

// Workgroup state beside the LDS vector.
struct ResShared {
  double red[2][2 * kResNW];
  double tot[2];
  int ok, next;
};

__device__ __forceinline__ void st_agent(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_agent(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The value itself, as something the compiler cannot carry over from an earlier
// use: the per-row addresses and conditions of an unrolled pass are then formed
// in the pass, instead of being kept for the whole solve (RP of each, which
// spilled thousands of registers).
__device__ __forceinline__ int fresh_s(int v) {
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
  return v;
}
__device__ __forceinline__ int fresh_v(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// i * 8 < left as a condition of its own: the compiler would otherwise thread
// the branches of an unrolled pass (one that fails implies the rest), which
// multiplies its code and its live registers.
__device__ __forceinline__ bool res_on(int left, int i) {
  asm volatile("" : "+s"(left));
  return i * kResNW < left;
}

// One member's part of one system.  TIMED: the first wavefront of the first member
// also sums the time its products and its update and preconditioner passes take
// (the same operations in the same order otherwise).
template <int RP, bool W8, bool MR, bool TIMED>
__device__ __forceinline__ void res_cg(const ResView& V, const ResMember& m, const ResArgs& a, double* lds,
                                       ResShared& sh) {
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int own = m.nsl * kWave;  // LDS: own rows (whole slices), halo rows, one zero
  const int T = m.T;
  // Row i of a thread: slice w + i*8 of the member, its lane.  With eight rows of
  // the matrix in registers x lies in LDS, behind p; with four the preconditioner
  // and the first halo rows' numbers are held in registers too.
  constexpr bool XL = MR && RP > kResRowsMini, KEEP = MR && RP <= kResRowsMini;
  constexpr int HU = 4;  // halo rows per thread and step
  double x[XL ? 1 : RP], r[RP], q[RP], dreg[KEEP ? RP : 1];
  int hreg[KEEP ? HU : 1];
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    if constexpr (!XL) x[i] = 0.0;
    r[i] = q[i] = 0.0;
  }
  double* xl = lds + own + m.nhalo + 1;
  auto xv = [&](int i, int l) -> double& {
    if constexpr (XL) return xl[l];
    else return x[i];
  };
  // lane i holds the slot and group offsets and the export bit of slice w + i*8
  int kreg = 0, wreg = 1, greg = 0;
  bool ereg = false;
  {
    const int s = w + lane * kResNW;
    if (lane < RP && s < m.nsl) {
      kreg = V.slice_ptr[m.slice0 + s];
      wreg = V.slice_ptr[m.slice0 + s + 1] - kreg;
      greg = V.g_ptr[m.slice0 + s];
      ereg = T > 1 && V.expf[m.slice0 + s] != 0;
    }
  }
  const unsigned long long exports = __ballot(ereg);
  // A pass over the thread's rows: f(i, l, real, g) with l the row's LDS index,
  // real whether it is a row of the system, g its global row (lanes past the
  // system's last row take that row).
  auto for_rows = [&](auto&& f) {
    const int left = fresh_s(m.nsl - w), l0 = fresh_v(w * kWave + lane), g0 = fresh_s(m.row0), last = fresh_s(m.nown - 1);
#pragma unroll
    for (int i = 0; i < RP; ++i)
      if (res_on(left, i)) {
        const int l = l0 + i * (kResNW * kWave);
        f(i, l, l <= last, g0 + (l < last ? l : last));
      }
  };

  // ---- reductions -------------------------------------------------------------
  // Sums two values over the system: wavefront butterfly, wavefronts in order,
  // members by one butterfly over their ranks -- the same bits in every member.
  // A member posts its sums as four 64-bit words, each half of a value with the
  // number of the reduction as a tag; one wavefront of every member polls the
  // words of all members and has the values as soon as the tags agree, without
  // a counter or a second round trip.  Two alternating sets: a set is rewritten
  // after a reduction that every member joined having read it.  The exported
  // rows' write-through stores are waited for before the sums are posted, so a
  // member that has read them may load those rows.
  // Bounded: a wait that gives up raises the abort flag, after which every wait
  // of the launch ends.  (Decisions taken from LDS values go through
  // readfirstlane: the branches are uniform; a divergent loop exit would copy
  // every live register.)
  unsigned epoch = 0;
  auto sum = [&](double& s0, double& s1) -> bool {
    ++epoch;
    double* red = sh.red[epoch & 1];
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    if (lane == 0) {
      red[2 * w] = s0;
      red[2 * w + 1] = s1;
    }
    if (T > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    s0 = red[0];
    s1 = red[1];
#pragma unroll
    for (int k = 1; k < kResNW; ++k) {
      s0 += red[2 * k];
      s1 += red[2 * k + 1];
    }
    if (T == 1) return true;
    if (w == 0) {
      unsigned long long* ps = V.part + ((size_t)m.team * 2 + (epoch & 1)) * (4 * kResTeamMax);
      if (lane < 4) {
        const unsigned long long v = __double_as_longlong(lane < 2 ? s0 : s1);
        const unsigned half = (lane & 1) ? (unsigned)(v >> 32) : (unsigned)v;
        __hip_atomic_store(ps + 4 * m.rank + lane, (unsigned long long)epoch << 32 | half, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
      constexpr int NL = 4 * kResTeamMax / kWave;  // words per lane
      unsigned long long word[NL];
      bool ok = true;
      long long t0 = 0;
      for (int k = 0;; ++k) {
        bool all = true;
#pragma unroll
        for (int u = 0; u < NL; ++u) {
          const int i = u * kWave + lane;
          word[u] = (unsigned long long)epoch << 32;
          if (u * kWave < 4 * T)
            word[u] = __hip_atomic_load(ps + (i < 4 * T ? i : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int u = 0; u < NL; ++u) all &= (unsigned)(word[u] >> 32) == epoch;
        if (__all(all)) break;
        if ((k & 15) == 15) {  // the clock and the abort flag every 16 polls
          const long long now = (long long)wall_clock64();
          if (t0 == 0) t0 = now;
          if (__hip_atomic_load(V.ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || k >= kResSpinMax ||
              now - t0 > V.limit) {
            __hip_atomic_store(V.ctl + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(V.sticky, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ok = false;
            break;
          }
        }
      }
      // lanes 4k, 4k+1 hold the halves of a member's first sum, 4k+2, 4k+3 of its second
      double tot = 0.0;
#pragma unroll
      for (int u = 0; u < NL; ++u) {
        const unsigned mine = (unsigned)word[u];
        const unsigned other = (unsigned)__builtin_amdgcn_update_dpp(0, (int)mine, 0xB1, 0xf, 0xf, true);  // lane ^ 1
        const unsigned long long v = (lane & 1) ? (unsigned long long)mine << 32 | other
                                                : (unsigned long long)other << 32 | mine;
        tot += u * kWave + lane < 4 * T ? __longlong_as_double(v) : 0.0;
      }
      tot += dpp_move<0x114>(tot);  // row_shr 4 and 8: lanes 12..15 of a row sum its four members
      tot += dpp_move<0x118>(tot);
      const double tot0 = (read_lane(tot, 12) + read_lane(tot, 28)) + (read_lane(tot, 44) + read_lane(tot, 60));
      const double tot1 = (read_lane(tot, 14) + read_lane(tot, 30)) + (read_lane(tot, 46) + read_lane(tot, 62));
      if (lane == 0) {
        sh.tot[0] = tot0;
        sh.tot[1] = tot1;
      }
      if (lane == 0) sh.ok = ok;
    }
    __syncthreads();
    s0 = sh.tot[0];
    s1 = sh.tot[1];
    return __builtin_amdgcn_readfirstlane(sh.ok) != 0;
  };

  // ---- q = A v for v in LDS -----------------------------------------------------
  auto unpack = [](const uint4& c, int u) {
    const unsigned wd = u < 2 ? c.x : u < 4 ? c.y : u < 6 ? c.z : c.w;
    return (u & 1) ? wd >> 16 : wd & 0xffffu;
  };
  // Slots past the slice's width re-read its last slot; their index is the zero
  // entry.  Offsets are formed in scalar registers, the lane's part in one vector.
  auto fetch = [&](int k0, int left, int g, int ln, uint4& c, double(&v)[8]) {
    c = (V.lcol + (size_t)g * kWave)[ln];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      v[u] = __builtin_nontemporal_load((V.val + (size_t)(k0 + (u < left ? u : left - 1)) * kWave) + ln);
  };
  auto accumulate = [&](const uint4& c, const double(&v)[8], double& acc) {
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = fma(v[u], lds[unpack(c, u)], acc);
  };
  uint4 mc[MR ? RP : 1];
  double mv[MR ? RP : 1][8];
  if constexpr (MR) {
    const int left = fresh_s(m.nsl - w);
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      mc[i] = make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 8; ++u) mv[i][u] = 0.0;
      if (res_on(left, i))
        fetch(__builtin_amdgcn_readlane(kreg, i), __builtin_amdgcn_readlane(wreg, i),
              __builtin_amdgcn_readlane(greg, i), lane, mc[i], mv[i]);
    }
  }
  auto product = [&]() {
    const int left = fresh_s(m.nsl - w), ln = fresh_v(lane);
    if constexpr (MR) {
#pragma unroll
      for (int i = 0; i < RP; ++i)
        if (res_on(left, i)) {
          uint4 c = mc[i];  // unpacked here, not once for the solve
          asm volatile("" : "+v"(c.x), "+v"(c.y), "+v"(c.z), "+v"(c.w));
          double acc = 0.0;
          accumulate(c, mv[i], acc);
          q[i] = acc;
        }
      return;
    }
    const int kr = fresh_v(kreg), wr = fresh_v(wreg), gr = fresh_v(greg);
    auto slot = [&](int i) { return __builtin_amdgcn_readlane(kr, i); };
    auto width = [&](int i) { return __builtin_amdgcn_readlane(wr, i); };
    auto group = [&](int i) { return __builtin_amdgcn_readlane(gr, i); };
    if constexpr (W8) {
      // the next slice's entries are in flight while this one's are used
      uint4 c[2];
      double v[2][8];
      if (left > 0) fetch(slot(0), width(0), group(0), ln, c[0], v[0]);
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        if (res_on(left, i)) {
          if (i + 1 < RP && res_on(left, i + 1))
            fetch(slot(i + 1), width(i + 1), group(i + 1), ln, c[(i + 1) & 1], v[(i + 1) & 1]);
          double acc = 0.0;
          accumulate(c[i & 1], v[i & 1], acc);
          q[i] = acc;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        if (res_on(left, i)) {
          const int k0 = slot(i), g0 = group(i), wd = width(i);
          double acc = 0.0;
          for (int k = 0; k < wd; k += 8) {
            uint4 c;
            double v[8];
            fetch(k0 + k, wd - k, g0 + k / 8, ln, c, v);
            accumulate(c, v, acc);
          }
          q[i] = acc;
        }
      }
    }
  };
  const int* halo = V.halo + m.halo_off;
  // LDS <- the vector whose own rows are f(i, l, g) and whose halo rows are in `src`
  auto load_vec = [&](auto&& f, const double* src) {
    for_rows([&](int i, int l, bool, int g) { lds[l] = f(i, l, g); });
    for (int h = threadIdx.x; h < m.nhalo; h += kResNT) lds[own + h] = src ? ld_agent(src + halo[h]) : 0.0;
    __syncthreads();
  };
  if constexpr (KEEP) {
    for_rows([&](int i, int, bool, int g) { dreg[i] = a.precond ? V.dinv[g] : 1.0; });
#pragma unroll
    for (int u = 0; u < HU; ++u) {
      const int h = threadIdx.x + u * kResNT;
      hreg[u] = m.nhalo > 0 ? halo[h < m.nhalo ? h : 0] : 0;
    }
  }
  auto fail = [&]() {
    if (threadIdx.x == 0)
      __hip_atomic_fetch_max(a.out.status + m.sys, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto store_x = [&](bool zero) {
    for_rows([&](int i, int l, bool real, int g) {
      if (real) a.x[g] = zero ? 0.0 : xv(i, l);
    });
  };
  long long t_start = 0, t_lap = 0, t_product = 0, t_update = 0;
  // the time since the last call, after which q holds its results
  auto lap = [&]() {
#pragma unroll
    for (int i = 0; i < RP; ++i) asm volatile("" : "+v"(q[i]));
    const long long now = (long long)wall_clock64(), d = now - t_lap;
    t_lap = now;
    return d;
  };
  if constexpr (TIMED) t_start = (long long)wall_clock64();
  auto finish = [&](int iters, double resid, int st) {
    if (threadIdx.x == 0) {
      if (m.rank == 0) {
        if constexpr (TIMED) {
          a.ticks[0] = t_product;
          a.ticks[1] = t_update;
          a.ticks[2] = (long long)wall_clock64() - t_start;
        }
        a.out.iters[m.sys] = iters;
        a.out.resid[m.sys] = resid;
      }
      __hip_atomic_fetch_max(a.out.status + m.sys, st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  if (threadIdx.x == 0) lds[own + m.nhalo] = 0.0;
  const bool init = a.init_x != 0;
  for_rows([&](int i, int l, bool, int g) { xv(i, l) = init ? 0.0 : a.x[g]; });
  load_vec([&](int i, int l, int) { return xv(i, l); }, init ? nullptr : a.x);
  // One loop body holds the only matrix product and the only preconditioner
  // pass.  LDS holds x when `resid_step` (the initial residual and the
  // replacement every 200 iterations), else p.
  bool resid_step = true;
  double B2 = 0.0, rho = 0.0, beta = 0.0, resid = 1.0;
  int it = 0;
  for (;;) {
    if constexpr (TIMED) lap();
    product();
    if constexpr (TIMED) t_product += lap();
    double rr = 0.0, rz = 0.0, none = 0.0;
    double alpha = 0.0;
    if (!resid_step) {
      for_rows([&](int i, int l, bool, int) { rr = fma(lds[l], q[i], rr); });
      if (!sum(rr, none)) return fail();
      alpha = rho / rr;  // (p, q)
      rr = 0.0;
      for_rows([&](int i, int l, bool, int) { xv(i, l) = fma(alpha, lds[l], xv(i, l)); });
      if (it % kResIterRR == 0) {
        // the true residual: p is set aside while LDS holds x
        for_rows([&](int i, int l, bool real, int g) {
          if (real) {
            st_agent(a.p + g, lds[l]);
            st_agent(a.xe + g, xv(i, l));
          }
        });
        if (T == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        double none2 = 0.0;
        if (!sum(none, none2)) return fail();
        load_vec([&](int i, int l, int) { return xv(i, l); }, a.xe);
        resid_step = true;
        continue;
      }
    }
    // r, then z = M^-1 r (kept in q's registers), (r, r), (r, z); z of exported slices goes out
    if constexpr (TIMED) lap();
    for_rows([&](int i, int, bool real, int g) {
      double d;
      if constexpr (KEEP) d = dreg[i];
      else d = a.precond ? V.dinv[g] : 1.0;
      double rv = resid_step ? a.b[g] - q[i] : fma(-alpha, q[i], r[i]);
      rv = real ? rv : 0.0;
      const double zv = a.precond ? d * rv : rv;
      r[i] = rv;
      q[i] = zv;
      rr = fma(rv, rv, rr);
      rz = fma(rv, zv, rz);
      if ((exports >> i) & 1)
        if (real) st_agent(a.z + g, zv);
    });
    if constexpr (TIMED) t_update += lap();
    if (resid_step) {
      __syncthreads();  // LDS reads of the product are done
      load_vec([&](int, int, int g) { return it > 0 ? ld_agent(a.p + g) : 0.0; }, it > 0 ? a.p : nullptr);
      resid_step = false;
    }
    if (!sum(rr, rz)) return fail();
    if (it == 0) {
      B2 = rr;
      if (__builtin_amdgcn_readfirstlane(B2 == 0.0)) {  // mat_converge.f90:40-48
        store_x(true);
        return finish(0, 0.0, 2);
      }
    } else {
      resid = sqrt(rr / B2);
      if (a.hist && m.rank == 0 && threadIdx.x == 0) a.hist[it] = resid;
      const bool conv = __builtin_amdgcn_readfirstlane(resid < a.tol);
      if (conv || it >= a.max_iter) {
        store_x(false);
        return finish(it, resid, conv ? 0 : 1);
      }
      beta = rz / rho;
    }
    rho = rz;
    ++it;
    // p = z + beta p (CG.f90:80-84; p = 0 before the first iteration), own rows and halo copies
    auto halo_step = [&](int h0, auto&& row) {
      double zv[HU];
#pragma unroll
      for (int u = 0; u < HU; ++u) zv[u] = ld_agent(a.z + row(u, h0 + u * kResNT));
#pragma unroll
      for (int u = 0; u < HU; ++u) {
        const int h = h0 + u * kResNT;
        if (h < m.nhalo) lds[own + h] = fma(beta, lds[own + h], zv[u]);
      }
    };
    auto listed = [&](int, int h) { return halo[h < m.nhalo ? h : 0]; };
    int h0 = threadIdx.x;
    if constexpr (KEEP) {
      if (h0 < m.nhalo) halo_step(h0, [&](int u, int) { return hreg[u]; });
      h0 += HU * kResNT;
    }
    for (; h0 < m.nhalo; h0 += HU * kResNT) halo_step(h0, listed);
    for_rows([&](int i, int l, bool, int) { lds[l] = fma(beta, lds[l], q[i]); });
    __syncthreads();
  }
}

// Persistent: workgroups take members in order from one counter.  A team's
// members are consecutive, so at most one team is incomplete at any time and a
// member waiting for a teammate that has not started waits only for running
// workgroups to finish their own complete teams.  Members of teams that start
// after a wait gave up report it at once (the workgroup's first thread alone: a
// branch around the solver's call raised its spilled registers from 8 to 37).
template <int RP, bool MR, bool TIMED>
__global__ void __launch_bounds__(kResNT) __attribute__((amdgpu_waves_per_eu(RP <= kResRowsSmall && !MR ? 4 : 2)))
    k_res_cg(ResView V, ResArgs a) {
  extern __shared__ double res_lds[];
  __shared__ ResShared sh;
  for (;;) {
    if (threadIdx.x == 0) {
      auto take = [&]() { return __hip_atomic_fetch_add(V.ctl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
      // both on their way at once
      const int aborted = __hip_atomic_load(V.ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int k = take();
      if (aborted != 0)
        for (; k < V.nmem && V.mem[k].T > 1; k = take())
          __hip_atomic_fetch_max(a.out.status + V.mem[k].sys, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.next = k;
    }
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(sh.next);
    if (k >= V.nmem) break;
    const ResMember m = V.mem[k];
    if constexpr (MR) {
      res_cg<RP, true, true, TIMED>(V, m, a, res_lds, sh);
    } else {
      if (m.w8) res_cg<RP, true, false, TIMED>(V, m, a, res_lds, sh);
      else res_cg<RP, false, false, TIMED>(V, m, a, res_lds, sh);
    }
    __syncthreads();
  }
}

// One system of a plan.
struct ResSystem {
  int slice0, nsl, row0, rows;
  double work;  // estimated work of the system (any unit)
};

// Members, halo lists and LDS indices of a set of systems (per pattern).
struct ResPlan {
  bool fits = false;
  int nmem = 0, nteam = 0, grid = 0, rp = 0;
  bool mr = false;  // the members' matrix stays in registers
  size_t lds_bytes = 0;
  double ticks_per_s = 0;
  DevArray<unsigned char> mem, expf, lcol;
  DevArray<int> halo, g_ptr, ctl, sticky;
  DevArray<unsigned long long> part;
  void clear();  // no plan, no memory
};

// slice_ptr: host slot offsets of every slice; d_slice_ptr / d_col: the device
// arrays (global 0-based columns); rowlen (per SELL row) or rowptr (per row)
// gives the row lengths.  Plan.fits is false when a system needs more members than
// a team may have or a member's rows and halo exceed LDS.  cus: the GPU's CUs, the
// workgroups that the systems share.  A plan that does not fit, or that there is
// no memory for, is cleared.
void res_plan_build(ResPlan& plan, const std::vector<ResSystem>& sys, const int* slice_ptr, int nslices,
                   const int* d_slice_ptr, const int* d_col, const int* rowlen, const int* rowptr, int cus,
                   hipStream_t s);
// Zeroes the counters and enqueues the solver (both capturable).  A wait of a
// team's member for another lasts at most wait_s seconds; 0: teams give up at once.
// With a.ticks the solve is timed.
int res_launch(const ResPlan& plan, const int* d_slice_ptr, const double* val, const double* dinv, const ResArgs& a,
               int nsys, double wait_s, hipStream_t s);
// 1 when a team wait gave up in any launch since the last call (synchronises).
int res_aborted(ResPlan& plan, int* aborted, hipStream_t s);

}  // namespace mh
