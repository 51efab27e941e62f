// Plans and launches of the on-chip CG (mh_resident.hpp).
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "mh_resident.hpp"

namespace mh {

namespace {

// One workgroup per member: marks the columns outside the member's rows in a
// bitmap of its system, numbers them (the halo list, ascending), flags the
// slices they lie in as exported, and writes every own entry's LDS index.
// Padding entries point at the zero behind the halo.
__global__ void __launch_bounds__(kResNT) k_res_build(ResMember* mem, const int* __restrict__ slice_ptr,
                                                      const int* __restrict__ g_ptr, const int* __restrict__ col,
                                                      const int* __restrict__ rowlen, const int* __restrict__ rowptr,
                                                      unsigned char* __restrict__ expf, int* __restrict__ halo,
                                                      uint4* __restrict__ lcol, int* __restrict__ bad) {
  extern __shared__ unsigned bits[];  // words, then the number of marked rows before each word
  __shared__ int wsum[kResNW];
  const ResMember m = mem[blockIdx.x];
  const int words = (m.sysrows + 31) / 32;
  int* pre = reinterpret_cast<int*>(bits + words);
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int m0 = m.row0 - m.sysrow0, m1 = m0 + m.nown;  // own rows inside the system
  auto len_of = [&](int s) {
    const int l = s * kWave + lane;
    if (l >= m.nown) return 0;
    return rowlen ? rowlen[(size_t)(m.slice0 + s) * kWave + lane] : rowptr[m.row0 + l + 1] - rowptr[m.row0 + l];
  };
  for (int i = threadIdx.x; i < words; i += kResNT) bits[i] = 0;
  __syncthreads();
  for (int s = w; s < m.nsl; s += kResNW) {
    const int k0 = slice_ptr[m.slice0 + s], len = len_of(s);
    for (int k = 0; k < len; ++k) {
      const int l = col[((size_t)k0 + k) * kWave + lane] - m.sysrow0;
      if (l < m0 || l >= m1) atomicOr(&bits[l >> 5], 1u << (l & 31));
    }
  }
  __syncthreads();
  // exclusive prefix of the words' counts: a chunk of words per thread
  const int per = (words + kResNT - 1) / kResNT, i0 = min(words, (int)threadIdx.x * per), i1 = min(words, i0 + per);
  int mine = 0;
  for (int i = i0; i < i1; ++i) mine += __popc(bits[i]);
  int scan = mine;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int v = __shfl_up(scan, o, kWave);
    if (lane >= o) scan += v;
  }
  if (lane == kWave - 1) wsum[w] = scan;
  __syncthreads();
  int base = scan - mine, total = 0;
  for (int k = 0; k < kResNW; ++k) {
    if (k < w) base += wsum[k];
    total += wsum[k];
  }
  for (int i = i0; i < i1; ++i) {
    pre[i] = base;
    base += __popc(bits[i]);
  }
  __syncthreads();
  if (total > m.halo_cap) {
    if (threadIdx.x == 0) atomicOr(bad, 1);
    return;
  }
  for (int i = threadIdx.x; i < words; i += kResNT) {
    unsigned v = bits[i];
    int rank = pre[i];
    while (v) {
      const int l = i * 32 + __ffs(v) - 1;
      v &= v - 1;
      halo[m.halo_off + rank++] = m.sysrow0 + l;
      expf[m.sysslice0 + l / kWave] = 1;
    }
  }
  if (threadIdx.x == 0) mem[blockIdx.x].nhalo = total;
  const int own = m.nsl * kWave;
  for (int s = w; s < m.nsl; s += kResNW) {
    const int k0 = slice_ptr[m.slice0 + s], wd = slice_ptr[m.slice0 + s + 1] - k0, len = len_of(s);
    for (int g = 0; g < (wd + 7) / 8; ++g) {
      unsigned c[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int k = g * 8 + u;
        c[u] = (unsigned)(own + total);
        if (k < len) {
          const int l = col[((size_t)k0 + k) * kWave + lane] - m.sysrow0;
          c[u] = l >= m0 && l < m1
                     ? (unsigned)(l - m0)
                     : (unsigned)(own + pre[l >> 5] + __popc(bits[l >> 5] & ((1u << (l & 31)) - 1)));
        }
      }
      lcol[((size_t)g_ptr[m.slice0 + s] + g) * kWave + lane] =
          make_uint4(c[0] | c[1] << 16, c[2] | c[3] << 16, c[4] | c[5] << 16, c[6] | c[7] << 16);
    }
  }
}

// Per-launch reset (a kernel, so that a captured graph holds no memset nodes).
// `abort`: no member of a team may wait at all.
__global__ void k_res_reset(int nsys, int* iters, double* resid, int* status, int* ctl, int abort, int* sticky,
                            unsigned long long* part, int npart) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nsys) {
    iters[i] = -1;
    resid[i] = 0.0;
    status[i] = -1;
  }
  if (i < 2) ctl[i] = i == 1 ? abort : 0;
  if (i == 0 && abort) *sticky = 1;
  if (i < npart) part[i] = 0;  // no tag of an earlier launch
}

// LDS of k_res_build's bitmap and its prefix (491,520 rows).
constexpr size_t kResBuildLds = (size_t)120 << 10;

// The attribute belongs to the kernel, which all plans of the process share: it
// is set to the most that any of them takes, never to one plan's own size (a
// smaller plan would lower it below what an earlier one launches with).
template <int RP, bool MR>
int occupancy(size_t lds, int* per_cu) {
  auto* k = &k_res_cg<RP, MR, false>;
  for (auto* f : {k, &k_res_cg<RP, MR, true>})
    MH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(kResLds * sizeof(double))));
  *per_cu = 0;
  MH_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, k, kResNT, lds));
  return 0;
}

}  // namespace

void ResPlan::clear() {
  fits = false;
  for (auto* d : {&mem, &expf, &lcol}) d->release();
  for (auto* d : {&halo, &g_ptr, &ctl, &sticky}) d->release();
  part.release();
}

static int build(ResPlan& plan, const std::vector<ResSystem>& sys, const int* slice_ptr, int nslices,
                 const int* d_slice_ptr, const int* d_col, const int* rowlen, const int* rowptr, int cus,
                 hipStream_t s) {
  double W = 0.0;
  int maxrows = 1;
  for (const ResSystem& q : sys) {
    W += q.work;
    maxrows = std::max(maxrows, q.rows);
  }
  const size_t build_lds = (size_t)((maxrows + 31) / 32) * 2 * sizeof(unsigned);
  if (maxrows > kResTeamMax * kResRowsLarge * kResNT || build_lds > kResBuildLds) return 0;
  struct Task {
    int sys, T;
    double d;
  };
  std::vector<Task> tasks;
  for (size_t k = 0; k < sys.size(); ++k) {
    const ResSystem& q = sys[k];
    const int T = res_members(q.nsl, (int)((double)cus * q.work / std::max(W, 1e-300)), cus);
    if (T == 0) return 0;
    tasks.push_back(Task{(int)k, T, ((double)q.rows / T + 1500.0) * std::cbrt((double)q.rows)});
  }
  std::stable_sort(tasks.begin(), tasks.end(), [](const Task& a, const Task& b) { return a.d > b.d; });
  std::vector<ResMember> mem;
  long long halo_total = 0;
  int nteam = 0, max_nsl = 0;
  for (const Task& t : tasks) {
    const ResSystem& q = sys[t.sys];
    const int team = t.T > 1 ? nteam++ : -1;
    for (int r = 0; r < t.T; ++r) {
      ResMember m{};
      const int a0 = (int)((long long)q.nsl * r / t.T), a1 = (int)((long long)q.nsl * (r + 1) / t.T);
      m.sys = t.sys;
      m.rank = r;
      m.T = t.T;
      m.team = team;
      m.slice0 = q.slice0 + a0;
      m.nsl = a1 - a0;
      m.row0 = q.row0 + a0 * kWave;
      m.nown = std::min(a1 * kWave, q.rows) - a0 * kWave;
      m.sysrow0 = q.row0;
      m.sysslice0 = q.slice0;
      m.sysrows = q.rows;
      m.halo_off = (int)halo_total;
      m.halo_cap = t.T > 1 ? std::min(kResLds - 1 - m.nsl * kWave, q.rows - m.nown) : 0;
      m.w8 = 1;
      for (int i = m.slice0; i < m.slice0 + m.nsl; ++i)
        if (slice_ptr[i + 1] - slice_ptr[i] > 8 || slice_ptr[i + 1] == slice_ptr[i]) m.w8 = 0;
      if (m.nsl > kResRowsLarge * kResNW || m.nown < 1) return 0;
      max_nsl = std::max(max_nsl, m.nsl);
      halo_total += m.halo_cap;
      if (halo_total >= (1LL << 31)) return 0;
      mem.push_back(m);
    }
  }
  std::vector<int> g_ptr((size_t)nslices + 1, 0);
  long long groups = 0;
  for (int i = 0; i < nslices; ++i) {
    g_ptr[i] = (int)groups;
    groups += (slice_ptr[i + 1] - slice_ptr[i] + 7) / 8;
    if (groups >= (1LL << 31)) return 0;
  }
  g_ptr[nslices] = (int)groups;
  plan.nmem = (int)mem.size();
  plan.nteam = nteam;
  MH_TRY(plan.mem.alloc(mem.size() * sizeof(ResMember)));
  MH_TRY(plan.expf.alloc((size_t)nslices));
  MH_TRY(plan.lcol.alloc((size_t)std::max(groups, 1LL) * kWave * sizeof(uint4)));
  MH_TRY(plan.halo.alloc((size_t)std::max(halo_total, 1LL)));
  MH_TRY(plan.g_ptr.alloc((size_t)nslices + 1));
  MH_TRY(plan.ctl.alloc(2));
  MH_TRY(plan.part.alloc((size_t)std::max(nteam, 1) * 8 * kResTeamMax));
  MH_TRY(plan.sticky.alloc(2));  // [1]: a halo that does not fit (build only)
  MH_TRY(upload(plan.mem.p, mem.data(), mem.size() * sizeof(ResMember), s));
  MH_TRY(upload(plan.g_ptr.p, g_ptr.data(), sizeof(int) * ((size_t)nslices + 1), s));
  MH_HIP(hipMemsetAsync(plan.expf.p, 0, (size_t)nslices, s));
  MH_HIP(hipMemsetAsync(plan.sticky.p, 0, 2 * sizeof(int), s));
  MH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_res_build), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)kResBuildLds));
  k_res_build<<<plan.nmem, kResNT, build_lds, s>>>((ResMember*)plan.mem.p, d_slice_ptr, plan.g_ptr.p, d_col, rowlen,
                                                   rowptr, plan.expf.p, plan.halo.p, (uint4*)plan.lcol.p,
                                                   plan.sticky.p + 1);
  MH_HIP(hipGetLastError());
  int bad[2] = {0, 0};
  MH_HIP(hipMemcpyAsync(mem.data(), plan.mem.p, mem.size() * sizeof(ResMember), hipMemcpyDeviceToHost, s));
  MH_HIP(hipMemcpyAsync(bad, plan.sticky.p, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (bad[1]) return 0;
  // Members of at most kResRowsSmall rows per thread: the matrix in registers
  // too (and x in LDS) if every row has at most 8 entries, else two workgroups
  // per CU.
  const bool small = max_nsl <= kResRowsSmall * kResNW;
  int lds = 0, lds_mr = 0;
  bool w8 = true;
  for (const ResMember& m : mem) {
    lds = std::max(lds, m.nsl * kWave + m.nhalo + 1);
    lds_mr = std::max(lds_mr, 2 * m.nsl * kWave + m.nhalo + 1);
    w8 = w8 && m.w8;
  }
  const bool mini = max_nsl <= kResRowsMini * kResNW && w8;
  plan.mr = mini || (small && w8 && lds_mr <= kResLds);
  plan.lds_bytes = (size_t)(plan.mr && !mini ? lds_mr : lds) * sizeof(double);
  int per_cu = 0;
  plan.rp = mini ? kResRowsMini : plan.mr || (small && plan.lds_bytes <= ((size_t)79 << 10)) ? kResRowsSmall : kResRowsLarge;
  if (mini) MH_TRY((occupancy<kResRowsMini, true>(plan.lds_bytes, &per_cu)));
  else if (plan.mr) MH_TRY((occupancy<kResRowsSmall, true>(plan.lds_bytes, &per_cu)));
  else if (plan.rp == kResRowsSmall) MH_TRY((occupancy<kResRowsSmall, false>(plan.lds_bytes, &per_cu)));
  else MH_TRY((occupancy<kResRowsLarge, false>(plan.lds_bytes, &per_cu)));
  if (per_cu < 1) return 0;
  plan.grid = std::min(plan.nmem, per_cu * cus);
  int dev = 0, khz = 0;
  MH_HIP(hipGetDevice(&dev));
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0) khz = 100000;
  plan.ticks_per_s = (double)khz * 1000.0;
  plan.fits = true;
  return 0;
}

void res_plan_build(ResPlan& plan, const std::vector<ResSystem>& sys, const int* slice_ptr, int nslices,
                    const int* d_slice_ptr, const int* d_col, const int* rowlen, const int* rowptr, int cus,
                    hipStream_t s) {
  plan.fits = false;
  if (!made_plan([&] {
        return build(plan, sys, slice_ptr, nslices, d_slice_ptr, d_col, rowlen, rowptr, cus, s);
      })) {
    plan.fits = false;
    clear_error();
  }
  if (!plan.fits) plan.clear();
}

int res_launch(const ResPlan& plan, const int* d_slice_ptr, const double* val, const double* dinv, const ResArgs& a,
               int nsys, double wait_s, hipStream_t s) {
  const int npart = plan.nteam * 8 * kResTeamMax;
  k_res_reset<<<(std::max(nsys, npart + 2) + kBlock - 1) / kBlock, kBlock, 0, s>>>(
      nsys, a.out.iters, a.out.resid, a.out.status, plan.ctl.p, plan.nteam > 0 && wait_s == 0.0, plan.sticky.p,
      plan.part.p, npart);
  MH_HIP(hipGetLastError());
  const ResView V{plan.nmem, (const ResMember*)plan.mem.p, d_slice_ptr, plan.g_ptr.p, val, (const uint4*)plan.lcol.p,
                  plan.expf.p, dinv, plan.halo.p, plan.ctl.p, plan.part.p, (long long)(plan.ticks_per_s * wait_s),
                  plan.sticky.p};
  auto launch = [&](auto rp, auto mr) {
    auto* k = a.ticks ? &k_res_cg<decltype(rp)::value, decltype(mr)::value, true>
                      : &k_res_cg<decltype(rp)::value, decltype(mr)::value, false>;
    k<<<plan.grid, kResNT, plan.lds_bytes, s>>>(V, a);
  };
  using Mini = std::integral_constant<int, kResRowsMini>;
  using Small = std::integral_constant<int, kResRowsSmall>;
  using Large = std::integral_constant<int, kResRowsLarge>;
  if (plan.rp == kResRowsMini) launch(Mini{}, std::true_type{});
  else if (plan.mr) launch(Small{}, std::true_type{});
  else if (plan.rp == kResRowsSmall) launch(Small{}, std::false_type{});
  else launch(Large{}, std::false_type{});
  MH_HIP(hipGetLastError());
  return 0;
}

int res_aborted(ResPlan& plan, int* aborted, hipStream_t s) {
  int flag = 0;
  MH_HIP(hipMemcpyAsync(&flag, plan.sticky.p, sizeof(int), hipMemcpyDeviceToHost, s));
  MH_HIP(hipStreamSynchronize(s));
  if (flag) {
    MH_HIP(hipMemsetAsync(plan.sticky.p, 0, sizeof(int), s));
    MH_HIP(hipStreamSynchronize(s));
  }
  *aborted = flag != 0;
  return 0;
}

}  // namespace mh
