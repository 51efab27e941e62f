// How many workgroups solve a system on chip (host code without a GPU header).
#pragma once

#include <algorithm>
#include <exception>

namespace mh {

// Whether build() made its plan: one that fails (memory) or throws is a system
// that does not run on chip, not a failed call.
template <class F>
bool made_plan(F&& build) {
  try {
    return build() == 0;
  } catch (const std::exception&) {
    return false;
  }
}

constexpr int kResNT = 512;                 // threads per member: two wavefronts per SIMD, 256 VGPRs each
constexpr int kResNW = kResNT / 64;         // its wavefronts, one 64-row slice each at a time
constexpr int kResTeamMax = 128;            // workgroups per team at most (one wavefront polls 4 words of each)
constexpr int kResRowsLarge = 26;           // RP: 13,312 rows per member (150 VGPRs of vectors)
constexpr int kResRowsMini = 4;             // RP: 2,048 rows
constexpr int kResRowsSmall = 8;            // RP: 4,096 rows (with the matrix in registers: 208 VGPRs of data)

// Members of a system of nsl slices whose share of the launch is `fair`
// workgroups, on a GPU of `cus` CUs; 0: the system does not fit.
// More members than capacity asks for, while the system's share of the
// workgroups allows: down to one row per thread (7-point systems, us per
// iteration with 64 / 128 members: 48^3 10.3 / 8.1, 64^3 19.7 / 11.2, 78^3
// 34.8 / 19.8; 32^3 is flat from 32 to 128 at 7.0-7.3).  Up to four rows per
// thread one workgroup alone is faster (10^3: 4.0 against 5.7 with four
// members, 12^3: 4.5 against 6.0): a team's two exchanges cost about 1 us each.
// Never more than the CUs: a CU may have room for no more than one member, and
// a team's members wait for one another, so all of them have to run at once.
inline int res_members(int nsl, int fair, int cus) {
  const int most = std::min(kResTeamMax, cus);
  const int need = (nsl + kResRowsLarge * kResNW - 1) / (kResRowsLarge * kResNW);
  if (nsl < 1 || need > most) return 0;
  if (nsl <= kResRowsMini * kResNW) return 1;
  return std::max(need, std::min(std::min(most, fair), nsl / kResNW));
}

}  // namespace mh
