"""Team sizes of the on-chip CG (monolis_amd/csrc/mh_resident_plan.hpp), compiled for the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "mh_resident_plan.hpp"
using namespace mh;
int main() {
  const int cap = kResRowsLarge * kResNW;
  for (int cus : {1, 2, 8, 32, 38, 64, 127, 128, 256})
    for (int nsl = 0; nsl <= cap * 130; nsl += nsl < 600 ? 1 : 37)
      for (int fair : {0, 1, 3, cus / 2, cus}) {
        const int T = res_members(nsl, fair, cus), most = kResTeamMax < cus ? kResTeamMax : cus;
        const bool can = nsl >= 1 && (long long)nsl <= (long long)cap * most;
        // as many as run at once, none without a slice, none with more than it can hold
        if ((T > 0) != can || T > most || T > nsl || (T > 0 && (nsl + T - 1) / T > cap) ||
            (T > 1 && nsl <= kResRowsMini * kResNW)) {
          std::printf("cus %d nsl %d fair %d: %d members\n", cus, nsl, fair, T);
          return 1;
        }
      }
  // one 32^3 system on 256 CUs, on 32 of them (a partition), and as one of many systems
  std::printf("%d %d %d\n", res_members(512, 256, 256), res_members(512, 32, 32), res_members(512, 1, 256));
  return 0;
}
"""


def _run(tmp_path, program):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(program)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "monolis_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
    return r.stdout.split()


def test_a_plan_without_memory_is_no_plan_and_no_error(tmp_path):
    _run(tmp_path, r"""
#include <new>
#include <vector>
#include "mh_resident_plan.hpp"
int main() {
  const bool ok = mh::made_plan([] { return 0; }) && !mh::made_plan([] { return -1; }) &&
                  !mh::made_plan([]() -> int { throw std::bad_alloc(); }) &&
                  !mh::made_plan([]() -> int { std::vector<int> v; return v.at(3); });
  return ok ? 0 : 1;
}
""")


def test_members_of_a_team_fit_on_the_gpu_at_once(tmp_path):
    assert _run(tmp_path, PROGRAM) == ["64", "32", "3"]
