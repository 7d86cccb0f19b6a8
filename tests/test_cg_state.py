"""The CG recurrences of csrc/cg_state.hpp, built by a host compiler.

A finalisation that rides in a hop shares its launch with workgroups that read `done` and
`reliable`.  It must leave both words alone, raise the same bits in `stop`, and agree with
the finalisation launched by itself in every other field.

The poll interval of a multi-shift solve follows the running shift that needs most.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nissa_amd", "csrc")

RIDING = r"""
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include "cg_state.hpp"
using namespace nq;

int main()
{
  const double nan = std::nan("");
  // |r|^2 of the p update, <p, A p>, iterations left: goes on, converged, below delta of
  // the last update, out of iterations, not a number, <p, A p> not positive
  const struct { double rr, pap; int left; } cases[] = {{0.5, 2, 9}, {1e-30, 2, 9}, {1e-3, 2, 9}, {0.5, 2, 1},
                                                        {nan, 2, 9}, {0.5, 0, 9}, {0.5, nan, 9}};
  for (int pending : {(int)FIN_NONE, (int)FIN_RR, (int)FIN_RR_SLOPPY})
    for (auto& c : cases) {
      CgState s;
      std::memset(&s, 0, sizeof s);
      s.rr = 1; s.r0 = 1; s.alpha = 3; s.xlag = 1; s.iter = 4; s.niter = 4 + c.left;
      s.target = 1e-20; s.delta = 0.1; s.rr_new = c.rr; s.pending = pending;
      CgState own = s, riding = s;
      finalize<false>(&own, FIN_PAP, c.pap);
      finalize<true>(&riding, FIN_PAP, c.pap);
      const int bits = own.done | own.reliable << 1;
      const bool kept = riding.done == 0 && riding.reliable == 0 && riding.stop == bits && own.stop == 0;
      riding.done = own.done; riding.reliable = own.reliable; riding.stop = 0;
      std::printf("%d %d %d\n", (int)kept, (int)!std::memcmp(&own, &riding, sizeof own), bits);
    }
}
"""


# smallest mass first; it has the looser residue and has stopped
POLL = r"""
#include <cstdio>
#include <cstring>
#include "cg_state.hpp"
using namespace nq;

int main()
{
  CgmState s;
  std::memset(&s, 0, sizeof s);
  s.nshift = 2; s.iter = 40;
  s.run[1] = 1;
  s.res[0] = 9e-5; s.target[0] = 1e-4;
  s.res[1] = 1e-10; s.target[1] = 1e-12;
  std::printf("%d\n", next_chunk_cgm(s, 16));  // 40 iterations for ten decades: 8 for two, and one
  s.target[1] = 0;
  std::printf("%d\n", next_chunk_cgm(s, 16));
  s.run[0] = 1; s.res[0] = 1e-3; s.target[1] = 1e-12;  // both run: 14 for the first
  std::printf("%d\n", next_chunk_cgm(s, 16));
  s.res[0] = 2;  // no estimate for it yet
  std::printf("%d\n", next_chunk_cgm(s, 16));
  s.run[0] = s.run[1] = 0;
  std::printf("%d\n", next_chunk_cgm(s, 16));
}
"""


def run_host(tmp_path, source):
    (tmp_path / "t.cpp").write_text(source)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", CSRC, str(tmp_path / "t.cpp"), "-o", exe],
                   check=True)
    return [l.split() for l in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_riding_finalisation_leaves_done_and_reliable(tmp_path):
    out = run_host(tmp_path, RIDING)
    assert len(out) == 21 and all(l[0] == "1" and l[1] == "1" for l in out), out
    # nothing pending: only <p, A p> can stop; a plain and a mixed CG with |r|^2 pending
    assert [int(l[2]) for l in out] == [0, 0, 0, 0, 0, 1, 1] + [0, 1, 0, 1, 1, 1, 1] + [0, 2, 2, 2, 1, 1, 1], out


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_poll_interval_of_a_multi_shift_solve(tmp_path):
    assert [int(l[0]) for l in run_host(tmp_path, POLL)] == [9, 64, 15, 16, 16]
