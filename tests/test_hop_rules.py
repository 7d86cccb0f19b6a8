"""Kernel and cache policy of the twisted-mass hop (csrc/hop_rules.hpp), built by a host
compiler and walked over lattices, precisions and link kinds."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nissa_amd", "csrc")

SRC = r"""
#include <cstdio>
#include "hop_rules.hpp"
using namespace nq;

int main()
{
  // spinor, link and tail precisions of the instances; clover blocks; batched residual
  const struct { int sp, lk, xp, clover, per_rhs; } inst[] = {
      {SP_F64, LK_F64_18, SP_F64, 0, 0}, {SP_F64, LK_F64_12, SP_F64, 0, 0}, {SP_F64, LK_F64_18, SP_F32, 0, 0},
      {SP_F64, LK_F64_12, SP_F32, 0, 0}, {SP_F64, LK_F64_18, SP_F64, 1, 0}, {SP_F32, LK_F32_18, SP_F32, 0, 0},
      {SP_F32, LK_F32_18, SP_F32, 1, 0}, {SP_F16, LK_F32_12, SP_F32, 0, 0}, {SP_F16, LK_F32_12, SP_F32, 1, 0},
      {SP_F16, LK_F16_12, SP_F32, 0, 0}, {SP_F16, LK_F16_12, SP_F32, 1, 0}, {SP_F64, LK_F64_18, SP_F32, 0, 1},
      {SP_F64, LK_F64_12, SP_F32, 0, 1}};
  for (auto& i : inst)
    for (int64_t Vh = 8; Vh < (int64_t(1) << 22); Vh += 1 + Vh / 200) {
      const HopRoute r = hop_route(Vh, i.sp, i.lk, i.xp, i.clover, 1, i.per_rhs, true);
      std::printf("%d %d %d %d %d %lld %d %d\n", i.sp, i.lk, i.xp, i.clover, i.per_rhs, (long long)Vh, r.kernel, r.keep);
    }
}
"""
F64, F32, F16 = 0, 1, 2
LINK = {0: 144, 1: 72, 2: 48, 3: 24, 4: 96}  # bytes of a link
PLAIN, LDS, SPLIT = 0, 1, 2


SMALL = r"""
#include <cstdio>
#include <initializer_list>
#include "hop_rules.hpp"
using namespace nq;

int main()
{
  for (int64_t blocks : {1, 16, 45, 68, 110, 126, 160, 256, 375, 625, 1296, 4096})
    for (int nr = 2; nr <= 16; nr++)
      for (int sp : {SP_F64, SP_F32, SP_F16})
        std::printf("%d %d %d %d %d %d\n", (int)blocks, nr, sp, stage_batch(256 * blocks, sp, 1, nr, 256),
                    stage_batch(256 * blocks, sp, 4, nr, 256), sp == SP_F16 ? 0 : st_block(256 * blocks, nr, sp, 256));
  for (int T : {4, 8, 16, 22, 30, 32, 36, 48, 64})
    for (int64_t Vh : {8, 65535, 65536, 1048576}) std::printf("%d %d %d\n", T, (int)Vh, z_tile(T, Vh));
}
"""


def numbers(tmp_path_factory, source):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "t.cpp").write_text(source)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t")],
                   check=True)
    out = subprocess.run([str(d / "t")], check=True, capture_output=True, text=True).stdout
    return [tuple(int(v) for v in l.split()) for l in out.splitlines()]


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    return numbers(tmp_path_factory, SRC)


@pytest.fixture(scope="module")
def small(tmp_path_factory):
    return numbers(tmp_path_factory, SMALL)


def test_one_policy_for_every_kernel(routes):
    """Default cache policy when links, clover blocks, input and output fit 224 MB, whichever
    kernel runs: split ones too, among which only the FP64 residual hop can exceed it."""
    seen = set()
    for sp, lk, xp, clover, per_rhs, Vh, kernel, keep in routes:
        eb = {F64: 16, F32: 8, F16: 4}[sp]
        site = 16 * LINK[lk] + 24 * eb + (108 * eb if clover else 0)
        assert keep == (site * Vh <= 224 << 20), (sp, lk, Vh)
        if kernel == SPLIT and not keep and (sp, xp, clover) != (F64, F64, 0):
            assert (sp, xp, clover) == (F64, F32, 0)
            seen.add(lk)
    assert seen == {0, 4}


def test_staged_hops_that_keep_their_links(routes):
    """The instances left out (hop_lds_keeps) are those that no lattice comes to: staging with
    the default policy happens in FP64 clover hops and batched residuals only."""
    kept = {(sp, clover, per_rhs) for sp, lk, xp, clover, per_rhs, Vh, kernel, keep in routes if kernel == LDS and keep}
    assert kept == {(F64, 1, 0), (F64, 0, 1)}


def test_batches_stage_where_they_fill_the_card(small):
    """A staged batch has more blocks, over all of its right-hand sides, than there are CUs."""
    for blocks, nr, sp, rb1, rb4, _ in (l for l in small if len(l) == 6):
        assert rb1 == (blocks * nr > 256)
        assert rb4 == (rb1 and sp == F16)  # LDS for four right-hand sides: FP16 only


def test_staggered_block_shrinks_with_the_lattice(small):
    """One source per wavefront only while all blocks of all sources leave the card near
    empty; the block never shrinks on the way to a larger lattice."""
    last = {}
    for blocks, nr, sp, _, _, v in (l for l in small if len(l) == 6):
        if sp == F16:
            continue
        full = 6 if sp == F32 and nr >= 5 else 4
        assert v in (1, 2, 4, 6) and v <= full and v >= last.get((nr, sp), 1)
        last[nr, sp] = v
        if v == 1:
            assert blocks * nr <= (256 if sp == F64 else 512)
        if blocks >= 512:
            assert v == full


def test_z_tile(small):
    for T, Vh, z in (l for l in small if len(l) == 3):
        assert z == (8 if Vh < 65536 else 4 if T % 8 else 2)
