"""The host's choice of kernel, tile and K-split (mkernel_amd/csrc/mk_plan.h),
compiled with the system C++ compiler: what the GPU tests' shapes are listed
for is what they run on 256 CUs."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

import test_gpu_fused_small as fused
import test_gpu_gemm as dense
import test_gpu_gemm_small as small
import test_zz_no_alloc as noalloc

ROOT = Path(__file__).resolve().parent.parent

PROG = r"""
#include "mk_plan.h"
static const mk::SmallSpace kSpace[2] = {{0, 0}, {496, 256LL * 262144}};
extern "C" {
int n_tiles() { return sizeof mk::kTiles / sizeof mk::kTiles[0]; }
int fold_only(int i) { return mk::kTiles[i].fold_only; }
// a workspace that holds `tiles` partial tiles of 128 x 256
int gemm_within(int64_t M, int64_t N, int64_t K, int64_t tiles) {
  mk::GemmSmallPlan p = {};
  return mk::gemm_runs_small(M, N, K, K, N, 256, {496, tiles * 131072}, &p);
}
// out: tile, workgroups, parts along K
int gemm(int64_t M, int64_t N, int64_t K, int ws, int* out) {
  mk::GemmSmallPlan p = {};
  const bool s = mk::gemm_runs_small(M, N, K, K, N, 256, kSpace[ws], &p);
  out[0] = p.tile, out[1] = p.grid, out[2] = p.split;
  return s;
}
int fused(int64_t M, int64_t N, int64_t K, int peers, int64_t rows, int blocks, int second, int* out) {
  const mk::FusedPlan f = mk::plan_fused(M, N, K, K, N, 256, {peers, rows}, blocks, second, true);
  out[0] = f.plan.tile;
  return f.small + 2 * f.first;
}
int parts(int rest, int64_t K, int bm, int n_cons, int reduce) { return mk::tail_parts(rest, K, bm, n_cons, reduce); }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("plans")
    (d / "plans.cpp").write_text(PROG)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", str(ROOT / "mkernel_amd" / "csrc"),
                    str(d / "plans.cpp"), "-o", str(d / "plans.so")], check=True, capture_output=True)
    lib = C.CDLL(str(d / "plans.so"))
    i64, i32 = C.c_int64, C.c_int
    lib.gemm_within.argtypes = [i64, i64, i64, i64]
    lib.gemm.argtypes = [i64, i64, i64, i32, C.c_void_p]
    lib.fused.argtypes = [i64, i64, i64, i32, i64, i32, i32, C.c_void_p]
    lib.parts.argtypes = [i32, i64, i32, i32, i32]
    return lib


def _gemm(plans, M, N, K, ws=1):
    out = (C.c_int * 3)()
    return bool(plans.gemm(M, N, K, ws, out)), *out


def _fused(plans, *a):
    out = (C.c_int * 1)()
    f = plans.fused(*a, out)
    return bool(f & 1), bool(f & 2), out[0]


def test_small_gemm_shapes(plans):
    """Each plain tile shape, and one to four parts along K, all in the small
    kernel, with and without a workspace."""
    got = [_gemm(plans, *s) for s in small.SHAPES]
    assert all(g[0] for g in got) and all(_gemm(plans, *s, ws=0)[0] for s in small.SHAPES)
    assert {g[1] for g in got} == {i for i in range(plans.n_tiles()) if not plans.fold_only(i)}
    assert {g[3] for g in got} == {1, 2, 3, 4}


@pytest.mark.parametrize("M,N,K,persistent", [(4224, 2048, 5504, 1), (36992, 256, 4096, 1), (4224, 2048, 3072, 0),
                                              (14720, 768, 13472, 1), (8320, 2048, 5024, 1), (22400, 768, 9056, 1),
                                              (15232, 1280, 4928, 0), (26240, 1024, 7712, 1), (22400, 1536, 4832, 0),
                                              (26752, 512, 10016, 0), (16512, 1024, 8192, 1), (32640, 512, 8192, 0)])
def test_odd_row_blocks(plans, M, N, K, persistent):
    """Odd numbers of 128-row blocks go to the persistent kernel where its last
    round is split along K and K is long for the number of rounds; without a
    workspace, or with one that is a tile too small, there is no split."""
    assert _gemm(plans, M, N, K)[0] != bool(persistent) and _gemm(plans, M, N, K, ws=0)[0]
    if persistent:
        rest = M // 128 * (N // 256) % 256
        tiles = rest * (plans.parts(rest, K, 128, 256, 0) - 1)
        assert not plans.gemm_within(M, N, K, tiles) and plans.gemm_within(M, N, K, tiles - 1)


def _blocks(world, rows, copies=1):
    return copies * (world - 1) * rows // 128


def test_fused_shapes(plans):
    """Every tile shape a fold may get comes up in each operation's list, staged
    first; the AllGather and ReduceScatter lists end in a launch that stages
    first and then runs the persistent kernel."""
    folds = {i for i in range(plans.n_tiles()) if 256 % (64, 128, 128, 192, 128, 128, 64)[i] == 0}
    ag = [_fused(plans, M, N, K, -1, 0, M // 128, 0) for _, M, N, K, _ in fused.AG]
    assert all(s and f for s, f, _ in ag[:-1]) and ag[-1][:2] == (False, True)
    assert {t for _, _, t in ag[:-1]} == {i for i in range(plans.n_tiles()) if not plans.fold_only(i)}
    rs = [_fused(plans, M, N, K, w - 1, M // w, _blocks(w, M // w), 0) for w, _, M, N, K in fused.RS]
    assert all(s and f == (c[0] > 1) for (s, f, _), c in zip(rs[:-1], fused.RS)) and rs[-1][:2] == (False, True)
    assert {t for _, _, t in rs[:-1]} == folds
    ar = [_fused(plans, M, N, K, w - 1, M, _blocks(w, M), 0) for w, M, N, K in fused.AR]
    ar2 = [_fused(plans, M, N, K, w - 1, M // w, _blocks(w, M // w, 2), 1) for w, _, M, N, K in fused.AR2]
    done = [_fused(plans, M, N, K, w - 1, M // w if two else M, _blocks(w, M // w if two else M, 1 + two), two)
            for w, M, N, K, two in fused.DONE]
    assert all(s and f for s, f, _ in ar + ar2 + done)
    assert {t for _, _, t in done} == folds


def test_split_tail_shapes(plans):
    """The dense K-split tests' tail tiles are split as their lists say, with
    two, three and four parts among them."""
    seen = set()

    def partials(tiles, K, bm, cus, reduce=0):
        cus = min(cus, tiles)  # the grid
        rest = tiles % cus
        s = plans.parts(rest, K, bm, cus, reduce)
        seen.add(s)
        return rest * (s - 1) * bm // 256

    for M, N, K, bm, cus, want in dense.SPLIT_TAIL:
        assert partials((M // bm) * (N // 256), K, bm, cus or 256) == want
    for M, N, K, cus, waves, want in dense.SPLIT_EXCHANGE:
        assert want == (0 if waves == 4 else partials((M // 256) * (N // 256), K, 256, cus))
    for world, rows, K, N, want in noalloc.NOALLOC_SPLIT:
        assert partials(world * rows // 256 * (N // 256), K, 256, 256) == want
    assert seen >= {2, 3, 4}
    # with the fold, 16 tiles on 5, 3 and 11 workgroups
    assert [plans.parts(16 % c, K, 256, c, 1) for c, K in ((5, 14336), (3, 16384), (11, 21504), (5, 4096))] == [4, 3, 2, 1]
