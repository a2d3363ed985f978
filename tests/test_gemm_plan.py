"""The launch-shape rules of the gather-GEMM (tenes_amd/csrc/gemm_plan.hpp),
compiled for the host."""
import ctypes as C
import os
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "tenes_amd" / "csrc"
SRC = r"""
#include "gemm_plan.hpp"
using namespace tn::kern;
extern "C" void plan(int M, int N, int K, int bm, int splits, int f64, int *out) {
  const GemmPlan g{bm, splits};
  const Plan p = plan_for(M, N, K, bm ? &g : nullptr, f64 != 0);
  out[0] = p.BM; out[1] = p.splits; out[2] = p.kps; out[3] = p.sk;
}
extern "C" int cands(int M, int N, int K, int f64, int *out) {
  int n = 0;
  for (const GemmPlan &g : candidates(M, N, K, f64 != 0)) { out[2 * n] = g.bm; out[2 * n++ + 1] = g.splits; }
  return n;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "p.cpp").write_text(SRC)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    f"-I{CSRC}", str(d / "p.cpp"), "-o", str(d / "p.so")], check=True)
    return C.CDLL(str(d / "p.so"))


def plan(lib, M, N, K, f64, shape=(0, 0)):
    out = (C.c_int * 4)()
    lib.plan(M, N, K, shape[0], shape[1], int(f64), out)
    return tuple(out)


def candidates(lib, M, N, K, f64):
    out = (C.c_int * 64)()
    n = lib.cands(M, N, K, int(f64), out)
    return [(out[2 * i], out[2 * i + 1]) for i in range(n)]


SHAPES = [(M, N, K) for M in (1, 9, 32, 33, 128, 333, 1024, 2500) for N in (1, 16, 32, 100, 128, 1024, 4096)
          for K in (1, 15, 16, 64, 100, 128, 333, 400, 401, 2500, 8192, 18225, 131072)]


@pytest.mark.parametrize("f64", [True, False])
def test_candidates_start_with_the_untuned_shape(lib, f64):
    """The autotuner's candidates in FP64 and in the mixed modes: the shape the
    same arithmetic takes untuned comes first, 32 x 32 tiles only in FP64 (no
    other kernel has them), and the untuned shape of the 64 and 128 tiles is
    among them in either."""
    for M, N, K in SHAPES:
        cs = [plan(lib, M, N, K, f64, c) for c in candidates(lib, M, N, K, f64)]
        assert cs[0][:2] == plan(lib, M, N, K, f64)[:2], (M, N, K)
        assert len(set(cs)) == len(cs), (M, N, K, cs)
        assert plan(lib, M, N, K, False)[:2] in [c[:2] for c in cs], (M, N, K)
        assert f64 or all(c[0] != 32 for c in cs)


@pytest.mark.parametrize("f64", [True, False])
def test_splits_cover_k(lib, f64):
    """Every split of every shape has work and the splits cover K."""
    for M, N, K in SHAPES:
        for c in [(0, 0)] + candidates(lib, M, N, K, f64):
            bm, splits, kps, _ = plan(lib, M, N, K, f64, c)
            assert bm in (32, 64, 128) and kps % 16 == 0
            assert (splits - 1) * kps < K <= splits * kps, (M, N, K, c)


@pytest.mark.parametrize("M", [2097120, 2097121, 4194240])
@pytest.mark.parametrize("N", [1, 32, 33])
@pytest.mark.parametrize("K", [1, 400, 8192])
def test_tall_products_stay_in_the_grid(lib, M, N, K):
    """65535 workgroups in y: M up to 64 x 65535 has a launch, as it had with
    64 x 64 tiles alone, tuned or not."""
    for f64 in (True, False):
        bm = plan(lib, M, N, K, f64)[0]
        assert -(-M // bm) <= 65535, (bm, f64)
        assert all(c[0] != 32 for c in candidates(lib, M, N, K, f64)) or M <= 2097120
