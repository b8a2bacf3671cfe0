"""Which kernel variant each shape of tests/test_gpu_gemm_tiles.py takes, by the
plan functions of csrc/api.cpp compiled for the host: every variant is reached,
with one chunk of K and (where it has them) several; and a weight's scratch
holds every plan."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import PKG
from test_gpu_gemm_tiles import SHAPES

GLUE = """
#include <algorithm>
#include <cmath>
#include <cstddef>
constexpr int kMfmaWaves = 8, kCounters = 8192;
struct GemmTilePlan { int mt, mb, nw, nb, kc, cs; };
%s
extern "C" void plan(int M, int K, int N, int *o) {  // {kind, a, b, K chunks, partial floats, split rows}
    if (two_passes(M, K, N)) { o[0] = 3; o[1] = o[2] = o[3] = o[4] = o[5] = 0; return; }
    if (M <= kMfma16Rows) {
        o[0] = 0; o[2] = 0; mfma16_plan(K, N, &o[1], &o[3]); o[4] = o[3] > 1 ? o[3] * 16 * N : 0; o[5] = 32;
    } else if (M <= kMfmaPassRows) {
        o[0] = 1; o[2] = M > 32 ? 2 : 1; mfma_plan(K, N, &o[1], &o[3]);
        o[4] = o[3] > 1 ? o[3] * 32 * o[2] * N : 0; o[5] = 32 * o[2];
    } else {
        const GemmTilePlan t = tile_plan(M, K, N);
        o[0] = 2; o[1] = t.mt; o[2] = t.nw; o[3] = t.kc; o[4] = (int)tile_part_floats(t); o[5] = 32 * t.mt * t.mb;
    }
}
extern "C" void scratch(int K, int N, size_t *x, size_t *part) { mfma_scratch(K, N, x, part); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    src = open(os.path.join(PKG, "csrc", "api.cpp")).read()
    plans = src[src.index("// Steps per wave and K chunks of the product of 17 to 64 rows"):
                src.index("// The MFMA operand copy of a panel-major weight")]
    d = tmp_path_factory.mktemp("plans")
    (d / "p.cpp").write_text(GLUE % plans)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", str(d / "p.cpp"), "-o", str(d / "p.so")], check=True)
    return C.CDLL(str(d / "p.so"))


def _plan(lib, M, K, N):
    o = (C.c_int * 6)()
    lib.plan(M, K, N, o)
    return list(o)


def test_shapes_reach_every_variant(lib):
    got = set()
    for M, K, N in SHAPES:
        kind, a, b, kc, _, _ = _plan(lib, min(M, 4096), K, N)
        got.add((kind, a, b, kc > 1))
    want = {(0, steps, 0, False) for steps in (1, 2, 4, 8)} | {(0, 4, 0, True), (0, 8, 0, True)}  # k_gemm_mfma16
    for mt in (1, 2):  # k_gemm_mfma; the fewest steps hold all of K
        want |= {(1, steps, mt, False) for steps in (1, 2, 4, 8, 16)} | {(1, steps, mt, True) for steps in (4, 8, 16)}
    for mt, nw in ((1, 4), (2, 4), (3, 4), (4, 4), (4, 8)):  # k_gemm_mfma_tile
        want |= {(2, mt, nw, False), (2, mt, nw, True)}
    want.add((3, 0, 0, False))  # two passes
    assert want <= got, want - got


@pytest.mark.parametrize("K,N", sorted({s[1:] for s in SHAPES} | {(8192, 32768), (8192, 32), (16, 32768), (2048, 1024)}))
def test_scratch_holds_every_plan(lib, K, N):
    x, part = C.c_size_t(), C.c_size_t()
    lib.scratch(K, N, C.byref(x), C.byref(part))
    for M in list(range(8, 260)) + list(range(260, 4097, 37)) + [4096]:
        kind, _, _, _, floats, rows = _plan(lib, M, K, N)
        assert floats <= part.value, M
        # 16-row operands: 16 rows of whole 32-row K steps; then the row exponents
        need = 2 * 16 * ((K + 31) // 32 * 32) + 32 if kind == 0 else 2 * rows * K + 2 * rows
        assert need <= x.value, M
