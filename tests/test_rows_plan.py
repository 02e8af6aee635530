"""Launch shapes of the 16-row-tile kernels (csrc/gguf_rows_plan.h), compiled as plain host code (CPU only)."""

from __future__ import annotations

import ctypes as c
import subprocess
from pathlib import Path

import pytest

from tensor_amd.gguf import quant as Q

CSRC = Path(__file__).resolve().parents[1] / "tensor_amd" / "csrc"
SOURCE = """
#include "gguf_rows_plan.h"
using namespace tensor_gguf;
extern "C" void gemm_rows(const int* n, int count, int m, int k, double bytes, int* out) {
  const GemmRowsPlan p = plan_gemm_rows(n, count, m, k, bytes, false);
  out[0] = p.t, out[1] = p.per, out[2] = p.m_splits;
}
extern "C" void gemv_rows(const int* n, int count, int m, int pair, int* out) {
  const GemvRowsPlan p = plan_gemv_rows(n, count, m, pair);
  out[0] = p.groups, out[1] = p.waves;
}
extern "C" int gemv_group(const int* n, int count, int m, int k) { return gemv_rows_group_better(n, count, m, k); }
extern "C" int gemv_single(int type, int m, int n, int k) { return gemv_rows_single_better(type, m, n, k); }
extern "C" int gemv_pair(int type, int m, int n, int k) { return gemv_rows_pair_better(type, m, n, k); }
extern "C" int gemm_skinny(int type, int m, int n, int k, int f32) { return gemm_skinny_better(type, m, n, k, f32); }
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rows_plan")
    (folder / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(CSRC),
                    str(folder / "plan.cpp"), "-o", str(folder / "plan.so")], check=True, capture_output=True)
    return c.CDLL(str(folder / "plan.so"))


def blocks(rows, per):
    return sum(-(-(-(-n // 16)) // per) for n in rows)


def gemm_rows(library, encoding, m, k, rows):
    qk, size = Q.GEOMETRY[Q.ggml_type(encoding)]
    out = (c.c_int * 3)()
    library.gemm_rows((c.c_int * len(rows))(*rows), len(rows), m, k, c.c_double(size / qk), out)
    return tuple(out)


@pytest.mark.parametrize("encoding", ["q2_k", "q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("rows,k", [((4096, 1024, 1024), 4096), ((4096, 4096, 4096), 4096), ((2048, 2048, 2048), 2048),
                                    ((8192, 1024, 1024), 8192), ((2560, 640, 640), 2560), ((12288, 12288), 4096),
                                    ((1, 17, 33), 256), ((64000,), 4096)])
def test_streaming_gemm_counts_the_workgroups_it_launches(library, encoding, rows, k):
    """Workgroups round up per matrix; no (t, per) that the plan could take has fewer rounds with as little
    work in each (an extra round for a few workgroups costs as much as a full one)."""
    def rounds(t, per, m_splits):  # of an XCD's 32 CUs: it takes every eighth set of weight rows
        return -(-(-(-blocks(rows, per) // 8) * m_splits) // 32)

    for m in (9, 16, 17, 32, 33, 48, 64):
        t, per, m_splits = gemm_rows(library, encoding, m, k, rows)
        m16 = -(-m // 16)
        assert t in (1, 2, 4) and 1 <= per <= 12 and m_splits == -(-m16 // t)
        assert t == 1 or t < 2 * m16  # no more activation rows than M has
        mine = rounds(t, per, m_splits)
        for other_t in (1, 2, 4):
            for other in range(1, per + 1):
                splits = -(-m16 // other_t)
                if other_t <= t and (other_t, other) != (t, per):
                    assert rounds(other_t, other, splits) > mine, (m, (t, per), (other_t, other))


def test_streaming_gemm_keeps_ordinary_groups_in_one_round(library):
    for m, rows in ((32, (4096, 1024, 1024)), (64, (4096, 1024, 1024)), (32, (4096, 4096, 4096)),
                    (32, (2048, 2048, 2048)), (48, (2560, 640, 640))):
        t, per, m_splits = gemm_rows(library, "q4_k", m, 4096, rows)
        assert -(-blocks(rows, per) // 8) * m_splits <= 32, (m, rows, t, per)


def test_decode_gemv_takes_one_round_of_the_workgroups_it_launches(library):
    """Up to six row tiles a workgroup (eight where M > 4, four gate / up pairs), the fewest that leave at
    most 256 workgroups; beyond, workgroups of four and 8 waves."""
    def plan(rows, m=1, pair=False):
        out = (c.c_int * 2)()
        library.gemv_rows((c.c_int * len(rows))(*rows), len(rows), m, int(pair), out)
        return tuple(out)

    assert plan((4096, 4096, 4096)) == (4, 12)  # three tiles each would be 258 workgroups
    assert plan((4096, 1024, 1024)) == (2, 12)
    assert plan((12288, 12288)) == (6, 12)
    assert plan((14336, 14336), 4) == (4, 8) and plan((14336, 14336), 5) == (7, 12)
    for rows in ((1,), (4096,), (4097,), (12288,), (4096, 1024, 1024), (4100, 4100), (5120, 5120, 5120), (64000,),
                 (24576,), (24577,), (32768,), (8192, 8192, 8192)):
        for m, pair in ((1, False), (4, False), (5, False), (8, False), (1, True), (8, True)):
            if pair and len(rows) > 1:
                continue
            groups, waves = plan(rows, m, pair)
            fits = [g for g in range(1, 5 if pair else 9 if m > 4 else 7) if blocks(rows, g) <= 256]
            assert (groups, waves) == ((fits[0], 12) if fits else (4, 8)), (rows, m, pair)
            assert groups * (2 if pair else 1) <= waves


@pytest.mark.parametrize("rows,k", [((12288, 12288), 4096), ((28672, 28672), 7168), ((28672, 28672), 8192),
                                    ((12288, 12288), 12288), ((8192, 8192), 2048)])
def test_groups_of_more_rows_than_one_go_in_one_launch(library, rows, k):
    """Wide ones too, whatever the single-matrix kernels would hold in LDS at that K."""
    for m in range(2, 9):
        assert library.gemv_group((c.c_int * len(rows))(*rows), len(rows), m, k)
    assert not library.gemv_group((c.c_int * len(rows))(*rows), len(rows), 1, k - k % 2048 + 2048)
    assert library.gemv_group((c.c_int * 3)(1024, 128, 128), 3, 1, 2048)


@pytest.mark.parametrize("encoding,m,n,k,rows", [
    ("q4_0", 3, 3000, 1056, False), ("q4_0", 3, 2048, 1536, False), ("q4_0", 3, 6912, 2560, True),
    ("q8_0", 4, 3000, 1056, False), ("q8_0", 6, 2048, 1056, False), ("q8_0", 8, 12288, 4096, True),
    ("q4_1", 6, 1024, 6912, False), ("q5_1", 4, 1024, 6912, False), ("q4_1", 6, 4096, 2048, True),
    ("q2_k", 2, 6912, 1024, False), ("q2_k", 1, 2560, 6912, False), ("q2_k", 2, 6912, 1536, True),
    ("q6_k", 3, 1024, 4096, False), ("q6_k", 6, 1024, 6912, False), ("q6_k", 3, 4096, 4096, True),
    ("q4_k", 1, 2560, 2048, False), ("q4_k", 1, 2560, 2560, True), ("q4_0", 2, 4096, 4096, False),
    ("q6_k", 3, 2560, 2560, True), ("q4_0", 2, 5120, 4096, False), ("q4_0", 1, 5120, 6912, False),
])
def test_decode_gemv_leaves_single_matrices_that_the_vector_kernels_do_sooner(library, encoding, m, n, k, rows):
    """Both kernels timed at each: 1.04 to 1.8 times as long on the one that is not taken."""
    assert bool(library.gemv_single(Q.ggml_type(encoding), m, n, k)) == rows


@pytest.mark.parametrize("encoding", ["q4_0", "q4_k", "q8_0"])
def test_decode_gemv_lines_follow_size(library, encoding):
    """More rows of the same length never go back to the vector kernels, nor do pairs of them; the tuned M = 1 row
    lengths stay there at every size."""
    type_ = Q.ggml_type(encoding)
    for take in (library.gemv_single, library.gemv_pair):
        for m in range(1, 9):
            for k in (256, 1024, 1536, 2048, 2560, 6912):
                taken = [bool(take(type_, m, n, k)) for n in (1, 16, 640, 1024, 3000, 4096, 12288, 151936)]
                assert taken == sorted(taken), (m, k)
    assert not library.gemv_single(type_, 1, 151936, 4096)


def test_swiglu_pairs_of_one_pass_rows_stay_on_the_vector_kernels(library):
    for encoding, m, n, k, rows in (("q4_0", 1, 4096, 2048, False), ("q4_k", 1, 4096, 2048, False),
                                    ("q8_0", 4, 2000, 1056, False), ("q8_0", 2, 4096, 2048, True),
                                    ("q4_0", 1, 6912, 2560, True), ("q4_k", 2, 1, 256, True),
                                    ("q5_k", 1, 4096, 4096, False)):
        assert bool(library.gemv_pair(Q.ggml_type(encoding), m, n, k)) == rows, (encoding, m, n, k)


@pytest.mark.parametrize("encoding,m,n,k,skinny", [
    ("q2_k", 32, 8192, 256, True), ("q5_1", 12, 8192, 256, True), ("q5_1", 48, 4096, 1056, True),
    ("q8_0", 64, 3000, 1056, True), ("q4_k", 16, 1024, 1024, True), ("q4_k", 64, 320, 256, True),
    ("q6_k", 16, 640, 256, True), ("q5_0", 48, 2560, 1056, True), ("q4_1", 24, 12288, 384, True),
    ("q3_k", 24, 6000, 512, False), ("q5_k", 64, 6000, 512, False), ("q2_k", 48, 6000, 256, True),
    ("q6_k", 16, 4096, 512, False), ("q4_k", 32, 2560, 2560, False), ("q3_k", 9, 1024, 512, False),
    ("q8_0", 16, 8192, 512, False), ("q2_k", 16, 20000, 256, False), ("q5_0", 32, 8192, 1056, False),
])
def test_streaming_gemm_leaves_short_rows_to_the_small_m_kernel(library, encoding, m, n, k, skinny):
    """Both kernels timed at each."""
    assert bool(library.gemm_skinny(Q.ggml_type(encoding), m, n, k, 0)) == skinny


def test_fp32_activations_move_the_lines_of_the_small_m_kernel(library):
    for encoding, m, n, k, half, single in (("q4_1", 32, 2560, 1280, 1, 0), ("q5_1", 32, 2048, 2048, 0, 1),
                                            ("q8_0", 64, 4096, 1024, 1, 0), ("q4_0", 16, 2560, 1280, 1, 1)):
        type_ = Q.ggml_type(encoding)
        assert bool(library.gemm_skinny(type_, m, n, k, 0)) == bool(half), (encoding, m, n, k)
        assert bool(library.gemm_skinny(type_, m, n, k, 1)) == bool(single), (encoding, m, n, k)


def test_small_m_kernel_keeps_no_long_rows(library):
    for encoding in ("q4_0", "q5_0", "q4_k", "q3_k"):
        for m in (2, 9, 32, 64):
            for n in (1, 1024, 4096, 8192, 151936):
                assert not library.gemm_skinny(Q.ggml_type(encoding), m, n, 2048, 0)
                assert not library.gemm_skinny(Q.ggml_type(encoding), m, 151936, 256, 1)
