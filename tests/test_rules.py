"""The dispatch rules of vkml-framework_amd/csrc/rules.hpp, compiled with the
host's compiler: which kernel a call takes, without a GPU."""
import ctypes as C
import os
import subprocess

import pytest

from vkml_amd import hip as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
K_SCALAR, K_VEC_B, K_VEC_AB = 0, 1, 2


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rules") / "librules.so")
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "vkml-framework_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "rules_c.cpp"), "-o", so], check=True)
    return C.CDLL(so)


def _matmul(m, n, k, b_type, transposed, stride=0, batches=1, causal=0, offset=0):
    return H.MatmulParams(m, n, k, stride, 1, batches, transposed, b_type, H.F16, causal, offset)


@pytest.mark.parametrize("b_type", [H.F32, H.F16, H.BF16])
@pytest.mark.parametrize("m,n,k,transposed", [(16, 151936, 8192, 1), (16, 8192, 151936, 0), (9, 256000, 4096, 1), (9, 300, 1 << 24, 1),
                                              (2048, 4096, 128, 1), (2048, 128, 4096, 0)])
def test_aligned_float_products_load_vec4s_at_any_size(rules, b_type, m, n, k, transposed):
    # b's of 2^30 elements and more and rows past 2^22 among them
    assert rules.float_loads_c(C.byref(_matmul(m, n, k, b_type, transposed)), C.c_uint64(4096), C.c_uint64(1 << 33)) == K_VEC_AB


def test_float_products_off_alignment_load_elements(rules):
    def loads(p, a=0, b=0):
        return rules.float_loads_c(C.byref(p), C.c_uint64(a), C.c_uint64(b))
    for t, n, k in ((1, 7, 8), (0, 8, 7)):
        assert loads(_matmul(9, n, k, H.F32, t)) == (K_VEC_AB if t else K_VEC_B)
    assert loads(_matmul(9, 8, 7, H.F16, 1)) == K_SCALAR
    assert loads(_matmul(9, 7, 8, H.F16, 0)) == K_SCALAR
    for b_type, unit in ((H.F32, 16), (H.F16, 8), (H.BF16, 8)):
        for t in (0, 1):
            p = _matmul(9, 8, 8, b_type, t, stride=64, batches=2)
            assert loads(p, 32, unit) == K_VEC_AB
            assert loads(p, 32, unit // 2) == K_SCALAR
            assert loads(p, 4, unit) == (K_SCALAR if t else K_VEC_B)
            assert loads(_matmul(9, 8, 8, b_type, t, stride=66, batches=2), 32, unit) == K_SCALAR
    # a tile's offsets past 32 bits
    assert loads(_matmul(9, 8, 1 << 25, H.F16, 1)) == K_SCALAR
    assert loads(_matmul(9, 8, 1 << 25, H.F16, 0)) == K_VEC_B
    assert loads(_matmul(9, 1 << 25, 8, H.F16, 0)) == K_VEC_B


# us of vkml_matmul with each wave tile (32 x 64, 32 x 32, 16 x 32, 16 x 16)
QUANT_TILES = [
    (H.Q4_K, 9, 4096, 4096, (585, 283, 189, 113)), (H.Q4_K, 64, 8192, 2048, (292, 144, 97.5, 70.8)),
    (H.Q4_K, 131, 8192, 2048, (297, 190, 158, 146)), (H.Q4_K, 200, 4096, 4096, (599, 289, 232, 227)),
    (H.Q4_K, 300, 4096, 4096, (603, 382, 316, 292)), (H.Q4_K, 300, 8192, 2048, (383, 270, 234, 259)),
    (H.Q4_K, 512, 2048, 2048, (304, 148, 121, 118)), (H.Q4_K, 512, 4096, 4096, (611, 383, 387, 418)),
    (H.Q4_K, 512, 8192, 2048, (387, 335, 350, 401)), (H.Q4_K, 1000, 2048, 2048, (309, 193, 195, 211)),
    (H.Q4_K, 2048, 14336, 4096, (4244, 4109, None, None)), (H.Q4_K, 4096, 14336, 1024, (2085, 2048, None, None)),
    (H.Q4_1, 512, 4096, 4096, (512, 365, 375, 382)), (H.Q4_1, 512, 8192, 2048, (331, 321, 346, 361)),
    (H.Q4_1, 200, 8192, 2048, (259, 183, 187, 171)), (H.Q4_1, 4096, 14336, 1024, (1946, 2000, None, None)),
    (H.Q8_0, 512, 8192, 2048, (337, 324, 321, 349)), (H.Q8_0, 300, 8192, 2048, (337, 263, 219, 229)),
    (H.Q8_0, 2048, 14336, 4096, (3879, 3984, None, None)), (H.Q4_0, 300, 8192, 2048, (321, 259, 231, 222)),
]


@pytest.mark.parametrize("b_type,m,n,k,us", QUANT_TILES)
def test_quantized_products_take_a_tile_within_5_percent_of_the_fastest(rules, b_type, m, n, k, us):
    picked = (42, 22, 21, 11).index(rules.wave_tile_c(C.byref(_matmul(m, n, k, b_type, 1))))
    assert us[picked] <= 1.05 * min(u for u in us if u)


def test_short_sums_that_end_in_a_chunks_first_half_are_cut(rules):
    def cut(k, b_type=H.F16, t=1):
        return bool(rules.cut_last_chunk_c(C.byref(_matmul(512, 512, k, b_type, t))))
    assert all(cut(k, b) for k in (1, 16, 72, 80, 144, 240) for b in (H.F32, H.F16, H.BF16))
    assert not any(cut(k) for k in (17, 32, 64, 96, 120, 128, 256, 272, 2064))  # (whole chunks and long sums lose by it)
    assert not cut(80, t=0)


# us of probs v (f16, heads, queries, first query's position, head_dim)
PROBS_V_TILES = [
    (8, 1000, 0, 80, (118, 67.6, 44, 28.5)),
    (8, 2048, 2048, 128, (476, 295, 268, 251)),
    (32, 512, 0, 64, (62.5, 35.8, 23.7, 16.1)),
    (32, 1000, 0, 64, (130, 73, 51.1, 45.6)),
    (32, 300, 0, 128, (38.5, 23.3, 15.9, 12.9)),
    (32, 512, 2000, 128, (294, 202, 194, 190)),
    (32, 2048, 2048, 128, (963, 884, 946, 1010)),
    (32, 2048, 0, 128, (368, 307, 321, 349)),
    (32, 1000, 3000, 64, (574, 313, 302, 298)),
    (64, 2048, 2048, 64, (1340, 936, 1010, 1080)),
    (64, 1000, 0, 128, (180, 156, 161, 174)),
    (40, 1700, 0, 128, (316, 273, 286, 302)),
]


@pytest.mark.parametrize("heads,rows,first,hd,us", PROBS_V_TILES)
def test_masked_probs_v_takes_a_tile_within_5_percent_of_the_fastest(rules, heads, rows, first, hd, us):
    p = _matmul(rows, hd, rows + first, H.F16, 0, stride=hd * (rows + first), batches=heads, causal=1, offset=first)
    picked = (42, 22, 21, 11).index(rules.wave_tile_c(C.byref(p)))
    assert us[picked] <= 1.05 * min(us)


# times as fast as the kernel that staged nothing, with chunks of four rounds, two, one (30000 outputs, 2 to 8 rows)
@pytest.mark.parametrize("k,speed", [(32, (0.79, 1.01, 1.21)), (256, (0.76, 0.99, 1.21)), (512, (0.79, 1.04, 1.24)), (768, (0.93, 1.19, 1.28)),
                                     (1024, (1.03, 1.32, 1.34)), (1536, (1.18, 1.23, 1.35)), (2048, (1.27, 1.31, 1.34))])
def test_several_row_gemv_loses_nothing_at_short_rows(rules, k, speed):
    assert speed[(4, 2, 1).index(rules.rows_chunk_c(k))] > 1


# times as fast as the element-wise kernel at k of up to 128: several rows of b a half wave, one
@pytest.mark.parametrize("m,n,batches,speed", [(1, 1, 1, (0.97, 1.04)), (1, 256, 1, (0.91, 1.06)), (2, 1000, 1, (0.86, 1.16)),
                                               (2, 4000, 1, (0.96, 1.22)), (5, 40, 8, (0.98, 1.12)), (8, 64000, 1, (1.19, 0.92)), (5, 4000, 32, (1.35, 1.13)),
                                               (1, 8000, 1, (1.24, 1.32)), (2, 250, 32, (1.16, 1.32)), (3, 4000, 1, (1.15, 1.18)), (3, 8000, 1, (1.29, 1.24)),
                                               (5, 250, 32, (1.21, 1.17))])
def test_float_gemv_of_short_rows_loses_nothing(rules, m, n, batches, speed):
    picked = speed[rules.gemv_row_each_c(m, n, batches)]
    assert picked > 1 and picked > 0.9 * max(speed)


# us of one row of a by an f32 b from memory: a staged, a from the caches
@pytest.mark.parametrize("n,k,us", [(12000, 8192, (73.6, 69.2)), (16000, 8192, (93.3, 90.6)), (32000, 4096, (85.7, 84.7)),
                                    (8192, 8192, (50.6, 52.2)), (32000, 2048, (42.8, 43.9)), (2048, 8192, (16.4, 17.8))])
def test_one_row_by_a_large_f32_b_takes_the_faster_form(rules, n, k, us):
    p = H.GemvParams(1, n, k, H.F32, H.F16, 0, 1, 1)
    assert us[rules.gemv_row_cached_c(C.byref(p))] == min(us)
    for m, b_type in ((2, H.F32), (1, H.F16), (1, H.BF16)):
        assert not rules.gemv_row_cached_c(C.byref(H.GemvParams(m, n, k, b_type, H.F16, 0, 1, 1)))


# (wave tile, k, us of the last chunk with all its blocks, cut)
@pytest.mark.parametrize("rt,ct,k,masked,cut", [(2, 2, 32, 5.7, 4.4), (2, 2, 128, 5.7, 5.0), (2, 2, 224, 5.8, 5.7), (1, 1, 32, 3.1, 2.9), (1, 1, 224, 3.13, 3.3),
                                                (1, 1, 2080, 10.9, 11.3)])
def test_last_chunk_of_matmul_dot(rules, rt, ct, k, masked, cut):
    assert rules.dot_tail_c(rt, ct, k) == (2 if cut < masked else 1)
    assert all(rules.dot_tail_c(rt, ct, whole) == 0 for whole in (256, 512, 4096))
