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
    (32, 147, 0, 128, (22, 11, 8.85, 7.02)),
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


# us of vkml_matmul_dot with tiles of 64 x 128, 32 x 128, 16 x 128 and 16 x 64 outputs (f16 scales or f32)
DOT_TILES = [
    (H.Q4_1, 1, 909, 1737, 4096, (None, 52.8, 71.5, 58.4)), (H.Q4_1, 1, 909, 1664, 4096, (None, 52.2, 49.2, 52.8)), (H.Q4_0, 1, 909, 1664, 4096, (None, 50.6, 47.9, 50)),
    (H.Q4_1, 1, 1000, 1800, 1024, (None, 16.3, 20.7, 19.3)), (H.Q4_1, 0, 909, 1737, 4096, (None, 55.3, 57.2, 59.8)),
    (H.Q4_0, 1, 160, 9216, 4096, (70.3, 50, 47.8, 49.5)),
    (H.Q4_0, 1, 265, 5574, 1056, (20.6, 16.1, 15.6, 16.5)),
    (H.Q4_1, 1, 160, 9216, 4096, (85.3, 52.7, 48.6, 50.8)),
    (H.Q4_1, 1, 352, 4096, 4096, (83.6, 52.7, 48.2, 49.7)),
    (H.Q4_1, 1, 265, 5574, 1056, (23.9, 17.3, 16.1, 18.7)),
    (H.Q4_K, 1, 16, 4096, 4096, (66.4, 38.7, 25.5, 19.7)),
    (H.Q4_K, 1, 64, 8192, 2048, (35.5, 20.8, 14.4, 13.7)),
    (H.Q4_K, 1, 128, 8192, 2048, (35.7, 21.2, 18, 19.4)),
    (H.Q4_K, 1, 131, 8192, 2048, (35.8, 25.4, 22.2, 24.9)),
    (H.Q4_K, 1, 131, 2048, 8192, (130, 75.4, 49.5, 46.6)),
    (H.Q4_K, 1, 256, 4096, 4096, (67.2, 39.2, 32.9, 35.5)),
    (H.Q4_K, 1, 300, 4096, 4096, (67.4, 48.3, 41.4, 46.8)),
    (H.Q4_K, 1, 300, 8192, 2048, (44.8, 34.1, 34.1, 42)),
    (H.Q4_K, 1, 512, 3072, 2048, (36, 26.1, 22.7, 28.2)),
    (H.Q4_K, 1, 512, 4096, 4096, (68.6, 50.2, 52.1, 65.6)),
    (H.Q4_K, 1, 512, 14336, 4096, (161, 137, 165, 226)),
    (H.Q4_K, 1, 800, 2048, 8192, (133, 94.8, 97.9, 114)),
    (H.Q4_K, 1, 1000, 4096, 4096, (87.5, 81.9, 95.9, 123)),
    (H.Q4_K, 1, 2048, 4096, 4096, (162, 154, 185, 241)),
    (H.Q4_K, 1, 3000, 6144, 4096, (325, 329, 405, 519)),
    (H.Q4_K, 1, 4096, 4096, 4096, (293, 296, 362, 471)),
    (H.Q8_0, 1, 16, 4096, 4096, (64.8, 38.9, 30, 18.9)),
    (H.Q8_0, 1, 64, 8192, 2048, (35.4, 21, 17.1, 13.4)),
    (H.Q8_0, 1, 128, 8192, 2048, (35.7, 21.7, 20.2, 19.1)),
    (H.Q8_0, 1, 131, 8192, 2048, (35.7, 25.3, 26.7, 26.3)),
    (H.Q8_0, 1, 131, 2048, 8192, (131, 76.3, 58.2, 39.1)),
    (H.Q8_0, 1, 256, 4096, 4096, (67.3, 40.3, 36.1, 33.8)),
    (H.Q8_0, 1, 300, 4096, 4096, (67.8, 48.1, 50.7, 47.2)),
    (H.Q8_0, 1, 300, 8192, 2048, (44.4, 35.4, 41.5, 41.2)),
    (H.Q8_0, 1, 512, 3072, 2048, (36, 26.1, 27.5, 26.8)),
    (H.Q8_0, 1, 512, 4096, 4096, (71.5, 51.6, 71.8, 62)),
    (H.Q8_0, 1, 512, 14336, 4096, (166, 148, 211, 224)),
    (H.Q8_0, 1, 800, 2048, 8192, (139, 97.4, 141, 107)),
    (H.Q8_0, 1, 1000, 4096, 4096, (88.5, 92.5, 120, 118)),
    (H.Q8_0, 1, 2048, 4096, 4096, (171, 161, 232, 230)),
    (H.Q8_0, 1, 3000, 6144, 4096, (379, 345, 504, 495)),
    (H.Q8_0, 1, 4096, 4096, 4096, (334, 307, 449, 448)),
    (H.Q8_0, 0, 16, 4096, 4096, (56.2, 31.6, 22.4, 13.6)),
    (H.Q8_0, 0, 64, 8192, 2048, (31.2, 17.7, 13.2, 11.5)),
    (H.Q8_0, 0, 128, 8192, 2048, (31.4, 18, 18.7, 17.8)),
    (H.Q8_0, 0, 131, 8192, 2048, (31.5, 24.2, 24.1, 21.3)),
    (H.Q8_0, 0, 131, 2048, 8192, (113, 61, 43.1, 35.8)),
    (H.Q8_0, 0, 256, 4096, 4096, (58.6, 32.9, 33.4, 30.3)),
    (H.Q8_0, 0, 300, 4096, 4096, (59.1, 45.7, 43.9, 38.3)),
    (H.Q8_0, 0, 300, 8192, 2048, (41.4, 32.5, 37.4, 37.4)),
    (H.Q8_0, 0, 512, 3072, 2048, (31.8, 25, 24.6, 23.8)),
    (H.Q8_0, 0, 512, 4096, 4096, (62.5, 48, 59.5, 56.3)),
    (H.Q8_0, 0, 512, 14336, 4096, (156, 136, 204, 241)),
    (H.Q8_0, 0, 800, 2048, 8192, (120, 89.1, 113, 96)),
    (H.Q8_0, 0, 1000, 4096, 4096, (81.6, 80.6, 106, 107)),
    (H.Q8_0, 0, 2048, 4096, 4096, (156, 147, 204, 209)),
    (H.Q8_0, 0, 3000, 6144, 4096, (342, 315, 454, 457)),
    (H.Q8_0, 0, 4096, 4096, 4096, (304, 281, 403, 413)),
    (H.Q4_0, 1, 16, 4096, 4096, (66.6, 41.9, 28.5, 17.8)),
    (H.Q4_0, 1, 64, 8192, 2048, (36.2, 22.5, 16.3, 12.1)),
    (H.Q4_0, 1, 128, 8192, 2048, (36.4, 22.9, 20.3, 17.4)),
    (H.Q4_0, 1, 131, 8192, 2048, (36.5, 26.3, 25.4, 19.3)),
    (H.Q4_0, 1, 131, 2048, 8192, (134, 81.7, 55.9, 38.1)),
    (H.Q4_0, 1, 256, 4096, 4096, (69, 42.8, 36.6, 31.2)),
    (H.Q4_0, 1, 300, 4096, 4096, (69.2, 49.8, 47.4, 35.4)),
    (H.Q4_0, 1, 300, 8192, 2048, (45.2, 37, 39.3, 34.6)),
    (H.Q4_0, 1, 512, 3072, 2048, (36.8, 27.2, 26.3, 26.4)),
    (H.Q4_0, 1, 512, 4096, 4096, (70.7, 51.6, 57.4, 57.6)),
    (H.Q4_0, 1, 512, 14336, 4096, (158, 134, 169, 175)),
    (H.Q4_0, 1, 800, 2048, 8192, (142, 100, 107, 96.1)),
    (H.Q4_0, 1, 1000, 4096, 4096, (88.5, 82.3, 101, 101)),
    (H.Q4_0, 1, 2048, 4096, 4096, (159, 149, 191, 193)),
    (H.Q4_0, 1, 3000, 6144, 4096, (308, 312, 410, 417)),
    (H.Q4_0, 1, 4096, 4096, 4096, (279, 282, 370, 378)),
    (H.Q4_1, 1, 16, 4096, 4096, (80, 40.7, 30.1, 18.3)),
    (H.Q4_1, 1, 64, 8192, 2048, (43.4, 22, 16.9, 13.1)),
    (H.Q4_1, 1, 128, 8192, 2048, (43.6, 22.4, 20, 19.2)),
    (H.Q4_1, 1, 131, 8192, 2048, (43.6, 27.9, 26.1, 24.4)),
    (H.Q4_1, 1, 131, 2048, 8192, (162, 80.4, 58.2, 41)),
    (H.Q4_1, 1, 256, 4096, 4096, (83.2, 42, 36, 34.3)),
    (H.Q4_1, 1, 300, 4096, 4096, (83.3, 52.4, 48.4, 46.8)),
    (H.Q4_1, 1, 300, 8192, 2048, (49.2, 37, 40.6, 41)),
    (H.Q4_1, 1, 512, 3072, 2048, (43.9, 28.7, 27.2, 27.6)),
    (H.Q4_1, 1, 512, 4096, 4096, (84.7, 54.2, 74.9, 63)),
    (H.Q4_1, 1, 512, 14336, 4096, (182, 141, 197, 209)),
    (H.Q4_1, 1, 800, 2048, 8192, (170, 103, 142, 111)),
    (H.Q4_1, 1, 1000, 4096, 4096, (98.1, 84.6, 115, 119)),
    (H.Q4_1, 1, 2048, 4096, 4096, (184, 157, 225, 231)),
    (H.Q4_1, 1, 3000, 6144, 4096, (349, 332, 479, 504)),
    (H.Q4_1, 1, 4096, 4096, 4096, (311, 299, 433, 453)),
    (H.Q4_1, 0, 16, 4096, 4096, (73.6, 42.4, 26.8, 17.6)),
    (H.Q4_1, 0, 64, 8192, 2048, (39.6, 23.1, 15.7, 13.1)),
    (H.Q4_1, 0, 128, 8192, 2048, (39.9, 23.4, 19.6, 20)),
    (H.Q4_1, 0, 131, 8192, 2048, (40, 29.2, 25.1, 24.4)),
    (H.Q4_1, 0, 131, 2048, 8192, (147, 82, 52.7, 42.9)),
    (H.Q4_1, 0, 256, 4096, 4096, (75.7, 43.1, 35.9, 37)),
    (H.Q4_1, 0, 300, 4096, 4096, (75.8, 55.4, 46.6, 45.5)),
    (H.Q4_1, 0, 300, 8192, 2048, (48.6, 40.9, 38, 42)),
    (H.Q4_1, 0, 512, 3072, 2048, (40.3, 29.9, 25.5, 27.6)),
    (H.Q4_1, 0, 512, 4096, 4096, (78, 57.7, 58.8, 67)),
    (H.Q4_1, 0, 512, 14336, 4096, (187, 160, 188, 232)),
    (H.Q4_1, 0, 800, 2048, 8192, (155, 108, 113, 116)),
    (H.Q4_1, 0, 1000, 4096, 4096, (96, 95.6, 107, 124)),
    (H.Q4_1, 0, 2048, 4096, 4096, (189, 180, 207, 246)),
    (H.Q4_1, 0, 3000, 6144, 4096, (422, 386, 456, 567)),
    (H.Q4_1, 0, 4096, 4096, 4096, (375, 347, 406, 517)),
    (H.Q4_K, 1, 64, 8192, 2048, (35.5, 21, 14.6, 13.9)),
    (H.Q4_K, 1, 128, 8192, 2048, (35.7, 21.2, 18.1, 19.5)),
    (H.Q4_K, 1, 512, 4096, 4096, (68.7, 50.2, 52.2, 65.7)),
    (H.Q4_K, 1, 64, 8192, 2048, (35.6, 21.1, 14.6, 13.9)),
    (H.Q4_K, 1, 128, 8192, 2048, (35.7, 21.2, 18, 19.5)),
    (H.Q4_K, 1, 512, 4096, 4096, (68.5, 50.4, 51.6, 65.6)),
    (H.Q8_0, 1, 64, 8192, 2048, (35.4, 21.1, 17, 13.3)),
    (H.Q8_0, 1, 128, 8192, 2048, (35.7, 21.9, 20.2, 19)),
    (H.Q8_0, 1, 512, 4096, 4096, (71.4, 51.7, 71.6, 62.5)),
    (H.Q8_0, 0, 64, 8192, 2048, (31.1, 17.7, 13.2, 11.6)),
    (H.Q8_0, 0, 128, 8192, 2048, (31.4, 18.2, 18.9, 17.9)),
    (H.Q8_0, 0, 512, 4096, 4096, (62.5, 47.8, 59.5, 56.9)),
    (H.Q4_0, 1, 64, 8192, 2048, (36.1, 22.3, 15.8, 11.7)),
    (H.Q4_0, 1, 128, 8192, 2048, (36.4, 22.9, 19.9, 17)),
    (H.Q4_0, 1, 512, 4096, 4096, (70.8, 51.2, 56.4, 57)),
    (H.Q4_1, 1, 64, 8192, 2048, (43.2, 21.7, 16.4, 12.6)),
    (H.Q4_1, 1, 128, 8192, 2048, (43.6, 22.5, 19.8, 18.9)),
    (H.Q4_1, 1, 512, 4096, 4096, (84.6, 54, 74.2, 62.9)),
    (H.Q4_1, 0, 64, 8192, 2048, (39.6, 22.9, 15.3, 12.7)),
    (H.Q4_1, 0, 128, 8192, 2048, (39.9, 23.4, 19.3, 19.7)),
    (H.Q4_1, 0, 512, 4096, 4096, (78.7, 56.9, 58.1, 66.2)),
]


@pytest.mark.parametrize("b_type,f16,m,n,k,us", DOT_TILES)
def test_matmul_dot_takes_a_tile_within_9_percent_of_the_fastest(rules, b_type, f16, m, n, k, us):
    # (two of 300 x 8192 x 2048 are past 6)
    picked = (42, 22, 12, 11).index(rules.dot_tile_c(b_type, f16, m, n))
    assert us[picked] <= 1.09 * min(u for u in us if u)


# us of vkml_attend_prompt_fast with blocks of 32 and of 64 keys: (heads, kv_heads, head_dim, first, queries)
PROMPT_BLOCKS = [
    (32, 8, 128, 0, 9, 4.31, 4.9), (32, 8, 128, 0, 40, 5.59, 5.77), (32, 8, 128, 0, 64, 6.36, 5.96), (32, 8, 128, 25, 40, 6.77, 7.19),
    (32, 8, 128, 0, 90, 7.52, 7.78), (32, 8, 128, 0, 128, 8.79, 7.88), (32, 8, 128, 0, 150, 9.86, 9.71), (32, 8, 128, 0, 192, 11.0, 9.85),
    (32, 8, 128, 0, 300, 15.6, 13.7), (32, 8, 128, 1000, 64, 42.2, 34.6), (32, 8, 128, 37, 1000, 43.1, 38.3), (32, 8, 128, 0, 1100, 46.2, 39.7),
    (32, 8, 128, 0, 1500, 61.6, 53.3), (32, 8, 128, 0, 2048, 88.6, 93.2), (32, 8, 128, 4000, 1100, 236, 273), (64, 8, 128, 0, 700, 33.6, 29.2),
    (64, 8, 128, 0, 1000, 48.4, 53.1), (8, 2, 128, 0, 4096, 146, 124), (32, 8, 64, 0, 9, 3.41, 3.82), (32, 8, 64, 0, 64, 4.56, 4.33),
    (32, 8, 64, 1, 64, 5.37, 5.57), (32, 8, 64, 0, 128, 6.22, 5.54), (32, 8, 64, 0, 1000, 28.8, 23.1), (64, 8, 64, 2048, 2048, 272, 257),
]


@pytest.mark.parametrize("heads,kv_heads,hd,first,t,narrow,wide", PROMPT_BLOCKS)
def test_prompt_attention_takes_the_faster_block(rules, heads, kv_heads, hd, first, t, narrow, wide):
    p = H.AttendPromptParams(heads, kv_heads, hd, first + t, t, first, H.F16, 1.0, 0.0)
    workgroups = -(-t // 16) * kv_heads * max(1, heads // kv_heads // 4)
    assert rules.wide_blocks_c(C.byref(p), workgroups, 256) == (wide < narrow)


@pytest.mark.parametrize("rows,columns", [(8, 9), (8, 15), (54, 73), (63, 71), (9, 100), (301, 86), (128, 17), (27, 1187), (65, 9)])
def test_bands_hold_every_tile_once_and_few_columns_an_xcd(rules, rows, columns):
    tiles = (C.c_uint32 * (rows * columns + 8))()
    count = rules.dot_bands_c(rows, columns, tiles)
    assert rows * columns <= count < rows * columns + 8
    order = list(tiles[:count])
    assert sorted(t for t in order if t != 0xFFFFFFFF) == sorted(65536 * r + c for r in range(rows) for c in range(columns))
    for xcd in range(8):
        mine = [t for t in order[xcd::8] if t != 0xFFFFFFFF]
        assert len(mine) <= -(-rows * columns // 8)
        assert len({t % 65536 for t in mine}) <= 2 * -(-columns // 8) + 1  # parts of two bands, at the end of three


def test_whole_eights_of_columns_and_small_and_huge_launches_keep_the_plain_grid(rules):
    # (the huge ones: 256 work items a tile along x would pass 32 bits)
    for rows, columns in ((100, 8), (100, 72), (7, 73), (300, 5), (1, 1187), (31250, 1187), (65535, 129)):
        assert rules.dot_bands_c(rows, columns, None) == 0


# us of transposed f16 products of short sums, wave tiles as above
SHORT_SUMS = [
    (64, 1000, 8, (4.24, 3.75, 3.13, 3.34)),
    (64, 1000, 64, (9.96, 6.19, 4.46, 3.34)),
    (130, 9532, 32, (7.08, 5.82, 5.35, 8.11)),
    (130, 9532, 72, (11.96, 10.47, 8.71, 12.06)),
    (130, 9532, 128, (17.79, 13.44, 11.38, 12.05)),
    (235, 12080, 12, (7.61, 6.63, 6.86, 13.83)),
    (235, 12080, 80, (17.37, 14.54, 14.14, 20.96)),
    (518, 5040, 16, (7.72, 6.61, 6.45, 12.93)),
    (518, 5040, 144, (27.11, 21.93, 20.76, 26.8)),
    (1188, 2272, 88, (18.85, 15.64, 16.38, 19.9)),
    (1188, 2272, 192, (34.77, 26.74, 26.86, 27.19)),
    (2008, 6992, 16, (18.67, 19.68, 19.16, 51.29)),
    (400, 1000, 16, (5.18, 3.93, 3.3, 4.29)),
    (400, 1000, 80, (12.18, 7.71, 5.65, 5.89)),
]


@pytest.mark.parametrize("m,n,k,us", SHORT_SUMS)
def test_short_sums_take_a_tile_within_10_percent_of_the_fastest(rules, m, n, k, us):
    picked = (42, 22, 21, 11).index(rules.wave_tile_c(C.byref(_matmul(m, n, k, H.F16, 1))))
    assert us[picked] <= 1.1 * min(us)
