"""CPU: how a Q8_0 GEMV launch is cut up (ferrum_amd/csrc/fkv_gemv_plan.h) and which kernel
a batched GEMM runs (fkv_gemm_plan.h), at sizes where both sides were measured or a limit
lies; neither changes a result, so only the choice is checked."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def _cuts(tmp_path, sizes, program="gemv_plan_print"):
    exe = tmp_path / program
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-o", str(exe),
                    os.path.join(HERE, "gemm", program + ".cpp")], check=True)
    text = "".join("%d %d %d\n" % s for s in sizes)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True)
    return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]


def test_wide_matrices_of_few_rows_take_one_token(tmp_path):
    """(rows, cols, tokens) -> (tokens a workgroup, row split). us at one / two tokens."""
    want = {
        (16, 14336, 2): (1, 2),       # 8.6 / 13.1
        (16, 14336, 128): (1, 2),     # 9.5 / 14.0
        (256, 12352, 8): (1, 2),      # 9.4 / 13.8
        (1024, 16384, 3): (1, 2),     # 12.2 / 15.6
        (2048, 14336, 2): (1, 2),     # 12.8 / 14.8
        (4096, 14336, 2): (2, 1),     # 24.6 / 19.9
        (1024, 14336, 8): (2, 1),     # 17.0 / 14.4
        (256, 14336, 64): (2, 1),     # 28.8 / 19.0
        (16, 12288, 8): (2, 1),       # two tokens within 64 KiB
        (16, 16416, 8): (1, 2),       # two tokens past half a CU's LDS
        (16, 14336, 1): (1, 2),
    }
    got = _cuts(tmp_path, list(want))
    assert {k: c[:2] for k, c in zip(want, got)} == want


def test_two_or_four_tokens(tmp_path):
    """(rows, cols, tokens) -> tokens a workgroup. us at two / four tokens."""
    want = {
        (11264, 4096, 7): 4,     # 30.4 / 25.5
        (11264, 4096, 8): 4,     # 30.9 / 26.4
        (8192, 4096, 7): 4,      # 20.1 / 18.1
        (4096, 2048, 20): 4,     # 12.9 / 11.8
        (1024, 832, 64): 4,      # 10.0 / 9.4
        (256, 1536, 256): 4,     # 10.2 / 9.6
        (6144, 3072, 10): 2,     # 17.7 / 19.4
        (3072, 2752, 24): 2,     # 19.0 / 20.3
        (11264, 2048, 5): 2,     # 11.9 / 12.7
        (2048, 2048, 8): 2,      # latency of few workgroups
        (8192, 5632, 8): 2,      # 31.2 / 32.3
        (11264, 5632, 6): 2,     # 35.5 / 40.2
        (16384, 5632, 8): 4,     # 64.2 / 60.9
        (8192, 4096, 3): 4,      # 12.3 / 12.1
        (6144, 4096, 4): 2,      # 10.7 / 12.9
        (28672, 4096, 2): 2,
        (28672, 8192, 8): 2,     # four past 64 KiB of LDS
    }
    got = _cuts(tmp_path, list(want))
    assert {k: c[0] for k, c in zip(want, got)} == want
    assert all(c[1] == 1 for c in got)


def test_batches_that_the_gemv_takes(tmp_path):
    """(rows, cols, tokens) -> all workgroups at once. us as a GEMV / on the matrix cores."""
    want = {
        (16, 64, 256): 1,        # 3.7 / 5.2
        (256, 576, 64): 1,       # 4.6 / 6.6
        (256, 576, 256): 0,      # 10.4 / 6.8
        (1024, 832, 17): 1,      # 5.0 / 6.1
        (1024, 4096, 24): 1,     # 9.3 / 10.7
        (1024, 4096, 32): 0,     # 11.2 / 10.4
        (1024, 5632, 17): 1,     # 11.6 / 13.1
        (2048, 2752, 12): 1,     # 8.6 / 8.7
        (2048, 2752, 16): 0,     # 10.3 / 8.6
        (4096, 4096, 8): 0,      # 11.5 / 10.2
        (4096, 4096, 12): 0,     # 15.4 / 10.2: 768 workgroups of four tokens
        (1024, 4096, 48): 0,     # 13.7 / 10.7
        (16, 14336, 256): 1,     # 12.2 / 30.6
        (256, 14336, 24): 1,     # 14.8 / 25.5
        (1024, 14336, 32): 0,    # 36 / 26.1: two workgroups a CU
        (1024, 28672, 8): 1,     # 24.8 / 40.6
        (1024, 28672, 16): 0,    # 45.7 / 40.6
    }
    got = _cuts(tmp_path, list(want))
    assert {k: c[2] for k, c in zip(want, got)} == want


def test_launches_stay_within_one_grid(tmp_path):
    """(rows, cols, tokens) -> 64 x 64 tiles? Sizes up to the card's memory and past it."""
    want = {
        (64, 64, 64 * (1 << 21) - 64): 1,     # 2^24 - 8 workgroups of 256
        (64, 64, 64 * (1 << 21)): 0,          # 2^32 threads
        (128, 64, 1 << 30): 0,
        (131072, 64, 64 * 8191): 1,
        (131072, 64, 64 * 8192): 0,
    }
    got = _cuts(tmp_path, list(want), "gemm_plan_print")
    assert {k: g[0] for k, g in zip(want, got)} == want
    for (rows, cols, tokens), g in zip(want, got):
        assert not g[0] or g[1] < 2 ** 32
        assert g[2] == -(-tokens // 16) * 16 * cols // 8
    past = _cuts(tmp_path, [(64, 5632, 6_200_000)], "gemm_plan_print")[0][2]
    assert past > 2 ** 32 - 1                 # the caller then runs the GEMV


def test_which_matrix_core_kernel(tmp_path):
    """(rows, cols, tokens) -> 64 x 64 tiles? us of 64 x 64 / 16 x 16, weights from HBM."""
    want = {
        (28672, 4096, 32): 0,     # 48.5 / 47.2
        (28672, 4096, 33): 1,     # 50.0 / 53.7
        (20480, 4096, 33): 0,     # 48.8 / 41
        (20480, 4096, 64): 0,     # 50.0 / 44.3
        (12288, 4096, 33): 0,     # 28.7 / 25.8
        (14336, 4096, 33): 1,     # 29.1 / 33.0
        (11264, 2048, 64): 0,     # 17.0 / 15.8
        (11264, 2048, 65): 0,     # 20.6 / 19.0
        (11264, 2048, 97): 1,     # 21.4 / 24.3
        (4096, 4096, 192): 0,     # 26.6 / 23.4
        (4096, 4096, 200): 1,     # 26.9 / 28.6
        (5120, 5120, 129): 0,     # 31.6 / 28.4
        (5120, 5120, 160): 1,     # 32.4 / 34.7
        (8192, 8192, 129): 0,     # 74.1 / 66.8
        (8192, 8192, 192): 1,     # 76.1 / 80.8
        (4096, 14336, 200): 1,    # 78.4 / 83.6
        (4096, 14336, 320): 0,    # 123.4 / 100.7
        (4096, 14336, 512): 1,    # 129.8 / 159.3
        (4480, 832, 256): 1,      # 13.8 / 16.1: 26 blocks run as 32
        (17408, 4096, 65): 0,     # 57.5 / 48.5
        (6144, 4096, 384): 1,     # 47.9 / 57.0
    }
    got = _cuts(tmp_path, list(want), "gemm_plan_print")
    assert {k: g[0] for k, g in zip(want, got)} == want


def test_cut_of_the_16x16_kernel(tmp_path):
    """(rows, cols, tokens) -> token tiles a workgroup, wide chunks, groups ahead, spare LDS."""
    want = {
        (4096, 4096, 16): (1, 0, 4, 0),
        (4096, 14336, 16): (1, 0, 8, 0),          # 26.4 us, 4 ahead 30.7
        (8192, 8192, 8): (1, 0, 8, 0),            # 21.4, 23.5
        (11264, 8192, 16): (1, 0, 4, 0),
        (14336, 4096, 16): (1, 0, 4, 0),          # 23.0, three a CU 27.5
        (22528, 4096, 16): (1, 0, 4, 35840),      # 30.6, eight a CU 35.5
        (4096, 4096, 32): (2, 0, 4, 0),
        (4096, 14336, 32): (2, 1, 8, 0),          # 28.3, 33.6
        (20480, 4096, 32): (2, 0, 4, 0),          # 35.4, three a CU 37.2
        (28672, 8192, 32): (2, 1, 8, 35840),      # 82.2, 86.0
        (4096, 4096, 33): (3, 1, 4, 0),
        (4096, 14336, 33): (3, 1, 8, 0),
        (17408, 4096, 33): (3, 1, 4, 35840),      # 35.9, 38.3
        (1024, 8192, 192): (4, 1, 4, 0),          # 20.3, 8 ahead 20.5
        (4096, 14336, 64): (4, 1, 8, 0),          # 30.5, 35.8
        (4096, 14336, 65): (3, 1, 4, 0),
        (4096, 14336, 128): (4, 1, 4, 0),
        (4096, 14336, 129): (3, 1, 4, 0),         # 9 tiles: 3 groups of 3
        (4096, 14336, 145): (4, 1, 4, 0),
    }
    got = _cuts(tmp_path, list(want), "gemm_plan_print")
    assert {k: tuple(g[3:]) for k, g in zip(want, got)} == want
