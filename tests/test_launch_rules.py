"""CPU: the rules that choose a kernel from sizes alone (csrc/launch_rules.h),
compiled with g++, on both sides of their lines for a card of 256 CUs."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256
I64 = ctypes.c_int64


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rules") / "rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "host", "launch_rules.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


# (tokens, columns): sizes timed on both kernels, and which was the faster
@pytest.mark.parametrize("n_tok,n,per_block", [
    (1, 5120, 1), (51, 5120, 1), (52, 5120, 0), (33, 8192, 0), (2048, 5120, 0), (257, 1024, 0),
    (16, 17408, 1), (28, 17408, 1), (32, 17408, 0), (48, 17408, 0),
    (15, 18432, 1), (36, 18432, 1), (30, 24576, 1), (24, 32768, 1), (28, 32768, 0), (20, 33792, 1), (24, 33792, 0),
    (12, 65536, 1), (14, 65536, 0), (6, 131072, 1), (3, 262144, 1), (1, 1048576, 1), (2, 1048576, 0), (1, 2097152, 0),
    ((1 << 31) - 1, 1024, 0), ((1 << 31) - 1, (1 << 31) - 1024, 0)])
def test_rms_prepass_kernel(rules, n_tok, n, per_block):
    assert rules.rms_per_block(I64(n_tok), I64(n // 1024), I64(CUS)) == per_block


# rows of a workgroup and waves over K of the streamed kernel for 9 to 16 tokens
@pytest.mark.parametrize("n_out,n_in,rows,waves", [
    (1, 5120, 16, 8), (4096, 5120, 16, 8), (4097, 5120, 16, 4), (4224, 5120, 16, 4), (4225, 5120, 32, 8),
    (7168, 5120, 32, 8), (7169, 5120, 16, 4), (8192, 5120, 16, 4), (10240, 5120, 16, 4),
    (4096, 6144, 16, 8), (4097, 6144, 32, 8), (8192, 6144, 32, 8), (8193, 6144, 16, 4), (5120, 17408, 32, 8),
    (1024, 4992, 16, 4), (8192, 4096, 16, 4), ((1 << 31) - 1, 5120, 16, 4)])
def test_streamed_shape_9_to_16_tokens(rules, n_out, n_in, rows, waves):
    assert rules.small_shape(I64(n_out), n_in // 128, I64(CUS)) == 100 * rows + waves


# sizes with every shape timed: the pick, and the time measured for it (us), which
# the estimate has to meet within a quarter
@pytest.mark.parametrize("n_out,n_in,n_tok,bm,bn,us", [
    (17408, 5120, 17, 80, 32, 17.4), (17408, 5120, 33, 80, 48, 22.5), (17408, 5120, 100, 80, 16, 47.1),
    (8703, 5120, 100, 80, 16, 26.5), (2560, 17408, 140, 48, 16, 37.8), (4096, 1024, 80, 48, 16, 5.6),
    (512, 5120, 64, 48, 16, 9.1), (4096, 1024, 33, 32, 32, 5.0), (6144, 5120, 50, 48, 32, 13.4),
    (5120, 17408, 80, 64, 32, 39.8), (10240, 5120, 140, 64, 48, 36.3), (6144, 5120, 140, 80, 48, 22.1)])
def test_small_tile_shape(rules, n_out, n_in, n_tok, bm, bn, us):
    assert rules.mid_pick(I64(n_out), I64(n_tok), n_in // 128, CUS) == 1000 * bm + bn
    rules.mid_us.restype = ctypes.c_float
    assert 0.75 * us < rules.mid_us(I64(n_out), I64(n_tok), n_in // 128, CUS) < 1.25 * us
