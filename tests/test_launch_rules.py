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


def plan(rules, n_out, n_in, n_tok, wide=1, small=1):
    out = (ctypes.c_int64 * 3)()
    rules.prefill_plan(wide, small, I64(n_out), I64(n_tok), n_in // 128, CUS, out)
    return tuple(out)


# tokens and rows of the large tiles, and the height of their wide tiles (0: all
# on the 128-row kernel); the tokens past them are on the small tiles
@pytest.mark.parametrize("n_out,n_in,n_tok,cols,rows,bm", [
    # small tiles only
    (17408, 5120, 17, 0, 0, 0), (17408, 5120, 33, 0, 0, 0), (17408, 5120, 100, 0, 0, 0), (5120, 17408, 100, 0, 0, 0),
    (1024, 5120, 512, 0, 0, 0), (1000, 5120, 200, 0, 0, 0), (129, 1024, 130, 0, 0, 0),
    # large tiles, and the tokens past them on small ones
    (10240, 5120, 777, 768, 0, 0), (17408, 5120, 777, 768, 17408, 256), (17408, 5120, 400, 384, 0, 0),
    (12288, 5120, 1300, 1280, 12288, 256), (17408, 5120, 2100, 2048, 16384, 256), (5120, 17408, 800, 768, 0, 0),
    # 128-row tiles only
    (17408, 5120, 384, 384, 0, 0), (17408, 5120, 300, 300, 0, 0), (10240, 5120, 768, 768, 0, 0),
    (6144, 5120, 1280, 1280, 0, 0), (12288, 5120, 640, 640, 0, 0), (4096, 4096, 2048, 2048, 0, 0),
    # wide tiles: whole rounds, one round of 256 or of 160 rows
    (17408, 5120, 2048, 2048, 16384, 256), (17408, 5120, 768, 768, 17408, 256), (17408, 5120, 512, 512, 17408, 160),
    (5120, 6144, 2048, 2048, 5120, 160),
    # one round of 256-row tiles, not three full ones of 128 x 128
    (6144, 5120, 2048, 2048, 6144, 256), (12288, 5120, 1024, 1024, 12288, 256), (12288, 4096, 1024, 1024, 12288, 256),
    (8192, 2048, 1536, 1536, 8192, 256), (6144, 5120, 1950, 1950, 0, 0),
    # 256-row tiles and three full rounds of 128 x 128 for the rows past them
    (28672, 8192, 1061, 1024, 16384, 256)])
def test_prefill_plan(rules, n_out, n_in, n_tok, cols, rows, bm):
    assert plan(rules, n_out, n_in, n_tok) == (cols, rows, bm)


@pytest.mark.parametrize("n_tok", [17, 33, 100, 384, 512, 768, 777, 1300, 2048, 4096, 100000])
@pytest.mark.parametrize("n_out,n_in", [(17408, 5120), (5120, 17408), (10240, 5120), (1024, 5120), (300, 3072), (77, 1024)])
def test_prefill_plan_is_launchable(rules, n_out, n_in, n_tok):
    """Token ranges and rows that the launches take: the large tiles' tokens are
    all or whole tiles, the wide rows all or whole tiles, and a kernel that the
    pointers rule out is not used."""
    for wide in (0, 1):
        for small in (0, 1):
            cols, rows, bm = plan(rules, n_out, n_in, n_tok, wide, small)
            assert 0 <= cols <= n_tok and (cols == n_tok or cols % (256 if rows else 128) == 0)
            assert 0 <= rows <= n_out and (rows in (0, n_out) or rows % bm == 0) and (rows > 0) == (bm > 0)
            assert wide or rows == 0
            assert small or cols == n_tok
