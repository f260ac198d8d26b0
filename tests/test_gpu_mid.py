"""The small-tile GEMM for a few dozen to a few hundred tokens (gemm_mid.hip):
every tile shape at the edges of its tiles and of K, against the oracle and
the 128-row kernel, exact where the result is an integer, and with block and
activation scales at the ends of fp16."""
import numpy as np
import pytest

from test_gpu_exact import (B, O, case, check_exact, dev, host, integer_tokens, run_gemm, sample_rows, torch,
                            unit_scale_weights)

pytestmark = pytest.mark.gpu

# fp32 sums of nb block terms, each a sum of 4 chunk terms: (nb + 4) roundings of
# 2^-24 at most, against the largest output; 1e-5 is the bar of every GEMM here
TOL = 1e-5
SHAPES = {1: (80, 48), 2: (48, 32), 3: (80, 32), 4: (64, 32), 5: (64, 48), 6: (32, 32), 7: (80, 16), 8: (80, 16), 9: (48, 16)}


def normwise(a, ref):
    return float(np.max(np.abs(a.astype(np.float64) - ref)) / np.max(np.abs(ref)))


def gemm(W, Xq, n_out, n_in, n_tok):
    Y = torch.full((n_out, n_tok), float("nan"), dtype=torch.float32, device="cuda")
    B.gemm(W, Xq, Y, n_out, n_in, n_tok)
    return host(Y)


def sizes(shape):
    bm, bn = SHAPES[shape]
    # one row and one column past a tile; less than a tile; whole tiles; token
    # counts of every alignment; 1, 2 and 17 steps of 8 blocks
    return [(bm + 1, 1024, bn + 1), (bm - 1, 2048, 17), (2 * bm, 1024, 2 * bn), (5, 17408, 18), (3 * bm - 7, 5120, 3 * bn - 1)]


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_mid_shapes(shape, knobs):
    for n_out, n_in, n_tok in sizes(shape):
        case(f"mid GEMM shape {shape}: {n_out}x{n_in}x{n_tok}")
        W = O.gen_weights(6100 + n_out, n_out, n_in)
        X = O.gen_normal(6101 + n_tok, n_tok * n_in).reshape(n_tok, n_in)
        Xq = O.quantize_chunk_major(X)
        Wd, Xd = dev(W), dev(Xq)
        knobs.set("BONSAI_GEMM_MID", shape)
        got = gemm(Wd, Xd, n_out, n_in, n_tok)
        knobs.set("BONSAI_GEMM_MID", 0)
        other = gemm(Wd, Xd, n_out, n_in, n_tok)
        ref = O.gemm(W, Xq, n_out, n_in, n_tok, nthreads=16)
        assert np.all(np.isfinite(got))
        assert normwise(got, ref) <= TOL
        assert normwise(got, other) <= TOL


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_mid_integer_sums_exact(shape, knobs):
    """Unit scales: every output is an integer below 2^24, so the chunk dots
    (and the offsets that the operands carry) have to be exact."""
    bm, bn = SHAPES[shape]
    n_out, n_in, n_tok = bm + 3, 5120, bn + 5
    knobs.set("BONSAI_GEMM_MID", shape)
    case(f"mid GEMM shape {shape}, exact integers {n_out}x{n_in}x{n_tok}")
    W, X = unit_scale_weights(6200 + shape, n_out, n_in), integer_tokens(6201 + shape, n_tok, n_in)
    check_exact(run_gemm(W, X, n_out, n_in, n_tok), W, X, sample_rows(n_out), n_in)


def test_mid_scales_at_the_ends(knobs):
    """Block scales that are zero, subnormal, or large beside code 3, saturated
    q, and activations whose scale is zero or infinite: an infinite d gives
    what the reference's fp32 arithmetic gives."""
    knobs.set("BONSAI_GEMM_MID", 1)
    case("mid GEMM 200x2048x50, scales at the ends of fp16")
    n_out, n_in, n_tok = 200, 2048, 50
    nb = n_in // 128
    W = O.gen_weights(6300, n_out, n_in).copy()
    rng = np.random.default_rng(63)
    blocks = W.reshape(n_out, nb, 34)
    for r in range(n_out):
        for b in rng.choice(nb, 3, replace=False):
            d = rng.integers(0x7800, 0x7C00) if r % 3 == 0 else rng.integers(0, 1024)
            blocks[r, b, :2] = np.frombuffer(np.uint16(d | (0x8000 if rng.random() < 0.5 else 0)).tobytes(), np.uint8)
            if r % 3 == 0:
                blocks[r, b, 2:] = rng.integers(0, 256, 32, dtype=np.uint8)
    X = O.gen_normal(6301, n_tok * n_in).reshape(n_tok, n_in)
    X[3] = 0
    X[4] = np.where(rng.random(n_in) < 0.5, 1.0, -1.0)                    # every q is +-127
    Xq = O.quantize_chunk_major(X).copy()
    Wd = dev(W)
    got = gemm(Wd, dev(Xq), n_out, n_in, n_tok)
    assert np.all(np.isfinite(got)) and np.all(got[:, 3] == 0)
    assert normwise(got, O.gemm(W, Xq, n_out, n_in, n_tok, nthreads=16)) <= TOL
    q = Xq.reshape(n_in // 32, n_tok, 36)
    q[7, 11, :2] = np.frombuffer(np.uint16(0x7C00).tobytes(), np.uint8)    # d = inf in one chunk of token 11
    got = gemm(Wd, dev(Xq), n_out, n_in, n_tok)
    ref = O.gemm(W, Xq, n_out, n_in, n_tok, nthreads=16)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    inf = np.isinf(ref)
    assert inf.any() and np.array_equal(got[inf], ref[inf])
    fine = np.isfinite(ref)
    assert np.max(np.abs(got[fine] - ref[fine])) <= TOL * np.max(np.abs(ref[fine]))


# the last figure is the tokens that stay on the large tiles (or, up to 16, on the
# streamed kernel)
@pytest.mark.parametrize("n_out,n_in,n_tok,cols", [
    (1024, 5120, 512, 0), (5120, 17408, 100, 0), (17408, 5120, 33, 0), (17408, 5120, 12, 0), (6144, 5120, 651, 640),
    (10240, 5120, 777, 768), (17408, 5120, 400, 384), (17408, 5120, 2100, 2048)])
def test_mid_default_dispatch(n_out, n_in, n_tok, cols, knobs):
    """Shapes the default rule gives to this kernel, whole or the tokens past the
    large tiles' whole ones, with and without a workspace (the same bytes), on a
    row sample.  Without this kernel (BONSAI_GEMM_MID=0) the tokens before those
    keep their bytes and the others, whose sums it adds in another order, do not."""
    case(f"mid GEMM by default: {n_out}x{n_in}x{n_tok}")
    W = O.gen_weights(6400 + n_out, n_out, n_in)
    X = O.gen_normal(6401 + n_tok, n_tok * n_in).reshape(n_tok, n_in)
    Xq = O.quantize_chunk_major(X)
    Wd, Xd = dev(W), dev(Xq)
    got = gemm(Wd, Xd, n_out, n_in, n_tok)
    ws = torch.full((B.gemm_workspace_bytes(n_in, n_tok),), 255, dtype=torch.uint8, device="cuda")
    Y = torch.full((n_out, n_tok), float("nan"), dtype=torch.float32, device="cuda")
    B.gemm_ws(Wd, Xd, Y, n_out, n_in, n_tok, ws)
    assert np.array_equal(got.view(np.uint32), host(Y).view(np.uint32))
    rows = np.r_[0:24, n_out // 2 - 12:n_out // 2 + 12, n_out - 24:n_out]
    rb = n_in // 128 * 34
    Ws = np.concatenate([W[r * rb:(r + 1) * rb] for r in rows])
    assert np.all(np.isfinite(got))
    assert normwise(got[rows], O.gemm(Ws, Xq, rows.size, n_in, n_tok, nthreads=16)) <= TOL
    knobs.set("BONSAI_GEMM_MID", 0)
    without = gemm(Wd, Xd, n_out, n_in, n_tok)
    np.testing.assert_array_equal(got[:, :cols].view(np.uint32), without[:, :cols].view(np.uint32))
    assert np.all(np.any(got[:, cols:] != without[:, cols:], axis=0))


def test_mid_stored_sum_up_to_16_tokens(knobs):
    """Batches of up to 16 tokens subtract each activation block's stored s,
    whatever it is: the 80 x 16 tiles as the streamed kernel of those sizes, and
    as the reference."""
    n_out, n_in, n_tok = 83, 5120, 13
    case(f"mid GEMM {n_out}x{n_in}x{n_tok}, stored sums that are not the sums")
    W = O.gen_weights(6500, n_out, n_in)
    Xq = O.quantize_chunk_major(O.gen_normal(6501, n_tok * n_in).reshape(n_tok, n_in)).copy()
    s = np.random.default_rng(65).integers(-32768, 32768, Xq.size // 36, dtype=np.int16)
    Xq.reshape(-1, 36)[:, 2:4] = s.view(np.uint8).reshape(-1, 2)
    Wd, Xd = dev(W), dev(Xq)
    ref = O.gemm(W, Xq, n_out, n_in, n_tok, nthreads=16)
    for knob in (7, 0):
        knobs.set("BONSAI_GEMM_MID", knob)
        assert normwise(gemm(Wd, Xd, n_out, n_in, n_tok), ref) <= TOL


@pytest.mark.parametrize("n_out,n_in,n_tok", [(1000, 5120, 17), (1000, 5120, 200), (300, 6144, 77), (129, 1024, 130),
                                              (200, 2048, 64), (10240, 5120, 777)])
def test_f16_knobs_reach_the_128_row_kernel(n_out, n_in, n_tok, knobs):
    """Sizes that the default rule gives to the small tiles, wholly or in part:
    with a knob of the 128-row kernel set (its token tile, split and waves) that
    kernel runs, every token of it: the bytes of BONSAI_GEMM_WIDE=0, which are
    others than the small tiles' (another order of the sums)."""
    case(f"gemm {n_out}x{n_in}x{n_tok}, the 128-row kernel's knobs")
    W = O.gen_weights(6600 + n_out, n_out, n_in)
    Xq = O.quantize_chunk_major(O.gen_normal(6601 + n_tok, n_tok * n_in).reshape(n_tok, n_in))
    Wd, Xd = dev(W), dev(Xq)
    knobs.set("BONSAI_GEMM_WIDE", 0)
    large = gemm(Wd, Xd, n_out, n_in, n_tok)
    knobs.unset("BONSAI_GEMM_WIDE")
    assert np.any(large != gemm(Wd, Xd, n_out, n_in, n_tok))
    for name, value in (("BN", 64), ("BN", 128), ("SPLIT", 0), ("SPLIT", 1), ("WAVES", 8), ("WAVES", 16)):
        knobs.set("BONSAI_GEMM_F16_" + name, value)
        np.testing.assert_array_equal(gemm(Wd, Xd, n_out, n_in, n_tok).view(np.uint32), large.view(np.uint32),
                                      err_msg=f"{name} = {value}")
        knobs.unset("BONSAI_GEMM_F16_" + name)
