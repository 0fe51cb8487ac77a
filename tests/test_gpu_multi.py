"""GPU parity of matmul_bt at a few tokens (batched decode: Weight::matmul_bt,
quant.rs:751-907, as forward_each calls it, llama.rs:418-434), which the
library runs as a multi-token GEMV that streams the weights once for every
token: on the VALU (dot4 per row and token; two token rows, or any with
KVAD_MMA_MIN above m) or on the matrix cores (one v_mfma_i32_16x16x32_i8
per block of 16 rows x 16 tokens; from five token rows).

Bar: f32 outputs within 1e-5 x max|ref| of the oracle's matmul.  On the VALU
path each token's row equals, to the bit, a single-token matvec of that
token (the per-token arithmetic is the GEMV's, term for term); on the matrix
cores the exact i32 block dots are scaled and summed in another order, so
the row is held to 1e-5 x max|row| of the matvec.  Shapes cover ragged row
counts (a last 16-row group part-filled), k tails (widths not a multiple of
four blocks), rows of one and of several segments, widths whose staged
codes take more than one launch of token slots, and, on the matrix cores,
more than 16 tokens (a launch per 16).
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

import kvad_amd as K  # noqa: E402  (fails loudly without libkvad_hip.so)

from test_gpu_gemm import oracle_matmul  # noqa: E402
from test_gpu_gemv import close, make, say  # noqa: E402

# (rows, cols) per precision: ragged rows, one segment, several segments,
# Qwen2.5-0.5B FFN shapes, a Llama-3-8B down row width
SHAPES = {
    "q8": [(37, 64), (130, 2048), (4864, 896), (896, 4864)],
    "q4": [(37, 64), (130, 2048), (896, 4864)],
    "q4k": [(37, 256), (130, 4096), (300, 14336)],
}


PATHS = {"valu": "99", "mma": "2"}  # KVAD_MMA_MIN: the matrix cores from this many rows


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("prec", ["q8", "q4", "q4k"])
@pytest.mark.parametrize("m", [2, 3, 4, 5, 8])
def test_few_tokens_match_the_oracle_and_single_matvecs(ctx, monkeypatch, path, prec, m):
    monkeypatch.setenv("KVAD_MMA_MIN", PATHS[path])
    for rows, cols in SHAPES[prec]:
        say("multi-token matmul", path, prec, m, rows, cols)
        w, parts = make(ctx, prec, rows, cols, seed=rows + cols + m)
        xs = O.normal(rows * 7 + m, m * cols)
        bias = O.normal(rows + 3, rows)
        for b in (None, bias):
            got = w.matmul_bt(xs, m, b)
            close(got, oracle_matmul(prec, parts, rows, cols, xs, m, b))
            got = got.reshape(m, rows)
            for t in range(m):
                one = w.matvec_bt(xs[t * cols:(t + 1) * cols], b)
                if path == "valu":
                    np.testing.assert_array_equal(got[t], one)
                else:
                    close(got[t], one)


@pytest.mark.parametrize("prec,rows,cols", [("q8", 8960, 1536), ("q8", 65552, 256), ("q4", 11008, 2048),
                                            ("q4k", 14336, 2048), ("q4k", 4096, 4096)])
def test_up_to_four_rows_are_their_matvecs(ctx, prec, rows, cols):
    # over large matrices too, where the matrix cores would be a little ahead
    say("four rows", prec, rows, cols)
    w, _ = make(ctx, prec, rows, cols, seed=rows)
    for m in (2, 3, 4):
        xs = O.normal(cols + m, m * cols)
        got = w.matmul_bt(xs, m).reshape(m, rows)
        for t in range(m):
            np.testing.assert_array_equal(got[t], w.matvec_bt(xs[t * cols:(t + 1) * cols]))


# the matrix cores: ragged 16-row groups, k tails of 1..3 blocks past whole
# four-block units, Q4_K's minimum terms over several super-blocks, and
# Qwen2.5-0.5B / Llama-3-8B widths
MMA_SHAPES = {
    "q8": [(1, 32), (17, 96), (37, 160), (130, 2048), (896, 4864), (64, 14336)],
    "q4": [(1, 32), (17, 96), (37, 224), (130, 2048), (896, 4864)],
    "q4k": [(1, 256), (17, 768), (130, 4096), (64, 14336)],
}


@pytest.mark.parametrize("prec", ["q8", "q4", "q4k"])
@pytest.mark.parametrize("m", [3, 8, 9, 16, 17, 40])
def test_matrix_core_tokens_match_the_oracle(ctx, monkeypatch, prec, m):
    # up to 40 rows through the matrix-core path (KVAD_MULTI_TOKENS,
    # KVAD_MMA_MIN): tiles of 16 tokens, one or two a workgroup; 17 and 40 take
    # several, each writing its own rows of y
    monkeypatch.setenv("KVAD_MULTI_TOKENS", "64")
    monkeypatch.setenv("KVAD_MMA_MIN", "2")
    for rows, cols in MMA_SHAPES[prec]:
        say("matrix-core matmul", prec, m, rows, cols)
        w, parts = make(ctx, prec, rows, cols, seed=3 * rows + cols + m)
        xs = O.normal(rows * 5 + m, m * cols)
        bias = O.normal(rows + 7, rows)
        for b in (None, bias):
            close(w.matmul_bt(xs, m, b), oracle_matmul(prec, parts, rows, cols, xs, m, b))


# k-ranges at the edges of the matrix-core kernel's slices: a wave holds 1, 2,
# 4, 7 (Q4_K, 256 wide) or 1, 2, 4, 8, 14 (q8 / q4, 128 wide) units of the
# row, eight waves a workgroup; past the widest slice the row takes a second
# range, past 16 tokens a split over the grid.  Tails of one block included.
EDGE_COLS = {
    "q8": [128, 512, 544, 1056, 2048, 2080, 4096, 4128, 8224, 14368],
    "q4": [512, 1024, 1056, 2080, 4128, 8192, 14336, 14368],
    "q4k": [256, 1024, 1280, 2048, 2304, 4096, 4352, 8192, 8448, 14336, 14592],
}


@pytest.mark.parametrize("prec", list(EDGE_COLS))
@pytest.mark.parametrize("m", [5, 16, 17, 33])
def test_matrix_core_k_ranges_match_the_oracle(ctx, monkeypatch, prec, m):
    monkeypatch.setenv("KVAD_MULTI_TOKENS", "64")
    rows = 35  # three 16-row groups, the last part-filled
    for cols in EDGE_COLS[prec]:
        say("matrix-core k-range", prec, m, rows, cols)
        w, parts = make(ctx, prec, rows, cols, seed=cols + m)
        xs = O.normal(cols + 11 * m, m * cols)
        bias = O.normal(rows + 5, rows)
        close(w.matmul_bt(xs, m, bias), oracle_matmul(prec, parts, rows, cols, xs, m, bias))


@pytest.mark.parametrize("prec", ["q8", "q4", "q4k"])
@pytest.mark.parametrize("rows,cols", [(4113, 256), (8210, 512), (33001, 256), (4500, 2304)])
def test_matrix_core_groups_in_turn_match_the_oracle(ctx, monkeypatch, prec, rows, cols):
    # more 16-row groups than workgroups: one, two or a few groups a
    # workgroup, and two workgroups a CU from eight groups a CU
    monkeypatch.setenv("KVAD_MULTI_TOKENS", "64")
    for m in (5, 19):
        say("matrix-core groups", prec, m, rows, cols)
        w, parts = make(ctx, prec, rows, cols, seed=rows + m)
        xs = O.normal(rows + 3 * m, m * cols)
        close(w.matmul_bt(xs, m), oracle_matmul(prec, parts, rows, cols, xs, m))


def test_matrix_core_keeps_odd_values_to_their_rows(ctx, monkeypatch):
    # an infinite or NaN scale in one weight row or token stays in that row:
    # the k tail's lanes read the next row's scale
    monkeypatch.setenv("KVAD_MULTI_TOKENS", "64")
    rows, cols, m = 40, 160, 6
    s, q = O.quantize_q8(O.normal(3, rows * cols, 0.02), rows, cols)
    s = s.reshape(rows, cols // 32).copy()
    s[7, 0], s[21, 1] = np.inf, np.nan
    xs = O.normal(4, m * cols)
    w = K.Weight.from_q8(ctx, rows, cols, s.ravel(), q)
    got = w.matmul_bt(xs, m).reshape(m, rows)
    bad = np.zeros(rows, bool)
    bad[[7, 21]] = True
    assert not np.isfinite(got[:, bad]).any()
    s[7, 0] = s[21, 1] = 0.0
    want = O.matmul_q8(s.ravel(), q, rows, cols, xs, m).reshape(m, rows)
    close(got[:, ~bad].ravel(), np.ascontiguousarray(want[:, ~bad]).ravel())


def test_many_token_slots_stream_in_launches(ctx, monkeypatch):
    # the VALU path, 8 tokens at a width whose codes fill the LDS stage for 2
    # at a time
    monkeypatch.setenv("KVAD_MMA_MIN", "99")
    rows, cols, m = 64, 14336, 8
    say("multi-token matmul, staged in launches")
    w, parts = make(ctx, "q4k", rows, cols, seed=5)
    xs = O.normal(6, m * cols)
    got = w.matmul_bt(xs, m)
    close(got, oracle_matmul("q4k", parts, rows, cols, xs, m))


@pytest.mark.parametrize("path", list(PATHS))
def test_zero_and_edge_tokens(ctx, monkeypatch, path):
    # a token of zeros quantises to zero codes (scale 0): its row is the bias
    monkeypatch.setenv("KVAD_MMA_MIN", PATHS[path])
    rows, cols, m = 96, 512, 3
    w, parts = make(ctx, "q8", rows, cols, seed=9)
    xs = O.normal(10, m * cols)
    xs[cols:2 * cols] = 0.0
    bias = O.normal(11, rows)
    got = w.matmul_bt(xs, m, bias).reshape(m, rows)
    np.testing.assert_array_equal(got[1], bias.astype(np.float32))
    close(got.ravel(), oracle_matmul("q8", parts, rows, cols, xs, m, bias))


@pytest.mark.parametrize("prec,rows,cols,m,bound", [("q4k", 512, 14336, 12, 1.9e-7), ("q4k", 512, 4096, 12, 1.48e-7),
                                                    ("q8", 512, 14336, 12, 1.25e-7), ("q4", 512, 4864, 16, 0.95e-7)])
def test_few_row_sums_stay_near_64_bits(ctx, monkeypatch, prec, rows, cols, m, bound):
    # A wave adds each unit's blocks up by themselves before the group's sum
    # takes them: in one chain over its share of the row the 2-norm of the error
    # was 2.25e-7, 1.55e-7, 1.49e-7 and 1.01e-7; the sums of units give 1.50e-7,
    # 1.40e-7, 1.03e-7 and 0.86e-7.
    say("few-row error", prec, rows, cols, m)
    rng = np.random.default_rng(cols)
    xs = (rng.standard_normal((m, cols)) * np.exp(0.5 * rng.standard_normal(cols))).astype(np.float32)
    b = xs.reshape(m, -1, 32)
    scale = (np.abs(b).max(2, keepdims=True) / np.float32(127)).astype(np.float32)
    t = (b * (np.float32(1) / scale)).astype(np.float64)
    x64 = (np.clip(np.sign(t) * np.floor(np.abs(t) + 0.5), -127, 127) * scale.astype(np.float64)).reshape(m, cols)
    if prec == "q4k":
        n, sup = rows, cols // 256
        sc, mn = rng.integers(20, 64, (2, n, sup, 8)).astype(np.uint8)
        q = np.clip(np.round(7.5 + 3.0 * rng.standard_normal((n, sup, 8, 32))), 0, 15).astype(np.uint8)
        d = (1.6e-4 * np.exp(0.2 * rng.standard_normal((n, sup)))).astype(np.float16)
        dmin = (7.5 * d.astype(np.float32)).astype(np.float16)
        blk = np.empty((n, sup, 144), np.uint8)
        blk[:, :, 0:2] = d.reshape(n, sup, 1).view(np.uint8)
        blk[:, :, 2:4] = dmin.reshape(n, sup, 1).view(np.uint8)
        blk[:, :, 4:8] = sc[:, :, :4] | (sc[:, :, 4:] >> 4 << 6)
        blk[:, :, 8:12] = mn[:, :, :4] | (mn[:, :, 4:] >> 4 << 6)
        blk[:, :, 12:16] = (sc[:, :, 4:] & 15) | ((mn[:, :, 4:] & 15) << 4)
        blk[:, :, 16:] = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(n, sup, 128)
        w = K.Weight.from_q4k(ctx, rows, cols, blk.ravel())
        w64 = ((d.astype(np.float64)[:, :, None] * sc)[..., None] * q
               - (dmin.astype(np.float64)[:, :, None] * mn)[..., None]).reshape(rows, cols)
    else:
        s = (0.02 / 3 * np.exp(0.2 * rng.standard_normal((rows, cols // 32))) / (40 if prec == "q8" else 2.5)).astype(np.float32)
        lim = 127 if prec == "q8" else 8
        q = np.clip(np.round(rng.standard_normal((rows, cols // 32, 32)) * lim / 3), -lim, lim - 1).astype(np.int8)
        w64 = (q * s.astype(np.float64)[:, :, None]).reshape(rows, cols)
        if prec == "q8":
            w = K.Weight.from_q8(ctx, rows, cols, s.ravel(), q.ravel())
        else:  # byte i of a block: weight i (low nibble), 16 + i (high), code + 8
            u = (q + 8).astype(np.uint8)
            w = K.Weight.from_q4(ctx, rows, cols, s.ravel(), (u[:, :, :16] | (u[:, :, 16:] << 4)).ravel())
    want = x64 @ w64.T
    got = w.matmul_bt(xs.ravel(), m).reshape(m, rows)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    say("few-row error", f"{err:.2e}")
    assert err <= bound
