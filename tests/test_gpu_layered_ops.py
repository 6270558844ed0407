"""Every mechanism of the layered decoders on its own, against the plain restatement (plain_stack.py).

Both element types: fp32 has to agree to fp32 rounding, bfloat16 to the rounding of its inputs and outputs
(the oracle gets the same rounded inputs).  Sizes are chosen to be ragged: nothing here is a multiple of
what a kernel's tile happens to be.
"""
import ctypes as C

import numpy as np
import pytest

import gemm_plan
import plain_stack as S
from layered_helpers import BF16, BOTH, F32, call, close, get, get_ints, gpu, ints, pack_gated, pad, put, rounded, up64, zeros  # noqa: F401

pytestmark = pytest.mark.gpu


# ---- linear ---------------------------------------------------------------------------------------------
@BOTH
@pytest.mark.parametrize("M,K,N", [(1, 64, 5), (3, 192, 70), (37, 320, 100), (64, 128, 129), (130, 256, 200), (300, 448, 2048),
                                   (513, 128, 4100), (2, 1024, 300), (31, 2048, 1100), (48, 1536, 65), (64, 512, 3000)])
def test_linear_with_bias_and_gelu_columns(gpu, dt, M, K, N):
    rng = np.random.default_rng(M * 7 + N)
    x, w, b = rounded(rng.standard_normal((M, K))), rounded(rng.standard_normal((N, K)) / K ** 0.5), rng.standard_normal(N)
    cut, ldo = N // 3, up64(N)
    out = zeros(gpu, (M, ldo), dt)
    call(gpu, "lcu_linear", out, 0, ldo, put(gpu, x, dt), put(gpu, w, dt), put(gpu, b), cut, dt, M, K, N)
    want = x @ w.T + b
    want[:, :cut] = S.gelu_tanh(want[:, :cut])
    got = get(gpu, out, (M, ldo), dt)
    close(got[:, :N], want, dt)
    assert (got[:, N:] == 0).all()                                    # the padding of the rows is left alone
    out = zeros(gpu, (M, N))
    call(gpu, "lcu_linear", out, 1, N, put(gpu, x, dt), put(gpu, w, dt), None, 0, dt, M, K, N)
    close(get(gpu, out, (M, N)), x @ w.T, F32)                        # fp32 output of either type
    gpu.release()


# tiles of 256 rows in bfloat16 with ragged rows and columns, a single K stage, and tiles of 128 rows; the last four columns as fp32 of their own
@pytest.mark.parametrize("M,K,N", [(2049, 192, 4100), (4096, 64, 4096), (300, 320, 12804), (100, 192, 20484), (127, 64, 35000),
                                   (257, 64, 6790), (1100, 320, 3684)])
def test_linear_large_tiles(gpu, M, K, N):
    rng = np.random.default_rng(N)
    x, w, b = rounded(rng.standard_normal((M, K))), rounded(rng.standard_normal((N, K)) / K ** 0.5), rng.standard_normal(N)
    xd, wd, ldo, tail = put(gpu, x, BF16), put(gpu, w, BF16), up64(N), 4
    want = x @ w.T + b
    want[:, :100] = S.gelu_tanh(want[:, :100])
    out = zeros(gpu, (M, ldo), BF16)
    call(gpu, "lcu_linear", out, 0, ldo, xd, wd, put(gpu, b), 100, BF16, M, K, N)
    got = get(gpu, out, (M, ldo), BF16)
    close(got[:, :N], want, BF16)
    assert (got[:, N:] == 0).all()
    last = zeros(gpu, (M, tail))
    out = zeros(gpu, (M, ldo), BF16)
    call(gpu, "lcu_linear_tail", out, ldo, last, tail, N - tail, xd, wd, BF16, M, K, N)
    close(get(gpu, out, (M, ldo), BF16)[:, :N - tail], (x @ w.T)[:, :-tail], BF16)
    close(get(gpu, last, (M, tail)), (x @ w.T)[:, -tail:], F32)
    out = zeros(gpu, (M, N + 1))
    call(gpu, "lcu_linear", out, 1, N + 1, xd, wd, None, 0, BF16, M, K, N)   # rows off any 16-byte boundary
    close(get(gpu, out, (M, N + 1))[:, :N], x @ w.T, F32)
    out = zeros(gpu, (M, N + 1), BF16)
    call(gpu, "lcu_linear", out, 0, N + 1, xd, wd, None, 0, BF16, M, K, N)
    close(get(gpu, out, (M, N + 1), BF16)[:, :N], x @ w.T, BF16)
    assert (get(gpu, out, (M, N + 1), BF16)[:, N:] == 0).all()
    gpu.release()


@pytest.mark.parametrize("M,K,ff", [(4096, 64, 2048), (2050, 128, 4100), (100, 64, 10250), (70, 128, 17000), (300, 64, 4000)])
def test_gated_linear_large_tiles(gpu, M, K, ff):
    rng = np.random.default_rng(ff)
    x, gw, uw = rounded(rng.standard_normal((M, K))), rounded(rng.standard_normal((ff, K)) / K ** 0.5), \
        rounded(rng.standard_normal((ff, K)) / K ** 0.5)
    ld = up64(ff)
    out = zeros(gpu, (M, ld), BF16)
    gate = gpu.B.GateParams(0.75, 1.702, 1.0)
    call(gpu, "lcu_linear_gated", out, ld, put(gpu, x, BF16), put(gpu, pack_gated(gw, uw, ld), BF16), C.byref(gate), BF16, M, K, 2 * ld)
    close(get(gpu, out, (M, ld), BF16)[:, :ff], S.expert(x, gw, uw, np.eye(ff), 0.75), BF16)
    gpu.release()


# few rows of weights that come from memory, marked as read once: one launch with what follows (6 and 5 rows) and two, one to four row tiles, ragged columns
@pytest.mark.parametrize("gated,M,K,N", [(False, 6, 4096, 8301), (False, 16, 4096, 8300), (False, 30, 4096, 8300), (False, 60, 4096, 8300), (False, 9, 1024, 33000),
                                         (True, 5, 4096, 4160), (True, 15, 4096, 4160), (True, 31, 2048, 8320), (True, 50, 4096, 4224)])
def test_linear_of_weights_from_memory(gpu, gated, M, K, N):
    known, outs = 13 << 30, up64(N)
    assert gemm_plan.few_rows("bf16", M, K, 2 * outs if gated else N, known=known)[1:] == (True, True)
    rng = np.random.default_rng(M)
    x = rounded(rng.standard_normal((M, K)))
    ws = [rounded(rng.standard_normal((N, K)) / K ** 0.5) for _ in range(2 if gated else 1)]
    xd, wd, gate = put(gpu, x, BF16), put(gpu, pack_gated(*ws, outs) if gated else ws[0], BF16), gpu.B.GateParams(7.0, 1.702, 1.0)
    results = []
    for bytes_known in (known, 0):
        gpu.B.check(gpu.L().lcu_stream_weights(gpu.stream, bytes_known))
        out = zeros(gpu, (M, outs), BF16 if gated else F32)
        if gated:
            call(gpu, "lcu_linear_gated", out, outs, xd, wd, C.byref(gate), BF16, M, K, 2 * outs)
        else:
            call(gpu, "lcu_linear", out, 1, outs, xd, wd, None, 0, BF16, M, K, N)
        results.append(get(gpu, out, (M, outs), BF16 if gated else F32)[:, :N])
    assert (results[0] == results[1]).all()
    close(results[0], S.expert(x, *ws, np.eye(N), 7.0) if gated else x @ ws[0].T, BF16 if gated else F32)
    gpu.release()


# products of 65 and more rows with few tiles over a long K, whose K is never split: a layer's roundings decide which experts a token takes, so the
# order of the sums hangs neither on the stream nor on its workspace
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("M,K,N", [(65, 4096, 1530), (65, 4096, 4096), (100, 2048, 2816), (129, 2880, 2045), (300, 4096, 6146), (513, 5632, 2061), (900, 10752, 1030)])
def test_linear_same_bits_on_every_stream(gpu, M, K, N, gated):
    rng = np.random.default_rng(N)
    x = rounded(rng.standard_normal((M, K)))
    gate, ld = gpu.B.GateParams(7.0, 1.702, 1.0), up64(N)
    ws = [rounded(rng.standard_normal((N, K)) / K ** 0.5) for _ in range(2 if gated else 1)]
    xd, wd = put(gpu, x, BF16), put(gpu, pack_gated(*ws, ld) if gated else ws[0], BF16)
    results = []
    for stream in (gpu.stream, None):  # one of its own workspace, and one that shares the device's
        out = zeros(gpu, (M, ld), BF16 if gated else F32)
        gpu.B.check(gpu.L().lcu_sync(gpu.stream))
        if gated:
            gpu.B.check(gpu.L().lcu_linear_gated(out.ptr, ld, xd.ptr, wd.ptr, C.byref(gate), BF16, M, K, 2 * ld, stream))
        else:
            gpu.B.check(gpu.L().lcu_linear(out.ptr, 1, ld, xd.ptr, wd.ptr, None, 0, BF16, M, K, N, stream))
        gpu.B.check(gpu.L().lcu_sync(stream))
        results.append(get(gpu, out, (M, ld), BF16 if gated else F32))
    assert np.array_equal(*results)
    if not gated:
        close(results[0][:, :N], x.astype(np.float32) @ ws[0].T.astype(np.float32), F32)
    gpu.release()


# few rows whose splits are added up where they end: one to four row tiles, odd and ragged columns, lhs that just fits beside the rings (24x2048) and
# that does not (25x2048), outputs over lhs, which may only be written when all of lhs has been read
@pytest.mark.parametrize("M,K,N", [(1, 2048, 1531), (2, 512, 515), (16, 2048, 3071), (24, 2048, 1000), (25, 2048, 1000), (31, 1024, 2047), (64, 512, 4100)])
def test_linear_few_rows_in_one_launch(gpu, M, K, N):
    test_linear_large_tiles(gpu, M, K, N)
    rng = np.random.default_rng(N)
    x, w = rounded(rng.standard_normal((M, K))), rounded(rng.standard_normal((N, K)) / K ** 0.5)
    whole = np.zeros((1, M * max(K, N)))
    whole[0, :M * K] = x.reshape(-1)
    both = put(gpu, whole, BF16)
    call(gpu, "lcu_linear", both, 0, N, both, put(gpu, w, BF16), None, 0, BF16, M, K, N)
    close(get(gpu, both, (1, M * max(K, N)), BF16)[0, :M * N].reshape(M, N), (x.astype(np.float32) @ w.T.astype(np.float32)).astype(np.float64), BF16)
    gpu.release()


@pytest.mark.parametrize("M,K,ff", [(1, 1024, 1000), (16, 2048, 2816), (17, 1920, 700), (33, 896, 2030), (64, 512, 1990)])
def test_gated_linear_few_rows_in_one_launch(gpu, M, K, ff):
    test_gated_linear_large_tiles(gpu, M, K, ff)


# 128 columns over a short K; gated tiles of 128x128 that outnumber the compute units, on both sides of theirs
@pytest.mark.parametrize("M,K,N", [(1441, 512, 8900), (1441, 640, 8900),
                                   (8, 512, 30000), (40, 640, 25000),  # few rows in two rounds of workgroups
                                   (56, 512, 16580), (56, 640, 16580), (56, 512, 5000)])  # runs of 4 and of 5, more and fewer tiles
def test_linear_large_tiles_by_length(gpu, M, K, N):
    test_linear_large_tiles(gpu, M, K, N)


# 192 and 256 columns alone, ragged ends
@pytest.mark.parametrize("M,K,N,columns", [(263, 2048, 16470, 192), (600, 4096, 16830, 256)])
def test_linear_wide_tiles(gpu, M, K, N, columns):
    assert gemm_plan.large("bf16", M, K, N, ragged=False) == (columns, 0, 0, 0, 0)
    test_linear_large_tiles(gpu, M, K, N)


# whole rounds of 128, 192 and 256 columns and what is left of them in tiles of 128x128 and of 256 rows
@pytest.mark.parametrize("M,K,N,plan", [(773, 2048, 12296, (128, 64, 8192, 128, 128)), (1027, 2048, 13178, (192, 51, 9792, 128, 128)),
                                        (1033, 2048, 13392, (192, 51, 9792, 256, 128)), (1282, 4096, 13464, (256, 42, 10752, 128, 128))])
def test_linear_columns_left_of_whole_rounds(gpu, M, K, N, plan):
    assert gemm_plan.large("bf16", M, K, N, ragged=False) == plan
    test_linear_large_tiles(gpu, M, K, N)


# tiles below 128x64, either side of where a round of the narrowest ends
@pytest.mark.parametrize("M,K,N,tile", [(66, 64, 4096, (64, 32)), (300, 192, 1590, (64, 32)), (300, 128, 1640, (64, 64)), (129, 320, 4094, (64, 64))])
def test_linear_smaller_tiles(gpu, M, K, N, tile):
    assert gemm_plan.tile_size(M, N, 1, (64, 64), True) == tile and gemm_plan.rows(M, 128, N)[0] == "halves"
    test_linear_large_tiles(gpu, M, K, N)


# columns of one tile: the workgroup that stores rows has read them, so outputs may lie over lhs
@pytest.mark.parametrize("M", [65, 300])
def test_linear_of_few_columns_over_lhs(gpu, M):
    rng = np.random.default_rng(M)
    x, w = rounded(rng.standard_normal((M, 64))), rounded(rng.standard_normal((64, 64)) / 8)
    xd, wd, out = put(gpu, x, BF16), put(gpu, w, BF16), zeros(gpu, (M, 64), BF16)
    call(gpu, "lcu_linear", out, 0, 64, xd, wd, None, 0, BF16, M, 64, 64)
    call(gpu, "lcu_linear", xd, 0, 64, xd, wd, None, 0, BF16, M, 64, 64)
    assert np.array_equal(get(gpu, xd, (M, 64), BF16), get(gpu, out, (M, 64), BF16))
    close(get(gpu, out, (M, 64), BF16), x @ w.T, BF16)
    gpu.release()


@pytest.mark.parametrize("M,K,ff,plan", [(1030, 1024, 6560, (192, 51, 9792, 128, 128)), (1025, 1024, 6750, (192, 51, 9792, 256, 128)),
                                         (1282, 2048, 6752, (256, 42, 10752, 128, 128)), (1990, 1024, 10980, (256, 64, 16384, 256, 192))])
def test_gated_linear_columns_left_of_whole_rounds(gpu, M, K, ff, plan):
    assert gemm_plan.large("gated", M, K, 2 * up64(ff)) == plan
    test_gated_linear_large_tiles(gpu, M, K, ff)


# gated outputs of few 128x64 tiles, either side of K = 1792 where weights come from memory, and where they may not
@pytest.mark.parametrize("known", [0, 13 << 30])
@pytest.mark.parametrize("M,K,ff", [(66, 1728, 1500), (66, 1792, 1500), (129, 1856, 2000), (200, 2048, 70)])
def test_gated_linear_few_tiles(gpu, M, K, ff, known):
    assert gemm_plan.gated_tiles(M, K, 2 * up64(ff), known) == (K >= 1792 and known > 0)
    gpu.B.check(gpu.L().lcu_stream_weights(gpu.stream, known))
    try:
        test_gated_linear_large_tiles(gpu, M, K, ff)
    finally:
        gpu.B.check(gpu.L().lcu_stream_weights(gpu.stream, 0))


# gated outputs of 192 columns: one round of them, ragged ends, a short K
@pytest.mark.parametrize("M,K,ff", [(300, 1024, 10900), (500, 640, 10920), (500, 576, 10920)])
def test_gated_linear_192_columns(gpu, M, K, ff):
    assert gemm_plan.large("gated", M, K, 2 * up64(ff)) == (192, 0, 0, 0, 0)
    test_gated_linear_large_tiles(gpu, M, K, ff)


@pytest.mark.parametrize("M,K,ff", [(1100, 1216, 1850), (1100, 1280, 1850), (1441, 640, 4400), (20, 512, 13000), (6, 2816, 1020)])
def test_gated_linear_tiles_by_length(gpu, M, K, ff):
    test_gated_linear_large_tiles(gpu, M, K, ff)


@BOTH
@pytest.mark.parametrize("M,K,ff", [(1, 64, 32), (5, 128, 40), (66, 192, 100), (200, 128, 640), (700, 64, 1000), (2, 1024, 70), (40, 768, 500)])
def test_gated_linear_clamps(gpu, dt, M, K, ff):
    rng = np.random.default_rng(ff)
    x, gw, uw = rounded(2 * rng.standard_normal((M, K))), rounded(rng.standard_normal((ff, K)) / K ** 0.5), \
        rounded(rng.standard_normal((ff, K)) / K ** 0.5)
    limit, ld = 0.75, up64(ff)
    packed = pack_gated(gw, uw, ld)
    out = zeros(gpu, (M, ld), dt)
    gate = gpu.B.GateParams(limit, 1.702, 1.0)
    call(gpu, "lcu_linear_gated", out, ld, put(gpu, x, dt), put(gpu, packed, dt), C.byref(gate), dt, M, K, 2 * ld)
    want = S.expert(x, gw, uw, np.eye(ff), limit)
    assert (x @ gw.T > limit).any() and (np.abs(x @ uw.T) > limit).any()
    close(get(gpu, out, (M, ld), dt)[:, :ff], want, dt)
    gpu.release()


# ---- norms and the residual -----------------------------------------------------------------------------
@BOTH
@pytest.mark.parametrize("width,groups", [(96, 1), (100, 5), (192, 3), (512, 2), (768, 3), (1280, 5), (2048, 8), (3000, 4), (4352, 17), (12288, 2), (10000, 2000)])
@pytest.mark.parametrize("rows", [1, 3])
def test_grouped_norm_residual_and_embedding(gpu, dt, width, groups, rows):
    rng = np.random.default_rng(width + groups)
    ld, eps, vocab, n_pos, start = up64(width), 1e-3, 11, 9, 4
    ws = [1 + 0.3 * rng.standard_normal(width) for _ in range(3)]
    dw = [put(gpu, pad(w, ld)) for w in ws]
    # parts of very different size: a norm over the wrong part shows
    part = np.repeat(10.0 ** rng.integers(-2, 3, groups), width // groups)
    table, pos = rounded(part * rng.standard_normal((vocab, width))), rounded(part * rng.standard_normal((n_pos, width)))
    ids = rng.integers(0, vocab, rows)
    x, h = zeros(gpu, (rows, ld)), zeros(gpu, (rows, ld), dt)
    call(gpu, "lcu_embed_pos_norm", x, h, ints(gpu, ids), rows, put(gpu, pad(table, ld), dt), vocab, put(gpu, pad(pos, ld), dt), n_pos,
         ints(gpu, [start]), dw[0], dw[1], dt, width, ld, groups, eps)
    e = S.group_rms_norm(table[ids] + pos[start:start + rows], ws[0], groups, eps)
    close(get(gpu, x, (rows, ld))[:, :width], e, F32)
    close(get(gpu, h, (rows, ld), dt)[:, :width], S.group_rms_norm(e, ws[1], groups, eps), dt)
    # the sum of two expert rows and a gated shared one, from scattered places
    out, shared, gate = part * rng.standard_normal((2 * rows, width)), part * rng.standard_normal((rows, width)), rng.random(rows)
    inverse = rng.permutation(2 * rows)
    call(gpu, "lcu_residual_norm", x, h, put(gpu, pad(out, ld)), ints(gpu, inverse), 2, put(gpu, pad(shared, ld)), put(gpu, gate),
         dw[1], dw[2], dt, rows, width, ld, groups, eps)
    m = out[inverse].reshape(rows, 2, width).sum(1) + gate[:, None] * shared
    want = e + S.group_rms_norm(m, ws[1], groups, eps)
    got = get(gpu, x, (rows, ld))
    close(got[:, :width], want, F32)
    assert (got[:, width:] == 0).all()
    close(get(gpu, h, (rows, ld), dt)[:, :width], S.group_rms_norm(want, ws[2], groups, eps), dt)
    call(gpu, "lcu_group_norm", h, x, ints(gpu, [rows - 1]), dw[0], dt, 1, width, ld, groups, eps)
    close(get(gpu, h, (1, ld), dt)[:, :width], S.group_rms_norm(want[-1:], ws[0], groups, eps), dt)
    gpu.release()


# a row that is not finite keeps its padding: parts of whole pieces of 256 columns with padding behind them, and a width that is none
@BOTH
@pytest.mark.parametrize("width,groups,ld", [(512, 1, 640), (256, 1, 1088), (1024, 2, 1152), (768, 1, 2112), (500, 1, 640)])
@pytest.mark.parametrize("rows", [1, 3])
def test_padding_of_rows_that_are_not_finite(gpu, dt, width, groups, ld, rows):
    rng = np.random.default_rng(width)
    out = rng.standard_normal((rows, width))
    out[0, 3] = np.nan
    ones = put(gpu, pad(np.ones(width), ld))
    x, h = zeros(gpu, (rows, ld)), zeros(gpu, (rows, ld), dt)
    call(gpu, "lcu_residual_norm", x, h, put(gpu, pad(out, ld)), None, 1, None, None, ones, ones, dt, rows, width, ld, groups, 1e-5)
    for got in (get(gpu, x, (rows, ld)), get(gpu, h, (rows, ld), dt)):
        assert np.isnan(got[0, :width // groups]).all() and np.isfinite(got[1:]).all()
        assert (got[:, width:] == 0).all()
    gpu.release()


@pytest.mark.parametrize("width,groups,experts,top", [(96, 1, 5, 1), (320, 5, 12, 3), (1024, 2, 40, 2), (4352, 17, 70, 4), (9216, 9, 17, 2), (12288, 3, 512, 5), (11000, 1000, 20, 1)])
def test_one_row_step_with_router(gpu, width, groups, experts, top):
    rng = np.random.default_rng(width)
    ld, eps = up64(width), 1e-5
    x, out, gate = rng.standard_normal(width), rng.standard_normal((2, width)), np.array([0.3])
    shared = rng.standard_normal(width)
    wa, wn = 1 + 0.2 * rng.standard_normal(width), 1 + 0.2 * rng.standard_normal(width)
    router = rounded(rng.standard_normal((experts + 1, width)) / width ** 0.5)
    dx, dh = put(gpu, pad(x, ld)), zeros(gpu, ld, BF16)
    e, w, sg = ints(gpu, np.zeros(top)), zeros(gpu, top), zeros(gpu, 1)
    call(gpu, "lcu_decode_residual_router", dx, dh, put(gpu, pad(out, ld)), 2, put(gpu, pad(shared, ld)), put(gpu, gate),
         put(gpu, pad(wa, ld)), put(gpu, pad(wn, ld)), width, ld, groups, eps, put(gpu, pad(router, ld), BF16), experts, top, e, w, sg)
    want = x + S.group_rms_norm(out.sum(0) + gate * shared, wa, groups, eps)
    close(get(gpu, dx, (ld,))[:width], want, F32)
    h = get(gpu, dh, (ld,), BF16)[:width]
    close(h, S.group_rms_norm(want, wn, groups, eps), BF16)
    order, scores = S.route(router[:experts] @ h, top)
    assert list(get_ints(gpu, e, (top,))) == order
    close(get(gpu, w, (top,)), scores, F32)
    close(get(gpu, sg, (1,)), S.sigmoid(router[experts] @ h), F32)
    gpu.release()


# ---- recurrence -----------------------------------------------------------------------------------------
def block_layout(width, blocks):
    """(channel -> padded channel, padded block, row stride)."""
    cb = width // blocks
    bw = (cb + 31) // 32 * 32
    c = np.arange(width)
    return c // cb * bw + c % cb, bw, up64(blocks * bw)


@BOTH
@pytest.mark.parametrize("width,blocks,taps", [(60, 3, 2), (96, 2, 4), (70, 1, 1), (128, 4, 3), (320, 2, 6), (512, 2, 4), (384, 3, 5)])
@pytest.mark.parametrize("cuts", [(150,), (1, 2, 2, 61, 3, 64, 17), (2,) * 5 + (140,)])
def test_recurrence_in_portions(gpu, dt, width, blocks, taps, cuts):
    """Convolution, gates and state over any cut of the tokens; in bfloat16 the one-token kernels take the
    portions of one token."""
    rng = np.random.default_rng(width + taps)
    to, bw, ld = block_layout(width, blocks)
    T, cb = sum(cuts), width // blocks
    z, y = rounded(rng.standard_normal((T, width))), rounded(rng.standard_normal((T, width)))
    cw, cbias = rng.standard_normal((width, taps)) / taps ** 0.5, 0.2 * rng.standard_normal(width)
    ra, ri = (rounded(rng.standard_normal((blocks, cb, cb)) / cb ** 0.5) for _ in range(2))
    ba, bi, lam = rng.standard_normal((blocks, cb)), rng.standard_normal((blocks, cb)), -4 + 3 * rng.standard_normal(width)

    def spread(v, shape):
        out = np.zeros(shape)
        out[..., to] = v
        return out

    def square(w):
        out = np.zeros((blocks, bw, bw))
        out[:, :cb, :cb] = w
        return out

    decay = -8.0 * S.softplus(lam)
    args = dict(conv=put(gpu, spread(cw.T, (taps, ld))), convb=put(gpu, spread(cbias, ld)), wr=put(gpu, square(ra), dt),
                wi=put(gpu, square(ri), dt), br=put(gpu, spread(ba.ravel(), ld)), bi=put(gpu, spread(bi.ravel(), ld)),
                decay=put(gpu, spread(decay, ld)))
    conv_state, state = zeros(gpu, (max(taps - 1, 1), ld), dt), zeros(gpu, ld)
    channels = blocks * bw
    got_u, got_s, at = [], [], 0
    for n in cuts:
        dz, dy = put(gpu, spread(z[at:at + n], (n, ld)), dt), put(gpu, spread(y[at:at + n], (n, ld)), dt)
        u, out = zeros(gpu, (n, ld), dt), zeros(gpu, (n, ld), dt)
        call(gpu, "lcu_conv_causal", u, dz, ld, args["conv"], args["convb"], conv_state, taps, 0, dt, n, channels, ld)
        if n == 1 and dt == BF16:
            call(gpu, "lcu_decode_recurrent_step", out, u, dy, args["wr"], args["wi"], args["br"], args["bi"], args["decay"], state,
                 channels, bw)
        else:
            scratch = zeros(gpu, gpu.L().lcu_gated_recurrence_scratch(n, ld) // 4)
            call(gpu, "lcu_gated_recurrence", out, u, dy, ld, args["wr"], args["wi"], args["br"], args["bi"], args["decay"], state, scratch,
                 dt, n, channels, bw, ld)
        got_u.append(get(gpu, u, (n, ld), dt)[:, to])
        got_s.append(get(gpu, out, (n, ld), dt)[:, to])
        at += n
    u = S.causal_conv(z, cw, cbias)
    close(np.concatenate(got_u), u, dt)
    if dt == BF16:
        u = np.concatenate(got_u)   # the rest is held to the rounded inputs the kernels saw
    s = S.gated_linear_recurrence(u, S.block_gate(u, ra, ba), S.block_gate(u, ri, bi), lam)
    close(np.concatenate(got_s), s * y, dt)
    close(get(gpu, state, (ld,))[to], s[-1], F32, f32=2e-5)
    assert (get(gpu, state, (ld,))[np.setdiff1d(np.arange(channels), to)] == 0).all()
    gpu.release()


def test_recurrence_remembers_for_thousands_of_tokens(gpu):
    """A decay of almost one: an impulse at the first token is still in the state 5000 tokens later, to fp32."""
    width, T, ld = 32, 5000, 64
    lam = np.full(width, -14.0)                    # softplus ~ 8.3e-7: log a ~ -3.3e-6 per token
    u = np.zeros((T, width))
    u[0] = 1.0
    y = np.ones((T, width))
    wz = np.zeros((1, width, width))
    state = zeros(gpu, ld)
    scratch = zeros(gpu, gpu.L().lcu_gated_recurrence_scratch(T, ld) // 4)
    for dt in (BF16, F32):
        state = zeros(gpu, ld)
        out = zeros(gpu, (T, ld), dt)
        call(gpu, "lcu_gated_recurrence", out, put(gpu, pad(u, ld), dt), put(gpu, pad(y, ld), dt), ld, put(gpu, wz, dt), put(gpu, wz, dt),
             zeros(gpu, ld), zeros(gpu, ld), put(gpu, pad(-8.0 * S.softplus(lam), ld)), state, scratch, dt, T, width, width, ld)
        half = np.full((T, width), 0.5)
        want = S.gated_linear_recurrence(u, half, half, lam)
        close(get(gpu, state, (ld,))[:width], want[-1], F32, f32=1e-4)
        assert want[-1, 0] > 0.9 * want[0, 0]
    gpu.release()


# ---- attention ------------------------------------------------------------------------------------------
PADDED_V = {20: 32, 32: 32, 33: 64, 64: 64, 80: 128, 128: 128, 200: 256}


def attention_case(gpu, dt, heads, kv_heads, dim, vdim, window, keep, T, seed, far=None):
    rng = np.random.default_rng(seed)
    dk, dv = (dim + 31) // 32 * 32, PADDED_V[vdim]
    q, k, v = rng.standard_normal((T, heads, dim)), rng.standard_normal((T, kv_heads, dim)), rng.standard_normal((T, kv_heads, vdim))
    if far is not None:
        # queries `far` tokens behind a key all but copy it: one score stands out
        for i in range(far, T):
            for h in range(heads):
                q[i, h] = 3.0 * k[i - far, h // (heads // kv_heads)]
    q, k, v = rounded(q), rounded(k), rounded(v)
    scale, r1, r2 = 1.3 / dim ** 0.5, rng.random(heads), 0.05 + rng.random(heads)
    dr1, dr2 = put(gpu, r1), put(gpu, r2)
    wp = gpu.B.WindowParams(heads, kv_heads, dk, dv, window, keep, scale, dr1.ptr, dr2.ptr)
    want = S.windowed_attention(q, k, v, scale, r1, r2, window, keep)
    return dict(q=pad(q, dk), k=pad(k, dk), v=pad(v, dv), want=want, wp=wp, dk=dk, dv=dv, heads=heads, kv=kv_heads, vdim=vdim, T=T)


def run_attention(gpu, c, dt, cuts):
    heads, kv, dk, dv, T = c["heads"], c["kv"], c["dk"], c["dv"], c["T"]
    kc, vc = put(gpu, c["k"], dt), put(gpu, c["v"], dt)
    got, at = [], 0
    arrived = ints(gpu, np.zeros(kv))
    for n in cuts:
        ldq, ldo = heads * dk, heads * dv
        q, out = put(gpu, c["q"][at:at + n], dt), zeros(gpu, (n, ldo), dt)
        if n == 1 and dt == BF16:
            call(gpu, "lcu_attention_windowed_decode", out, q, kc, vc, ints(gpu, [at]), T, C.byref(c["wp"]), arrived)
        else:
            call(gpu, "lcu_attention_windowed", out, ldo, q, ldq, kc, vc, at, C.byref(c["wp"]), dt, n)
        got.append(get(gpu, out, (n, heads, dv), dt)[..., :c["vdim"]])
        at += n
    assert not get_ints(gpu, arrived, (kv,)).any()
    return np.concatenate(got)


@BOTH
@pytest.mark.parametrize("heads,kv,dim,vdim,window,keep", [
    (4, 2, 24, 20, 16, 0), (6, 1, 40, 33, 1, 3), (3, 3, 96, 64, 65, 1), (8, 2, 64, 128, 100, 70), (16, 1, 128, 128, 40, 5),
    (2, 2, 160, 200, 64, 64), (5, 5, 56, 80, 500, 2), (12, 2, 32, 32, 33, 130)])
def test_windowed_attention_in_portions(gpu, dt, heads, kv, dim, vdim, window, keep):
    T = 200
    c = attention_case(gpu, dt, heads, kv, dim, vdim, window, keep, T, heads * 100 + dim)
    whole = run_attention(gpu, c, dt, (T,))
    close(whole, c["want"], dt, bf16=2.0 ** -7)
    cut = run_attention(gpu, c, dt, (1, 1, 2, 3, 59, 64, 1, 2, 1, 37) + (1,) * 29)
    close(cut, c["want"], dt, bf16=2.0 ** -7)
    gpu.release()


# key sizes on both sides of what the tile kernel keeps registers for
@pytest.mark.parametrize("dim,vdim", [(128, 128), (129, 64), (192, 128), (193, 200), (256, 32), (64, 64), (65, 33)])
def test_windowed_attention_key_sizes(gpu, dim, vdim):
    c = attention_case(gpu, BF16, 4, 2, dim, vdim, 90, 3, 150, dim)
    close(run_attention(gpu, c, BF16, (150,)), c["want"], BF16, bf16=2.0 ** -7)
    gpu.release()


# values of 256 behind keys of up to 128, whose registers are cut to two wavefronts per SIMD, with and without a distance bias
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("dim,window,T", [(32, 90, 150), (64, 300, 193), (96, 10, 128), (128, 65, 257)])
def test_windowed_attention_of_wide_values(gpu, dim, window, T, bias):
    c = attention_case(gpu, BF16, 4, 2, dim, 200, window, 3, T, dim)
    if not bias:
        c["wp"].r1 = c["wp"].r2 = None
        c["want"] = S.windowed_attention(c["q"][..., :dim], c["k"][..., :dim], c["v"][..., :200], c["wp"].scale, np.zeros(4), np.zeros(4), window, 3)
    close(run_attention(gpu, c, BF16, (T,)), c["want"], BF16, bf16=2.0 ** -7)
    gpu.release()


# a maximum that grows from tile to tile by little (e in 100 keys), by more, by e^38, and one that falls
@pytest.mark.parametrize("growth", [0.01, 0.08, 0.6, -0.3])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (192, 128)])
def test_windowed_attention_of_growing_scores(gpu, dim, vdim, growth):
    heads, kv, T, window, keep = 3, 3, 330, 400, 0
    c = attention_case(gpu, BF16, heads, kv, dim, vdim, window, keep, T, dim)
    c["q"][..., 0] = 8.0
    c["k"][..., 0] = rounded(growth * np.arange(T) * dim ** 0.5 / 8.0 / 1.3)[:, None]  # a score grows by `growth` from key to key
    r1, r2 = (gpu.B.from_device(b, (heads,), np.float32).astype(float) for b in last_two_vectors(gpu))
    want = S.windowed_attention(c["q"][..., :dim], c["k"][..., :dim], c["v"][..., :vdim], c["wp"].scale, r1, r2, window, keep)
    close(run_attention(gpu, c, BF16, (T,)), want, BF16, bf16=2.0 ** -7)
    gpu.release()


@BOTH
@pytest.mark.parametrize("sink", [float(np.finfo(np.float32).min), -3e38, -2.4e38, -1e30])
def test_windowed_attention_of_sinks_that_are_switched_off(gpu, dt, sink):
    """A sink at the lowest float is no sink, also for rows whose window begins behind the first tile that their workgroup visits."""
    for heads, kv, dim, vdim, window, T in [(3, 3, 64, 64, 10, 128), (4, 2, 192, 128, 70, 200)]:
        c = attention_case(gpu, dt, heads, kv, dim, vdim, window, 0, T, dim)
        c["wp"].sink = put(gpu, np.full(heads, sink)).ptr
        close(run_attention(gpu, c, dt, (T,)), c["want"], dt, bf16=2.0 ** -7)
    gpu.release()


def test_windowed_attention_of_lowest_scores(gpu):
    """Scores down to -1e30, where a running maximum begins: the largest of a row takes all."""
    heads, T = 2, 130
    c = attention_case(gpu, BF16, heads, heads, 32, 32, T, 0, T, 5)
    c["wp"].scale, c["wp"].r1, c["wp"].r2 = 2.0 ** 96, None, None
    c["q"][:] = 0.0
    c["k"][:] = 0.0
    c["q"][..., 0] = 1.0
    c["k"][..., 0] = rounded(-np.random.default_rng(6).permutation(np.linspace(9.0, 12.5, T)))[:, None]  # scores of -7.1e29 to -9.9e29
    got, scores = run_attention(gpu, c, BF16, (T,)), c["k"][:, 0, 0]
    for i in range(T):
        first = np.flatnonzero(scores[:i + 1] == scores[:i + 1].max())
        assert np.allclose(got[i], c["v"][first].mean(0), rtol=2.0 ** -7, atol=0), i
    gpu.release()


# more workgroups than the chip holds at once, 768 and beyond of rows that fill their tiles and rows that do not
@pytest.mark.parametrize("heads,T", [(128, 384), (112, 390), (112, 449)])
def test_windowed_attention_many_workgroups(gpu, heads, T):
    c = attention_case(gpu, BF16, heads, 4, 120, 128, 90, 3, T, heads)
    close(run_attention(gpu, c, BF16, (T,)), c["want"], BF16, bf16=2.0 ** -7)
    gpu.release()


@BOTH
@pytest.mark.parametrize("window,keep,edge", [(48, 0, "window"), (64, 6, "window"), (65, 0, "window"), (32, 0, "window"), (20, 70, "keep")])
def test_attention_edges(gpu, dt, window, keep, edge):
    """One key stands out: just inside the window it decides the output, one token further it must not be seen;
    the same for the last kept token and the one behind it."""
    heads, kv, dim, vdim, T = 4, 2, 48, 20, 180
    for dist in (window - 1, window, window + 1):
        c = attention_case(gpu, dt, heads, kv, dim, vdim, window, keep, T, 7 + dist, far=dist)
        whole = run_attention(gpu, c, dt, (T,))
        close(whole, c["want"], dt, bf16=2.0 ** -7)
        close(run_attention(gpu, c, dt, (90,) + (1,) * 90), c["want"], dt, bf16=2.0 ** -7)
        seen = attention_case(gpu, dt, heads, kv, dim, vdim, window + 1, keep, T, 7 + dist, far=dist)["want"]
        if dist == window:   # a window one longer would have shown
            assert np.max(np.abs(seen - c["want"])) > 0.2
    if edge == "keep":
        rng = np.random.default_rng(3)
        for key in (keep - 1, keep):
            c = attention_case(gpu, dt, heads, kv, dim, vdim, window, keep, T, 5)
            c["q"][100:, :, :dim] = rounded(3.0 * np.repeat(c["k"][key, :, :dim], heads // kv, axis=0))
            r1, r2 = (gpu.B.from_device(b, (heads,), np.float32).astype(float) for b in last_two_vectors(gpu))
            c["want"] = S.windowed_attention(c["q"][..., :dim], c["k"][..., :dim], c["v"][..., :vdim], c["wp"].scale, r1, r2, window, keep)
            close(run_attention(gpu, c, dt, (60, 70) + (1,) * 50), c["want"], dt, bf16=2.0 ** -7)
            dominated = np.max(np.abs(c["want"][150, 0] - c["v"][key, 0, :vdim])) < 0.5
            assert dominated == (key < keep)
    gpu.release()


def last_two_vectors(gpu):
    """Device copies of r1 and r2 of the latest attention_case."""
    return gpu._keep[-2:]


def test_attention_far_key_over_a_long_window(gpu):
    """A key 900 tokens back among hundreds, in a prompt and token by token (several slices of keys)."""
    c = attention_case(gpu, BF16, 8, 2, 64, 64, 1000, 3, 1100, 1, far=900)
    close(run_attention(gpu, c, BF16, (1060,) + (1,) * 40), c["want"], BF16, bf16=2.0 ** -7)
    gpu.release()


@BOTH
def test_kv_rows_and_value_mixing(gpu, dt):
    rng = np.random.default_rng(0)
    n, ctx, qc, kc, vc, start = 5, 20, 32, 64, 32, 7
    ld = up64(qc + kc + vc)
    qkv = rounded(rng.standard_normal((n, ld)))
    first = rounded(rng.standard_normal((n, vc)))
    for mode, lam in ((0, 0.0), (1, 0.0), (2, 0.3)):
        kcache, vcache, vf = zeros(gpu, (ctx, kc), dt), zeros(gpu, (ctx, vc), dt), put(gpu, first, dt)
        call(gpu, "lcu_kv_store", kcache, vcache, put(gpu, qkv, dt), ld, qc, kc, vc, vf, mode, put(gpu, [lam]), ints(gpu, [start]), ctx, dt, n)
        k, v, f = get(gpu, kcache, (ctx, kc), dt), get(gpu, vcache, (ctx, vc), dt), get(gpu, vf, (n, vc), dt)
        own = qkv[:, qc + kc:qc + kc + vc]
        assert (k[start:start + n] == qkv[:, qc:qc + kc]).all() and not k[:start].any() and not k[start + n:].any()
        close(v[start:start + n], S.mix_values(own, first, lam) if mode == 2 else own, dt)
        assert (f == (own if mode == 1 else first)).all()
    gpu.release()


# ---- experts --------------------------------------------------------------------------------------------
@BOTH
@pytest.mark.parametrize("n,K,experts,top", [(1, 64, 3, 1), (5, 192, 12, 2), (70, 128, 17, 4), (33, 320, 70, 3), (40, 64, 1, 1), (18, 64, 200, 8), (20, 128, 512, 6)])
def test_router(gpu, dt, n, K, experts, top):
    rng = np.random.default_rng(K + experts)
    h, w = rounded(rng.standard_normal((n, K))), rounded(rng.standard_normal((experts + 1, K)) / K ** 0.5)
    e, wt, sg = ints(gpu, np.zeros((n, top))), zeros(gpu, (n, top)), zeros(gpu, n)
    call(gpu, "lcu_router", e, wt, sg, put(gpu, h, dt), put(gpu, w, dt), experts, top, dt, n, K)
    got, weights = get_ints(gpu, e, (n, top)), get(gpu, wt, (n, top))
    z = h @ w.T
    for t in range(n):
        order, s = S.route(z[t, :experts], top)
        assert list(got[t]) == order
        close(weights[t], s, F32)
    close(get(gpu, sg, (n,)), S.sigmoid(z[:, experts]), F32)
    gpu.release()


@BOTH
@pytest.mark.parametrize("n,K,ff,experts,top,tile", [(1, 64, 40, 3, 2, 64), (7, 128, 33, 5, 1, 64), (50, 64, 100, 4, 4, 128), (300, 128, 64, 3, 2, 256),
                                                     (150, 192, 70, 20, 2, 64)])
def test_experts(gpu, dt, n, K, ff, experts, top, tile):
    """Sorting by expert (one of them gets nothing, one gets every token), both products, and the inverse order."""
    rng = np.random.default_rng(n + ff)
    N, ld, tile = 96, up64(ff), 32 if dt == F32 else tile
    h = rounded(rng.standard_normal((n, K)))
    gate, up = (rounded(rng.standard_normal((experts, ff, K)) / K ** 0.5) for _ in range(2))
    down = rounded(rng.standard_normal((experts, N, ff)) / ff ** 0.5)
    choice = np.stack([rng.permutation(experts - 1)[:top] if experts > top else rng.permutation(experts)[:top] for _ in range(n)])
    weight = rng.random((n, top))
    rows, max_tiles = n * top, n * top // tile + experts
    plan = gpu.B.ExpertPlan()
    keep = {}
    for name, count in (("row_token", rows), ("row_weight", rows), ("inverse", rows), ("tile_expert", max_tiles), ("tile_row", max_tiles),
                        ("expert_end", experts), ("n_tiles", 1)):
        keep[name] = ints(gpu, np.zeros(count))
        setattr(plan, name, keep[name].ptr)
    plan.tile_rows, plan.max_tiles = tile, max_tiles
    call(gpu, "lcu_experts_plan", C.byref(plan), ints(gpu, choice), put(gpu, weight), n, top, experts)
    packed = np.stack([pack_gated(gate[e], up[e], ld) for e in range(experts)])
    es = 2 if dt == BF16 else 4
    hidden, out = zeros(gpu, (rows, ld), dt), zeros(gpu, (rows, N))
    g = gpu.B.GateParams(0.8, 1.702, 1.0)
    call(gpu, "lcu_experts_up", hidden, ld, put(gpu, h, dt), put(gpu, packed, dt), 2 * ld * K * es, C.byref(g), C.byref(plan), dt, n, K, 2 * ld)
    call(gpu, "lcu_experts_down", out, N, hidden, put(gpu, pad(down, ld), dt), N * ld * es, C.byref(plan), dt, rows, ld, N)
    got, inv = get(gpu, out, (rows, N)), get_ints(gpu, keep["inverse"], (n, top))
    assert sorted(inv.ravel()) == list(range(rows))
    want = np.stack([[S.expert(weight[t, k] * h[t], gate[e], up[e], down[e], 0.8) for k, e in enumerate(choice[t])] for t in range(n)])
    close(got[inv], want, dt)
    # the one-token kernels on the last token, with a shared expert of another size
    if dt == BF16:
        sff = ff + 50
        sld = up64(sff)
        sg, su, sd = (rounded(rng.standard_normal(s) / 8) for s in ((sff, K), (sff, K), (N, sff)))
        hid, shid, res = zeros(gpu, (top, ld), BF16), zeros(gpu, sld, BF16), zeros(gpu, (top + 1, N))
        ch, g2 = ints(gpu, choice[-1]), gpu.B.GateParams(0.5, 1.702, 1.0)
        call(gpu, "lcu_decode_experts_up", hid, shid, put(gpu, h[-1], BF16), ch, put(gpu, weight[-1]), put(gpu, packed, BF16),
             2 * ld * K * 2, C.byref(g), put(gpu, pack_gated(sg, su, sld), BF16), C.byref(g2), top, ld, sld, K)
        call(gpu, "lcu_decode_experts_down", res, N, hid, ch, put(gpu, pad(down, ld), BF16), N * ld * 2, top, ld, shid,
             put(gpu, pad(sd, sld), BF16), sld, N)
        got = get(gpu, res, (top + 1, N))
        close(got[:top], want[-1], BF16)
        close(got[top], S.expert(h[-1], sg, su, sd, 0.5), BF16)
    gpu.release()


@pytest.mark.parametrize("n,K,ff,experts,top,tile", [(4700, 64, 64, 3, 2, 64), (190, 64, 130, 100, 1, 64), (90, 128, 70, 65, 1, 128)])
def test_experts_lists_of_many_tiles(gpu, n, K, ff, experts, top, tile):
    """Lists of row tiles that 64 entries do not hold: runs of one expert across their edge, and many of one tile each."""
    test_experts(gpu, BF16, n, K, ff, experts, top, tile)


# one, some and many tiles to an expert, K and the hidden columns shorter and longer than the rings; few rows to a tile over a short and a long K
@pytest.mark.parametrize("n,K,ff,experts,top", [(700, 576, 500, 3, 2), (600, 64, 100, 5, 1), (50, 1024, 64, 9, 3), (60, 2112, 70, 9, 2)])
def test_experts_in_tiles_of_any_height(gpu, n, K, ff, experts, top):
    """Tiles of 64, 128 and 256 rows: the same sums in the same order, so the same bits."""
    rng = np.random.default_rng(n)
    N, ld, rows = 200, up64(ff), n * top
    h = put(gpu, rounded(rng.standard_normal((n, K))), BF16)
    gate, up = (rounded(rng.standard_normal((experts, ff, K)) / K ** 0.5) for _ in range(2))
    packed = put(gpu, np.stack([pack_gated(gate[e], up[e], ld) for e in range(experts)]), BF16)
    down = put(gpu, pad(rounded(rng.standard_normal((experts, N, ff)) / ff ** 0.5), ld), BF16)
    choice = ints(gpu, np.stack([rng.permutation(experts)[:top] for _ in range(n)]))
    weight, g = put(gpu, rng.random((n, top))), gpu.B.GateParams(0.8, 1.702, 1.0)
    got = []
    for tile, known in ((64, 0), (128, 0), (256, 0), (128, 13 << 30), (256, 13 << 30)):  # with weights from memory they are marked as read once
        gpu.B.check(gpu.L().lcu_stream_weights(gpu.stream, known))
        plan, keep, max_tiles = gpu.B.ExpertPlan(), {}, rows // tile + experts
        for name, count in (("row_token", rows), ("row_weight", rows), ("inverse", rows), ("tile_expert", max_tiles), ("tile_row", max_tiles),
                            ("expert_end", experts), ("n_tiles", 1)):
            keep[name] = ints(gpu, np.zeros(count))
            setattr(plan, name, keep[name].ptr)
        plan.tile_rows, plan.max_tiles = tile, max_tiles
        call(gpu, "lcu_experts_plan", C.byref(plan), choice, weight, n, top, experts)
        hidden, out = zeros(gpu, (rows, ld), BF16), zeros(gpu, (rows, N))
        call(gpu, "lcu_experts_up", hidden, ld, h, packed, 2 * ld * K * 2, C.byref(g), C.byref(plan), BF16, n, K, 2 * ld)
        call(gpu, "lcu_experts_down", out, N, hidden, down, N * ld * 2, C.byref(plan), BF16, rows, ld, N)
        got.append(get(gpu, out, (rows, N))[get_ints(gpu, keep["inverse"], (rows,))])
    assert np.isfinite(got[0]).all() and np.abs(got[0]).max() > 0.1
    gpu.B.check(gpu.L().lcu_stream_weights(gpu.stream, 0))
    assert all((got[0] == g).all() for g in got[1:])
    gpu.release()


@pytest.mark.parametrize("K,experts,top", [(320, 16, 2), (64, 70, 3)])
def test_router_tokens_to_a_workgroup(gpu, K, experts, top):
    """1030 tokens, sixteen to a workgroup, choose as the first 1, 3, 4, 5, 1023 and 1024 of them, four to one, to the bit."""
    rng = np.random.default_rng(K)
    h, w = put(gpu, rounded(rng.standard_normal((1030, K))), BF16), put(gpu, rounded(rng.standard_normal((experts + 1, K)) / K ** 0.5), BF16)
    results = {}
    for n in (1030, 1, 3, 4, 5, 1023, 1024):
        e, wt, sg = ints(gpu, np.full((n + 1, top), -7)), zeros(gpu, (n + 1, top)), zeros(gpu, n + 1)
        call(gpu, "lcu_router", e, wt, sg, h, w, experts, top, BF16, n, K)
        results[n] = get_ints(gpu, e, (n + 1, top)), get(gpu, wt, (n + 1, top)), get(gpu, sg, (n + 1,))
        assert (results[n][0][n] == -7).all() and not results[n][1][n].any() and results[n][2][n] == 0
        for got, want in zip(results[n], results[1030]):
            assert (got[:n] == want[:n]).all()
    gpu.release()


@pytest.mark.parametrize("n", [1, 7, 640, 32000, 50257])
def test_argmax_and_softmax(gpu, n):
    rng = np.random.default_rng(n)
    x = np.round(rng.standard_normal(n) * 4).astype(np.float32)     # ties: the first maximum counts
    idx, probs = ints(gpu, [0]), gpu.dev_keep(np.zeros(n, np.float16))
    dx = put(gpu, x)
    call(gpu, "lcu_argmax_f32", idx, dx, n)
    call(gpu, "lcu_softmax_f32", probs, dx, n, 0.7)
    gpu.B.check(gpu.L().lcu_sync(gpu.stream))
    assert get_ints(gpu, idx, (1,))[0] == x.argmax()
    p = np.exp((x.astype(float) - x.max()) / 0.7)
    assert np.max(np.abs(gpu.host(probs, (n,), np.float16) - p / p.sum())) < 1e-3
    gpu.release()


def test_unsupported_shapes_are_refused_before_any_launch(gpu):
    L, B = gpu.L(), gpu.B
    a = zeros(gpu, 4096)
    assert L.lcu_linear(a.ptr, 0, 64, a.ptr, a.ptr, None, 0, 0, 4, 40, 64, gpu.stream) == -2      # K not a multiple of 64
    assert L.lcu_linear(a.ptr, 0, 8, a.ptr, a.ptr, None, 0, 0, 4, 64, 64, gpu.stream) == -2       # rows shorter than N
    assert L.lcu_linear(a.ptr, 0, 64, a.ptr, a.ptr, None, 0, 7, 4, 64, 64, gpu.stream) == -2      # no such element type
    wp = B.WindowParams(3, 2, 64, 64, 8, 0, 1.0, a.ptr, a.ptr)                                    # 3 heads on 2
    assert L.lcu_attention_windowed(a.ptr, 192, a.ptr, 192, a.ptr, a.ptr, 0, C.byref(wp), 0, 1, gpu.stream) == -2
    assert L.lcu_router(a.ptr, a.ptr, None, a.ptr, a.ptr, 4, 5, 0, 1, 64, gpu.stream) == -2       # more choices than experts
    assert L.lcu_group_norm(a.ptr, a.ptr, None, a.ptr, 0, 1, 100, 128, 3, 1e-5, gpu.stream) == -2  # 100 in 3 parts
    assert L.lcu_gated_recurrence(*([a.ptr] * 3), 64, *([a.ptr] * 7), 0, 1, 64, 20, 64, gpu.stream) == -2  # block width
    gpu.release()
