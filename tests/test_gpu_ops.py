"""GPU parity of every kernel behind the C ABI against the CPU oracle, on the same seeded inputs.

Bars: bit-exact for the quantiser's codes and scales, for dequantisation, embedding, RoPE and the
argmax; max-abs-rel <= 1e-2 for every fp16 output that accumulates in fp32 (matmul, attention,
softmax, norm, silu)."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

TOL = 1e-2  # max-abs-rel bar for fp16 outputs with fp32 accumulation


@pytest.fixture(scope="module", autouse=True)
def gpu():
    import gpu_helpers as G
    G.setup()
    yield G
    G.release()


def normal(shape, seed, stream, std):
    n = int(np.prod(shape))
    return O.fill_normal_f16(n, seed, stream, std).reshape(shape)


def test_fill_normal_matches_oracle_bits(gpu):
    G = gpu
    for n, seed, stream, std in [(1000, 0, 1, 0.02), (1 << 20, 7, 33, 1.0), (12345, 2 ** 40 + 3, 2 ** 33, 0.5)]:
        buf = G.empty((n,))
        G.B.check(G.L().lcu_fill_normal_f16(buf.ptr, n, seed, stream, std, None))
        got = G.host(buf, (n,))
        assert (got.view(np.uint16) == O.fill_normal_f16(n, seed, stream, std).view(np.uint16)).all()


@pytest.mark.parametrize("rows,cols,block", [(64, 1024, 128), (7, 512, 32), (5, 2048, 1024), (33, 768, 256)])
def test_quantize_bit_exact(gpu, rows, cols, block):
    G = gpu
    w = normal((rows, cols), 3, 5, 0.02)
    w[0, :block] = 0  # an all-zero block
    w[1, 3] = np.float16(65504.0)
    w[2, :block] = np.float16(6e-8)  # scale underflows to zero
    codes_d, scales_d = G.empty((rows, cols), np.uint8), G.empty((rows, cols // block))
    wd = G.dev(w)
    G.B.check(G.L().lcu_quantize_absmax_u8(codes_d.ptr, scales_d.ptr, wd.ptr, rows, cols, block, None))
    codes, scales = G.host(codes_d, (rows, cols), np.uint8), G.host(scales_d, (rows, cols // block))
    ec, es = O.quantize_absmax_u8(w, block)
    assert (scales.view(np.uint16) == es.view(np.uint16)).all()
    assert (codes == ec).all()
    out_d = G.empty((rows, cols))
    G.B.check(G.L().lcu_dequantize_absmax_u8(out_d.ptr, scales_d.ptr, codes_d.ptr, rows, cols, block, None))
    assert (G.host(out_d, (rows, cols)).view(np.uint16) == O.dequantize_absmax_u8(ec, es, block).view(np.uint16)).all()


# one to sixty-four lanes a block, block sizes and places that take the general kernel, counts that end inside a workgroup
@pytest.mark.parametrize("rows,cols,block,shift", [(3, 8, 8, 0), (67, 112, 16, 0), (5, 96, 32, 0), (129, 64, 64, 0), (41, 256, 128, 0),
                                                   (9, 512, 256, 0), (3, 1536, 512, 0), (5, 72, 24, 0), (4, 100, 20, 0), (37, 256, 128, 1)])
def test_quantize_block_sizes_and_places(gpu, rows, cols, block, shift):
    G = gpu
    w = normal((rows, cols), 3, 6, 0.02)
    w[0, :block] = np.float16(np.inf)
    w[-1, -1] = np.float16(np.nan)
    w[1, :block] *= np.float16(2.0 ** -9)     # subnormal scale
    w[2, :block] = 0
    wd = G.dev_keep(np.concatenate([np.zeros(shift, np.float16), w.reshape(-1)]))
    codes_d, scales_d = G.empty((rows, cols), np.uint8), G.empty((rows, cols // block))
    G.B.check(G.L().lcu_quantize_absmax_u8(codes_d.ptr, scales_d.ptr, wd.ptr + 2 * shift, rows, cols, block, None))
    ec, es = O.quantize_absmax_u8(w, block)
    assert (G.host(scales_d, (rows, cols // block)).view(np.uint16) == es.view(np.uint16)).all()
    assert (G.host(codes_d, (rows, cols), np.uint8) == ec).all()
    G.release()


@pytest.mark.parametrize("rows,cols", [(4096, 4096), (11008, 4096), (4096, 11008)])
def test_quantize_bit_exact_at_llama7b_shapes(gpu, rows, cols):
    """the weight matrices of the int8 benchmark configuration, W ~ N(0, 0.02), block 128: every code and scale"""
    G = gpu
    x = normal((rows, cols), 0, 310, 0.02)
    codes_d, scales_d = G.empty((rows, cols), np.uint8), G.empty((rows, cols // 128))
    G.B.check(G.L().lcu_quantize_absmax_u8(codes_d.ptr, scales_d.ptr, G.dev_keep(x).ptr, rows, cols, 128, None))
    ec, es = O.quantize_absmax_u8(x, 128)
    assert (G.host(codes_d, (rows, cols), np.uint8) == ec).all()
    assert (G.host(scales_d, (rows, cols // 128)).view(np.uint16) == es.view(np.uint16)).all()
    back_d = G.empty((rows, cols))
    G.B.check(G.L().lcu_dequantize_absmax_u8(back_d.ptr, scales_d.ptr, codes_d.ptr, rows, cols, 128, None))
    assert (G.host(back_d, (rows, cols)).view(np.uint16) == O.dequantize_absmax_u8(ec, es, 128).view(np.uint16)).all()
    G.release()


def test_quantize_exhaustive_inputs_bit_exact(gpu):
    G = gpu
    allbits = np.arange(65536, dtype=np.uint16).view(np.float16)
    finite = allbits[np.isfinite(allbits)]
    for absmax in [np.float16(65504.0), np.float16(1.0), np.float16(0.0604), np.float16(3e-4)]:
        xs = finite[np.abs(finite) <= absmax]
        n = (len(xs) + 126) // 127
        blocks = np.zeros((n, 128), dtype=np.float16)
        blocks[:, 0] = absmax
        flat = np.zeros(n * 127, dtype=np.float16)
        flat[: len(xs)] = xs
        blocks[:, 1:] = flat.reshape(n, 127)
        codes_d, scales_d = G.empty((n, 128), np.uint8), G.empty((n, 1))
        G.B.check(G.L().lcu_quantize_absmax_u8(codes_d.ptr, scales_d.ptr, G.dev_keep(blocks).ptr, n, 128, 128, None))
        ec, es = O.quantize_absmax_u8(blocks, 128)
        assert (G.host(codes_d, (n, 128), np.uint8) == ec).all()
        assert (G.host(scales_d, (n, 1)).view(np.uint16) == es.view(np.uint16)).all()


def test_dequantize_all_codes_all_scales_bit_exact(gpu):
    G = gpu
    # every code against a sweep of scales including subnormal ones
    scales = np.concatenate([np.arange(0, 0x0500, 7, dtype=np.uint16), np.arange(0x0500, 0x5C00, 97, dtype=np.uint16)])
    scales = scales.view(np.float16).reshape(-1, 1)
    n = len(scales)
    codes = np.tile(np.arange(256, dtype=np.uint8), (n, 1))
    out_d = G.empty((n, 256))
    G.B.check(G.L().lcu_dequantize_absmax_u8(out_d.ptr, G.dev_keep(scales).ptr, G.dev_keep(codes).ptr, n, 256, 256, None))
    assert (G.host(out_d, (n, 256)).view(np.uint16) == O.dequantize_absmax_u8(codes, scales, 256).view(np.uint16)).all()


GEMV_SHAPES = [(4096, 11008), (4096, 4096), (11008, 4096), (256, 40), (1032, 77), (6656, 6656)]


@pytest.mark.parametrize("K,N", GEMV_SHAPES)
def test_gemv_f16(gpu, K, N):
    G = gpu
    x = normal((1, K), 0, 100, 1.0)
    w = normal((N, K), 0, 101, 0.02)
    got = G.gemm_f16(x, w)
    ref = O.matmul_nt(x, w)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.05  # same fp16 value except where fp32 summation order flips a rounding
    # against the oracle's restatement of this kernel's own summation order: every bit
    assert G.ulp_mismatch(got, O.matmul_nt(x, w, flavour=2)) == 0.0
    old = normal((1, N), 0, 102, 1.0)
    got = G.gemm_f16(x, w, beta=1.0, out=old)
    assert G.max_abs_rel(got, O.matmul_nt(x, w, beta=1.0, out=old)) <= TOL
    assert G.ulp_mismatch(got, O.matmul_nt(x, w, beta=1.0, out=old, flavour=2)) == 0.0
    G.release()


def test_gemv_exact_cases(gpu):
    G = gpu
    K = 512
    x = normal((1, K), 1, 1, 1.0)
    assert (G.gemm_f16(x, np.eye(K, dtype=np.float16)).view(np.uint16) == x.view(np.uint16)).all()
    w = normal((300, K), 1, 2, 0.02)
    onehot = np.zeros((1, K), dtype=np.float16)
    onehot[0, 129] = 1
    assert (G.gemm_f16(onehot, w)[0].view(np.uint16) == w[:, 129].view(np.uint16)).all()
    G.release()


# rows of one to six batches of the workgroup (4096 codes each): two to five are requested at once, one
# and six go through the loop; two and four rows per workgroup (N below / from 6144)
@pytest.mark.parametrize("K,N", [(4096, 4096), (4096, 11008), (11008, 4096), (256, 40), (1024 + 128, 77), (6656, 17920),
                                 (17920, 300), (13824, 100), (22016, 64), (8192, 6200), (17920, 6152)])
def test_gemv_u8(gpu, K, N):
    G = gpu
    x = normal((1, K), 0, 200, 1.0)
    w = normal((N, K), 0, 201, 0.02)
    codes, scales = O.quantize_absmax_u8(w, 128)
    got = G.gemm_u8(x, codes, scales, 128)
    ref = O.matmul_nt_u8(x, codes, scales, 128)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.05
    # the kernel-order flavour restates the kernel's sums down to the alignment inside
    # v_dot2_f32_f16: every output bit for bit
    assert G.ulp_mismatch(got, O.matmul_nt_u8(x, codes, scales, 128, flavour=2)) == 0.0
    old = normal((1, N), 0, 202, 1.0)
    got = G.gemm_u8(x, codes, scales, 128, beta=1.0, out=old)
    assert G.max_abs_rel(got, O.matmul_nt_u8(x, codes, scales, 128, beta=1.0, out=old)) <= TOL
    assert G.ulp_mismatch(got, O.matmul_nt_u8(x, codes, scales, 128, beta=1.0, out=old, flavour=2)) == 0.0
    G.release()


def test_gemv_u8_dequant_is_exact(gpu):
    # one-hot x picks single dequantised weights: they must be the reference's fp16 values exactly
    G = gpu
    K, N = 256, 64
    w = normal((N, K), 4, 1, 0.02)
    w[:, 128:] *= np.float16(1e-3)  # small scales, some products subnormal in fp16
    codes, scales = O.quantize_absmax_u8(w, 128)
    deq = O.dequantize_absmax_u8(codes, scales, 128)
    for k in (0, 5, 127, 128, 200, 255):
        x = np.zeros((1, K), dtype=np.float16)
        x[0, k] = 1
        got = G.gemm_u8(x, codes, scales, 128)[0]
        assert (got.view(np.uint16) == deq[:, k].view(np.uint16)).all(), k
    G.release()


# the shapes cover every tile configuration of the dispatcher: 128x64 with two wavefront groups,
# 256x128, 128x128 with eight wavefronts (160..255 tiles: N = 5120), 128x64 with two workgroups per
# compute unit (N = 4160), 128x128 with four wavefronts (M = 1024, N = 4096), ragged K / M / N, and
# grids with more tiles than the chip holds workgroups at once ((4096, 128, 4096) .. (2100, 128, 8200)); the
# last five are short prompts (2..64 rows), which split K over several workgroups per tile: 32- and 64-row
# tiles, uneven splits (11008 / 64 = 172 stages over 16 workgroups), ragged M and N
@pytest.mark.parametrize("M,K,N", [(512, 4096, 4096), (512, 4096, 11008), (512, 11008, 4096), (128, 256, 128),
                                   (7, 64, 24), (130, 200, 70), (33, 1024, 257), (512, 256, 5120), (512, 384, 4160),
                                   (1024, 256, 4096), (500, 128, 5100), (4096, 128, 4096), (512, 256, 17920), (2100, 128, 8200),
                                   (2, 4096, 4096), (17, 1024, 5000), (32, 11008, 4096), (33, 1024, 4100), (64, 4096, 11008)])
def test_gemm_f16(gpu, M, K, N):
    G = gpu
    x = normal((M, K), 0, 300, 1.0)
    w = normal((N, K), 0, 301, 0.02)
    got = G.gemm_f16(x, w)
    ref = O.matmul_nt(x, w)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.05
    # the kernel-order flavour restates the matrix cores' sums and the dispatcher's cut of K: bit for bit
    assert G.ulp_mismatch(got, O.matmul_nt(x, w, flavour=2)) == 0.0, O.gemm_plan(M, K, N)
    old = normal((M, N), 0, 302, 1.0)
    got = G.gemm_f16(x, w, beta=1.0, out=old)
    assert G.max_abs_rel(got, O.matmul_nt(x, w, beta=1.0, out=old)) <= TOL
    assert G.ulp_mismatch(got, O.matmul_nt(x, w, beta=1.0, out=old, flavour=2)) == 0.0
    G.release()


# tiles of 256 rows at their edges: 192 columns with rows of 4 halves past a 16-byte boundary, 256 columns, 128 columns of one
# row and column beyond a tile, and K split over workgroups with rows of 2 floats past one; a single K stage pair and many
@pytest.mark.parametrize("M,K,N", [(2049, 128, 4100), (4096, 256, 4090), (257, 384, 12929), (300, 5120, 1030),
                                   (65, 128, 20500), (127, 256, 35000), (100, 5120, 1030),  # and of 128 rows: 128 and 256 columns, K split
                                   (257, 128, 6790), (1100, 384, 3690)])  # with more rows: 160 tiles, 261
def test_gemm_f16_large_tiles_ragged(gpu, M, K, N):
    G = gpu
    x, w, old = normal((M, K), 0, 320, 1.0), normal((N, K), 0, 321, 0.02), normal((M, N), 0, 322, 1.0)
    assert G.ulp_mismatch(G.gemm_f16(x, w), O.matmul_nt(x, w, flavour=2)) == 0.0, O.gemm_plan(M, K, N)
    got = G.gemm_f16(x, w, beta=1.0, out=old)
    assert G.ulp_mismatch(got, O.matmul_nt(x, w, beta=1.0, out=old, flavour=2)) == 0.0
    G.release()


# both sides of the lengths of K that decide between the kernels: fp16 with 160 .. 255 tiles of 128x128 and more, 128 or 256 columns
# of large tiles; the cases above whose K is short, with a long one
@pytest.mark.parametrize("M,K,N,count", [(257, 1152, 6790, 1), (257, 1280, 6790, 1), (1100, 1152, 3690, 1), (1100, 1408, 3690, 1), (1100, 1536, 3690, 1),
                                         (1441, 512, 2900, 3), (1441, 640, 2900, 3), (2049, 640, 4100, 1), (300, 640, 12930, 1)])
def test_gemm_f16_short_and_long_k(gpu, M, K, N, count):
    G = gpu
    VP = G.B.vp
    x, ws = normal((M, K), 0, 330, 1.0), [normal((N, K), 0, 331 + g, 0.02) for g in range(count)]
    wd, outs = [G.dev_keep(w) for w in ws], [G.empty((M, N)) for _ in ws]
    G.B.check(G.L().lcu_gemm_f16_nt_multi((VP * count)(*[o.ptr for o in outs]), G.dev_keep(x).ptr, (VP * count)(*[w.ptr for w in wd]), count,
                                          M, K, N, 0.0, None))
    for o, w in zip(outs, ws):
        assert G.ulp_mismatch(G.host(o, (M, N)), O.matmul_nt_kernel_order(x, w, n_mats=count)) == 0.0, O.gemm_plan(M, K, N)
    G.release()


# the same for codes: 160 .. 255 tiles of 128x128, more, one round of large tiles and several
@pytest.mark.parametrize("M,K,N,block", [(257, 256, 6790, 128), (257, 384, 6790, 64), (1100, 1408, 3690, 128), (1100, 1536, 3690, 128),
                                         (1030, 512, 4100, 128), (1030, 640, 4100, 128), (2049, 384, 4100, 64), (2049, 512, 4100, 256)])
def test_gemm_u8_short_and_long_k(gpu, M, K, N, block):
    G = gpu
    x, w = normal((M, K), 0, 340, 1.0), normal((N, K), 0, 341, 0.02)
    codes, scales = O.quantize_absmax_u8(w, block)
    got = G.gemm_u8(x, codes, scales, block)
    assert G.ulp_mismatch(got, O.matmul_nt_u8(x, codes, scales, block, flavour=2)) == 0.0, O.gemm_plan(M, K, N, True)
    G.release()


def test_gemm_residual_into_an_output_that_is_not_16_byte_aligned(gpu):
    """beta = 1 with the output tile 8 bytes off a 16-byte boundary: the tile that fetches its old values in 16-byte
    pieces (512 x 4096 x 4096, the Wo product) must fall back to 2-byte reads; same bits as the aligned call."""
    G = gpu
    M, K, N = 512, 4096, 4096
    x = normal((M, K), 0, 310, 1.0)
    w = normal((N, K), 0, 311, 0.02)
    old = normal((M, N), 0, 312, 1.0)
    want = G.gemm_f16(x, w, beta=1.0, out=old)
    buf = G.empty((M * N + 8,))
    for shift in (4, 1):  # halves: 8 bytes and 2 bytes off
        padded = np.zeros(M * N + 8, dtype=np.float16)
        padded[shift:shift + M * N] = old.reshape(-1)
        G.B.check(G.L().lcu_h2d(buf.ptr, padded.ctypes.data, padded.nbytes, None))
        G.B.check(G.L().lcu_gemm_f16_nt(buf.ptr + 2 * shift, G.dev_keep(x).ptr, G.dev_keep(w).ptr, M, K, N, 1.0, None))
        got = G.host(buf, (M * N + 8,))[shift:shift + M * N].reshape(M, N)
        assert (got.view(np.uint16) == want.view(np.uint16)).all(), shift
    buf.free()
    G.release()


def test_gemm_exact_cases(gpu):
    G = gpu
    K = 256
    x = normal((40, K), 2, 1, 1.0)
    assert (G.gemm_f16(x, np.eye(K, dtype=np.float16)).view(np.uint16) == x.view(np.uint16)).all()
    # asymmetric operands: out[m, n] pairs lhs row m with rhs row n
    w = np.zeros((96, K), dtype=np.float16)
    w[70, 5] = 2
    x2 = np.zeros((40, K), dtype=np.float16)
    x2[33, 5] = 3
    out = G.gemm_f16(x2, w)
    assert out[33, 70] == 6 and np.count_nonzero(out) == 1
    G.release()


# Whole rounds of large tiles (of 128, 192 and 256 columns) and the columns behind them in smaller ones: 128x128, 128 and 192 columns of 256
# rows, ragged ones, one to three matrices; and one width alone.  Every output against the same rows in other calls, whose tiles are others and
# whose sums are one ascending chain too, and samples on both sides of every edge against that chain worked out by itself.
@pytest.mark.parametrize("u8,M,K,N,count,plan", [
    (False, 775, 1024, 12308, 1, (128, 64, 8192, 128, 128)), (False, 266, 1024, 12558, 3, (128, 256, 7424, 128, 128)),
    (False, 1034, 1152, 13072, 1, (192, 51, 9792, 128, 128)), (False, 514, 1024, 11432, 2, (192, 85, 4800, 256, 128)),
    (False, 700, 1024, 11003, 2, (192, 85, 5184, 256, 128)), (False, 1286, 1152, 13464, 1, (256, 42, 10752, 128, 128)),
    (False, 264, 1152, 12248, 3, (256, 128, 8192, 128, 128)), (False, 775, 1152, 12811, 2, (256, 64, 3328, 256, 192)),
    (False, 512, 2048, 11008, 2, (192, 0, 0, 0, 0)), (True, 770, 1152, 12507, 1, (128, 64, 8192, 128, 128)),
    (True, 1030, 1152, 13178, 1, (192, 51, 9792, 128, 128)), (True, 260, 1024, 10982, 3, (192, 128, 2304, 128, 128)),
    (True, 512, 1024, 17924, 2, (192, 128, 6528, 256, 128)), (True, 521, 1024, 13598, 2, (256, 85, 7936, 128, 128)),
    (True, 770, 1024, 12544, 3, (256, 128, 7680, 256, 128)), (True, 1987, 1024, 11008, 2, (256, 64, 5376, 256, 192)),
    (True, 384, 1024, 6656, 3, (192, 0, 0, 0, 0)), (False, 263, 256, 16437, 1, (192, 0, 0, 0, 0)), (False, 524, 2048, 17471, 1, (256, 0, 0, 0, 0)),
    (True, 513, 640, 16530, 1, (256, 0, 0, 0, 0))])
def test_gemm_columns_left_of_whole_rounds(gpu, u8, M, K, N, count, plan):
    import gemm_plan
    G = gpu
    VP, check, L = G.B.vp, G.B.check, G.L()
    kind = "u8" if u8 else "f16"
    assert gemm_plan.rows(M, K, N, count)[0] == "large" and gemm_plan.large(kind, M, K, N, count) == plan
    x, ws = normal((M, K), 0, 350, 1.0), [normal((N, K), 0, 351 + g, 0.02) for g in range(count)]
    w = [O.quantize_absmax_u8(v, 128) for v in ws] if u8 else [(v,) for v in ws]
    wd = [[G.dev_keep(part) for part in v] for v in w]
    ptrs = [(VP * count)(*[v[i].ptr for v in wd]) for i in range(len(w[0]))]
    if u8:
        ws = [O.dequantize_absmax_u8(*v, 128) for v in w]

    def product(rows, beta, old):
        outs = [G.dev_keep(o) for o in old]
        args = ((VP * count)(*[o.ptr for o in outs]), G.dev_keep(rows).ptr, *ptrs, count, len(rows), K, N)
        check(L.lcu_gemm_f16u8_nt_multi(*args, 128, beta, None) if u8 else L.lcu_gemm_f16_nt_multi(*args, beta, None))
        return [G.host(o, (len(rows), N)) for o in outs]

    step = 256 if M >= 512 else 128
    at = list(range(0, M - step + 1, step)) + [M]
    for a, b in zip(at, at[1:]):
        assert O.gemm_plan(b - a, K, N, u8, 128, count) == (1, 1)
        assert gemm_plan.rows(b - a, K, N, count)[0] != "large" or gemm_plan.large(kind, b - a, K, N, count) != plan
    rng = np.random.default_rng(M)
    edges = {e + d for e in (0, plan[0], plan[2], plan[2] + plan[4], 2 * plan[0], N) for d in (-2, -1, 0, 1, 127, 128)}
    columns = sorted({c for c in edges if 0 <= c < N} | set(map(int, rng.integers(0, N, 40))))
    rows = sorted({0, 127, 128, 255, 256, M - 1} | set(map(int, rng.integers(0, M, 8))))
    r, c = (v.ravel() for v in np.meshgrid(rows, columns, indexing="ij"))
    old = [normal((M, N), 0, 360 + g, 1.0) for g in range(count)]
    for beta in (0.0, 1.0):
        got = product(x, beta, old)
        for a, b in zip(at, at[1:]):
            for g, part in zip(got, product(x[a:b], beta, [o[a:b] for o in old])):
                assert G.ulp_mismatch(g[a:b], part) == 0.0, (a, b)
        for g, m, o in zip(got, ws, old):
            chain = O.mfma_f32_f16(x[r].view(np.uint16), m[c].view(np.uint16), np.zeros(len(r), np.float32))
            assert (g[r, c] == (chain + np.float32(beta) * o[r, c].astype(np.float32)).astype(np.float16)).all()
    G.release()


@pytest.mark.parametrize("M,K,N", [(512, 4096, 4096), (512, 4096, 11008), (512, 11008, 4096), (16, 256, 128),
                                   (130, 384, 70), (512, 256, 5120), (512, 384, 4160), (1024, 256, 4096),
                                   (500, 128, 5100), (40, 384, 300), (4096, 128, 4096), (512, 256, 17920),
                                   (5, 4096, 4096), (17, 1024, 5000), (32, 11008, 4096), (64, 1024, 4100), (512, 17920, 6656)])
def test_gemm_u8(gpu, M, K, N):
    G = gpu
    x = normal((M, K), 0, 400, 1.0)
    w = normal((N, K), 0, 401, 0.02)
    codes, scales = O.quantize_absmax_u8(w, 128)
    got = G.gemm_u8(x, codes, scales, 128)
    ref = O.matmul_nt_u8(x, codes, scales, 128)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.05
    assert G.ulp_mismatch(got, O.matmul_nt_u8(x, codes, scales, 128, flavour=2)) == 0.0, O.gemm_plan(M, K, N, True)
    # row r of the M-row product equals the single-row product (decode path) within tolerance
    one = G.gemm_u8(x[3:4], codes, scales, 128)
    assert G.max_abs_rel(one, got[3:4]) <= TOL
    G.release()


# few rows, codes: runs of K stages that begin in the middle of 128 codes, one to four row tiles, lhs in one piece and in
# chunks, one and two scales in 128 codes, and a block that takes the other kernel
@pytest.mark.parametrize("M,K,N,block", [(2, 1152, 520, 64), (16, 1152, 4100, 128), (17, 2560, 1000, 256), (33, 1152, 5000, 64),
                                         (64, 5888, 4100, 128), (64, 1152, 3000, 384), (7, 17920, 6656, 128),
                                         (16, 512, 32000, 128), (17, 512, 32000, 64), (20, 2560, 31010, 128)])  # two rounds of workgroups
def test_gemm_u8_few_rows(gpu, M, K, N, block):
    G = gpu
    x, w = normal((M, K), 0, 430, 1.0), normal((N, K), 0, 431, 0.02)
    codes, scales = O.quantize_absmax_u8(w, block)
    got = G.gemm_u8(x, codes, scales, block)
    assert G.ulp_mismatch(got, O.matmul_nt_u8(x, codes, scales, block, flavour=2)) == 0.0, O.gemm_plan(M, K, N, True)
    G.release()


# few rows, fp16: odd runs, rows past the last whole tile, columns past the last whole wavefront, lhs in chunks
@pytest.mark.parametrize("M,K,N", [(3, 1152, 520), (16, 1408, 4099), (31, 2944, 1000), (48, 5888, 4100), (64, 4096, 24000),
                                   (16, 5760, 4099), (31, 5760, 4099), (24, 4096, 4096), (28, 512, 16840),  # 264, 264, 256 and 264 tiles
                                   (8, 512, 32000), (40, 640, 31000),  # two rounds of workgroups: the other kernel
                                   (20, 2560, 31010), (24, 6144, 4099)])  # two rounds of long runs, one of them: weights from memory decide
def test_gemm_f16_few_rows(gpu, M, K, N):
    G = gpu
    x, w, old = normal((M, K), 0, 440, 1.0), normal((N, K), 0, 441, 0.02), normal((M, N), 0, 442, 1.0)
    assert G.ulp_mismatch(G.gemm_f16(x, w), O.matmul_nt(x, w, flavour=2)) == 0.0, O.gemm_plan(M, K, N)
    assert G.ulp_mismatch(G.gemm_f16(x, w, beta=1.0, out=old), O.matmul_nt(x, w, beta=1.0, out=old, flavour=2)) == 0.0
    G.release()


MODEL = 13 << 30  # bytes of weights between two uses of the same ones


@pytest.fixture
def model_stream(gpu):
    """A stream whose weights come from memory."""
    stream = gpu.B.vp()
    gpu.B.check(gpu.L().lcu_stream_create(C.byref(stream)))
    gpu.B.check(gpu.L().lcu_stream_weights(stream, MODEL))
    yield stream
    gpu.B.check(gpu.L().lcu_stream_destroy(stream))


# weights marked as read once, on a model's stream, against the oracle and against a stream that says nothing: one to four row tiles with a ragged last one, columns
# past the last whole sixteen, sums that are added up where they end and sums that are not, two rounds of workgroups
@pytest.mark.parametrize("kind,M,K,N,mats", [("f16", 3, 4096, 8300, 1), ("f16", 16, 5760, 6001, 1), ("f16", 24, 6144, 5500, 1), ("f16", 31, 2944, 11500, 1),
                                             ("f16", 40, 8192, 4101, 1), ("f16", 63, 4096, 8300, 1), ("f16", 20, 2560, 31010, 1), ("f16", 7, 4096, 2902, 3),
                                             ("f16", 45, 4096, 4104, 2), ("u8", 5, 6656, 10102, 1), ("u8", 20, 6656, 10102, 1), ("u8", 33, 6656, 10102, 1),
                                             ("u8", 60, 17920, 4006, 1), ("u8", 64, 5888, 11502, 1), ("u8", 9, 4096, 5502, 3), ("u8", 48, 6656, 5102, 2),
                                             ("u8", 17, 2560, 31010, 1)])
def test_few_rows_of_weights_from_memory(gpu, model_stream, kind, M, K, N, mats):
    import gemm_plan
    G = gpu
    check, L, VP = G.B.check, G.L(), G.B.vp
    assert gemm_plan.few_rows(kind, M, K, N, mats, known=MODEL)[1:] == (True, True) and not gemm_plan.few_rows(kind, M, K, N, mats)[2]
    x, ws = normal((M, K), 0, 460, 1.0), [normal((N, K), 0, 461 + g, 0.02) for g in range(mats)]
    codes = [O.quantize_absmax_u8(w, 128) for w in ws] if kind == "u8" else []
    xd, wd = G.dev_keep(x), [G.dev_keep(c[0]) for c in codes] or [G.dev_keep(w) for w in ws]
    sd, results = [G.dev_keep(c[1]) for c in codes], []
    for stream in (model_stream, None):
        outs = [G.empty((M, N)) for _ in range(mats)]
        arr = lambda items: (VP * mats)(*[i.ptr for i in items])
        if codes:
            check(L.lcu_gemm_f16u8_nt_multi(arr(outs), xd.ptr, arr(wd), arr(sd), mats, M, K, N, 128, 0.0, stream))
        else:
            check(L.lcu_gemm_f16_nt_multi(arr(outs), xd.ptr, arr(wd), mats, M, K, N, 0.0, stream))
        check(L.lcu_sync(stream))
        results.append([G.host(o, (M, N)) for o in outs])
        for o in outs:
            o.free()
    for g in range(mats):
        want = O.matmul_nt_kernel_order(x, codes=codes[g][0], scales=codes[g][1], block=128, n_mats=mats) if codes else \
            O.matmul_nt_kernel_order(x, ws[g], n_mats=mats)
        assert G.ulp_mismatch(results[0][g], want) == 0.0
        assert (results[0][g].view(np.uint16) == results[1][g].view(np.uint16)).all()
    G.release()


@pytest.mark.parametrize("B,u8", [(2, False), (9, False), (20, False), (50, False), (9, True), (40, True)])
def test_batch_steps_of_weights_from_memory(gpu, model_stream, B, u8):
    """The fused steps of a batch, their weights marked as read once, against the same on a stream that says nothing, bit for bit."""
    G = gpu
    check, L, VP = G.B.check, G.L(), G.B.vp
    dim, heads, ffn, ctx, block = (4992, 39, 13568, 8, 128) if u8 else (4096, 32, 8320, 8, 0)
    table = VP()
    check(L.lcu_rope_table_create(G.B.C.byref(table), ctx, dim // heads, 10000.0))

    def weights(rows, cols, stream):
        w = normal((rows, cols), 0, stream, 0.02)
        return [G.dev_keep(a) for a in (O.quantize_absmax_u8(w, block) if u8 else (w,))]

    qkv, up, w2 = [weights(dim, dim, 470 + g) for g in range(3)], [weights(ffn, dim, 480 + g) for g in range(2)], weights(dim, ffn, 490)
    arr = lambda items, at=0: (VP * len(items))(*[i[at].ptr for i in items])
    x, h, nw = normal((B, dim), 0, 491, 1.0), G.dev_keep(normal((B, ffn), 0, 492, 0.5)), G.dev_keep(normal((dim,), 0, 493, 1.0))
    xd, pos, results = G.dev_keep(x), G.dev_keep(np.arange(B, dtype=np.int32) % ctx), []
    for stream in (model_stream, None):
        kc, vc = [G.dev_keep(np.zeros((ctx, dim), np.float16)) for _ in range(B)], [G.dev_keep(np.zeros((ctx, dim), np.float16)) for _ in range(B)]
        kp, vp = (G.dev_keep(np.array([c.ptr for c in cs], dtype=np.uint64)) for cs in (kc, vc))
        q, k, v, t1, t3, act, norm, res = [G.dev_keep(np.zeros((B, n), np.float16)) for n in (dim, dim, dim, ffn, ffn, ffn, dim)] + [G.dev_keep(x)]
        check(L.lcu_batch_qkv(q.ptr, k.ptr, v.ptr, xd.ptr, arr(qkv), arr(qkv, 1) if u8 else None, block, B, dim, heads, kp.ptr, vp.ptr, pos.ptr, table, ctx, stream))
        check(L.lcu_batch_ffn_up(act.ptr, t1.ptr, t3.ptr, xd.ptr, arr(up), arr(up, 1) if u8 else None, block, B, dim, ffn, stream))
        check(L.lcu_batch_proj_norm(res.ptr, norm.ptr, h.ptr, w2[0].ptr, w2[1].ptr if u8 else None, block, B, ffn, dim, nw.ptr, 1e-6, stream))
        check(L.lcu_sync(stream))
        results.append([G.host(q, (B, dim)), G.host(act, (B, ffn)), G.host(res, (B, dim)), G.host(norm, (B, dim))] + [G.host(c, (ctx, dim)) for c in kc + vc])
    for a, b in zip(*results):
        assert (a.view(np.uint16) == b.view(np.uint16)).all() and np.abs(a.astype(np.float32)).max() > 0
    G.release()
    L.lcu_free(table)


def test_only_streams_of_the_library_take_a_size_of_weights(gpu, model_stream):
    L = gpu.L()
    assert L.lcu_stream_weights(None, 1) != 0 and b"lcu_stream_weights" in L.lcu_last_error()
    assert L.lcu_stream_weights(model_stream, 0) == 0


# few rows whose splits are added up where they end: one to four row tiles, workgroups that hold the last columns of one matrix and the first of
# the next, columns past the last whole sixteen, lhs that fills what the rings leave (12x4096, codes 11x4096) and lhs that does not fit (13x4096, codes 12x4096)
@pytest.mark.parametrize("M,K,N,mats,block", [(2, 512, 3000, 3, 0), (16, 2048, 1002, 3, 0), (17, 1920, 2034, 2, 0), (32, 1024, 1300, 3, 128), (33, 896, 3010, 3, 64),
                                              (64, 512, 4098, 3, 0), (64, 512, 4098, 2, 256), (11, 4096, 1346, 3, 128), (12, 4096, 1346, 3, 128), (12, 4096, 1346, 3, 0), (13, 4096, 1346, 3, 0), (3, 8192, 1026, 1, 0)])
def test_few_rows_added_up_where_they_end(gpu, M, K, N, mats, block):
    G = gpu
    check, L, VP = G.B.check, G.L(), G.B.vp
    x, ws = normal((M, K), 0, 450, 1.0), [normal((N, K), 0, 451 + g, 0.02) for g in range(mats)]
    codes = [O.quantize_absmax_u8(w, block) for w in ws] if block else []
    refs = ([O.matmul_nt_kernel_order(x, codes=c, scales=s, block=block, n_mats=mats) for c, s in codes] if block else
            [O.matmul_nt_kernel_order(x, w, n_mats=mats) for w in ws])
    wd, sd = [G.dev_keep(c[0]) for c in codes] or [G.dev_keep(w) for w in ws], [G.dev_keep(c[1]) for c in codes]
    w_arr, s_arr = (VP * mats)(*[w.ptr for w in wd]), (VP * mats)(*[s.ptr for s in sd]) if block else None
    # lhs by itself, then inside the first output, which may only be written when all of lhs has been read
    whole = np.zeros(M * max(K, N), dtype=np.float16)
    whole[:M * K] = x.reshape(-1)
    for same in (False, True):
        lhs = G.dev_keep(whole)
        outs = [lhs if same and g == 0 else G.empty((M, N)) for g in range(mats)]
        o_arr = (VP * mats)(*[o.ptr for o in outs])
        if block:
            check(L.lcu_gemm_f16u8_nt_multi(o_arr, lhs.ptr, w_arr, s_arr, mats, M, K, N, block, 0.0, None))
        else:
            check(L.lcu_gemm_f16_nt_multi(o_arr, lhs.ptr, w_arr, mats, M, K, N, 0.0, None))
        for o, ref in zip(outs, refs):
            assert G.ulp_mismatch(G.host(o, (M, N)), ref) == 0.0, O.gemm_plan(M, K, N, block > 0, block or 128, mats)
    G.release()


# uint8 tiles of 256 rows at their edges: 128 and 256 columns, K split over workgroups, blocks of one, two and four K
# stages, and a block that takes the other kernel
@pytest.mark.parametrize("M,K,N,block", [(2049, 256, 4100, 64), (4096, 128, 4090, 128), (2300, 512, 6000, 256), (300, 5120, 1030, 128),
                                         (2049, 128, 4100, 32), (65, 128, 20500, 64), (127, 256, 35000, 128), (100, 5120, 1030, 128),
                                         (257, 128, 6790, 64), (1100, 384, 3690, 128), (1100, 384, 3690, 32)])
def test_gemm_u8_large_tiles_ragged(gpu, M, K, N, block):
    G = gpu
    x, w = normal((M, K), 0, 420, 1.0), normal((N, K), 0, 421, 0.02)
    w[3] *= np.float16(2.0 ** -7)             # subnormal scales, and a row of zeros
    w[5] = 0
    codes, scales = O.quantize_absmax_u8(w, block)
    got = G.gemm_u8(x, codes, scales, block)
    assert G.ulp_mismatch(got, O.matmul_nt_u8(x, codes, scales, block, flavour=2)) == 0.0, O.gemm_plan(M, K, N, True)
    G.release()


@pytest.mark.parametrize("M,K,N,count", [(512, 512, 4096, 3), (8, 4096, 4096, 3), (40, 1024, 11008, 2), (300, 256, 700, 2),
                                          (33, 200, 70, 3), (1, 512, 300, 3),
                                          # uint8: each alone has few tiles, together they have many
                                          (512, 256, 3072, 3), (1000, 384, 1990, 2),
                                          # few rows whose columns take two and three rounds of one workgroup per compute unit
                                          (8, 640, 9664, 3), (33, 512, 9664, 3), (9, 512, 31990, 2)])
def test_gemm_multi_matches_separate_calls(gpu, M, K, N, count):
    """Several weight matrices of one shape in one launch (Wq, Wk, Wv; W1, W3): what separate calls give
    (to the matmul tolerance: the fused launch may pick another tile shape, hence another summation order)
    and what the oracle gives, for fp16 and uint8 weights, in every dispatch branch (large tiles,
    short-prompt split-K, ragged K, a single row)."""
    G = gpu
    L = G.L()
    VP = G.B.vp
    x = normal((M, K), 0, 1600, 1.0)
    xd = G.dev_keep(x)
    ws = [normal((N, K), 0, 1601 + g, 0.02) for g in range(count)]
    wd = [G.dev_keep(w) for w in ws]
    sep = [G.gemm_f16(x, w) for w in ws]
    outs = [G.empty((M, N)) for _ in range(count)]
    out_arr = (VP * count)(*[o.ptr for o in outs])
    w_arr = (VP * count)(*[w.ptr for w in wd])
    G.B.check(L.lcu_gemm_f16_nt_multi(out_arr, xd.ptr, w_arr, count, M, K, N, 0.0, None))
    for g in range(count):
        got = G.host(outs[g], (M, N))
        assert G.max_abs_rel(got, sep[g]) <= TOL and G.ulp_mismatch(got, sep[g]) < 0.05, g
        assert G.max_abs_rel(got, O.matmul_nt(x, ws[g])) <= TOL, g
        if K % 8 == 0:
            assert G.ulp_mismatch(got, O.matmul_nt_kernel_order(x, ws[g], n_mats=count)) == 0.0, g
    if K % 128 == 0:
        q = [O.quantize_absmax_u8(w, 128) for w in ws]
        cd = [G.dev_keep(c) for c, _ in q]
        sd = [G.dev_keep(sc) for _, sc in q]
        sep = [G.gemm_u8(x, c, sc, 128) for c, sc in q]
        c_arr = (VP * count)(*[c.ptr for c in cd])
        s_arr = (VP * count)(*[sc.ptr for sc in sd])
        G.B.check(L.lcu_gemm_f16u8_nt_multi(out_arr, xd.ptr, c_arr, s_arr, count, M, K, N, 128, 0.0, None))
        for g in range(count):
            got = G.host(outs[g], (M, N))
            assert G.max_abs_rel(got, sep[g]) <= TOL and G.ulp_mismatch(got, sep[g]) < 0.05, g
            assert G.max_abs_rel(got, O.matmul_nt_u8(x, q[g][0], q[g][1], 128)) <= TOL, g
            assert G.ulp_mismatch(got, O.matmul_nt_kernel_order(x, codes=q[g][0], scales=q[g][1], block=128,
                                                               n_mats=count)) == 0.0, g
    # beta = 1: every output starts from its own earlier contents
    olds = [normal((M, N), 0, 1650 + g, 1.0) for g in range(count)]
    for g in range(count):
        G.B.check(L.lcu_h2d(outs[g].ptr, olds[g].ctypes.data_as(VP), olds[g].nbytes, None))
    G.B.check(L.lcu_gemm_f16_nt_multi(out_arr, xd.ptr, w_arr, count, M, K, N, 1.0, None))
    for g in range(count):
        assert G.max_abs_rel(G.host(outs[g], (M, N)), O.matmul_nt(x, ws[g], beta=1.0, out=olds[g])) <= TOL, g
    assert L.lcu_gemm_f16_nt_multi(out_arr, xd.ptr, w_arr, 4, M, K, N, 0.0, None) == -2
    G.release()


def test_gemm_dispatch_sweep_bit_exact(gpu):
    """Seventy seeded shapes across the dispatcher's branches (few and many rows, K in whole stages or
    ragged, tile counts on both sides of every threshold, one to three matrices per launch, fp16 and
    uint8): the oracle's restatement of the cut of K must give the device's bits on all of them."""
    G = gpu
    L = G.L()
    VP = G.B.vp
    rng = np.random.default_rng(77)
    plans = set()
    for case in range(70):
        M = int(rng.choice([2, 7, 32, 33, 64, 65, 100, 256, 300, 512, 700, 1100]))
        K = int(rng.choice([64, 128, 136, 256, 384, 640, 1024, 2560, 5120]))
        N = int(rng.choice([24, 128, 1000, 2048, 4096, 5120, 8200, 11008, 17920]))
        nm = int(rng.choice([1, 1, 2, 3]))
        u8 = bool(rng.integers(0, 2)) and K % 128 == 0
        if M * K * N * nm > 2.5e10:
            K = 128
        x = normal((M, K), 5, 3 * case, 1.0)
        ws = [normal((N, K), 5, 3 * case + 1 + g, 0.02) for g in range(nm)]
        xd = G.dev_keep(x)
        outs = [G.empty((M, N)) for _ in range(nm)]
        out_arr = (VP * nm)(*[o.ptr for o in outs])
        if u8:
            q = [O.quantize_absmax_u8(w, 128) for w in ws]
            cd, sd = [G.dev_keep(c) for c, _ in q], [G.dev_keep(sc) for _, sc in q]
            G.B.check(L.lcu_gemm_f16u8_nt_multi(out_arr, xd.ptr, (VP * nm)(*[c.ptr for c in cd]), (VP * nm)(*[sc.ptr for sc in sd]),
                                                nm, M, K, N, 128, 0.0, None))
            want = [O.matmul_nt_kernel_order(x, codes=c, scales=sc, block=128, n_mats=nm) for c, sc in q]
        else:
            wd = [G.dev_keep(w) for w in ws]
            G.B.check(L.lcu_gemm_f16_nt_multi(out_arr, xd.ptr, (VP * nm)(*[w.ptr for w in wd]), nm, M, K, N, 0.0, None))
            want = [O.matmul_nt_kernel_order(x, w, n_mats=nm) for w in ws]
        plan = O.gemm_plan(M, K, N, u8, 128, nm)
        plans.add(plan)
        for g in range(nm):
            assert G.ulp_mismatch(G.host(outs[g], (M, N)), want[g]) == 0.0, (case, M, K, N, nm, u8, plan, g)
        G.release()
    assert len(plans) >= 6, plans  # single chains, two groups per stage, several depths of split


def test_streams_own_their_workspace(gpu):
    """Split-K products (2..64 rows) keep fp32 partial sums in scratch memory.  Every stream made by
    lcu_stream_create has a workspace of its own, so two host threads driving two streams at once
    get the results of a single undisturbed call, bit for bit."""
    import ctypes as C
    import threading
    G = gpu
    L = G.L()
    K, N = 4096, 4096
    cases = []
    for t in range(2):
        x = normal((8 + 8 * t, K), 3, 40 + t, 1.0)
        w = normal((N, K), 3, 50 + t, 0.02)
        cases.append((x, w, G.gemm_f16(x, w)))
    G.release()
    results = [None, None]

    def work(t):
        x, w, _ = cases[t]
        stream = G.B.vp()
        G.B.check(L.lcu_stream_create(C.byref(stream)))
        xd, wd, od = G.dev(x), G.dev(w), G.empty((x.shape[0], N))
        bad = 0
        for _ in range(200):
            G.B.check(L.lcu_gemm_f16_nt(od.ptr, xd.ptr, wd.ptr, x.shape[0], K, N, 0.0, stream))
        G.B.check(L.lcu_sync(stream))
        results[t] = G.host(od, (x.shape[0], N))
        G.B.check(L.lcu_stream_destroy(stream))
        for b in (xd, wd, od):
            b.free()

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for t in range(2):
        assert results[t] is not None and (results[t].view(np.uint16) == cases[t][2].view(np.uint16)).all()


# tiles below 128x64 and below those that K is dealt for, either side of where a round of them ends; ragged rows and columns, rows off 16 bytes
@pytest.mark.parametrize("M,K,N,splits,tile", [(66, 256, 1001, 0, (64, 32)), (65, 384, 4096, 0, (64, 32)), (67, 128, 4100, 0, (64, 64)),
                                               (130, 384, 5440, 0, (64, 64)), (130, 256, 5472, 0, (128, 64)), (193, 128, 2052, 0, (64, 64)),
                                               (66, 5120, 2056, 2, (64, 64)), (66, 5120, 4169, 2, (128, 64)), (130, 5120, 1100, 2, (64, 64)),
                                               (257, 5120, 2700, 2, (128, 128))])
@pytest.mark.parametrize("u8", [False, True])
def test_gemm_smaller_tiles_of_one_round(gpu, u8, M, K, N, splits, tile):
    import gemm_plan
    G = gpu
    assert gemm_plan.rows(M, K, N) == (("split_large", splits) if splits else ("halves", 1))
    largest = (128, 64) if not splits else (128, 128) if M <= 128 else (256, 128)
    narrowest = not splits and not u8
    assert gemm_plan.tile_size(M, N, max(splits, 1), largest, narrowest) == ((64, 64) if tile == (64, 32) and u8 else tile)
    x, w, old = normal((M, K), 0, 450, 1.0), normal((N, K), 0, 451, 0.02), normal((M, N), 0, 452, 1.0)
    if u8:
        codes, scales = O.quantize_absmax_u8(w, 128)
        assert G.ulp_mismatch(G.gemm_u8(x, codes, scales, 128), O.matmul_nt_u8(x, codes, scales, 128, flavour=2)) == 0.0
    else:
        assert G.ulp_mismatch(G.gemm_f16(x, w), O.matmul_nt(x, w, flavour=2)) == 0.0
        assert G.ulp_mismatch(G.gemm_f16(x, w, beta=1.0, out=old), O.matmul_nt(x, w, beta=1.0, out=old, flavour=2)) == 0.0
    G.release()


# products whose columns fit one tile of 64: the workgroup that stores rows has read them, so outputs may lie over lhs
@pytest.mark.parametrize("M,K,N,at", [(100, 128, 64, 0), (128, 256, 64, 0), (65, 384, 33, 128), (90, 128, 50, 4096), (128, 512, 64, 65536)])
@pytest.mark.parametrize("u8", [False, True])
def test_gemm_of_few_columns_over_lhs(gpu, u8, M, K, N, at):
    G = gpu
    x, w = normal((M, K), 0, 460, 1.0), normal((N, K), 0, 461, 0.02)
    if u8:
        codes, scales = O.quantize_absmax_u8(w, 64)
        want, args = G.gemm_u8(x, codes, scales, 64), (G.dev_keep(codes).ptr, G.dev_keep(scales).ptr)
    else:
        want, args = G.gemm_f16(x, w), (G.dev_keep(w).ptr,)
    held = G.dev_keep(x)
    call, tail = (G.L().lcu_gemm_f16u8_nt, (64, 0.0, None)) if u8 else (G.L().lcu_gemm_f16_nt, (0.0, None))
    G.B.check(call(held.ptr + at, held.ptr, *args, M, K, N, *tail))
    got = G.host(held, (M, K)).reshape(-1)[at // 2:at // 2 + M * N]
    assert np.array_equal(got.view(np.uint16), want.reshape(-1).view(np.uint16))
    G.release()


def test_gemm_rejects_bad_shapes(gpu):
    G = gpu
    a = G.dev(np.zeros((4, 12), dtype=np.float16))
    assert G.L().lcu_gemm_f16_nt(a.ptr, a.ptr, a.ptr, 4, 12, 4, 0.0, None) == -2  # K % 8
    assert G.L().lcu_gemm_f16_nt(None, a.ptr, a.ptr, 4, 16, 4, 0.0, None) == -2
    assert G.L().lcu_gemm_f16u8_nt(a.ptr, a.ptr, a.ptr, a.ptr, 1, 256, 4, 100, 0.0, None) == -2
    assert b"lcu_gemm_f16u8_nt" in G.L().lcu_last_error()
    assert G.L().lcu_gemm_f16_nt(a.ptr, a.ptr, a.ptr, 0, 16, 4, 0.0, None) == 0  # empty input is fine


@pytest.mark.parametrize("rows,cols", [(1, 4096), (512, 4096), (3, 6656), (5, 200)])
def test_rmsnorm(gpu, rows, cols):
    G = gpu
    x = normal((rows, cols), 0, 500, 1.0)
    w = (normal((cols,), 0, 501, 0.1).astype(np.float32) + 1).astype(np.float16)
    out_d = G.empty((rows, cols))
    G.B.check(G.L().lcu_rmsnorm(out_d.ptr, G.dev_keep(x).ptr, G.dev_keep(w).ptr, rows, cols, 1e-6, None))
    got = G.host(out_d, (rows, cols))
    ref = O.rms_norm(x, w, 1e-6)
    assert G.max_abs_rel(got, ref) <= TOL
    # same reduction order and IEEE 1/sqrt on both sides
    assert G.ulp_mismatch(got, ref) == 0.0
    G.release()


@pytest.mark.parametrize("rows,pos", [(1, 0), (1, 1337), (512, 0), (40, 2000)])
def test_rope_bit_exact(gpu, rows, pos):
    G = gpu
    heads, dim = 32, 4096
    x = normal((rows, dim), 0, 600, 1.0)
    tab = G.B.vp()
    G.B.check(G.L().lcu_rope_table_create(G.B.C.byref(tab), 2048, 128, 10000.0))
    out_d = G.empty((rows, dim))
    G.B.check(G.L().lcu_rope(out_d.ptr, G.dev_keep(x).ptr, rows, dim, heads, pos, tab, 2048, None))
    got = G.host(out_d, (rows, dim))
    assert G.ulp_mismatch(got, O.rotary(x, heads, pos_offset=pos)) == 0.0
    # in place
    xd = G.dev(x)
    G.B.check(G.L().lcu_rope(xd.ptr, xd.ptr, rows, dim, heads, pos, tab, 2048, None))
    assert G.ulp_mismatch(G.host(xd, (rows, dim)), got) == 0.0
    assert G.L().lcu_rope(xd.ptr, xd.ptr, rows, dim, heads, 2048 - rows + 1, tab, 2048, None) == -2  # past the table
    # two tensors in one launch
    y = normal((rows, dim), 0, 601, 1.0)
    ad, bd = G.dev(x), G.dev(y)
    G.B.check(G.L().lcu_rope_pair(ad.ptr, bd.ptr, rows, dim, heads, pos, tab, 2048, None))
    assert G.ulp_mismatch(G.host(ad, (rows, dim)), got) == 0.0
    assert G.ulp_mismatch(G.host(bd, (rows, dim)), O.rotary(y, heads, pos_offset=pos)) == 0.0
    assert G.L().lcu_rope_pair(ad.ptr, bd.ptr, rows, dim, heads, 2048 - rows + 1, tab, 2048, None) == -2
    G.release()
    G.L().lcu_free(tab)


@pytest.mark.parametrize("rows,w,temp", [(1, 32000, 0.8), (64, 512, 1.0), (3, 77, 1.0), (2, 2048, 0.9)])
def test_softmax_rows(gpu, rows, w, temp):
    G = gpu
    x = normal((rows, w), 0, 700, 2.0)
    if w > 100:
        x[:, w - 30:] = -np.inf
    out_d = G.empty((rows, w))
    G.B.check(G.L().lcu_softmax_rows(out_d.ptr, G.dev_keep(x).ptr, rows, w, temp, None))
    got = G.host(out_d, (rows, w))
    ref = O.softmax_rows(x, temp)
    assert G.ulp_mismatch(got, ref) == 0.0  # same association of the sums, same exponential: every bit
    if w > 100:
        assert (got[:, w - 30:] == 0).all()
    G.release()


def test_silu_mul(gpu):
    G = gpu
    n = 512 * 11008
    a, b = normal((n,), 0, 800, 2.0), normal((n,), 0, 801, 1.0)
    out_d = G.empty((n,))
    G.B.check(G.L().lcu_silu_mul(out_d.ptr, G.dev_keep(a).ptr, G.dev_keep(b).ptr, n, None))
    got = G.host(out_d, (n,))
    ref = O.silu_mul(a, b)
    assert G.ulp_mismatch(got, ref) == 0.0
    # ragged length (the last thread's eight elements are cut) and buffers off the 16-byte grid
    for n2, off in ((2051, 0), (1000, 3)):
        ad, bd, od = G.dev_keep(a[:n2 + off]), G.dev_keep(b[:n2 + off]), G.empty((n2 + off,))
        G.B.check(G.L().lcu_silu_mul(od.ptr + 2 * off, ad.ptr + 2 * off, bd.ptr + 2 * off, n2, None))
        got2 = G.host(od, (n2 + off,))[off:]
        assert (got2.view(np.uint16) == got[off:n2 + off].view(np.uint16)).all()
    G.release()


def test_silu_of_every_half(gpu):
    """The short forms of exponential and division against the general ones: every a, with b of every kind."""
    G = gpu
    a = np.arange(65536, dtype=np.uint16).view(np.float16)
    for value in (1.0, -0.37, 65504.0, 6e-8, -0.0, np.inf, np.nan, 0.5, 2.5, -4.5):  # the last three: ties of subnormal results where the quotient is a unit off
        b = np.full(65536, value, np.float16)
        out = G.dev_keep(np.zeros(65536, np.float16))
        G.B.check(G.L().lcu_silu_mul(out.ptr, G.dev_keep(a).ptr, G.dev_keep(b).ptr, 65536, None))
        got, want = G.host(out, (65536,), np.float16), O.silu_mul(a, b)
        assert (np.isnan(got) == np.isnan(want)).all()
        assert (got.view(np.uint16) == want.view(np.uint16))[~np.isnan(want)].all(), value
    G.release()


@pytest.mark.parametrize("n,dim,ffn", [(65, 128, 10240), (100, 128, 16400), (129, 256, 10256), (300, 384, 5136), (512, 1024, 11008), (773, 2048, 6160), (1027, 2048, 6592), (1033, 2048, 6704), (1024, 1024, 13392)])
def test_up_products_with_their_silu(gpu, n, dim, ffn):
    """Large tiles whose columns alternate between W1 and W3: the bits of the two products and lcu_silu_mul, whatever is behind the last row
    and column.  128, 192 and 256 columns, whole rounds and the rest, 128 rows."""
    G, L = gpu, gpu.L()
    rng = np.random.default_rng(n + ffn)
    x = G.dev_keep(rng.standard_normal((n, dim)).astype(np.float16))
    w = [G.dev_keep((rng.standard_normal((ffn, dim)) * 3 / dim ** 0.5).astype(np.float16)) for _ in range(2)]
    t1, t3, want, got = (G.dev_keep(np.full((n + 1, ffn), -7, np.float16)) for _ in range(4))
    ptrs = lambda bufs: (C.c_void_p * len(bufs))(*[b.ptr for b in bufs])
    G.B.check(L.lcu_gemm_f16_nt_multi(ptrs([t1, t3]), x.ptr, ptrs(w), 2, n, dim, ffn, 0.0, None))
    G.B.check(L.lcu_silu_mul(want.ptr, t1.ptr, t3.ptr, n * ffn, None))
    G.B.check(L.lcu_batch_ffn_up(got.ptr, t1.ptr, t3.ptr, x.ptr, ptrs(w), None, 0, n, dim, ffn, None))
    a, b = G.host(got, (n + 1, ffn), np.uint16), G.host(want, (n + 1, ffn), np.uint16)
    assert (a == b).all() and (a[n] == np.float16(-7).view(np.uint16)).all()
    G.release()


@pytest.mark.parametrize("n,dim,ffn,at", [(100, 128, 16400, 0), (512, 1024, 11008, 0), (512, 1024, 11008, 4000000), (1033, 2048, 6704, 0), (773, 2048, 6160, 773 * 6160 - 8)])
def test_up_products_over_their_lhs(gpu, n, dim, ffn, at):
    """Outputs in the buffer of lhs, from its first element on or with lhs at their element `at`: the products go to the temporaries first, as
    the workgroups of one launch would still be reading lhs."""
    G, L = gpu, gpu.L()
    rng = np.random.default_rng(n + ffn + at)
    x = rng.standard_normal((n, dim)).astype(np.float16)
    w = [G.dev_keep((rng.standard_normal((ffn, dim)) * 3 / dim ** 0.5).astype(np.float16)) for _ in range(2)]
    ptrs = lambda bufs: (C.c_void_p * len(bufs))(*[b.ptr for b in bufs])
    t1, t3, want, u1, u3 = (G.dev_keep(np.full((n, ffn), -7, np.float16)) for _ in range(5))
    G.B.check(L.lcu_gemm_f16_nt_multi(ptrs([t1, t3]), G.dev_keep(x).ptr, ptrs(w), 2, n, dim, ffn, 0.0, None))
    G.B.check(L.lcu_silu_mul(want.ptr, t1.ptr, t3.ptr, n * ffn, None))
    both = np.zeros(max(n * ffn, at + n * dim), np.float16)
    both[at:at + n * dim] = x.reshape(-1)
    both = G.dev_keep(both)
    G.B.check(L.lcu_batch_ffn_up(both.ptr, u1.ptr, u3.ptr, both.ptr + 2 * at, ptrs(w), None, 0, n, dim, ffn, None))
    for got, ref in ((both, want), (u1, t1), (u3, t3)):
        assert (G.host(got, (n, ffn), np.uint16) == G.host(ref, (n, ffn), np.uint16)).all()
    G.release()


def test_exp_bit_exact(gpu):
    """the exponential of every softmax and SiLU: host restatement and kernel agree on every bit"""
    G = gpu
    rng = np.random.default_rng(5)
    x = np.concatenate([np.linspace(-100, 95, 1 << 20), rng.normal(0, 4, 1 << 20), rng.uniform(-18, 0, 1 << 20),
                        [0.0, -0.0, np.inf, -np.inf, 88.72283, 88.72284, -87.33654, -87.33655, -87.3]]).astype(np.float32)
    out_d = G.B.empty(x.shape, np.float32)
    G.B.check(G.L().lcu_exp_f32(out_d.ptr, G.dev_keep(x).ptr, x.size, None))
    got = G.host(out_d, x.shape, np.float32)
    assert (got.view(np.uint32) == O.exp_f32(x).view(np.uint32)).all()
    G.release()


def test_embed_bit_exact(gpu):
    G = gpu
    vocab, dim = 1000, 512
    table = normal((vocab, dim), 0, 900, 0.02)
    ids = np.array([0, 999, 5, 5, 123], dtype=np.int16)
    out_d = G.empty((len(ids), dim))
    G.B.check(G.L().lcu_embed(out_d.ptr, G.dev_keep(ids).ptr, len(ids), dim, G.dev_keep(table).ptr, vocab, None))
    assert G.ulp_mismatch(G.host(out_d, (len(ids), dim)), O.embed(ids, table)) == 0.0
    codes, scales = O.quantize_absmax_u8(table, 128)
    G.B.check(G.L().lcu_embed_u8(out_d.ptr, G.dev_keep(ids).ptr, len(ids), dim, G.dev_keep(codes).ptr,
                                 G.dev_keep(scales).ptr, 128, vocab, None))
    assert G.ulp_mismatch(G.host(out_d, (len(ids), dim)), O.embed_u8(ids, codes, scales, 128)) == 0.0
    # an id outside the table gives zeros, not a stray read
    bad = np.array([1000, -1], dtype=np.int16)
    G.B.check(G.L().lcu_embed(out_d.ptr, G.dev_keep(bad).ptr, 2, dim, G.dev_keep(table).ptr, vocab, None))
    assert (G.host(out_d, (2, dim)) == 0).all()
    G.B.check(G.L().lcu_embed_u8(out_d.ptr, G.dev_keep(bad).ptr, 2, dim, G.dev_keep(codes).ptr,
                                 G.dev_keep(scales).ptr, 128, vocab, None))
    assert (G.host(out_d, (2, dim)) == 0).all()
    G.release()
    # uint8 rows of more than one piece of 4096 codes (sixteen codes per thread), and a block size that is
    # not a multiple of 16 (one code per thread)
    for vocab, dim, block in ((40, 6656, 128), (40, 4096 + 16, 16), (50, 480, 24)):
        table = normal((vocab, dim), 0, 901, 0.02)
        codes, scales = O.quantize_absmax_u8(table, block)
        ids = np.array([vocab - 1, 0, 7, vocab, 7], dtype=np.int16)
        out_d = G.empty((len(ids), dim))
        G.B.check(G.L().lcu_embed_u8(out_d.ptr, G.dev_keep(ids).ptr, len(ids), dim, G.dev_keep(codes).ptr,
                                     G.dev_keep(scales).ptr, block, vocab, None))
        got = G.host(out_d, (len(ids), dim))
        want = O.embed_u8(np.where(ids < vocab, ids, 0).astype(np.int16), codes, scales, block)
        want[3] = 0
        assert (got.view(np.uint16) == want.view(np.uint16)).all()
        G.release()


def test_embed_rmsnorm_equals_embed_then_rmsnorm(gpu):
    """The one-token step's first launch: the gathered row and its norm, to the bit what lcu_embed[_u8] and
    lcu_rmsnorm give one after the other (and so what the oracle gives for them)."""
    G = gpu
    for vocab, dim, block in ((300, 4096, 0), (300, 4096, 128), (100, 6656, 128), (64, 264, 0), (64, 264, 8), (20, 8192, 64)):
        table = normal((vocab, dim), 0, 910, 0.02)
        w = normal((dim,), 0, 911, 1.0)
        ids = np.array([vocab - 1, 0, 5, vocab, -3, 5], dtype=np.int16)
        x_d, n_d = G.empty((len(ids), dim)), G.empty((len(ids), dim))
        safe = np.where((ids >= 0) & (ids < vocab), ids, 0).astype(np.int16)
        if block:
            codes, scales = O.quantize_absmax_u8(table, block)
            G.B.check(G.L().lcu_embed_rmsnorm(x_d.ptr, n_d.ptr, G.dev_keep(ids).ptr, len(ids), dim, G.dev_keep(codes).ptr,
                                              G.dev_keep(scales).ptr, block, vocab, G.dev_keep(w).ptr, 1e-6, None))
            rows = O.embed_u8(safe, codes, scales, block)
        else:
            G.B.check(G.L().lcu_embed_rmsnorm(x_d.ptr, n_d.ptr, G.dev_keep(ids).ptr, len(ids), dim, G.dev_keep(table).ptr,
                                              None, 0, vocab, G.dev_keep(w).ptr, 1e-6, None))
            rows = O.embed(safe, table)
        rows[3] = 0
        rows[4] = 0
        assert (G.host(x_d, (len(ids), dim)).view(np.uint16) == rows.view(np.uint16)).all()
        assert (G.host(n_d, (len(ids), dim)).view(np.uint16) == O.rms_norm(rows, w, 1e-6).view(np.uint16)).all()
        G.release()
    out = G.empty((1, 8200))
    assert G.L().lcu_embed_rmsnorm(out.ptr, out.ptr, out.ptr, 1, 8200, out.ptr, None, 0, 10, out.ptr, 1e-6, None) != 0
    G.release()


def test_argmax_first_maximum(gpu):
    G = gpu
    out_d = G.empty((1,), np.int32)
    rng = np.random.default_rng(0)
    for n in (5, 1024, 32000, 40001):
        p = rng.random(n).astype(np.float16)
        m = p.max()
        ties = rng.choice(n, size=min(4, n), replace=False)
        p[ties] = m
        G.B.check(G.L().lcu_argmax_f16(out_d.ptr, G.dev_keep(p).ptr, n, None))
        expected = int(np.flatnonzero(p == m)[0])
        assert int(G.host(out_d, (1,), np.int32)[0]) == O.argmax_first(p) == expected
    G.release()


def test_error_stats(gpu):
    G = gpu
    for n in (1, 255, 4096, 1 << 20, (1 << 22) + 77):
        a = normal((n,), 8, 1, 1.0)
        b = normal((n,), 8, 2, 1.0)
        out = G.empty((3,), np.float32)
        da, db = G.dev_keep(a), G.dev_keep(b)
        G.B.check(G.L().lcu_error_stats(out.ptr, da.ptr, db.ptr, n, None))
        got = G.host(out, (3,), np.float32)
        want = O.error_stats(a, b)
        assert got[1] == want[1]                                  # the largest difference is exact
        assert np.allclose(got[[0, 2]], want[[0, 2]], rtol=1e-5)  # fp32 partial sums against double
        # run to run identical (the reference's atomics are not)
        G.B.check(G.L().lcu_error_stats(out.ptr, da.ptr, db.ptr, n, None))
        assert (G.host(out, (3,), np.float32) == got).all()
        G.B.check(G.L().lcu_error_stats(out.ptr, da.ptr, da.ptr, n, None))
        assert (G.host(out, (3,), np.float32) == 0).all()
        G.release()


def test_memset_and_copies(gpu):
    G = gpu
    for n in (1, 15, 16, 17, 4099, 1 << 20):
        buf = G.empty((n + 32,), np.uint8)
        G.B.check(G.L().lcu_memset(buf.ptr, 0xAB, n + 32, None))
        G.B.check(G.L().lcu_memset(buf.ptr + 3, 0x11, n, None))
        h = G.host(buf, (n + 32,), np.uint8)
        assert (h[:3] == 0xAB).all() and (h[3:3 + n] == 0x11).all() and (h[3 + n:] == 0xAB).all()


ATT_CASES = [(1, 1), (1, 2), (1, 255), (1, 256), (1, 257), (1, 577), (1, 2048), (5, 5), (64, 64), (70, 70),
             (512, 512), (3, 130), (40, 300), (300, 2100), (64, 4096), (1, 4096)]


@pytest.mark.parametrize("n,T", ATT_CASES)
def test_attention(gpu, n, T):
    G = gpu
    heads, dim = 4, 512
    start = T - n
    q = normal((n, dim), 0, 1000, 1.0)
    k = normal((T, dim), 0, 1001, 1.0)
    v = normal((T, dim), 0, 1002, 1.0)
    out_d = G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out_d.ptr, G.dev_keep(q).ptr, G.dev_keep(k).ptr, G.dev_keep(v).ptr, n, T, start, dim,
                                  heads, None))
    got = G.host(out_d, (n, dim))
    ref = O.attention(q, k, v, heads, start)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.05  # fp32 summation order only
    if start == 0:
        assert G.ulp_mismatch(got[0], v[0]) == 0.0  # causal row 0 sees only itself
    # the oracle restates the kernels' own sums (for several rows: the matrix cores' steps), every bit
    if n == 1:
        assert G.ulp_mismatch(got, O.attention_decode_kernel_order(q, k, v, heads)) == 0.0
    else:
        assert G.ulp_mismatch(got, O.attention_prefill_kernel_order(q, k, v, heads, start)) == 0.0
    G.release()


@pytest.mark.parametrize("n,T", [(512, 512), (1, 577), (1, 2048), (64, 1024), (512, 2048), (33, 1100)])
def test_attention_llama7b_heads(gpu, n, T):
    """32 heads at dim 4096, the shapes of the benchmark configurations."""
    G = gpu
    heads, dim = 32, 4096
    start = T - n
    q = normal((n, dim), 0, 1010, 1.0)
    k = normal((T, dim), 0, 1011, 1.0)
    v = normal((T, dim), 0, 1012, 1.0)
    out_d = G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out_d.ptr, G.dev_keep(q).ptr, G.dev_keep(k).ptr, G.dev_keep(v).ptr, n, T, start, dim,
                                  heads, None))
    got = G.host(out_d, (n, dim))
    ref = O.attention(q, k, v, heads, start)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.05
    if n == 1:
        assert G.ulp_mismatch(got, O.attention_decode_kernel_order(q, k, v, heads)) == 0.0
    else:
        assert G.ulp_mismatch(got, O.attention_prefill_kernel_order(q, k, v, heads, start)) == 0.0
    G.release()


# calls with enough scores for the kernel that stores none: ragged rows and columns, 64- and 128-row tiles, rows behind cached ones
@pytest.mark.parametrize("heads,n,T", [(40, 601, 601), (64, 350, 385), (64, 900, 931), (52, 449, 450)])
def test_attention_of_many_scores(gpu, heads, n, T):
    G = gpu
    dim, start = heads * 128, T - n
    q, k, v = normal((n, dim), 0, 1020, 1.0), normal((T, dim), 0, 1021, 1.0), normal((T, dim), 0, 1022, 1.0)
    out_d = G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out_d.ptr, G.dev_keep(q).ptr, G.dev_keep(k).ptr, G.dev_keep(v).ptr, n, T, start, dim, heads, None))
    assert G.ulp_mismatch(G.host(out_d, (n, dim)), O.attention_prefill_kernel_order(q, k, v, heads, start)) == 0.0
    G.release()


@pytest.mark.parametrize("shift", [1, 4])
def test_attention_of_many_scores_into_an_output_off_16_bytes(gpu, shift):
    """An output 2 bytes off any boundary goes to the kernel that stores 2 bytes at a time, one of 8 bytes need not; same bits."""
    G = gpu
    heads, n, dim = 40, 601, 5120
    q, k, v = normal((n, dim), 0, 1023, 1.0), normal((n, dim), 0, 1024, 1.0), normal((n, dim), 0, 1025, 1.0)
    qd, kd, vd = G.dev_keep(q), G.dev_keep(k), G.dev_keep(v)
    flat, out = G.dev(np.full(n * dim + 8, 9.0, np.float16)), G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out.ptr, qd.ptr, kd.ptr, vd.ptr, n, n, 0, dim, heads, None))
    G.B.check(G.L().lcu_attention(flat.ptr + 2 * shift, qd.ptr, kd.ptr, vd.ptr, n, n, 0, dim, heads, None))
    got = G.host(flat, (n * dim + 8,))
    assert G.ulp_mismatch(got[shift:shift + n * dim].reshape(n, dim), G.host(out, (n, dim))) == 0.0
    assert (got[:shift] == 9.0).all() and (got[shift + n * dim:] == 9.0).all()
    G.release()


def test_attention_of_many_scores_equals_portions(gpu):
    """One call against portions of 16 rows, which take the other kernel: the same bits, also with scores past the
    range of fp16, products past that of fp32 (infinite operands), NaN, and rows that see equal scores only."""
    G = gpu
    heads, n = 48, 520
    dim = heads * 128
    q, k, v = normal((n, dim), 0, 1030, 1.0), normal((n, dim), 0, 1031, 1.0), normal((n, dim), 0, 1032, 1.0)
    q[:, :128] *= 0                       # head 0: equal scores
    q[:, 128:256] *= 60                   # head 1: one score takes all, exponentials underflow
    k[100, 256:384] = 60000               # head 2: a score of +-infinity in fp16 from row 100 on
    q[:, 256:384] = 60000
    k[200, 384], k[300, 512] = np.inf, np.nan
    kd, vd = G.dev_keep(k), G.dev_keep(v)
    out_d = G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out_d.ptr, G.dev_keep(q).ptr, kd.ptr, vd.ptr, n, n, 0, dim, heads, None))
    got = G.host(out_d, (n, dim))
    part = G.empty((16, dim))
    for r in range(0, n, 16):
        rows = min(16, n - r)
        G.B.check(G.L().lcu_attention(part.ptr, G.dev_keep(q[r:r + rows]).ptr, kd.ptr, vd.ptr, rows, r + rows, r, dim, heads, None))
        want = G.host(part, (16, dim))[:rows]
        assert (np.isnan(got[r:r + rows]) == np.isnan(want)).all(), r
        same = got[r:r + rows].view(np.uint16) == want.view(np.uint16)
        assert (same | np.isnan(want)).all(), r
    assert np.isnan(got[250:, 384:512]).any() and not np.isnan(got[:200, 384:512]).any()
    G.release()


# the kernel that stores scores: a lane's pairs of a row in registers up to 256, 512 and 1024 columns, on both sides of each, and in
# LDS beyond; both sides of the line to the kernel above, with three strips and with one in a compute unit's LDS
@pytest.mark.parametrize("heads,n,T", [(4, 17, 256), (4, 20, 257), (4, 33, 512), (3, 18, 513), (3, 16, 1024), (3, 31, 1025), (64, 500, 500), (64, 560, 560),
                                       (17, 300, 1838), (14, 1250, 1990), (9, 1250, 1990)])
def test_attention_of_scores_in_registers(gpu, heads, n, T):
    test_attention_of_many_scores(gpu, heads, n, T)


# both sides of the line where two strips fit
@pytest.mark.parametrize("heads,n,T", [(52, 246, 1500), (52, 306, 1531)])
def test_attention_of_scores_where_two_strips_fit(gpu, heads, n, T):
    import gemm_plan
    assert gemm_plan.scores_again(heads, n, T) == (n > 300)
    test_attention_of_many_scores(gpu, heads, n, T)


@pytest.mark.parametrize("heads,n", [(64, 900), (64, 560), (5, 150)])
def test_attention_of_scores_at_both_ends_of_fp16(gpu, heads, n):
    """Every kernel for prompts against the oracle to the bit: scores among the subnormals, and scores on both sides of 62 000, where some wavefronts take
    the short forms and others do not."""
    G = gpu
    dim = heads * 128
    q, k, v = normal((n, dim), 0, 1050, 1.0), normal((n, dim), 0, 1051, 1.0), normal((n, dim), 0, 1052, 1.0)
    largest = lambda: np.abs(np.float64(q[:, 128:256]) @ np.float64(k[:, 128:256]).T).max(1)
    for x in (q, k):
        x[:, :128] *= np.float16(1e-3)
        x[:, 128:256] *= np.float16(100)
    q[:, 128:256] = (q[:, 128:256] * (7.3e5 / largest().max())).astype(np.float16)
    assert (largest() < 6.9e5).any() and 7.2e5 < largest().max() < 7.4e5  # beyond 7.41e5 a score is infinite
    out_d = G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out_d.ptr, G.dev_keep(q).ptr, G.dev_keep(k).ptr, G.dev_keep(v).ptr, n, n, 0, dim, heads, None))
    assert G.ulp_mismatch(G.host(out_d, (n, dim))[:, :256], O.attention_prefill_kernel_order(q[:, :256], k[:, :256], v[:, :256], 2, 0)) == 0.0
    G.release()


@pytest.mark.parametrize("heads,n", [(64, 560), (5, 150)])
def test_attention_of_extreme_scores(gpu, heads, n):
    """Both kernels for prompts against the oracle: equal scores, one that takes all, scores past fp16, products past fp32, NaN."""
    G = gpu
    dim = heads * 128
    q, k, v = normal((n, dim), 0, 1040, 1.0), normal((n, dim), 0, 1041, 1.0), normal((n, dim), 0, 1042, 1.0)
    q[:, :128] *= 0
    q[:, 128:256] *= 60
    k[100, 256:384] = 60000
    q[:, 256:384] = 60000
    k[60, 384], k[80, 512] = np.inf, np.nan
    out_d = G.empty((n, dim))
    G.B.check(G.L().lcu_attention(out_d.ptr, G.dev_keep(q).ptr, G.dev_keep(k).ptr, G.dev_keep(v).ptr, n, n, 0, dim, heads, None))
    got = G.host(out_d, (n, dim))
    assert G.ulp_mismatch(got[:, :256], O.attention_prefill_kernel_order(q[:, :256], k[:, :256], v[:, :256], 2, 0)) == 0.0
    # a score of +infinity or NaN leaves a row of NaN; one of -infinity is a probability of 0
    seen = np.tril(np.ones((n, n), bool))
    with np.errstate(all="ignore"):
        z = [np.float64(q[:, h * 128:h * 128 + 128]) @ np.float64(k[:, h * 128:h * 128 + 128]).T / 128 ** 0.5 for h in range(5)]
        lost = [(seen & ~(np.float32(x).astype(np.float16) < np.inf)).any(1) for x in z]
    assert lost[2][100:].all() and 0 < lost[3].sum() < n - 60 and lost[4].sum() == n - 80
    for h in (2, 3, 4):
        out = got[:, h * 128:h * 128 + 128]
        assert (np.isnan(out) == lost[h][:, None]).all(), h
        if h > 2:
            x = np.where(seen, np.where(lost[h][:, None], 0.0, z[h]), -np.inf)
            e = np.exp(x - x.max(1, keepdims=True))
            want = e @ np.float64(v[:, h * 128:h * 128 + 128]) / e.sum(1, keepdims=True)
            assert np.abs(out - want)[~lost[h]].max() < 1.6e-2  # values below 4: scores, probabilities and outputs in halves of 2^-11 each
    G.release()


def test_attention_decode_twice_reuses_workspace(gpu):
    # the split-T decode path keeps arrival counters in a workspace; back-to-back calls must agree
    G = gpu
    heads, dim, T = 32, 4096, 2048
    q = normal((1, dim), 0, 1100, 1.0)
    k = normal((T, dim), 0, 1101, 1.0)
    v = normal((T, dim), 0, 1102, 1.0)
    kd, vd, qd = G.dev_keep(k), G.dev_keep(v), G.dev_keep(q)
    ref = O.attention(q, k, v, heads, T - 1)
    out_d = G.empty((1, dim))
    for T_use in (T, 700, T):
        G.B.check(G.L().lcu_attention(out_d.ptr, qd.ptr, kd.ptr, vd.ptr, 1, T_use, T_use - 1, dim, heads, None))
        got = G.host(out_d, (1, dim))
        want = ref if T_use == T else O.attention(q, k[:T_use], v[:T_use], heads, T_use - 1)
        assert G.max_abs_rel(got, want) <= TOL
    assert G.L().lcu_attention(out_d.ptr, qd.ptr, kd.ptr, vd.ptr, 1, 10, 5, dim, heads, None) == -2
    assert G.L().lcu_attention(out_d.ptr, qd.ptr, kd.ptr, vd.ptr, 1, 10, 9, dim, 31, None) == -2
    G.release()


@pytest.mark.parametrize("heads,ctx", [(32, 1024), (52, 2048), (3, 4096)])
def test_attention_decode_spread_in_a_replayed_graph(gpu, heads, ctx):
    """lcu_attention_decode_spread (eight workgroups per head that hand their scores over inside the launch):
    two calls with different salts captured in one graph, replayed with the position and the step counter
    changed on the device between replays (positions going up and down, so rows hold scores of earlier
    epochs), every replay bit-exact against the kernel-order oracle and against lcu_attention_decode; no
    bounded wait ran out."""
    import ctypes as C
    G = gpu
    L = G.L()
    dim = heads * 128
    k = [normal((ctx, dim), 0, 1200 + i, 1.0) for i in range(2)]
    v = [normal((ctx, dim), 0, 1210 + i, 1.0) for i in range(2)]
    q = [normal((1, dim), 0, 1220 + i, 1.0) for i in range(2)]
    kd, vd, qd = [G.dev_keep(a) for a in k], [G.dev_keep(a) for a in v], [G.dev_keep(a) for a in q]
    out = [G.empty((1, dim)) for _ in range(2)]
    old = G.empty((1, dim))
    stream = C.c_void_p()
    G.B.check(L.lcu_stream_create(C.byref(stream)))
    state = G.B.DeviceBuffer(8)  # int32 position, uint32 step counter
    def set_state(pos, seq):
        a = np.array([pos, seq], dtype=np.uint32)
        G.B.check(L.lcu_h2d(state.ptr, a.ctypes.data_as(C.c_void_p), 8, stream))
        G.B.check(L.lcu_sync(stream))
    def enqueue():
        for i in range(2):
            G.B.check(L.lcu_attention_decode_spread(out[i].ptr, qd[i].ptr, kd[i].ptr, vd[i].ptr, state.ptr, state.ptr + 4,
                                                    i, ctx, dim, heads, stream))
    positions = [5, ctx - 1, 300, 0, 1023 if ctx > 1023 else ctx // 2, 17, ctx - 2]
    set_state(positions[0], 1)
    enqueue()  # eager
    G.B.check(L.lcu_sync(stream))
    G.B.check(L.lcu_graph_begin_capture(stream))
    enqueue()
    graph = C.c_void_p()
    G.B.check(L.lcu_graph_end_capture(stream, C.byref(graph)))
    for step, pos in enumerate(positions):
        set_state(pos, 2 + step)
        G.B.check(L.lcu_graph_launch(graph, stream))
        G.B.check(L.lcu_sync(stream))
        T = pos + 1
        for i in range(2):
            got = G.host(out[i], (1, dim))
            assert G.ulp_mismatch(got, O.attention_decode_kernel_order(q[i], k[i][:T], v[i][:T], heads)) == 0.0, (pos, i)
            G.B.check(L.lcu_attention_decode(old.ptr, qd[i].ptr, kd[i].ptr, vd[i].ptr, state.ptr, ctx, dim, heads, stream))
            G.B.check(L.lcu_sync(stream))
            assert G.ulp_mismatch(got, G.host(old, (1, dim))) == 0.0, (pos, i)
    # a step counter that has come round to the same low 21 bits: the caller clears the hand-over words first
    G.B.check(L.lcu_sync_reset(stream))
    set_state(300, 2 + (1 << 21))
    G.B.check(L.lcu_graph_launch(graph, stream))
    G.B.check(L.lcu_sync(stream))
    for i in range(2):
        assert G.ulp_mismatch(G.host(out[i], (1, dim)), O.attention_decode_kernel_order(q[i], k[i][:301], v[i][:301], heads)) == 0.0
    G.B.check(L.lcu_graph_begin_capture(stream))
    assert L.lcu_sync_reset(stream) == -2  # a memset node is not what a captured step may hold
    enqueue()
    graph2 = C.c_void_p()
    G.B.check(L.lcu_graph_end_capture(stream, C.byref(graph2)))
    G.B.check(L.lcu_graph_destroy(graph2))
    count = C.c_uint(123)
    G.B.check(L.lcu_sync_timeouts(stream, C.byref(count)))
    assert count.value == 0
    assert L.lcu_attention_decode_spread(out[0].ptr, qd[0].ptr, kd[0].ptr, vd[0].ptr, state.ptr, state.ptr + 4, 1024, ctx,
                                         dim, heads, stream) == -2
    assert L.lcu_attention_decode_spread(out[0].ptr, qd[0].ptr, kd[0].ptr, vd[0].ptr, state.ptr, None, 0, ctx, dim, heads,
                                         stream) == -2
    G.B.check(L.lcu_graph_destroy(graph))
    G.B.check(L.lcu_stream_destroy(stream))
    state.free()
    G.release()


@pytest.mark.parametrize("heads,ctx", [(32, 1024), (8, 640), (3, 1024), (24, 300)])
def test_decode_attention_wo_norm_equals_its_separate_operators(gpu, heads, ctx):
    """lcu_decode_attention_wo_norm (attention, x += att . Wo^T and the RMS norm behind it in one launch with
    in-launch hand-overs) against lcu_attention_decode + lcu_gemm_f16_nt (beta 1) + lcu_rmsnorm and against the
    kernel-order oracle, bit for bit: eager, captured and replayed with positions going up and down."""
    import ctypes as C
    G = gpu
    L = G.L()
    dim = heads * 128
    eps = 1e-5
    k, v = normal((ctx, dim), 0, 1300, 1.0), normal((ctx, dim), 0, 1301, 1.0)
    q, x0 = normal((1, dim), 0, 1302, 1.0), normal((1, dim), 0, 1303, 1.0)
    wo, nw = normal((dim, dim), 0, 1304, 0.02), normal((dim,), 1, 1305, 0.1)
    kd, vd, qd, wod, nwd = [G.dev_keep(a) for a in (k, v, q, wo, nw)]
    x_f, n_f = G.empty((1, dim)), G.empty((1, dim))       # fused
    x_s, n_s, att_s = G.empty((1, dim)), G.empty((1, dim)), G.empty((1, dim))  # separate
    stream = C.c_void_p()
    G.B.check(L.lcu_stream_create(C.byref(stream)))
    state = G.B.DeviceBuffer(8)
    def set_state(pos, seq):
        a = np.array([pos, seq], dtype=np.uint32)
        G.B.check(L.lcu_h2d(state.ptr, a.ctypes.data_as(C.c_void_p), 8, stream))
        for dst in (x_f, x_s):
            G.B.check(L.lcu_h2d(dst.ptr, x0.ctypes.data_as(C.c_void_p), x0.nbytes, stream))
        G.B.check(L.lcu_sync(stream))
    def fused():
        G.B.check(L.lcu_decode_attention_wo_norm(x_f.ptr, n_f.ptr, qd.ptr, kd.ptr, vd.ptr, wod.ptr, nwd.ptr, eps, state.ptr,
                                                 state.ptr + 4, 7, ctx, dim, heads, stream))
    def check(pos):
        G.B.check(L.lcu_attention_decode(att_s.ptr, qd.ptr, kd.ptr, vd.ptr, state.ptr, ctx, dim, heads, stream))
        G.B.check(L.lcu_gemm_f16_nt(x_s.ptr, att_s.ptr, wod.ptr, 1, dim, dim, 1.0, stream))
        G.B.check(L.lcu_rmsnorm(n_s.ptr, x_s.ptr, nwd.ptr, 1, dim, eps, stream))
        G.B.check(L.lcu_sync(stream))
        got_x, got_n = G.host(x_f, (1, dim)), G.host(n_f, (1, dim))
        assert G.ulp_mismatch(got_x, G.host(x_s, (1, dim))) == 0.0, pos
        assert G.ulp_mismatch(got_n, G.host(n_s, (1, dim))) == 0.0, pos
        T = pos + 1
        att = O.attention_decode_kernel_order(q, k[:T], v[:T], heads)
        want_x = O.matmul_nt(att, wo, flavour=2, beta=1.0, out=x0)
        assert G.ulp_mismatch(got_x, want_x) == 0.0, pos
        assert G.ulp_mismatch(got_n, O.rms_norm(want_x, nw, eps)) == 0.0, pos
    positions = [4, ctx - 1, 200, 0, ctx // 2, ctx - 2]
    set_state(positions[0], 1)
    fused()
    check(positions[0])
    set_state(positions[0], 2)
    G.B.check(L.lcu_graph_begin_capture(stream))
    fused()
    graph = C.c_void_p()
    G.B.check(L.lcu_graph_end_capture(stream, C.byref(graph)))
    for step, pos in enumerate(positions):
        set_state(pos, 3 + step)
        G.B.check(L.lcu_graph_launch(graph, stream))
        check(pos)
    count = C.c_uint(123)
    G.B.check(L.lcu_sync_timeouts(stream, C.byref(count)))
    assert count.value == 0
    assert L.lcu_decode_attention_wo_norm(x_f.ptr, n_f.ptr, qd.ptr, kd.ptr, vd.ptr, wod.ptr, nwd.ptr, eps, state.ptr,
                                          state.ptr + 4, 7, 1025, dim, heads, stream) == -2
    # more workgroups than compute units could not all be resident while they wait for one another
    assert L.lcu_decode_attention_wo_norm(x_f.ptr, n_f.ptr, qd.ptr, kd.ptr, vd.ptr, wod.ptr, nwd.ptr, eps, state.ptr,
                                          state.ptr + 4, 7, ctx, 52 * 128, 52, stream) == -2
    G.B.check(L.lcu_graph_destroy(graph))
    G.B.check(L.lcu_stream_destroy(stream))
    state.free()
    G.release()


@pytest.mark.parametrize("K,N,u8", [(11008, 4096, False), (17920, 6656, True), (4096, 4096, True), (2816, 1024, False),
                                    (512, 8, False), (1024, 8192, False)])
def test_decode_proj_norm_equals_its_separate_operators(gpu, K, N, u8):
    """lcu_decode_proj_norm (x += lhs . W^T and the RMS norm of the new x in one launch; an extra workgroup waits
    inside the launch for the rows) against lcu_gemm_* (beta 1) + lcu_rmsnorm and the kernel-order oracle, bit for
    bit, eager and replayed from a graph with the step counter changed between replays."""
    import ctypes as C
    G = gpu
    L = G.L()
    eps = 1e-6
    lhs = [normal((1, K), 0, 1400 + i, 1.0) for i in range(3)]
    x0 = normal((1, N), 0, 1410, 1.0)
    w, nw = normal((N, K), 0, 1411, 0.02), normal((N,), 1, 1412, 0.3)
    block = 128 if u8 else 0
    if u8:
        codes, scales = O.quantize_absmax_u8(w, block)
        wd, sd = G.dev_keep(codes), G.dev_keep(scales)
    else:
        wd, sd = G.dev_keep(w), None
    nwd = G.dev_keep(nw)
    lhs_d = G.empty((1, K))
    x_f, n_f, x_s, n_s = G.empty((1, N)), G.empty((1, N)), G.empty((1, N)), G.empty((1, N))
    stream = C.c_void_p()
    G.B.check(L.lcu_stream_create(C.byref(stream)))
    state = G.B.DeviceBuffer(8)
    def prepare(seq, which):
        a = np.array([0, seq], dtype=np.uint32)
        G.B.check(L.lcu_h2d(state.ptr, a.ctypes.data_as(C.c_void_p), 8, stream))
        G.B.check(L.lcu_h2d(lhs_d.ptr, lhs[which].ctypes.data_as(C.c_void_p), lhs[which].nbytes, stream))
        for dst in (x_f, x_s):
            G.B.check(L.lcu_h2d(dst.ptr, x0.ctypes.data_as(C.c_void_p), x0.nbytes, stream))
        G.B.check(L.lcu_sync(stream))
    def fused():
        G.B.check(L.lcu_decode_proj_norm(x_f.ptr, n_f.ptr, lhs_d.ptr, wd.ptr, sd.ptr if u8 else None, block, K, N, nwd.ptr,
                                         eps, state.ptr + 4, 3, stream))
    def check(which):
        if u8:
            G.B.check(L.lcu_gemm_f16u8_nt(x_s.ptr, lhs_d.ptr, wd.ptr, sd.ptr, 1, K, N, block, 1.0, stream))
        else:
            G.B.check(L.lcu_gemm_f16_nt(x_s.ptr, lhs_d.ptr, wd.ptr, 1, K, N, 1.0, stream))
        G.B.check(L.lcu_rmsnorm(n_s.ptr, x_s.ptr, nwd.ptr, 1, N, eps, stream))
        G.B.check(L.lcu_sync(stream))
        got_x, got_n = G.host(x_f, (1, N)), G.host(n_f, (1, N))
        assert G.ulp_mismatch(got_x, G.host(x_s, (1, N))) == 0.0, which
        assert G.ulp_mismatch(got_n, G.host(n_s, (1, N))) == 0.0, which
        if u8:
            want_x = O.matmul_nt_u8(lhs[which], codes, scales, block, beta=1.0, out=x0, flavour=2)
        else:
            want_x = O.matmul_nt(lhs[which], w, flavour=2, beta=1.0, out=x0)
        assert G.ulp_mismatch(got_x, want_x) == 0.0, which
        assert G.ulp_mismatch(got_n, O.rms_norm(want_x, nw, eps)) == 0.0, which
    prepare(1, 0)
    fused()
    check(0)
    prepare(2, 0)
    G.B.check(L.lcu_graph_begin_capture(stream))
    fused()
    graph = C.c_void_p()
    G.B.check(L.lcu_graph_end_capture(stream, C.byref(graph)))
    for step in range(4):
        prepare(3 + step, step % 3)
        G.B.check(L.lcu_graph_launch(graph, stream))
        check(step % 3)
    count = C.c_uint(123)
    G.B.check(L.lcu_sync_timeouts(stream, C.byref(count)))
    assert count.value == 0
    assert L.lcu_decode_proj_norm(x_f.ptr, n_f.ptr, lhs_d.ptr, wd.ptr, sd.ptr if u8 else None, block, K, 8200, nwd.ptr, eps,
                                  state.ptr + 4, 3, stream) == -2
    G.B.check(L.lcu_graph_destroy(graph))
    G.B.check(L.lcu_stream_destroy(stream))
    state.free()
    G.release()


@pytest.mark.parametrize("B,dim,heads,ffn,u8", [(8, 4096, 32, 11008, False), (8, 4096, 32, 11008, True), (33, 1024, 8, 2816, False),
                                                (3, 320, 2, 704, False), (1, 512, 4, 1408, True)])
def test_batch_fused_steps_equal_their_separate_operators(gpu, B, dim, heads, ffn, u8):
    """lcu_batch_qkv / lcu_batch_ffn_up / lcu_batch_proj_norm against the operators they fuse, bit for bit: on
    shapes that take the split-K path (partial sums added up by the fused kernel), on shapes that do not
    (dim 320: ragged K; one row) and with uint8 weights."""
    G = gpu
    L = G.L()
    VP = G.B.vp
    ctx, block = 16, (128 if u8 else 0)
    table = VP()
    G.B.check(L.lcu_rope_table_create(G.B.C.byref(table), ctx, dim // heads, 10000.0))
    pos = np.arange(B, dtype=np.int32) % ctx
    x = normal((B, dim), 0, 1700, 1.0)

    def weights(rows, cols, stream):
        w = normal((rows, cols), 0, stream, 0.02)
        if not u8:
            return G.dev_keep(w), None
        c, sc = O.quantize_absmax_u8(w, 128)
        return G.dev_keep(c), G.dev_keep(sc)

    def arr(items):
        return (VP * len(items))(*[(i.ptr if i is not None else None) for i in items])

    def caches():
        k = [G.dev_keep(np.zeros((ctx, dim), dtype=np.float16)) for _ in range(B)]
        v = [G.dev_keep(np.zeros((ctx, dim), dtype=np.float16)) for _ in range(B)]
        return k, v, G.dev_keep(np.array([d.ptr for d in k], dtype=np.uint64)), G.dev_keep(np.array([d.ptr for d in v], dtype=np.uint64))

    xd, pd = G.dev_keep(x), G.dev_keep(pos)
    # Wq, Wk, Wv + rotary + cache append
    qkv = [weights(dim, dim, 1701 + g) for g in range(3)]
    w_arr, s_arr = arr([w for w, _ in qkv]), arr([sc for _, sc in qkv])
    res = []
    for fused in (True, False):
        kc, vc, kptr, vptr = caches()
        q, kt, vt = G.empty((B, dim)), G.empty((B, dim)), G.empty((B, dim))
        if fused:
            G.B.check(L.lcu_batch_qkv(q.ptr, kt.ptr, vt.ptr, xd.ptr, w_arr, s_arr, block, B, dim, heads, kptr.ptr, vptr.ptr,
                                      pd.ptr, table, ctx, None))
        else:
            outs = arr([q, kt, vt])
            if u8:
                G.B.check(L.lcu_gemm_f16u8_nt_multi(outs, xd.ptr, w_arr, s_arr, 3, B, dim, dim, block, 0.0, None))
            else:
                G.B.check(L.lcu_gemm_f16_nt_multi(outs, xd.ptr, w_arr, 3, B, dim, dim, 0.0, None))
            G.B.check(L.lcu_rope_store_batch(q.ptr, kt.ptr, vt.ptr, kptr.ptr, vptr.ptr, pd.ptr, B, dim, heads, table, ctx, None))
        res.append([G.host(q, (B, dim))] + [G.host(c, (ctx, dim)) for c in kc + vc])
    for a, b in zip(*res):
        assert (a.view(np.uint16) == b.view(np.uint16)).all()
    assert np.abs(res[0][0].astype(np.float32)).max() > 0
    # W1, W3 + SiLU
    up = [weights(ffn, dim, 1710 + g) for g in range(2)]
    w_arr, s_arr = arr([w for w, _ in up]), arr([sc for _, sc in up])
    t1, t3, fused_out, sep_out = G.empty((B, ffn)), G.empty((B, ffn)), G.empty((B, ffn)), G.empty((B, ffn))
    G.B.check(L.lcu_batch_ffn_up(fused_out.ptr, t1.ptr, t3.ptr, xd.ptr, w_arr, s_arr, block, B, dim, ffn, None))
    outs = arr([t1, t3])
    if u8:
        G.B.check(L.lcu_gemm_f16u8_nt_multi(outs, xd.ptr, w_arr, s_arr, 2, B, dim, ffn, block, 0.0, None))
    else:
        G.B.check(L.lcu_gemm_f16_nt_multi(outs, xd.ptr, w_arr, 2, B, dim, ffn, 0.0, None))
    G.B.check(L.lcu_silu_mul(sep_out.ptr, t1.ptr, t3.ptr, B * ffn, None))
    assert (G.host(fused_out, (B, ffn)).view(np.uint16) == G.host(sep_out, (B, ffn)).view(np.uint16)).all()
    # W2 with the residual + the next norm
    h = normal((B, ffn), 0, 1720, 0.5)
    hd = G.dev_keep(h)
    w2, s2 = weights(dim, ffn, 1721)
    nw = G.dev_keep(normal((dim,), 0, 1722, 1.0))
    xa, xb, na, nb = G.dev(x), G.dev(x), G.empty((B, dim)), G.empty((B, dim))
    G.B.check(L.lcu_batch_proj_norm(xa.ptr, na.ptr, hd.ptr, w2.ptr, s2.ptr if s2 else None, block, B, ffn, dim, nw.ptr, 1e-6, None))
    if u8:
        G.B.check(L.lcu_gemm_f16u8_nt(xb.ptr, hd.ptr, w2.ptr, s2.ptr, B, ffn, dim, block, 1.0, None))
    else:
        G.B.check(L.lcu_gemm_f16_nt(xb.ptr, hd.ptr, w2.ptr, B, ffn, dim, 1.0, None))
    G.B.check(L.lcu_rmsnorm(nb.ptr, xb.ptr, nw.ptr, B, dim, 1e-6, None))
    assert (G.host(xa, (B, dim)).view(np.uint16) == G.host(xb, (B, dim)).view(np.uint16)).all()
    assert (G.host(na, (B, dim)).view(np.uint16) == G.host(nb, (B, dim)).view(np.uint16)).all()
    G.release()
    L.lcu_free(table)


@pytest.mark.parametrize("n", [1, 5, 1000, 1024, 32000, 32003])
def test_sample_row(gpu, n):
    # integer arithmetic on both sides: the drawn index must agree exactly
    G = gpu
    rng = np.random.default_rng(n)
    rows = [O.softmax_rows(normal((1, n), 0, 1300 + n, 2.0), 0.8)[0],          # a real distribution
            (rng.random(n) * 0.01).astype(np.float16),                         # does not sum to 1
            np.where(rng.random(n) < 0.9, 0, rng.random(n)).astype(np.float16)]  # mostly zeros
    special = (rng.random(n) * 0.5).astype(np.float16)
    special[::7] = np.float16(-1.0)
    special[::11] = np.float16(np.nan)
    special[n // 2] = np.float16(np.inf)
    rows.append(special)
    rows.append(np.zeros(n, dtype=np.float16))
    randoms = [0, 1, 2**63, 2**64 - 1] + [int(v) for v in rng.integers(0, 2**64, 12, dtype=np.uint64)]
    idx_d = G.empty((1,), np.int32)
    for p in rows:
        pd = G.dev_keep(p)
        for r in randoms:
            G.B.check(G.L().lcu_sample_row(idx_d.ptr, pd.ptr, n, r, None, None))
            assert int(G.host(idx_d, (1,), np.int32)[0]) == O.sample_row(p, r), (n, r)
    # the random bits read from device memory (what a captured launch does)
    r = randoms[-1]
    rd = G.dev_keep(np.array([r], dtype=np.uint64))
    G.B.check(G.L().lcu_sample_row(idx_d.ptr, G.dev_keep(rows[0]).ptr, n, 0, rd.ptr, None))
    assert int(G.host(idx_d, (1,), np.int32)[0]) == O.sample_row(rows[0], r)
    assert G.L().lcu_sample_row(idx_d.ptr, None, n, 0, None, None) == -2
    assert G.L().lcu_sample_row(idx_d.ptr, rd.ptr, 0, 0, None, None) == -2
    G.release()


def test_batch_step_operators(gpu):
    """The per-sequence parts of a batched decode step against their single-sequence forms, bit for bit:
    rotary + cache append with a position per row, attention over each sequence's own caches, softmax +
    argmax per row."""
    G = gpu
    L = G.L()
    dim, heads, ctx, B = 512, 4, 40, 3
    pos = np.array([17, 0, 39], dtype=np.int32)
    table = G.B.vp()
    G.B.check(L.lcu_rope_table_create(G.B.C.byref(table), ctx, dim // heads, 10000.0))
    q, k, v = normal((B, dim), 0, 1500, 1.0), normal((B, dim), 0, 1501, 1.0), normal((B, dim), 0, 1502, 1.0)
    kc = [normal((ctx, dim), 0, 1510 + b, 1.0) for b in range(B)]
    vc = [normal((ctx, dim), 0, 1520 + b, 1.0) for b in range(B)]
    kd, vd = [G.dev_keep(a) for a in kc], [G.dev_keep(a) for a in vc]
    kptr = G.dev_keep(np.array([d.ptr for d in kd], dtype=np.uint64))
    vptr = G.dev_keep(np.array([d.ptr for d in vd], dtype=np.uint64))
    qd, kn, vn, pd = G.dev_keep(q), G.dev_keep(k), G.dev_keep(v), G.dev_keep(pos)
    G.B.check(L.lcu_rope_store_batch(qd.ptr, kn.ptr, vn.ptr, kptr.ptr, vptr.ptr, pd.ptr, B, dim, heads, table, ctx, None))
    out_d = G.empty((B, dim))
    G.B.check(L.lcu_attention_decode_batch(out_d.ptr, qd.ptr, kptr.ptr, vptr.ptr, pd.ptr, B, ctx, dim, heads, None))
    q_rot, out = G.host(qd, (B, dim)), G.host(out_d, (B, dim))
    for b in range(B):
        p = int(pos[b])
        # single-sequence forms: lcu_rope on the row at its position, lcu_attention_decode on the caches
        row = G.empty((1, dim))
        G.B.check(L.lcu_rope(row.ptr, G.dev_keep(q[b:b + 1]).ptr, 1, dim, heads, p, table, ctx, None))
        assert (G.host(row, (1, dim)).view(np.uint16) == q_rot[b].view(np.uint16)).all()
        G.B.check(L.lcu_rope(row.ptr, G.dev_keep(k[b:b + 1]).ptr, 1, dim, heads, p, table, ctx, None))
        k_now, v_now = G.host(kd[b], (ctx, dim)), G.host(vd[b], (ctx, dim))
        assert (k_now[p].view(np.uint16) == G.host(row, (1, dim))[0].view(np.uint16)).all()
        assert (v_now[p].view(np.uint16) == v[b].view(np.uint16)).all()
        others = np.arange(ctx) != p
        assert (k_now[others].view(np.uint16) == kc[b][others].view(np.uint16)).all()
        one = G.empty((1, dim))
        G.B.check(L.lcu_attention_decode(one.ptr, G.dev_keep(q_rot[b:b + 1]).ptr, kd[b].ptr, vd[b].ptr,
                                         G.dev_keep(pos[b:b + 1]).ptr, ctx, dim, heads, None))
        assert (G.host(one, (1, dim))[0].view(np.uint16) == out[b].view(np.uint16)).all()
        # and the oracle on the same caches
        ref = O.attention(q_rot[b:b + 1], k_now[:p + 1], v_now[:p + 1], heads, p)
        assert G.max_abs_rel(out[b:b + 1], ref) <= TOL
    n = 1024
    x = normal((B, n), 0, 1530, 1.5)
    probs_d, idx_d = G.empty((B, n)), G.empty((B,), np.int32)
    G.B.check(L.lcu_softmax_argmax_rows(probs_d.ptr, idx_d.ptr, G.dev_keep(x).ptr, B, n, 0.8, None))
    probs, idx = G.host(probs_d, (B, n)), G.host(idx_d, (B,), np.int32)
    p1, i1 = G.empty((n,)), G.empty((1,), np.int32)
    for b in range(B):
        G.B.check(L.lcu_softmax_argmax(p1.ptr, i1.ptr, G.dev_keep(x[b:b + 1]).ptr, n, 0.8, None))
        assert (G.host(p1, (n,)).view(np.uint16) == probs[b].view(np.uint16)).all()
        assert int(G.host(i1, (1,), np.int32)[0]) == int(idx[b]) == O.argmax_first(probs[b])
    assert L.lcu_softmax_argmax_rows(probs_d.ptr, idx_d.ptr, G.dev_keep(x).ptr, B, 1001, 0.8, None) == -2
    assert L.lcu_attention_decode_batch(out_d.ptr, qd.ptr, kptr.ptr, vptr.ptr, pd.ptr, B, ctx, dim, 3, None) == -2
    G.release()


@pytest.mark.parametrize("n,temp", [(32000, 0.8), (32003, 0.9), (5, 1.0), (1024, 0.5)])
def test_softmax_argmax_fused(gpu, n, temp):
    G = gpu
    x = normal((1, n), 0, 1200, 1.3)
    x[0, n // 3] = x.max()  # two equal largest logits: the first index must win
    x[0, n // 3 * 2] = x.max()
    probs_d, idx_d = G.empty((n,)), G.empty((1,), np.int32)
    G.B.check(G.L().lcu_softmax_argmax(probs_d.ptr, idx_d.ptr, G.dev_keep(x).ptr, n, temp, None))
    got = G.host(probs_d, (1, n))
    ref = O.softmax_rows(x, temp)
    assert G.max_abs_rel(got, ref) <= TOL
    assert G.ulp_mismatch(got, ref) < 0.02
    if n % 8 == 0:  # the kernel's own association of the exponential sum, restated: every bit
        assert G.ulp_mismatch(got, O.softmax_logits_kernel_order(x[0], temp)) == 0.0
    assert int(G.host(idx_d, (1,), np.int32)[0]) == O.argmax_first(got) == int(np.flatnonzero(got[0] == got.max())[0])
    assert G.L().lcu_softmax_argmax(probs_d.ptr, idx_d.ptr, probs_d.ptr, n, temp, None) == -2
    G.release()


# more rows than the kernel of few rows takes: even and odd 64-blocks of K apart (one stage each, odd counts, ragged rows and columns, blocks of 64
# and 256 codes), too short a K for that, splits of large tiles and of 128 rows, a single chain, and a K that is no whole number of stages
@pytest.mark.parametrize("M,K,N,block", [(512, 4096, 4096, 0), (65, 128, 130, 0), (130, 384, 1030, 0), (511, 384, 2050, 0), (300, 1152, 1030, 64), (200, 2304, 4094, 256),
                                         (512, 11008, 4096, 0), (100, 11008, 4096, 128), (300, 5120, 8192, 128), (1000, 256, 8192, 0),
                                         (70, 320, 512, 0), (90, 256, 9000, 128)])
def test_product_residual_norm_of_many_rows(gpu, M, K, N, block):
    """lcu_batch_proj_norm against the product and the norm by themselves, bit for bit."""
    G = gpu
    check, L = G.B.check, G.L()
    x, lhs, w, nw = normal((M, N), 0, 1800, 1.0), normal((M, K), 0, 1801, 1.0), normal((N, K), 0, 1802, 0.02), normal((N,), 0, 1803, 1.0)
    wd = [G.dev_keep(part) for part in (O.quantize_absmax_u8(w, block) if block else (w,))]
    ld, nd = G.dev_keep(lhs), G.dev_keep(nw)
    xa, xb, na, nb = G.dev(x), G.dev(x), G.empty((M, N)), G.empty((M, N))
    check(L.lcu_batch_proj_norm(xa.ptr, na.ptr, ld.ptr, wd[0].ptr, wd[1].ptr if block else None, block, M, K, N, nd.ptr, 1e-6, None))
    if block:
        check(L.lcu_gemm_f16u8_nt(xb.ptr, ld.ptr, wd[0].ptr, wd[1].ptr, M, K, N, block, 1.0, None))
    else:
        check(L.lcu_gemm_f16_nt(xb.ptr, ld.ptr, wd[0].ptr, M, K, N, 1.0, None))
    check(L.lcu_rmsnorm(nb.ptr, xb.ptr, nd.ptr, M, N, 1e-6, None))
    assert (G.host(xa, (M, N)).view(np.uint16) == G.host(xb, (M, N)).view(np.uint16)).all()
    assert (G.host(na, (M, N)).view(np.uint16) == G.host(nb, (M, N)).view(np.uint16)).all()
    G.release()


@pytest.mark.parametrize("M,K,N,block", [(512, 4096, 4096, 0), (65, 128, 130, 0), (130, 384, 1030, 0), (511, 384, 2050, 0), (300, 1152, 1030, 64), (200, 2304, 4094, 256),
                                         (512, 11008, 4096, 0), (90, 4096, 4096, 128)])
def test_product_residual_norm_on_a_stream_of_its_own(gpu, M, K, N, block):
    """The same where the even and the odd stages are summed apart and added up by the norm's launch."""
    G = gpu
    check, L = G.B.check, G.L()
    stream = G.B.vp()
    check(L.lcu_stream_create(G.B.C.byref(stream)))
    x, lhs, w, nw = normal((M, N), 0, 1810, 1.0), normal((M, K), 0, 1811, 1.0), normal((N, K), 0, 1812, 0.02), normal((N,), 0, 1813, 1.0)
    wd = [G.dev_keep(part) for part in (O.quantize_absmax_u8(w, block) if block else (w,))]
    ld, nd = G.dev_keep(lhs), G.dev_keep(nw)
    xs, ns = [G.dev_keep(x) for _ in range(3)], [G.empty((M, N)) for _ in range(3)]
    for at, s in ((0, None), (1, stream)):
        check(L.lcu_batch_proj_norm(xs[at].ptr, ns[at].ptr, ld.ptr, wd[0].ptr, wd[1].ptr if block else None, block, M, K, N, nd.ptr, 1e-6, s))
    if block:
        check(L.lcu_gemm_f16u8_nt(xs[2].ptr, ld.ptr, wd[0].ptr, wd[1].ptr, M, K, N, block, 1.0, None))
    else:
        check(L.lcu_gemm_f16_nt(xs[2].ptr, ld.ptr, wd[0].ptr, M, K, N, 1.0, None))
    check(L.lcu_rmsnorm(ns[2].ptr, xs[2].ptr, nd.ptr, M, N, 1e-6, None))
    check(L.lcu_sync(stream))
    for got in (xs, ns):
        a, b, c = (G.host(t, (M, N)).view(np.uint16) for t in got)
        assert (a == c).all() and (b == c).all()
    G.release()
    check(L.lcu_stream_destroy(stream))


def test_product_residual_norm_overlaps_on_foreign_streams(gpu):
    """Two streams made elsewhere share the device's workspace; products whose kernel needs none may overlap on them."""
    import gemm_plan
    G = gpu
    C, check, L = G.B.C, G.B.check, G.L()
    hip = C.CDLL("libamdhip64.so")
    streams = [G.B.vp(), G.B.vp()]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    M, K, N, times = 200, 2048, 2048, 12
    assert gemm_plan.left_sums(M, K, N) == (2, 2) and gemm_plan.left_sums(M, K, N, owned=False) == (0, 1)
    nd = G.dev_keep(normal((N,), 0, 1823, 1.0))
    sides = []
    for t in range(2):
        x, lhs, w = normal((M, N), 0, 1820 + 10 * t, 1.0), G.dev_keep(normal((M, K), 0, 1821 + 10 * t, 1.0)), G.dev_keep(normal((N, K), 0, 1822 + 10 * t, 0.02))
        sides.append((lhs, w, [G.dev_keep(x) for _ in range(times + 1)], [G.empty((M, N)) for _ in range(times + 1)]))
    run = lambda t, i, s: check(L.lcu_batch_proj_norm(sides[t][2][i].ptr, sides[t][3][i].ptr, sides[t][0].ptr, sides[t][1].ptr, None, 0, M, K, N, nd.ptr, 1e-6, s))
    for t in range(2):
        run(t, times, None)
    G.sync()
    for i in range(times):
        for t in range(2):
            run(t, i, streams[t])
    G.sync()
    for _, _, xs, ns in sides:
        for got in (xs, ns):
            want = G.host(got[-1], (M, N)).view(np.uint16)
            assert all((G.host(o, (M, N)).view(np.uint16) == want).all() for o in got[:-1])
    G.release()
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0


# split sums of few rows (two kernels), tiles of 128 and 256 rows, ragged rows; kernels without a rotation of their
# own (half stages apart, K no whole number of stages, blocks of 96 codes), one row
@pytest.mark.parametrize("rows,dim,heads,first,block", [(24, 512, 4, 0, 0), (45, 4096, 32, 7, 0), (64, 1024, 8, 3, 128), (512, 4096, 32, 0, 0), (301, 4096, 32, 100, 0),
                                                        (700, 2048, 16, 9, 0), (1000, 4096, 32, 20, 0), (512, 6656, 52, 0, 128), (1500, 6656, 52, 11, 128),
                                                        (1500, 5120, 40, 0, 0), (200, 4096, 32, 1, 128), (100, 4096, 32, 5, 0), (90, 320, 2, 4, 0),
                                                        (300, 1152, 9, 2, 96), (1, 512, 4, 6, 0), (260, 3200, 100, 2, 128)])
def test_prompt_qkv(gpu, rows, dim, heads, first, block):
    """lcu_prompt_qkv against the products and lcu_rope_pair, bit for bit."""
    G = gpu
    check, L, VP = G.B.check, G.L(), G.B.vp
    table = VP()
    check(L.lcu_rope_table_create(G.B.C.byref(table), first + rows, dim // heads, 10000.0))
    x, ws = G.dev_keep(normal((rows, dim), 0, 1900, 1.0)), [normal((dim, dim), 0, 1901 + g, 0.02) for g in range(3)]
    wd = [[G.dev_keep(part) for part in (O.quantize_absmax_u8(w, block) if block else (w,))] for w in ws]
    w_arr, s_arr = (VP * 3)(*[w[0].ptr for w in wd]), (VP * 3)(*[w[1].ptr for w in wd]) if block else None
    outs, seps = [G.empty((rows, dim)) for _ in range(3)], [G.empty((rows, dim)) for _ in range(3)]
    check(L.lcu_prompt_qkv(outs[0].ptr, outs[1].ptr, outs[2].ptr, x.ptr, w_arr, s_arr, block, rows, dim, heads, first, table, first + rows, None))
    arr = (VP * 3)(*[o.ptr for o in seps])
    if block:
        check(L.lcu_gemm_f16u8_nt_multi(arr, x.ptr, w_arr, s_arr, 3, rows, dim, dim, block, 0.0, None))
    else:
        check(L.lcu_gemm_f16_nt_multi(arr, x.ptr, w_arr, 3, rows, dim, dim, 0.0, None))
    check(L.lcu_rope_pair(seps[0].ptr, seps[1].ptr, rows, dim, heads, first, table, first + rows, None))
    for a, b in zip(outs, seps):
        assert (G.host(a, (rows, dim)).view(np.uint16) == G.host(b, (rows, dim)).view(np.uint16)).all()
    assert L.lcu_prompt_qkv(outs[0].ptr, outs[1].ptr, outs[2].ptr, x.ptr, w_arr, s_arr, block, rows, dim, heads, first + 1, table, first + rows, None) == -2
    G.release()
    L.lcu_free(table)


# values' last columns in a launch of their own, which must not rotate them; from a column inside a head, ragged rows
@pytest.mark.parametrize("rows,dim,heads,first,block", [(1300, 4096, 32, 5, 0), (1300, 4096, 32, 0, 128), (800, 6656, 52, 3, 0), (801, 6656, 52, 3, 128)])
def test_prompt_qkv_columns_left_of_whole_rounds(gpu, rows, dim, heads, first, block):
    import gemm_plan
    columns, _, at, _, _ = gemm_plan.large("u8" if block else "f16", rows, dim, dim, 3)
    assert 0 < at < dim and gemm_plan.rows(rows, dim, dim, 3)[0] == "large"
    test_prompt_qkv(gpu, rows, dim, heads, first, block)
