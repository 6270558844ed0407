"""What a one-token step takes from the host: page-locked words that its first launch reads and copies to the device."""
import ctypes as C

import numpy as np
import pytest

from layered_helpers import BF16, F32, call, get, gpu, put, rounded, up64, zeros  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture
def words(gpu):
    """Page-locked memory as an array of 256 int32."""
    p = C.c_void_p()
    gpu.B.check(gpu.L().lcu_host_alloc(C.byref(p), 1024))
    yield np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_int32)), (256,))
    gpu.B.check(gpu.L().lcu_sync(gpu.stream))
    gpu.B.check(gpu.L().lcu_host_free(p))


def test_small_pieces_of_page_locked_memory(gpu):
    """More than a page of them: apart, zero, written by the device one by one, and taken anew after some have gone back."""
    L, check = gpu.L(), gpu.B.check

    def take(n):
        out = [C.c_void_p() for _ in range(n)]
        for p in out:
            check(L.lcu_host_alloc(C.byref(p), 64))
        return out

    def view(p):
        return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_int32)), (16,))

    pieces, source = take(150), gpu.dev_keep(np.arange(150, dtype=np.float32))
    for _ in range(2):
        at = sorted(p.value for p in pieces)
        assert all(b - a >= 64 for a, b in zip(at, at[1:])) and all(a % 64 == 0 for a in at)
        assert all((view(p) == 0).all() for p in pieces)
        for i, p in enumerate(pieces):
            check(L.lcu_argmax_f32(p, source.ptr, i + 1, gpu.stream))
        check(L.lcu_sync(gpu.stream))
        assert all(view(p)[0] == i and (view(p)[1:] == 0).all() for i, p in enumerate(pieces))
        for p in pieces[::2] + pieces[1:100:2]:
            check(L.lcu_host_free(p))
        kept = pieces[101::2]
        for p in kept:
            view(p)[:] = 0
        pieces = take(150 - len(kept)) + kept
    for p in pieces:
        check(L.lcu_host_free(p))
    gpu.release()


@pytest.mark.parametrize("n", [1, 6, 255, 256])
def test_fetched_words(gpu, words, n):
    words[:] = np.random.default_rng(n).integers(-2**31, 2**31, 256)
    out = zeros(gpu, 256)
    call(gpu, "lcu_fetch", out, words.ctypes.data, 4 * n)
    gpu.B.check(gpu.L().lcu_sync(gpu.stream))
    assert np.array_equal(gpu.host(out, (256,), np.int32), np.where(np.arange(256) < n, words, 0))
    assert gpu.L().lcu_fetch(out.ptr, words.ctypes.data, 6, gpu.stream) == -2
    gpu.release()


@pytest.mark.parametrize("dim,block,state", [(8, 0, 2), (512, 0, 6), (8192, 0, 256), (1024, 128, 6)])
def test_embedding_with_the_steps_state(gpu, words, dim, block, state):
    """The bits of lcu_embed_rmsnorm, and the state on the device."""
    rng = np.random.default_rng(dim)
    words[:] = rng.integers(-2**31, 2**31, 256)
    words[1] = 5
    ids, out = gpu.dev_keep(np.array([5], np.int16)), zeros(gpu, 256)
    table = gpu.dev_keep(rng.integers(0, 256, (9, dim)).astype(np.uint8) if block else rng.standard_normal((9, dim)).astype(np.float16))
    scales = gpu.dev_keep((0.01 * rng.random((9, max(1, dim // 128)))).astype(np.float16)) if block else None
    w = gpu.dev_keep(rng.standard_normal(dim).astype(np.float16))
    results = []
    for step in (False, True):
        x, h = (gpu.dev_keep(np.zeros(dim, np.float16)) for _ in range(2))
        if step:
            call(gpu, "lcu_step_embed_rmsnorm", out, words.ctypes.data, 4 * state, x, h, words.ctypes.data + 4, dim, table, scales, block, 9, w, 1e-6)
        else:
            call(gpu, "lcu_embed_rmsnorm", x, h, ids, 1, dim, table, scales, block, 9, w, 1e-6)
        gpu.B.check(gpu.L().lcu_sync(gpu.stream))
        results.append([gpu.host(b, (dim,), np.uint16) for b in (x, h)])
    assert all(np.array_equal(a, b) for a, b in zip(*results))
    assert np.array_equal(gpu.host(out, (256,), np.int32), np.where(np.arange(256) < state, words, 0))
    assert gpu.L().lcu_step_embed_rmsnorm(out.ptr, words.ctypes.data, 1028, x.ptr, h.ptr, words.ctypes.data, dim, table.ptr,
                                          scales.ptr if block else None, block, 9, w.ptr, 1e-6, gpu.stream) == -2
    gpu.release()


@pytest.mark.parametrize("width,learned", [(70, False), (4200, False), (960, True)])
def test_layered_embedding_with_the_steps_state(gpu, words, width, learned):
    """The bits of lcu_embed_scaled and lcu_embed_pos_norm at position 3, and position and id on the device."""
    rng = np.random.default_rng(width)
    ld = up64(width)
    padded = lambda a: np.pad(a, [(0, 0)] * (a.ndim - 1) + [(0, ld - width)])
    words[:2] = 3, 5
    pair, out = gpu.dev_keep(words[:2].copy()), zeros(gpu, 2)
    table, pos = (put(gpu, padded(rounded(rng.standard_normal((9, width)))), BF16) for _ in range(2))
    w1, w2 = (put(gpu, padded(rng.standard_normal(width))) for _ in range(2))
    shape = (w2, BF16, width, ld, 1, 1e-5)
    results = []
    for step in (False, True):
        x, h = zeros(gpu, ld), zeros(gpu, ld, BF16)
        if step:
            call(gpu, "lcu_step_embed", out, words.ctypes.data, x, h, table, 9, 2.5, *((pos, 9, w1) if learned else (None, 0, None)), *shape)
        elif learned:
            call(gpu, "lcu_embed_pos_norm", x, h, pair.ptr + 4, 1, table, 9, pos, 9, pair, w1, *shape)
        else:
            call(gpu, "lcu_embed_scaled", x, h, pair.ptr + 4, 1, table, 9, 2.5, *shape)
        results.append([get(gpu, x, (ld,), F32), get(gpu, h, (ld,), BF16)])
    assert all(np.array_equal(a, b) for a, b in zip(*results))
    assert np.array_equal(gpu.host(out, (2,), np.int32), words[:2])
    gpu.release()


@pytest.mark.parametrize("kind", ["fp16", "uint8", "layered", "batch"])
def test_a_calls_token_is_its_own(gpu, kind):
    """What a call returns is read as soon as it is there: after every one of many calls, short prompts and captured steps in turn, it is the first
    maximum of what that call left, and a context used again gives the same."""
    P = gpu.P
    if kind == "layered":
        model = P.Model(config={"architecture": "Logivik", "vocab": 301, "width": 64, "embedding": {"scale": 8.0}, "norm": {"eps": 1e-5}, "layers": [
            {"type": "latent_attention_2", "mlp": {"kind": "dense", "ff": 128},
             "mixer": {"heads": 2, "dim": 32, "vdim": 32, "kv_rank": 32, "q_rank": 32, "scale": 0.2, "mask": {"size": 64}}}]}, seed=4)
    else:
        model = P.Model(dim=256, multiple_of=128, n_heads=2, n_layers=1, n_vocab=512, seed=5, weight_std=0.05, q_type=int(kind == "uint8"), qblock=128)
    ctx = P.BatchContext(model, 3, context_len=96) if kind == "batch" else P.Context(model, context_len=96)
    ids = np.random.default_rng(1).integers(0, 301, 200).astype(np.int16)
    runs = []
    for _ in range(2):
        seen = []
        for b in range(3):
            ctx.clear_tokens(*([b] if kind == "batch" else []))
            if kind == "batch":
                ctx.next_token(b, ids[b:b + 2])
        for step in range(30):
            if kind == "batch":
                token = list(ctx.next_tokens(ids[3 * step:3 * step + 3]))
                rows = ctx.probs().reshape(3, -1)
            else:
                token = [ctx.next_token(ids[5 * step:5 * step + (3 if step % 7 == 3 else 1)])]
                rows = ctx.probs().reshape(1, -1)
            if kind != "layered":  # whose token is that of the fp32 logits: fp16 probabilities may tie
                assert token == [int(i) for i in rows.argmax(1)]
            assert all(rows[i, t] == rows[i].max() for i, t in enumerate(token))
            seen.append(token)
        runs.append(seen)
    assert runs[0] == runs[1] and len({tuple(t) for t in runs[0]}) > 3
    ctx.close()
    model.close()
