"""The general grouped kernel (k_grouped_rows): MUL_MAT_ID and layers over
many tokens, for every format it takes, at row counts and k that leave
partial tiles and a partial last step.

Its integer block sums are exact and its fp32 steps are the token-major
kernels' in their order, so the bar is bit-identity with the token-major path
(grouping off, or sabah_moe_layer_noalloc), and the oracle's parity bar.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from helpers import assert_bits_equal, assert_parity, random_blocks, token_major_layer

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q5_K, Q6_K, IQ3_XXS, IQ4_NL, IQ3_S, IQ4_XS = 8, 12, 13, 14, 18, 20, 21, 23
DEV = torch.device("cuda:0")
AUTO, NEVER, ALWAYS = 0, 1, 2


def T(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def vp(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.fixture
def grouping(hip_rt):
    lib = hip_rt.lib()

    def set_mode(mode):
        hip_rt.check(lib.sabah_rt_set_mmid_grouping(mode), "set grouping")

    yield set_mode
    set_mode(AUTO)


def bank_bytes(rng, qt, E, rows, k, scale=0.05):
    raw = random_blocks(rng, qt, E * rows, k)
    return raw.reshape(E, rows, -1)


def mmid(hip_rt, bank, qt, rows, k, E, x, ids, grouped):
    lib = hip_rt.lib()
    rb = hip_rt.row_bytes(qt, k)
    out = torch.full((ids.shape[0], ids.shape[1], rows), 7.0, dtype=torch.float32, device=DEV)
    before = hip_rt.snapshot()["grouped_calls"]
    hip_rt.check(lib.sabah_rt_mul_mat_id_v2(
        vp(bank), ctypes.c_size_t(rows * rb), ctypes.c_size_t(rb),
        vp(x), ctypes.c_size_t(x.stride(1) * 4), x.shape[1], ctypes.c_size_t(x.stride(0) * 4),
        vp(ids), ctypes.c_size_t(4), ctypes.c_size_t(ids.stride(0) * 4), ids.shape[1], ids.shape[0],
        vp(out), ctypes.c_size_t(out.stride(1) * 4), ctypes.c_size_t(out.stride(0) * 4), rows, k, E, qt,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), None), "v2")
    torch.cuda.synchronize()
    assert hip_rt.snapshot()["grouped_calls"] == before + int(grouped)
    return out.cpu().numpy()


# (k, rows, tokens): rows below, at and past a 64-row tile, one and several
# steps of k; 2 tokens leave most experts one pair, 40 give a heavy expert three
# or more pair tiles (two items); 6200 rows make 90 tokens' items four-tile ones, 13240
# rows give each wave two row groups
SHAPES = [(256, 17, 2), (768, 64, 40), (1280, 130, 40), (2560, 96, 90), (512, 6200, 90), (256, 13240, 40)]
# formats of 32-element blocks: k past a whole 256-step as well
ODD_K = [(32, 64, 40), (288, 65, 2), (992, 48, 90)]


@pytest.mark.parametrize("qt,k,rows,tokens",
                         [(qt, *s) for qt in (Q8_0, Q4_K, Q5_K, Q6_K, IQ3_XXS, IQ4_NL, IQ3_S, IQ4_XS) for s in SHAPES]
                         + [(qt, *s) for qt in (Q8_0, IQ4_NL) for s in ODD_K])
@pytest.mark.parametrize("slot_rows", [False, True])
def test_grouped_rows_is_bit_identical_to_token_major(hip_rt, orc, grouping, qt, k, rows, tokens, slot_rows):
    E, K = 7, 3
    rng = np.random.default_rng(qt * 1000 + k + rows + tokens + slot_rows)
    raw = bank_bytes(rng, qt, E, rows, k)
    ids = np.stack([rng.choice(E - 1, K, replace=False) for _ in range(tokens)]).astype(np.int32)
    ids[:, 0] = 2                                    # a heavy expert; expert E - 1 has no pair
    ids[1, 2] = ids[1, 0]                            # a duplicate
    x = rng.standard_normal((tokens, K if slot_rows else 1, k)).astype(np.float32)
    x[0, 0, :min(k, 256)] = 0.0                      # a block of zeros
    bank, xd, idd = T(raw), T(x), T(ids)
    grouping(ALWAYS)
    got = mmid(hip_rt, bank, qt, rows, k, E, xd, idd, grouped=True)
    grouping(NEVER)
    tok = mmid(hip_rt, bank, qt, rows, k, E, xd, idd, grouped=False)
    assert_bits_equal(got, tok, "qt=%d k=%d rows=%d tokens=%d" % (qt, k, rows, tokens))
    if rows <= 130 and tokens <= 40 and not slot_rows:
        assert_parity(got, orc.mul_mat_id(raw, x, ids, rows, k, qt), "oracle qt=%d k=%d" % (qt, k))


def test_a_bad_id_becomes_nan_and_is_reported(hip_rt, grouping):
    E, K, rows, k, tokens = 7, 3, 40, 256, 20
    rng = np.random.default_rng(5)
    raw = bank_bytes(rng, Q8_0, E, rows, k)
    ids = rng.integers(0, E, (tokens, K)).astype(np.int32)
    bad = ids.copy()
    bad[4, 1] = E
    x = T(rng.standard_normal((tokens, 1, k)).astype(np.float32))
    bank = T(raw)
    grouping(ALWAYS)
    want = mmid(hip_rt, bank, Q8_0, rows, k, E, x, T(ids), grouped=True)
    got = mmid(hip_rt, bank, Q8_0, rows, k, E, x, T(bad), grouped=True)
    assert np.isnan(got[4, 1]).all()
    got[4, 1] = want[4, 1]
    assert_bits_equal(got, want, "the other slots")
    assert hip_rt.lib().sabah_rt_check_errors() == -1
    assert hip_rt.lib().sabah_rt_check_errors() == 0


def test_calls_on_two_streams_and_under_capture(hip_rt, grouping):
    """Two streams' calls overlap with workspaces of their own, and a captured
    call (token-major) replays beside them."""
    E, K, rows, k, tokens = 7, 2, 960, 768, 200
    rng = np.random.default_rng(6)
    bank = T(bank_bytes(rng, IQ3_XXS, E, rows, k))
    xs = [T(rng.standard_normal((tokens, 1, k)).astype(np.float32)) for _ in range(2)]
    ids = [T(rng.integers(0, E, (tokens, K)).astype(np.int32)) for _ in range(2)]
    grouping(NEVER)
    want = [mmid(hip_rt, bank, IQ3_XXS, rows, k, E, xs[i], ids[i], grouped=False) for i in range(2)]
    grouping(AUTO)
    lib, rb = hip_rt.lib(), hip_rt.row_bytes(IQ3_XXS, k)
    outs = [torch.empty(tokens, K, rows, device=DEV) for _ in range(3)]

    def call(i, out, stream):
        hip_rt.check(lib.sabah_rt_mul_mat_id_v2(
            vp(bank), ctypes.c_size_t(rows * rb), ctypes.c_size_t(rb), vp(xs[i]), ctypes.c_size_t(k * 4), 1,
            ctypes.c_size_t(k * 4), vp(ids[i]), ctypes.c_size_t(4), ctypes.c_size_t(K * 4), K, tokens, vp(out),
            ctypes.c_size_t(rows * 4), ctypes.c_size_t(K * rows * 4), rows, k, E, IQ3_XXS,
            ctypes.c_void_p(stream.cuda_stream), None), "v2")

    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    before = hip_rt.snapshot()["grouped_calls"]
    with torch.cuda.graph(graph):
        call(0, outs[2], torch.cuda.current_stream())
    assert hip_rt.snapshot()["grouped_calls"] == before
    for _ in range(10):
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        graph.replay()
        for i in range(2):
            call(i, outs[i], streams[i])
        torch.cuda.synchronize()
        for got, i in zip(outs, (0, 1, 0)):
            assert_bits_equal(got.cpu().numpy(), want[i], "stream %d" % i)
    assert hip_rt.snapshot()["grouped_calls"] == before + 20


# Over 8 experts a launch of few pairs is k / 256 dependent steps whatever their
# number: the token-major kernels keep the calls below the line, by shape
@pytest.mark.parametrize("qt,k,rows,tokens,grouped", [
    (IQ4_XS, 2560, 640, 27, False), (IQ4_XS, 2560, 640, 60, True), (Q8_0, 2048, 768, 28, False),
    (Q8_0, 2048, 768, 50, True), (IQ3_XXS, 4096, 1536, 16, False), (IQ3_XXS, 4096, 1536, 40, True),
    (IQ4_XS, 4096, 1536, 9, False), (Q6_K, 2560, 640, 27, False)])
def test_few_pairs_over_few_experts_stay_token_major(hip_rt, grouping, qt, k, rows, tokens, grouped):
    E, K = 8, 2
    rng = np.random.default_rng(qt + k)
    bank = T(bank_bytes(rng, qt, E, rows, k))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    x = T(rng.standard_normal((tokens, 1, k)).astype(np.float32))
    grouping(AUTO)
    got = mmid(hip_rt, bank, qt, rows, k, E, x, ids, grouped=grouped)
    grouping(NEVER)
    assert_bits_equal(got, mmid(hip_rt, bank, qt, rows, k, E, x, ids, grouped=False), "qt=%d" % qt)


def hip_runtime():
    """The HIP runtime this process runs on."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(l.split()[-1] for l in f if "libamdhip64" in l))


@pytest.mark.parametrize("kind", ["twelve", "created and destroyed", "per thread"])
def test_more_streams_than_workspaces(hip_rt, grouping, kind):
    """Eight workspaces serve any number of streams: a further stream takes over
    the least recently used one, in order after its last call, and a
    destroyed stream holds none.  The per-thread default stream (one handle for every
    thread) is served token-major."""
    E, K, rows, k = 7, 2, 960, 768
    rng = np.random.default_rng(61)
    bank = T(bank_bytes(rng, IQ3_XXS, E, rows, k))
    lib, rb = hip_rt.lib(), hip_rt.row_bytes(IQ3_XXS, k)
    tokens = [200, 130, 333, 150]
    xs = [T(rng.standard_normal((t, 1, k)).astype(np.float32)) for t in tokens]
    ids = [T(rng.integers(0, E, (t, K)).astype(np.int32)) for t in tokens]
    grouping(NEVER)
    want = [mmid(hip_rt, bank, IQ3_XXS, rows, k, E, x, i, grouped=False) for x, i in zip(xs, ids)]
    grouping(AUTO)

    def call(i, out, handle):
        hip_rt.check(lib.sabah_rt_mul_mat_id_v2(
            vp(bank), ctypes.c_size_t(rows * rb), ctypes.c_size_t(rb), vp(xs[i]), ctypes.c_size_t(k * 4), 1,
            ctypes.c_size_t(k * 4), vp(ids[i]), ctypes.c_size_t(4), ctypes.c_size_t(K * 4), K, tokens[i], vp(out),
            ctypes.c_size_t(rows * 4), ctypes.c_size_t(K * rows * 4), rows, k, E, IQ3_XXS,
            ctypes.c_void_p(handle), None), "v2")

    n = 36
    outs = [torch.zeros(tokens[j % 4], K, rows, device=DEV) for j in range(n)]
    streams = [torch.cuda.Stream() for _ in range(12)]
    torch.cuda.synchronize()
    before = hip_rt.snapshot()["grouped_calls"]
    hip = hip_runtime()
    for j in range(n):                                  # back to back: nothing waits on the host
        if kind == "twelve":
            call(j % 4, outs[j], streams[j % 12].cuda_stream)
        elif kind == "per thread":
            call(j % 4, outs[j], 2)                     # hipStreamPerThread
        else:
            h = ctypes.c_void_p()
            assert hip.hipStreamCreateWithFlags(ctypes.byref(h), 1) == 0
            call(j % 4, outs[j], h.value)
            assert hip.hipStreamDestroy(h) == 0
    torch.cuda.synchronize()
    assert hip_rt.snapshot()["grouped_calls"] == before + (0 if kind == "per thread" else n)
    for j in range(n):
        assert_bits_equal(outs[j].cpu().numpy(), want[j % 4], "call %d" % j)


def test_a_call_that_allocates_beside_another_streams_capture(hip_rt, grouping):
    """A first call on its stream, whose workspace has to be allocated, while another
    stream is being captured: both go through."""
    E, K, rows, k, tokens = 7, 2, 960, 768, 20000      # larger than the other tests' workspaces
    rng = np.random.default_rng(62)
    bank = T(bank_bytes(rng, IQ3_XXS, E, rows, k))
    lib, rb = hip_rt.lib(), hip_rt.row_bytes(IQ3_XXS, k)
    x = T(rng.standard_normal((tokens, 1, k)).astype(np.float32))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    grouping(NEVER)
    want = mmid(hip_rt, bank, IQ3_XXS, rows, k, E, x, ids, grouped=False)
    grouping(AUTO)
    out = torch.zeros(tokens, K, rows, device=DEV)
    other, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    a, b = torch.ones(1000, device=DEV), torch.zeros(1000, device=DEV)
    torch.cuda.synchronize()
    before = hip_rt.snapshot()
    with torch.cuda.graph(graph):
        torch.add(a, 1.0, out=b)
        hip_rt.check(lib.sabah_rt_mul_mat_id_v2(
            vp(bank), ctypes.c_size_t(rows * rb), ctypes.c_size_t(rb), vp(x), ctypes.c_size_t(k * 4), 1,
            ctypes.c_size_t(k * 4), vp(ids), ctypes.c_size_t(4), ctypes.c_size_t(K * 4), K, tokens, vp(out),
            ctypes.c_size_t(rows * 4), ctypes.c_size_t(K * rows * 4), rows, k, E, IQ3_XXS,
            ctypes.c_void_p(other.cuda_stream), None), "v2")
    torch.cuda.synchronize()
    after = hip_rt.snapshot()
    assert after["grouped_calls"] == before["grouped_calls"] + 1
    assert after["scratch_bytes"] > before["scratch_bytes"]
    assert_bits_equal(out.cpu().numpy(), want, "the eager call")
    for _ in range(3):
        b.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert (b == 2.0).all()


def grouped_launches(hip_rt):
    """Group-major gate/up launches (kernel kind 4) since the last reading, with timing on."""
    ms, n = ctypes.c_double(), ctypes.c_ulonglong()
    hip_rt.check(hip_rt.lib().sabah_rt_get_kernel_timing(4, ctypes.byref(ms), ctypes.byref(n), 1), "timing")
    return n.value


def layer(hip_rt, fn, desc, x, ids, w, resid=None):
    out = torch.full_like(x, float("nan"))
    hip_rt.check(getattr(hip_rt.lib(), fn)(
        ctypes.byref(desc), vp(x), vp(ids), vp(w), ids.shape[1], ids.shape[0], vp(out),
        vp(resid) if resid is not None else None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), fn)
    torch.cuda.synchronize()
    return out.cpu().numpy()


# the tokens are the fewest that take the grouped form at the shape, and more; 16640 rows give
# each wave of the down kernel two row groups
LAYERS = [(IQ3_XXS, IQ4_NL, 2560, 640, (28, 61)), (Q8_0, Q8_0, 288, 96, (912, 1001)), (Q5_K, IQ4_XS, 512, 256, (194, 301)),
          (Q4_K, Q6_K, 256, 1280, (93, 150)), (Q6_K, Q8_0, 768, 352, (95, 150)), (IQ3_S, IQ3_S, 512, 512, (182, 301)),
          (IQ3_XXS, IQ4_NL, 16640, 64, (42, 61))]


@pytest.mark.parametrize("qtg,qtd,D,F,tokens", [(*c[:4], t) for c in LAYERS for t in c[4]])
def test_grouped_layer_is_bit_identical_to_token_major(hip_rt, qtg, qtd, D, F, tokens):
    from sabah.runtime import rt
    E, K = 6, 2
    rng = np.random.default_rng(qtg + qtd + D + tokens)
    banks = [T(bank_bytes(rng, q, E, rows, k)) for q, rows, k in ((qtg, F, D), (qtg, F, D), (qtd, D, F))]
    desc = rt.MoeLayerDesc()
    desc.gate, desc.up, desc.down = (b.data_ptr() for b in banks)
    desc.qt_gate = desc.qt_up = qtg
    desc.qt_down = qtd
    desc.d_model, desc.d_ff, desc.n_experts = D, F, E
    x = T(0.05 * rng.standard_normal((tokens, D)).astype(np.float32))
    ids = T(np.stack([rng.choice(E, K, replace=False) for _ in range(tokens)]).astype(np.int32))
    w = T(rng.random((tokens, K)).astype(np.float32))
    for resid in (None, T(rng.standard_normal((tokens, D)).astype(np.float32))):
        want = layer(hip_rt, "sabah_moe_layer_noalloc", desc, x, ids, w, resid)
        hip_rt.check(hip_rt.lib().sabah_rt_set_kernel_timing(1), "timing on")
        grouped_launches(hip_rt)
        got = layer(hip_rt, "sabah_moe_layer", desc, x, ids, w, resid)
        assert grouped_launches(hip_rt) > 0
        hip_rt.check(hip_rt.lib().sabah_rt_set_kernel_timing(0), "timing off")
        assert_bits_equal(got, want, "layer")
    # in place, then captured with the scratch in place
    y = x.clone()
    graph = torch.cuda.CUDAGraph()
    out = torch.empty_like(x)
    with torch.cuda.graph(graph):
        hip_rt.check(hip_rt.lib().sabah_moe_layer(
            ctypes.byref(desc), vp(y), vp(ids), vp(w), K, tokens, vp(out), vp(y),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "captured layer")
    want = layer(hip_rt, "sabah_moe_layer_noalloc", desc, x, ids, w, x)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), want, "replayed layer")


def typed_executor(rng, qtg, qtd, E, D, F, K, shared=None):
    """An executor over one layer of random valid blocks."""
    from sabah.runtime.bank import ExpertBank
    from sabah.runtime.executor import MoEExecutor
    bank = ExpertBank(1, E, D, F, {"gate": qtg, "up": qtg, "down": qtd}, device="cuda:0")
    for role, qt, rows, k in (("gate", qtg, F, D), ("up", qtg, F, D), ("down", qtd, D, F)):
        bank.load(0, role, bank_bytes(rng, qt, E, rows, k))
    return MoEExecutor(bank, max_used=K, shared=shared)


def layer_inputs(rng, E, D, K, tokens):
    ids = np.argsort(rng.random((tokens, E)), axis=1)[:, :K].astype(np.int32)
    ids[1, 1] = ids[1, 0]                            # a duplicate
    return (T(0.05 * rng.standard_normal((tokens, D)).astype(np.float32)), T(ids),
            T(rng.random((tokens, K)).astype(np.float32)))


# four-tile items: 602 pairs over 6 experts (at least 24 each on average; items of 64
# and a rest that ends inside a tile) at d_ff 4608 (72 row tiles x 15 items >= 1,024)
@pytest.mark.parametrize("qtg,qtd,D", [(Q4_K, Q6_K, 512), (Q6_K, Q4_K, 256), (Q4_K, Q8_0, 256), (Q5_K, IQ4_XS, 256),
                                       (IQ3_S, IQ3_S, 256), (IQ3_XXS, IQ4_NL, 512), (IQ4_XS, Q5_K, 256),
                                       (IQ4_NL, IQ3_XXS, 352)])
def test_grouped_layer_of_four_tile_items(hip_rt, qtg, qtd, D):
    E, K, F, tokens = 6, 2, 4608, 301
    rng = np.random.default_rng(1000 * qtg + qtd)
    ex = typed_executor(rng, qtg, qtd, E, D, F, K)
    x, ids, w = layer_inputs(rng, E, D, K, tokens)
    for resid in (None, x):
        got = ex.run_layer(0, x, ids, w, resid=resid)
        want = token_major_layer(ex, 0, x, ids, w, resid)
        assert_bits_equal(got.cpu().numpy(), want.cpu().numpy(), "layer %d/%d" % (qtg, qtd))


# sabah_moe_prefill_layer's batches on k_grouped_rows: from 10 pairs per expert and 512 in
# all (20 and 4,096 with an IQ3_S matrix), in two- and four-tile items (40 experts, 1,600 pairs)
@pytest.mark.parametrize("qtg,qtd,E,D,F,K,tokens", [
    (Q4_K, Q6_K, 6, 512, 256, 2, 256), (Q6_K, Q4_K, 51, 1024, 512, 3, 171), (Q4_K, Q6_K, 40, 512, 1024, 4, 401),
    (Q6_K, Q6_K, 40, 512, 1024, 4, 400), (Q4_K, Q4_K, 40, 2048, 1024, 4, 400), (IQ3_S, Q4_K, 200, 512, 512, 8, 513),
    (Q4_K, IQ3_S, 40, 512, 1024, 4, 1025), (IQ3_S, IQ3_S, 40, 512, 1024, 4, 1025)])
def test_prefill_layer_on_grouped_rows(hip_rt, qtg, qtd, E, D, F, K, tokens):
    rng = np.random.default_rng(100 * qtg + qtd + tokens)
    ex = typed_executor(rng, qtg, qtd, E, D, F, K)
    x, ids, w = layer_inputs(rng, E, D, K, tokens)
    want = token_major_layer(ex, 0, x, ids, w, x).cpu().numpy()
    hip_rt.check(hip_rt.lib().sabah_rt_set_kernel_timing(1), "timing on")
    try:
        grouped_launches(hip_rt)
        got = ex.run_prefill_layer(0, x, ids, w, resid=x)
        torch.cuda.synchronize()
        assert grouped_launches(hip_rt) == 3         # the grouping, x's rows and gate/up (the fixed-shape form times one)
    finally:
        hip_rt.check(hip_rt.lib().sabah_rt_set_kernel_timing(0), "timing off")
    assert_bits_equal(got.cpu().numpy(), want, "prefill %d/%d" % (qtg, qtd))


# k_group_pairs with its ids in 8 or 16 registers a thread, and read again: at most 8,192
# and 16,384 pairs, and more
@pytest.mark.parametrize("tokens", [2730, 2731, 5461, 5462, 7001])
def test_grouping_of_many_pairs(hip_rt, grouping, tokens):
    E, K, rows, k = 37, 3, 17, 256
    rng = np.random.default_rng(tokens)
    bank = T(bank_bytes(rng, IQ4_XS, E, rows, k))
    ids = rng.integers(0, E, (tokens, K)).astype(np.int32)
    ids[tokens - 1, 2] = E                           # a bad id, in the last pair
    x = T(rng.standard_normal((tokens, 1, k)).astype(np.float32))
    grouping(NEVER)
    tok = mmid(hip_rt, bank, IQ4_XS, rows, k, E, x, T(ids), grouped=False)
    assert hip_rt.lib().sabah_rt_check_errors() == -1
    grouping(ALWAYS)
    got = mmid(hip_rt, bank, IQ4_XS, rows, k, E, x, T(ids), grouped=True)
    assert hip_rt.lib().sabah_rt_check_errors() == -1
    assert np.isnan(got[tokens - 1, 2]).all() and np.isnan(tok[tokens - 1, 2]).all()
    got[tokens - 1, 2] = tok[tokens - 1, 2] = 0
    assert_bits_equal(got, tok, "%d pairs" % (tokens * K))


def test_runs_of_tokens_beside_a_gated_shared_expert(hip_rt):
    """70,010 pairs in two runs of tokens, each with the shared expert on the side
    stream beside it and the residual."""
    from sabah.runtime.bank import DenseExpert
    E, D, F, K, tokens = 12, 256, 256, 10, 7001
    rng = np.random.default_rng(71)
    shared = DenseExpert(D, 256, Q8_0, device="cuda:0")
    for role in ("gate", "up", "down"):
        shared.load(role, random_blocks(rng, Q8_0, 256, 256))
    shared.set_gate((0.05 * rng.standard_normal(D)).astype(np.float32))
    ex = typed_executor(rng, Q5_K, Q8_0, E, D, F, K, shared)
    x, ids, w = layer_inputs(rng, E, D, K, tokens)
    got = ex.run_layer(0, x, ids, w, resid=x)
    want = token_major_layer(ex, 0, x, ids, w, x)
    assert_bits_equal(got.cpu().numpy(), want.cpu().numpy(), "layer")


def test_a_smaller_token_major_layer_is_captured_after_a_grouped_one(hip_rt):
    """An eager call that runs group-major leaves room for a smaller, token-major
    call of the same layer inside a capture, which cannot allocate."""
    from sabah.runtime import rt
    E, K, D, F, tokens, small = 6, 3, 1024, 2304, 700, 5
    rng = np.random.default_rng(77)
    banks = [T(bank_bytes(rng, q, E, rows, k)) for q, rows, k in ((Q5_K, F, D), (Q5_K, F, D), (Q5_K, D, F))]
    desc = rt.MoeLayerDesc()
    desc.gate, desc.up, desc.down = (b.data_ptr() for b in banks)
    desc.qt_gate = desc.qt_up = desc.qt_down = Q5_K
    desc.d_model, desc.d_ff, desc.n_experts = D, F, E
    x = T(0.05 * rng.standard_normal((tokens, D)).astype(np.float32))
    ids = T(np.stack([rng.choice(E, K, replace=False) for _ in range(tokens)]).astype(np.int32))
    w = T(rng.random((tokens, K)).astype(np.float32))
    got = layer(hip_rt, "sabah_moe_layer", desc, x, ids, w)
    for t in range(0, tokens, 100):
        s = slice(t, t + 100)
        want = layer(hip_rt, "sabah_moe_layer_noalloc", desc, x[s].contiguous(), ids[s].contiguous(), w[s].contiguous())
        assert_bits_equal(got[s], want, "the eager layer, tokens from %d" % t)
    want = layer(hip_rt, "sabah_moe_layer_noalloc", desc, x[:small], ids[:small], w[:small])
    out = torch.empty_like(x[:small])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hip_rt.check(hip_rt.lib().sabah_moe_layer(
            ctypes.byref(desc), vp(x), vp(ids), vp(w), K, small, vp(out), None,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "captured layer")
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), want, "replayed layer")


def test_a_large_layers_scratch_is_one_runs(hip_rt):
    """200,000 pairs run in four runs of tokens (three of 65,536 pairs and a rest):
    the scratch is one run's (h of the whole batch alone would be 3.3 GB), and every
    run's tokens are the token-major layer's."""
    from sabah.runtime import rt
    E, K, D, F, tokens = 6, 2, 64, 4096, 100000
    rng = np.random.default_rng(41)
    banks = [T(bank_bytes(rng, Q8_0, E, rows, k)) for rows, k in ((F, D), (F, D), (D, F))]
    desc = rt.MoeLayerDesc()
    desc.gate, desc.up, desc.down = (b.data_ptr() for b in banks)
    desc.qt_gate = desc.qt_up = desc.qt_down = Q8_0
    desc.d_model, desc.d_ff, desc.n_experts = D, F, E
    x = T(0.05 * rng.standard_normal((tokens, D)).astype(np.float32))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    w = T(rng.random((tokens, K)).astype(np.float32))
    before = hip_rt.snapshot()["scratch_bytes"]
    got = layer(hip_rt, "sabah_moe_layer", desc, x, ids, w, x)
    assert hip_rt.snapshot()["scratch_bytes"] - before < 2.5e9
    for t in (0, 32768 - 60, 2 * 32768 - 60, 3 * 32768 - 60, tokens - 120):
        s = slice(t, t + 120)                     # across the runs' ends
        want = layer(hip_rt, "sabah_moe_layer_noalloc", desc, *(a[s].contiguous() for a in (x, ids, w, x)))
        assert_bits_equal(got[s], want, "tokens from %d" % t)


def test_a_smaller_fixed_shape_prefill_is_captured_after_a_grouped_rows_one(hip_rt):
    """4,096 experts: 90,000 pairs take k_grouped_rows in runs of 65,536, and the
    80,000 pairs captured after them the fixed-shape kernels, in one piece."""
    from sabah.runtime.bank import ExpertBank
    from sabah.runtime.executor import MoEExecutor
    E, K, D, F, tokens, small = 4096, 10, 512, 256, 9000, 8000
    rng = np.random.default_rng(42)
    bank = ExpertBank(1, E, D, F, {"gate": IQ3_S, "up": IQ3_S, "down": Q6_K}, device="cuda:0")
    bank.fill_synthetic(seed=5)
    ex = MoEExecutor(bank, max_used=K)
    x = T(rng.standard_normal((tokens, D)).astype(np.float32))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    w = T(rng.random((tokens, K)).astype(np.float32))
    big = ex.run_prefill_layer(0, x, ids, w)
    out = torch.empty_like(x[:small])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ex.run_prefill_layer(0, x[:small], ids[:small], w[:small], out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), big[:small].cpu().numpy(), "replayed prefill")


# q8 rows past 2 GiB and past 2^21 chunks in all: in the general form with one x row
# per slot (450,000 rows of 4,864 bytes) and in the fixed-shape form (900,000 of 2,464)
@pytest.mark.parametrize("qt,k,tokens,K,slot_rows", [(Q8_0, 4096, 45000, 10, True), (Q4_K, 2048, 45000, 20, False)])
def test_quantised_rows_past_2_gib(hip_rt, grouping, qt, k, tokens, K, slot_rows):
    E, rows = 16, 64
    rng = np.random.default_rng(k)
    bank = T(bank_bytes(rng, qt, E, rows, k))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    g = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn((tokens, K if slot_rows else 1, k), device=DEV, generator=g)
    grouping(NEVER)
    tok = mmid(hip_rt, bank, qt, rows, k, E, x, ids, grouped=False)
    grouping(AUTO)
    got = mmid(hip_rt, bank, qt, rows, k, E, x, ids, grouped=True)
    assert_bits_equal(got, tok, "qt=%d" % qt)


def test_a_layers_quantised_h_rows_past_2_gib(hip_rt):
    """One run of 65,000 pairs at d_ff 28,672: 2.2 GB of q8 rows of h."""
    from sabah.runtime import rt
    E, K, D, F, tokens = 4, 1, 64, 28672, 65000
    rng = np.random.default_rng(28)
    banks = [T(bank_bytes(rng, Q8_0, E, rows, k)) for rows, k in ((F, D), (F, D), (D, F))]
    desc = rt.MoeLayerDesc()
    desc.gate, desc.up, desc.down = (b.data_ptr() for b in banks)
    desc.qt_gate = desc.qt_up = desc.qt_down = Q8_0
    desc.d_model, desc.d_ff, desc.n_experts = D, F, E
    x = T(0.05 * rng.standard_normal((tokens, D)).astype(np.float32))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    w = T(rng.random((tokens, K)).astype(np.float32))
    got = layer(hip_rt, "sabah_moe_layer", desc, x, ids, w)
    for t in (0, 20000, 40000, tokens - 40):
        s = slice(t, t + 40)                      # as many tokens as the token-major call's static scratch holds
        want = layer(hip_rt, "sabah_moe_layer_noalloc", desc, x[s].contiguous(), ids[s].contiguous(), w[s].contiguous())
        assert_bits_equal(got[s], want, "tokens from %d" % t)


def test_calls_whose_optional_scratch_is_refused_run_token_major(hip_rt, grouping):
    """A device with no room for the grouped form's scratch: the call and the
    layer take the kernels that need none, and no error is left for either."""
    from sabah.runtime import rt
    lib = hip_rt.lib()
    E, K, D, F, tokens = 6, 2, 512, 256, 301
    rng = np.random.default_rng(91)
    banks = [T(bank_bytes(rng, Q5_K, E, rows, k)) for rows, k in ((F, D), (F, D), (D, F))]
    desc = rt.MoeLayerDesc()
    desc.gate, desc.up, desc.down = (b.data_ptr() for b in banks)
    desc.qt_gate = desc.qt_up = desc.qt_down = Q5_K
    desc.d_model, desc.d_ff, desc.n_experts = D, F, E
    x = T(0.05 * rng.standard_normal((tokens, D)).astype(np.float32))
    ids = T(rng.integers(0, E, (tokens, K)).astype(np.int32))
    w = T(rng.random((tokens, K)).astype(np.float32))
    x3 = x.view(tokens, 1, D)
    want = mmid(hip_rt, banks[0], Q5_K, F, D, E, x3, ids, grouped=True)
    want_layer = layer(hip_rt, "sabah_moe_layer", desc, x, ids, w)
    hip_rt.check(lib.sabah_rt_set_scratch_refusal(1), "refusal on")
    hip_rt.check(lib.sabah_rt_set_kernel_timing(1), "timing on")
    try:
        assert_bits_equal(mmid(hip_rt, banks[0], Q5_K, F, D, E, x3, ids, grouped=False), want, "MUL_MAT_ID")
        grouped_launches(hip_rt)
        assert_bits_equal(layer(hip_rt, "sabah_moe_layer", desc, x, ids, w), want_layer, "layer")
        assert grouped_launches(hip_rt) == 0
    finally:
        lib.sabah_rt_set_kernel_timing(0)
        lib.sabah_rt_set_scratch_refusal(0)
    assert_bits_equal(mmid(hip_rt, banks[0], Q5_K, F, D, E, x3, ids, grouped=True), want, "grouped again")
