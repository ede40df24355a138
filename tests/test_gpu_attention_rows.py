"""Attention of several tokens on the bf16 matrix cores (attention_prefill.hip) and the quad RoPE + append.

Outputs against 64-bit attention: the scores and sums are f32 sums of exact
products, so an output differs by a few units of 2^-24 of the largest value
times the chain of roundings in a weight (scores of up to about 30 in size).
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from leaf_amd import runtime
    runtime.library()
    return runtime


def exact(q, keys, values, position, window):
    heads, tokens, dim = q.shape
    group = heads // keys.shape[0]
    out = np.empty((tokens, heads, dim))
    for h in range(heads):
        k, v = (a[h // group].astype(np.float64) for a in (keys, values))
        for t in range(tokens):
            end = position + t + 1
            begin = max(0, end - window) if window else 0
            s = k[begin:end] @ q[h, t].astype(np.float64) / np.sqrt(dim)
            p = np.exp(s - s.max())
            out[t, h] = (p / p.sum()) @ v[begin:end]
    return out


def call(rt, q, keys, values, position, window):
    heads, tokens, dim = q.shape
    kv, capacity, _ = keys.shape
    dq, dk, dv = (rt.DeviceArray.of(a) for a in (q, keys, values))
    out = rt.DeviceArray((tokens, heads, dim), np.float32)
    rt.check(rt.library().lh_attention(dq.ptr, dk.ptr, dv.ptr, capacity, heads, kv, dim, tokens, position, window,
                                       out.ptr, None))
    return out.numpy()


def inputs(rng, tokens, position, heads, kv, dim):
    total, capacity = position + tokens, position + tokens + 37
    q = rng.standard_normal((heads, tokens, dim), dtype=np.float32)
    keys, values = (rng.standard_normal((kv, capacity, dim), dtype=np.float32) for _ in range(2))
    keys[:, total:] = values[:, total:] = np.nan      # never written
    return q, keys, values


# Row tiles (128 rows, 64 beyond 64 values) cut by the token count, groups that
# do not divide them, one part and several (few rows over long caches), every
# padded width, windows shorter and longer than a step of 64 keys.
@pytest.mark.parametrize("tokens,position,heads,kv,dim,window", [
    (2, 0, 12, 12, 64, 0), (2, 700, 14, 2, 64, 0), (3, 64, 7, 1, 32, 0), (17, 0, 15, 5, 64, 0), (33, 191, 4, 1, 128, 0),
    (64, 0, 32, 4, 64, 0), (65, 1, 6, 2, 80, 0), (130, 40, 5, 5, 96, 0), (40, 0, 3, 3, 4, 0), (50, 90, 4, 2, 20, 33),
    (90, 300, 6, 3, 64, 100), (70, 500, 8, 2, 128, 64), (5, 1500, 32, 8, 128, 0), (300, 20, 2, 1, 36, 7)])
def test_against_64_bits(rt, tokens, position, heads, kv, dim, window):
    rng = np.random.default_rng(tokens * 31 + position + dim)
    q, keys, values = inputs(rng, tokens, position, heads, kv, dim)
    got, want = call(rt, q, keys, values, position, window), exact(q, keys, values, position, window)
    assert np.isfinite(got).all()
    # weights to 2^-24 (|score| + 8), so outputs to that of the largest value
    assert np.max(np.abs(got - want)) <= 2.0 ** -24 * 40 * np.nanmax(np.abs(values))


@pytest.mark.parametrize("tokens,position,dim", [(70, 10, 64), (4, 900, 64), (20, 100, 128)])
def test_values_that_do_not_split(rt, tokens, position, dim):
    # Keys of minus infinity weigh nothing, infinite and NaN values reach the
    # rows that see them and no other.
    rng = np.random.default_rng(dim + tokens)
    heads, kv = 4, 2
    q, keys, values = inputs(rng, tokens, position, heads, kv, dim)
    q[:, :, 0] = np.abs(q[:, :, 0]) + 0.1
    keys[0, 5, 0] = -np.inf
    values[1, position + 1, 3] = np.inf
    values[1, position + tokens - 1, 2] = np.nan
    got = call(rt, q, keys, values, position, 0)
    with np.errstate(all="ignore"):
        want = exact(q, keys, values, position, 0)
    # a weight that underflows to 0 times an infinite value is NaN on either side of f32's range
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    plain = np.isfinite(want)
    assert np.max(np.abs(got[plain] - want[plain])) <= 2.0 ** -24 * 40 * 5


@pytest.mark.parametrize("special", [np.nan, np.inf])
@pytest.mark.parametrize("tokens,position,dim", [(70, 10, 64), (4, 900, 64), (20, 100, 128)])
def test_keys_that_spoil_a_row(rt, tokens, position, dim, special):
    # A NaN score, or one of infinity less its own maximum, makes its row NaN,
    # as in plain f32; rows and heads that do not see the key keep their values.
    rng = np.random.default_rng(dim + tokens)
    q, keys, values = inputs(rng, tokens, position, 4, 2, dim)
    q[:, :, 1] = np.abs(q[:, :, 1]) + 0.1
    keys[1, position + tokens // 2, 1] = special
    got = call(rt, q, keys, values, position, 0)
    with np.errstate(all="ignore"):
        want = exact(q, keys, values, position, 0)
    assert np.array_equal(np.isfinite(got), np.isfinite(want)) and not np.isfinite(want).all()
    plain = np.isfinite(want)
    assert np.max(np.abs(got[plain] - want[plain])) <= 2.0 ** -24 * 40 * 5


@pytest.mark.parametrize("heads,kv,dim,rotary,tokens", [(14, 2, 64, 64, 5), (4, 2, 64, 32, 3), (3, 1, 80, 80, 2),
                                                        (2, 2, 36, 24, 4), (5, 5, 64, 0, 1), (4, 1, 20, 12, 3)])
def test_rope_append(rt, heads, kv, dim, rotary, tokens):
    # widths of whole quads and (rotary 12) not: the same arithmetic
    rng = np.random.default_rng(heads + dim + rotary)
    position, capacity, half = 7, 20, rotary // 2
    qkv = rng.standard_normal((tokens, heads + 2 * kv, dim), dtype=np.float32)
    cos, sin = (rng.standard_normal((capacity, max(half, 1)), dtype=np.float32) for _ in range(2))
    dq, dc, ds = (rt.DeviceArray.of(a) for a in (qkv, cos, sin))
    q = rt.DeviceArray((heads, tokens, dim), np.float32)
    keys, values = (rt.DeviceArray((kv, capacity, dim), np.float32).zero() for _ in range(2))
    rt.check(rt.library().lh_rope_kv(dq.ptr, tokens, heads, kv, dim, rotary, position, dc.ptr, ds.ptr, q.ptr, keys.ptr,
                                     values.ptr, capacity, None))
    turned = qkv[:, :heads + kv].copy()
    c, s = (a[position:position + tokens, None, :half] for a in (cos, sin))
    a, b = qkv[:, :heads + kv, :half], qkv[:, :heads + kv, half:rotary]
    turned[..., :half], turned[..., half:rotary] = a * c - b * s, b * c + a * s
    assert np.array_equal(q.numpy(), turned[:, :heads].transpose(1, 0, 2))
    assert np.array_equal(keys.numpy()[:, position:position + tokens], turned[:, heads:].transpose(1, 0, 2))
    assert np.array_equal(values.numpy()[:, position:position + tokens], qkv[:, heads + kv:].transpose(1, 0, 2))


# Rows whose visible scores in a whole part of the keys are NaN or minus
# infinity: split over two parts, over five and more, and not split (a short
# cache).  Row `position` is the first key of its last part in the split calls.
@pytest.mark.parametrize("tokens,position,heads,kv,dim", [(100, 128, 2, 2, 64), (100, 512, 2, 2, 64), (4, 900, 4, 2, 64),
                                                          (50, 128, 2, 2, 128), (20, 0, 4, 2, 64)])
@pytest.mark.parametrize("spoilt", ["query", "own key", "every key", "masked value"])
def test_parts_without_a_usable_score(rt, tokens, position, heads, kv, dim, spoilt):
    rng = np.random.default_rng(tokens + position + dim)
    q, keys, values = inputs(rng, tokens, position, heads, kv, dim)
    q[:, :, 0] = np.abs(q[:, :, 0]) + 0.1
    if spoilt == "query":
        q[1, tokens // 2, 3] = np.nan
    elif spoilt == "own key":
        keys[0, position, 2] = np.nan
    elif spoilt == "every key":
        keys[0, :position + tokens, 0] = -np.inf
    else:
        keys[:, position, 0], values[0, position, 3] = -np.inf, np.inf      # weight 0 of an infinite value: NaN
    got = call(rt, q, keys, values, position, 0)
    with np.errstate(all="ignore"):
        want = exact(q, keys, values, position, 0)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any()
    plain = np.isfinite(want)
    assert np.max(np.abs(got[plain] - want[plain])) <= 2.0 ** -24 * 40 * 5


@pytest.mark.parametrize("tokens,position,heads,kv,dim,window", [(33, 191, 4, 1, 64, 0), (20, 1000, 6, 3, 128, 0),
                                                                 (64, 0, 6, 2, 80, 33)])
def test_unaligned_arrays(rt, tokens, position, heads, kv, dim, window):
    # every array one float past a 16-byte boundary
    rng = np.random.default_rng(tokens + dim)
    arrays = inputs(rng, tokens, position, heads, kv, dim)
    q, keys, values = arrays
    dq, dk, dv = (rt.DeviceArray.of(np.concatenate([np.zeros(1, np.float32), a.reshape(-1)])) for a in arrays)
    out = rt.DeviceArray((1 + tokens * heads * dim,), np.float32).zero()
    rt.check(rt.library().lh_attention(dq.ptr + 4, dk.ptr + 4, dv.ptr + 4, keys.shape[1], heads, kv, dim, tokens, position,
                                       window, out.ptr + 4, None))
    got, want = out.numpy()[1:].reshape(tokens, heads, dim), exact(q, keys, values, position, window)
    assert np.max(np.abs(got - want)) <= 2.0 ** -24 * 40 * np.nanmax(np.abs(values))


# The general kernel (head dims beyond 128, arrays that are not aligned): NaN
# and minus infinity as in the kernel above, also where the first 256 keys have
# no weight.
@pytest.mark.parametrize("dim,offset", [(160, 0), (64, 1)])
@pytest.mark.parametrize("spoilt", ["query", "key", "early keys", "every key"])
def test_general_kernel_without_a_usable_score(rt, dim, offset, spoilt):
    tokens, position, heads, kv = 20, 300, 4, 2
    rng = np.random.default_rng(dim)
    q, keys, values = inputs(rng, tokens, position, heads, kv, dim)
    q[:, :, 0] = np.abs(q[:, :, 0]) + 0.1
    if spoilt == "query":
        q[1, 7, 3] = np.nan
    elif spoilt == "key":
        keys[0, position + 4, 2] = np.nan
    else:
        keys[0, :position + tokens if spoilt == "every key" else 290, 0] = -np.inf
    dq, dk, dv = (rt.DeviceArray.of(np.concatenate([np.zeros(offset, np.float32), a.reshape(-1)])) for a in (q, keys, values))
    out = rt.DeviceArray((tokens, heads, dim), np.float32)
    rt.check(rt.library().lh_attention(dq.ptr + 4 * offset, dk.ptr + 4 * offset, dv.ptr + 4 * offset, keys.shape[1], heads,
                                       kv, dim, tokens, position, 0, out.ptr, None))
    got = out.numpy()
    with np.errstate(all="ignore"):
        want = exact(q, keys, values, position, 0)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    plain = np.isfinite(want)
    assert np.max(np.abs(got[plain] - want[plain])) <= 2.0 ** -24 * 40 * 5


# Up to 40, 48 and 80 keys (one block per head and token) and just beyond, with windows,
# dims with and without a remainder of eight, and a NaN in between.
@pytest.mark.parametrize("tokens,position,heads,kv,dim,window", [
    (2, 0, 12, 12, 64, 0), (40, 0, 4, 2, 128, 0), (17, 23, 6, 2, 80, 9), (5, 35, 8, 1, 32, 0), (3, 20, 4, 4, 36, 5),
    (40, 0, 3, 3, 4, 0), (50, 0, 3, 3, 4, 0), (9, 32, 4, 2, 128, 12), (20, 28, 4, 2, 96, 0), (7, 60, 6, 2, 64, 0),
    (24, 56, 32, 8, 128, 0), (25, 56, 4, 4, 32, 0), (16, 64, 8, 1, 32, 50)])
def test_few_keys(rt, tokens, position, heads, kv, dim, window):
    rng = np.random.default_rng(tokens + dim)
    q, keys, values = inputs(rng, tokens, position, heads, kv, dim)
    q[0, tokens // 2, 0] = np.nan
    got, want = call(rt, q, keys, values, position, window), exact(q, keys, values, position, window)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any()
    plain = np.isfinite(want)
    assert np.max(np.abs(got[plain] - want[plain])) <= 2.0 ** -24 * 40 * np.nanmax(np.abs(values))


def test_decoder_prompt_in_chunks(rt, oracle, artifacts):
    # a decoder's chunks behind cached keys, which share those keys out over
    # blocks: every row of logits against the CPU path (1e-3 of the largest, as
    # for any FP32-math decoder)
    dec, cpu = rt.Decoder(artifacts["qwen"], max_prefill=512), oracle.decoder(artifacts["qwen"], 32, False)
    prompt = np.random.default_rng(5).integers(0, dec.vocabulary_size, 900).astype(np.uint32)
    start = 0
    for tokens in (512, 300, 60, 16, 10, 2):
        ids = prompt[start:start + tokens]
        got, want = dec.forward(ids, all_logits=True), cpu.forward(ids, all_logits=True)
        assert np.max(np.abs(got - want)) <= 1e-3 * np.max(np.abs(want))
        start += tokens


@pytest.mark.parametrize("every", [False, True])
def test_nan_queries_cost_little(rt, every):
    # Their rows are computed again, which ends at the first NaN score: about 1.1
    # times the call's time for one, 7 times for all (3 and over 90 in two passes).
    import ctypes as C
    rng = np.random.default_rng(2)
    heads, kv, dim, tokens = 14, 2, 64, 300
    q, keys, values = inputs(rng, tokens, 0, heads, kv, dim)
    dk, dv, out, lib = rt.DeviceArray.of(keys), rt.DeviceArray.of(values), rt.DeviceArray((tokens, heads, dim), np.float32), rt.library()

    def milliseconds(q):
        dq, best = rt.DeviceArray.of(q), np.inf
        for _ in range(5):
            timer, ms = C.c_void_p(), C.c_double()
            for timed in (False, True):
                if timed:
                    rt.check(lib.lh_timer_start(None, C.byref(timer)))
                for _ in range(5):
                    rt.check(lib.lh_attention(dq.ptr, dk.ptr, dv.ptr, keys.shape[1], heads, kv, dim, tokens, 0, 0, out.ptr, None))
            rt.check(lib.lh_timer_stop(timer, None, C.byref(ms)))
            best = min(best, ms.value)
        return best

    plain = milliseconds(q)
    spoilt = q.copy()
    if every:
        spoilt[:, :, 1] = np.nan
    else:
        spoilt[0, tokens // 2, 1] = np.nan
    assert milliseconds(spoilt) <= (25 if every else 2) * plain
