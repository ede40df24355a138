"""FP32-math linears of five and more tokens: the bf16-split GEMM (gemm_f32.hip).

Every output is compared with its 64-bit value under the bound of a plain f32
dot of K terms, K 2^-24 sum|x w|, and all of them together under a bound that
follows the kernel.  It rounds a sum once per MFMA, 3 of them for each 32 columns
(6 where the weight is split too), once per scale group, and once or twice at the
end; each rounding is at most 2^-24 of a partial sum of random sign, whose size
is that of sqrt(sum (x w)^2), and they are independent: 2^-24 sqrt(roundings)
sqrt(sum (x w)^2) in the 2-norm over the outputs.  The products left out, and a
dequantized weight's rounding, are 2^-24 of a term or less: one rounding more.
A kernel without the third bf16 value of x would be off by about 2^-18.8 of
sqrt(sum (x w)^2), 1.7 times that bound at the longest rows here and 4 at 960
columns.
"""
from __future__ import annotations

import numpy as np
import pytest

from leaf_amd.artifact import quantize

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from leaf_amd import runtime
    runtime.library()
    return runtime


def weights(rng, bits, N, K, group):
    """(storage, scales, group, the weights in 64 bits)"""
    w = (0.02 * rng.standard_normal((N, K))).astype(np.float32)
    if bits == 32:
        return w, None, 0, w.astype(np.float64)
    if bits == 16:
        data = (w.view(np.uint32) >> 16).astype(np.uint16)
        return data, None, 0, (data.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    data, scales = quantize(w, bits, group)
    q = data
    if bits == 4:
        q = np.empty((N, K), np.int8)
        q[:, ::2], q[:, 1::2] = data & 15, data >> 4
        q[q >= 8] -= 16
    return data, scales, group, q.astype(np.float64) * np.repeat(scales.astype(np.float64), group, axis=1)


def run(rt, bits, data, scales, group, bias, x):
    dw = rt.DeviceWeight(data, bits, x.shape[1], scales, group, bias)
    dx, dy = rt.DeviceArray.of(x), rt.DeviceArray((x.shape[0], data.shape[0]), np.float32)
    rt.linear(dw, dx, x.shape[0], 32, dy)
    return dy.numpy()


def within_bound(y, x, wd, bias):
    e = x.astype(np.float64) @ wd.T
    size = np.abs(x).astype(np.float64) @ np.abs(wd).T
    bound = (x.shape[1] + 1) * 2.0 ** -24 * size + 2.0 ** -23 * (np.abs(e) + np.abs(bias))
    return bool(np.all(np.abs(y - (e + bias)) <= bound))


def share_of_bound(y, x, wd, bias, split_weights, groups=1):
    """The error's 2-norm over the bound above."""
    K = x.shape[1]
    x = x.astype(np.float64)
    roundings = (6 if split_weights else 3) * -(-K // 32) + groups + 3
    size = np.sqrt(((x ** 2) @ (wd ** 2).T).sum() + (bias.astype(np.float64) ** 2).sum() * len(x))
    return float(np.linalg.norm(y - (x @ wd.T + bias)) / (2.0 ** -24 * np.sqrt(roundings) * size))


def bf16(v):
    """f32 values rounded to bf16 (ties to even)."""
    u = v.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)


@pytest.mark.parametrize("K", [64, 960, 4864])
@pytest.mark.parametrize("split_weights", [False, True])
def test_bound_finds_a_missing_plane(K, split_weights):
    # the oracle's sums in 64 bits, with all of x and with two of its three bf16 values
    rng = np.random.default_rng(K)
    x = rng.standard_normal((40, K), dtype=np.float32)
    w = rng.standard_normal((60, K), dtype=np.float32)
    w = w if split_weights else bf16(w)
    bias = np.zeros(60, np.float32)
    hi = bf16(x)
    two = hi.astype(np.float64) + bf16(x - hi)
    assert share_of_bound(x.astype(np.float64) @ w.astype(np.float64).T, x, w.astype(np.float64), bias, split_weights) < 1e-3
    assert share_of_bound(two @ w.astype(np.float64).T, x, w.astype(np.float64), bias, split_weights) > 1.1


# Token and row counts at the edges of the blocks (16 to 128 of either), grids
# that choose each of them, K of one stage and odd counts of stages.
@gpu
@pytest.mark.parametrize("bits,group", [(32, 0), (16, 0), (8, 0), (8, 64), (4, 32)])
@pytest.mark.parametrize("M,K,N", [(5, 64, 1), (16, 1984, 130), (33, 448, 777), (65, 64, 2051), (129, 960, 515),
                                   (300, 4864, 96), (513, 192, 1030), (700, 896, 2100), (1100, 64, 33)])
def test_shapes(rt, bits, group, M, K, N):
    rng = np.random.default_rng(M + K + N + bits)
    data, scales, group, wd = weights(rng, bits, N, K, group or K)
    bias = (0.1 * rng.standard_normal(N)).astype(np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32)
    x[rng.random((M, K)) < 0.001] *= np.float32(20)
    y = run(rt, bits, data, scales, group, bias, x)
    assert within_bound(y, x, wd, bias)
    assert share_of_bound(y, x, wd, bias, bits == 32, K // group if bits <= 8 else 1) <= 1


# Every block forced, with rows that end inside its tiles and (FP32, BF16) inside
# a stage; 15 stages leave the last waves of a "few" block one fewer.
@gpu
@pytest.mark.parametrize("shape", ["128x64", "64x128", "128x128", "64x64", "few16x16", "few32x16", "few16x32", "few32x32",
                                   "few64x32"])
@pytest.mark.parametrize("bits,K,group", [(32, 480, 0), (32, 484, 0), (16, 480, 0), (16, 20, 0), (8, 480, 0), (8, 480, 96),
                                          (4, 480, 32), (4, 480, 20)])
def test_every_block(rt, monkeypatch, shape, bits, K, group):
    rng = np.random.default_rng(K + bits)
    for M, N in ((5, 33), (70, 131), (131, 70)):
        data, scales, g, wd = weights(rng, bits, N, K, group or K)
        bias = (0.1 * rng.standard_normal(N)).astype(np.float32)
        x = rng.standard_normal((M, K), dtype=np.float32)
        monkeypatch.setenv("LEAF_F32_GEMM_TILE", shape)
        y = run(rt, bits, data, scales, g, bias, x)
        assert within_bound(y, x, wd, bias)
        split = bits == 32 or bits <= 8 and g != K and g % 32 != 0
        assert share_of_bound(y, x, wd, bias, split, K // g if bits <= 8 else 1) <= 1


# Two to four tokens: int4 groups of whole stages take the GEMM too, up to 4096 columns.
@gpu
@pytest.mark.parametrize("M", [2, 3, 4])
@pytest.mark.parametrize("K,N,group", [(64, 5, 32), (960, 1030, 64), (4096, 96, 32), (4128, 96, 32)])
def test_few_tokens_int4(rt, M, K, N, group):
    rng = np.random.default_rng(M + K)
    data, scales, group, wd = weights(rng, 4, N, K, group)
    bias = (0.1 * rng.standard_normal(N)).astype(np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32)
    y = run(rt, 4, data, scales, group, bias, x)
    assert within_bound(y, x, wd, bias)
    if K <= 4096:      # the GEMM's own
        assert share_of_bound(y, x, wd, bias, False, K // group) <= 1


# Rows that end inside a 32-value stage, and scale groups that are not whole stages.
@gpu
@pytest.mark.parametrize("bits,K,group", [(32, 36, 0), (32, 772, 0), (16, 100, 0), (16, 1028, 0), (8, 100, 100),
                                          (8, 96, 4), (8, 432, 48), (4, 100, 20), (4, 144, 16), (4, 1200, 100)])
@pytest.mark.parametrize("M,N", [(7, 17), (77, 131), (400, 1000)])
def test_ragged_rows_and_groups(rt, bits, K, group, M, N):
    rng = np.random.default_rng(K + M)
    data, scales, group, wd = weights(rng, bits, N, K, group)
    bias = (0.1 * rng.standard_normal(N)).astype(np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32)
    y = run(rt, bits, data, scales, group, bias, x)
    assert within_bound(y, x, wd, bias)
    assert share_of_bound(y, x, wd, bias, bits != 16, K // group if bits <= 8 else 1) <= 1


@gpu
@pytest.mark.parametrize("bits,K", [(32, 256), (16, 256), (8, 256), (4, 256), (32, 260)])
@pytest.mark.parametrize("M,N", [(6, 40), (200, 1030)])
def test_values_that_do_not_split(rt, bits, K, M, N):
    # Infinities, NaN and values that round past bf16's largest: what a chain
    # of f32 multiply-adds gives, in the outputs they reach and no other.
    rng = np.random.default_rng(5 + bits)
    data, scales, group, wd = weights(rng, bits, N, K, 32 if bits == 4 else K)
    x = rng.standard_normal((M, K), dtype=np.float32)
    huge = np.finfo(np.float32).max
    x[0, 3], x[1, 5], x[2, 7], x[3, 9] = np.inf, -np.inf, np.nan, huge
    x[4, 1], x[4, 2] = np.inf, -np.inf
    if bits == 32:
        data[11, 20] = np.inf
        wd = data.astype(np.float64)
    y = run(rt, bits, data, scales, group, None, x)
    with np.errstate(all="ignore"):
        e = x.astype(np.float64) @ wd.T
        e = np.where(np.abs(e) > huge, np.sign(e) * np.inf, e)
        assert np.array_equal(np.isnan(y), np.isnan(e))
        assert np.array_equal(np.isinf(y), np.isinf(e)) and np.array_equal(np.sign(y[np.isinf(y)]), np.sign(e[np.isinf(e)]))
        plain = np.isfinite(e)
        assert np.all(np.abs(y - e)[plain] <= 1e-4 * (1 + np.abs(e[plain])))


@gpu
@pytest.mark.parametrize("bits,M", [(32, 300), (16, 300), (4, 300), (16, 16)])
def test_one_infinite_activation_costs_little(rt, bits, M):
    # The outputs it spoils are computed again, by whole waves: 3 to 6 times the
    # call's time as they are spread here (over 50 times as one chain per lane).
    import ctypes as C
    rng = np.random.default_rng(3)
    K, N = 960, 5120
    data, scales, group, _ = weights(rng, bits, N, K, 32 if bits == 4 else 0)
    dw = rt.DeviceWeight(data, bits, K, scales, group)
    x = rng.standard_normal((M, K), dtype=np.float32)
    dy, lib = rt.DeviceArray((M, N), np.float32), rt.library()

    def milliseconds(dx):
        best = np.inf
        for _ in range(5):
            timer, ms = C.c_void_p(), C.c_double()
            rt.linear(dw, dx, M, 32, dy)
            rt.check(lib.lh_timer_start(None, C.byref(timer)))
            for _ in range(5):
                rt.linear(dw, dx, M, 32, dy)
            rt.check(lib.lh_timer_stop(timer, None, C.byref(ms)))
            best = min(best, ms.value)
        return best

    plain = milliseconds(rt.DeviceArray.of(x))
    x[M // 2, K // 3] = np.inf
    assert milliseconds(rt.DeviceArray.of(x)) <= 12 * plain
