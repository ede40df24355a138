"""Integer-activation linears with scale groups: the int8 MFMA GEMM (gemm_grouped.hip).

Outputs and group accumulators are bit-identical to the oracle's for every
route: groups of one, two or four steps of 32 values, of whole stages of 128
or anything else, rows that end inside a stage, both block sizes, with the
accumulators (the general kernel) and without.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from leaf_amd.artifact import quantize

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from leaf_amd import runtime
    runtime.library()
    return runtime


@pytest.fixture(scope="module")
def oracle():
    from oracle.bindings import oracle as load
    return load()


@pytest.mark.parametrize("bits,K,group", [(8, 96, 32), (8, 128, 64), (8, 960, 64), (8, 2048, 128), (8, 768, 256),
                                          (8, 480, 96), (8, 960, 960), (8, 32, 32), (4, 896, 32), (4, 192, 64),
                                          (4, 1280, 128), (4, 288, 96), (4, 896, 896), (4, 32, 32)])
@pytest.mark.parametrize("M,N", [(1, 40), (5, 97), (33, 256), (130, 31), (300, 3100), (513, 1030)])
def test_grouped_gemm_bit_exact(rt, oracle, bits, K, group, M, N):
    rng = np.random.default_rng(bits * 100000 + K * 10 + M)
    w = (0.02 * rng.standard_normal((N, K))).astype(np.float32)
    wq, ws = quantize(w, bits, group)
    bias = rng.standard_normal(N, dtype=np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32)
    x[rng.random((M, K)) < 0.002] *= np.float32(20)
    x[M // 2] = 0.0
    dw = rt.DeviceWeight(wq, bits, K, ws, group, bias)
    dx, dy = rt.DeviceArray.of(x), rt.DeviceArray((M, N), np.float32)
    q, _ = oracle.quantize_rows(x)
    oracle.set_vnni_policy(0)
    expected = oracle.linear_int(bits, N, K, group, wq, ws, bias, x)
    rt.linear(dw, dx, M, 8, dy)
    assert np.array_equal(dy.numpy().view(np.uint32), expected.view(np.uint32))
    dacc = rt.DeviceArray((M, N, K // group), np.int32)
    dy.zero()
    rt.linear(dw, dx, M, 8, dy, dacc)
    assert np.array_equal(dy.numpy().view(np.uint32), expected.view(np.uint32))
    assert np.array_equal(dacc.numpy(), oracle.int_accumulators(bits, N, K, group, wq, q))
    # the same input given quantized, its copy not 16-byte aligned: any kernel, the same bits
    dq, ds = rt.DeviceArray.of(np.concatenate([np.zeros(4, np.int8), q.reshape(-1)])), None
    scale = np.maximum(np.abs(x).max(axis=1) / np.float32(127), np.float32(1e-12)).astype(np.float32)
    ds = rt.DeviceArray.of(scale)
    dy.zero()
    rt.check(rt.library().lh_linear_q(C.byref(dw.desc), dq.ptr + 4, ds.ptr, M, dy.ptr, None, None))
    assert np.array_equal(dy.numpy().view(np.uint32), expected.view(np.uint32))


# An input that is not aligned and may not be copied (the stream captures): every
# weight width and kind of group, rows that end inside a stage, both block sizes.
@pytest.mark.parametrize("bits,K,group", [(8, 96, 32), (8, 2048, 128), (8, 960, 960), (4, 896, 32), (4, 288, 96)])
@pytest.mark.parametrize("M,N,offset", [(5, 97, 1), (33, 256, 4), (300, 3100, 7), (513, 1030, 8)])
def test_captured_unaligned_input_bit_exact(rt, oracle, bits, K, group, M, N, offset):
    rng = np.random.default_rng(bits * 1000 + K + M)
    wq, ws = quantize((0.02 * rng.standard_normal((N, K))).astype(np.float32), bits, group)
    bias = rng.standard_normal(N, dtype=np.float32)
    x = rng.standard_normal((M, K), dtype=np.float32)
    dw = rt.DeviceWeight(wq, bits, K, ws, group, bias)
    q, _ = oracle.quantize_rows(x)
    oracle.set_vnni_policy(0)
    expected = oracle.linear_int(bits, N, K, group, wq, ws, bias, x)
    dq = rt.DeviceArray.of(np.concatenate([np.zeros(offset, np.int8), q.reshape(-1)]))
    ds = rt.DeviceArray.of(np.maximum(np.abs(x).max(axis=1) / np.float32(127), np.float32(1e-12)).astype(np.float32))
    dy, dacc = rt.DeviceArray((M, N), np.float32), rt.DeviceArray((M, N, K // group), np.int32)
    stream = rt.Stream()

    def call():
        rt.check(rt.library().lh_linear_q(C.byref(dw.desc), dq.ptr + offset, ds.ptr, M, dy.ptr, dacc.ptr, stream.handle))

    call()                                             # sizes the stream's scratch
    stream.synchronize()
    graph = rt.Graph(stream, call)
    for _ in range(2):
        dy.zero()
        dacc.zero()
        rt.synchronize()
        graph.launch()
        stream.synchronize()
        assert np.array_equal(dy.numpy().view(np.uint32), expected.view(np.uint32))
        assert np.array_equal(dacc.numpy(), oracle.int_accumulators(bits, N, K, group, wq, q))
    graph.close()
    stream.close()
