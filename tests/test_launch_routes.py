"""Which kernel a call takes, on the host with a HIP runtime that records launches (fake_hip.py)."""
from __future__ import annotations

import pytest

from tests.fake_hip import fake_hip  # noqa: F401  (fixture)


@pytest.mark.parametrize("argument", ["q", "out"])
def test_attention_alignment(fake_hip, argument):  # noqa: F811
    # 16-byte loads and stores only where every row is 16-byte aligned; the
    # general kernel moves single values
    aligned, unaligned = fake_hip(f"""
        assert attention(64, 1000, dim=80) == 0
        aligned = kernels()
        assert attention(64, 1000, dim=80, {argument}=buffer.ptr + 4) == 0
        result = aligned, kernels()
    """)
    assert "attention_rows_kernel" in aligned[0]
    assert len(unaligned) == 1 and "16attention_kernelILi0E" in unaligned[0]


# up to 40 keys; up to 48, and from 65 to 80, where heads, tokens and dims are few
@pytest.mark.parametrize("tokens,position,small", [(2, 0, True), (4, 36, True), (40, 0, True), (2, 46, True), (2, 47, False),
                                                   (4, 60, False), (4, 61, True), (16, 64, True), (16, 65, False),
                                                   (200, 0, False)])
@pytest.mark.parametrize("heads,kv,dim", [(32, 8, 128), (8, 1, 32), (14, 2, 64)])
def test_attention_over_few_keys(fake_hip, heads, kv, dim, tokens, position, small):  # noqa: F811
    launched = fake_hip(f"""
        assert attention({tokens}, {position}, {heads}, {kv}, {dim}) == 0
        result = kernels()
    """)
    assert len(launched) <= 2 and (f"16attention_kernelILi{1 if dim > 32 else 2}E" if small else "attention_rows_kernel") in launched[0]


@pytest.mark.parametrize("rows,width,waves", [(767, 960, False), (768, 1024, True), (1000, 2048, False), (1535, 1025, False),
                                              (1536, 2048, True), (4096, 2049, False)])
def test_norm_rows(fake_hip, rows, width, waves):  # noqa: F811
    # a wave per row only where that is the faster one
    launched = fake_hip(f"""
        rt.check(lib.lh_rmsnorm(buffer.ptr, {rows}, {width}, buffer.ptr, 1e-5, 0, buffer.ptr, None))
        result = kernels()
    """)
    assert len(launched) == 1 and ("norm_wave_rows_kernel" in launched[0]) == waves


@pytest.mark.parametrize("tokens,small", [(24, True), (25, False)])
def test_attention_over_few_keys_of_many_heads(fake_hip, tokens, small):  # noqa: F811
    launched = fake_hip(f"""
        assert attention({tokens}, {72 - tokens}, 32, 8, 128) == 0
        result = kernels()
    """)
    assert len(launched) == 1 and ("16attention_kernelILi1E" if small else "attention_rows_kernel") in launched[0]
