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
    assert len(unaligned) == 1 and "16attention_kernel" in unaligned[0]
