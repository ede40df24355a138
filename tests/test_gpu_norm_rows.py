"""Norms of many rows (a wave per row) equal those of few (sixteen waves per row) bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [1, 64, 77, 128, 500, 960, 1024, 1025, 2048])
@pytest.mark.parametrize("rows", [768, 1031, 1536])
def test_many_rows_equal_few(width, rows):
    from leaf_amd import runtime as rt
    rng = np.random.default_rng(width + rows)
    x = (rng.standard_normal((rows, width)) * np.exp(rng.standard_normal((rows, 1)))).astype(np.float32)
    g, b = (rng.standard_normal(width).astype(np.float32) for _ in range(2))
    dx, dg, db, dy = rt.DeviceArray.of(x), rt.DeviceArray.of(g), rt.DeviceArray.of(b), rt.DeviceArray((rows, width), np.float32)
    lib, eps, part = rt.library(), np.float32(1e-5), 300
    for layer in (False, True):
        def norm(first, count):
            at = 4 * first * width
            if layer:
                rt.check(lib.lh_layernorm(dx.ptr + at, count, width, dg.ptr, db.ptr, eps, dy.ptr + at, None))
            else:
                rt.check(lib.lh_rmsnorm(dx.ptr + at, count, width, dg.ptr, eps, 0, dy.ptr + at, None))
        dy.zero()
        norm(0, rows)
        many = dy.numpy()
        dy.zero()
        for first in range(0, rows, part):
            norm(first, min(part, rows - first))
        assert np.array_equal(many.view(np.uint32), dy.numpy().view(np.uint32))
