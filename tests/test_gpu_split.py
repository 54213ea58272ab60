"""The tiled layout conversion against the general one (any block count and
alignment, byte by byte), which a destination one step off 16-byte alignment
selects: every byte the same, both ways, at block counts around the tile of
128, several matrices."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BYTES = {8: 34, 12: 144, 13: 176, 14: 210}


@pytest.fixture(scope="module")
def gpu():
    from styx_amd import Gpu
    g = Gpu(0)
    yield g
    g.close()


@pytest.mark.parametrize("t", [8, 12, 13, 14])
@pytest.mark.parametrize("nblocks,nmat", [(8, 1), (120, 3), (128, 2), (136, 5), (1000, 2)])
def test_tiled_conversion_matches_the_general_one(gpu, t, nblocks, nmat):
    from styx_amd import _lib as L
    n = nblocks * nmat * BYTES[t]
    a = np.random.default_rng(nblocks + t).integers(0, 256, n).astype(np.uint8)
    src, fast, slow, back = gpu.from_numpy(a), gpu.zeros(n + 64), gpu.zeros(n + 64), gpu.zeros(n + 64)
    to, frm = gpu.lib.styx_op_to_split, gpu.lib.styx_op_from_split
    L.check(to(gpu.h, t, src.ptr, fast.ptr, nblocks, nmat))
    L.check(to(gpu.h, t, src.ptr, slow.ptr + 8, nblocks, nmat))
    gpu.sync()
    f = fast.download()
    assert np.array_equal(f[:n], slow.download()[8:n + 8])
    assert not f[n:].any()
    L.check(frm(gpu.h, t, fast.ptr, back.ptr, nblocks, nmat))
    gpu.sync()
    b = back.download()
    assert np.array_equal(b[:n], a) and not b[n:].any()
