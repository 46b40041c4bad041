"""orc_embed and orc_dequant, one thread per eight values: rows of every type
bit for bit the oracle's dequantized rows, at row lengths that end inside a
workgroup, with ids outside the table reading row 0 and rows ldy apart."""
import numpy as np
import pytest

import oracle_lib as ol
from conftest import rand_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt,n_in", [(ol.Q4_K, 256), (ol.Q4_K, 3072), (ol.Q6_K, 256), (ol.Q6_K, 1280), (ol.Q8_0, 32),
                                     (ol.Q8_0, 1056), (ol.Q4_0, 96), (ol.F16, 992), (ol.BF16, 160), (ol.F32, 32)])
def test_embed_rows(dev, oracle, qt, n_in):
    print(f"[gpu] embed type={qt} n_in={n_in}", flush=True)
    rng = np.random.default_rng(n_in + qt)
    rows, ids = 9, np.array([3, 0, 8, -1, 9, 5, 3], np.int32)
    if qt in (ol.F32, ol.BF16):
        v = rng.normal(0, 1, (rows, n_in)).astype(np.float32)
        raw = v.view(np.uint32) if qt == ol.F32 else (v.view(np.uint32) >> 16).astype(np.uint16)
        want = v if qt == ol.F32 else (raw.astype(np.uint32) << 16).view(np.float32)
    else:
        raw = rand_blocks(qt, rows * n_in, rng)
        want = oracle.dequant(qt, raw, rows * n_in).reshape(rows, n_in)
    ldy = n_in + 4
    dw, di, dy = dev.upload(raw), dev.upload(ids), dev.upload(np.full((ids.size, ldy), 7.5, np.float32))
    dev.check(dev.L.orc_embed(qt, dw.ptr, n_in, rows, di.ptr, ids.size, dy.ptr, ldy, None))
    got = dy.read(np.float32).reshape(ids.size, ldy)
    src = np.where((ids < 0) | (ids >= rows), 0, ids)
    assert np.array_equal(got[:, :n_in].view(np.uint32), want[src].view(np.uint32))
    assert np.all(got[:, n_in:] == 7.5)
    dd = dev.alloc(4 * rows * n_in)
    dev.check(dev.L.orc_dequant(qt, dw.ptr, rows * n_in, dd.ptr, None))
    assert np.array_equal(dd.read(np.uint32).reshape(rows, n_in), want.view(np.uint32))
