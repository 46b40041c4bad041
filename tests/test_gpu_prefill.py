"""The prefill GEMM over split activations (csrc/orc_pf.hip): calls of 24
tokens and more on Q4_K, Q6_K, Q8_0 (GGUF and regrouped), Q4_0, F16 and BF16
weights, against the float64 product of the oracle's dequantized rows; the
kernels that captured calls of that size take; the prefill attention.

Bound of the GEMM, per (token, row), relative to sum |w x|: 2^-22 = 2.4e-7 for
the activations' split; in a 32-value block at most 12 roundings of the matrix
cores (two steps of up to three pieces, two roundings each) of 2^-23, which
round toward minus infinity: 1.4e-6; 8 blocks per 256 values, 16 superblocks of
a range and 16 ranges at 2^-24 each: 2.4e-6. That is 4.1e-6 if every rounding
had its full size and one sign; but half of the blocks are stored negated and
the roundings of the sums have either sign, so the tests hold 2e-6, as the wider
tests of the same entry points (256 tokens and more) do.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as ol
from conftest import rand_blocks

pytestmark = pytest.mark.gpu


def _weights(dev, oracle, qt, n_out, n_in, rng):
    """(device buffer, weight type of the call, float64 values)"""
    if qt == ol.BF16:
        bits = (rng.normal(0, 0.05, n_out * n_in).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        return dev.upload(bits), qt, (bits.astype(np.uint32) << 16).view(np.float32).reshape(n_out, n_in).astype(np.float64)
    gguf = ol.Q8_0 if qt == ol.Q8_0_X8 else qt
    raw = rand_blocks(gguf, n_out * n_in, rng)
    w = dev.upload(raw)
    if qt == ol.Q8_0_X8:
        dev.check(dev.L.orc_q8_0_regroup(w.ptr, n_out * n_in // 256, None))
    return w, qt, oracle.dequant(gguf, raw, n_out * n_in).reshape(n_out, n_in).astype(np.float64)


def _gemm(dev, qt, w, X, n_out, stream=None):
    n_tok, n_in = X.shape
    dx, dy = dev.upload(X), dev.alloc(n_tok * n_out * 4)
    dev.sync()
    dev.check(dev.L.orc_gemm(qt, w.ptr, n_tok, n_out, n_in, dx.ptr, n_in, dy.ptr, n_out, stream))
    dev.sync()
    return dy.read(np.float32).reshape(n_tok, n_out)


def _check(got, X, W, tol=2e-6):
    X = X.astype(np.float64)
    err, scale = np.abs(got - X @ W.T), np.abs(X) @ np.abs(W).T
    assert np.all(err <= tol * scale + 1e-30), float(np.max(err / (scale + 1e-300)))


# tile edges: 32 / 64 / 128 tokens, 32 and 128 rows; K of less than a
# superblock, of whole and of partial ones (896 and 1120 values: Q8_0, Q4_0
# and dense rows), and long enough to be split into several ranges
CASES = [(ol.Q4_K, 24, 31, 256), (ol.Q4_K, 33, 130, 2304), (ol.Q6_K, 32, 33, 256), (ol.Q6_K, 65, 127, 4352),
         (ol.Q8_0, 25, 129, 32), (ol.Q8_0, 64, 64, 896), (ol.Q8_0, 129, 97, 1120), (ol.Q8_0_X8, 128, 32, 2048),
         (ol.Q4_0, 31, 40, 1120), (ol.Q4_0, 193, 128, 96), (ol.F16, 63, 257, 4352), (ol.F16, 127, 16, 160),
         (ol.BF16, 40, 96, 4352), (ol.BF16, 130, 161, 96), (ol.Q6_K, 130, 17000, 256), (ol.F16, 300, 17000, 64)]


@pytest.mark.parametrize("qt,nt,n_out,n_in", CASES)
def test_against_float64(dev, oracle, qt, nt, n_out, n_in):
    print(f"[gpu] pf gemm type={qt} nt={nt} {n_out}x{n_in}", flush=True)
    rng = np.random.default_rng(nt + n_out)
    w, ty, W = _weights(dev, oracle, qt, n_out, n_in, rng)
    X = (rng.normal(0, 1, (nt, n_in)) * 10.0 ** rng.integers(-6, 6, (nt, 1))).astype(np.float32)
    X[nt // 2] = 0.0
    got = _gemm(dev, ty, w, X, n_out)
    _check(got, X, W)
    assert not got[nt // 2].any()
    # a token's row does not depend on the other tokens of a call of this size
    Y = rng.normal(0, 1, X.shape).astype(np.float32)
    Y[3] = X[3]
    assert np.array_equal(_gemm(dev, ty, w, Y, n_out)[3], got[3])


@pytest.mark.parametrize("qt,nt,n_in", [(ol.Q4_K, 50, 512), (ol.Q8_0, 40, 864), (ol.F16, 140, 4352)])
def test_epilogues(dev, oracle, qt, nt, n_in):
    """RMSNorm prologue with bias into three segments, SwiGLU pairs (rows not a
    multiple of 16) and residual accumulation, in float64."""
    _epilogues(dev, oracle, qt, nt, n_in, (45, 33, 50))


def _epilogues(dev, oracle, qt, nt, n_in, rows):
    import orc

    print(f"[gpu] pf epilogues type={qt} nt={nt} n_in={n_in} rows={rows}", flush=True)
    rng = np.random.default_rng(7 * nt)
    ws = [_weights(dev, oracle, qt, r, n_in, rng) for r in rows]
    X = rng.normal(0, 3, (nt, n_in)).astype(np.float32)
    g = rng.uniform(0.5, 1.5, n_in).astype(np.float32)
    dx, dg = dev.upload(X), dev.upload(g)
    Xd = X.astype(np.float64)
    Xn = Xd / np.sqrt((Xd ** 2).mean(1, keepdims=True) + 1e-5) * g
    dot = [Xn @ W.T for _, _, W in ws]
    scale = [np.abs(Xn) @ np.abs(W).T for _, _, W in ws]
    ld = sum(rows)
    bias = rng.normal(0, 1, rows[1]).astype(np.float32)
    db, dy = dev.upload(bias), dev.alloc(nt * ld * 4)
    offs = np.cumsum((0,) + rows)
    segs = (orc.Seg * 3)(*[orc.Seg(w[0].ptr, r, dy.ptr + int(o) * 4, db.ptr if i == 1 else None)
                           for i, (w, r, o) in enumerate(zip(ws, rows, offs))])
    dev.check(dev.L.orc_gemm_fused(qt, segs, 3, nt, n_in, dx.ptr, n_in, ld, dg.ptr, C.c_float(1e-5), orc.EPI_STORE,
                                   None))
    got = dy.read(np.float32).reshape(nt, ld)
    for i, r in enumerate(rows):
        want = dot[i] + (bias if i == 1 else 0)
        assert np.all(np.abs(got[:, offs[i]:offs[i + 1]] - want) <= 2e-6 * scale[i] + 3e-7 * np.abs(want)), i
    # SwiGLU over the first rows of two segments
    ff = rows[1]
    segs = (orc.Seg * 2)(orc.Seg(ws[0][0].ptr, ff, dy.ptr, None), orc.Seg(ws[1][0].ptr, ff, dy.ptr, None))
    dev.check(dev.L.orc_gemm_fused(qt, segs, 2, nt, n_in, dx.ptr, n_in, ff, dg.ptr, C.c_float(1e-5), orc.EPI_SWIGLU,
                                   None))
    got = dy.read(np.float32, nt * ff).reshape(nt, ff)
    gt, up = dot[0][:, :ff], dot[1]
    want = gt / (1 + np.exp(-gt)) * up
    tol = 3e-6 * (scale[0][:, :ff] * np.abs(up) + scale[1] * np.abs(gt)) + 1e-6 * np.abs(want) + 1e-30
    assert np.all(np.abs(got - want) <= tol)  # |silu'| <= 1.1
    res = rng.normal(0, 1, (nt, rows[2])).astype(np.float32)
    dr = dev.upload(res)
    segs = (orc.Seg * 1)(orc.Seg(ws[2][0].ptr, rows[2], dr.ptr, None))
    dev.check(dev.L.orc_gemm_fused(qt, segs, 1, nt, n_in, dx.ptr, n_in, rows[2], None, C.c_float(0), orc.EPI_ACCUM,
                                   None))
    W = ws[2][2]
    want = res + Xd @ W.T
    assert np.all(np.abs(dr.read(np.float32).reshape(nt, -1) - want) <=
                  2e-6 * (np.abs(Xd) @ np.abs(W).T) + 1.2e-7 * np.abs(want))


def test_mixed_segments(dev, oracle):
    """Q4_K and Q6_K segments of one call (a Q4_K_M layer's Q|K|V) share one split."""
    _mixed(dev, oracle, 1024, (96, 32, 64), 70)


def _mixed(dev, oracle, n_in, rows, nt):
    import orc

    rng = np.random.default_rng(5)
    types = (ol.Q4_K, ol.Q6_K, ol.Q6_K)
    ws = [_weights(dev, oracle, t, r, n_in, rng) for t, r in zip(types, rows)]
    X = rng.normal(0, 1, (nt, n_in)).astype(np.float32)
    dx, dy = dev.upload(X), dev.alloc(nt * sum(rows) * 4)
    offs = np.cumsum((0,) + rows)
    segs = (orc.Seg * 3)(*[orc.Seg(w[0].ptr, r, dy.ptr + int(o) * 4, None) for w, r, o in zip(ws, rows, offs)])
    ty = (C.c_int32 * 3)(*types)
    dev.check(dev.L.orc_gemm_fused_mixed(ty, segs, 3, nt, n_in, dx.ptr, n_in, sum(rows), None, C.c_float(0),
                                         orc.EPI_STORE, None))
    got = dy.read(np.float32).reshape(nt, -1)
    for i in range(3):
        _check(got[:, offs[i]:offs[i + 1]], X, ws[i][2])


# K-quants at sizes that go to the prefill kernels (smaller matrices stay with
# the verify kernels for these token counts): the tile edges of CASES
K_CASES = [(ol.Q4_K, 24, 8223, 256), (ol.Q4_K, 33, 4226, 2304), (ol.Q6_K, 32, 8225, 256), (ol.Q6_K, 65, 1151, 4352),
           (ol.Q4_K, 130, 1090, 1280), (ol.Q6_K, 257, 65, 512)]


@pytest.mark.parametrize("qt,nt,n_out,n_in", K_CASES)
def test_k_quants_against_float64(dev, oracle, qt, nt, n_out, n_in):
    test_against_float64(dev, oracle, qt, nt, n_out, n_in)


@pytest.mark.parametrize("qt,nt,n_in,rows", [(ol.Q4_K, 50, 512, (4173, 4161, 50)), (ol.Q6_K, 140, 2304, (1061, 1041, 33))])
def test_k_quant_epilogues(dev, oracle, qt, nt, n_in, rows):
    _epilogues(dev, oracle, qt, nt, n_in, rows)


def test_mixed_segments_at_prefill_sizes(dev, oracle):
    _mixed(dev, oracle, 1024, (2080, 1040, 1056), 70)


@pytest.mark.parametrize("qt", [ol.Q8_0, ol.F16, ol.BF16])
def test_infinities_and_nan_stay_in_their_token(dev, oracle, qt):
    """An infinite activation gives the infinity (or NaN) of the fp32 product
    in its own row, whatever else the row holds; other tokens are untouched."""
    rng = np.random.default_rng(3)
    n_in, n_out, nt = 512, 40, 30
    w, ty, W = _weights(dev, oracle, qt, n_out, n_in, rng)
    X = rng.normal(0, 1, (nt, n_in)).astype(np.float32)
    clean = _gemm(dev, ty, w, X, n_out)
    X[4, 100] = np.inf
    X[4, 101] = 1e6  # finite neighbours keep their scale
    X[9, 7] = np.nan
    got = _gemm(dev, ty, w, X, n_out)
    W32 = W[:, 100]
    assert np.array_equal(got[4][W32 > 0], np.full((W32 > 0).sum(), np.inf, np.float32))
    assert np.array_equal(got[4][W32 < 0], np.full((W32 < 0).sum(), -np.inf, np.float32))
    assert np.isnan(got[9]).all()
    keep = [t for t in range(nt) if t not in (4, 9)]
    assert np.array_equal(got[keep], clean[keep])


def test_streams_take_the_workspace_in_turn(dev, oracle):
    """Calls interleaved on two streams, without waiting in between, equal
    the same calls one after another bit for bit."""
    rng = np.random.default_rng(11)
    n_in, n_out, nt = 2048, 512, 200
    w, ty, W = _weights(dev, oracle, ol.Q6_K, n_out, n_in, rng)
    Xs = [rng.normal(0, 1, (nt, n_in)).astype(np.float32) for _ in range(6)]
    want = [_gemm(dev, ty, w, X, n_out) for X in Xs]
    dxs, dys = [dev.upload(X) for X in Xs], [dev.alloc(nt * n_out * 4) for _ in Xs]
    streams = [C.c_void_p() for _ in range(2)]
    for s in streams:
        dev.check(dev.L.orc_stream_create(C.byref(s)))
    dev.sync()
    for i, (dx, dy) in enumerate(zip(dxs, dys)):
        dev.check(dev.L.orc_gemm(ty, w.ptr, nt, n_out, n_in, dx.ptr, n_in, dy.ptr, n_out, streams[i % 2]))
    dev.sync()
    for dy, e in zip(dys, want):
        assert np.array_equal(dy.read(np.float32).reshape(nt, n_out), e)
    for s in streams:
        dev.check(dev.L.orc_stream_destroy(s))


def test_captured_calls_do_not_use_the_workspace(dev, oracle):
    """A captured call (it keeps the kernels that stage x themselves) replays
    to the same values while other calls use the workspace in between."""
    rng = np.random.default_rng(12)
    n_in, n_out, nt = 1024, 256, 48
    w, ty, W = _weights(dev, oracle, ol.Q4_K, n_out, n_in, rng)
    X = rng.normal(0, 1, (nt, n_in)).astype(np.float32)
    dx, dy = dev.upload(X), dev.alloc(nt * n_out * 4)
    s, graph = C.c_void_p(), C.c_void_p()
    dev.check(dev.L.orc_stream_create(C.byref(s)))
    dev.check(dev.L.orc_graph_begin(s))
    dev.check(dev.L.orc_gemm(ty, w.ptr, nt, n_out, n_in, dx.ptr, n_in, dy.ptr, n_out, s))
    dev.check(dev.L.orc_graph_end(s, C.byref(graph)))
    outs = []
    for _ in range(3):
        dev.check(dev.L.orc_graph_launch(graph, s))
        _check(_gemm(dev, ty, w, X[::-1].copy(), n_out), X[::-1], W)  # eager work beside the replay
        dev.sync()
        outs.append(dy.read(np.float32).reshape(nt, n_out))
        _check(outs[-1], X, W)
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    dev.check(dev.L.orc_graph_destroy(graph))
    dev.check(dev.L.orc_stream_destroy(s))


def test_token_chunks(dev, oracle):
    """More tokens than the workspace holds at once go in chunks."""
    rng = np.random.default_rng(13)
    n_in, n_out, nt = 18944, 20, 3600
    w, ty, W = _weights(dev, oracle, ol.Q6_K, n_out, n_in, rng)
    X = rng.standard_normal((nt, n_in), np.float32)
    got = _gemm(dev, ty, w, X, n_out)
    pick = np.r_[0:40, 3400:3600]  # both sides of the chunk boundary
    _check(got[pick], X[pick], W)


@pytest.mark.parametrize("H,KVH,hd,sp,nt", [(8, 1, 64, 0, 1), (7, 7, 128, 31, 33), (24, 8, 128, 4000, 30),
                                            (28, 4, 128, 95, 129), (16, 2, 64, 640, 600), (7, 7, 128, 287, 33),
                                            (3, 3, 64, 96, 33), (2, 2, 64, 60, 68), (8, 4, 128, 10, 54), (6, 2, 128, 56, 8)])
def test_prefill_attention(dev, H, KVH, hd, sp, nt):
    """The prefill attention (over split K and V, csrc/orc_attn_pf.hip, and
    k_attn_pf for the short contexts of few query heads) against float64: block
    edges of 32 positions, padded row tiles, key ranges merged
    over workgroups (few rows over a long cache), values whose scale differs by
    2^20 between key blocks and dimensions. Scores are fp32-like (2^-22 per
    product, |score| up to ~30): 4e-6 of the row's largest output. A repeat
    gives the same bits; the cache rows past the pass are untouched."""
    print(f"[gpu] pf attention H={H} KVH={KVH} hd={hd} sp={sp} nt={nt}", flush=True)
    rng = np.random.default_rng(sp + nt)
    ctx, ld = sp + nt + 40, (H + 2 * KVH) * hd
    qkv = rng.normal(0, 1, (nt, ld)).astype(np.float32)
    K, V = (rng.normal(0, 1, (KVH, ctx, hd)).astype(np.float32) for _ in range(2))
    V *= (2.0 ** rng.integers(-10, 10, (KVH, ctx // 32 + 1))).repeat(32, 1)[:, :ctx, None].astype(np.float32)
    K[:, :, : hd // 8] *= 2.0 ** -20
    th = np.arange(ctx)[:, None] / 1e4 ** (np.arange(hd // 2) * 2.0 / hd)
    tab = np.stack([np.cos(th), np.sin(th)], -1).astype(np.float32)
    dq, dt, do = dev.upload(qkv), dev.upload(tab), dev.alloc(nt * H * hd * 4)
    outs = []
    for _ in range(2):
        dK, dV = dev.upload(K), dev.upload(V)
        dev.check(dev.L.orc_attn_prefill(dq.ptr, ld, nt, H, KVH, hd, sp, dt.ptr, dK.ptr, dV.ptr, ctx, do.ptr, H * hd,
                                         None))
        outs.append(do.read(np.float32).reshape(nt, H, hd))
    assert np.array_equal(outs[0], outs[1])
    got = outs[0]
    x = qkv.astype(np.float64).reshape(nt, H + 2 * KVH, hd)
    c, s = (tab[sp:sp + nt, None, :, i].astype(np.float64) for i in range(2))

    def rope(v):
        a, b = v[..., : hd // 2], v[..., hd // 2:]
        return np.concatenate([a * c - b * s, a * s + b * c], -1)

    q, k = rope(x[:, :H]), rope(x[:, H:H + KVH])
    k64, v64 = K.astype(np.float64), V.astype(np.float64)
    k64[:, sp:sp + nt], v64[:, sp:sp + nt] = k.transpose(1, 0, 2), x[:, H + KVH:].transpose(1, 0, 2)
    Kc, Vc = dK.read(np.float32).reshape(K.shape), dV.read(np.float32).reshape(V.shape)
    assert np.allclose(Kc[:, :sp + nt], k64[:, :sp + nt], rtol=1e-6, atol=1e-6)
    assert np.array_equal(Vc[:, :sp + nt], v64[:, :sp + nt].astype(np.float32))
    assert np.array_equal(Kc[:, sp + nt:], K[:, sp + nt:]) and np.array_equal(Vc[:, sp + nt:], V[:, sp + nt:])
    mask = np.arange(sp + nt)[None] > sp + np.arange(nt)[:, None]
    for h in range(H):
        g = h // (H // KVH)
        sc = q[:, h] @ k64[g, :sp + nt].T / np.sqrt(hd)
        sc[mask] = -np.inf
        p = np.exp(sc - sc.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        want, scale = p @ v64[g, :sp + nt], p @ np.abs(v64[g, :sp + nt])
        assert np.all(np.abs(got[:, h] - want) <= 4e-6 * scale.max(1, keepdims=True)), h


def test_prefill_attention_captured_and_streams(dev):
    """A captured call keeps the kernel without the workspace and replays to
    fp32 rounding of the other; calls on a second stream take the workspace in
    turn (same bits)."""
    rng = np.random.default_rng(4)
    H, KVH, hd, sp, nt = 8, 2, 64, 50, 70
    ctx, ld = 128, (H + 2 * KVH) * hd
    qkv = rng.normal(0, 1, (nt, ld)).astype(np.float32)
    K, V = (rng.normal(0, 1, (KVH, ctx, hd)).astype(np.float32) for _ in range(2))
    th = np.arange(ctx)[:, None] / 1e4 ** (np.arange(hd // 2) * 2.0 / hd)
    dt = dev.upload(np.stack([np.cos(th), np.sin(th)], -1).astype(np.float32))
    dq, dK, dV = dev.upload(qkv), dev.upload(K), dev.upload(V)
    dos = [dev.alloc(nt * H * hd * 4) for _ in range(5)]

    def run(do, s):
        dev.check(dev.L.orc_attn_prefill(dq.ptr, ld, nt, H, KVH, hd, sp, dt.ptr, dK.ptr, dV.ptr, ctx, do.ptr, H * hd,
                                         s))

    s, graph = C.c_void_p(), C.c_void_p()
    dev.check(dev.L.orc_stream_create(C.byref(s)))
    run(dos[0], None)
    dev.sync()
    want = dos[0].read(np.float32)
    for i, st in enumerate((s, None, s)):
        run(dos[1 + i], st)
    dev.sync()
    for i in range(3):
        assert np.array_equal(dos[1 + i].read(np.float32), want), i
    dev.check(dev.L.orc_graph_begin(s))
    run(dos[4], s)
    dev.check(dev.L.orc_graph_end(s, C.byref(graph)))
    for _ in range(3):
        dev.check(dev.L.orc_graph_launch(graph, s))
        run(dos[0], None)
        dev.sync()
        assert np.array_equal(dos[0].read(np.float32), want)
        assert np.allclose(dos[4].read(np.float32), want, rtol=0, atol=4e-6 * np.abs(want).max())
    dev.check(dev.L.orc_graph_destroy(graph))
    dev.check(dev.L.orc_stream_destroy(s))
    run(dos[0], None)  # the workspace's last use was on the destroyed stream or on this one
    dev.sync()
    assert np.array_equal(dos[0].read(np.float32), want)


# narrow matrices above 32 tokens (32-token tiles, a short K in up to four
# ranges): one and several ranges, ragged tokens and rows, and on both sides
# of the line to 64-token tiles (256 workgroups of those: 16 row blocks here)
@pytest.mark.parametrize("qt,nt,n_out,n_in", [(ol.Q8_0, 33, 896, 896), (ol.Q8_0, 257, 129, 896), (ol.Q8_0, 1023, 896, 896),
                                              (ol.Q4_0, 512, 33, 96), (ol.Q4_K, 48, 3072, 3072), (ol.Q6_K, 97, 130, 1280),
                                              (ol.BF16, 190, 96, 1024), (ol.F16, 95, 31, 4352), (ol.Q8_0, 1024, 2048, 64),
                                              (ol.Q8_0, 960, 2048, 64)])
def test_narrow_matrices(dev, oracle, qt, nt, n_out, n_in):
    print(f"[gpu] pf narrow type={qt} nt={nt} {n_out}x{n_in}", flush=True)
    rng = np.random.default_rng(nt + n_in)
    w, ty, W = _weights(dev, oracle, qt, n_out, n_in, rng)
    X = rng.normal(0, 1, (nt, n_in)).astype(np.float32)
    _check(_gemm(dev, ty, w, X, n_out), X, W)


def _attn_case(dev, H, KVH, hd, sp, nt, S, K, V, qkv):
    """orc_attn_prefill without rotation (angles 0), and the float64 result
    over each row's own positions: (got, weights p [nt, H, S], float64 V)."""
    ctx, ld = K.shape[1], (H + 2 * KVH) * hd
    tab = np.zeros((ctx, hd // 2, 2), np.float32)
    tab[..., 0] = 1
    dq, dt, dK, dV = dev.upload(qkv), dev.upload(tab), dev.upload(K), dev.upload(V)
    do = dev.alloc(nt * H * hd * 4)
    dev.check(dev.L.orc_attn_prefill(dq.ptr, ld, nt, H, KVH, hd, sp, dt.ptr, dK.ptr, dV.ptr, ctx, do.ptr, H * hd, None))
    got = do.read(np.float32).reshape(nt, H, hd)
    x = qkv.astype(np.float64).reshape(nt, H + 2 * KVH, hd)
    k64, v64 = K.astype(np.float64), V.astype(np.float64)
    k64[:, sp:sp + nt], v64[:, sp:sp + nt] = x[:, H:H + KVH].transpose(1, 0, 2), x[:, H + KVH:].transpose(1, 0, 2)
    p = np.zeros((nt, H, S))
    for t in range(nt):
        for h in range(H):
            s = x[t, h] @ k64[h // (H // KVH), :sp + t + 1].T / np.sqrt(hd)
            with np.errstate(invalid="ignore"):  # a row that sees an infinity
                e = np.exp(s - s.max())
                p[t, h, :sp + t + 1] = e / e.sum()
    return got, p, v64


def _scored(rng, H, KVH, hd, sp, nt, score, vscale):
    """Inputs whose score of position j is score[j] (every query is the same
    unit vector, every key that many times it) and whose V row j has the
    magnitude vscale[j]."""
    S = sp + nt
    u = rng.normal(0, 1, hd)
    u *= np.sqrt(np.sqrt(hd) / (u @ u))  # u . u / sqrt(hd) = 1
    k = (score[:, None] * u).astype(np.float32)
    qkv = np.zeros((nt, H + 2 * KVH, hd), np.float32)
    qkv[:, :H] = u
    K, V = np.zeros((KVH, S + 8, hd), np.float32), np.zeros((KVH, S + 8, hd), np.float32)
    v = (rng.normal(0, 1, (KVH, S, hd)) * vscale[None, :, None]).astype(np.float32)
    K[:, :sp], V[:, :sp] = k[:sp], v[:, :sp]
    qkv[:, H:H + KVH], qkv[:, H + KVH:] = k[sp:, None], v[:, sp:].transpose(1, 0, 2)
    return S, K, V, qkv.reshape(nt, -1)


def _rows_within(got, p, v64, R, tol=6e-6):
    """|error| <= tol times the row's sum of p_j max |v_j|: rounding in fp32 or
    22 bits (2.4e-7 a product) of the two factors of every product, the
    weights' own error (scores up to 40: 40 * 2^-24 = 2.4e-6) and the sums."""
    v = np.repeat(v64, R, 0)
    want, scale = np.einsum("ths,hsd->thd", p, v[:, :p.shape[2]]), np.einsum("ths,hs->th", p, np.abs(v[:, :p.shape[2]]).max(2))
    err = np.abs(got - want).max(2) / scale
    assert err.max() <= tol, (float(err.max()), np.unravel_index(err.argmax(), err.shape))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("big,drop", [(24, 40), (40, 60), (24, 17), (40, 28), (60, 80), (-40, 0)])
def test_prefill_attention_v_ranges_over_blocks(dev, hd, big, drop):
    """V of some blocks of 32 positions 2^big times the others', with scores
    that give those positions exp(-drop) of the weight: a negligible large V, a
    large V whose contribution is comparable, and a small V that carries all."""
    print(f"[gpu] pf attention V range hd={hd} 2^{big} drop {drop}", flush=True)
    rng = np.random.default_rng(hd + big + drop)
    H, KVH, sp, nt = 4, 2, 300, 70
    S = sp + nt
    j = np.arange(S)
    for blocks in ([0, 1], [4], [10], [0, 3, 6, 9]):
        m = np.isin(j // 32, blocks)
        score = np.where(m, -float(drop), rng.uniform(-2, 0, S))
        vscale = np.where(m, 2.0 ** big, 1.0)
        got, p, v64 = _attn_case(dev, H, KVH, hd, sp, nt, *_scored(rng, H, KVH, hd, sp, nt, score, vscale))
        _rows_within(got, p, v64, H // KVH)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("what", ["v", "v_comparable", "v_later", "k_later", "k_low"])
def test_prefill_attention_ranges_inside_a_block(dev, hd, what):
    """V (or K) rows 2^20 to 2^50 apart inside a block of 32 positions, the
    large ones of little weight, of comparable weight, or not seen by the
    earlier tokens of the pass."""
    print(f"[gpu] pf attention range in a block hd={hd} {what}", flush=True)
    rng = np.random.default_rng(hd + len(what))
    H, KVH, sp, nt = 6, 2, 77, 90
    S = sp + nt
    j = np.arange(S)
    score, vscale = rng.uniform(-2, 0, S), np.ones(S)
    big = (j % 5 == 2) & (j > 20)
    if what == "v":
        score[big], vscale[big] = -60.0, 2.0 ** rng.integers(20, 50, big.sum())
    elif what == "v_comparable":
        b = rng.integers(20, 50, big.sum())
        score[big], vscale[big] = -b * np.log(2.0) + rng.uniform(-2, 2, big.sum()), 2.0 ** b
    elif what == "v_later":
        vscale[j >= sp + 50] = 2.0 ** 40
    elif what == "k_later":
        score[j >= sp + 50] = 2.0 ** 30 * rng.choice([-1, 1], nt - 50)
    else:
        score[big] = -2.0 ** 30
    got, p, v64 = _attn_case(dev, H, KVH, hd, sp, nt, *_scored(rng, H, KVH, hd, sp, nt, score, vscale))
    n = 50 if what == "k_later" else nt  # (scores near 2^30 tie in fp32: tokens that see them are not compared)
    _rows_within(got[:n], p[:n], v64, H // KVH)


@pytest.mark.parametrize("H,KVH,hd,nt", [(4, 4, 64, 150), (8, 2, 64, 40), (4, 4, 128, 150), (14, 2, 128, 70)])
def test_prefill_attention_infinities_reach_no_earlier_token(dev, H, KVH, hd, nt):
    """A V or K row with an infinity or NaN changes no token before its
    position; later tokens have it in the dimensions it is in."""
    print(f"[gpu] pf attention infinities H={H} KVH={KVH} hd={hd} nt={nt}", flush=True)
    rng = np.random.default_rng(H + hd)
    sp = 45
    S, K, V, qkv = _scored(rng, H, KVH, hd, sp, nt, rng.uniform(-2, 0, sp + nt), np.ones(sp + nt))
    qkv = qkv.reshape(nt, H + 2 * KVH, hd)
    at = nt - 7
    want, p, v64 = _attn_case(dev, H, KVH, hd, sp, nt, S, K, V, qkv.reshape(nt, -1))
    for bad in (np.inf, -np.inf, np.nan):
        q = qkv.copy()
        q[at, H + KVH:, 3] = bad
        got, _, _ = _attn_case(dev, H, KVH, hd, sp, nt, S, K, V, q.reshape(nt, -1))
        _rows_within(got[:at], p[:at], v64, H // KVH)
        assert np.array_equal(got[at:, :, 3], np.full((nt - at, H), bad, np.float32), equal_nan=True)
        rest = np.r_[0:3, 4:hd]
        assert np.allclose(got[at:][:, :, rest], want[at:][:, :, rest], rtol=0, atol=2e-5)
        q = qkv.copy()
        q[at, H:H + KVH, 3] = bad
        got, _, _ = _attn_case(dev, H, KVH, hd, sp, nt, S, K, V, q.reshape(nt, -1))
        _rows_within(got[:at], p[:at], v64, H // KVH)
    # in the cache before the pass: every token has it
    V2 = V.copy()
    V2[:, 40, 5] = np.inf
    got, _, _ = _attn_case(dev, H, KVH, hd, sp, nt, S, K, V2, qkv.reshape(nt, -1))
    assert np.isposinf(got[:, :, 5]).all() and np.isfinite(np.delete(got, 5, 2)).all()


def test_tall_dense_matrix_in_chunks(dev, oracle):
    """A tall F16 matrix of long rows: the sums of its two ranges leave room
    for 64 tokens at a time. 262144 rows that repeat 64."""
    print("[gpu] pf tall F16 262144 x 8192, 130 tokens", flush=True)
    rng = np.random.default_rng(14)
    n_in, base, n_out, nt = 8192, 64, 262144, 130
    w, ty, W = _weights(dev, oracle, ol.F16, base, n_in, rng)
    big = dev.alloc(n_out * n_in * 2)
    done = base * n_in * 2
    dev.check(dev.L.orc_memcpy_d2d(big.ptr, w.ptr, done, None))
    while done < n_out * n_in * 2:
        dev.check(dev.L.orc_memcpy_d2d(big.ptr + done, big.ptr, done, None))
        done *= 2
    X = rng.normal(0, 1, (nt, n_in)).astype(np.float32)
    got = _gemm(dev, ty, big, X, n_out).reshape(nt, -1, base)
    _check(got[:, 0], X, W)
    assert (got == got[:, :1]).all()


def _captured(dev, call, outs, runs=3):
    """call(stream) captured on a stream of its own and replayed `runs` times,
    with eager work between; the outputs of every replay are the same bits."""
    s, graph = C.c_void_p(), C.c_void_p()
    dev.check(dev.L.orc_stream_create(C.byref(s)))
    dev.check(dev.L.orc_graph_begin(s))
    call(s)
    dev.check(dev.L.orc_graph_end(s, C.byref(graph)))
    got = []
    for _ in range(runs):
        for o in outs:
            dev.check(dev.L.orc_fill(o.ptr, 0xFF, o.nbytes, s))
        dev.check(dev.L.orc_graph_launch(graph, s))
        dev.sync()
        got.append([o.read(np.float32) for o in outs])
        call(None)  # the same call eagerly, over the workspace
        dev.sync()
    for g in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(g, got[0]))
    dev.check(dev.L.orc_graph_destroy(graph))
    dev.check(dev.L.orc_stream_destroy(s))
    return got[0]


@pytest.mark.parametrize("qt,nt,n_out,n_in", [(ol.Q4_K, 300, 300, 3072), (ol.Q6_K, 263, 200, 18944), (ol.Q6_K, 256, 130, 2048),
                                              (ol.Q8_0, 263, 200, 896), (ol.Q8_0, 256, 70, 4864),
                                              (ol.Q8_0_X8, 256, 257, 3072), (ol.Q4_0, 256, 40, 1120), (ol.F16, 260, 40, 512)])
def test_captured_prefill_gemm(dev, oracle, qt, nt, n_out, n_in):
    """Captured calls of 256 tokens and more: k_mmq_pf for the K-quants and
    Q8_0 (64 tokens per workgroup), the vector kernels' token blocks else."""
    print(f"[gpu] captured gemm type={qt} nt={nt} {n_out}x{n_in}", flush=True)
    rng = np.random.default_rng(nt + n_in)
    w, ty, W = _weights(dev, oracle, qt, n_out, n_in, rng)
    X = rng.normal(0, 1, (nt, n_in)).astype(np.float32)
    dx, dy = dev.upload(X), dev.alloc(nt * n_out * 4)
    got, = _captured(dev, lambda s: dev.check(dev.L.orc_gemm(ty, w.ptr, nt, n_out, n_in, dx.ptr, n_in, dy.ptr, n_out, s)), [dy])
    _check(got.reshape(nt, n_out), X, W)


@pytest.mark.parametrize("qt", [ol.Q4_K, ol.Q6_K, ol.Q8_0])
def test_captured_prefill_epilogues(dev, oracle, qt):
    """k_mmq_pf's norm, bias, SwiGLU (Q8_0: two passes over the output) and
    residual sums against float64; no pass reads what a replay before it left."""
    import orc

    rng = np.random.default_rng(20)
    nt, n_in, rows = 300, 1024, (144, 80)
    ws = [_weights(dev, oracle, qt, r, n_in, rng) for r in rows]
    X = rng.normal(0, 2, (nt, n_in)).astype(np.float32)
    g, bias = rng.uniform(0.5, 1.5, n_in).astype(np.float32), rng.normal(0, 1, rows[1]).astype(np.float32)
    dx, dg, db, dy, dh = dev.upload(X), dev.upload(g), dev.upload(bias), dev.alloc(nt * sum(rows) * 4), dev.alloc(nt * 80 * 4)
    print(f"[gpu] captured epilogues type={qt}", flush=True)

    def call(s):
        segs = (orc.Seg * 2)(orc.Seg(ws[0][0].ptr, rows[0], dy.ptr, None), orc.Seg(ws[1][0].ptr, rows[1], dy.ptr + 4 * rows[0], db.ptr))
        dev.check(dev.L.orc_gemm_fused(qt, segs, 2, nt, n_in, dx.ptr, n_in, sum(rows), dg.ptr, C.c_float(1e-5), orc.EPI_STORE, s))
        segs = (orc.Seg * 2)(orc.Seg(ws[0][0].ptr, 80, dh.ptr, None), orc.Seg(ws[1][0].ptr, 80, dh.ptr, None))
        dev.check(dev.L.orc_gemm_fused(qt, segs, 2, nt, n_in, dx.ptr, n_in, 80, dg.ptr, C.c_float(1e-5), orc.EPI_SWIGLU, s))
        segs = (orc.Seg * 1)(orc.Seg(ws[1][0].ptr, 80, dh.ptr, None))
        dev.check(dev.L.orc_gemm_fused(qt, segs, 1, nt, n_in, dx.ptr, n_in, 80, None, C.c_float(0), orc.EPI_ACCUM, s))

    y, h = _captured(dev, call, [dy, dh])
    Xd = X.astype(np.float64)
    Xn = Xd / np.sqrt((Xd ** 2).mean(1, keepdims=True) + 1e-5) * g
    dot, scale = [Xn @ w[2].T for w in ws], [np.abs(Xn) @ np.abs(w[2]).T for w in ws]
    want = np.concatenate([dot[0], dot[1] + bias], 1)
    assert np.all(np.abs(y.reshape(nt, -1) - want) <= 2e-6 * np.concatenate(scale, 1) + 3e-7 * np.abs(want))
    gt, up = dot[0][:, :80], dot[1]
    act = gt / (1 + np.exp(-gt)) * up
    res = Xd @ ws[1][2].T
    tol = 3e-6 * (scale[0][:, :80] * np.abs(up) + scale[1] * np.abs(gt)) + 2e-6 * (np.abs(Xd) @ np.abs(ws[1][2]).T) + 1e-6 * np.abs(act)
    assert np.all(np.abs(h.reshape(nt, -1) - (act + res)) <= tol)  # |silu'| <= 1.1


@pytest.mark.parametrize("H,KVH,hd,sp,nt", [(8, 2, 128, 500, 70), (14, 2, 64, 700, 33)])
def test_captured_attention_of_long_contexts(dev, H, KVH, hd, sp, nt):
    """k_attn_pf, which an eager call of these sizes does not take, against
    the eager call: both within 4e-6 of float64 (the largest output)."""
    print(f"[gpu] captured attention H={H} KVH={KVH} hd={hd} sp={sp} nt={nt}", flush=True)
    rng = np.random.default_rng(sp)
    ctx, ld = sp + nt, (H + 2 * KVH) * hd
    qkv = rng.normal(0, 1, (nt, ld)).astype(np.float32)
    K, V = (rng.normal(0, 1, (KVH, ctx, hd)).astype(np.float32) for _ in range(2))
    th = np.arange(ctx)[:, None] / 1e4 ** (np.arange(hd // 2) * 2.0 / hd)
    dt = dev.upload(np.stack([np.cos(th), np.sin(th)], -1).astype(np.float32))
    dq, dK, dV, do = dev.upload(qkv), dev.upload(K), dev.upload(V), dev.alloc(nt * H * hd * 4)

    def call(s):
        dev.check(dev.L.orc_attn_prefill(dq.ptr, ld, nt, H, KVH, hd, sp, dt.ptr, dK.ptr, dV.ptr, ctx, do.ptr, H * hd, s))

    got, = _captured(dev, call, [do])
    want = do.read(np.float32)  # the last eager call's
    assert np.allclose(got, want, rtol=0, atol=8e-6 * np.abs(want).max())


@pytest.mark.parametrize("H,KVH,hd,nt", [(8, 1, 64, 200), (28, 4, 128, 40)])
def test_prefill_attention_of_one_key(dev, H, KVH, hd, nt):
    """The first token's weight is 1 exactly: its output is V to the split of
    V alone, at most 2^-23 of a value and 2^-23 / sqrt(3) = 6.9e-8 over many."""
    print(f"[gpu] pf attention of one key H={H} KVH={KVH} hd={hd} nt={nt}", flush=True)
    rng = np.random.default_rng(hd)
    num = den = 0.0
    for _ in range(8):
        qkv = rng.normal(0, 1, (nt, (H + 2 * KVH) * hd)).astype(np.float32)
        K = np.zeros((KVH, nt, hd), np.float32)
        got, _, v64 = _attn_case(dev, H, KVH, hd, 0, nt, nt, K, K.copy(), qkv)
        v = np.repeat(v64[:, 0], H // KVH, 0)
        num, den = num + ((got[0] - v) ** 2).sum(), den + (v ** 2).sum()
    assert np.sqrt(num / den) <= 6.9e-8, np.sqrt(num / den)
