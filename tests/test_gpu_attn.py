"""GPU tests of the attention kernels' dispatch edges (csrc/uq_attn.hip):
softmax rows around every row-kernel size, outputs that sit on f32 rounding
midpoints (the reference's sequential sum replayed by a workgroup), the
prefill's tile kernels against single-query steps over long caches and for
every head group, undecided outputs in them, and operands that are zero, huge,
infinite or NaN. Every comparison is bit for bit (a NaN equals a NaN): the
kernels' contract is the reference's own bits.
"""
import numpy as np
import pytest

import oracle as O
import uq
import uq.synth as S
from uq import layer as L
from uq import ops
from helpers import microseconds
from test_gpu_layer_prefill import prefill_rows
from test_gpu_layers import SMALL, Model, nodes_of
from test_gpu_ops import assert_bitwise, check_attn, softmax_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows", [(1, 3), (255, 2), (256, 2), (257, 2), (3, 5000), (200, 3000), (1024, 2),
                                    (1025, 2), (4096, 2), (4097, 2), (8193, 2), (16385, 2), (32768, 2), (32769, 2),
                                    (1500, 600), (2049, 600), (4095, 600)])
def test_softmax_rows_at_the_row_kernels_edges(n, rows):
    rng = np.random.default_rng(n + rows)
    X = rng.standard_normal((rows, n)).astype(np.float32) * 5
    d = uq.DeviceArray.from_numpy(X)
    ops.softmax_d(d, d, n, rows, 0.5)
    uq.synchronize()
    got = d.download(np.float32, rows * n).reshape(rows, n)
    for r in {0, 1, rows - 1}:
        assert_bitwise(got[r], softmax_model(X[r], 0.5), f"softmax n={n} row {r}")


def midpoint_column(rng, n, w):
    """n f32 values whose sum of w v in position order is within an f64 ulp or
    two of the midpoint of two f32 values: ever smaller values close the gap."""
    v = rng.standard_normal(n).astype(np.float32)
    v[-6:] = 0.0
    s = float(np.add.accumulate(w * v.astype(np.float64))[-1])
    lo = np.float32(s)
    mid = (float(lo) + float(np.nextafter(lo, np.float32(np.inf)))) / 2
    for k in range(n - 6, n):
        v[k] = np.float32((mid - s) / w)
        s = float(np.add.accumulate(w * v.astype(np.float64))[-1])
    assert abs(s - mid) <= 4 * np.spacing(abs(mid)), "the column does not reach the midpoint"
    return v


@pytest.mark.parametrize("n_ctx", [40, 160, 161, 320, 321, 1000, 5000, 20000])
@pytest.mark.parametrize("cols", [(5,), (0, 1, 17, 18, 63), tuple(range(16, 27))])
def test_attn_decode_outputs_on_midpoints(n_ctx, cols):
    """Equal weights, value columns planted on f32 midpoints: no bound decides
    them. One, a few (over more than 160 positions an output a workgroup replays
    each) and eleven of one workgroup's columns (each lane its own)."""
    hd = 64
    rng = np.random.default_rng(n_ctx + len(cols))
    w = float(O.softmax(np.zeros(n_ctx, np.float32), 1.0)[0])
    vc = rng.standard_normal((n_ctx, hd)).astype(np.float32)
    for c in cols:
        vc[:, c] = midpoint_column(rng, n_ctx, w)
    check_attn(np.ones(hd, np.float32), np.ones(n_ctx * hd, np.float32), vc.reshape(-1), n_ctx, 1, 1, hd, 1.0,
               f"midpoints n={n_ctx}", bit_exact_soft=True)


def attn_layer(m, X, K, V, n_ctx_max, pos0, prefill):
    d, (nt, n) = m.d, X.shape
    kc, vc, dx, dl = (uq.DeviceArray.from_numpy(a) for a in (K, V, X, np.zeros_like(X)))
    ws = uq.DeviceArray(4 * max(L.ws_floats(d, n_ctx_max), L.prefill_ws_floats(d, nt, attn=m.aw, n_ctx_max=n_ctx_max)))
    out = np.empty_like(X)
    if prefill:
        L.attn_prefill(d, m.aw, kc, vc, n_ctx_max, pos0, nt, dx, dl, ws)
        out = dl.download(np.float32, nt * n).reshape(nt, n)
    else:
        for t in range(nt):
            one = uq.DeviceArray.from_numpy(X[t])
            L.attn_step(d, m.aw, kc, vc, n_ctx_max, pos0 + t, one, dl, ws)
            out[t] = dl.download(np.float32, n)
            one.free()
    for a in (kc, vc, dx, dl, ws):
        a.free()
    return out


@pytest.mark.parametrize("shape,nt,pos0", [
    (dict(n_head=8, n_head_kv=2, head_dim=64), 3, 1700),  # queries by themselves
    (dict(n_head=8, n_head_kv=2, head_dim=64), 90, 1009),  # scores in tiles, values by themselves
    (dict(n_head=8, n_head_kv=2, head_dim=64), 333, 29),  # both in tiles
    (dict(n_embd=1280, n_v_heads=20, n_head=5, n_head_kv=1, head_dim=256), 65, 1100),  # group 5
    (dict(n_embd=768, n_v_heads=12, n_head=6, n_head_kv=2, head_dim=128), 130, 2051),  # group 3
    (dict(n_head=1, n_head_kv=1, head_dim=512, n_rot=32), 140, 600)])  # scores by themselves, values in tiles
def test_attn_prefill_over_a_long_cache_equals_steps(shape, nt, pos0):
    m = Model(dict(SMALL, **shape), seed=71 + nt)
    c = m.cfg
    rng = np.random.default_rng(nt + pos0)
    n_ctx_max = pos0 + nt + 3
    K, V = (rng.standard_normal(n_ctx_max * c.n_head_kv * c.head_dim).astype(np.float32) for _ in range(2))
    X = rng.standard_normal((nt, c.n_embd)).astype(np.float32)
    ref = attn_layer(m, X, K, V, n_ctx_max, pos0, False)
    got = attn_layer(m, X, K, V, n_ctx_max, pos0, True)
    for t in range(nt):
        assert_bitwise(got[t], ref[t], f"attn {shape} token {t} of {nt} at {pos0}")
    ref, _ = gated_rows(m, X, K, V, n_ctx_max, pos0, False)
    got, _ = gated_rows(m, X, K, V, n_ctx_max, pos0, True)
    for t in range(nt):
        assert_bitwise(got[t], ref[t], f"gated attn {shape} token {t} of {nt} at {pos0}")
    m.free()


def gated_rows(m, X, K, V, n_ctx_max, pos0, prefill):
    """The attention outputs times the gates, before the output projection
    quantizes them to eight bits, and the V cache: by one prefill or by steps."""
    d, (nt, n) = m.d, X.shape
    kc, vc, dx, dl = (uq.DeviceArray.from_numpy(a) for a in (K, V, X, np.zeros_like(X)))
    ws = uq.DeviceArray(4 * max(L.ws_floats(d, n_ctx_max), L.prefill_ws_floats(d, nt, attn=m.aw, n_ctx_max=n_ctx_max)))
    if prefill:
        L.attn_prefill(d, m.aw, kc, vc, n_ctx_max, pos0, nt, dx, dl, ws)
        out = prefill_rows(m, ws, nt, n_ctx_max, "gated")
    else:
        out = np.empty((nt, m.cfg.n_head * m.cfg.head_dim), np.float32)
        for t in range(nt):
            one = uq.DeviceArray.from_numpy(X[t])
            L.attn_step(d, m.aw, kc, vc, n_ctx_max, pos0 + t, one, dl, ws)
            out[t] = nodes_of(d, ws, ["gated"], n_ctx_max)["gated"]
            one.free()
    V = vc.download(np.float32, vc.nbytes // 4).reshape(n_ctx_max, m.cfg.n_head_kv, m.cfg.head_dim)
    for a in (kc, vc, dx, dl, ws):
        a.free()
    return out, V


@pytest.mark.parametrize("shape,nt,pos0", [
    (dict(n_embd=768, n_v_heads=12, n_head=6, n_head_kv=2, head_dim=128), 301, 9),  # 3
    (dict(n_embd=1280, n_v_heads=20, n_head=5, n_head_kv=1, head_dim=256), 250, 0),  # 5
    (dict(n_embd=768, n_v_heads=12, n_head=12, n_head_kv=2, head_dim=64), 601, 3),  # 6
    (dict(n_embd=1792, n_v_heads=28, n_head=7, n_head_kv=1, head_dim=256), 203, 21),  # 7
    (dict(n_embd=1024, n_v_heads=16, n_head=8, n_head_kv=1, head_dim=128), 500, 29)])  # 8
def test_attn_prefill_pair_tiles_of_every_head_group(shape, nt, pos0):
    """Tokens enough for the values' pair tiles (1.4 to 2 times the rule's
    line), groups that do not divide a tile's 64 pairs among them: a tile
    starts and ends inside a token, the last one partly filled."""
    m = Model(dict(SMALL, **shape), seed=101 + nt)
    c = m.cfg
    rng = np.random.default_rng(nt)
    n_ctx_max = pos0 + nt + 2
    K, V = (rng.standard_normal((n_ctx_max, c.n_head_kv, c.head_dim)).astype(np.float32) for _ in range(2))
    X = rng.standard_normal((nt, c.n_embd)).astype(np.float32)
    ref, _ = gated_rows(m, X, K, V, n_ctx_max, pos0, False)
    got, _ = gated_rows(m, X, K, V, n_ctx_max, pos0, True)
    for t in range(nt):
        assert_bitwise(got[t], ref[t], f"attn {shape} token {t} of {nt} at {pos0}")
    m.free()


@pytest.mark.parametrize("pos0", [28, 428])
def test_attn_prefill_undecided_outputs_in_pair_tiles(pos0):
    """Zero tokens weigh every position alike, and cached V columns of
    [2^62, 1, -2^62, 1] then cancel: their sums depend on the order and no bound
    decides them. Tokens 7 and 21, 21, 75, 105, 200, 329 put 1 to 4 pairs into
    tiles (groups of 3: token 21 lies in two of them), times two columns of a
    workgroup's 64 (at most eight, replayed by the workgroup over more than 160
    positions) or four (each lane its own), in every quarter of a tile's columns
    and of its pairs."""
    m = Model(dict(SMALL, n_embd=768, n_v_heads=12, n_head=6, n_head_kv=2, head_dim=128), seed=103)
    c, nt, zero = m.cfg, 330, [7, 21, 75, 105, 200, 329]
    planted = [(0, 5), (0, 60), (0, 64 + 19), (0, 64 + 33), (1, 0), (1, 17), (1, 33), (1, 50)]
    rng = np.random.default_rng(8)
    K, V = (rng.standard_normal((pos0 + nt, c.n_head_kv, c.head_dim)).astype(np.float32) for _ in range(2))
    for kv, col in planted:
        V[:pos0, kv, col] = np.tile(np.array([2.0 ** 62, 1.0, -(2.0 ** 62), 1.0], np.float32), pos0 // 4)
    X = rng.standard_normal((nt, c.n_embd)).astype(np.float32)
    X[zero] = 0.0
    ref, _ = gated_rows(m, X, K, V, pos0 + nt, pos0, False)
    got, after = gated_rows(m, X, K, V, pos0 + nt, pos0, True)
    for z in zero:  # the reference's sum, its gate sigmoid(0) = 0.5
        n = pos0 + z + 1
        t = float(O.softmax(np.zeros(n, np.float32), 1.0)[0]) * after[:n].astype(np.float64)
        seq = np.add.accumulate(t)[-1].astype(np.float32)
        other = np.add.accumulate(t[::-1])[-1].astype(np.float32)
        assert all(seq[p] != other[p] for p in planted), "another order gives the planted columns' values too"
        assert_bitwise(got[z], np.repeat(np.float32(0.5) * seq, c.n_head // c.n_head_kv, axis=0).reshape(-1), f"zero token {z}")
    for t in range(nt):
        assert_bitwise(got[t], ref[t], f"attn undecided, token {t}")
    m.free()


def test_attn_prefill_later_infinity_stays_out_of_earlier_tokens():
    """Token 200's value row overflows to infinity. Tokens 192 .. 199 share
    its pair tile, where the row meets their masked (zero) weights; the
    reference, and the steps, read no position past a token's own."""
    m = Model(dict(SMALL, n_head=8, n_head_kv=2, head_dim=64), seed=83)
    c, nt, pos0, late = m.cfg, 333, 29, 200
    nv = c.n_head_kv * c.head_dim
    wv = S.weights(S.Q4_K, nv, c.n_embd, seed=5, sigma=0.05).reshape(-1, S.BLOCK_BYTES[S.Q4_K])
    wv[:, 2:4] = 0  # dmin 0: an overflowing value is an infinity, never inf - inf
    norm = m.ah["attn_norm"].copy()
    norm[7] = 1e37
    extra = uq.Weights(wv.reshape(-1), S.Q4_K, c.n_embd, nv), uq.DeviceArray.from_numpy(norm)
    m.dev += extra
    m.aw.attn_v, m.aw.attn_norm = extra
    rng = np.random.default_rng(4)
    X = rng.standard_normal((nt, c.n_embd)).astype(np.float32)
    X[:, 7] = 0.0  # only the late token meets the large norm weight
    X[late] = 0.0
    X[late, 7] = 1.0
    n_ctx_max = pos0 + nt
    K, V = (rng.standard_normal((n_ctx_max, nv)).astype(np.float32) for _ in range(2))
    ref = attn_layer(m, X[:late + 1], K, V, n_ctx_max, pos0, False)
    got = attn_layer(m, X, K, V, n_ctx_max, pos0, True)
    assert not np.isfinite(ref[late]).all(), "the late token's values do not overflow"
    for t in range(late):
        assert_bitwise(got[t], ref[t], f"attn token {t}, an infinite value row at token {late}")
    m.free()


@pytest.mark.parametrize("n_ctx", [40, 1100, 5000])
def test_attn_decode_huge_values_under_underflowed_weights(n_ctx):
    """|V| of 3e38 wherever the weight underflows to zero: finite, and zero in
    the reference's sum, though a few such |V| added in f32 are infinite."""
    hd = 64
    rng = np.random.default_rng(n_ctx)
    far = np.arange(n_ctx) % 16 == 3
    kc = np.where(far[:, None], -3.0, 1.0).astype(np.float32) * np.ones((n_ctx, hd), np.float32)
    vc = rng.standard_normal((n_ctx, hd)).astype(np.float32)
    vc[far] = rng.choice([-3e38, 3e38], (int(far.sum()), hd)).astype(np.float32)
    got = check_attn(np.ones(hd, np.float32), kc.reshape(-1), vc.reshape(-1), n_ctx, 1, 1, hd, 1.0,
                     f"huge values n={n_ctx}", bit_exact_soft=True)
    assert np.isfinite(got).all()


@pytest.mark.parametrize("hd,nh,nhkv", [(64, 8, 2), (256, 6, 1), (512, 2, 2)])
def test_attn_decode_zero_rows(hd, nh, nhkv):
    """A zero q head, zero K rows (one K row whose norm leaves the f32 range
    beside them) and zero V columns."""
    n_ctx = 700
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((nh, hd)).astype(np.float32)
    K, V = (rng.standard_normal((n_ctx, nhkv, hd)).astype(np.float32) for _ in range(2))
    q[1] = 0.0
    K[5:40] = 0.0
    K[11] = -0.0
    K[300] = 1e25
    V[:, :, 3:9] = 0.0
    V[::2, :, 10] = -0.0
    check_attn(q.reshape(-1), K.reshape(-1), V.reshape(-1), n_ctx, nh, nhkv, hd, 0.1, f"zero rows hd={hd}")


def test_attn_decode_infinities_and_nans():
    """One infinite or NaN element in q, K or V of each kv head: the outputs it
    reaches, and no others, are the reference's infinities and NaNs."""
    n_ctx, nh, nhkv, hd = 500, 10, 5, 64
    group = nh // nhkv
    rng = np.random.default_rng(12)
    q = rng.standard_normal((nh, hd)).astype(np.float32)
    K, V = (rng.standard_normal((n_ctx, nhkv, hd)).astype(np.float32) for _ in range(2))
    K[17, 0, 3] = np.nan  # all weights of its heads
    V[100, 1, 5], V[200, 1, 6], V[201, 1, 7] = np.nan, np.inf, -np.inf
    V[300, 1, 8], V[301, 1, 8] = np.inf, -np.inf
    K[50, 2, 9] = np.inf
    q[4, 9], q[5, 9] = -1.0, 1.0  # a weight of zero; infinity - infinity
    V[50, 2, 4] = np.inf  # under that weight of zero
    q[6, 1], q[7, 1] = np.nan, np.inf
    ref, rsoft = O.attn_decode(q.reshape(-1), K.reshape(-1), V.reshape(-1), n_ctx, nh, nhkv, hd, 0.125)
    dq, dk, dv = (uq.DeviceArray.from_numpy(a) for a in (q, K, V))
    dout, dsoft = uq.DeviceArray(4 * nh * hd), uq.DeviceArray(4 * nh * n_ctx)
    ops.attn_decode_d(dout, dsoft, dq, dk, dv, n_ctx, nh, nhkv, hd, 0.125)
    uq.synchronize()
    out, soft = dout.download(np.float32, nh * hd).reshape(nh, hd), dsoft.download(np.float32, nh * n_ctx)
    ref, rsoft, soft = np.reshape(ref, (nh, hd)), np.reshape(rsoft, (nh, n_ctx)), soft.reshape(nh, n_ctx)
    assert np.isnan(rsoft).any(1).tolist() == [True, True, False, False, False, True, True, True, False, False]
    assert np.isnan(ref[2]).sum() == 2 and np.isinf(ref[2]).sum() == 2 and np.isnan(ref[4]).sum() == 1
    for h in range(nh):
        assert np.array_equal(np.isnan(soft[h]), np.isnan(rsoft[h])), f"head {h}: NaN weights"
        assert np.array_equal(np.isnan(out[h]), np.isnan(ref[h])), f"head {h}: NaN outputs"
        # softmax's expf may differ from the C library's by an ulp: the sums in order of the device's own weights
        v = V[:, h // group].astype(np.float64)
        with np.errstate(invalid="ignore"):
            seq = np.add.accumulate(soft[h].astype(np.float64)[:, None] * v)[-1].astype(np.float32)
        ok = ~np.isnan(ref[h])
        assert_bitwise(out[h][ok], seq[ok], f"head {h}")
        np.testing.assert_allclose(out[h], ref[h], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("zero", ["q", "k", "v"])
def test_attn_decode_zero_operands_take_no_replays(zero):
    """Scores of zero rows and sums of zero columns are decided: with the
    scores replayed one by one a call took 1.9 times as long."""
    n_ctx, nh, nhkv, hd = 4096, 16, 4, 256
    rng = np.random.default_rng(1)
    a = {n: rng.standard_normal(m).astype(np.float32) for n, m in
         (("q", nh * hd), ("k", n_ctx * nhkv * hd), ("v", n_ctx * nhkv * hd))}
    dout, dsoft = uq.DeviceArray(4 * nh * hd), uq.DeviceArray(4 * nh * n_ctx)
    us = []
    for z in (None, zero):
        dq, dk, dv = (uq.DeviceArray.from_numpy(a[n] * np.float32(n != z)) for n in "qkv")
        us.append(microseconds(lambda: ops.attn_decode_d(dout, dsoft, dq, dk, dv, n_ctx, nh, nhkv, hd, 0.0625)))
        for d in (dq, dk, dv):
            d.free()
    print(f"random operands {us[0]:.0f} us, {zero} zero {us[1]:.0f} us", flush=True)
    assert us[1] < 1.5 * us[0]


def decode_us(q, k, v, n_ctx, nh, nhkv, hd):
    dq, dk, dv = (uq.DeviceArray.from_numpy(np.ascontiguousarray(a, np.float32)) for a in (q, k, v))
    dout, dsoft = uq.DeviceArray(4 * nh * hd), uq.DeviceArray(4 * nh * n_ctx)
    us = microseconds(lambda: ops.attn_decode_d(dout, dsoft, dq, dk, dv, n_ctx, nh, nhkv, hd, 0.0625))
    for d in (dq, dk, dv, dout, dsoft):
        d.free()
    return us


@pytest.mark.parametrize("qs,ks", [(1e-30, 1.0), (1.0, 1e-30), (1e-30, 1e-30), (1.0, 1e25), (1e20, 1e-5)])
def test_attn_decode_small_and_large_operands_take_no_replays(qs, ks):
    """Operands whose squares leave the f32 range: the bound follows them, the
    scores are the reference's, and a call takes the time of other operands
    (with norms in the f32 range every score was replayed)."""
    nh, nhkv, hd = 16, 4, 256
    rng = np.random.default_rng(3)
    q, k, v = rng.standard_normal((nh, hd)), rng.standard_normal((4000, nhkv * hd)), rng.standard_normal((4000, nhkv * hd))
    small = [(a * b).astype(np.float32) for a, b in ((q, qs), (k[:70], ks), (v[:70], 1.0))]
    check_attn(*(a.reshape(-1) for a in small), 70, nh, nhkv, hd, 0.0625, f"q x {qs} k x {ks}")
    us = decode_us(q, k, v, 4000, nh, nhkv, hd), decode_us(q * qs, k * ks, v, 4000, nh, nhkv, hd)
    log = f"random operands {us[0]:.0f} us, q x {qs} k x {ks} {us[1]:.0f} us"
    print(log, flush=True)
    assert us[1] < 1.5 * us[0], log


@pytest.mark.parametrize("n_ctx", [500, 4000])
def test_attn_decode_infinite_values_take_no_replays(n_ctx):
    """One infinite V row: every output is infinite, as the sum of the same
    terms in any order is, and a call takes the time of other operands."""
    nh, nhkv, hd = 16, 4, 256
    rng = np.random.default_rng(4)
    q, k, v = rng.standard_normal((nh, hd)), rng.standard_normal((n_ctx, nhkv * hd)), rng.standard_normal((n_ctx, nhkv * hd))
    us = [decode_us(q, k, v, n_ctx, nh, nhkv, hd)]
    v[7] = np.where(v[7] > 0, np.inf, -np.inf)
    got = check_attn(*(a.astype(np.float32).reshape(-1) for a in (q, k, v)), n_ctx, nh, nhkv, hd, 0.0625, "infinite V row")
    assert np.isinf(got).all()
    us.append(decode_us(q, k, v, n_ctx, nh, nhkv, hd))
    print(f"random operands {us[0]:.0f} us, an infinite V row {us[1]:.0f} us", flush=True)
    assert us[1] < 1.5 * us[0]


@pytest.mark.parametrize("n_ctx", [2, 4, 16, 64])
def test_attn_decode_midpoints_over_few_positions_replay_fast(n_ctx):
    """A zero q over few positions weighs them by a power of two, and many sums
    of such products end on an f32 midpoint: the lanes replay theirs side by
    side (a workgroup, output by output, took up to 80 us more)."""
    nh, nhkv, hd = 16, 4, 256
    rng = np.random.default_rng(5)
    q, k, v = rng.standard_normal((nh, hd)), rng.standard_normal((n_ctx, nhkv * hd)), rng.standard_normal((n_ctx, nhkv * hd))
    check_attn(*(a.astype(np.float32).reshape(-1) for a in (0 * q, k, v)), n_ctx, nh, nhkv, hd, 0.0625, f"equal weights n={n_ctx}",
               bit_exact_soft=True)
    us = decode_us(q, k, v, n_ctx, nh, nhkv, hd), decode_us(0 * q, k, v, n_ctx, nh, nhkv, hd)
    print(f"random q {us[0]:.0f} us, zero {us[1]:.0f} us", flush=True)
    assert us[1] < 1.8 * us[0]


@pytest.mark.parametrize("shape,nt,pos0", [
    (dict(n_head=8, n_head_kv=2, head_dim=64), 333, 29), (dict(n_head=8, n_head_kv=2, head_dim=64), 9, 300),
    (dict(n_embd=1024, n_v_heads=16, n_head=4, n_head_kv=1, head_dim=256), 300, 1500)])
def test_attn_prefill_zero_operands(shape, nt, pos0):
    """Zero tokens (q, and their own K and V rows) over a cache with zero V
    columns and rows: the steps' bits, and about the time of other operands
    (the values replayed, it was 6 to 8 times as much in the pair tiles)."""
    m = Model(dict(SMALL, **shape), seed=91)
    c = m.cfg
    rng = np.random.default_rng(nt)
    n_ctx_max = pos0 + nt
    K, V = (rng.standard_normal((n_ctx_max, c.n_head_kv, c.head_dim)).astype(np.float32) for _ in range(2))
    Z = V.copy()
    Z[:, :, 1::2] = 0.0
    Z[::3] = 0.0
    X = np.zeros((nt, c.n_embd), np.float32)
    steps = range(0, nt, max(1, nt // 40))
    got = attn_layer(m, X, K, Z, n_ctx_max, pos0, True)
    for t in steps:  # zero tokens: a step at each position by itself
        own = Z.copy()
        own[pos0:pos0 + t] = 0.0
        assert_bitwise(got[t], attn_layer(m, X[t:t + 1], K * (np.arange(n_ctx_max) < pos0)[:, None, None], own,
                                          n_ctx_max, pos0 + t, False)[0], f"zero token {t} of {nt}")
    ws = uq.DeviceArray(4 * L.prefill_ws_floats(m.d, nt, attn=m.aw, n_ctx_max=n_ctx_max))
    us = []
    for x, v in ((rng.standard_normal(X.shape).astype(np.float32), V), (X, Z)):
        kc, vc, dx, dl = (uq.DeviceArray.from_numpy(b) for b in (K, v, x, X))
        us.append(microseconds(lambda: L.attn_prefill(m.d, m.aw, kc, vc, n_ctx_max, pos0, nt, dx, dl, ws)))
        for d in (kc, vc, dx, dl):
            d.free()
    ws.free()
    m.free()
    print(f"random operands {us[0]:.0f} us, zero {us[1]:.0f} us", flush=True)
    assert us[1] < 1.5 * us[0]
