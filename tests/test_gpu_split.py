"""Products on bf16 parts (ft_split.hip) at the edges of their tiles, K steps and dispatch, against f64.

Tolerance: the operands are held whole, so an element is off by the roundings of its sum alone: at most n matrix
instructions follow each other on one accumulator (six per K step of 16, the K steps shared by at least two waves),
then the waves' sums are added; each may be off by 2^-23 of the sum of the absolute products so far, or, among subnormal
numbers, by their distance 2^-149.
"""
import contextlib
import ctypes

import numpy as np
import pytest

from tests.gpu_util import make_ctx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    ctx, eng = make_ctx()
    yield ctx, eng
    ctx.close()


def rnd(seed, *shape, scale=1.0):
    return (np.random.default_rng(seed).standard_normal(shape) * scale).astype(np.float32)


def up(ctx, x):
    from ferrotensor_amd import UnifiedTensor
    return UnifiedTensor.new(ctx, np.ascontiguousarray(x), list(x.shape))


def up16(ctx, x):
    from ferrotensor_amd import UnifiedTensor
    return UnifiedTensor.from_f32_as_f16(ctx, np.ascontiguousarray(x), list(x.shape))


def empty(ctx, *shape):
    from ferrotensor_amd import UnifiedTensor
    return UnifiedTensor.empty(ctx, list(shape))


@contextlib.contextmanager
def on_bf16_parts(ctx):
    """What runs inside is here to test gemm_split_kernel: sizes that take another one say so."""
    from ferrotensor_amd import _lib
    lib = _lib.load()
    assert lib.ft_profile_begin(ctx.handle) == 0
    yield
    n = ctypes.c_size_t()
    assert lib.ft_profile_end(ctx.handle, ctypes.byref(n)) == 0
    names = []
    for i in range(n.value):
        name, launches, x = ctypes.c_char_p(), ctypes.c_uint64(), [ctypes.c_double() for _ in range(3)]
        assert lib.ft_profile_kernel(ctx.handle, i, ctypes.byref(name), ctypes.byref(launches), *(ctypes.byref(v) for v in x)) == 0
        names.append(name.value.decode())
    products = [x for x in names if x.startswith(("gemm", "splitk"))]
    assert products and all(x.startswith("gemm_split_kernel") for x in products), names


def check(name, got, terms, K):
    """terms: (a, b) pairs whose products add up."""
    want = sum(a.astype(np.float64) @ b.astype(np.float64) for a, b in terms)
    size = sum(np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64) for a, b in terms)
    limit = (6 * (K // 16 // 2 + 1) + 32) * (2.0 ** -23 * size + 2.0 ** -149)
    got = np.asarray(got, np.float64).reshape(want.shape)
    assert np.all(np.isfinite(got)), name
    worst = np.max(np.abs(got - want) / np.maximum(limit, 1e-300))
    assert worst <= 1.0, "%s: %.3g of the bound" % (name, worst)


# Each tile and wave count of the dispatch, one row or column more and less than a tile, K with no whole step left over,
# 1, 4, 15 left over, and rows of every alignment, K of two steps and a rest on.
SHAPES = [(4, 48, 8), (4, 33, 9), (31, 52, 33), (33, 47, 31), (32, 64, 32), (100, 333, 517), (257, 733, 1001), (65, 96, 63),
          (700, 161, 1024), (1023, 101, 641), (1025, 66, 1101), (2113, 64, 1100), (1100, 127, 1029), (1088, 576, 1152), (5, 2561, 9)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_f32_layouts(g, M, K, N):
    ctx, eng = g
    a, b = rnd(M + K, M, K), rnd(N + K, K, N)
    out = empty(ctx, M, N)
    for name, run in (("a@b", lambda: eng.matmul(ctx, up(ctx, a), up(ctx, b), out)),
                      ("a@bT", lambda: eng.matmul_bt(ctx, up(ctx, a), up(ctx, b.T), out)),
                      ("aT@b", lambda: eng.matmul_at(ctx, up(ctx, a.T), up(ctx, b), out))):
        with on_bf16_parts(ctx):
            run()
        check("%s %dx%dx%d" % (name, M, K, N), out.to_vec(), [(a, b)], K)


@pytest.mark.parametrize("M,K,N,r", [(4, 48, 8, 4), (33, 64, 40, 8), (17, 96, 1000, 16), (257, 736, 1000, 32), (700, 1024, 1024, 8),
                                     (2113, 64, 1104, 16), (1100, 352, 1032, 3),
                                     # widths that are no multiple of 8 (f16) or 4: loads from 2- and 4-byte boundaries, a last
                                     # K step (dx: of N) element by element, every tile size
                                     (5, 33, 9, 4), (33, 70, 41, 8), (100, 100, 333, 8), (257, 733, 1001, 16), (700, 161, 1023, 8),
                                     (1100, 127, 1029, 8), (1090, 577, 1150, 4)])
def test_adapted_linear_both_ways(g, M, K, N, r):
    ctx, eng = g
    x, w, t, b = rnd(M, M, K), rnd(K, K, N, scale=0.05), rnd(r, M, r), rnd(N, r, N)
    dy, dt, a, res = rnd(M + 1, M, N), rnd(r + 1, M, r), rnd(K + 1, K, r), rnd(M + 2, M, K)
    w16 = w.astype(np.float16).astype(np.float32)
    for half in (True, False):
        W, wv = (up16(ctx, w), w16) if half else (up(ctx, w), w)
        y, dx = empty(ctx, M, N), empty(ctx, M, K)
        with on_bf16_parts(ctx):
            eng.lora_linear(ctx, up(ctx, x), W, up(ctx, t), up(ctx, b), y)
        check("y", y.to_vec(), [(x, wv), (t, b)], K)
        with on_bf16_parts(ctx) if N >= 48 else contextlib.nullcontext():   # (a sum over N)
            eng.lora_linear_dx(ctx, up(ctx, dy), W, up(ctx, dt), up(ctx, a), dx, residual=up(ctx, res))
        check("dx", dx.to_vec(), [(dy, wv.T), (dt, a.T), (res, np.eye(K, dtype=np.float32))], N)


@pytest.mark.parametrize("half", [False, True])
def test_wide_range_of_values_in_one_row(g, half):
    """Exponents from -60 to 40, and 100 on columns that meet zeros: no scale per row, so an outlier costs its neighbours
    nothing."""
    ctx, eng = g
    M, K, N = 96, 192, 96
    rng = np.random.default_rng(3)
    a = (rnd(1, M, K) * np.exp2(rng.integers(-60, 40, (M, K)))).astype(np.float32)
    w = rnd(2, K, N, scale=0.05)
    w[rng.integers(0, K, 40)] = 0.0   # whole rows of zeros: the outliers that meet them must not show
    a[:, np.all(w == 0.0, axis=1)] *= np.float32(2.0 ** 60)
    wv = w.astype(np.float16).astype(np.float32) if half else w
    out = empty(ctx, M, N)
    if half:
        eng.lora_linear(ctx, up(ctx, a), up16(ctx, w), None, None, out)
    else:
        eng.matmul(ctx, up(ctx, a), up(ctx, w), out)
    check("wide", out.to_vec(), [(a, wv)], K)


# Tiles of every shape; K with whole steps only, and with a rest.
@pytest.mark.parametrize("M,K,N", [(40, 64, 48), (96, 200, 960), (300, 192, 1100), (1025, 100, 1104)])
@pytest.mark.parametrize("kind", ["all", "few", "products"])
def test_values_below_what_three_bf16_parts_hold(g, M, K, N, kind):
    """Values down to the last subnormal against large ones: all of an operand, single ones that alone decide a result (the
    others meet zeros), and ordinary values whose products are subnormal."""
    ctx, eng = g
    rng = np.random.default_rng(K)
    a, b = rnd(1, M, K), rnd(2, K, N)
    if kind == "all":
        a, b = np.ldexp(a, rng.integers(-149, -108, a.shape)), np.ldexp(b, 100)
    elif kind == "few":
        b[K // 2] = 0.0
        a[1:, K // 2] = np.ldexp(a[1:, K // 2], 60)
        a[M // 2, :] = 0.0
        a[M // 2, K // 2 - 1] = np.ldexp(np.float32(1.2345678), -121)   # this row's only value
        b[K // 2 - 1] = np.ldexp(b[K // 2 - 1], 90)
        a[M // 2 + 1 :, K // 2 - 1] = 0.0
    else:
        a, b = np.ldexp(a, -70), np.ldexp(b, -68)
    a, b = a.astype(np.float32), b.astype(np.float32)
    out, w = empty(ctx, M, N), up(ctx, b)
    for name, run in (("a@b", lambda: eng.matmul(ctx, up(ctx, a), w, out)), ("a@bT", lambda: eng.matmul_bt(ctx, up(ctx, a), up(ctx, b.T), out)),
                      ("aT@b", lambda: eng.matmul_at(ctx, up(ctx, a.T), w, out))):
        with on_bf16_parts(ctx):
            run()
        check("%s %s" % (kind, name), out.to_vec(), [(a, b)], K)
    out = empty(ctx, N, M)   # as the second operand
    eng.matmul(ctx, up(ctx, b.T), up(ctx, a.T), out)
    check("%s second" % kind, out.to_vec(), [(b.T, a.T)], K)


@pytest.mark.parametrize("half", [False, True])
def test_values_below_what_three_bf16_parts_hold_in_the_fused_launches(g, half):
    ctx, eng = g
    M, K, N = 100, 144, 128
    x = np.ldexp(rnd(1, M, K), np.random.default_rng(1).integers(-149, -108, (M, K))).astype(np.float32)
    w1, w2 = rnd(2, K, N), rnd(3, K, N)
    make = up16 if half else up
    w1, w2 = (w.astype(np.float16).astype(np.float32) if half else w for w in (w1, w2))
    y1, y2 = empty(ctx, M, N), empty(ctx, M, N)
    scale = np.float32(1.0) if half else np.ldexp(np.float32(1.0), 100)
    eng.lora_linear_group(ctx, up(ctx, x), [(make(ctx, w1 * scale), None, None, y1, None), (make(ctx, w2 * scale), None, None, y2, None)])
    check("group 1", y1.to_vec(), [(x, w1 * scale)], K)
    check("group 2", y2.to_vec(), [(x, w2 * scale)], K)
    gate, u, act = (empty(ctx, M, N) for _ in range(3))
    eng.mlp_gate_up(ctx, up(ctx, x), make(ctx, w1 * scale), make(ctx, w2 * scale), gate, u, act)
    check("gate", gate.to_vec(), [(x, w1 * scale)], K)
    check("up", u.to_vec(), [(x, w2 * scale)], K)


@pytest.mark.parametrize("M,N", [(70, 96), (520, 1100)])
def test_infinities_and_nan_as_f32_products_give_them(g, M, N):
    ctx, eng = g
    K = 81
    a, b = np.abs(rnd(5, M, K)) + 0.1, np.abs(rnd(6, K, N)) + 0.1
    a[3, 7], a[9, 20], a[40, 3], a[41, 70] = np.inf, np.nan, 3.4e38, -np.inf
    b[30, 11], b[70, 50], b[3, 60] = np.inf, 0.0, 1e-30
    out = empty(ctx, M, N)
    with on_bf16_parts(ctx):
        eng.matmul(ctx, up(ctx, a), up(ctx, b), out)
    got = np.asarray(out.to_vec(), np.float32).reshape(M, N)
    with np.errstate(all="ignore"):
        want = np.zeros((M, N))
        for k in range(K):
            want = want + a[:, k:k + 1].astype(np.float64) * b[k:k + 1].astype(np.float64)
    want[np.abs(want) > 3.4028235e38] = np.sign(want[np.abs(want) > 3.4028235e38]) * np.inf
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(np.sign(got[np.isinf(got)]), np.sign(want[np.isinf(want)]))
    fine = np.isfinite(want)
    np.testing.assert_allclose(got[fine], want[fine], rtol=1e-5)


def test_sums_the_same_twice(g):
    ctx, eng = g
    a, b = up(ctx, rnd(8, 300, 700)), up(ctx, rnd(9, 700, 500))
    o1, o2 = empty(ctx, 300, 500), empty(ctx, 300, 500)
    eng.matmul(ctx, a, b, o1)
    eng.matmul(ctx, a, b, o2)
    assert np.array_equal(np.asarray(o1.to_vec()).view(np.uint32), np.asarray(o2.to_vec()).view(np.uint32))


def rope_table(ctx, seq, theta=10000.0):
    pos, i = np.arange(seq)[:, None], np.arange(32)[None, :]
    angle = pos * theta ** (-2.0 * i / 64)
    t = np.stack([np.cos(angle), np.sin(angle)], axis=-1).astype(np.float32)
    return up(ctx, t.reshape(seq, 64)), t


@pytest.mark.parametrize("M,K,widths,half", [(4, 32, (64, 64, 64), True), (33, 100, (128, 64, 72), False), (96, 960, (960, 320, 320), True),
                                             (520, 250, (1088, 64, 64), True), (1040, 64, (1024, 128, 8), False),
                                             (33, 100, (64, 64, 73), True), (520, 251, (1024, 64, 70), True), (1040, 193, (1024, 128, 9), False)])
def test_group_with_rotation_and_residual(g, M, K, widths, half):
    """Two rotated products and one with a residual and a rank-r term, every tile height and wave count."""
    ctx, eng = g
    x, seq = rnd(M, M, K), M // 4 if M % 4 == 0 else M
    table, t = rope_table(ctx, seq)
    linears, want = [], []
    for i, n in enumerate(widths):
        w, f, b = rnd(n + i, K, n, scale=0.05), rnd(i, M, 8), rnd(i + 9, 8, n)
        wv = w.astype(np.float16).astype(np.float32) if half else w
        res = rnd(i + 20, M, n) if i == 2 else None
        y = empty(ctx, M, n)
        linears.append((up16(ctx, w) if half else up(ctx, w), up(ctx, f), up(ctx, b), y, up(ctx, res) if i == 2 else None))
        terms = [(x, wv), (f, b)] + ([(res, np.eye(n, dtype=np.float32))] if i == 2 else [])
        plain = sum(p.astype(np.float64) @ q.astype(np.float64) for p, q in terms)
        size = sum(np.abs(p).astype(np.float64) @ np.abs(q).astype(np.float64) for p, q in terms)
        if i < 2:
            c, s = (np.tile(t[..., k].astype(np.float64), (M // seq, 1))[:, None, :] for k in (0, 1))
            h, hs = plain.reshape(M, n // 64, 2, 32), size.reshape(M, n // 64, 2, 32)
            plain = np.stack([h[:, :, 0] * c - h[:, :, 1] * s, h[:, :, 0] * s + h[:, :, 1] * c], 2).reshape(M, n)
            size = np.stack([hs[:, :, 0] + hs[:, :, 1]] * 2, 2).reshape(M, n)
        want.append((plain, size))
    with on_bf16_parts(ctx):
        eng.lora_linear_group(ctx, up(ctx, x), linears, rope_table=table, rope_seq=seq, n_rope=2)
    for (w, f, b, y, r), (plain, size) in zip(linears, want):
        limit = (6 * (K // 16 // 4 + 1) + 36) * 2.0 ** -23 * size
        got = np.asarray(y.to_vec(), np.float64).reshape(plain.shape)
        assert np.all(np.abs(got - plain) <= limit), (y.shape, np.max(np.abs(got - plain) / limit))


@pytest.mark.parametrize("M,K,N,half", [(4, 32, 8, True), (33, 100, 41, False), (96, 960, 2560, True), (300, 200, 1000, True), (1040, 64, 1024, False), (33, 101, 41, True),
                                        (520, 205, 1003, True)])
def test_gate_up(g, M, K, N, half):
    ctx, eng = g
    x, wg, wu = rnd(M, M, K), rnd(N, K, N, scale=0.05), rnd(N + 1, K, N, scale=0.05)
    gv, uv = (w.astype(np.float16).astype(np.float32) if half else w for w in (wg, wu))
    make = up16 if half else up
    gate, u, act = (empty(ctx, M, N) for _ in range(3))
    with on_bf16_parts(ctx):
        eng.mlp_gate_up(ctx, up(ctx, x), make(ctx, wg), make(ctx, wu), gate, u, act)
    check("gate", gate.to_vec(), [(x, gv)], K)
    check("up", u.to_vec(), [(x, uv)], K)
    gt, ut = (np.asarray(o.to_vec(), np.float64) for o in (gate, u))
    want = gt / (1.0 + np.exp(-gt)) * ut
    np.testing.assert_allclose(np.asarray(act.to_vec(), np.float64), want, rtol=2e-6, atol=1e-30)


@pytest.mark.parametrize("half", [False, True])
def test_group_whose_linears_feed_each_other(g, half):
    """Down to the rank, up again with it as the factor, and a third that adds to the second's output: in order, as three calls."""
    ctx, eng = g
    M, K, N, r = 300, 96, 640, 8
    x, a, w, b, v = rnd(1, M, K), rnd(2, K, r), rnd(3, K, N, scale=0.05), rnd(4, r, N), rnd(5, K, N, scale=0.05)
    make = up16 if half else up
    seen = (lambda m: m.astype(np.float16).astype(np.float32)) if half else (lambda m: m)
    t, y, z = empty(ctx, M, r), empty(ctx, M, N), empty(ctx, M, N)
    eng.lora_linear_group(ctx, up(ctx, x), [(make(ctx, a), None, None, t, None), (make(ctx, w), t, up(ctx, b), y, None),
                                            (make(ctx, v), None, None, z, y)])
    got = np.asarray(t.to_vec(), np.float32).reshape(M, r)
    check("t", got, [(x, seen(a))], K)
    check("y", y.to_vec(), [(x, seen(w)), (got, b)], K)
    check("z", z.to_vec(), [(x, seen(v)), (np.asarray(y.to_vec(), np.float32).reshape(M, N), np.eye(N, dtype=np.float32))], K)


@pytest.mark.parametrize("half", [False, True])
def test_gate_up_with_the_activation_in_the_place_of_its_input(g, half):
    ctx, eng = g
    M, K = 300, 192
    x, wg, wu = rnd(1, M, K), rnd(2, K, K, scale=0.05), rnd(3, K, K, scale=0.05)
    make = up16 if half else up
    outs = []
    for inplace in (False, True):
        X, gate, u = up(ctx, x), empty(ctx, M, K), empty(ctx, M, K)
        act = X if inplace else empty(ctx, M, K)
        eng.mlp_gate_up(ctx, X, make(ctx, wg), make(ctx, wu), gate, u, act)
        outs.append([np.asarray(o.to_vec(), np.float32) for o in (gate, u, act)])
    for a, b in zip(*outs):
        np.testing.assert_allclose(b, a, rtol=2e-6, atol=2e-6)   # one launch or three: sums in another order


def attention64(q, k, v, causal, offset):
    """f64 attention of [B, Sq, H, D] over [B, Sk, Hkv, D]; log-sum-exp too."""
    B, Sq, H, D = q.shape
    rep = H // k.shape[2]
    k, v = np.repeat(k, rep, axis=2).astype(np.float64), np.repeat(v, rep, axis=2).astype(np.float64)
    s = np.matmul(q.astype(np.float64).transpose(0, 2, 1, 3), k.transpose(0, 2, 3, 1)) / np.sqrt(D)
    if causal:
        s = np.where(np.arange(k.shape[1])[None, :] <= np.arange(Sq)[:, None] + offset, s, -np.inf)
    m = s.max(-1, keepdims=True)
    e = np.exp(s - m)
    z = e.sum(-1, keepdims=True)
    return np.matmul(e / z, v.transpose(0, 2, 1, 3)).transpose(0, 2, 1, 3), (m + np.log(z))[..., 0]


def on_parts(ctx, B, Sq, Sk, H, Hkv, causal, forward_only=0):
    """Do these sizes take the kernels on bf16 parts on this device?"""
    from ferrotensor_amd import _lib
    lib = ctypes.CDLL(_lib.LIB_PATH)
    return lib.ft_internal_attention_split(*(ctypes.c_size_t(x) for x in (lib.ft_internal_num_cus(ctx.handle), B, Sq, Sk, H, Hkv)),
                                           int(causal), forward_only)


# Ragged queries and keys, heads without a group, a group added by the second kernel, a group too large for its scratch,
# fewer queries than keys with an offset, no mask.
ATTENTION = [(8, 200, 200, 32, 32, True, 0), (4, 397, 461, 32, 16, True, 64), (8, 150, 190, 32, 32, False, 0), (4, 300, 333, 32, 16, False, 0),
             (8, 400, 400, 32, 8, True, 0), (12, 96, 200, 32, 32, True, 104), (8, 385, 400, 32, 8, False, 0)]


@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,causal,offset", ATTENTION)
def test_attention_forward(g, B, Sq, Sk, H, Hkv, causal, offset):
    from ferrotensor_amd import AttentionOptions
    ctx, eng = g
    assert on_parts(ctx, B, Sq, Sk, H, Hkv, causal)
    q, k, v = rnd(1, B, Sq, H, 64), rnd(2, B, Sk, Hkv, 64), rnd(3, B, Sk, Hkv, 64)
    o, stats = empty(ctx, B, Sq, H, 64), empty(ctx, B * H * Sq, 2)
    eng.flash_attention_v2_with_stats(ctx, up(ctx, q), up(ctx, k), up(ctx, v), o, stats, AttentionOptions(causal=causal, causal_offset=offset))
    want, lse = attention64(q, k, v, causal, offset)
    # probabilities to 2^-18 of themselves (scores of a few units, exp2 in f32), then averages of values near 1
    np.testing.assert_allclose(np.asarray(o.to_vec(), np.float64).reshape(want.shape), want, atol=2e-5)
    np.testing.assert_allclose(np.asarray(stats.to_vec(), np.float64).reshape(B, H, Sq, 2)[..., 1], lse, atol=1e-5)


# Tiles of 32 rows (few workgroups) and of 64, ragged, an offset, no mask.
@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,causal,offset", [(1, 40, 40, 3, 1, True, 0), (1, 7, 9, 3, 1, True, 2), (2, 65, 129, 4, 2, True, 64), (1, 200, 200, 9, 3, False, 0),
                                                         (1, 256, 256, 3, 1, True, 0), (8, 130, 130, 16, 4, True, 0), (8, 127, 200, 16, 16, False, 0)])
def test_attention_forward_alone(g, B, Sq, Sk, H, Hkv, causal, offset):
    """The entry that a model's forward pass takes, which no operator call reaches at these sizes."""
    from ferrotensor_amd import _lib
    ctx, eng = g
    assert on_parts(ctx, B, Sq, Sk, H, Hkv, causal, 1)
    q, k, v = rnd(1, B, Sq, H, 64), rnd(2, B, Sk, Hkv, 64), rnd(3, B, Sk, Hkv, 64)
    o, t = empty(ctx, B, Sq, H, 64), [up(ctx, x) for x in (q, k, v)]
    opts = _lib.AttentionOptionsC(int(causal), offset, 0, 0.0, 0)
    run = ctypes.CDLL(_lib.LIB_PATH).ft_internal_attention_forward_only
    assert run(ctx.handle, *(ctypes.c_void_p(x.ptr) for x in (*t, o)), *(ctypes.c_size_t(x) for x in (B, Sq, Sk, H, Hkv, 64)), ctypes.byref(opts)) == 0
    want, _ = attention64(q, k, v, causal, offset)
    np.testing.assert_allclose(np.asarray(o.to_vec(), np.float64).reshape(want.shape), want, atol=2e-5)


def test_attention_with_infinite_and_nan_values_as_the_f32_kernel(g):
    """V and K of some heads hold an infinity, a NaN, a value at the top of f32: the queries that see them come out as from
    the f32 kernel (where a tile crosses the diagonal, a NaN score counts as masked), the others as ever."""
    from ferrotensor_amd import AttentionOptions
    ctx, eng = g
    B, S, H = 8, 160, 32
    assert on_parts(ctx, B, S, S, H, H, True)
    q, k, v = rnd(1, B, S, H, 64), rnd(2, B, S, H, 64), rnd(3, B, S, H, 64)
    v[0, 50, 3, 7], v[1, 100, 5, 9], k[2, 70, 1, 4] = np.inf, np.nan, np.nan
    v[3, 20, 2, 11] = 3.4e38   # finite, but its first bf16 part is not
    o, stats = empty(ctx, B, S, H, 64), empty(ctx, B * H * S, 2)
    eng.flash_attention_v2_with_stats(ctx, up(ctx, q), up(ctx, k), up(ctx, v), o, stats, AttentionOptions(causal=True))
    got = np.asarray(o.to_vec(), np.float64).reshape(B, S, H, 64)
    fine = np.isfinite(got)
    assert not fine[0, 50:, 3, 7].any() and not fine[1, 100:, 5, 9].any() and not fine[2, 128:, 1].any()
    with np.errstate(all="ignore"):
        want, _ = attention64(q, k, np.where(np.isfinite(v), v, 0.0), True, 0)
    ok = fine & np.isfinite(want)
    ok[3, :, 2, 11] = False
    np.testing.assert_allclose(got[ok], want[ok], atol=2e-5)
    np.testing.assert_allclose(got[3, :, 2, 11], want[3, :, 2, 11], rtol=1e-4, atol=2e-5)
    assert fine[[0, 1, 3]][:, :, [0, 4, 6]].all()   # the other heads


def backward64(q, k, v, do, causal, offset):
    B, Sq, H, D = q.shape
    Hkv = k.shape[2]
    rep = H // Hkv
    qt, dt = (x.astype(np.float64).transpose(0, 2, 1, 3) for x in (q, do))
    kt, vt = (np.repeat(x, rep, axis=2).astype(np.float64).transpose(0, 2, 1, 3) for x in (k, v))
    s = np.matmul(qt, kt.transpose(0, 1, 3, 2)) / np.sqrt(D)
    if causal:
        s = np.where(np.arange(k.shape[1])[None, :] <= np.arange(Sq)[:, None] + offset, s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    dp = np.matmul(dt, vt.transpose(0, 1, 3, 2))
    ds = p * (dp - (p * dp).sum(-1, keepdims=True)) / np.sqrt(D)
    back = lambda x: x.transpose(0, 2, 1, 3)
    group = lambda x: back(x).reshape(B, -1, Hkv, rep, D).sum(3)
    return back(np.matmul(ds, kt)), group(np.matmul(ds.transpose(0, 1, 3, 2), qt)), group(np.matmul(p.transpose(0, 1, 3, 2), dt))


def run_attention(ctx, eng, q, k, v, do, causal, offset):
    from ferrotensor_amd import AttentionOptions
    B, Sq, H, D = q.shape
    t = [up(ctx, x) for x in (q, k, v)]
    o, stats = empty(ctx, *q.shape), empty(ctx, B * H * Sq, 2)
    dq, dk, dv = empty(ctx, *q.shape), empty(ctx, *k.shape), empty(ctx, *k.shape)
    opts = AttentionOptions(causal=causal, causal_offset=offset)
    eng.flash_attention_v2_with_stats(ctx, *t, o, stats, opts)
    eng.flash_attention_v2_backward_with_stats(ctx, *t, o, up(ctx, do), dq, dk, dv, stats, opts)
    return [np.asarray(x.to_vec(), np.float32).reshape(y.shape) for x, y in ((dq, q), (dk, k), (dv, k))]


@pytest.mark.parametrize("B,Sq,Sk,H,Hkv,causal,offset", ATTENTION)
def test_attention_backward(g, B, Sq, Sk, H, Hkv, causal, offset):
    ctx, eng = g
    assert on_parts(ctx, B, Sq, Sk, H, Hkv, causal)
    q, k, v, do = rnd(1, B, Sq, H, 64), rnd(2, B, Sk, Hkv, 64), rnd(3, B, Sk, Hkv, 64), rnd(4, B, Sq, H, 64, scale=1e-2)
    for name, got, want in zip(("dq", "dk", "dv"), run_attention(ctx, eng, q, k, v, do, causal, offset), backward64(q, k, v, do, causal, offset)):
        # probabilities to 2^-18 of themselves, sums of at most a few hundred rounded terms
        assert np.max(np.abs(got - want)) <= 2e-5 * np.max(np.abs(want)), name


def test_attention_backward_with_infinite_and_nan_values_as_the_f32_kernels(g):
    """The batch takes the kernels on bf16 parts; its sequences one at a time do not: the same values are not finite."""
    ctx, eng = g
    B, S, H = 8, 200, 32
    assert on_parts(ctx, B, S, S, H, H, True) and not on_parts(ctx, 1, S, S, H, H, True)
    q, k, v, do = rnd(1, B, S, H, 64), rnd(2, B, S, H, 64), rnd(3, B, S, H, 64), rnd(4, B, S, H, 64, scale=1e-2)
    v[0, 50, 3, 7], do[1, 100, 5, 9], k[2, 70, 1, 4], q[3, 190, 2, 1], do[4, 3, 7, 0] = np.inf, np.nan, np.nan, np.inf, 3.4e38
    batch = run_attention(ctx, eng, q, k, v, do, True, 0)
    for i in range(5):
        one = run_attention(ctx, eng, *(x[i:i + 1] for x in (q, k, v, do)), True, 0)
        for name, a, b in zip(("dq", "dk", "dv"), batch, one):
            assert np.array_equal(np.isfinite(a[i]), np.isfinite(b[0])), (i, name)
            fine = np.isfinite(b[0])
            np.testing.assert_allclose(a[i][fine], b[0][fine], rtol=2e-4, atol=2e-6)


@pytest.mark.parametrize("B,S,heads,kv", [(1, 8, 3, 1), (2, 50, 4, 2), (2, 70, 16, 8), (3, 150, 12, 4)])
def test_model_forward_attention_at_small_sizes(B, S, heads, kv):
    """A forward pass takes attention on bf16 parts at these sizes (32- and 64-row tiles): logits against the oracle's."""
    from ferrotensor_amd import HipContext
    from ferrotensor_amd.trainer import Lfm2Model, ModelConfig
    from oracle import reference_step as rs
    H, F, V = heads * 64, 128, 64
    cfg = ModelConfig(vocab_size=V, hidden_size=H, intermediate_size=F, num_hidden_layers=2, num_attention_heads=heads,
                      num_key_value_heads=kv, tie_word_embeddings=True, f16_linears=False)
    t = {"model.embed_tokens.weight": rnd(1, V, H, scale=0.5), "model.norm.weight": np.ones(H, np.float32)}
    for l in range(2):
        p = "model.layers.%d." % l
        t[p + "input_layernorm.weight"] = t[p + "post_attention_layernorm.weight"] = np.ones(H, np.float32)
        for i, (n, o, k) in enumerate((("self_attn.q_proj", H, H), ("self_attn.k_proj", kv * 64, H), ("self_attn.v_proj", kv * 64, H),
                                       ("self_attn.o_proj", H, H), ("mlp.gate_proj", F, H), ("mlp.up_proj", F, H), ("mlp.down_proj", H, F))):
            t[p + n + ".weight"] = rnd(10 * l + i + 2, o, k, scale=0.05)
    ctx = HipContext(0)
    hip = Lfm2Model(ctx, cfg)
    hip.load_tensors(t)
    orc = rs.Model.from_hf_tensors(rs.ModelConfig(V, H, F, 2, heads, kv, cfg.rms_norm_eps, cfg.rope_theta, True), t, f16_linears=False)
    rows = np.random.default_rng(S).integers(0, V, (B, S)).astype(np.uint32)
    want, _ = orc.forward(rows)
    got = hip.forward_batch(rows)
    # The suite's parity bar, its absolute term (for values near 1) times the logits' rms, which is 12 to 20 here: a pass on
    # the f32 kernels is off the oracle by as much (2.8e-4 at 2 x 70 tokens, 16 heads; this one 2.7e-4).
    want = np.asarray(want).reshape(-1)
    assert np.all(np.abs(got.reshape(-1) - want) <= 1e-4 * np.sqrt(np.mean(want ** 2)) + 1e-3 * np.abs(want))
    ctx.close()


def test_attention_results_in_the_place_of_an_operand(g):
    """o over q, dq over out, dk over k and dv over v, with values that send some workgroups back to the f32 code (which reads
    the operands again): the same bits as with buffers of their own."""
    from ferrotensor_amd import AttentionOptions
    ctx, eng = g
    B, S, H = 3, 512, 32
    assert on_parts(ctx, B, S, S, H, H, True)
    q, k, v, do = rnd(1, B, S, H, 64), rnd(2, B, S, H, 64), rnd(3, B, S, H, 64), rnd(4, B, S, H, 64, scale=1e-2)
    v[0, 50, 3, 7], k[1, 100, 5, 9], do[2, 70, 1, 4] = np.inf, np.nan, 3.4e38
    opts = AttentionOptions(causal=True)
    results = []
    for inplace in (False, True):
        Q, K, V, DO = (up(ctx, x) for x in (q, k, v, do))
        stats, o = empty(ctx, B * H * S, 2), Q if inplace else empty(ctx, *q.shape)
        eng.flash_attention_v2_with_stats(ctx, Q, K, V, o, stats, opts)
        out = o.to_vec()
        if inplace:   # the backward needs q
            Q, o = up(ctx, q), up(ctx, np.asarray(out, np.float32).reshape(q.shape))
        dq, dk, dv = (o, K, V) if inplace else (empty(ctx, *q.shape), empty(ctx, *k.shape), empty(ctx, *v.shape))
        eng.flash_attention_v2_backward_with_stats(ctx, Q, K, V, o, DO, dq, dk, dv, stats, opts)
        results.append([np.asarray(x, np.float32) for x in (out, dq.to_vec(), dk.to_vec(), dv.to_vec())])
    for name, a, b in zip(("o", "dq", "dk", "dv"), *results):
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)]), name


# (which operand is scaled by which power of two, and what else)
@pytest.mark.parametrize("case", ["v", "k", "q", "one v", "one do", "do", "ds", "none"])
def test_attention_with_values_below_what_three_bf16_parts_hold(g, case):
    """Operands below 2^-110 (all of one, against a large other one; a single value that decides a result), and dO and V whose
    product is: relative to the largest of a head's results, as ordinary values. Also against the f32 kernels (the batch's
    first sequence alone)."""
    from ferrotensor_amd import AttentionOptions
    ctx, eng = g
    B, S, H = 3, 512, 32
    assert on_parts(ctx, B, S, S, H, H, True)
    q, k, v, do = rnd(1, B, S, H, 64), rnd(2, B, S, H, 64), rnd(3, B, S, H, 64), rnd(4, B, S, H, 64, scale=1e-2)
    ld = lambda x, e: np.ldexp(x, e).astype(np.float32)
    if case == "v":
        v = ld(v, -124)
    elif case == "k":
        k, q = ld(k, -120), ld(q, 119)
    elif case == "q":
        q, k = ld(q, -124), ld(k, 123)
    elif case == "one v":
        v[0, :, 3, 7] = 0.0
        v[0, 5, 3, 7] = np.ldexp(1.2345678, -121)
    elif case == "one do":
        do[0, :, 3] = 0.0
        do[0, 300, 3, 7] = np.ldexp(1.2345678, -121)
        v[0, :, 3] = ld(v[0, :, 3], 60)
    elif case == "do":
        do = ld(do, -112)
    elif case == "ds":
        do, v, k = ld(do, -60), ld(v, -60), ld(k, 60)
        q = ld(q, -60)
    opts = AttentionOptions(causal=True)
    o, stats = empty(ctx, *q.shape), empty(ctx, B * H * S, 2)
    eng.flash_attention_v2_with_stats(ctx, up(ctx, q), up(ctx, k), up(ctx, v), o, stats, opts)
    got = [np.asarray(o.to_vec(), np.float32).reshape(q.shape), *run_attention(ctx, eng, q, k, v, do, True, 0)]
    want = [attention64(q, k, v, True, 0)[0], *backward64(q, k, v, do, True, 0)]
    alone = [x[:1] for x in (q, k, v, do)]
    o1, s1 = empty(ctx, 1, S, H, 64), empty(ctx, H * S, 2)
    eng.flash_attention_v2_with_stats(ctx, *(up(ctx, x) for x in alone[:3]), o1, s1, opts)
    f32 = [np.asarray(o1.to_vec(), np.float32).reshape(1, S, H, 64), *run_attention(ctx, eng, *alone, True, 0)]
    for name, a, b, c in zip(("o", "dq", "dk", "dv"), got, want, f32):
        for h in (0, 3, 31):
            scale = np.max(np.abs(b[0, :, h]))
            err, err32 = (np.max(np.abs(x[0, :, h] - b[0, :, h])) for x in (a, c))
            # as test_attention_backward, or among subnormal results their distance; where cancellation is all there is
            # (dS of a head with hardly any dP), as far off as the f32 kernels
            assert err <= max(2e-5 * scale, 64 * 2.0 ** -149, 2 * err32), (name, h, err, scale, err32)


def replays_match(ctx, call, outputs, eager_call, eager_outputs, bound):
    """Captures `call` on the context's stream, then replays it three times, with the eager call between the replays."""
    from ferrotensor_amd import _lib
    hip, lib = ctypes.CDLL("libamdhip64.so.7"), _lib.load()
    stream, graph, run = ctypes.c_void_p(lib.ft_context_stream(ctx.handle)), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    call()
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    for i in range(3):
        assert hip.hipGraphLaunch(run, stream) == 0
        ctx.synchronize()
        eager_call()
        for n, (a, b) in enumerate(zip(outputs, eager_outputs)):
            x, y = (np.asarray(t.to_vec(), np.float32) for t in (a, b))
            assert np.max(np.abs(x - y)) <= bound * np.max(np.abs(y)), (i, n)
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0


def test_attention_backward_is_captured_without_a_warm_up():
    """A context that has run nothing yet: the group's shares have no scratch, and under capture none can be allocated; the f32
    kernels need none at these sizes."""
    from ferrotensor_amd import AttentionOptions
    B, S, H, Hkv = 3, 512, 32, 8
    host = [rnd(1, B, S, H, 64), rnd(2, B, S, Hkv, 64), rnd(3, B, S, Hkv, 64), rnd(4, B, S, H, 64, scale=1e-2)]
    opts = AttentionOptions(causal=True)
    ctx, eng = make_ctx()
    assert on_parts(ctx, B, S, S, H, Hkv, True)
    q, k, v, do = (up(ctx, x) for x in host)
    o, stats = empty(ctx, *host[0].shape), empty(ctx, B * H * S, 2)
    out, eager = ([empty(ctx, *x.shape) for x in host[:3]] for _ in range(2))
    eng.flash_attention_v2_with_stats(ctx, q, k, v, o, stats, opts)
    ctx.synchronize()
    back = lambda to: eng.flash_attention_v2_backward_with_stats(ctx, q, k, v, o, do, *to, stats, opts)
    # heads added in another order: sums of at most a few thousand rounded terms
    replays_match(ctx, lambda: back(out), out, lambda: back(eager), eager, 2e-5)
    ctx.close()


def test_f32_product_with_long_k_is_captured_without_a_warm_up():
    """The same for a product whose K the f32 kernel shares out over workgroups, which add through scratch memory."""
    ctx, eng = make_ctx()
    a, b = up(ctx, rnd(1, 64, 4096)), up(ctx, rnd(2, 4096, 256))
    out, eager = empty(ctx, 64, 256), empty(ctx, 64, 256)
    ctx.synchronize()
    # 4096 fused multiply-adds in one chain or in eight
    replays_match(ctx, lambda: eng.matmul(ctx, a, b, out), [out], lambda: eng.matmul(ctx, a, b, eager), [eager], 4096 * 2.0 ** -24)
    ctx.close()
