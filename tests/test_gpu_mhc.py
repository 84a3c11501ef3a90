"""GPU parity of the mHC hyper-connections (hc_split_sinkhorn_scalar,
hc_pre_into, hc_post_into; E/compute.rs:4945-5092) against the oracle: the
Sinkhorn split and hc_post bit for bit; hc_pre bit for bit under exact
numerics (the reference's serial dot and sum-of-squares order) and within
1e-5 of the largest value with exact numerics off (tree sums), at the
model's shape (hc 4 x hidden 4096, 24 mix rows, 20 rounds) and small
ones."""
import numpy as np
import pytest

from test_gpu_mla import Dev

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.fixture
def dev(ctx):
    d = Dev(ctx)
    yield d
    d.free()
    ctx.set_exact_numerics(True)


def _params(rng, hc, hidden):
    mix_hc = (2 + hc) * hc
    fn = (rng.standard_normal((mix_hc, hc * hidden)) * (1.0 / np.sqrt(hc * hidden))).astype(np.float32)
    scale = (0.5 + rng.random(3)).astype(np.float32)
    base = (rng.standard_normal(mix_hc) * 0.5).astype(np.float32)
    return fn, scale, base


@pytest.mark.parametrize("hc,iters", [(4, 20), (4, 1), (4, 0), (1, 20), (2, 3), (14, 20)])
def test_split_sinkhorn_bit_exact(ctx, oracle, dev, hc, iters):
    rng = np.random.default_rng(hc * 10 + iters)
    mix_hc = (2 + hc) * hc
    mixes = rng.standard_normal(mix_hc).astype(np.float32) * 2
    scale = (0.5 + rng.random(3)).astype(np.float32)
    base = rng.standard_normal(mix_hc).astype(np.float32)
    pp, qp, cp = dev.empty(hc * 4), dev.empty(hc * 4), dev.empty(hc * hc * 4)
    ctx.hc_split_sinkhorn_async(dev.put(mixes), dev.put(scale), dev.put(base), hc, iters, 1e-6, pp, qp, cp)
    ctx.synchronize()
    want = oracle.hc_split_sinkhorn(mixes, scale, base, hc, iters, 1e-6)
    for got, w in zip((dev.get(pp, hc), dev.get(qp, hc), dev.get(cp, hc * hc)), want):
        assert np.array_equal(bits(got), bits(w))


@pytest.mark.parametrize("hc,hidden", [(4, 4096), (2, 3), (3, 1001), (4, 64)])
def test_hc_pre_post_exact(ctx, oracle, dev, hc, hidden):
    rng = np.random.default_rng(hc * 7 + hidden)
    fn, scale, base = _params(rng, hc, hidden)
    x = rng.standard_normal(hc * hidden).astype(np.float32)
    yp, qp, cp, op = dev.empty(hidden * 4), dev.empty(hc * 4), dev.empty(hc * hc * 4), dev.empty(hc * hidden * 4)
    xp = dev.put(x)
    ctx.set_exact_numerics(True)
    ctx.hc_pre_async(dev.put(fn), dev.put(scale), dev.put(base), hc, hidden, 20, 1e-6, xp, yp, qp, cp)
    ctx.synchronize()
    y, pre, post, comb, _ = oracle.hc_pre(fn, scale, base, x, hc, hidden, 20, 1e-6)
    assert np.array_equal(bits(dev.get(yp, hidden)), bits(y))
    assert np.array_equal(bits(dev.get(qp, hc)), bits(post))
    assert np.array_equal(bits(dev.get(cp, hc * hc)), bits(comb))
    # hc_post with a sub-block output of its own
    ys = rng.standard_normal(hidden).astype(np.float32)
    ctx.hc_post_async(dev.put(ys), xp, qp, cp, op, hc, hidden)
    ctx.synchronize()
    assert np.array_equal(bits(dev.get(op, hc * hidden)), bits(oracle.hc_post(ys, x, post, comb, hc, hidden)))


def test_hc_pre_fast_within_tolerance(ctx, oracle, dev):
    hc, hidden = 4, 4096
    rng = np.random.default_rng(44)
    fn, scale, base = _params(rng, hc, hidden)
    x = rng.standard_normal(hc * hidden).astype(np.float32)
    yp, qp, cp = dev.empty(hidden * 4), dev.empty(hc * 4), dev.empty(hc * hc * 4)
    args = (dev.put(fn), dev.put(scale), dev.put(base), hc, hidden, 20, 1e-6, dev.put(x), yp, qp, cp)
    y, pre, post, comb, _ = oracle.hc_pre(fn, scale, base, x, hc, hidden, 20, 1e-6)
    times = {}
    for exact in (True, False):
        ctx.set_exact_numerics(exact)
        ctx.hc_pre_async(*args)
        ctx.synchronize()
        ctx.timer_start()
        for _ in range(20):
            ctx.hc_pre_async(*args)
        times[exact] = ctx.timer_stop() / 20
        ctx.synchronize()
    # the last run is the tree-sum one
    for got, want in ((dev.get(yp, hidden), y), (dev.get(qp, hc), post), (dev.get(cp, hc * hc), comb)):
        assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))
    print(f"hc_pre 4 x 4096: exact {times[True]:.1f} us, tree sums {times[False]:.1f} us")


def _terms(kind, rng, n):
    """x and a weight row whose products take a sequential f32 sum through
    the cases of the chunked one."""
    x = rng.standard_normal(n).astype(np.float32)
    w = rng.standard_normal(n).astype(np.float32)
    if kind == "ties":        # few mantissa bits: most additions round a tie
        x = np.round(x * 4) / 4 + 0.25
        w = np.exp2(rng.integers(-3, 4, n)) * np.sign(w)
    elif kind == "range":     # 2^-40 .. 2^40, cancelling pairs
        w = w * np.exp2(rng.uniform(-40, 40, n))
        w[1::2] = -w[:n - n % 2:2]
    elif kind == "zeros":
        x[rng.random(n) < 0.9] = 0.0
    elif kind == "huge":      # overflows to infinity part of the way
        x = x * np.float32(1e19)
        w = np.abs(w) * np.float32(1e18)
    return x.astype(np.float32), w.astype(np.float32)


@pytest.mark.parametrize("kind", ["normal", "ties", "range", "zeros", "huge"])
@pytest.mark.parametrize("hc,hidden", [(1, 31), (1, 1024), (1, 1025), (4, 1024), (4, 1025), (1, 8192), (1, 8193),
                                       (4, 4096), (4, 4097), (2, 17000)])
def test_hc_pre_ordered_sums(ctx, oracle, dev, kind, hc, hidden):
    """The chunked sequential sums at the edges of their chunk sizes and past
    one segment (16384 terms), bit for bit."""
    rng = np.random.default_rng(hidden + hc)
    mix_hc, n = (2 + hc) * hc, hc * hidden
    x, w0 = _terms(kind, rng, n)
    fn = np.stack([w0] + [_terms(kind, rng, n)[1] for _ in range(mix_hc - 1)])
    scale, base = np.full(3, 1e-3, np.float32), rng.standard_normal(mix_hc).astype(np.float32)
    yp, qp, cp = dev.empty(hidden * 4), dev.empty(hc * 4), dev.empty(hc * hc * 4)
    ctx.set_exact_numerics(True)
    ctx.hc_pre_async(dev.put(fn), dev.put(scale), dev.put(base), hc, hidden, 2, 1e-6, dev.put(x), yp, qp, cp)
    ctx.synchronize()
    with np.errstate(all="ignore"):
        y, _, post, comb, _ = oracle.hc_pre(fn, scale, base, x, hc, hidden, 2, 1e-6)
    for got, w in zip((dev.get(yp, hidden), dev.get(qp, hc), dev.get(cp, hc * hc)), (y, post, comb)):
        w = np.asarray(w).reshape(-1)
        assert np.array_equal(np.isnan(got), np.isnan(w))
        assert np.array_equal(bits(got)[~np.isnan(w)], bits(w)[~np.isnan(w)])


@pytest.mark.parametrize("kind", ["normal", "ties", "range", "zeros"])
@pytest.mark.parametrize("n", [1, 512, 513, 1024, 1025, 4095, 4096])
@pytest.mark.parametrize("rows", [1, 16])
def test_rms_norm_ordered_sum(ctx, oracle, dev, kind, n, rows):
    """The norm's sequential sum of squares over both workgroup sizes, bit
    for bit."""
    rng = np.random.default_rng(n)
    x = np.stack([_terms(kind, rng, n)[0] * np.float32(1.5 ** r) for r in range(rows)])
    if kind == "range":
        x = (x * np.exp2(rng.uniform(-30, 30, x.shape))).astype(np.float32)
    xp, op = dev.put(x), dev.empty(x.nbytes)
    ctx.set_exact_numerics(True)
    ctx.rms_norm_async(xp, op, rows, n)
    ctx.synchronize()
    want = np.stack([oracle.rms_norm(r) for r in x])
    assert np.array_equal(bits(dev.get(op, x.size)), bits(want).reshape(-1))


def _cancelling(rng, n, closeness):
    """Products whose even ones cancel the odd ones to `closeness`."""
    x, w = rng.standard_normal(n), rng.standard_normal(n)
    w[1::2] = -(w * x)[0::2] * (1.0 + closeness * rng.standard_normal(n // 2)) / x[1::2]
    return x.astype(np.float32), w.astype(np.float32)


@pytest.mark.parametrize("closeness", [1e-1, 3e-2, 1e-2, 1e-3, 1e-6, 0.0])
@pytest.mark.parametrize("hc,hidden", [(1, 1500), (2, 2048), (4, 2048), (4, 4096), (2, 17000)])
def test_hc_pre_cancelling_sums(ctx, oracle, dev, closeness, hc, hidden):
    """Sums that the chunked sequential sum finishes one term at a time, from
    the first and from later groups of chunks, bit for bit."""
    rng = np.random.default_rng(hidden)
    mix_hc, n = (2 + hc) * hc, hc * hidden
    x, _ = _cancelling(rng, n, closeness)
    fn = np.empty((mix_hc, n), np.float32)
    for r in fn:
        w = rng.standard_normal(n)
        w[1::2] = -(w * x)[0::2] * (1.0 + closeness * rng.standard_normal(n // 2)) / x[1::2]
        r[:] = w
    scale, base = np.ones(3, np.float32), rng.standard_normal(mix_hc).astype(np.float32)
    yp, qp, cp = dev.empty(hidden * 4), dev.empty(hc * 4), dev.empty(hc * hc * 4)
    ctx.set_exact_numerics(True)
    ctx.hc_pre_async(dev.put(fn), dev.put(scale), dev.put(base), hc, hidden, 2, 1e-6, dev.put(x), yp, qp, cp)
    ctx.synchronize()
    y, _, post, comb, _ = oracle.hc_pre(fn, scale, base, x, hc, hidden, 2, 1e-6)
    for got, w in zip((dev.get(yp, hidden), dev.get(qp, hc), dev.get(cp, hc * hc)), (y, post, comb)):
        assert np.array_equal(bits(got), bits(np.asarray(w).reshape(-1)))


def _hc_pre_us(ctx, dev, hc, hidden, x, fn):
    """Time of one hc_pre call, 20 in a graph."""
    mix_hc = (2 + hc) * hc
    out = [dev.empty(k * 4) for k in (hidden, hc, hc * hc)]
    scale, base = dev.put(np.ones(3, np.float32)), dev.put(np.zeros(mix_hc, np.float32))
    xp, fp = dev.put(x), dev.put(fn)
    ctx.hc_pre_async(fp, scale, base, hc, hidden, 2, 1e-6, xp, *out)
    ctx.synchronize()
    g = ctx.graph_capture(lambda: [ctx.hc_pre_async(fp, scale, base, hc, hidden, 2, 1e-6, xp, *out)
                                   for _ in range(20)])
    us = []
    for _ in range(6):
        ctx.timer_start()
        ctx.graph_launch(g)
        us.append(ctx.timer_stop() / 20)
    ctx.graph_release(g)
    return min(us)


def test_hc_pre_cancelling_sums_time(ctx, dev):
    """One chunk after the other is the most that the values can make of a
    sequential sum: 16384 adds of 8.6 cycles are 59 us at 2.4 GHz, 3.2 times
    the whole call on N(0, 1) products (22 us); with a round for every chunk
    it was 6.5 times."""
    hc, hidden = 4, 4096
    n, mix_hc = hc * hidden, (2 + hc) * hc
    rng = np.random.default_rng(8)
    ctx.set_exact_numerics(True)
    x, w = _cancelling(rng, n, 1e-4)
    slow = _hc_pre_us(ctx, dev, hc, hidden, x, np.tile(w, (mix_hc, 1)))
    plain = _hc_pre_us(ctx, dev, hc, hidden, rng.standard_normal(n).astype(np.float32),
                       rng.standard_normal((mix_hc, n)).astype(np.float32))
    print(f"hc_pre 4 x 4096: N(0, 1) {plain:.1f} us, cancelling {slow:.1f} us")
    assert slow <= 4.5 * plain


@pytest.mark.parametrize("hc,hidden", [(1, 1), (1, 255), (1, 257), (3, 85), (1, 1279), (1, 1280), (1, 1281), (2, 1024)])
@pytest.mark.parametrize("kind", ["normal", "range"])
def test_hc_pre_short_rows(ctx, oracle, dev, hc, hidden, kind):
    """Rows that one lane adds, and the first above them, bit for bit."""
    test_hc_pre_ordered_sums(ctx, oracle, dev, kind, hc, hidden)


def test_hc_pre_short_rows_time(ctx, dev):
    """Rows of 256 terms: 256 ordered adds are 1 us, so exact numerics take
    about the order-free call's time (9.5 against 9.3 us; through the chunked
    sum 12)."""
    rng = np.random.default_rng(9)
    x, fn = rng.standard_normal(256).astype(np.float32), rng.standard_normal((24, 256)).astype(np.float32)
    us = {}
    for exact in (False, True):
        ctx.set_exact_numerics(exact)
        try:
            us[exact] = _hc_pre_us(ctx, dev, 4, 64, x, fn)
        finally:
            ctx.set_exact_numerics(True)
    print(f"hc_pre 4 x 64: exact {us[True]:.1f} us, order-free {us[False]:.1f} us")
    assert us[True] <= 1.18 * us[False]


@pytest.mark.parametrize("kind", ["normal", "ties", "range"])
@pytest.mark.parametrize("n", [575, 576, 577, 1500, 2047, 2048, 2049])
@pytest.mark.parametrize("rows", [3, 17])
def test_rms_norm_ordered_sum_edges(ctx, oracle, dev, kind, n, rows):
    """The last row that one lane adds and the chunk sizes after it, bit for
    bit."""
    test_rms_norm_ordered_sum(ctx, oracle, dev, kind, n, rows)


def test_rms_norm_one_wave_more_than_512(ctx, dev):
    """One row of 513 terms, one more than a row of 512 whose adds one lane
    makes: 3.8 us against 3.65 (through the chunked sum 4.4 or more)."""
    us = {}
    ctx.set_exact_numerics(True)
    for n in (512, 513):
        x, o = dev.put(np.random.default_rng(n).standard_normal(n).astype(np.float32)), dev.empty(4 * n)
        g = ctx.graph_capture(lambda: [ctx.rms_norm_async(x, o, 1, n) for _ in range(50)])
        t = []
        for _ in range(8):
            ctx.timer_start()
            ctx.graph_launch(g)
            t.append(ctx.timer_stop() / 50)
        ctx.graph_release(g)
        us[n] = min(t)
    print(f"norm of one row: 512 {us[512]:.2f} us, 513 {us[513]:.2f} us")
    assert us[513] <= 1.12 * us[512]
