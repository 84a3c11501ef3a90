"""GPU parity of the batched MLA attention of prefill and MTP verify
(wh_mla_attention_decode_batch_async, compute_deepseek_v4_mla_attention_batch,
E/compute.rs:4307-4641).  The reference batches the projections with
gemv_fp8_e4m3_ue8m0_rows_multi, whose every input is bit-identical to the
single-input kernel (E/compute.rs:6447-6452), writes every position's KV row
before the window loop, and reads in each position's window only rows at or
before its own; so with exact numerics the batch must equal the single-token
layer run position by position, bit for bit, and the oracle's single-token
restatement (mla_attention_decode) run the same way: a sliding-window layer
over a cache with earlier rows, a compressed YaRN layer with per-position
compressed rows, and 16 positions in order-free numerics (the projections on
MFMA) within a loose bound of the exact result."""
import numpy as np
import pytest

import wohper_amd
from parity_util import bits
from test_gpu_mla import HEAD_DIM, HEADS, NOPE, ROPE, GROUPS, O_LORA, Dev, _layer, _proj
from wohper_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture
def dev(ctx):
    d = Dev(ctx)
    yield d
    d.free()
    ctx.set_exact_numerics(True)


def _sequential(ctx, dev, L, xs, positions, cache0, ld, comps=None):
    """The single-token layer at each position in order, on its own cache."""
    cap = cache0.shape[0]
    kvp = dev.put(cache0)
    outs = []
    for i, p in enumerate(positions):
        hp = dev.put(xs[i])
        if comps:
            ctx.mla_attention_decode_async(L, p, hp, kvp, ld, cap, comps[i][0], comps[i][1])
        else:
            ctx.mla_attention_decode_async(L, p, hp, kvp, ld, cap)
        ctx.synchronize()
        outs.append(dev.get(hp, wl.HIDDEN))
    return np.stack(outs), dev.get(kvp, (cap, ld))


def _batch(ctx, dev, L, xs, positions, cache0, ld, comps=None):
    cap = cache0.shape[0]
    kvp, hp = dev.put(cache0), dev.put(np.ascontiguousarray(xs))
    ctx.mla_attention_decode_batch_async(L, positions, hp, kvp, ld, cap, comps)
    ctx.synchronize()
    return dev.get(hp, (len(positions), wl.HIDDEN)), dev.get(kvp, (cap, ld))


def test_mla_batch_window_layer(ctx, oracle, dev):
    """Layer 0 (sliding window, theta 10000): positions 5..9 after five
    earlier cache rows, against the single-token layer and the oracle."""
    ctx.set_exact_numerics(True)
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 0)
    proj = _proj(oracle, host)
    cap, ld = 16, HEAD_DIM + 64
    rng = np.random.default_rng(11)
    cache0 = np.zeros((cap, ld), np.float32)
    cache0[:5] = (rng.standard_normal((5, ld)) * 0.3).astype(np.float32)
    positions = [5, 6, 7, 8, 9]
    xs = rng.standard_normal((len(positions), wl.HIDDEN)).astype(np.float32)
    got, got_cache = _batch(ctx, dev, L, xs, positions, cache0, ld)
    want, want_cache = _sequential(ctx, dev, L, xs, positions, cache0, ld)
    assert np.array_equal(bits(got_cache), bits(want_cache))
    assert np.array_equal(bits(got), bits(want)), int(np.count_nonzero(bits(got) != bits(want)))
    cache = cache0.copy()
    for i, p in enumerate(positions):
        w = oracle.mla_attention_decode(xs[i], proj, qn, kn, sink, HEADS, NOPE, ROPE, GROUPS, O_LORA, 0, p, cache)
        assert np.array_equal(bits(got[i]), bits(w)), p
    assert np.array_equal(bits(got_cache), bits(cache))
    for h in handles.values():
        ctx.release(h)


def test_mla_batch_compressed_layer(ctx, oracle, dev):
    """Layer 2 (theta 160000 with YaRN), positions 300..302 with a full
    window and 75, 75, 76 compressed rows of their own, plain norms, no
    sink."""
    ctx.set_exact_numerics(True)
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 2, with_norms=False, with_sink=False)
    proj = _proj(oracle, host)
    cap, ld = 320, HEAD_DIM
    rng = np.random.default_rng(12)
    cache0 = (rng.standard_normal((cap, ld)) * 0.3).astype(np.float32)
    positions = [300, 301, 302]
    comps_h = [(rng.standard_normal((k, HEAD_DIM)) * 0.3).astype(np.float32) for k in (75, 75, 76)]
    comps = [(dev.put(cmp), cmp.shape[0]) for cmp in comps_h]
    xs = rng.standard_normal((len(positions), wl.HIDDEN)).astype(np.float32)
    got, got_cache = _batch(ctx, dev, L, xs, positions, cache0, ld, comps)
    want, want_cache = _sequential(ctx, dev, L, xs, positions, cache0, ld, comps)
    assert np.array_equal(bits(got_cache), bits(want_cache))
    assert np.array_equal(bits(got), bits(want))
    cache = cache0.copy()
    for i, p in enumerate(positions):
        w = oracle.mla_attention_decode(xs[i], proj, None, None, None, HEADS, NOPE, ROPE, GROUPS, O_LORA, 2, p, cache,
                                        comps_h[i])
        assert np.array_equal(bits(got[i]), bits(w)), p
    for h in handles.values():
        ctx.release(h)


def test_mla_batch_many_positions(ctx, dev):
    """35 positions in one launch, with key lists from a few rows to 700, so
    that it holds short and long ones: bit for bit the single-token layer's
    outputs."""
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 2)
    cap, ld = 240, HEAD_DIM
    rng = np.random.default_rng(14)
    cache0 = (rng.standard_normal((cap, ld)) * 0.3).astype(np.float32)
    positions = list(range(3, 3 + 18)) + list(range(200, 217))
    comp = dev.put((rng.standard_normal((700, HEAD_DIM)) * 0.3).astype(np.float32))
    comps = [(comp, int(k)) for k in rng.integers(1, 701, len(positions))]
    xs = rng.standard_normal((len(positions), wl.HIDDEN)).astype(np.float32)
    got, got_cache = _batch(ctx, dev, L, xs, positions, cache0, ld, comps)
    want, want_cache = _sequential(ctx, dev, L, xs, positions, cache0, ld, comps)
    assert np.array_equal(bits(got_cache), bits(want_cache))
    assert np.array_equal(bits(got), bits(want))
    for h in handles.values():
        ctx.release(h)


def test_mla_batch_two_launches(ctx, dev):
    """131 positions, three more than one launch of the rows and the window
    attention takes, with uneven compressed lists: at the first positions and
    about the launches' edge bit for bit the single-token layer over the
    batch's cache, whose rows up to a position are that position's."""
    ctx.set_exact_numerics(True)
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 2)
    n, cap, ld = 131, 400, HEAD_DIM
    rng = np.random.default_rng(15)
    cache0 = (rng.standard_normal((cap, ld)) * 0.3).astype(np.float32)
    positions = list(range(3, 3 + 18)) + list(range(200, 200 + n - 18))
    comp = dev.put((rng.standard_normal((700, HEAD_DIM)) * 0.3).astype(np.float32))
    comps = [(comp + 4 * HEAD_DIM * int(o), int(k)) for o, k in zip(rng.integers(0, 300, n), rng.integers(1, 401, n))]
    xs = rng.standard_normal((n, wl.HIDDEN)).astype(np.float32)
    got, cache = _batch(ctx, dev, L, xs, positions, cache0, ld, comps)
    for i in (0, 1, 17, 18, 126, 127, 128, 129, 130):
        want, after = _sequential(ctx, dev, L, xs[i:i + 1], positions[i:i + 1], cache, ld, comps[i:i + 1])
        assert np.array_equal(bits(after), bits(cache)), i
        assert np.array_equal(bits(got[i]), bits(want[0])), i
    for h in handles.values():
        ctx.release(h)


def _one_hot(ctx, rng, rows, cols):
    """A resident matrix whose rows pick one column each, plus or minus it:
    one product a row, the same bits in any order of summation."""
    w = np.zeros((rows, cols), np.uint8)
    pick = np.concatenate([rng.permutation(cols) for _ in range(-(-rows // cols))])[:rows]
    w[np.arange(rows), pick] = rng.choice(np.array([0x38, 0xB8], np.uint8), rows)
    return ctx.store_fp8(w, rows, cols, np.ones((rows // 128, cols // 128), np.float32), rows // 128, cols // 128,
                         wohper_amd.SCALE_F32)


@pytest.mark.parametrize("heads", [64, 48])
@pytest.mark.parametrize("n", [5, 17, 33, 131])
def test_mla_batch_order_free_window_alone(ctx, dev, heads, n):
    """The order-free window kernels of a batch (from 16 positions on 32 heads
    x 64 dims a workgroup, 48 heads with half a last one, and the score tiles),
    uneven key lists, with nothing else that could differ from exact numerics:
    one-hot projections, and inputs of 4 to 8 whose squares add exactly in any
    order.  The caches are then the same bits.  The attention's values differ
    by rounding, about 1e-6 of themselves, and are rounded to E4M3 twice, which
    turns such a difference into a step for about 4e-5 of them (two boundaries
    a step of 1/16 to 1/8); 1e-3 is the bound.  A key left out of 700 moves a
    value by 4 percent of itself and so about half of them by a step."""
    rng = np.random.default_rng(n + heads)
    q_lora, out = 1024, GROUPS * O_LORA
    shapes = {"wq_a": (q_lora, wl.HIDDEN), "wq_b": (heads * HEAD_DIM, q_lora), "wkv": (HEAD_DIM, wl.HIDDEN),
              "wo_a": (out, heads * HEAD_DIM // GROUPS), "wo_b": (wl.HIDDEN, out)}
    t = {k: _one_hot(ctx, rng, *v) for k, v in shapes.items()}
    ones = {k: dev.put(np.full(k, 0x3F80, np.uint16)) for k in (q_lora, HEAD_DIM)}
    sink = dev.put(rng.standard_normal(heads).astype(np.float32))
    L = wohper_amd.WhMlaLayer(2, heads, NOPE, ROPE, GROUPS, O_LORA, t["wq_a"], t["wq_b"], t["wkv"], t["wo_a"], t["wo_b"],
                              ones[q_lora], ones[HEAD_DIM], sink)
    cap = 400
    cache0 = rng.standard_normal((cap, HEAD_DIM)).astype(np.float32)
    few = min(n // 2, 18)
    positions = list(range(3, 3 + few)) + list(range(200, 200 + n - few))
    comp = dev.put(rng.standard_normal((1000, HEAD_DIM)).astype(np.float32))
    comps = [(comp + 4 * HEAD_DIM * int(o), int(k)) for o, k in zip(rng.integers(0, 300, n), rng.integers(1, 701, n))]
    xs = (rng.integers(4, 9, (n, wl.HIDDEN)) * rng.choice([-1, 1], (n, wl.HIDDEN))).astype(np.float32)
    got = {}
    for exact in (True, False):
        ctx.set_exact_numerics(exact)
        got[exact] = _batch(ctx, dev, L, xs, positions, cache0, HEAD_DIM, comps)
    assert np.array_equal(bits(got[True][1]), bits(got[False][1]))
    a, b = got[True][0], got[False][0]
    differ = (a != b).mean(1)
    print(f"{heads} heads, {n} positions: share of values a step apart, most of a position {differ.max():.2e}, "
          f"all {differ.mean():.2e}")
    assert np.count_nonzero(a) > 0.99 * a.size and np.all(np.isfinite(b))
    assert differ.mean() <= 1e-3 and differ.max() <= 5e-3
    for h in t.values():
        ctx.release(h)


def test_mla_batch_order_free_16(ctx, dev):
    """16 positions: with exact numerics the batch equals the single-token
    layer position by position (the decode-once kernels at 16 inputs); with
    exact numerics off (the projections on bf16 MFMA, exact products, fp32
    accumulation order only; the norms' sums as trees) each position stays
    within 1e-2 of the exact output in norm.  The bound is loose because an
    act-quant between the projections can round a near-tie the other way:
    one such element moves a wo_b output by a whole E4M3 step of its input
    (the per-matvec tolerance of the projections is checked in
    test_gpu_fp8_mfma)."""
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 0)
    cap, ld = 32, HEAD_DIM
    rng = np.random.default_rng(13)
    cache0 = (rng.standard_normal((cap, ld)) * 0.3).astype(np.float32)
    positions = list(range(4, 20))
    xs = rng.standard_normal((len(positions), wl.HIDDEN)).astype(np.float32)
    ctx.set_exact_numerics(True)
    want, _ = _batch(ctx, dev, L, xs, positions, cache0, ld)
    seq, _ = _sequential(ctx, dev, L, xs, positions, cache0, ld)
    assert np.array_equal(bits(want), bits(seq))  # exact: 16 inputs through the decode-once kernels
    ctx.set_exact_numerics(False)
    got, _ = _batch(ctx, dev, L, xs, positions, cache0, ld)
    assert np.all(np.isfinite(got))
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    print("per-position ||diff|| / ||value||:", np.array2string(rel, precision=6))
    assert float(rel.max()) <= 1e-2
    for h in handles.values():
        ctx.release(h)


@pytest.mark.parametrize("n", [35, 131])
def test_mla_batch_order_free_many(ctx, dev, n):
    """Exact numerics off, key lists from a few rows to 700 in one launch (32
    heads x 64 keys a workgroup, partial and missing key tiles; 131: more
    positions than one launch takes): nine of ten positions within 1e-2 of the
    exact output in norm, as above, and every one within 0.1: an act-quant
    that rounds a near-tie the other way moves one element by up to 1/16 of
    its value, and of this many positions some have several on the way (a
    wrong key, head or position is a deviation of order one)."""
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 2)
    cap, ld = 400, HEAD_DIM
    rng = np.random.default_rng(n)
    cache0 = (rng.standard_normal((cap, ld)) * 0.3).astype(np.float32)
    positions = list(range(3, 3 + 18)) + list(range(200, 200 + n - 18))
    comp = dev.put((rng.standard_normal((700, HEAD_DIM)) * 0.3).astype(np.float32))
    comps = [(comp, int(k)) for k in rng.integers(1, 701, n)]
    xs = rng.standard_normal((n, wl.HIDDEN)).astype(np.float32)
    ctx.set_exact_numerics(True)
    want, _ = _batch(ctx, dev, L, xs, positions, cache0, ld, comps)
    ctx.set_exact_numerics(False)
    got, _ = _batch(ctx, dev, L, xs, positions, cache0, ld, comps)
    ctx.set_exact_numerics(True)
    assert np.all(np.isfinite(got))
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    print("per-position ||diff|| / ||value||:", np.array2string(rel, precision=6))
    assert float(np.quantile(rel, 0.9)) <= 1e-2 and float(rel.max()) <= 0.1
    for h in handles.values():
        ctx.release(h)


def test_mla_batch_errors(ctx, dev):
    L, host, qn, kn, sink, handles = _layer(ctx, dev, 0)
    cap, ld = 8, HEAD_DIM
    kvp, hp = dev.put(np.zeros((cap, ld), np.float32)), dev.put(np.zeros((2, wl.HIDDEN), np.float32))
    with pytest.raises(wohper_amd.DeepSeekV4KernelError) as e:
        ctx.mla_attention_decode_batch_async(L, [3, 2], hp, kvp, ld, cap)  # positions must ascend
    assert e.value.name == "InvalidArgument"
    with pytest.raises(wohper_amd.DeepSeekV4KernelError) as e:
        ctx.mla_attention_decode_batch_async(L, [], hp, kvp, ld, cap)
    assert e.value.name == "InvalidShape"
    with pytest.raises(wohper_amd.DeepSeekV4KernelError) as e:
        ctx.mla_attention_decode_batch_async(L, [6, cap], hp, kvp, ld, cap)  # past the cache
    assert e.value.name == "InvalidShape"
    for h in handles.values():
        ctx.release(h)
