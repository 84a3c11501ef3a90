"""GPU parity of the batched DeepSeek-V4 layer of prefill and MTP verify
(wh_deepseek_mhc_layer_batch_async, E/server/generation.rs:2437-2590:
compute_layer_deepseek_mhc_phase1_batch, the router per position, the union
MoE, finish_layer_deepseek_mhc_phase2_batch) at the model's shapes with a
32-expert router, against the oracle's composition of the same steps
(oracle.mhc_decode_layer_batch).  Exact numerics: bit for bit, positions
after earlier cache rows; the batch MoE divides each position's router
weights by their sum as the reference's batch path does, so a one-position
batch differs from the single-token layer only through that division.
Exact numerics off: within a loose norm bound of the exact batch."""
import numpy as np
import pytest

from parity_util import bits
from test_gpu_decode_layer import HC, Dev, _setup
from test_gpu_mla import HEAD_DIM
import wohper_amd
from wohper_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture
def dev(ctx):
    d = Dev(ctx)
    yield d
    d.free()
    ctx.set_exact_numerics(True)


def _run(ctx, dev, L, h0, positions, kv0, ld):
    cap = kv0.shape[0]
    hp, kvp = dev.put(np.ascontiguousarray(h0)), dev.put(kv0)
    ctx.deepseek_mhc_layer_batch_async(L, positions, hp, kvp, ld, cap)
    ctx.synchronize()
    return dev.get(hp, (len(positions), HC * wl.HIDDEN)), dev.get(kvp, (cap, ld))


def test_decode_layer_batch_bit_exact(ctx, oracle, dev):
    ctx.set_exact_numerics(True)
    L, want, handles = _setup(ctx, oracle, dev)
    cap, ld = 16, HEAD_DIM + 64
    rng = np.random.default_rng(21)
    kv0 = np.zeros((cap, ld), np.float32)
    kv0[:3] = (rng.standard_normal((3, ld)) * 0.3).astype(np.float32)
    positions = [3, 4, 5, 6]
    h0 = (rng.standard_normal((len(positions), HC * wl.HIDDEN)) * 0.5).astype(np.float32)
    got, got_kv = _run(ctx, dev, L, h0, positions, kv0, ld)
    cache = kv0.copy()
    wanted, ids, w = want.batch(h0, positions, cache)
    print("routes:", ids.tolist())
    assert np.array_equal(bits(got_kv), bits(cache))
    for i in range(len(positions)):
        assert np.array_equal(bits(got[i]), bits(wanted[i])), (i, int(np.count_nonzero(bits(got[i]) != bits(wanted[i]))))
    for t in handles.values():
        ctx.release(t)


def test_decode_layer_batch_order_free(ctx, oracle, dev):
    """Exact numerics off (the projections, the expert matvecs and hc_pre's
    sums on the order-free kernels): each position within 10% of the exact
    batch in norm, the median position within 3%.  The layer is not
    continuous in its inputs: an act-quant can round a near-tie the other way
    (one E4M3 step of one element), and the biased top-6 can swap a near-tied
    sixth expert (several percent of the output at this weight); the
    synthetic layer amplifies its input about 2e4 times, so such flips are
    not damped by the residual.  The single-token layer on the first
    position's input deviates by the same 4.4% in the same mode.  Every
    order-free kernel has its own tolerance test; the batch's composition is
    pinned bit for bit by the exact test above."""
    L, want, handles = _setup(ctx, oracle, dev)
    cap, ld = 16, HEAD_DIM + 64
    rng = np.random.default_rng(22)
    kv0 = (rng.standard_normal((cap, ld)) * 0.3).astype(np.float32)
    positions = list(range(2, 10))
    h0 = (rng.standard_normal((len(positions), HC * wl.HIDDEN)) * 0.5).astype(np.float32)
    ctx.set_exact_numerics(True)
    exact, _ = _run(ctx, dev, L, h0, positions, kv0, ld)
    ctx.set_exact_numerics(False)
    got, _ = _run(ctx, dev, L, h0, positions, kv0, ld)
    assert np.all(np.isfinite(got))
    rel = np.linalg.norm(got - exact, axis=1) / np.linalg.norm(exact, axis=1)
    print("per-position ||diff|| / ||value||:", np.array2string(rel, precision=6))
    assert float(rel.max()) <= 0.1
    assert float(np.median(rel)) <= 3e-2
    for t in handles.values():
        ctx.release(t)


@pytest.mark.parametrize("n", [5, 16, 17, 33, 131])
def test_decode_layer_batch_matches_small(ctx, oracle, dev, n):
    """Exact numerics: n positions in one call against calls of at most four,
    bit for bit: the projections and the router of 16 inputs on matrix
    instructions with a partial last tile, and more positions than one launch
    of the window attention takes."""
    ctx.set_exact_numerics(True)
    L, _, handles = _setup(ctx, oracle, dev)
    cap, ld = n + 3, HEAD_DIM
    rng = np.random.default_rng(n)
    kv0 = np.zeros((cap, ld), np.float32)
    kv0[:3] = (rng.standard_normal((3, ld)) * 0.3).astype(np.float32)
    positions = list(range(3, 3 + n))
    h0 = (rng.standard_normal((n, HC * wl.HIDDEN)) * 0.5).astype(np.float32)
    got, got_kv = _run(ctx, dev, L, h0, positions, kv0, ld)
    want, want_kv = np.empty_like(got), kv0
    for i in range(0, n, 4):
        want[i:i + 4], want_kv = _run(ctx, dev, L, h0[i:i + 4], positions[i:i + 4], want_kv, ld)
    assert np.array_equal(bits(got_kv), bits(want_kv))
    for i in range(n):
        assert np.array_equal(bits(got[i]), bits(want[i])), (i, int(np.count_nonzero(bits(got[i]) != bits(want[i]))))
    for t in handles.values():
        ctx.release(t)


def test_decode_layer_batch_order_free_many(ctx, oracle, dev):
    """Exact numerics off, 33 positions in one call (hc_pre's sums of four
    streams a workgroup, a partial last one) against calls of at most 8: the
    bounds of the test above against the exact batch, for the same reasons."""
    L, _, handles = _setup(ctx, oracle, dev)
    n, ld = 33, HEAD_DIM
    rng = np.random.default_rng(23)
    kv0 = (rng.standard_normal((n + 2, ld)) * 0.3).astype(np.float32)
    positions = list(range(2, 2 + n))
    h0 = (rng.standard_normal((n, HC * wl.HIDDEN)) * 0.5).astype(np.float32)
    ctx.set_exact_numerics(False)
    got, _ = _run(ctx, dev, L, h0, positions, kv0, ld)
    want = np.empty_like(got)
    kv = kv0
    for i in range(0, n, 8):
        want[i:i + 8], kv = _run(ctx, dev, L, h0[i:i + 8], positions[i:i + 8], kv, ld)
    assert np.all(np.isfinite(got))
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    print("per-position ||diff|| / ||value||:", np.array2string(rel, precision=6))
    assert float(rel.max()) <= 0.1
    assert float(np.median(rel)) <= 3e-2
    for t in handles.values():
        ctx.release(t)


def test_decode_layer_batch_errors(ctx, oracle, dev):
    L, want, handles = _setup(ctx, oracle, dev)
    cap, ld = 8, HEAD_DIM
    hp, kvp = dev.put(np.zeros((2, HC * wl.HIDDEN), np.float32)), dev.put(np.zeros((cap, ld), np.float32))
    with pytest.raises(wohper_amd.DeepSeekV4KernelError) as e:
        ctx.deepseek_mhc_layer_batch_async(L, [], hp, kvp, ld, cap)
    assert e.value.name == "InvalidShape"
    with pytest.raises(wohper_amd.DeepSeekV4KernelError) as e:
        ctx.deepseek_mhc_layer_batch_async(L, [4, 3], hp, kvp, ld, cap)
    assert e.value.name == "InvalidArgument"
    for t in handles.values():
        ctx.release(t)
