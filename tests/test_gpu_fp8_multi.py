"""GPU parity of the exact multi-input FP8 GEMV (k_fp8_gemv_multi: each
weight byte decoded once for every input, each input's dot in the
single-input kernel's order) against the oracle's restatement of
gemv_fp8_e4m3_ue8m0_rows_multi (E/compute.rs:6384-6577), bit for bit: the
decode layer's shapes at batch 16, partial input blocks (2, 5, 9, 20
inputs), unaligned row ranges, UE8M0 and f32 scales, the +-480 codes, the
pair entry point (wq_a + wkv on one input set) and row groups with their
own inputs (wo_a)."""
import numpy as np
import pytest

import wohper_amd
from parity_util import bits
from wohper_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def exact(ctx):
    ctx.set_exact_numerics(True)
    yield


def _tensor(ctx, rows, cols, seed, ue8m0=False, special=False):
    case = wl.fp8_gemv_case(rows, cols, seed=seed, ue8m0_compatible=ue8m0)
    w = case.w.copy()
    if special:
        rng = np.random.default_rng(seed)
        w[rng.integers(0, rows, 64), rng.integers(0, cols, 64)] = 0x7F
        w[rng.integers(0, rows, 64), rng.integers(0, cols, 64)] = 0xFF
    if ue8m0:
        sb = (np.log2(case.scales).astype(np.int32) + 127).astype(np.uint8)
        t = ctx.store_fp8(w, rows, cols, sb, rows // 128, cols // 128, wohper_amd.SCALE_UE8M0)
    else:
        t = ctx.store_fp8(w, rows, cols, case.scales, rows // 128, cols // 128, wohper_amd.SCALE_F32)
    return t, w, case.scales


def _run(ctx, t, xs, r0, r1):
    n, cols = xs.shape
    xd, yd = ctx.device_alloc(xs.nbytes), ctx.device_alloc(n * (r1 - r0) * 4)
    ctx.to_device(xd, np.ascontiguousarray(xs))
    ctx.fp8_gemv_multi_async(t, r0, r1, xd, n, cols, yd, r1 - r0)
    ys = np.empty((n, r1 - r0), np.float32)
    ctx.synchronize()
    ctx.from_device(ys, yd)
    ctx.device_free(xd)
    ctx.device_free(yd)
    return ys


@pytest.mark.parametrize("rows,cols,n,r0,r1,ue8m0", [
    (4096, 4096, 16, 0, 4096, False), (32768, 1024, 16, 0, 32768, True), (4096, 8192, 16, 0, 4096, False),
    (1024, 2048, 5, 100, 900, True), (512, 4096, 9, 3, 509, False), (1024, 1024, 2, 0, 1024, True),
    (1024, 4096, 20, 64, 1024, False), (4096, 4096, 7, 0, 4096, True), (8192, 2048, 3, 128, 8064, False)])
def test_multi_exact_matches_rows_multi(ctx, oracle, rows, cols, n, r0, r1, ue8m0):
    t, w, scales = _tensor(ctx, rows, cols, rows + cols + n, ue8m0)
    xs = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    ys = _run(ctx, t, xs, r0, r1)
    want = oracle.fp8_gemv_rows_multi(w, rows, cols, scales, rows // 128, cols // 128, xs, r0, r1)
    for i in range(n):
        assert np.array_equal(bits(ys[i]), bits(want[i])), (i, int(np.count_nonzero(bits(ys[i]) != bits(want[i]))))
    ctx.release(t)


@pytest.mark.parametrize("rows,cols,n,r0,r1,ue8m0", [
    (4096, 8192, 2, 0, 4096, False), (4224, 1024, 13, 16, 4209, True), (4224, 2048, 18, 0, 4224, False),
    (8320, 2048, 9, 0, 8320, True), (8320, 3072, 25, 128, 8320, False), (32768, 1024, 29, 0, 32768, False)])
def test_multi_exact_matrix_instructions(ctx, oracle, rows, cols, n, r0, r1, ue8m0):
    """The one-term matrix instructions: one and two row tiles a wave, a partial
    last row tile, partial tiles of inputs, two and more chunks of columns; an
    input of tiny values (products and sums below the normal range) and one of
    large ones keep their own columns."""
    t, w, scales = _tensor(ctx, rows, cols, rows + cols + n, ue8m0)
    xs = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    xs[0] *= np.float32(2.0 ** -126)
    xs[n - 1] *= np.float32(1e30)
    ys = _run(ctx, t, xs, r0, r1)
    want = oracle.fp8_gemv_rows_multi(w, rows, cols, scales, rows // 128, cols // 128, xs, r0, r1)
    assert np.array_equal(bits(ys), bits(np.stack(want)))
    ctx.release(t)


def test_multi_exact_special_codes(ctx, oracle):
    rows, cols, n = 1024, 2048, 16
    t, w, scales = _tensor(ctx, rows, cols, 17, special=True)
    xs = np.random.default_rng(4).standard_normal((n, cols)).astype(np.float32)
    ys = _run(ctx, t, xs, 0, rows)
    want = oracle.fp8_gemv_rows_multi(w, rows, cols, scales, rows // 128, cols // 128, xs)
    assert np.array_equal(bits(ys), bits(want))
    ctx.release(t)


def test_multi_exact_pair_and_groups(ctx, oracle):
    """wq_a + wkv on one set of 16 inputs in one launch, and wo_a's 8 row
    groups of 1024 each on its own 16 inputs."""
    n = 16
    ta, wa, sa = _tensor(ctx, 1024, 4096, 31)
    tk, wk, sk = _tensor(ctx, 512, 4096, 32)
    xs = np.random.default_rng(8).standard_normal((n, 4096)).astype(np.float32)
    xd = ctx.device_alloc(xs.nbytes)
    ctx.to_device(xd, xs)
    ya, yk = ctx.device_alloc(n * 1024 * 4), ctx.device_alloc(n * 512 * 4)
    ctx.fp8_gemv_multi_pair_async(ta, 0, 1024, ya, 1024, tk, 0, 512, yk, 512, xd, n, 4096)
    ctx.synchronize()
    got_a, got_k = np.empty((n, 1024), np.float32), np.empty((n, 512), np.float32)
    ctx.from_device(got_a, ya)
    ctx.from_device(got_k, yk)
    assert np.array_equal(bits(got_a), bits(oracle.fp8_gemv_rows_multi(wa, 1024, 4096, sa, 8, 32, xs)))
    assert np.array_equal(bits(got_k), bits(oracle.fp8_gemv_rows_multi(wk, 512, 4096, sk, 4, 32, xs)))
    for p in (xd, ya, yk):
        ctx.device_free(p)
    # wo_a: 8 groups of 1024 rows, group g reads its own 16 inputs
    to, wo, so = _tensor(ctx, 8192, 4096, 33)
    xg = np.random.default_rng(9).standard_normal((n, 8, 4096)).astype(np.float32)
    xd, yd = ctx.device_alloc(xg.nbytes), ctx.device_alloc(n * 8192 * 4)
    ctx.to_device(xd, xg)
    ctx.fp8_gemv_multi_groups_async(to, 0, 8192, 1024, xd, 4096, n, 8 * 4096, yd, 8192)
    ctx.synchronize()
    got = np.empty((n, 8192), np.float32)
    ctx.from_device(got, yd)
    for g in range(8):
        want = oracle.fp8_gemv_rows_multi(wo, 8192, 4096, so, 64, 32, xg[:, g], 1024 * g, 1024 * (g + 1))
        assert np.array_equal(bits(got[:, 1024 * g:1024 * (g + 1)]), bits(want)), g
    ctx.device_free(xd)
    ctx.device_free(yd)
    for t in (ta, tk, to):
        ctx.release(t)


@pytest.mark.parametrize("rows,cols,n,r0,r1,ue8m0,special", [
    (4096, 4096, 2, 0, 4089, True, True), (4096, 2048, 6, 16, 4096, False, False),
    (4096, 1024, 13, 0, 4096, True, False),     # one round of 16-row tiles
    (6144, 2048, 12, 16, 6137, False, True), (8192, 2048, 13, 16, 8185, True, False),   # two, a partial last one
    (6144, 2048, 24, 16, 6137, True, True), (16384, 1024, 15, 0, 16377, False, False),  # 32-row tiles
    (32768, 1024, 15, 0, 32761, False, False)])
def test_multi_exact_matrix_instructions_full_rounds(ctx, oracle, rows, cols, n, r0, r1, ue8m0, special):
    """Products that the one-term matrix instructions take: rounds of 256
    workgroups that are full enough, with partial tiles of rows and inputs."""
    t, w, scales = _tensor(ctx, rows, cols, rows + n, ue8m0, special)
    xs = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    xs[0] *= np.float32(2.0 ** -126)
    xs[n - 1] *= np.float32(1e30)
    ys = _run(ctx, t, xs, r0, r1)
    want = oracle.fp8_gemv_rows_multi(w, rows, cols, scales, rows // 128, cols // 128, xs, r0, r1)
    assert np.array_equal(bits(ys), bits(np.stack(want)))
    ctx.release(t)


@pytest.mark.parametrize("rows,cols,n,most", [(5120, 2048, 9, 1.2), (6144, 3072, 9, 1.15), (5120, 1024, 13, 1.32)])
def test_multi_exact_time_follows_inputs(ctx, rows, cols, n, most):
    """Products that fill less than half of a round of the matrix
    instructions' workgroups stay with the vector kernel: one more input than
    a whole block of it costs 1.07, 1.04 and 1.19 times as much, not the 1.31,
    1.24 and 1.41 times of a tile of 16."""
    t = ctx.store_fp8_synthetic(rows, cols, 3, 1, np.full((rows // 128, cols // 128), 2.0 ** -10, np.float32))
    x = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    xd, y = ctx.device_alloc(x.nbytes), ctx.device_alloc(4 * n * rows)
    ctx.to_device(xd, x)
    us = {}
    for k in (n - 1, n):
        ctx.fp8_gemv_multi_async(t, 0, rows, xd, k, cols, y, rows)
        ctx.synchronize()
        g = ctx.graph_capture(lambda: [ctx.fp8_gemv_multi_async(t, 0, rows, xd, k, cols, y, rows) for _ in range(20)])
        v = []
        for _ in range(6):
            ctx.timer_start()
            ctx.graph_launch(g)
            v.append(ctx.timer_stop() / 20)
        ctx.graph_release(g)
        us[k] = min(v)
    print(f"{rows} x {cols}: {n - 1} inputs {us[n - 1]:.2f} us, {n} inputs {us[n]:.2f} us")
    ctx.release(t)
    ctx.device_free(xd)
    ctx.device_free(y)
    assert us[n] <= most * us[n - 1]
