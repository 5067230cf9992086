"""Dispatch rules by their times: of two calls that share the work, or whose work
differs by a known factor, neither may take far longer than the other.  Each
bound lies between what a right choice and a wrong one measured on MI355X, at
least a fifth away from the right one."""
import itertools

import pytest

pytestmark = pytest.mark.gpu


def torch():
    import torch as t
    return t


def times(*calls):
    """Best time in us of each call among 24 queued ones, the calls timed in turn."""
    t = torch()
    best = [float("inf")] * len(calls)
    for call in calls:
        call()
    t.cuda.synchronize()
    for _ in range(7):
        for i, call in enumerate(calls):
            start, end = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(24):
                call()
            end.record()
            end.synchronize()
            best[i] = min(best[i], start.elapsed_time(end) * 1e3 / 24)
    return best


def attention(ops, batch, heads, nq, nk, d, causal):
    t = torch()
    gen = t.Generator(device="cuda").manual_seed(batch)
    q, k, v = (t.randn(batch, heads, n, d, generator=gen, device="cuda").half() for n in (nq, nk, nk))
    off = [nk - nq] * batch
    return lambda: ops.attention(q, k, v, query_offsets=off, causal=causal)


@pytest.mark.parametrize("d", [64, 128])
def test_few_attention_rows_use_every_xcd(ops, d):
    """4 heads of 4096 queries against 8: half the work (28 and 58 us at 64 dims;
    57 and 58 with whole rows on single XCDs)."""
    print("[case] attention rows", d, flush=True)
    half, whole = times(attention(ops, 1, 4, 4096, 4096, d, False), attention(ops, 1, 8, 4096, 4096, d, False))
    assert half < 0.75 * whole, (half, whole)


@pytest.mark.parametrize("causal", [False, True])
def test_many_attention_rows_keep_their_l2_share(ops, causal):
    """32 requests against 8 of the same shape: four times the work (295 and 85 us
    without a mask; 555 and 101 with every row of an XCD in flight)."""
    print("[case] attention batch", causal, flush=True)
    small, large = times(attention(ops, 8, 25, 333, 1500, 128, causal), attention(ops, 32, 25, 333, 1500, 128, causal))
    assert large < 4.6 * small, (small, large)


def linear(ops, kind, m, k, n, out="f16"):
    """An int8 or fp16 linear over weights that rotate, as a model's layers."""
    t = torch()
    gen = t.Generator(device="cuda").manual_seed(m + k + n)
    a = t.randn(m, k, generator=gen, device="cuda").half()
    sets = max(1, min(24, (300 << 20) // (k * n)))
    w = t.randint(-127, 128, (sets, k, n), generator=gen, device="cuda", dtype=t.int8)
    if kind == "fp16":
        w = w.half()
    s = t.rand(n, generator=gen, device="cuda") * 1e-3
    dtype = t.float32 if out == "f32" else t.float16
    at = itertools.count()

    def call():
        held = w[next(at) % sets]
        return ops.gemm_int8(a, held, s, output_dtype=dtype) if kind == "int8" else ops.gemm(a, held, output_dtype=dtype)
    return call


@pytest.mark.parametrize("kind,k", [("int8", 3072), ("fp16", 6400)])
def test_few_columns_above_1024_rows_split_k(ops, kind, k):
    """fp32 outputs take the kernel that splits K; fp16 ones of the same product
    need not be slower (int8: 15 and 15 us; 42 and 15 as one chain over K)."""
    print("[case] few columns", kind, k, flush=True)
    half, single = times(linear(ops, kind, 1100, k, 64), linear(ops, kind, 1100, k, 64, out="f32"))
    assert half < 1.6 * single, (half, single)


@pytest.mark.parametrize("m,k,n", [(866, 3072, 1600), (523, 2160, 2304)])
def test_long_sums_over_few_tiles_cut_k(ops, m, k, n):
    """fp32 outputs take the kernel that cuts K over waves; fp16 ones of the same
    product need not be slower (35 and 37 us; 53 as one chain over K)."""
    print("[case] long sums", m, k, n, flush=True)
    half, single = times(linear(ops, "int8", m, k, n), linear(ops, "int8", m, k, n, out="f32"))
    assert half < 1.2 * single, (half, single)


def test_odd_wide_rows_at_short_k(ops):
    """int8 rows of any alignment at short K are no slower than fp16 ones of twice
    the bytes (105 and 97 us; 241 with each weight converted once per 32 rows)."""
    print("[case] odd wide rows", flush=True)
    int8, fp16 = times(linear(ops, "int8", 1024, 64, 50257), linear(ops, "fp16", 1024, 64, 50257))
    assert int8 < 1.5 * fp16, (int8, fp16)
