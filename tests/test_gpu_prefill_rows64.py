"""The 64-rows-per-wave prefill kernel (prefill_rows64.hip): the layouts that
attention_generic took before (64-dim heads, KV heads shared by other than a
multiple of four query heads), against that kernel on the same inputs, and the
middle range of the model's layout, against the fp64 oracle."""
import numpy as np
import pytest
import torch

import oracle
from helpers import assert_close

pytestmark = pytest.mark.gpu


def inputs(N, Hq, Hkv, D, pad, seed, grow=False):
    """Q rows of a fused [Q | K | V] buffer, K and V rows of a cache; `pad`
    elements past each row.  grow: scores rise along the keys, so that the
    running maximum is raised again and again."""
    rng = np.random.default_rng(seed)
    qs, ks = (Hq + 2 * Hkv) * D + pad, Hkv * D + pad
    q = rng.standard_normal((N, qs)).astype(np.float16)
    k = rng.standard_normal((N, ks)).astype(np.float16)
    v = rng.standard_normal((N, ks)).astype(np.float16)
    if grow:
        k = (k * np.linspace(0.1, 6.0, N)[:, None]).astype(np.float16)
    return q, k, v, qs, ks


def run(attn, device, q, k, v, Hq, Hkv, D, qs, ks):
    N = q.shape[0]
    d = [torch.from_numpy(x.copy()).to(device) for x in (q, k, v)]
    guard = 64
    out = torch.full((N * Hq * D + 2 * guard,), 77.0, dtype=torch.float16, device=device)
    attn.prefill(*d, out[guard:].data_ptr(), N, Hq, Hkv, D, qs, ks)
    torch.cuda.synchronize()
    o = out.cpu().numpy()
    assert (o[:guard] == 77).all() and (o[-guard:] == 77).all(), "write outside out"
    return o[guard:-guard].reshape(N, Hq * D)


def run_generic(attn, device, *args):
    attn.set_option("prefill_force_generic", 1)
    try:
        return run(attn, device, *args)
    finally:
        attn.set_option("prefill_force_generic", 0)


def assert_as_generic(got, ref, v):
    # both sum fp32 products of fp32 (or 22-bit) weights: they differ by fp32
    # rounding of sums of terms up to max|v| (2e-6 of it, ~30 roundings of
    # 2^-24), and then by at most one rounding to fp16 (2^-10 of the value)
    ref, got = ref.astype(np.float64), got.astype(np.float64)
    bound = 2.0 ** -10 * np.abs(ref) + 2e-6 * np.abs(v.astype(np.float64)).max() + 2.0 ** -24
    bad = ~(np.abs(got - ref) <= bound)
    assert not bad.any(), (int(bad.sum()), np.argwhere(bad)[:4], np.abs(got - ref).max())


# the shortest prompt of the kernel by the number of heads; one token less is
# attention_generic's, bit for bit
@pytest.mark.parametrize("Hq,Hkv,D,least", [(20, 10, 128, 64), (16, 16, 128, 74), (10, 5, 128, 84),
                                            (9, 9, 128, 104), (4, 4, 128, 112), (3, 3, 128, 136),
                                            (1, 1, 128, 136), (8, 8, 64, 64), (2, 1, 64, 66)])
def test_rows64_from_where_it_is_faster(attn, gpu, Hq, Hkv, D, least):
    q, k, v, qs, ks = inputs(least, Hq, Hkv, D, 0, 9)
    for N in (least - 1, least):
        print(f"[case] rows64 route Hq={Hq} D={D} N={N}", flush=True)
        args = (q[:N], k[:N], v[:N], Hq, Hkv, D, qs, ks)
        got, ref = run(attn, gpu, *args), run_generic(attn, gpu, *args)
        assert_as_generic(got, ref, v)
        if N < least:
            assert np.array_equal(got.view(np.uint16), ref.view(np.uint16))


# one and several key units per wave, the last query tile full, one row and one
# block long; past two rounds of workgroups (1041 and 576 of them) two key parts
@pytest.mark.parametrize("Hq,Hkv,D,N,pad", [
    (16, 16, 128, 64, 0), (16, 16, 128, 65, 0), (20, 20, 128, 64, 0), (20, 10, 128, 65, 0),
    (16, 16, 128, 74, 0), (3, 3, 128, 136, 0), (16, 8, 128, 97, 8), (6, 2, 128, 130, 24),
    (5, 5, 128, 300, 0), (16, 16, 128, 1000, 0), (32, 16, 128, 1100, 8),
    (16, 4, 64, 64, 0), (16, 4, 64, 95, 8), (8, 8, 64, 128, 0), (3, 1, 64, 129, 16),
    (16, 4, 64, 1025, 0), (16, 8, 64, 4161, 0)])
@pytest.mark.parametrize("grow", [False, True])
def test_rows64_as_generic(attn, gpu, Hq, Hkv, D, N, pad, grow):
    print(f"[case] rows64 Hq={Hq} Hkv={Hkv} D={D} N={N} pad={pad} grow={grow}", flush=True)
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, pad, N + Hq, grow)
    args = (q, k, v, Hq, Hkv, D, qs, ks)
    got = run(attn, gpu, *args)
    assert_as_generic(got, run_generic(attn, gpu, *args), v)


@pytest.mark.parametrize("Hq,Hkv,D,N", [(16, 16, 128, 300), (16, 4, 64, 300), (16, 8, 64, 4200)])
def test_rows64_infinities_and_nans(attn, gpu, Hq, Hkv, D, N):
    """An infinity or NaN in K or V reaches exactly the rows that see its key."""
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, 0, 5)
    v[N - 60, 3] = np.inf
    v[N - 40, D + 7] = np.nan
    k[N - 20, 1] = np.nan
    v[N - 10, 5] = -np.inf
    print(f"[case] rows64 inf/nan Hq={Hq} Hkv={Hkv} D={D} N={N}", flush=True)
    args = (q, k, v, Hq, Hkv, D, qs, ks)
    got, ref = run(attn, gpu, *args), run_generic(attn, gpu, *args)
    assert np.isfinite(ref[:N - 60]).all() and not np.isfinite(ref[N - 1]).all()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fine = np.isfinite(ref)
    assert_as_generic(np.where(fine, got, 0), np.where(fine, ref, 0),
                      np.where(np.isfinite(v), v, 0))


# 16 heads: the first and the last length of the range (192 and 256 workgroups),
# with one row and 32 rows in the last tile; 32, 24 and 12 heads (up to 512)
@pytest.mark.parametrize("Hq,Hkv,N,pad", [
    (16, 4, 704, 0), (16, 4, 705, 0), (16, 4, 736, 8), (16, 4, 800, 0), (16, 4, 1024, 0),
    (32, 8, 353, 0), (32, 4, 1023, 8), (24, 3, 700, 0), (12, 3, 1000, 0)])
@pytest.mark.parametrize("grow", [False, True])
def test_rows64_model_layout(attn, gpu, Hq, Hkv, N, pad, grow):
    D = 128
    print(f"[case] rows64 model layout Hq={Hq} Hkv={Hkv} N={N} grow={grow}", flush=True)
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, pad, 3 * N, grow)
    got = run(attn, gpu, q, k, v, Hq, Hkv, D, qs, ks)
    rows = np.unique(np.concatenate([np.arange(0, N, 17), np.arange(max(0, N - 66), N)]))
    _, e32 = oracle.attention(q.view(np.uint16).ravel(), k.view(np.uint16).ravel(),
                              v.view(np.uint16).ravel(), N, Hq, Hkv, D, qs, ks, N, causal=True,
                              rows=rows)
    assert_close(got[rows].reshape(-1).view(np.uint16), e32.reshape(-1), 2e-3, 1e-2, f"N={N}")


def test_rows64_prefix_invariance(attn, gpu):
    """A row depends on the rows up to it only, bit for bit, also where the
    prefix ends inside its query tile."""
    q, k, v, qs, ks = inputs(1020, 16, 4, 128, 0, 8)
    whole = run(attn, gpu, q, k, v, 16, 4, 128, qs, ks)
    for n in (705, 766, 960):
        part = run(attn, gpu, q[:n], k[:n], v[:n], 16, 4, 128, qs, ks)
        assert np.array_equal(part.view(np.uint16), whole[:n].view(np.uint16)), n


# the model's layout, and both numbers of key parts of the others
@pytest.mark.parametrize("Hq,Hkv,D,N", [(16, 4, 128, 1000), (16, 16, 128, 300), (16, 4, 64, 300),
                                        (32, 16, 128, 1100), (16, 8, 64, 4161)])
def test_rows64_row_independence(attn, gpu, Hq, Hkv, D, N):
    """A row's output does not depend on the other queries of its tile, bit for
    bit, where their growing scores raise their maxima again and again."""
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, 0, 11)
    others = np.arange(N) % 32 >= 16
    sharp = q.copy()
    sharp[others] *= np.float16(24)
    print(f"[case] rows64 row independence Hq={Hq} Hkv={Hkv} D={D} N={N}", flush=True)
    a = run(attn, gpu, q, k, v, Hq, Hkv, D, qs, ks)
    b = run(attn, gpu, sharp, k, v, Hq, Hkv, D, qs, ks)
    assert np.array_equal(a[~others].view(np.uint16), b[~others].view(np.uint16))
    assert not np.array_equal(a[others], b[others])


@pytest.mark.parametrize("N", [705, 800, 1024])
def test_rows64_model_layout_infinities_and_nans(attn, gpu, N):
    """The model's layout: an infinity or NaN in V reaches exactly the rows that
    see its key, not the earlier rows of the tile."""
    Hq, Hkv, D = 16, 4, 128
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, 0, 6)
    v[N - 30, 3] = np.inf
    v[N - 20, D + 7] = np.nan
    v[N - 10, 2 * D + 5] = -np.inf
    v[500, 3 * D + 9] = np.inf
    print(f"[case] rows64 model layout inf/nan N={N}", flush=True)
    args = (q, k, v, Hq, Hkv, D, qs, ks)
    got, ref = run(attn, gpu, *args), run_generic(attn, gpu, *args)
    assert np.isfinite(ref[:500]).all() and not np.isfinite(ref[N - 1]).all()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fine = np.isfinite(ref)
    assert_close(np.where(fine, got, 0).astype(np.float16).reshape(-1).view(np.uint16),
                 np.where(fine, ref, 0).astype(np.float32).reshape(-1), 2e-3, 1e-2, f"N={N}")


@pytest.mark.parametrize("Hq,Hkv,N,form", [
    # the all-tiles form up to 256 tokens, the 32-query streaming form where its
    # workgroups are few, else this kernel
    (64, 16, 150, 2), (64, 16, 256, 2), (128, 32, 65, 2), (128, 32, 192, 2),
    (64, 16, 257, 4), (64, 16, 288, 4), (48, 12, 340, 4), (40, 10, 416, 4),
    (64, 16, 289, 0), (40, 10, 417, 0), (96, 24, 257, 0), (40, 10, 384, 0)])
def test_rows64_grouped_layout_routes(attn, gpu, Hq, Hkv, N, form):
    """Many heads of the grouped layout: the form that is fastest there (256 CUs)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are in workgroups per CU, the sizes for 256 CUs")
    D = 128
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, 0, 10)
    print(f"[case] rows64 grouped route Hq={Hq} N={N}", flush=True)
    args = (q, k, v, Hq, Hkv, D, qs, ks)
    got = run(attn, gpu, *args).view(np.uint16)
    try:
        attn.set_option("prefill_split_keys", form or 4)
        forced = run(attn, gpu, *args).view(np.uint16)
    finally:
        attn.set_option("prefill_split_keys", 0)
    assert np.array_equal(got, forced) == (form != 0)
    assert_close(got.reshape(-1), forced.astype(np.uint16).view(np.float16).astype(np.float32)
                 .reshape(-1), 2e-3, 1e-2, f"{Hq}/{Hkv} N={N}")


def prefill_us(attn, device, q, k, v, Hq, Hkv, D, qs, ks):
    d = [torch.from_numpy(x.copy()).to(device) for x in (q, k, v)]
    out = torch.empty(q.shape[0] * Hq * D, dtype=torch.float16, device=device)
    times = []
    for _ in range(4):
        e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        e0.record()
        attn.prefill(*d, out, q.shape[0], Hq, Hkv, D, qs, ks)
        e1.record()
        e1.synchronize()
        times.append(1e3 * e0.elapsed_time(e1))
    return min(times)


@pytest.mark.parametrize("Hq,Hkv,D,where", [
    (16, 4, 128, "all"), (16, 16, 128, "all"), (16, 4, 64, "all"),
    (16, 4, 128, "k"), (16, 16, 128, "k"), (16, 4, 64, "k"), (16, 4, 128, "v")])
def test_rows64_nan_inputs_cost_no_more(attn, gpu, Hq, Hkv, D, where):
    """Rows whose scores are NaN are NaN without being computed again key by key,
    and so, in the grouped layout, are rows that no later key has spoilt: with NaN
    inputs a call takes less than attention_generic (0.3 ms and more; 10 ms where
    every row was computed again)."""
    N = 1000
    q, k, v, qs, ks = inputs(N, Hq, Hkv, D, 0, 14)
    if where == "all":
        q, k, v = (np.full_like(x, np.nan) for x in (q, k, v))
    else:
        (k if where == "k" else v)[3] = np.nan
    print(f"[case] rows64 nan Hq={Hq} Hkv={Hkv} D={D} {where}", flush=True)
    args = (q, k, v, Hq, Hkv, D, qs, ks)
    got, ref = run(attn, gpu, *args), run_generic(attn, gpu, *args)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    us = prefill_us(attn, gpu, *args)
    try:
        attn.set_option("prefill_force_generic", 1)
        generic_us = prefill_us(attn, gpu, *args)
    finally:
        attn.set_option("prefill_force_generic", 0)
    print(f"  {us:.0f} us against {generic_us:.0f}", flush=True)
    assert us < generic_us


def sink_inputs(N, Hq, Hkv, D, nats, sinks, seed):
    """Keys `sinks` score about `nats` above the others and carry V = 0; V is large
    enough that what the other keys leave is a normal fp16 value."""
    rng = np.random.default_rng(seed)
    u = rng.choice([-1.0, 1.0], (Hkv, D))
    q = 2.0 * np.repeat(u, Hq // Hkv, 0)[None] + 0.2 * rng.standard_normal((N, Hq, D))
    k = 0.3 * rng.standard_normal((N, Hkv, D))
    v = 4096.0 * (1.0 + 0.3 * rng.standard_normal((N, Hkv, D)))
    k[sinks] = nats / (2.0 * np.sqrt(D)) * u
    v[sinks] = 0.0
    return [x.reshape(N, -1).astype(np.float16) for x in (q, k, v)]


# one sink in the first unit of 32 keys and in a later one, one in every unit;
# both numbers of key parts
@pytest.mark.parametrize("Hq,Hkv,D,N", [(4, 4, 128, 300), (8, 2, 64, 300), (32, 16, 128, 1100),
                                        (16, 8, 64, 4161)])
@pytest.mark.parametrize("sinks", [[0], [100], list(range(3, 300, 29))])
@pytest.mark.parametrize("nats", [6, 12, 16, 20])
def test_rows64_small_weights_beside_sinks(attn, gpu, Hq, Hkv, D, N, sinks, nats):
    """Weights far below the largest keep their bits: no further from 64 bits than
    attention_generic's fp32 weights (whose own error is the fp16 rounding of the
    output; 2 % for another order of the sums)."""
    q, k, v = sink_inputs(N, Hq, Hkv, D, nats, sinks, 13 + nats)
    print(f"[case] rows64 sinks Hq={Hq} D={D} N={N} nats={nats} at={sinks[:2]}", flush=True)
    args = (q, k, v, Hq, Hkv, D, Hq * D, Hkv * D)
    rows = np.arange(1, N, 1 if N <= 300 else 23)
    _, e32 = oracle.attention(q.view(np.uint16).ravel(), k.view(np.uint16).ravel(),
                              v.view(np.uint16).ravel(), N, Hq, Hkv, D, Hq * D, Hkv * D, N,
                              causal=True, rows=rows)
    exact = e32.reshape(len(rows), -1).astype(np.float64)
    got, ref = (run_(attn, gpu, *args)[rows].astype(np.float64) for run_ in (run, run_generic))
    for name, part in (("all", slice(None)), ("first", rows < 128), ("last", rows >= N - 128)):
        err = [np.linalg.norm(x[part] - exact[part]) / np.linalg.norm(exact[part])
               for x in (got, ref)]
        print(f"  {name}: {err[0]:.3e} against {err[1]:.3e}", flush=True)
        assert err[0] <= 1.02 * err[1] + 1e-6, (name, err)
