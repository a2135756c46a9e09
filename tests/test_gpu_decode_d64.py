"""Split decode of 64-dim heads (decode_d64.hip) against attention_generic, which
took these heads before, on the same inputs; and its graph nodes."""
import numpy as np
import pytest
import torch

import oracle
from attn_mi355x import hipgraph
from helpers import assert_close

pytestmark = pytest.mark.gpu
D = 64
SENTINEL = 123.0


def inputs(L, Hq, Hkv, stride, seed, device):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal(Hq * D).astype(np.float16)
    k = rng.standard_normal((L + 2, stride)).astype(np.float16)
    v = rng.standard_normal((L + 2, stride)).astype(np.float16)
    k[L:] = v[L:] = SENTINEL
    return (q, k, v), [torch.from_numpy(x).to(device) for x in (q, k, v)]


def workspace(attn, Hq, L, device):
    # NaN-filled and guarded: every state read must have been written, and
    # nothing past the documented capacity is
    n = attn.decode_workspace_states(Hq, L)
    return [torch.full((m + 8,), float("nan"), device=device) for m in (n * D, n, n)], n


def decode(attn, d, L, Hq, Hkv, stride, device):
    ws, n = workspace(attn, Hq, L, device)
    for w in ws:
        w[-8:] = 7.0
    out = torch.full((Hq * D + 8,), 77.0, dtype=torch.float16, device=device)
    attn.decode(*d, out, *ws, 1, L, L - 1, Hq, Hkv, D, 0, stride)
    torch.cuda.synchronize()
    assert all((w[-8:] == 7).all() for w in ws) and (out[-8:] == 77).all()
    return out[:-8].cpu().numpy()


def generic(attn, *args):
    attn.set_option("decode_force_generic", 1)
    try:
        return decode(attn, *args)
    finally:
        attn.set_option("decode_force_generic", 0)


def assert_as_generic(got, ref, v):
    # fp32 sums of the same terms in another order: at most ~2e-6 of the largest
    # |v| apart, then one rounding to fp16 (2^-10 of the value)
    ref, got = ref.astype(np.float64), got.astype(np.float64)
    bound = 2.0 ** -10 * np.abs(ref) + 2e-6 * np.abs(v.astype(np.float64)).max() + 2.0 ** -24
    assert (np.abs(got - ref) <= bound).all(), np.abs(got - ref).max()


# one chunk and several, ragged quarters of a wave, more than one round per
# wave, up to 64 and 256 states; groups of 1, 2, 3, 4, 8 and 12 query heads
@pytest.mark.parametrize("Hq,Hkv,pad", [(16, 4, 0), (8, 8, 0), (4, 2, 8), (6, 2, 0), (16, 2, 0),
                                        (12, 1, 24)])
@pytest.mark.parametrize("L", [1, 7, 12, 31, 64, 65, 127, 200, 1000, 3000, 20001])
def test_decode_d64_as_generic(attn, gpu, Hq, Hkv, pad, L):
    stride = Hkv * D + pad
    print(f"[case] decode d64 Hq={Hq} Hkv={Hkv} pad={pad} L={L}", flush=True)
    (q, k, v), d = inputs(L, Hq, Hkv, stride, L + Hq, gpu)
    got = decode(attn, d, L, Hq, Hkv, stride, gpu)
    assert_as_generic(got, generic(attn, d, L, Hq, Hkv, stride, gpu), v[:L])
    _, e32 = oracle.attention(q.view(np.uint16), k.view(np.uint16).ravel(),
                              v.view(np.uint16).ravel(), 1, Hq, Hkv, D, Hq * D, stride, L,
                              causal=False)
    assert_close(got.view(np.uint16), e32.reshape(-1), 2e-3, 1e-2, f"L={L}")


def test_decode_d64_large_scores_and_nan(attn, gpu):
    """Scores that rise along the keys, and a NaN in V: the NaN reaches its dim
    of its KV head's query heads only."""
    Hq, Hkv, L = 16, 4, 1500
    (q, k, v), d = inputs(L, Hq, Hkv, Hkv * D, 2, gpu)
    k[:L] = (k[:L] * np.linspace(0.1, 8.0, L)[:, None]).astype(np.float16)
    v[700, 2 * D + 5] = np.nan
    d[1], d[2] = (torch.from_numpy(x).to(gpu) for x in (k, v))
    got = decode(attn, d, L, Hq, Hkv, Hkv * D, gpu).reshape(Hq, D)
    ref = generic(attn, d, L, Hq, Hkv, Hkv * D, gpu).reshape(Hq, D)
    where = np.isnan(got)
    assert np.array_equal(where, np.isnan(ref)) and where[8:12, 5].all() and where.sum() == 4
    assert_as_generic(np.where(where, 0, got), np.where(where, 0, ref), np.nan_to_num(v[:L]))


def captured(attn, d, out, ws, L, Hq, Hkv, stride):
    """One captured call of L keys: graph, executable graph, its last node, its
    number of kernels."""
    import ctypes
    stream = torch.cuda.Stream()
    sp = stream.cuda_stream
    torch.cuda.synchronize()
    hipgraph.begin_capture(sp)
    attn.decode(*d, out, *ws, 1, L, L - 1, Hq, Hkv, D, 0, stride, stream=sp)
    node = hipgraph.last_captured_node(sp)
    graph, exe = hipgraph.end_capture(sp)
    n = ctypes.c_size_t()
    assert hipgraph._hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    return stream, graph, exe, node, n.value


@pytest.mark.parametrize("Hq,Hkv,least", [(8, 8, 64), (4, 2, 64), (6, 2, 104), (16, 4, 104),
                                          (16, 2, 192), (12, 1, 192)])
def test_decode_d64_from_where_it_is_faster(attn, gpu, Hq, Hkv, least):
    """The shortest context of the two kernels; below it the one generic kernel runs,
    bit for bit."""
    (q, k, v), d = inputs(least, Hq, Hkv, Hkv * D, 6, gpu)
    ws, _ = workspace(attn, Hq, least, gpu)
    out = torch.zeros(Hq * D, dtype=torch.float16, device=gpu)
    for L, kernels in ((1, 1), (least - 1, 1), (least, 2)):
        print(f"[case] decode d64 route Hq={Hq} Hkv={Hkv} L={L}", flush=True)
        stream, graph, exe, _, n = captured(attn, d, out, ws, L, Hq, Hkv, Hkv * D)
        hipgraph.destroy(graph, exe)
        assert n == kernels, (L, n)
        if kernels == 1:
            got, ref = (f(attn, d, L, Hq, Hkv, Hkv * D, gpu) for f in (decode, generic))
            assert np.array_equal(got.view(np.uint16), ref.view(np.uint16))


# contexts below those, through a captured pair moved to them
@pytest.mark.parametrize("Hq,Hkv,pad", [(16, 4, 0), (8, 8, 0), (4, 2, 8), (6, 2, 0), (16, 2, 0),
                                        (12, 1, 24)])
def test_decode_d64_short_contexts_of_a_patched_pair(attn, gpu, Hq, Hkv, pad):
    stride, L0 = Hkv * D + pad, 1000
    (q, k, v), d = inputs(L0, Hq, Hkv, stride, 7, gpu)
    ws, _ = workspace(attn, Hq, L0, gpu)
    out = torch.zeros(Hq * D, dtype=torch.float16, device=gpu)
    stream, graph, exe, node, n = captured(attn, d, out, ws, L0, Hq, Hkv, stride)
    assert n == 2
    try:
        for L in (1, 7, 12, 31, 64, 65, 127, L0):
            print(f"[case] decode d64 patched Hq={Hq} Hkv={Hkv} L={L}", flush=True)
            assert attn.lib().attn_update_decode_node(exe, node, L) == 0
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            hipgraph.launch(exe, stream.cuda_stream)
            hipgraph.synchronize(stream.cuda_stream)
            assert_as_generic(out.cpu().numpy(), generic(attn, d, L, Hq, Hkv, stride, gpu), v[:L])
    finally:
        hipgraph.destroy(graph, exe)


@pytest.mark.parametrize("updater", ["decode", "merge", "split"])
def test_decode_d64_captured_and_patched(attn, gpu, updater):
    """A captured call replays as the eager one; a node of it moves to other
    contexts (shorter and longer, within the capturing call's states)."""
    Hq, Hkv, L0 = 16, 4, 3000
    (q, k, v), d = inputs(8000, Hq, Hkv, Hkv * D, 4, gpu)
    ws, _ = workspace(attn, Hq, 8000, gpu)
    out = torch.zeros(Hq * D, dtype=torch.float16, device=gpu)
    stream = torch.cuda.Stream()
    sp = stream.cuda_stream
    torch.cuda.synchronize()
    hipgraph.begin_capture(sp)
    attn.decode(*d, out, *ws, 1, L0, L0 - 1, Hq, Hkv, D, 0, 0, stream=sp)
    node = hipgraph.last_captured_node(sp)
    graph, exe = hipgraph.end_capture(sp)
    lib = attn.lib()
    if updater == "split":
        import ctypes
        hip = hipgraph._hip
        near, n = (ctypes.c_void_p * 4)(), ctypes.c_size_t(4)
        hip.hipGraphNodeGetDependencies.argtypes = [ctypes.c_void_p, ctypes.c_void_p,
                                                    ctypes.c_void_p]
        assert hip.hipGraphNodeGetDependencies(node, near, ctypes.byref(n)) == 0 and n.value == 1
        node = near[0]
    patch = lib.attn_update_merge_node if updater == "merge" else lib.attn_update_decode_node
    try:
        for L in (L0, 100, 1, 2999, 8000, 64, L0):
            assert patch(exe, node, L) == 0, L
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            hipgraph.launch(exe, sp)
            hipgraph.synchronize(sp)
            got = out.cpu().numpy()
            assert_as_generic(got, generic(attn, d, L, Hq, Hkv, Hkv * D, gpu), v[:L])
        assert patch(exe, node, 0) != 0
    finally:
        hipgraph.destroy(graph, exe)
