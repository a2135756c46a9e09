"""Workloads of the attention path, one pass each through the Python binding.

Two kinds, both over the layers of a model whose hidden size is 2048:

* "prompt": the attention path of a prompt of `tokens` tokens, per layer the
  QKV projection, RoPE + KV-cache append and causal attention; `fused` folds
  RoPE and append into the projection (two calls per layer instead of three).
  Prompts short enough to be launch-bound run all `layers` layers from one
  captured graph, longer ones call one layer directly.
* "decode": the attention path of one token at context length `context`, all
  layers from one captured graph, as the engine decodes: QKV projection, RoPE +
  append, Flash-Decode and the output projection added to the hidden state.
  `form` says which launches are folded: "plain" (none), "qkv" (RoPE + append
  into the projection) or "attention" (RoPE + append into the decode).

Every fourth layer takes no rotation (NoPE), as in the model.  Every layer has
weights, activations and cache rows of its own.
"""
import math
import pathlib
import sys

import torch

HIDDEN = 2048
THETA = 5.0e6
# (query heads, KV heads, head dim): the model's own, then other grouped-query,
# multi-head and 64-dim layouts
MODEL = (16, 4, 128)
OTHERS = ((16, 8, 128), (16, 16, 128), (8, 2, 128), (16, 4, 64), (8, 8, 64), (32, 8, 64))


def _binding():
    path = str(pathlib.Path.cwd() / "llm-inference_amd" / "python")
    if path not in sys.path:
        sys.path.insert(0, path)
    import attn_mi355x
    return attn_mi355x


def _case(kind, layout, **more):
    heads, kv_heads, head_dim = layout
    return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, **more}


def _prompt(layout, tokens, layers, fused):
    return _case("prompt", layout, tokens=tokens, layers=layers, fused=fused)


def _decode(layout, context, layers, form):
    return _case("decode", layout, context=context, layers=layers, form=form)


def listed():
    return [
        # a one-line question: every launch is latency
        {"name": "prompt_24", **_prompt(MODEL, 24, 36, True)},
        # a paragraph, the length the reference's tests use, on its own three launches
        {"name": "prompt_254", **_prompt(MODEL, 254, 36, False)},
        # a page of text or a chat with some history, odd length
        {"name": "prompt_999", **_prompt(MODEL, 999, 1, True)},
        # a few pages, ragged against every tile
        {"name": "prompt_2500", **_prompt(MODEL, 2500, 1, False)},
        # a long document chunk just past a power of two
        {"name": "prompt_4100", **_prompt(MODEL, 4100, 1, True)},
        # the benchmark's long prompt
        {"name": "prompt_8192", **_prompt(MODEL, 8192, 1, False)},
        # one token of a short chat
        {"name": "decode_254", **_decode(MODEL, 254, 36, "plain")},
        # one token of a longer conversation, RoPE + append folded into the decode
        {"name": "decode_4001", **_decode(MODEL, 4001, 36, "attention")},
        # one token over a long document: the benchmark's headline length
        {"name": "decode_32768", **_decode(MODEL, 32768, 36, "qkv")},
        # a multi-head layout (no grouping): a page of text
        {"name": "prompt_mha_1000", **_prompt((16, 16, 128), 1000, 1, False)},
        # 64-dim heads, grouped: a page and a half of text
        {"name": "prompt_d64_1500", **_prompt((16, 4, 64), 1500, 1, False)},
        # 64-dim heads: one token of a longer conversation
        {"name": "decode_d64_3000", **_decode((16, 4, 64), 3000, 12, "plain")},
    ]


def _between(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("prompt", "prompt", "decode"))
    if rng.random() < 0.3:
        layout = rng.choice(OTHERS)
        if kind == "prompt":
            return _prompt(layout, _between(rng, 100, 1500), 1, rng.random() < 0.5)
        return _decode(layout, _between(rng, 100, 4096), 12, rng.choice(("plain", "qkv", "attention")))
    if kind == "prompt":
        tokens = _between(rng, 8, 8192)
        return _prompt(MODEL, tokens, 36 if tokens <= 320 else 1, rng.random() < 0.5)
    return _decode(MODEL, _between(rng, 100, 32768), 36, rng.choice(("plain", "qkv", "attention")))


def _dims(case):
    q_dim = case["heads"] * case["head_dim"]
    kv_dim = case["kv_heads"] * case["head_dim"]
    return q_dim, kv_dim, q_dim + 2 * kv_dim


def _rotates(layer):
    return layer % 4 != 3


def _tables(rows, head_dim):
    """fp16 cos/sin [rows, head_dim / 2], angles in 32 bits as the engine makes them."""
    half = head_dim // 2
    exponent = torch.arange(half, dtype=torch.float32) * 2 / head_dim
    angle = torch.arange(rows, dtype=torch.float32)[:, None] / torch.pow(THETA, exponent)[None]
    return angle.cos().half(), angle.sin().half()


def _inputs(case, seed):
    """The inputs of a case, from the seed alone: normalised hidden states,
    weights that keep their variance, a cache of unit-variance keys and values."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(*shape, sigma=1.0):
        return torch.empty(*shape, dtype=torch.float16, device="cuda").normal_(0.0, sigma, generator=gen)

    q_dim, kv_dim, total = _dims(case)
    layers = case["layers"]
    rows = case["tokens"] if case["kind"] == "prompt" else case["context"]
    cos, sin = _tables(rows, case["head_dim"])
    t = {"cos": cos.cuda(), "sin": sin.cuda(),
         "w_qkv": normal(layers, total, HIDDEN, sigma=HIDDEN ** -0.5)}
    if case["kind"] == "prompt":
        t["x"] = normal(layers, rows, HIDDEN)
        t["cache"] = torch.zeros(layers, 2, rows, kv_dim, dtype=torch.float16, device="cuda")
    else:
        t["x"] = normal(layers, HIDDEN)
        t["w_o"] = normal(layers, HIDDEN, q_dim, sigma=q_dim ** -0.5)
        t["residual"] = normal(layers, HIDDEN)
        t["cache"] = normal(layers, 2, rows, kv_dim)
    return t


class _State:
    def __init__(self, case, seed):
        self.A = _binding()
        self.case = case
        self.t = _inputs(case, seed)
        q_dim, kv_dim, total = _dims(case)
        layers = case["layers"]

        def empty(*shape):
            return torch.zeros(*shape, dtype=torch.float16, device="cuda")

        if case["kind"] == "prompt":
            self.qkv = empty(layers, case["tokens"], total)
            self.out = empty(layers, case["tokens"], q_dim)
            self.enqueue = self._prompt
        else:
            self.qkv = empty(layers, total)
            self.out = empty(layers, q_dim)
            self.hidden = empty(layers, HIDDEN)
            self.partials = self.A.decode_workspace(case["heads"], case["context"], case["head_dim"])
            self.enqueue = self._decode
        self.graph = None
        if layers > 1:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                self.enqueue()
                side.synchronize()
                self.graph = torch.cuda.CUDAGraph()
                self.graph.capture_begin(capture_error_mode="relaxed")
                self.enqueue()
                self.graph.capture_end()
            torch.cuda.current_stream().wait_stream(side)

    def _prompt(self):
        A, c, t = self.A, self.case, self.t
        heads, kv_heads, head_dim, n = c["heads"], c["kv_heads"], c["head_dim"], c["tokens"]
        q_dim, kv_dim, total = _dims(c)
        for layer in range(c["layers"]):
            k_cache, v_cache = t["cache"][layer]
            x, w, y, rotate = t["x"][layer], t["w_qkv"][layer], self.qkv[layer], _rotates(layer)
            if c["fused"]:
                A.qkv_gemm_rope_store_kv(x, y, w, k_cache, v_cache, t["cos"], t["sin"], n, HIDDEN,
                                         heads, kv_heads, head_dim, 0, rotate)
            else:
                at = y.data_ptr()
                A.qkv_gemm(x, y, w, n, HIDDEN, total)
                A.rope_store_kv(at, at + 2 * q_dim, at + 2 * (q_dim + kv_dim), k_cache, v_cache,
                                t["cos"], t["sin"], n, heads, kv_heads, head_dim, total, total, 0,
                                rotate)
            A.prefill(y, k_cache, v_cache, self.out[layer], n, heads, kv_heads, head_dim, total,
                      kv_dim)

    def _decode(self):
        A, c, t = self.A, self.case, self.t
        heads, kv_heads, head_dim, length = c["heads"], c["kv_heads"], c["head_dim"], c["context"]
        q_dim, kv_dim, total = _dims(c)
        row = length - 1
        for layer in range(c["layers"]):
            k_cache, v_cache = t["cache"][layer]
            x, w, y, rotate = t["x"][layer], t["w_qkv"][layer], self.qkv[layer], _rotates(layer)
            at = y.data_ptr()
            q, k, v = at, at + 2 * q_dim, at + 2 * (q_dim + kv_dim)
            if c["form"] == "qkv":
                A.qkv_rope_store_kv_decode(x, y, w, k_cache, v_cache, t["cos"], t["sin"], HIDDEN,
                                           heads, kv_heads, head_dim, row, rotate)
            else:
                A.qkv_decode(x, y, w, HIDDEN, total)
            if c["form"] == "attention":
                A.rope_store_kv_decode(q, k, v, k_cache, v_cache, t["cos"], t["sin"],
                                       self.out[layer], *self.partials, length, row, heads,
                                       kv_heads, head_dim, rotate, kv_dim)
            else:
                if c["form"] == "plain":
                    A.rope_store_kv(q, k, v, k_cache, v_cache, t["cos"], t["sin"], 1, heads,
                                    kv_heads, head_dim, total, total, row, rotate)
                A.decode(q, k_cache, v_cache, self.out[layer], *self.partials, 1, length, row,
                         heads, kv_heads, head_dim, 0, kv_dim)
            A.out_proj_decode(self.out[layer], self.hidden[layer], t["w_o"][layer], HIDDEN, heads,
                              head_dim, 1.0)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    if state.case["kind"] == "decode":
        # the layers add to the hidden states that the blocks before them left
        state.hidden.copy_(state.t["residual"])
    if state.graph is not None:
        state.graph.replay()
    else:
        state.enqueue()
    result = {"qkv": state.qkv, "cache": state.t["cache"], "out": state.out}
    if state.case["kind"] == "decode":
        result["hidden"] = state.hidden
    return result


def work(case):
    q_dim, kv_dim, total = _dims(case)
    layers, heads, head_dim = case["layers"], case["heads"], case["head_dim"]
    if case["kind"] == "prompt":
        n = case["tokens"]
        # x and the weights read; Q/K/V, the cache rows and the output written; the tables once
        values = n * HIDDEN + total * HIDDEN + n * (total + 2 * kv_dim + q_dim)
        flops = 2 * n * HIDDEN * total + 4 * head_dim * heads * (n * (n + 1) // 2)
        tables = n * head_dim
    else:
        length = case["context"]
        # both weights, x, the residual and the cached rows read; Q/K/V, the
        # new rows, the output and the hidden state written
        values = (HIDDEN * (total + q_dim) + 3 * HIDDEN + 2 * kv_dim * length + total + q_dim)
        flops = 2 * HIDDEN * (total + q_dim) + 4 * head_dim * heads * length
        tables = head_dim
    return {"bytes": 2 * (layers * values + tables), "flops": layers * flops}


def tolerance(case):
    # fp16 outputs of 32-bit sums; attention weights rounded to fp16
    return {"rel": 2e-3, "max": 4e-2}


def exact(case, seed):
    t = _inputs(case, seed)
    heads, kv_heads, head_dim = case["heads"], case["kv_heads"], case["head_dim"]
    q_dim, kv_dim, total = _dims(case)
    half, group, layers = head_dim // 2, heads // kv_heads, case["layers"]
    prompt = case["kind"] == "prompt"
    n = case["tokens"] if prompt else 1
    first = 0 if prompt else case["context"] - 1
    cos = t["cos"][first:first + n].double()[:, None]
    sin = t["sin"][first:first + n].double()[:, None]

    def rotated(v):
        v = v.view(n, -1, head_dim)
        a, b = v[..., :half], v[..., half:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1).reshape(n, -1)

    def new(*shape):
        return torch.empty(*shape, dtype=torch.float64, device="cuda")

    cache = t["cache"].double()
    qkv, out, hidden = new(layers, n, total), new(layers, n, q_dim), new(layers, HIDDEN)
    for layer in range(layers):
        y = t["x"][layer].double().view(n, HIDDEN) @ t["w_qkv"][layer].double().t()
        q, k, v = y.split((q_dim, kv_dim, kv_dim), 1)
        q, k = q.contiguous(), k.contiguous()
        k_new = k
        if _rotates(layer):
            # only the cache's keys are rotated; Q is rotated in place.  The
            # three-launch and the folded forms leave K and V as projected
            q, k_new = rotated(q), rotated(k)
        cache[layer, 0, first:first + n] = k_new
        cache[layer, 1, first:first + n] = v
        qkv[layer] = torch.cat((q, k, v), 1)
        keys, values = cache[layer]
        for head in range(heads):
            g = head // group
            one = slice(head * head_dim, (head + 1) * head_dim)
            kv = slice(g * head_dim, (g + 1) * head_dim)
            s = q[:, one] @ keys[:, kv].t().contiguous() / math.sqrt(head_dim)
            if prompt:
                s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
            out[layer][:, one] = torch.softmax(s, 1) @ values[:, kv].contiguous()
        if not prompt:
            hidden[layer] = t["residual"][layer].double() + t["w_o"][layer].double() @ out[layer, 0]
    if prompt:
        return {"qkv": qkv, "cache": cache, "out": out}
    return {"qkv": qkv[:, 0], "cache": cache, "out": out[:, 0], "hidden": hidden}
