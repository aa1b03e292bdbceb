"""Performance cases of the fused-MoE operator: what a serving or evaluation
program calls, over the range of batch sizes, layer shapes, weight formats and
entry points the package supports.

A case is a dict of plain values:
  op       "fused"   fused_moe from given router logits
           "layer"   fused_moe from hidden states: router GEMM, routed experts
                     and an always-on shared expert in one call
           "routed"  fused_moe_routed: one expert-parallel rank's experts on
                     the token rows and routing that a dispatch delivered
           "rows"    run_kernel: rows already grouped and padded by expert
  fmt      "fp16", "int8" or "fp8" expert weights
  tokens, hidden, inter, experts, top_k     the layer ("routed": `experts`
           routed in all, `local` of them held here; "rows": `tokens` valid
           rows, of which `high` experts share what the others' `low` rows
           each leave)
  bias     "none", "normal" or "zipf": the expert bias added to the logits
"""
from __future__ import annotations

import math

import torch

import muxi_race_amd as moe

# (hidden, inter, experts, top_k): the layers of this repository's benchmark
DSV3 = (7168, 2048, 256, 8)
MIXTRAL = (4096, 14336, 8, 2)
MID = (7168, 2048, 64, 6)
SMALL = (1024, 512, 8, 2)
# (experts, hidden, inter, valid rows, high experts, low rows): run_kernel's published cases
ROWS = ((16, 2048, 8192, 2272, 8, 124), (32, 7168, 2048, 4544, 22, 112), (64, 7168, 2048, 9088, 23, 127))


def _layer(op, fmt, tokens, shape, bias="none", **more):
    h, i, e, k = shape
    return dict(op=op, fmt=fmt, tokens=tokens, hidden=h, inter=i, experts=e, top_k=k, bias=bias, **more)


def _rows(which):
    e, h, i, valid, high, low = ROWS[which]
    return dict(op="rows", fmt="fp16", tokens=valid, hidden=h, inter=i, experts=e, top_k=1, bias="none",
                high=high, low=low)


def listed():
    return [
        # a small model's layer at a modest batch: launches and latency
        dict(_layer("fused", "fp16", 128, SMALL), name="small_128"),
        # one user's next token through the large layer: eight experts read once
        dict(_layer("fused", "fp16", 1, DSV3), name="large_1"),
        # a decode batch whose tokens share popular experts
        dict(_layer("fused", "fp16", 32, DSV3, "zipf"), name="large_32_zipf"),
        # a whole layer from hidden states: a large decode batch or one chunk of a prompt
        dict(_layer("layer", "fp16", 601, DSV3), name="layer_601"),
        # a prompt's prefill through the large layer (the headline benchmark)
        dict(_layer("fused", "fp16", 4096, DSV3, "normal"), name="large_4096"),
        # a prompt's prefill through few wide experts: the matrix-core end of the range
        dict(_layer("fused", "fp16", 2048, MIXTRAL), name="wide_2048"),
        # decode on 8-bit weights, both formats: the reason a server quantises
        dict(_layer("fused", "int8", 24, MID), name="int8_24"),
        dict(_layer("fused", "fp8", 129, MID), name="fp8_129"),
        # prefill on 8-bit weights
        dict(_layer("fused", "int8", 2048, MID), name="int8_2048"),
        dict(_layer("fused", "fp8", 2048, MID), name="fp8_2048"),
        # one of eight expert-parallel ranks, on the rows that a dispatch delivered to it
        dict(_layer("routed", "fp16", 777, DSV3, local=32), name="rank_777"),
        # the pre-grouped operator on its second published case
        dict(_rows(1), name="rows_4544"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("fused", "fused", "int8", "fp8", "layer", "routed", "rows"))
    if kind == "rows":
        e, h, i, _, _, _ = rng.choice(ROWS)
        high, low = rng.randint(1, e - 1), rng.randint(1, 128)
        valid = (e - high) * low + high * rng.randint(1, 380)
        return dict(op="rows", fmt="fp16", tokens=valid, hidden=h, inter=i, experts=e, top_k=1, bias="none",
                    high=high, low=low)
    if kind == "fused":
        shape = rng.choice((DSV3, MIXTRAL, MID, SMALL))
        return _layer("fused", "fp16", _log_int(rng, 1, 4096), shape, rng.choice(("none", "normal", "zipf")))
    if kind in ("int8", "fp8"):
        shape = rng.choice((MID, MID, MIXTRAL, SMALL))
        return _layer("fused", kind, _log_int(rng, 1, 4096), shape, rng.choice(("none", "normal")))
    if kind == "layer":
        return _layer("layer", "fp16", _log_int(rng, 1, 2048), rng.choice((DSV3, MID)), rng.choice(("none", "normal")))
    return _layer("routed", "fp16", _log_int(rng, 16, 4096), DSV3, local=rng.choice((16, 32, 64)))


def _group_sizes(c):
    """`low` rows for each expert but `high`, which share the rest evenly; interleaved."""
    sizes = [c["low"]] * (c["experts"] - c["high"])
    rest = c["tokens"] - sum(sizes)
    q, r = divmod(rest, c["high"])
    sizes += [q + (i < r) for i in range(c["high"])]
    return sizes[::2] + sizes[1::2]


def _held(c):
    """Experts whose weights this program holds."""
    return c["local"] if c["op"] == "routed" else c["experts"]


def _normal(shape, std, gen, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _quantised(w, fmt):
    """Symmetric 8-bit codes and fp32 scales of each row of w [E, N, K], expert by expert."""
    q = torch.empty(w.shape, dtype=torch.int8 if fmt == "int8" else torch.float8_e4m3fn, device=w.device)
    s = torch.empty(w.shape[:-1], dtype=torch.float32, device=w.device)
    top = 127.0 if fmt == "int8" else 448.0
    for lo in range(0, w.shape[0], 8):
        f = w[lo:lo + 8].float()
        amax = f.abs().amax(-1, keepdim=True).clamp_min(1e-20)
        s[lo:lo + 8] = (amax / top)[..., 0]
        f = (f * (top / amax)).clamp_(-top, top)
        q[lo:lo + 8] = f.round_().to(torch.int8) if fmt == "int8" else f.to(torch.float8_e4m3fn)
    return q, s


def _bias(c, gen):
    if c["bias"] == "normal":
        return _normal((c["experts"],), 0.5, gen, torch.float32)
    if c["bias"] == "zipf":  # expert popularity falls with the index
        return -1.2 * torch.log(torch.arange(c["experts"], dtype=torch.float32, device="cuda") + 1.0)
    return None


def _top_k(logits, bias, k):
    """(ids, weights) of the k largest logits, softmax renormalised over them, in the logits' precision."""
    v = logits if bias is None else logits + bias.to(logits.dtype)
    top, ids = v.topk(k, dim=-1)
    return ids, torch.softmax(top, dim=-1)


def prepare(case, seed):
    """Activations as a norm leaves them (N(0, 1)), weights N(0, 0.02), routing from N(0, 1) logits."""
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T, H, I, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"]
    El = _held(c)
    st = dict(case=c)
    w = [_normal(shape, 0.02, gen) for shape in ((El, I, H), (El, I, H), (El, H, I))]
    if c["fmt"] == "fp16":
        st["w"] = w
    else:
        parts = []
        while w:
            parts += _quantised(w.pop(0), c["fmt"])
        st["w"] = parts
        st["w8a8"] = moe.W8A8Weights(*parts)
    if c["op"] == "rows":
        sizes = _group_sizes(c)
        padded = [(n + 127) // 128 * 128 for n in sizes]
        i32 = dict(dtype=torch.int32, device="cuda")
        st["sizes"], st["starts"] = sizes, [sum(padded[:e]) for e in range(E)]
        st["gs"] = torch.tensor(sizes, **i32)
        st["go"] = torch.tensor([sum(sizes[:e]) for e in range(E + 1)], **i32)
        st["gpo"] = torch.tensor([sum(padded[:e]) for e in range(E + 1)], **i32)
        st["gidx"] = torch.tensor([e for e in range(E) for _ in range(padded[e] // 128)], **i32)
        st["x"] = _normal((sum(padded), H), 1.0, gen)
        st["routed"] = torch.rand((T,), generator=gen, device="cuda")
        st["out"] = torch.empty_like(st["x"])
        return st
    st["x"] = _normal((T, H), 1.0, gen)
    st["bias"] = _bias(c, gen)
    if c["op"] == "layer":
        st["router"] = _normal((E, H), 0.02, gen)
        st["shared"] = tuple(_normal(shape, 0.02, gen) for shape in ((I, H), (I, H), (H, I)))
    else:
        st["logits"] = _normal((T, E), 1.0, gen, torch.float32)
    if c["op"] == "routed":
        # a dispatch sends a token to this rank if at least one choice lies here:
        # one choice of every row is moved into the range
        ids, wts = _top_k(st["logits"], None, k)
        there = (ids < El).any(-1)
        own = torch.randint(0, El, (T,), generator=gen, device="cuda")
        ids[:, 0] = torch.where(there, ids[:, 0], own)
        st["ids"], st["wts"] = ids.to(torch.int32).contiguous(), wts.contiguous()
    return st


def run(state):
    c, w = state["case"], state["w"]
    if c["op"] == "rows":
        moe.run_kernel(state["x"], *w, state["routed"], state["gs"], state["go"], state["gpo"], state["gidx"], state["out"])
        return state["out"]
    if c["op"] == "routed":
        return moe.fused_moe_routed(state["x"], state["ids"], state["wts"], *w, num_experts=c["experts"])
    if c["op"] == "layer":
        return moe.fused_moe(state["x"], None, *w, c["top_k"], expert_bias=state["bias"],
                             router_weight=state["router"], shared_expert=state["shared"])
    if c["fmt"] != "fp16":
        return moe.fused_moe(state["x"], state["logits"], None, None, None, c["top_k"], expert_bias=state["bias"],
                             w8a8=state["w8a8"])
    return moe.fused_moe(state["x"], state["logits"], *w, c["top_k"], expert_bias=state["bias"])


def _mlp64(x, wg, wu, wd):
    g = x @ wg.T
    return (g * torch.sigmoid(g) * (x @ wu.T)) @ wd.T


def exact(case, seed):
    """The layer in float64 from the same inputs; 8-bit weights dequantised, activations not quantised."""
    c, st = case, prepare(case, seed)
    El = _held(c)

    def weight(j, e):
        if c["fmt"] == "fp16":
            return st["w"][j][e].double()
        return st["w"][2 * j][e].to(torch.float32).double() * st["w"][2 * j + 1][e].double()[:, None]

    x = st["x"].double()
    out = torch.zeros_like(x)
    if c["op"] == "rows":
        first = 0
        for e, (n, start) in enumerate(zip(st["sizes"], st["starts"])):
            if n:
                y = _mlp64(x[start:start + n], *(weight(j, e) for j in range(3)))
                out[start:start + n] = y * st["routed"][first:first + n].double()[:, None]
            first += n
        return out
    if c["op"] == "routed":
        ids, wts = st["ids"], st["wts"].double()
    elif c["op"] == "layer":
        ids, wts = _top_k(x @ st["router"].double().T, st["bias"], c["top_k"])
    else:
        ids, _ = _top_k(st["logits"], st["bias"], c["top_k"])  # the choice is made in the logits' fp32
        v = st["logits"].double() if st["bias"] is None else (st["logits"] + st["bias"]).double()
        wts = torch.softmax(v.gather(1, ids.long()), dim=-1)
    for e in range(El):
        t, j = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            out.index_add_(0, t, _mlp64(x[t], *(weight(m, e) for m in range(3))) * wts[t, j][:, None])
    if c["op"] == "layer":
        out += _mlp64(x, *(m.double() for m in st["shared"]))
    return out


def _touched(c):
    """(experts read, routed rows) of one pass: counted on a sample routing of the case's kind."""
    T, E, k = c["tokens"], c["experts"], c["top_k"]
    gen = torch.Generator().manual_seed(1)
    logits = torch.randn((T, E), generator=gen)
    if c["bias"] == "normal":
        logits += 0.5 * torch.randn((E,), generator=gen)
    elif c["bias"] == "zipf":
        logits -= 1.2 * torch.log(torch.arange(E, dtype=torch.float32) + 1.0)
    ids = logits.topk(k, dim=-1).indices
    if c["op"] != "routed":
        return ids.unique().numel(), T * k
    here = ids < c["local"]
    # every row has at least one choice here
    rows = int(here.sum()) + int((~here.any(-1)).sum())
    return min(c["local"], rows), rows


def work(case):
    c = case
    T, H, I, E, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"]
    wb = 2 if c["fmt"] == "fp16" else 1
    if c["op"] == "rows":
        sizes = _group_sizes(c)
        experts, rows = sum(n > 0 for n in sizes), T
        io = 2 * T * H + 2 * H * sum((n + 127) // 128 * 128 for n in sizes) + 4 * T
    else:
        experts, rows = _touched(c)
        io = 4 * T * H + (8 * T * k if c["op"] == "routed" else 4 * T * E)
    flops, data = 6.0 * rows * H * I, experts * 3 * H * I * wb
    if wb == 1:
        data += experts * 4 * (2 * I + H)
    if c["op"] == "layer":
        flops += 6.0 * T * H * I + 2.0 * T * H * E
        data += 3 * H * I * 2 + E * H * 2
        io -= 4 * T * E  # no logits are given
    return {"bytes": float(data + io), "flops": flops}


def tolerance(case):
    # fp16: the intermediate and each choice's row are rounded to fp16 (2^-11), so
    # sums in another order move a result by about 2e-4.  From hidden states a
    # near-tie of two experts may also fall the other way in one token.  8-bit: an
    # activation's code at a rounding tie may fall the other way.
    if case["fmt"] != "fp16":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 4e-3, "max": 0.5} if case["op"] == "layer" else {"rel": 1e-3, "max": 0.02}
