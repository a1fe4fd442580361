"""Performance cases: the calls a program makes on this library, at the
shapes it makes them.

A MoE engine calls the library for one token at a time (decode: bound
experts, whole layer chains, the LM head), for a few tokens at once
(multi-token decode, a dense matmul that verifies a draft) and for a prompt
chunk (router, grouped experts, the whole MoE block, projections). The
listed cases hold each of these once, at the model shapes the tests and the
benchmark use; `draw` spreads over the same ranges.

Inputs have the distributions the layers see: codes uniform, scales
bf16 |N(0, .02)|, biases bf16 N(0, .01), router and gate N(0, .02),
normalised hidden rows N(0, 1), Zipf(1.1) expert popularity.
"""
import math

import torch

import streamoe_amd as sa

DEV = "cuda:0"
EPS = 1e-6

# name: hidden, inter, experts, top-k, renormalised top-k, shared expert.
MODELS = {
    "a3b": (2048, 512, 256, 8, True, True),
    "olmoe": (2048, 1024, 64, 8, False, False),
    "flash-next": (2560, 640, 512, 10, True, True),
    "h4096": (4096, 1024, 512, 10, True, True),
    "cogito": (7168, 2048, 256, 8, True, True),
}


def listed():
    return [
        # The engine's per-token expert dispatch with the routing on the
        # host: eight bound blobs, one call, the smallest unit of work.
        dict(name="experts_a3b", kind="experts", model="a3b", k=8, bits=4, shared=True),
        # One token through the 40 MoE blocks of the A3B model, replayed
        # from a HIP graph: the decode loop itself.
        dict(name="decode_a3b_40", kind="decode", model="a3b", layers=40, bits=4, tokens=1),
        # Four tokens at once through packed 3-bit layers (speculative or
        # batched decode).
        dict(name="decode_a3b_3bit_t4", kind="decode", model="a3b", layers=16, bits=3, tokens=4),
        # Decode at widths that are not a power of two, 512 experts, top-10.
        dict(name="decode_flash_next", kind="decode", model="flash-next", layers=8, bits=4, tokens=1),
        # The LM head with the greedy pick, once per decoded token.
        dict(name="lm_head", kind="lm_head", out_dim=151936, in_dim=2048),
        # The LM head over a few positions (draft verification, prompt
        # scoring): a wide matrix, few rows.
        dict(name="qmm_vocab_16", kind="qmm", n=16, out_dim=151936, in_dim=2048, bits=4, group=64),
        # A dense projection over a prompt chunk with a ragged tail.
        dict(name="qmm_proj", kind="qmm", n=500, out_dim=4096, in_dim=2048, bits=4, group=64),
        # The router of a prompt chunk: logits, softmax, top-k.
        dict(name="router_512", kind="router", model="a3b", n=512),
        # The MoE block of a prompt chunk (routed and shared experts, gate,
        # residual).
        dict(name="prefill_a3b_block", kind="block", model="a3b", n=512, bits=4, x="bf16"),
        # A short prompt through packed 3-bit experts, f32 hidden rows.
        dict(name="prefill_a3b_short", kind="prefill", model="a3b", n=37, bits=3, x="f32"),
        # The largest prompt chunk through the largest resident layer.
        dict(name="prefill_h4096", kind="prefill", model="h4096", n=1000, bits=4, x="bf16"),
        # A prompt chunk at the widths that are not multiples of 256.
        dict(name="prefill_flash_next", kind="prefill", model="flash-next", n=512, bits=4, x="bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["experts", "decode", "decode", "lm_head", "qmm", "qmm", "router", "block", "prefill", "prefill"])
    if kind == "experts":
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), k=rng.randint(1, 10), bits=rng.choice([3, 4]),
                    shared=rng.random() < 0.7)
    if kind == "decode":
        model = rng.choice(["a3b", "olmoe", "flash-next", "h4096"])
        most = {"a3b": 40, "olmoe": 40, "flash-next": 16, "h4096": 6}[model]
        return dict(kind=kind, model=model, layers=_log_int(rng, 1, most), bits=rng.choice([3, 4]),
                    tokens=rng.choice([1, 1, 2, 3, 4]), k=rng.randint(2, 10))
    if kind == "lm_head":
        return dict(kind=kind, out_dim=_log_int(rng, 500, 151936), in_dim=rng.choice([2048, 2560, 4096]))
    if kind == "qmm":
        out_dim, in_dim = rng.choice([(512, 2048), (2048, 512), (4096, 2048), (640, 2560), (2560, 640), (1024, 4096),
                                      (4096, 1024), (_log_int(rng, 1000, 151936), 2048)])
        most = 64 if out_dim > 16384 else 1024
        return dict(kind=kind, n=_log_int(rng, 2, most), out_dim=out_dim, in_dim=in_dim, bits=rng.choice([3, 4]),
                    group=rng.choice([32, 64, 128]))
    if kind == "router":
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), n=_log_int(rng, 1, 1024), k=rng.randint(2, 10))
    model = rng.choice(["a3b", "olmoe", "h4096"] if kind == "block" else ["a3b", "olmoe", "h4096", "flash-next"])
    return dict(kind=kind, model=model, n=_log_int(rng, 2, 512 if model == "flash-next" else 1000),
                bits=rng.choice([3, 4]), x=rng.choice(["bf16", "f32"]), k=rng.randint(2, 10))


def _model(case):
    """The case's model, with its own top-k where the case names one."""
    H, I, E, k, norm, shared = MODELS[case["model"]]
    return H, I, E, case.get("k", k), norm, shared


# -- inputs ------------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + salt) % (1 << 62))


def _normal(g, *shape, sigma=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * sigma


def _matrices(g, count, rows, cols, bits, group):
    """`count` packed matrices, each [codes | bf16 scales | bf16 biases], as
    bytes [count, size]."""
    codes = rows * cols * bits // 8
    sb = rows * (cols // group) * 2
    buf = torch.empty((count, codes + 2 * sb), dtype=torch.uint8, device=DEV)
    buf[:, :codes] = torch.randint(0, 256, (count, codes), generator=g, device=DEV, dtype=torch.uint8)
    s = _normal(g, count, sb // 2, sigma=0.02).abs_().to(torch.bfloat16)
    buf[:, codes:codes + sb] = s.view(torch.uint8).view(count, sb)
    b = _normal(g, count, sb // 2, sigma=0.01).to(torch.bfloat16)
    buf[:, codes + sb:] = b.view(torch.uint8).view(count, sb)
    return buf


def _experts(g, count, hidden, inter, bits, group=64):
    """Expert blobs [gate | up | down] as bytes [count, size]. The three
    blocks have the same size, so gate and up come as [inter, hidden] and
    down as [hidden, inter]."""
    return _matrices(g, 3 * count, inter, hidden, bits, group).view(count, -1)


def _routing(g, n, experts, k):
    """n tokens' k distinct experts, popularity Zipf(1.1) over a random
    permutation of the experts, and softmax weights."""
    order = torch.randperm(experts, generator=g, device=DEV)
    logp = torch.empty(experts, device=DEV)
    logp[order] = -1.1 * torch.log(torch.arange(1, experts + 1, device=DEV, dtype=torch.float32))
    u = torch.rand((n, experts), generator=g, device=DEV).clamp_(1e-20, 1 - 1e-7)
    idx = torch.topk(logp - torch.log(-torch.log(u)), k, dim=1).indices.to(torch.int32)
    w = torch.softmax(_normal(g, n, k), dim=1)
    return idx.contiguous(), w.contiguous()


def _inputs(case, seed):
    """Every tensor of a case, from the case and the seed alone."""
    g = _gen(seed, 17)
    kind = case["kind"]
    if kind == "lm_head":
        m = _matrices(g, 1, case["out_dim"], case["in_dim"], 4, 64)[0]
        return dict(w=m, x=_normal(g, case["in_dim"]))
    if kind == "qmm":
        m = _matrices(g, 1, case["out_dim"], case["in_dim"], case["bits"], case["group"])[0]
        return dict(w=m, x=_normal(g, case["n"], case["in_dim"]))
    H, I, E, k, _, shared = _model(case)
    if kind == "experts":
        d = dict(blobs=_experts(g, case["k"], H, I, case["bits"]), x=_normal(g, H), h_mid=_normal(g, H),
                 w=torch.softmax(_normal(g, case["k"]), 0))
        if case["shared"]:
            d["shared_out"] = _normal(g, H, sigma=0.3)
        return d
    if kind == "router":
        return dict(router=_normal(g, E, H, sigma=0.02), x=_normal(g, case["n"], H))
    if kind == "decode":
        layers = []
        for l in range(case["layers"]):
            gl = _gen(seed, 1000 + l)
            d = dict(experts=_experts(gl, E, H, I, case["bits"]), router=_normal(gl, E, H, sigma=0.02),
                     norm=(1 + _normal(gl, H, sigma=0.1)).to(torch.bfloat16))
            if shared:
                d["shared"] = _experts(gl, 1, H, I, 4)[0]
                d["gate"] = _normal(gl, H, sigma=0.02)
            layers.append(d)
        T = case["tokens"]
        return dict(layers=layers, x=_normal(g, T, H), resid=_normal(g, T, H), attn=_normal(g, T, H, sigma=0.3))
    n = case["n"]
    idx, w = _routing(g, n, E, k)
    x = _normal(g, n, H)
    d = dict(experts=_experts(g, E, H, I, case["bits"]), idx=idx, w=w,
             x=x.to(torch.bfloat16) if case["x"] == "bf16" else x)
    if kind == "block":
        d["h_mid"] = _normal(g, n, H)
        if shared:
            d["shared"] = _experts(g, 1, H, I, 4)[0]
            d["gate"] = _normal(g, H, sigma=0.02)
    return d


# -- the calls ---------------------------------------------------------------


def _qweights(m, out_dim, in_dim, bits, group):
    codes = out_dim * in_dim * bits // 8
    return sa.QuantWeights(m, 0, codes, codes + out_dim * (in_dim // group) * 2, group, bits)


def prepare(case, seed):
    st = dict(_inputs(case, seed), case=case)
    kern = st["kern"] = sa.Kernels(0)
    kind = case["kind"]
    empty = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device=DEV)
    if kind == "lm_head":
        st["qw"] = _qweights(st["w"], case["out_dim"], case["in_dim"], 4, 64)
        st["y"] = empty(case["out_dim"])
        st["pick"] = empty(1, dtype=torch.int32)
        return st
    if kind == "qmm":
        st["qw"] = _qweights(st["w"], case["out_dim"], case["in_dim"], case["bits"], case["group"])
        st["y"] = empty(case["n"], case["out_dim"])
        st["ws"] = empty(kern.qmm_workspace_size(case["in_dim"], case["group"], case["n"]), dtype=torch.uint8)
        return st
    H, I, E, k, norm, shared = _model(case)
    if H > 4096:
        kern.reserve(H, I, 1024)
    if kind == "router":
        n = case["n"]
        st.update(idx=empty(n, k, dtype=torch.int32), w=empty(n, k), logits=empty(n, E))
        return st
    lay = st["lay"] = sa.ExpertLayout(H, I, case["bits"], 64)
    if kind == "experts":
        st["bind"] = [(st["blobs"], s * lay.expert_size) for s in range(case["k"])]
        st["wh"] = st["w"].tolist()
        st["out"] = empty(H)
        return st
    if kind == "decode":
        T = case["tokens"]
        st["io"], st["work"] = empty(T, H), empty(T, H)
        layers = [kern.layer(lay, d["experts"], lay.expert_size, E, k, norm, d["router"], d.get("shared"), d.get("gate"))
                  for d in st["layers"]]
        norms = [d["norm"] for d in st["layers"]]

        def step():
            # h_mid = residual + attention output, then the MoE blocks.
            torch.add(st["resid"], st["attn"], out=st["io"])
            if T == 1:
                sa.check(kern.moe_decode_layers(layers, norms, EPS, st["x"], st["io"], st["work"]), "decode")
            else:
                sa.check(kern.moe_decode_tokens(layers, norms, EPS, T, st["x"], st["io"], st["work"]), "decode")

        st["graph"] = sa.capture_graph(kern, step)
        return st
    n = case["n"]
    st["out"] = empty(n, H)
    if kind == "block":
        size = kern.moe_prefill_block_workspace_size(lay, n, E, k, shared)
    else:
        size = kern.moe_prefill_workspace_size(lay, n, E, k)
    st["ws"] = empty(size, dtype=torch.uint8)
    return st


def run(st):
    case, kern = st["case"], st["kern"]
    kind = case["kind"]
    if kind == "lm_head":
        sa.check(kern.qmv_argmax(st["qw"], st["x"], st["y"], case["out_dim"], case["in_dim"], st["pick"]), "lm_head")
        return st["y"], st["pick"]
    if kind == "qmm":
        sa.check(kern.qmm(st["qw"], st["x"], st["y"], case["out_dim"], case["in_dim"], case["n"], st["ws"]), "qmm")
        return st["y"]
    H, I, E, k, norm, _ = _model(case)
    if kind == "router":
        sa.check(kern.router(st["router"], st["x"], case["n"], E, H, k, norm, st["idx"], st["w"], st["logits"]), "router")
        return st["idx"], st["w"], st["logits"]
    if kind == "experts":
        sa.check(kern.experts_decode(st["lay"], st["bind"], st["wh"], st["x"], st["h_mid"], st.get("shared_out"), 0.5,
                                     st["out"]), "experts")
        return st["out"]
    if kind == "decode":
        st["graph"].replay()
        return st["io"]
    args = (st["lay"], st["experts"], st["lay"].expert_size, E, st["idx"], st["w"], st["x"], case["x"] == "bf16",
            case["n"], k)
    if kind == "block":
        sa.check(kern.moe_prefill_block(*args, st.get("shared"), st.get("gate"), st["h_mid"], st["out"], st["ws"]), "block")
    else:
        sa.check(kern.moe_prefill(*args, st["out"], st["ws"]), "prefill")
    return st["out"]


# -- what a pass cannot do without -------------------------------------------


def _matrix_bytes(rows, cols, bits, group=64):
    return rows * cols * bits // 8 + 4 * rows * (cols // group)


def _hit(n, experts, k):
    """Expected number of distinct experts of n tokens under Zipf(1.1), each
    token's k draws without replacement taken as k independent ones whose
    shares are capped at one per token."""
    p = [1 / r ** 1.1 for r in range(1, experts + 1)]
    s = sum(p)
    q = [min(1.0, k * v / s) for v in p]
    scale = (k - sum(v for v in q if v >= 1)) / max(1e-9, sum(v for v in q if v < 1))
    q = [v if v >= 1 else min(1.0, v * scale) for v in q]
    return sum(1 - (1 - v) ** n for v in q)


def work(case):
    kind = case["kind"]
    if kind in ("lm_head", "qmm"):
        n, o, i = case.get("n", 1), case["out_dim"], case["in_dim"]
        return dict(bytes=_matrix_bytes(o, i, case.get("bits", 4), case.get("group", 64)) + 4 * n * (o + i),
                    flops=2 * n * o * i)
    H, I, E, k, _, shared = _model(case)
    if kind == "router":
        n = case["n"]
        return dict(bytes=4 * (E * H + n * H + n * E + 2 * n * k), flops=2 * n * E * H)
    expert = 3 * _matrix_bytes(I, H, case["bits"])
    flops = 6 * H * I
    if kind == "experts":
        return dict(bytes=case["k"] * expert + 4 * H * (4 if case["shared"] else 3), flops=case["k"] * flops)
    extra = 3 * _matrix_bytes(I, H, 4) + 4 * H if shared else 0
    if kind == "decode":
        T = case["tokens"]
        per = T * k * expert + extra + 4 * E * H + 2 * H
        return dict(bytes=case["layers"] * per + 4 * 4 * T * H,
                    flops=case["layers"] * T * ((k + bool(shared)) * flops + 2 * E * H))
    n = case["n"]
    x = (2 if case["x"] == "bf16" else 4) * n * H
    bytes_ = _hit(n, E, k) * expert + x + 4 * n * H + 8 * n * k
    if kind == "block":
        return dict(bytes=bytes_ + extra + 4 * n * H, flops=n * (k + bool(shared)) * flops)
    return dict(bytes=bytes_, flops=n * k * flops)


def tolerance(case):
    # About four times the largest distance from `exact` seen over the
    # ranges below.
    kind = case["kind"]
    if kind == "decode":
        # 3.7e-7 after 40 layers: a rounding in one travels through the rest.
        return {"rel": 2e-6}
    if kind == "experts":
        return {"rel": 1e-6}
    if kind == "lm_head":
        return {"rel": 2e-6}
    if kind == "router":
        # Slots of experts whose logits tie to f32 rounding may exchange.
        return {"rel": 1e-6, "differ": 2e-3}
    if kind == "qmm":
        # f32 rows as bf16 pairs (2.8e-6).
        return {"rel": 1.2e-5}
    if case["model"] == "flash-next":
        # f32 activations (5.7e-8).
        return {"rel": 4e-7}
    # Grouped GEMMs over fp16 activations (1e-5 to 4e-5, the most with the
    # fewest tokens).
    return {"rel": 1.5e-4}


# -- the same in 64 bits -----------------------------------------------------


def _dequant(m, rows, cols, bits, group):
    """One packed matrix (bytes) as float64 [rows, cols]."""
    cb = rows * cols * bits // 8
    sb = rows * (cols // group) * 2
    raw = m[:cb]
    if bits == 4:
        q = torch.stack((raw & 15, raw >> 4), dim=-1).view(rows, cols)
    else:
        p = raw.view(-1, 3).to(torch.int32)
        p = p[:, 0] | (p[:, 1] << 8) | (p[:, 2] << 16)
        q = torch.stack([(p >> (3 * i)) & 7 for i in range(8)], dim=-1).view(rows, cols)
    s = m[cb:cb + sb].clone().view(torch.bfloat16).to(torch.float64).view(rows, -1, 1)
    b = m[cb + sb:cb + 2 * sb].clone().view(torch.bfloat16).to(torch.float64).view(rows, -1, 1)
    return (q.to(torch.float64).view(rows, cols // group, group) * s + b).view(rows, cols)


def _ffn(blob, x, hidden, inter, bits):
    """One expert on float64 rows x [m, hidden]."""
    part = blob.numel() // 3
    gate = x @ _dequant(blob[:part], inter, hidden, bits, 64).T
    up = x @ _dequant(blob[part:2 * part], inter, hidden, bits, 64).T
    act = gate / (1 + torch.exp(-gate)) * up
    return act @ _dequant(blob[2 * part:], hidden, inter, bits, 64).T


def _route(logits, k, norm):
    p = torch.softmax(logits, dim=-1)
    w, idx = torch.topk(p, k, dim=-1)
    return idx, (w / w.sum(-1, keepdim=True) if norm else w)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    f64 = torch.float64
    if kind == "lm_head":
        y = _dequant(d["w"], case["out_dim"], case["in_dim"], 4, 64) @ d["x"].to(f64)
        return y, y.argmax().view(1).to(torch.int32)
    if kind == "qmm":
        w = d["w"]
        return d["x"].to(f64) @ _dequant(w, case["out_dim"], case["in_dim"], case["bits"], case["group"]).T
    H, I, E, k, norm, shared = _model(case)
    if kind == "router":
        logits = d["x"].to(f64) @ d["router"].to(f64).T
        return _scan_slots(torch.softmax(logits, -1), k, norm) + (logits,)
    bits = case["bits"]
    if kind == "experts":
        x = d["x"].to(f64).view(1, H)
        out = d["h_mid"].to(f64)
        for s in range(case["k"]):
            out = out + d["w"][s].to(f64) * _ffn(d["blobs"][s], x, H, I, bits)[0]
        if case["shared"]:
            out = out + d["shared_out"].to(f64) / (1 + math.exp(-0.5))
        return out
    if kind == "decode":
        r = (d["resid"] + d["attn"]).to(f64)
        x = d["x"].to(f64)
        for l, p in enumerate(d["layers"]):
            if l:
                x = r / torch.sqrt((r * r).mean(-1, keepdim=True) + EPS) * p["norm"].to(f64)
            idx, w = _route(x @ p["router"].to(f64).T, k, norm)
            add = torch.zeros_like(r)
            for t in range(case["tokens"]):
                for s in range(k):
                    add[t] += w[t, s] * _ffn(p["experts"][idx[t, s]], x[t:t + 1], H, I, bits)[0]
            if shared:
                g = torch.sigmoid(x @ p["gate"].to(f64)).view(-1, 1)
                add = add + g * _ffn(p["shared"], x, H, I, 4)
            r = r + add
        return r
    x = d["x"].to(f64)
    out = torch.zeros_like(x)
    idx = d["idx"].to(torch.int64)
    for e in idx.unique().tolist():
        t, s = (idx == e).nonzero(as_tuple=True)
        out.index_add_(0, t, _ffn(d["experts"][e], x[t], H, I, bits) * d["w"][t, s].to(f64).view(-1, 1))
    if kind == "block":
        if shared:
            out += torch.sigmoid(x @ d["gate"].to(f64)).view(-1, 1) * _ffn(d["shared"], x, H, I, 4)
        out += d["h_mid"].to(f64)
    return out


def _scan_slots(p, k, norm):
    """The routers' slot order: scan the experts in index order, replace the
    smallest slot (the lowest on ties) by every strictly larger score."""
    n, experts = p.shape
    val = torch.full((n, k), -1e30, dtype=torch.float64, device=p.device)
    idx = torch.zeros((n, k), dtype=torch.int64, device=p.device)
    rows = torch.arange(n, device=p.device)
    for e in range(experts):
        low = val.argmin(dim=1)
        take = p[:, e] > val[rows, low]
        val[rows[take], low[take]] = p[take, e]
        idx[rows[take], low[take]] = e
    w = val / val.sum(-1, keepdim=True) if norm else val
    return idx.to(torch.int32), w
