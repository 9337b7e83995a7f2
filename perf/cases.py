"""The work a user of this package has it do, as cases that can be timed.

Every case runs through the package's public entry points:

  linear   one LittleBitLinear module call, decode to prefill row counts
  mlp      the MLP block as a decoder runs it: gate/up of RMSNorm(x) as one
           group call, down of SiLU(gate) * up added to x in place
  layer    one decoder layer (projections, attention, norms) on a KV cache
  step     one greedy draft token as a captured HIP graph: layers, final
           norm, Q4_0 head (logits and argmax)
  head     the Q4_0 head alone
  tree     a target model's verify of a token tree behind a cached prefix
  prompt   a target model's forward of a fresh prompt

Weights are random sign words with scales |N(0, 1)| + 0.05 (divided by the
square root of the length they are summed over, so that outputs stay O(1) as
in a trained model), activations N(0, 1): the distributions of the package's
own benchmark.  `exact` computes the same in float64 with plain torch.
"""
from __future__ import annotations

import math

import torch

from littlebit_amd import LittleBitBranch, LittleBitLinear, LittleBitProjection, LittleBitProjectionGroup
from littlebit_amd.decode import DecoderConfig, GPUTargetModel, LittleBitDecoder
from littlebit_amd.lm_head import Q4LMHead
from littlebit_amd.ops import PrivateWorkspace, private_workspace
from littlebit_amd.synthetic import synthetic_runtime_state

DEV = "cuda"
EPS = 1e-6

# hidden, intermediate, heads, kv heads, draft ranks (attention, MLP), residual ranks
FAMILIES = {
    "llama2-7b": (4096, 11008, 32, 32, (205, 298), (1843, 2686)),
    "llama3-8b": (4096, 14336, 32, 8, (204, 318), (1843, 2867)),
    "small": (1536, 4100, 24, 8, (77, 110), (700, 993)),  # head_dim 64, K and ranks off every tile
}
VOCAB = 32000


def listed():
    return [
        # a draft o_proj at batch 1, called as a module: the smallest call, launch and host latency
        {"name": "linear decode f32", "kind": "linear", "M": 1, "K": 4096, "N": 4096, "r0": 205, "r1": 0,
         "bf16": False, "bias": False},
        # a target down_proj of a bf16 model on a few rows (a short speculation), with a bias
        {"name": "linear few rows bf16", "kind": "linear", "M": 3, "K": 11008, "N": 4096, "r0": 298, "r1": 2686,
         "bf16": True, "bias": True},
        # q_proj of the target on a short prompt in the decoders' fp32
        {"name": "linear prompt f32", "kind": "linear", "M": 300, "K": 4096, "N": 4096, "r0": 205, "r1": 1843,
         "bf16": False, "bias": False},
        # gate_proj of a long bf16 prefill: the largest matrix products
        {"name": "linear prefill bf16", "kind": "linear", "M": 2048, "K": 4096, "N": 14336, "r0": 318, "r1": 2867,
         "bf16": True, "bias": False},
        # the target's MLP block verifying 8 drafted tokens
        {"name": "mlp verify", "kind": "mlp", "family": "llama2-7b", "M": 8, "residual": True},
        # the same for a 33-node token tree
        {"name": "mlp tree", "kind": "mlp", "family": "llama2-7b", "M": 33, "residual": True},
        # a whole target layer verifying 8 tokens on a 1,024-token context
        {"name": "layer verify", "kind": "layer", "family": "llama2-7b", "N": 8, "start": 1024, "residual": True},
        # a whole target layer (grouped-query attention) on a fresh, ragged prompt
        {"name": "layer prompt", "kind": "layer", "family": "llama3-8b", "N": 700, "start": 0, "residual": True},
        # one draft token on a 512-token context, an 8-layer draft model, graph replay
        {"name": "draft step", "kind": "step", "family": "llama2-7b", "layers": 8, "pos": 512, "residual": False},
        # the draft model's quantised head
        {"name": "head q4", "kind": "head", "vocab": VOCAB, "hidden": 4096},
        # a target model's verify of a 33-node tree behind a 1,000-token prefix
        {"name": "model tree", "kind": "tree", "family": "llama2-7b", "layers": 4, "T": 33, "prefix": 1000,
         "residual": True},
        # a target model's forward of a fresh 1,024-token prompt
        {"name": "model prompt", "kind": "prompt", "family": "llama2-7b", "layers": 4, "N": 1024, "residual": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "layer", "layer", "step", "head", "tree", "prompt"])
    family = rng.choice(sorted(FAMILIES))
    H, I, _, _, dr, rr = FAMILIES[family]
    if kind == "linear":
        residual = rng.random() < 0.6
        if rng.random() < 0.5:
            K, N, b = rng.choice([(H, H, 0), (H, I, 1), (I, H, 1)])
            r0, r1 = dr[b], rr[b] if residual else 0
        else:
            K, N = _log_int(rng, 256, 8192), _log_int(rng, 256, 8192)
            if rng.random() < 0.7:
                K = 8 * (K // 8)
            r0 = _log_int(rng, 16, 320)
            r1 = _log_int(rng, 64, 2048) if residual else 0
        return {"kind": kind, "M": _log_int(rng, 1, 2048), "K": K, "N": N, "r0": r0, "r1": r1,
                "bf16": rng.random() < 0.5, "bias": rng.random() < 0.3}
    if kind == "mlp":
        return {"kind": kind, "family": family, "M": _log_int(rng, 1, 160), "residual": rng.random() < 0.7}
    if kind == "layer":
        return {"kind": kind, "family": family, "N": _log_int(rng, 2, 1024), "start": rng.choice([0, rng.randint(1, 3000)]),
                "residual": rng.random() < 0.7}
    if kind == "step":
        return {"kind": kind, "family": family, "layers": rng.randint(2, 10), "pos": _log_int(rng, 1, 3000),
                "residual": rng.random() < 0.3}
    if kind == "head":
        return {"kind": kind, "vocab": rng.randint(1000, 64000), "hidden": 32 * rng.randint(24, 160)}
    if kind == "tree":
        return {"kind": kind, "family": family, "layers": rng.randint(1, 4), "T": _log_int(rng, 2, 64),
                "prefix": _log_int(rng, 16, 3000), "residual": True}
    return {"kind": kind, "family": family, "layers": rng.randint(1, 4), "N": _log_int(rng, 2, 1024),
            "residual": rng.random() < 0.7}


# ---------------------------------------------------------------------------
# inputs (made from the seed alone, on the GPU)
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV)


def _branch(gen, K, R, N):
    def words(rows, cols):
        w = torch.randint(-2**31, 2**31, (rows, -(-cols // 32)), generator=gen, dtype=torch.int64, device=DEV)
        if cols % 32:
            w[:, -1] &= (1 << (cols % 32)) - 1
        return w.to(torch.int32)

    def scales(n, div):
        return ((_randn(gen, n).abs() + 0.05) / div).contiguous()

    return {"v": words(R, K), "u": words(N, R), "g": scales(K, K ** 0.5), "l": scales(R, R ** 0.5),
            "h": scales(N, 1.0)}


def _branches(gen, K, N, ranks):
    return [_branch(gen, K, R, N) for R in ranks]


def _linear_inputs(case, seed):
    gen = _gen(seed)
    br = _branches(gen, case["K"], case["N"], [r for r in (case["r0"], case["r1"]) if r])
    x = _randn(gen, case["M"], case["K"])
    bias = _randn(gen, case["N"]) if case["bias"] else None
    return br, x.to(torch.bfloat16) if case["bf16"] else x, bias


def _mlp_inputs(case, seed):
    H, I, _, _, dr, rr = FAMILIES[case["family"]]
    ranks = [dr[1]] + ([rr[1]] if case["residual"] else [])
    gen = _gen(seed)
    gate, up, down = _branches(gen, H, I, ranks), _branches(gen, H, I, ranks), _branches(gen, I, H, ranks)
    w = 1 + 0.1 * _randn(gen, H)
    return gate, up, down, w, _randn(gen, case["M"], H)


def _config(case, layers):
    H, I, heads, kv, _, _ = FAMILIES[case["family"]]
    return DecoderConfig(hidden_size=H, intermediate_size=I, num_hidden_layers=layers, num_attention_heads=heads,
                         num_key_value_heads=kv, vocab_size=VOCAB, rms_norm_eps=EPS)


def _state(case, layers, seed, embed):
    _, _, _, _, dr, rr = FAMILIES[case["family"]]
    res = {"attn": rr[0], "mlp": rr[1]} if case["residual"] else None
    return synthetic_runtime_state(_config(case, layers), {"attn": dr[0], "mlp": dr[1]}, res, seed=seed, device=DEV,
                                   normalized=True, embed=embed)


def _cache(case, layers, length, seed):
    """Keys and values of the positions before the call."""
    c = _config(case, layers)
    gen = _gen(seed + 7919)
    shape = (layers, c.num_key_value_heads, length, c.head_dim)
    return _randn(gen, *shape), _randn(gen, *shape)


def _chain_mask(T):
    """Ancestor mask of a tree of T nodes: node i's parent is node (i - 1) // 2."""
    m = torch.zeros((T, T), dtype=torch.bool)
    for i in range(T):
        j = i
        while True:
            m[i, j] = True
            if j == 0:
                break
            j = (j - 1) // 2
    return m


def _tokens(seed, n):
    return torch.randint(0, VOCAB, (1, n), generator=torch.Generator().manual_seed(int(seed) + 31))


# ---------------------------------------------------------------------------
def _projection(br, bias=None):
    return LittleBitProjection([LittleBitBranch(v_sign=b["v"], u_sign=b["u"], v2=b["g"], mid=b["l"], u1=b["h"])
                                for b in br], bias)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        br, x, bias = _linear_inputs(case, seed)
        m = LittleBitLinear.from_packed(
            case["K"], case["N"], [{"u_packed": b["u"], "v_packed": b["v"], "u1": b["h"].reshape(1, -1),
                                    "v2": b["g"].reshape(1, -1), "mid": b["l"].reshape(1, -1)} for b in br],
            bias=bias, device=DEV)
        m(x[:1])  # a program's first call: the module lays its factors out
        return {"kind": kind, "module": m, "x": x}
    if kind == "mlp":
        gate, up, down, w, x = _mlp_inputs(case, seed)
        return {"kind": kind, "group": LittleBitProjectionGroup([_projection(gate), _projection(up)]),
                "down": _projection(down), "w": w, "x": x}
    if kind == "layer":
        dec = LittleBitDecoder(_state(case, 1, seed, False), _config(case, 1), DEV, case["start"] + case["N"])
        k, v = _cache(case, 1, case["start"], seed)
        dec.k_cache[:, :, :case["start"]] = k
        dec.v_cache[:, :, :case["start"]] = v
        return {"kind": kind, "dec": dec, "x": _randn(_gen(seed + 13), case["N"], dec.config.hidden_size),
                "start": case["start"]}
    if kind == "step":
        st = _state(case, case["layers"], seed, True)
        dec = LittleBitDecoder(st, _config(case, case["layers"]), DEV, case["pos"] + 64)
        k, v = _cache(case, case["layers"], case["pos"], seed)
        dec.k_cache[:, :, :case["pos"]] = k
        dec.v_cache[:, :, :case["pos"]] = v
        embed, head = st["model.embed_tokens.weight"], Q4LMHead(st["lm_head.weight"])
        tok = _tokens(seed, 1)[0].to(DEV)
        pos = torch.full((1,), case["pos"], dtype=torch.int64, device=DEV)
        logits, token = torch.empty(VOCAB, device=DEV), torch.empty(1, dtype=torch.int64, device=DEV)
        ws, stream = PrivateWorkspace(), torch.cuda.Stream()

        def step():
            h = dec.forward_hidden(embed.index_select(0, tok), 0, pos_t=pos, final_norm=False)
            head.argmax(h, dec.final_norm, EPS, out=token, logits=logits)
            return h

        stream.wait_stream(torch.cuda.current_stream())
        with private_workspace(ws), torch.no_grad():
            with torch.cuda.stream(stream):
                step()
            stream.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                h = step()
        torch.cuda.synchronize()
        return {"kind": kind, "graph": graph, "hidden": h, "logits": logits, "token": token,
                "keep": (dec, embed, head, tok, pos, ws, stream)}
    if kind == "head":
        gen = _gen(seed)
        head = Q4LMHead(_randn(gen, case["vocab"], case["hidden"]))
        w = 1 + 0.1 * _randn(gen, case["hidden"])
        return {"kind": kind, "head": head, "w": w, "x": _randn(gen, 1, case["hidden"]),
                "logits": torch.empty(case["vocab"], device=DEV)}
    st = _state(case, case["layers"], seed, True)
    n = case["prefix"] if kind == "tree" else case["N"]
    model = GPUTargetModel(draft_state=st, config=_config(case, case["layers"]), device=DEV,
                           torch_dtype=torch.bfloat16, max_seq_len=n + 64)
    ids = _tokens(seed, n)
    if kind == "tree":
        tree = [int(ids[0, -1])] + _tokens(seed + 1, case["T"] - 1)[0].tolist()
        model.forward(ids)  # the prefix is cached
        return {"kind": kind, "model": model, "ids": ids, "tree": tree, "mask": _chain_mask(case["T"]).to(DEV)}
    return {"kind": kind, "model": model, "ids": ids}


def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if kind == "linear":
            return state["module"](state["x"])
        if kind == "mlp":
            x = state["x"].clone()
            g, u = state["group"].forward(x, rms_weight=state["w"], rms_eps=EPS)
            state["down"].forward(g, out=x, residual=x, x_up=u)
            return [g, u, x]
        if kind == "layer":
            dec = state["dec"]
            y = dec.forward_hidden(state["x"], state["start"], final_norm=False)
            return [y, dec.k_cache, dec.v_cache]
        if kind == "step":
            state["graph"].replay()
            return [state["hidden"], state["logits"]]
        if kind == "head":
            token = state["head"].argmax(state["x"], state["w"], EPS, logits=state["logits"])
            return [state["logits"], token]
        if kind == "tree":
            return state["model"].forward_tree(state["ids"], state["tree"], state["mask"])
        state["model"].reset_cache()
        return state["model"].forward(state["ids"])


# ---------------------------------------------------------------------------
def _proj_work(M, K, N, ranks, sx=4, sy=4):
    b = sum(4 * (R * -(-K // 32) + N * -(-R // 32) + K + R + N) for R in ranks)
    return b + M * (K * sx + N * sy), sum(2 * M * R * (K + N) for R in ranks)


def _layer_work(case, M, start):
    H, I, heads, kv, dr, rr = FAMILIES[case["family"]]
    kvd = H // heads * kv
    ra = [dr[0]] + ([rr[0]] if case["residual"] else [])
    rm = [dr[1]] + ([rr[1]] if case["residual"] else [])
    parts = [_proj_work(M, H, H, ra), _proj_work(M, H, kvd, ra), _proj_work(M, H, kvd, ra), _proj_work(M, H, H, ra),
             _proj_work(M, H, I, rm), _proj_work(M, H, I, rm), _proj_work(M, I, H, rm)]
    b = sum(p[0] for p in parts) + 4 * 2 * (start + M) * kvd + 4 * 2 * M * kvd
    f = sum(p[1] for p in parts) + 4 * H * M * (start + (M + 1) / 2)  # causal q.k and p.v
    return b, f


def _q4_bytes(vocab, hidden):
    return vocab * hidden // 2 + vocab * hidden // 16


def work(case):
    kind = case["kind"]
    if kind == "linear":
        s = 2 if case["bf16"] else 4
        b, f = _proj_work(case["M"], case["K"], case["N"], [r for r in (case["r0"], case["r1"]) if r], s, s)
    elif kind == "mlp":
        H, I, _, _, dr, rr = FAMILIES[case["family"]]
        ranks = [dr[1]] + ([rr[1]] if case["residual"] else [])
        gu, dn = _proj_work(case["M"], H, I, ranks), _proj_work(case["M"], I, H, ranks)
        b, f = 2 * gu[0] + dn[0], 2 * gu[1] + dn[1]
    elif kind == "layer":
        b, f = _layer_work(case, case["N"], case["start"])
    elif kind == "step":
        H = FAMILIES[case["family"]][0]
        b, f = _layer_work(case, 1, case["pos"])
        b, f = case["layers"] * b + _q4_bytes(VOCAB, H) + 4 * VOCAB, case["layers"] * f + 2 * VOCAB * H
    elif kind == "head":
        b, f = _q4_bytes(case["vocab"], case["hidden"]) + 4 * case["vocab"], 2 * case["vocab"] * case["hidden"]
    else:
        H = FAMILIES[case["family"]][0]
        M, start = (case["T"], case["prefix"] - 1) if kind == "tree" else (case["N"], 0)
        b, f = _layer_work(case, M, start)
        b, f = case["layers"] * b + 2 * VOCAB * H + 4 * M * VOCAB, case["layers"] * f + 2 * M * VOCAB * H
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear" and case["bf16"]:
        return {"rel": 1e-2, "max": 0.1}  # bf16 outputs; the latent vector in bf16 on long inputs
    if kind in ("linear", "mlp", "layer"):
        return {"rel": 4e-5, "max": 4e-4}  # fp32 sums of 16-bit mantissa pairs
    if kind == "head":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "step":
        return {"rel": 2e-3, "max": 2e-2}  # logits of an 8-bit copy of the hidden state
    return {"rel": 1e-2, "max": 0.1}  # logits of a bf16 head


# ---------------------------------------------------------------------------
# float64
# ---------------------------------------------------------------------------
def _pm1(w, cols):
    bits = (w.unsqueeze(-1) >> torch.arange(32, dtype=torch.int32, device=w.device)) & 1
    return (1 - 2 * bits).reshape(w.shape[0], -1)[:, :cols].to(torch.float64)


def _linear64(x, br, bias=None):
    y = 0
    for b in br:
        t = (x * b["g"].double()) @ _pm1(b["v"], b["g"].numel()).t().contiguous() * b["l"].double()
        y = y + t @ _pm1(b["u"], b["l"].numel()).t().contiguous() * b["h"].double()
    return y if bias is None else y + bias.double()


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attention64(q, k, v, kc, vc, start, heads, mask):
    """q [M, H]; new k, v [M, kv * hd] written into kc, vc [kv, S, hd] at start."""
    M, kv, hd = q.shape[0], kc.shape[0], kc.shape[2]
    kc[:, start:start + M] = k.view(M, kv, hd).transpose(0, 1)
    vc[:, start:start + M] = v.view(M, kv, hd).transpose(0, 1)
    S = start + M
    allowed = torch.ones((M, S), dtype=torch.bool, device=q.device)
    allowed[:, start:] = mask
    out = torch.empty_like(q).view(M, heads, hd)
    for h in range(heads):
        j = h // (heads // kv)
        s = (q.view(M, heads, hd)[:, h] @ kc[j, :S].t().contiguous()) * hd ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(~allowed, float("-inf")), -1) @ vc[j, :S]
    return out.reshape(M, -1)


def _state_branches(st, p):
    out = [{"v": st[p + ".v_sign_rt"], "u": st[p + ".u_sign_rt"], "g": st[p + ".v2"].reshape(-1),
            "l": st[p + ".mid"].reshape(-1), "h": st[p + ".u1"].reshape(-1)}]
    if p + ".u_sign_r_rt" in st:
        out.append({"v": st[p + ".v_sign_r_rt"], "u": st[p + ".u_sign_r_rt"], "g": st[p + ".v2_r"].reshape(-1),
                    "l": st[p + ".mid_r"].reshape(-1), "h": st[p + ".u1_r"].reshape(-1)})
    return out


def _layer64(x, st, i, c, kc, vc, start, mask):
    p = f"model.layers.{i}."
    lin = lambda h, n: _linear64(h, _state_branches(st, p + n))  # noqa: E731
    h = _norm64(x, st[p + "input_layernorm.weight"])
    a = _attention64(lin(h, "self_attn.q_proj"), lin(h, "self_attn.k_proj"), lin(h, "self_attn.v_proj"), kc, vc, start,
                     c.num_attention_heads, mask)
    x = x + lin(a, "self_attn.o_proj")
    h = _norm64(x, st[p + "post_attention_layernorm.weight"])
    g = lin(h, "mlp.gate_proj")
    return x + lin(g / (1 + torch.exp(-g)) * lin(h, "mlp.up_proj"), "mlp.down_proj")


def _causal(M):
    return torch.ones((M, M), dtype=torch.bool, device=DEV).tril()


def _fp16_trunc(d):
    """The float32 scales as fp16 with the mantissa cut off, exponents in fp16's normal range."""
    return (d.to(torch.float32).view(torch.int32) & ~0x1FFF).view(torch.float32).double()


def _head64(weight, x, w):
    """Q4_0 weight times the Q8_0 hidden state (blocks of 32)."""
    rows, cols = weight.shape
    h = _norm64(x.double(), w).reshape(-1, 32)
    d8 = h.abs().amax(-1, keepdim=True) / 127
    q8 = torch.trunc(h / d8 + torch.sign(h) * 0.5) * _fp16_trunc(d8)
    out = []
    for part in weight.split(8192):
        blk = part.view(part.shape[0], cols // 32, 32)
        m = torch.gather(blk, -1, blk.abs().argmax(-1, keepdim=True))
        d = m / -8.0
        q = torch.clamp((blk * (1.0 / d) + 8.5).to(torch.int32), max=15) - 8
        out.append(((q.double() * _fp16_trunc(d)) * q8).sum((1, 2)))
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "linear":
            br, x, bias = _linear_inputs(case, seed)
            return _linear64(x.double(), br, bias)
        if kind == "mlp":
            gate, up, down, w, x = _mlp_inputs(case, seed)
            h = _norm64(x.double(), w)
            g, u = _linear64(h, gate), _linear64(h, up)
            return [g, u, x.double() + _linear64(g / (1 + torch.exp(-g)) * u, down)]
        if kind == "head":
            gen = _gen(seed)
            weight = _randn(gen, case["vocab"], case["hidden"])
            w = 1 + 0.1 * _randn(gen, case["hidden"])
            logits = _head64(weight, _randn(gen, 1, case["hidden"]), w)
            return [logits, None]
        if kind == "layer":
            c = _config(case, 1)
            st = _state(case, 1, seed, False)
            total = case["start"] + case["N"]
            kc, vc = (torch.zeros((1, c.num_key_value_heads, total, c.head_dim), dtype=torch.float64, device=DEV)
                      for _ in range(2))
            k, v = _cache(case, 1, case["start"], seed)
            kc[:, :, :case["start"]], vc[:, :, :case["start"]] = k.double(), v.double()
            x = _randn(_gen(seed + 13), case["N"], c.hidden_size).double()
            y = _layer64(x, st, 0, c, kc[0], vc[0], case["start"], _causal(case["N"]))
            return [y, kc, vc]
        layers = case["layers"]
        c = _config(case, layers)
        st = _state(case, layers, seed, True)
        embed, head = st["model.embed_tokens.weight"].double(), st["lm_head.weight"]
        if kind == "step":
            k, v = _cache(case, layers, case["pos"], seed)
            x = embed[_tokens(seed, 1)[0].to(DEV)]
            for i in range(layers):
                kc, vc = (torch.cat([t[i].double(), torch.zeros_like(t[i, :, :1]).double()], 1) for t in (k, v))
                x = _layer64(x, st, i, c, kc, vc, case["pos"], _causal(1))
            return [x, _head64(head, x, st["model.norm.weight"])]
        head = head.to(torch.bfloat16).double()
        if kind == "prompt":
            ids, mask, rows = _tokens(seed, case["N"])[0], _causal(case["N"]), slice(0, None)
        else:  # the prefix but its last token (the root), then the tree
            ids, T = _tokens(seed, case["prefix"])[0], case["T"]
            ids = torch.cat([ids, _tokens(seed + 1, T - 1)[0]])
            P = case["prefix"] - 1
            mask = _causal(P + T)
            mask[P:, P:] = _chain_mask(T).to(DEV)
            rows = slice(P, None)
        x = embed[ids.to(DEV)]
        for i in range(layers):
            kc, vc = (torch.zeros((c.num_key_value_heads, len(ids), c.head_dim), dtype=torch.float64, device=DEV)
                      for _ in range(2))
            x = _layer64(x, st, i, c, kc, vc, 0, mask)
        logits = _norm64(x, st["model.norm.weight"])[rows] @ head.t().contiguous()
        return logits if kind == "tree" else logits.unsqueeze(0)
