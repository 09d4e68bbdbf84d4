"""The timed cases of this library: what a serving or loading program has it do, through the
public Python entry points, from one-row decode calls to a 4096-token prefill chunk.

  kind "dense"       one W4A16 projection (DenseW4A16.forward), a few rows to a chunk.
  kind "ffn"         one expert's MLP (ExpertFFN.forward) at a decode batch, replayed as a graph.
  kind "kimi_decode" a Kimi-K2 MoE decode layer on one GPU's 48 of 384 experts: shared expert,
                     router select, routed experts, residual join, replayed as a graph (as a
                     decode loop replays its layers).
  kind "kimi_prefill" the MoE block of a Kimi-K2 prefill chunk: router GEMM + select, routed
                     experts, shared expert, residual join, issued eagerly.
  kind "kimi_zipf"   the routed experts alone under skewed (Zipf) local routing.
  kind "dsv2"        a DeepSeek-V2-Lite MoE layer (64 routed experts, top-6, shared expert):
                     up to 64 tokens as a graph (decode), above eagerly (prefill chunk).
  kind "expanded"    the expert-parallel receive side: an expert-major buffer of worst-case
                     capacity with the routed total known on the device only.
  kind "repack"      loading a layer: checkpoint INT4 gate and up projections into the fused
                     device package.
"""
import math

import torch

from pegainfer_amd import layer, ops

KIMI_H, KIMI_I, KIMI_E, KIMI_N, KIMI_TOPK = 7168, 2048, 48, 384, 8
DSV2_H, DSV2_I, DSV2_E, DSV2_TOPK = 2048, 1408, 64, 6
GRAPH_TOKENS = 64  # DeepSeek-V2-Lite batches up to this replay a graph


def listed():
    return [
        # one token through a Qwen3-4B-shaped MLP projection: the smallest call there is
        {"name": "dense_r1", "kind": "dense", "rows": 1, "n": 9728, "k": 2560},
        # one expert's MLP for an odd handful of tokens (speculative decode, tiny batches)
        {"name": "ffn_r5", "kind": "ffn", "rows": 5, "h": KIMI_H, "i": KIMI_I},
        # a near-idle server: three sequences decoding
        {"name": "kimi_decode_t3", "kind": "kimi_decode", "tokens": 3},
        # the headline decode batch
        {"name": "kimi_decode_t64", "kind": "kimi_decode", "tokens": 64},
        # a busy server's decode batch, past the block sizes of the small-batch kernels
        {"name": "kimi_decode_t160", "kind": "kimi_decode", "tokens": 160},
        # an ordinary ragged prefill chunk, the whole MoE block
        {"name": "kimi_prefill_t1000", "kind": "kimi_prefill", "tokens": 1000},
        # the full prefill chunk with skewed experts: the largest call
        {"name": "kimi_zipf_t4096", "kind": "kimi_zipf", "tokens": 4096},
        # a small model's decode batch
        {"name": "dsv2_decode_t24", "kind": "dsv2", "tokens": 24},
        # a small model's prefill chunks, ordinary and large
        {"name": "dsv2_prefill_t512", "kind": "dsv2", "tokens": 512},
        {"name": "dsv2_prefill_t2500", "kind": "dsv2", "tokens": 2500},
        # decode on the expert-parallel receive side: 512 rows arrive in a buffer sized for the worst
        {"name": "expanded_r512", "kind": "expanded", "rows": 512, "capacity": 4480},
        # one layer of a rank's checkpoint becoming a device package
        {"name": "repack_e48", "kind": "repack", "experts": KIMI_E, "k": KIMI_H, "i": KIMI_I},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["dense", "ffn", "kimi_decode", "kimi_decode", "kimi_prefill", "kimi_zipf",
                       "dsv2", "dsv2", "expanded", "repack"])
    if kind == "dense":
        return {"kind": kind, "rows": _log_int(rng, 1, 512), "n": 64 * _log_int(rng, 16, 224),
                "k": 64 * _log_int(rng, 16, 112)}
    if kind == "ffn":
        return {"kind": kind, "rows": _log_int(rng, 1, 16), "h": 64 * _log_int(rng, 32, 112),
                "i": 64 * _log_int(rng, 16, 48)}
    if kind == "kimi_decode":
        return {"kind": kind, "tokens": _log_int(rng, 1, 256)}
    if kind == "kimi_prefill":
        return {"kind": kind, "tokens": _log_int(rng, 256, 2048)}
    if kind == "kimi_zipf":
        return {"kind": kind, "tokens": _log_int(rng, 512, 4000)}
    if kind == "dsv2":
        return {"kind": kind, "tokens": _log_int(rng, 1, 3000)}
    if kind == "expanded":
        rows = _log_int(rng, 32, 2048)
        return {"kind": kind, "rows": rows, "capacity": rows * rng.randint(1, 8) + 8 * KIMI_E}
    return {"kind": "repack", "experts": rng.randint(8, 47), "k": 64 * _log_int(rng, 32, 112),
            "i": 64 * _log_int(rng, 16, 32)}


# ------------------------------------------------------------------ inputs, from the seed alone
def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed(seed * 1009 + stream)


def _ckpt(g, experts, out_dim, in_dim):
    """Checkpoint tensors: offset-binary nibbles, scales |N(0, 0.02)| / 7."""
    packed = torch.randint(0, 256, (experts, out_dim, in_dim // 2), dtype=torch.uint8,
                           device="cuda", generator=g)
    scale = torch.randn(experts, out_dim, in_dim // 32, device="cuda", generator=g)
    return packed, (scale.abs_() * (0.02 / 7)).to(torch.bfloat16)


def _normal(g, *shape, std=1.0):
    return (torch.randn(*shape, device="cuda", generator=g) * std).to(torch.bfloat16)


def _reorder(ckpt):
    packed, scale = ckpt
    e, n, half = packed.shape
    return ops.marlin_int4_reorder(packed, scale, e, 2 * half, n)


def _experts(seed, stream, e, h, i):
    """The gate, up and down checkpoint pairs of e experts."""
    g = _gen(seed, stream)
    return _ckpt(g, e, i, h), _ckpt(g, e, i, h), _ckpt(g, e, h, i)


def _package(gate, up, down):
    return ops.marlin_int4_fuse_w13(_reorder(gate), _reorder(up)), _reorder(down)


def _kimi_inputs(seed, t):
    g = _gen(seed, 2)
    return {"normed": _normal(g, t, KIMI_H), "hidden": _normal(g, t, KIMI_H),
            "bias": torch.randn(KIMI_N, device="cuda", generator=g) * 0.05,
            "logits": torch.randn(t, KIMI_N, device="cuda", generator=g),
            "gate_up": _normal(g, 2 * KIMI_I, KIMI_H, std=0.02),
            "down": _normal(g, KIMI_H, KIMI_I, std=0.02),
            "router": _normal(g, KIMI_N, KIMI_H, std=KIMI_H ** -0.5)}


def _zipf_inputs(seed, t):
    """Each token has one or two (60%) local experts of a Zipf(1.2) popularity; the rest of
    its eight routes belong to other GPUs."""
    g = _gen(seed, 3)
    prob = torch.arange(1, KIMI_E + 1, device="cuda", dtype=torch.float64).pow(-1.2)
    prob = prob[torch.randperm(KIMI_E, device="cuda", generator=g)].float()
    local = torch.multinomial(prob.expand(t, -1), 2, generator=g)
    other = torch.rand(t, KIMI_N - KIMI_E, device="cuda", generator=g).argsort(1)[:, :KIMI_TOPK]
    idx = other + KIMI_E
    idx[:, 0] = local[:, 0]
    two = torch.rand(t, device="cuda", generator=g) < 0.6
    idx[:, 1] = torch.where(two, local[:, 1], idx[:, 1])
    order = torch.rand(t, KIMI_TOPK, device="cuda", generator=g).argsort(1)
    idx = idx.gather(1, order).to(torch.int32).contiguous()
    w = torch.rand(t, KIMI_TOPK, device="cuda", generator=g) + 0.1
    return idx, (w / w.sum(1, keepdim=True)).contiguous(), _normal(g, t, KIMI_H)


def _expanded_inputs(seed, rows, capacity):
    """rows received rows of random experts, expert-major, each segment starting at a
    multiple of 8; pad rows are zero.  Returns psum, x, w and the expert of each row (-1 pad)."""
    g = _gen(seed, 4)
    expert = torch.randint(0, KIMI_E, (rows,), device="cuda", generator=g)
    counts = torch.bincount(expert, minlength=KIMI_E).tolist()
    psum, owner, cur = [], torch.full((capacity,), -1, device="cuda"), 0
    for e, c in enumerate(counts):
        cur = -(-cur // 8) * 8
        owner[cur:cur + c] = e
        cur += c
        psum.append(cur)
    psum.append(-(-cur // 8) * 8)
    real = (owner >= 0).unsqueeze(1)
    x = _normal(g, capacity, KIMI_H) * real
    w = (torch.rand(capacity, device="cuda", generator=g) + 0.1) * real.squeeze(1)
    return torch.tensor(psum, dtype=torch.int32, device="cuda"), x, w, owner


# ------------------------------------------------------------------ a program's state, and a pass
def prepare(case, seed):
    s = dict(case)
    kind = case["kind"]
    bf = dict(dtype=torch.bfloat16, device="cuda")
    if kind == "dense":
        g = _gen(seed, 1)
        s["layer"] = layer.DenseW4A16(_reorder(_ckpt(g, 1, case["n"], case["k"])),
                                      max_rows=case["rows"])
        s["x"] = _normal(g, case["rows"], case["k"])
        s["y"] = torch.zeros(case["rows"], case["n"], **bf)
    elif kind == "ffn":
        ffn = layer.ExpertFFN(*_package(*_experts(seed, 1, 1, case["h"], case["i"])),
                              max_rows=case["rows"])
        x = _normal(_gen(seed, 2), case["rows"], case["h"])
        y = torch.zeros(case["rows"], case["h"], **bf)
        s.update(layer=ffn, x=x, out=y, graph=layer.capture_graph(lambda: ffn.forward(x, y)))
    elif kind in ("kimi_decode", "kimi_prefill"):
        t = case["tokens"]
        s.update(_kimi_inputs(seed, t))
        routed = layer.RoutedExperts(
            *_package(*_experts(seed, 1, KIMI_E, KIMI_H, KIMI_I)), max_tokens=t, topk=KIMI_TOPK,
            block_size=ops.kimi_marlin_block_size(t))
        shared = layer.KimiSharedExpert(s["gate_up"], s["down"], max_tokens=t)
        s["out"] = torch.zeros(t, KIMI_H, **bf)
        if kind == "kimi_decode":
            moe = layer.KimiMoeDecodeLayer(routed, shared)
            s.update(layer=moe, graph=layer.capture_graph(
                lambda: moe.forward(s["hidden"], s["normed"], s["logits"], s["bias"], s["out"])))
        else:
            s.update(routed=routed, shared=shared, projected=torch.zeros(t, KIMI_H, **bf),
                     routed_f32=torch.zeros(t, KIMI_H, device="cuda"),
                     scores=torch.zeros(t, KIMI_N, device="cuda"),
                     topk_w=torch.zeros(t, KIMI_TOPK, device="cuda"),
                     topk_idx=torch.zeros(t, KIMI_TOPK, dtype=torch.int32, device="cuda"))
    elif kind == "kimi_zipf":
        t = case["tokens"]
        s["topk_idx"], s["topk_w"], s["hidden"] = _zipf_inputs(seed, t)
        s["layer"] = layer.RoutedExperts(
            *_package(*_experts(seed, 1, KIMI_E, KIMI_H, KIMI_I)), max_tokens=t, topk=KIMI_TOPK,
            block_size=ops.kimi_marlin_block_size(t))
        s["out"] = torch.zeros(t, KIMI_H, device="cuda")
    elif kind == "dsv2":
        t = case["tokens"]
        routed = layer.RoutedExperts(
            *_package(*_experts(seed, 1, DSV2_E, DSV2_H, DSV2_I)), max_tokens=t, topk=DSV2_TOPK,
            block_size=ops.kimi_marlin_block_size(t, topk=DSV2_TOPK, local_experts=DSV2_E))
        shared = layer.ExpertFFN(*_package(*_experts(seed, 5, 1, DSV2_H, 2 * DSV2_I)), max_rows=t)
        moe = layer.Dsv2MoeLayer(routed, shared)
        g = _gen(seed, 2)
        hidden = _normal(g, t, DSV2_H)
        logits = torch.randn(t, DSV2_E, device="cuda", generator=g)
        out = torch.zeros(t, DSV2_H, **bf)
        s.update(layer=moe, hidden=hidden, logits=logits, out=out)
        if t <= GRAPH_TOKENS:
            s["graph"] = layer.capture_graph(lambda: moe.forward(hidden, logits, out))
    elif kind == "expanded":
        cap = case["capacity"]
        s["psum"], s["x"], s["w"], _ = _expanded_inputs(seed, case["rows"], cap)
        s["w13"], s["w2"] = _package(*_experts(seed, 1, KIMI_E, KIMI_H, KIMI_I))
        s["route_ws"] = ops.KimiMarlinRouteWorkspace(cap, 8)
        s["gemm_ws"] = ops.KimiMarlinWna16Workspace(-(-cap // 8), KIMI_H, 8)
        s.update(w13_out=torch.zeros(cap, 2 * KIMI_I, **bf), act=torch.zeros(cap, KIMI_I, **bf),
                 out=torch.zeros(cap, KIMI_H, **bf))
    else:
        s["gate"], s["up"], _ = _experts(seed, 1, case["experts"], case["k"], case["i"])
    return s


def run(s):
    kind = s["kind"]
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    if kind == "dense":
        return s["layer"].forward(s["x"], s["y"])
    if kind == "kimi_prefill":
        t = s["tokens"]
        ops.kimi_k2_router_noaux_tc(s["normed"], s["router"], s["bias"], s["scores"], s["topk_w"],
                                    s["topk_idx"], t, t)
        s["shared"].forward(s["normed"], s["projected"])
        s["routed"].forward(s["normed"], s["topk_idx"], s["topk_w"], s["routed_f32"])
        ops.kimi_residual_add_scaled_f32(s["hidden"], s["projected"], s["routed_f32"],
                                         ops.KIMI_K2_ROUTER_SCALE, s["out"])
        return {"scores": s["scores"], "topk_idx": s["topk_idx"], "out": s["out"]}
    if kind == "kimi_zipf":
        return s["layer"].forward(s["hidden"], s["topk_idx"], s["topk_w"], s["out"])
    if kind == "dsv2":
        return s["layer"].forward(s["hidden"], s["logits"], s["out"])
    if kind == "expanded":
        routing = ops.kimi_deepep_build_marlin_routing_on_stream(s["route_ws"], s["psum"], 8,
                                                                 s["capacity"])
        ops.kimi_marlin_wna16_expanded_w13_gemm(s["gemm_ws"], routing, s["x"], s["w13"], s["w"],
                                                s["w13_out"])
        ops.kimi_marlin_w13_swiglu_expanded(s["w13_out"], routing.num_tokens_post_padded, s["act"],
                                            s["capacity"], KIMI_I)
        ops.kimi_marlin_wna16_expanded_w2_gemm(s["gemm_ws"], routing, s["act"], s["w2"], s["w"],
                                               s["out"])
        return s["out"]
    w13 = ops.marlin_int4_fuse_w13(_reorder(s["gate"]), _reorder(s["up"]))
    return w13.weight_packed_uint4b8, w13.weight_scale_permuted


# ------------------------------------------------------------------ what a pass cannot do without
def _touched(experts, tokens, share):
    """Expected experts with a route when each token picks each with probability share."""
    return experts * (1.0 - (1.0 - share) ** tokens)


def _expert_work(experts, rows, h, i):
    """Weights and scales of the experts, and the products of their rows."""
    return experts * 3 * h * i * (0.5 + 2 / 32), rows * 6.0 * h * i


def work(case):
    kind, t = case["kind"], case.get("tokens", 0)
    if kind == "dense":
        r, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k * (0.5 + 2 / 32) + 2 * r * (n + k), "flops": 2.0 * r * n * k}
    if kind == "ffn":
        b, f = _expert_work(1, case["rows"], case["h"], case["i"])
        return {"bytes": b + 4 * case["rows"] * case["h"], "flops": f}
    if kind in ("kimi_decode", "kimi_prefill"):
        b, f = _expert_work(_touched(KIMI_E, t, KIMI_TOPK / KIMI_N),
                            t * KIMI_TOPK * KIMI_E / KIMI_N, KIMI_H, KIMI_I)
        b += 3 * KIMI_H * KIMI_I * 2 + t * (KIMI_H * 6 + KIMI_N * 4)
        f += t * 6.0 * KIMI_H * KIMI_I
        if kind == "kimi_prefill":
            b, f = b + KIMI_N * KIMI_H * 2, f + 2.0 * t * KIMI_N * KIMI_H
        return {"bytes": b, "flops": f}
    if kind == "kimi_zipf":
        b, f = _expert_work(KIMI_E, 1.6 * t, KIMI_H, KIMI_I)
        return {"bytes": b + t * KIMI_H * 6, "flops": f}
    if kind == "dsv2":
        b, f = _expert_work(_touched(DSV2_E, t, DSV2_TOPK / DSV2_E), t * DSV2_TOPK, DSV2_H, DSV2_I)
        sb, sf = _expert_work(1, t, DSV2_H, 2 * DSV2_I)
        return {"bytes": b + sb + t * (DSV2_H * 4 + DSV2_E * 4), "flops": f + sf}
    if kind == "expanded":
        b, f = _expert_work(_touched(KIMI_E, case["rows"], 1 / KIMI_E), case["rows"], KIMI_H, KIMI_I)
        return {"bytes": b + 4 * case["rows"] * KIMI_H, "flops": f}
    w = 2 * case["experts"] * case["k"] * case["i"] * (0.5 + 2 / 32)
    return {"bytes": 2 * w, "flops": 0}


# Measured against 64 bits: the bf16 result of one projection is 1.6e-3 off, that of a chain of
# two or three with bf16 rows between them 3.9e-3 to 4.5e-3 (fp32 sums of bf16 rows the same), the
# router's fp32 scores 4e-7.
def tolerance(case):
    if case["kind"] == "repack":
        return "exact"
    if case["kind"] == "dense":
        return {"rel": 6e-3}
    if case["kind"] == "kimi_prefill":  # the fp32 scores decide ids: a tie may fall either way
        return {"rel": 1e-2, "differ": 1e-3}
    return {"rel": 1e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _dequant(ckpt, e):
    """Expert e's weights as the format defines them: bf16(q * scale)."""
    packed, scale = ckpt
    p, n = packed[e], packed.shape[1]
    q = torch.stack((p & 15, p >> 4), -1).reshape(n, -1).float() - 8
    return (q.reshape(n, -1, 32) * scale[e].float().unsqueeze(-1)).to(torch.bfloat16).reshape(n, -1).double()


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _mlp(x, gate, up, down, e):
    return _silu_mul(x @ _dequant(gate, e).T, x @ _dequant(up, e).T) @ _dequant(down, e).T


def _routed(x, idx, w, ckpts, experts):
    out = torch.zeros(x.shape[0], x.shape[1], dtype=torch.float64, device="cuda")
    for e in range(experts):
        t, k = (idx == e).nonzero(as_tuple=True)
        if t.numel():
            out.index_add_(0, t, _mlp(x[t], *ckpts, e) * w[t, k].double().unsqueeze(1))
    return out


def _sigmoid_top8(logits, bias):
    score = 1 / (1 + torch.exp(-logits))
    idx = (score + bias.double()).topk(KIMI_TOPK, 1).indices
    w = score.gather(1, idx)
    return idx, w / w.sum(1, keepdim=True)


def exact(case, seed):
    kind = case["kind"]
    if kind == "dense":
        g = _gen(seed, 1)
        w = _ckpt(g, 1, case["n"], case["k"])
        return _normal(g, case["rows"], case["k"]).double() @ _dequant(w, 0).T
    if kind == "ffn":
        return _mlp(_normal(_gen(seed, 2), case["rows"], case["h"]).double(),
                    *_experts(seed, 1, 1, case["h"], case["i"]), 0)
    if kind in ("kimi_decode", "kimi_prefill"):
        v = _kimi_inputs(seed, case["tokens"])
        x = v["normed"].double()
        logits = v["logits"].double() if kind == "kimi_decode" else x @ v["router"].double().T
        idx, w = _sigmoid_top8(logits, v["bias"])
        gu = x @ v["gate_up"].double().T
        projected = _silu_mul(gu[:, :KIMI_I], gu[:, KIMI_I:]) @ v["down"].double().T
        routed = _routed(x, idx, w, _experts(seed, 1, KIMI_E, KIMI_H, KIMI_I), KIMI_E)
        out = v["hidden"].double() + projected + routed * 2.827
        return out if kind == "kimi_decode" else {"scores": logits, "topk_idx": None, "out": out}
    if kind == "kimi_zipf":
        idx, w, x = _zipf_inputs(seed, case["tokens"])
        return _routed(x.double(), idx, w, _experts(seed, 1, KIMI_E, KIMI_H, KIMI_I), KIMI_E)
    if kind == "dsv2":
        g = _gen(seed, 2)
        x = _normal(g, case["tokens"], DSV2_H).double()
        p = torch.softmax(torch.randn(case["tokens"], DSV2_E, device="cuda", generator=g).double(), 1)
        w, idx = p.topk(DSV2_TOPK, 1)
        return (_routed(x, idx, w, _experts(seed, 1, DSV2_E, DSV2_H, DSV2_I), DSV2_E)
                + _mlp(x, *_experts(seed, 5, 1, DSV2_H, 2 * DSV2_I), 0))
    if kind == "expanded":
        _, x, w, owner = _expanded_inputs(seed, case["rows"], case["capacity"])
        return _routed(x.double(), owner.unsqueeze(1), w.unsqueeze(1),
                       _experts(seed, 1, KIMI_E, KIMI_H, KIMI_I), KIMI_E)
    return None
