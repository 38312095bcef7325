"""The measured cases: what a program that runs quantized models on this library has it do.

Each case is a dict of plain values; `kind` names the entry point:

- matvec: `matvec_any` over `copies` tensors, one token's projections (or its router);
- attention: `gqa_causal_attention_f32` of one token over the K/V caches of `layers` layers;
- gemm: `quantize_act` and `gemm`, one projection of a prompt's rows;
- moe: `dispatch_qwen3_moe_ffn`, one expert layer for `tokens` tokens;
- decode / prefill: `DecodeModel`, a whole token (a captured step, replayed) or a whole prompt;
- forward: `ForwardModel.evaluate`, the int8 model's greedy loop.

Weights are random GGUF blocks whose values have a variance of 1 / n_in, so that activations keep
their size through a stack of layers; activations are normal with per-channel scales that spread
as a language model's do.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jero-engine_amd"))
import jero_hip as J  # noqa: E402

QUANT = {"F32": J.F32, "F16": J.F16, "BF16": J.BF16, "Q4_0": J.Q4_0, "Q8_0": J.Q8_0, "Q4_K": J.Q4_K, "Q6_K": J.Q6_K}
BLOCK = {"F32": (1, 4), "F16": (1, 2), "BF16": (1, 2), "Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144),
         "Q6_K": (256, 210)}
EPS = 1e-6

# The dense 8B and the 30B mixture shapes of bench.py, cut to a few layers (a layer costs what it costs in the
# whole model; the head is whole).
DENSE_8B = dict(hidden=4096, ffn=12288, heads=32, kv_heads=8, head_dim=128, vocab=151936, theta=1e6, qk_norm=True,
                experts=0, top_k=0, mix="Q4_K_M", kv="f16")
MOE_30B = dict(hidden=2048, ffn=768, heads=32, kv_heads=4, head_dim=128, vocab=151936, theta=1e6, qk_norm=True,
               experts=128, top_k=8, mix="Q4_K_M", kv="f16")


def listed():
    return [
        # an expert layer's router: one small float product, the smallest call a layer makes
        dict(name="matvec_f32_router", kind="matvec", quant="F32", laid=False, n_in=2048, n_out=128, copies=1),
        # one token through 8 FFN-sized Q4_K projections, in the layout weights are loaded into
        dict(name="matvec_q4k", kind="matvec", quant="Q4_K", laid=True, n_in=4096, n_out=12288, copies=8),
        # the same for a Q8_0 model's square projections, straight from the file's blocks
        dict(name="matvec_q8_0", kind="matvec", quant="Q8_0", laid=False, n_in=4096, n_out=4096, copies=8),
        # one token's attention in 8 layers over a 4096-token cache
        dict(name="attention_4096", kind="attention", heads=32, kv_heads=8, head_dim=128, seq=4096, layers=8, kv="f16"),
        # a 512-token prompt through an FFN projection
        dict(name="gemm_q4k_512", kind="gemm", quant="Q4_K", laid=True, n_in=4096, n_out=14336, tokens=512),
        # a short prompt (or a chunk of one) through a down projection
        dict(name="gemm_q6k_37", kind="gemm", quant="Q6_K", laid=True, n_in=12288, n_out=4096, tokens=37),
        # an expert layer for one token (decode), and for a batch of 64
        dict(name="moe_1", kind="moe", tokens=1, experts=128, top_k=8, hidden=2048, ffn=768, down="Q6_K", laid=True),
        dict(name="moe_64", kind="moe", tokens=64, experts=128, top_k=8, hidden=2048, ffn=768, down="Q6_K", laid=True),
        # one decode step with the cache full
        dict(name="decode_8b_layers", kind="decode", layers=6, capacity=4096, pos=4095, **DENSE_8B),
        # a prompt of odd length, dense and mixture
        dict(name="prefill_8b_layers", kind="prefill", layers=4, capacity=1024, tokens=509, **DENSE_8B),
        dict(name="prefill_30b_layers", kind="prefill", layers=2, capacity=1024, tokens=512, **MOE_30B),
        # the matrix bench's run of the int8 model
        dict(name="forward_int8", kind="forward", vocab=256, positions=64, prompt=11),
    ]


def _between(rng, lo, hi, step=1):
    """A multiple of `step` from [lo, hi], spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["matvec", "attention", "gemm", "moe", "decode", "prefill", "forward"])
    if kind == "matvec":
        quant = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q8_0", "Q4_0", "F32", "F16", "BF16"])
        n_out = _between(rng, 64, 16384) if rng.random() < 0.8 else _between(rng, 16384, 151936)
        return dict(kind=kind, quant=quant, laid=quant in ("Q4_K", "Q6_K") and rng.random() < 0.7,
                    n_in=_between(rng, 512, 14336, 256), n_out=n_out, copies=rng.randint(1, 4 if n_out <= 16384 else 1))
    if kind == "attention":
        kv_heads = rng.choice([2, 4, 8])
        return dict(kind=kind, heads=kv_heads * rng.choice([1, 2, 4, 8]), kv_heads=kv_heads,
                    head_dim=rng.choice([64, 128, 128]), seq=_between(rng, 1, 32768), layers=rng.randint(1, 6),
                    kv=rng.choice(["f16", "f16", "f32"]))
    if kind == "gemm":
        quant = rng.choice(["Q4_K", "Q4_K", "Q6_K"])
        return dict(kind=kind, quant=quant, laid=rng.random() < 0.8, n_in=_between(rng, 1024, 12288, 256),
                    n_out=_between(rng, 1024, 14336, 32), tokens=_between(rng, 8, 1024))
    if kind == "moe":
        experts = rng.choice([64, 128])
        return dict(kind=kind, tokens=_between(rng, 1, 768), experts=experts, top_k=rng.choice([4, 6, 8]),
                    hidden=rng.choice([1024, 2048]), ffn=rng.choice([512, 768, 1024]), down=rng.choice(["Q4_K", "Q6_K"]),
                    laid=rng.random() < 0.8)
    if kind == "forward":
        return dict(kind=kind, vocab=_between(rng, 32, 1024), positions=64, prompt=rng.randint(3, 40))
    if rng.random() < 0.3:
        model = dict(MOE_30B, layers=2)
    else:
        model = dict(DENSE_8B, layers=rng.randint(2, 4))
        model["hidden"] = rng.choice([1024, 2048, 2560, 4096])
        model["ffn"] = _between(rng, 2048, 12288, 256)
        model["heads"], model["kv_heads"] = rng.choice([(16, 8), (32, 8), (16, 4), (32, 32)])
        model["mix"] = rng.choice(["Q4_K_M", "Q4_K_M", "Q8_0"])
        model["qk_norm"] = rng.random() < 0.7
    model["vocab"] = rng.choice([32000, 128256, 151936])
    model["kv"] = rng.choice(["f16", "f16", "f32"])
    if kind == "decode":
        capacity = rng.choice([512, 2048, 8192])
        return dict(kind=kind, capacity=capacity, pos=_between(rng, 1, capacity - 1), **model)
    return dict(kind=kind, capacity=1024, tokens=_between(rng, 8, 512), **model)


# ------------------------------------------------------------------ inputs


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _blocks(quant, n_in, rows, g, gain=1.0):
    """Random weights of variance about gain^2 / n_in, as the bytes of a GGUF tensor [n_in, rows]."""
    size = gain / math.sqrt(n_in)
    if BLOCK[quant][0] == 1:
        w = torch.randn(rows * n_in, generator=g, device="cuda") * size
        return w.to({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[quant]).view(torch.uint8)
    be, bb = BLOCK[quant]
    nb = rows * (n_in // be)
    b = torch.randint(0, 1 << 32, ((nb * bb + 3) // 4,), generator=g, device="cuda").to(torch.uint32)
    b = b.view(torch.uint8)[:nb * bb].view(nb, bb)
    spread = torch.rand(nb, generator=g, device="cuda") * 0.6 + 0.7
    # the standard deviation of a weight whose scale is 1
    one = {"Q4_K": 300.0, "Q6_K": 680.0, "Q8_0": 73.0, "Q4_0": 4.6}[quant]
    d = (spread * (size / one)).half().view(torch.uint8).view(nb, 2)
    if quant == "Q6_K":
        b[:, 192:208] = torch.randint(-64, 64, (nb, 16), dtype=torch.int8, generator=g, device="cuda").view(torch.uint8)
        b[:, 208:210] = d
    else:
        b[:, 0:2] = d
    if quant == "Q4_K":  # minima that bring the mean to about zero
        b[:, 2:4] = (7.5 * spread * (size / one)).half().view(torch.uint8).view(nb, 2)
    return b.reshape(-1)


def _acts(rows, n, g):
    scale = torch.exp(0.5 * torch.randn(n, generator=g, device="cuda"))
    return torch.randn(rows, n, generator=g, device="cuda") * scale


def _view(quant, dims, data):
    return J.TensorView("w", QUANT[quant], list(dims), data)


def _q6k_layer(i, n):
    """The Q4_K_M mix: attn_v and ffn_down of these layers are Q6_K."""
    return i < n // 8 or i >= 7 * n // 8 or (i - n // 8) % 3 == 2


def _model_tensors(c, seed):
    """(name, quant, dims, bytes) of every tensor of a decode / prefill case."""
    H, F, V, hd = c["hidden"], c["ffn"], c["vocab"], c["head_dim"]
    Q, KV, E = c["heads"] * hd, c["kv_heads"] * hd, c["experts"]
    low, high = ("Q4_K", "Q6_K") if c["mix"] == "Q4_K_M" else ("Q8_0", "Q8_0")
    spec = [("token_embd.weight", low, (H, V)), ("output.weight", high, (H, V)), ("output_norm.weight", "norm", (H,))]
    for i in range(c["layers"]):
        v = high if _q6k_layer(i, c["layers"]) else low
        p = "blk.%d." % i
        spec += [(p + "attn_norm.weight", "norm", (H,)), (p + "ffn_norm.weight", "norm", (H,)),
                 (p + "attn_q.weight", low, (H, Q)), (p + "attn_k.weight", low, (H, KV)),
                 (p + "attn_v.weight", v, (H, KV)), (p + "attn_output.weight", low, (Q, H))]
        if c["qk_norm"]:
            spec += [(p + "attn_q_norm.weight", "norm", (hd,)), (p + "attn_k_norm.weight", "norm", (hd,))]
        if E:
            spec += [(p + "ffn_gate_inp.weight", "F32", (H, E)), (p + "ffn_gate_exps.weight", low, (H, F, E)),
                     (p + "ffn_up_exps.weight", low, (H, F, E)), (p + "ffn_down_exps.weight", v, (F, H, E))]
        else:
            spec += [(p + "ffn_gate.weight", low, (H, F)), (p + "ffn_up.weight", low, (H, F)),
                     (p + "ffn_down.weight", v, (F, H))]
    for n, (name, quant, dims) in enumerate(spec):
        g = _gen(seed, 100 + n)
        if quant == "norm":
            yield name, "F32", dims, (1 + 0.1 * torch.randn(dims[0], generator=g, device="cuda")).view(torch.uint8)
        else:
            # a sublayer adds a fraction of what the residual stream holds, as in a trained model: with more, the
            # int8 roundings that two correct programs take differently would grow from layer to layer
            gain = math.sqrt(H) if name == "token_embd.weight" else 0.2 if "attn_output" in name or "ffn_down" in name else 1.0
            yield name, quant, dims, _blocks(quant, dims[0], math.prod(dims[1:]), g, gain)


def _rings(c, seed, layer):
    g = _gen(seed, 50000 + layer)
    shape = (2, c["capacity"], c["kv_heads"] * c["head_dim"])
    return torch.randn(shape, generator=g, device="cuda").to(torch.float16 if c["kv"] == "f16" else torch.float32)


def _tokens(c, seed):
    n = c["tokens"] if c["kind"] == "prefill" else 1
    return np.random.default_rng(seed).integers(0, c["vocab"], n).astype(np.int32)


class _Raw:
    """A device address as an array that torch can view; the view keeps the memory's owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=tuple(shape), typestr=typestr, version=2)


def _at(owner, ptr, shape, typestr):
    return torch.as_tensor(_Raw(owner, ptr, shape, typestr), device="cuda")


def _prepare_model(c, seed):
    moe = (c["experts"], c["top_k"], c["ffn"], False) if c["experts"] else None
    m = J.DecodeModel(c["hidden"], c["ffn"], c["layers"], c["vocab"], c["heads"], c["kv_heads"], c["head_dim"], EPS,
                      c["theta"], c["capacity"], J.KV_F16 if c["kv"] == "f16" else J.KV_F32, c["qk_norm"], moe)
    for name, quant, dims, data in _model_tensors(c, seed):
        m.set_tensor(name, QUANT[quant], data, dims[0], math.prod(dims[1:]))
    m.finalize()
    kvd, f = c["kv_heads"] * c["head_dim"], "<f2" if c["kv"] == "f16" else "<f4"
    state = dict(model=m)
    first, n = (c["pos"], 1) if c["kind"] == "decode" else (0, c["tokens"])
    out = {"logits": _at(m, m.state_ptrs()[2], (m.logits_len(),), "<f4")}
    for layer in range(c["layers"]):
        kv = _rings(c, seed, layer)
        torch.cuda.synchronize()
        m.write_kv(layer, kv[0], kv[1])
        k, v = m.kv_ptrs(layer)
        # what the call appends to the cache
        out["k%d" % layer] = _at(m, k, (c["capacity"], kvd), f)[first:first + n]
        out["v%d" % layer] = _at(m, v, (c["capacity"], kvd), f)[first:first + n]
    state["out"] = out
    tokens = _tokens(c, seed)
    if c["kind"] == "decode":
        state["token"], state["pos"] = int(tokens[0]), c["pos"]
        m.set_position(state["token"], state["pos"])
        m.decode_step()
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            m.decode_step()
    else:
        state["tokens"] = torch.from_numpy(tokens).pin_memory()
        m.prefill(state["tokens"], 0)  # a server's warm-up: the row buffers and the layouts of the weights
    return state


def prepare(case, seed):
    c = case
    J.init(0)
    if c["kind"] in ("decode", "prefill"):
        return dict(kind=c["kind"], **_prepare_model(c, seed))
    if c["kind"] == "matvec":
        w = []
        for i in range(c["copies"]):
            t = _view(c["quant"], (c["n_in"], c["n_out"]), _blocks(c["quant"], c["n_in"], c["n_out"], _gen(seed, i)))
            w.append(J.repack(t) if c["laid"] else t)
        x, y = _acts(c["copies"], c["n_in"], _gen(seed, 90)), torch.empty(c["copies"], c["n_out"], device="cuda")
        return dict(kind=c["kind"], calls=list(zip(y, w, x)), y=y,
                    ws=torch.empty(2 * c["n_in"], dtype=torch.uint8, device="cuda"))
    if c["kind"] == "attention":
        q, kv = _attention_inputs(c, seed)
        y = torch.empty_like(q)
        return dict(kind=c["kind"], calls=list(zip(y, q, kv[:, 0], kv[:, 1])), y=y,
                    shape=(c["heads"], c["kv_heads"], c["head_dim"], c["seq"], 1 / math.sqrt(c["head_dim"])),
                    ws=torch.empty(_attention_workspace(c), dtype=torch.uint8, device="cuda"))
    if c["kind"] == "gemm":
        t = _view(c["quant"], (c["n_in"], c["n_out"]), _blocks(c["quant"], c["n_in"], c["n_out"], _gen(seed, 0)))
        xq = torch.empty(c["tokens"] * J.row_bytes(J.Q8_K, c["n_in"]), dtype=torch.uint8, device="cuda")
        return dict(kind=c["kind"], w=J.repack_gemm(t) if c["laid"] else t, x=_acts(c["tokens"], c["n_in"], _gen(seed, 90)),
                    xq=xq, y=torch.empty(c["tokens"], c["n_out"], device="cuda"))
    if c["kind"] == "moe":
        w, x, logits = _moe_inputs(c, seed)
        return dict(kind=c["kind"], w=[J.repack(t) if c["laid"] else t for t in w], x=x, logits=logits, top_k=c["top_k"],
                    ws=J.moe_workspace(c["tokens"], c["experts"], c["top_k"], c["hidden"], c["ffn"]),
                    y=torch.empty_like(x))
    prompt = [int(t) for t in np.random.default_rng(seed).integers(0, c["vocab"], c["prompt"])]
    return dict(kind=c["kind"], model=J.ForwardModel(seed, c["vocab"], c["positions"]), prompt=prompt,
                n=c["positions"] - c["prompt"])


def _attention_workspace(c):
    """Room for one (max, sum, row) of floats per head and 64 positions."""
    return 4 * c["heads"] * (c["head_dim"] + 2) * (c["seq"] // 64 + 2) + (1 << 16)


def _attention_inputs(c, seed):
    g = _gen(seed, 0)
    q = torch.randn(c["layers"], c["heads"] * c["head_dim"], generator=g, device="cuda") * 1.5
    kv = torch.randn(c["layers"], 2, c["seq"], c["kv_heads"] * c["head_dim"], generator=g, device="cuda")
    return q, kv.to(torch.float16 if c["kv"] == "f16" else torch.float32)


def _moe_inputs(c, seed):
    E, H, F = c["experts"], c["hidden"], c["ffn"]
    shapes = [("Q4_K", (H, F, E)), ("Q4_K", (H, F, E)), (c["down"], (F, H, E))]
    w = [_view(q, s, _blocks(q, s[0], s[1] * s[2], _gen(seed, i))) for i, (q, s) in enumerate(shapes)]
    g = _gen(seed, 90)
    x = _acts(c["tokens"], H, g)
    return w, x, torch.randn(c["tokens"], E, generator=g, device="cuda")


def run(state):
    s, kind = state, state["kind"]
    if kind == "matvec":
        for y, w, x in s["calls"]:
            J.matvec_any(y, w, x, s["ws"])
        return s["y"]
    if kind == "attention":
        for y, q, k, v in s["calls"]:
            J.gqa_causal_attention_f32(y, q, k, v, *s["shape"], s["ws"])
        return s["y"]
    if kind == "gemm":
        J.quantize_act(J.Q8_K, s["x"], s["xq"])
        return J.gemm(s["w"], s["xq"], s["x"].shape[0], s["y"])
    if kind == "moe":
        idx, weight = J.dispatch_qwen3_moe_ffn(s["y"], s["x"], s["logits"], s["top_k"], *s["w"], workspace=s["ws"])
        return {"y": s["y"], "experts": idx, "weights": weight}
    if kind == "decode":
        s["model"].set_position(s["token"], s["pos"])
        s["graph"].replay()
        return s["out"]
    if kind == "prefill":
        s["model"].prefill(s["tokens"], 0)
        return s["out"]
    s["model"].reset()
    return np.array(s["model"].evaluate(s["prompt"], s["n"]), np.int64)


# ------------------------------------------------------------------ what a pass cannot do without


def _row_bytes(quant, n):
    return n // BLOCK[quant][0] * BLOCK[quant][1]


def work(case):
    c = case
    if c["kind"] == "matvec":
        one = c["n_out"] * _row_bytes(c["quant"], c["n_in"]) + 4 * (c["n_in"] + c["n_out"])
        return dict(bytes=c["copies"] * one, flops=2 * c["copies"] * c["n_in"] * c["n_out"])
    if c["kind"] == "attention":
        per = 2 * c["kv_heads"] * c["head_dim"] * (2 if c["kv"] == "f16" else 4)
        return dict(bytes=c["layers"] * (c["seq"] * per + 8 * c["heads"] * c["head_dim"]),
                    flops=4 * c["layers"] * c["seq"] * c["heads"] * c["head_dim"])
    if c["kind"] == "gemm":
        return dict(bytes=c["n_out"] * _row_bytes(c["quant"], c["n_in"]) + 4 * c["tokens"] * (c["n_in"] + c["n_out"]),
                    flops=2 * c["tokens"] * c["n_in"] * c["n_out"])
    if c["kind"] == "forward":
        # 8.4 million int8 weights a token, read once for the prompt and once for each further token
        steps = c["positions"] - c["prompt"]
        weights = 4 * (4 * 512 * 512 + 2 * 512 * 1024) + 512 * c["vocab"]
        return dict(bytes=weights * steps, flops=2 * weights * c["positions"])
    H, F, E = c["hidden"], c["ffn"], c["experts"]
    T = 1 if c["kind"] == "decode" else c["tokens"]
    used = E * (1 - (1 - c["top_k"] / E) ** T) if E else 0  # experts that some token is routed to
    if c["kind"] == "moe":
        one = 2 * F * _row_bytes("Q4_K", H) + H * _row_bytes(c["down"], F)
        return dict(bytes=int(used * one + T * (8 * H + 4 * E)), flops=6 * T * c["top_k"] * H * F)
    Q, KV = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    low, high = ("Q4_K", "Q6_K") if c["mix"] == "Q4_K_M" else ("Q8_0", "Q8_0")
    total = c["vocab"] * _row_bytes(high, H)
    flops = 2 * H * c["vocab"]
    seen = c["pos"] + 1 if c["kind"] == "decode" else T
    for i in range(c["layers"]):
        v = high if _q6k_layer(i, c["layers"]) else low
        total += (Q + KV) * _row_bytes(low, H) + KV * _row_bytes(v, H) + H * _row_bytes(low, Q)
        ffn = 2 * F * _row_bytes(low, H) + H * _row_bytes(v, F)
        total += used * ffn + 4 * H * E if E else ffn
        total += 2 * seen * KV * (2 if c["kv"] == "f16" else 4)
        attended = seen if c["kind"] == "decode" else T * (T + 1) // 2
        flops += 2 * T * (2 * H * (Q + KV) + 3 * H * F * (c["top_k"] or 1)) + 4 * attended * Q
    return dict(bytes=int(total), flops=int(flops))


def tolerance(case):
    # The products' and the attention's 32-bit sums come within 1.3e-7 and 5e-7 of 64 bits.  An expert layer quantizes
    # its inner activations to int8 again, where values that lie on a rounding boundary may go either way (up to 4e-4); in a
    # whole model such roundings, and those of the f16 caches, travel through every later layer.
    return {"matvec": {"rel": 1e-6}, "attention": {"rel": 2e-6}, "gemm": {"rel": 1e-6}, "moe": {"rel": 1.5e-3},
            "decode": {"rel": 3e-2, "max": 0.5}, "prefill": {"rel": 3e-2, "max": 0.9}, "forward": "exact"}[case["kind"]]


# ------------------------------------------------------------------ the same in 64 bits


def _weights64(quant, data, n_in):
    """The values of a GGUF tensor's bytes, [rows, n_in]."""
    f = torch.float64
    if BLOCK[quant][0] == 1:
        return data.view({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[quant]).to(f).view(-1, n_in)
    b = data.view(-1, BLOCK[quant][1])
    if quant == "Q8_0":
        return (b[:, :2].clone().view(torch.float16).to(f) * b[:, 2:].view(torch.int8)).reshape(-1, n_in)
    if quant == "Q4_0":
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(torch.int16) - 8
        return (b[:, :2].clone().view(torch.float16).to(f) * q).reshape(-1, n_in)
    if quant == "Q4_K":
        s, qs = b[:, 4:16], b[:, 16:].view(-1, 4, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        d, dmin = (b[:, i:i + 2].clone().view(torch.float16).to(f) for i in (0, 2))
        return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).view(-1, n_in)
    ql, qh = b[:, :128].view(-1, 2, 64), b[:, 128:192].view(-1, 2, 32)
    part = [(ql[:, :, :32] & 15) | ((qh & 3) << 4), (ql[:, :, 32:] & 15) | (((qh >> 2) & 3) << 4),
            (ql[:, :, :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 32:] >> 4) | ((qh >> 6) << 4)]
    q = torch.stack(part, 2).view(-1, 16, 16).to(torch.int16) - 32
    d = b[:, 208:210].clone().view(torch.float16).to(f)
    return ((d * b[:, 192:208].view(torch.int8))[:, :, None] * q).view(-1, n_in)


def _acts64(quant, x):
    """The values that rows `x` have once they are quantized for weights of `quant`."""
    x = x.float()
    if quant in ("F32", "F16", "BF16"):
        return x.double()
    if quant in ("Q8_0", "Q4_0"):  # blocks of 32: d = max|x| / 127
        b = x.view(-1, 32)
        d = b.abs().amax(1, keepdim=True) / 127
        q = torch.round(b * torch.where(d == 0, 0, 1 / d))
        return (q.double() * d).view(x.shape)
    b = x.view(-1, 256)  # blocks of 256: the largest element becomes -127
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = torch.where(top == 0, 0, -127 / top)
    q = torch.round(inv * b).clamp(max=127)
    return (q.double() * torch.where(top == 0, 0, 1 / inv)).view(x.shape)


def _product64(quant, data, x):
    """Rows `x` times a GGUF tensor, taken in parts that keep the 64-bit weights small."""
    n = x.shape[1]
    a, part = _acts64(quant, x), 16384 * _row_bytes(quant, n)
    return torch.cat([a @ _weights64(quant, data[i:i + part], n).T for i in range(0, data.numel(), part)], 1)


def _swiglu64(gate, up):
    return gate * torch.sigmoid(gate) * up


def _attend64(q, k, v, kv_heads, first):
    """q [T, heads, hd] of tokens first.. over k, v [S, kv_heads, hd], causal."""
    group = q.shape[1] // kv_heads
    out = []
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // group].T / math.sqrt(q.shape[2])
        last = torch.arange(first, first + q.shape[0], device="cuda")[:, None]
        s = s.masked_fill(torch.arange(k.shape[0], device="cuda")[None] > last, -math.inf)
        out.append(torch.softmax(s, 1) @ v[:, h // group])
    return torch.stack(out, 1).reshape(q.shape[0], -1)


def _experts64(w, x, logits, top_k):
    """(y, experts, weights) of an expert layer; w: (quant, dims, bytes) of gate, up and down."""
    p = torch.softmax(logits.double(), 1)
    order = torch.argsort(logits, dim=1, descending=True, stable=True)[:, :top_k]
    weight = p.gather(1, order)
    weight = weight / weight.sum(1, keepdim=True)
    y = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for e in torch.unique(order).tolist():
        rows, slot = torch.where(order == e)
        gate, up, down = ((q, b.view(dims[2], -1)[e]) for q, dims, b in w)
        a = _swiglu64(_product64(*gate, x[rows]), _product64(*up, x[rows]))
        y[rows] += weight[rows, slot][:, None] * _product64(*down, a)
    return y, order, weight


def _norm64(x, w, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope64(x, positions, theta):
    """x [T, heads, hd], neighbouring pairs rotated by position / theta^(2i / hd) (in 32 bits, as it is defined)."""
    hd = x.shape[2]
    expo = torch.arange(0, hd, 2, dtype=torch.float32, device="cuda") / hd
    angle = (positions.float()[:, None] / torch.pow(torch.tensor(theta, device="cuda"), expo)).double()[:, None]
    a, b = x[:, :, 0::2], x[:, :, 1::2]
    c, s = torch.cos(angle), torch.sin(angle)
    return torch.stack([a * c - b * s, a * s + b * c], 3).view(x.shape)


def _model64(c, seed):
    tokens = torch.from_numpy(_tokens(c, seed)).cuda().long()
    first = c["pos"] if c["kind"] == "decode" else 0
    at = torch.arange(first, first + tokens.numel(), device="cuda")
    hd, nkv, T = c["head_dim"], c["kv_heads"], tokens.numel()
    kv_type = torch.float16 if c["kv"] == "f16" else torch.float32
    w = {name: (quant, dims, data) for name, quant, dims, data in _model_tensors(c, seed)}

    def norm(name, x):
        return _norm64(x, _weights64(*[w[name][i] for i in (0, 2)], w[name][1][0])[0])

    def product(name, x):
        return _product64(w[name][0], w[name][2], x)

    quant, _, data = w["token_embd.weight"]
    x = _weights64(quant, data.view(c["vocab"], -1)[tokens].reshape(-1), c["hidden"])
    out = {}
    for i in range(c["layers"]):
        p = "blk.%d." % i
        n = norm(p + "attn_norm.weight", x)
        q, k, v = (product(p + t + ".weight", n).view(T, -1, hd) for t in ("attn_q", "attn_k", "attn_v"))
        if c["qk_norm"]:
            q, k = norm(p + "attn_q_norm.weight", q), norm(p + "attn_k_norm.weight", k)
        q, k = _rope64(q, at, c["theta"]), _rope64(k, at, c["theta"])
        out["k%d" % i], out["v%d" % i] = k.reshape(T, -1), v.reshape(T, -1)
        if c["kind"] == "decode":
            old = _rings(c, seed, i)[:, :first].double().view(2, first, nkv, hd)
        else:
            old = torch.empty(2, 0, nkv, hd, dtype=torch.float64, device="cuda")
        k, v = torch.cat([old[0], k.to(kv_type).double()]), torch.cat([old[1], v.to(kv_type).double()])
        x = x + product(p + "attn_output.weight", _attend64(q, k, v, nkv, first))
        n = norm(p + "ffn_norm.weight", x)
        if c["experts"]:
            logits = product(p + "ffn_gate_inp.weight", n)
            x = x + _experts64([w[p + "ffn_%s_exps.weight" % t] for t in ("gate", "up", "down")], n, logits, c["top_k"])[0]
        else:
            x = x + product(p + "ffn_down.weight", _swiglu64(product(p + "ffn_gate.weight", n), product(p + "ffn_up.weight", n)))
    out["logits"] = product("output.weight", norm("output_norm.weight", x[-1:]))[0]
    return out


def exact(case, seed):
    c = case
    if c["kind"] in ("decode", "prefill"):
        return _model64(c, seed)
    if c["kind"] == "matvec":
        x = _acts(c["copies"], c["n_in"], _gen(seed, 90))
        w = (_blocks(c["quant"], c["n_in"], c["n_out"], _gen(seed, i)) for i in range(c["copies"]))
        return torch.cat([_product64(c["quant"], t, x[i:i + 1]) for i, t in enumerate(w)])
    if c["kind"] == "attention":
        q, kv = _attention_inputs(c, seed)
        q = q.double().view(c["layers"], 1, c["heads"], c["head_dim"])
        kv = kv.view(c["layers"], 2, c["seq"], c["kv_heads"], c["head_dim"])
        return torch.cat([_attend64(q[i], kv[i, 0].double(), kv[i, 1].double(), c["kv_heads"], c["seq"] - 1)
                          for i in range(c["layers"])])
    if c["kind"] == "gemm":
        return _product64(c["quant"], _blocks(c["quant"], c["n_in"], c["n_out"], _gen(seed, 0)),
                          _acts(c["tokens"], c["n_in"], _gen(seed, 90)))
    if c["kind"] == "moe":
        w, x, logits = _moe_inputs(c, seed)
        names = {v: k for k, v in QUANT.items()}
        y, _, weight = _experts64([(names[t.quant], t.shape, t.data) for t in w], x, logits, c["top_k"])
        return {"y": y, "experts": None, "weights": weight}
    return None  # whole numbers
