"""What a user of this library has it do, as cases to be timed: one call of the MoE FFN layer (`ember_moe_ffn`,
router, routing, dispatch, experts, combine) on a layer resident in HBM, over the layer shapes, encodings and
batch sizes that this repository's configurations and tests name.

An inference engine calls it once per layer and step: one token when a single user decodes, a few to a few
dozen tokens when a server batches decode steps, hundreds to thousands when a prompt is prefilled. Expert
stacks come as the GGUF file holds them (Q8_0, Q4_K, BF16, F16) or, as the tuned llama engine uploads them, in
F32; Q8_0 / Q4_K / BF16 layers usually carry the prefill pack, which the C++ drop-in call does not pass.

A case: `shape` (SHAPES), `type` of the expert stacks, `pack`, `T` tokens, and for drawn cases the router
options. Weights are N(0, 0.02), the router N(0, 1/d), hidden states N(0, 1)."""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ember.cpp_amd"))
import ember_moe as em  # noqa: E402

SHAPES = {
    # the toy layer of the F32 correctness configuration
    "toy": dict(d=256, d_ff=688, E=8, k=2),
    # a small dense-trained MoE that is served in F32
    "small": dict(d=1024, d_ff=2816, E=8, k=2),
    "mixtral": dict(d=4096, d_ff=14336, E=8, k=2),
    "qwen": dict(d=2048, d_ff=768, E=128, k=8),
    "qwen_large": dict(d=4096, d_ff=1536, E=128, k=8),
    # 64 routed experts, two shared ones as one of twice the width, a selection bias
    "deepseek": dict(d=2048, d_ff=1408, E=64, k=6, d_ff_shared=2816, bias_std=2.0),
}
TYPES = {"f32": em.F32, "f16": em.F16, "bf16": em.BF16, "q8_0": em.Q8_0, "q4_k": em.Q4_K}
BYTES = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q8_0": 34 / 32, "q4_k": 144 / 256}


def listed():
    return [
        # the smallest call there is: one token of the toy layer, launches and latency only
        dict(name="toy_f32_t1", shape="toy", type="f32", pack=False, T=1),
        # a prompt through an F32 layer, as the drop-in call of the tuned engine runs it
        dict(name="small_f32_t400", shape="small", type="f32", pack=False, T=400),
        # one user's decode step of a Mixtral-shaped layer: the weights of two experts from HBM
        dict(name="mixtral_q8_t1", shape="mixtral", type="q8_0", pack=True, T=1),
        # a batched decode step: nearly every expert hit, a few rows each
        dict(name="mixtral_q8_t13", shape="mixtral", type="q8_0", pack=True, T=13),
        # a short prompt through the drop-in call, which passes the GGUF rows and no pack
        dict(name="mixtral_q8_rows_t129", shape="mixtral", type="q8_0", pack=False, T=129),
        # a long prompt: the matrix cores' case
        dict(name="mixtral_q8_t2048", shape="mixtral", type="q8_0", pack=True, T=2048),
        # the 512-token prompt of the end-to-end model
        dict(name="mixtral_q4k_t512", shape="mixtral", type="q4_k", pack=True, T=512),
        # many small experts: one token, a batched decode step, a long prompt
        dict(name="qwen_q4k_t1", shape="qwen", type="q4_k", pack=True, T=1),
        dict(name="qwen_q4k_t48", shape="qwen", type="q4_k", pack=True, T=48),
        dict(name="qwen_q4k_t4096", shape="qwen", type="q4_k", pack=True, T=4096),
        # routed and shared experts with a selection bias: one token, a ragged prompt
        dict(name="deepseek_bf16_t1", shape="deepseek", type="bf16", pack=True, T=1),
        dict(name="deepseek_bf16_t1500", shape="deepseek", type="bf16", pack=True, T=1500),
    ]


def draw(rng):
    """A layer of one of the shapes in one of its encodings, with or without the pack, raw or renormalised
    gates, and for the bias router softmax or sigmoid scores; T spread over the logarithm of its range."""
    shape, types, t_max = rng.choice([
        ("toy", ["f32"], 1024),
        ("small", ["f32", "f16", "q8_0"], 768),
        ("mixtral", ["q8_0", "q4_k"], 1536),
        ("mixtral", ["q8_0", "q4_k", "bf16"], 256),
        ("qwen", ["q4_k", "q8_0", "bf16"], 4000),
        ("qwen_large", ["q4_k", "q8_0"], 1536),
        ("deepseek", ["bf16", "q8_0", "f16"], 2000),
    ])
    t = rng.choice(types)
    T = int(round(math.exp(rng.uniform(0.0, math.log(t_max)))))
    T = max(1, min(t_max, T + rng.choice([-1, 0, 0, 1])))
    c = dict(shape=shape, type=t, pack=t in ("q8_0", "q4_k", "bf16") and rng.random() < 0.75, T=T,
             renorm=rng.random() < 0.75)
    if shape == "deepseek":
        if t == "q8_0" or rng.random() < 0.5:  # the same layer without its bias, or with the sigmoid router
            c["sigmoid"] = rng.random() < 0.5
            c["bias"] = c["sigmoid"]
    return c


# ---- inputs

def _options(case):
    s = SHAPES[case["shape"]]
    sigmoid = bool(case.get("sigmoid", False))
    bias_std = s.get("bias_std", 0.0) if case.get("bias", True) else 0.0
    return s, bool(case.get("renorm", True)), sigmoid, (1.0 if sigmoid and bias_std else bias_std)


def _q8_0(w):
    """[n, 32 m] f32 -> Q8_0 bytes: per 32 values an fp16 scale and 32 signed bytes."""
    b = w.view(-1, 32)
    d = (b.abs().amax(1, keepdim=True) / 127.0).half()
    q = torch.round(b / d.float().clamp_min(1e-30)).clamp_(-127, 127).to(torch.int8)
    return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1).view(-1)


def _q4_k(w):
    """[n, 256 m] f32 -> Q4_K bytes: per 256 values fp16 d and dmin, eight 6-bit scales and mins, 128 nibble
    bytes."""
    b = w.view(-1, 8, 32)
    lo = b.amin(2).clamp_max(0.0)
    step = (b.amax(2) - lo) / 15.0
    d, dm = (step.amax(1, keepdim=True) / 63.0).half(), ((-lo).amax(1, keepdim=True) / 63.0).half()
    sc = torch.round(step / d.float().clamp_min(1e-30)).clamp_(0, 63)
    mn = torch.round(-lo / dm.float().clamp_min(1e-30)).clamp_(0, 63)
    scale, off = (d.float() * sc).unsqueeze(2).clamp_min(1e-30), (dm.float() * mn).unsqueeze(2)
    q = torch.round((b + off) / scale).clamp_(0, 15).to(torch.uint8).view(-1, 4, 2, 32)
    nib = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    s6 = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                    (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    return torch.cat([d.view(torch.uint8), dm.view(torch.uint8), s6, nib], 1).view(-1)


def _encode(w, t):
    if t == "f32":
        return w.reshape(-1).view(torch.uint8)
    if t == "f16":
        return w.half().reshape(-1).view(torch.uint8)
    if t == "bf16":
        return w.bfloat16().reshape(-1).view(torch.uint8)
    return _q8_0(w) if t == "q8_0" else _q4_k(w)


def _tensors(case, seed):
    """The layer's tensors as a GGUF upload leaves them, and the hidden states, from the seed alone."""
    s, _, _, bias_std = _options(case)
    d, f, E, t = s["d"], s["d_ff"], s["E"], case["type"]
    g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))

    def normal(*n, std=1.0):
        return torch.randn(*n, generator=g, device="cuda", dtype=torch.float32) * std

    def stack(experts, rows, cols):
        out = None
        per = max(1, (1 << 27) // (rows * cols))  # experts encoded at once
        for e in range(0, experts, per):
            n = min(per, experts - e)
            b = _encode(normal(n * rows, cols, std=0.02), t)
            if out is None:
                out = torch.empty(b.numel() // n * experts, dtype=torch.uint8, device="cuda")
            out[b.numel() // n * e:][:b.numel()] = b
        return out

    r = dict(x=normal(case["T"], d), router=normal(E, d, std=d ** -0.5))
    r.update(gate=stack(E, f, d), up=stack(E, f, d), down=stack(E, d, f))
    if bias_std:
        r["bias"] = normal(E, std=bias_std)
    fs = s.get("d_ff_shared", 0)
    if fs:
        r.update(gate_sh=stack(1, fs, d), up_sh=stack(1, fs, d), down_sh=stack(1, d, fs))
    return r


def prepare(case, seed):
    s, renorm, sigmoid, _ = _options(case)
    t = _tensors(case, seed)
    w = em.Layer()
    w.d, w.d_ff, w.E, w.k = s["d"], s["d_ff"], s["E"], s["k"]
    w.renorm, w.scoring = int(renorm), em.SCORE_SIGMOID if sigmoid else em.SCORE_SOFTMAX
    w.out_scale = 1.0
    w.groups_n = w.groups_top = 1
    ty = TYPES[case["type"]]
    w.router, w.gate, w.up, w.down = (t[n].data_ptr() for n in ("router", "gate", "up", "down"))
    w.gate_type = w.up_type = w.down_type = ty
    if "bias" in t:
        w.selection_bias = t["bias"].data_ptr()
    if "gate_sh" in t:
        w.d_ff_shared = s["d_ff_shared"]
        w.gate_shared, w.up_shared, w.down_shared = (t[n].data_ptr() for n in ("gate_sh", "up_sh", "down_sh"))
        w.gate_shared_type = w.up_shared_type = w.down_shared_type = ty
    if case["pack"]:
        t["pack"] = torch.empty(em.prefill_pack_bytes(w), dtype=torch.uint8, device="cuda")
        em.prefill_pack(w, t["pack"])
    need = em.scratch_bytes(w, case["T"])
    return dict(layer=w, tensors=t, x=t["x"], out=torch.empty_like(t["x"]),
                scratch=torch.empty(need, dtype=torch.uint8, device="cuda"))


def run(state):
    x = state["x"]
    st = em.moe_ffn(state["layer"], x, x.shape[0], state["out"], state["scratch"])
    if st:
        raise em.EmberError(st, "ember_moe_ffn")
    return state["out"]


# ---- what a pass cannot do without, and what it should give

def work(case):
    s = SHAPES[case["shape"]]
    d, f, E, k, T = s["d"], s["d_ff"], s["E"], s["k"], case["T"]
    fs = s.get("d_ff_shared", 0)
    hit = E * (1.0 - (1.0 - k / E) ** T)  # distinct experts of T tokens
    return {"bytes": (hit * 3 * d * f + 3 * d * fs) * BYTES[case["type"]] + E * d * 4 + 2 * T * d * 4,
            "flops": 2.0 * T * (k * 3 * d * f + 3 * d * fs) + 2.0 * T * E * d}


def tolerance(case):
    # about four times what the path shows against `exact`: F32 dots 1.8e-7 over all batch sizes; one token of
    # half stacks 1.9e-7 (f32 activations) and of Q8_0 4.5e-5 (int16 activations); batches of Q8_0 and half
    # stacks 5.1e-4 (fp16 operands); Q4_K 1.2e-3 (group factors held in fp16)
    t, one = case["type"], case["T"] == 1
    if t == "f32":
        return {"rel": 1e-6}
    if t == "q4_k":
        return {"rel": 5e-3}
    return {"rel": (2e-4 if t == "q8_0" else 1e-6) if one else 2e-3}


def _decode(raw, t):
    """f64 values of encoded rows."""
    if t == "f32":
        return raw.view(torch.float32).double()
    if t == "f16":
        return raw.view(torch.float16).double()
    if t == "bf16":
        return raw.view(torch.bfloat16).double()
    if t == "q8_0":
        b = raw.view(-1, 34)
        return (b[:, :2].contiguous().view(torch.float16).double() * b[:, 2:].contiguous().view(torch.int8).double()).view(-1)
    b = raw.view(-1, 144)
    d = b[:, :4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double() * d[:, :1]
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double() * d[:, 1:]
    q = b[:, 16:].view(-1, 4, 32)
    q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
    return (q * sc.unsqueeze(2) - mn.unsqueeze(2)).view(-1)


def _ffn(x, wg, wu, wd):
    g = x @ wg.t()
    return (g * torch.sigmoid(g) * (x @ wu.t())) @ wd.t()


def exact(case, seed):
    s, renorm, sigmoid, _ = _options(case)
    t = _tensors(case, seed)
    d, f, E, k, ty = s["d"], s["d_ff"], s["E"], s["k"], case["type"]
    x = t["x"].double()
    # the router's logits are f32 values by definition, and the picks are made on them
    logits = (x @ t["router"].double().t()).float().double()
    score = torch.sigmoid(logits) if sigmoid else torch.softmax(logits, 1)
    sel = score + t["bias"].double() if "bias" in t else logits
    idx = torch.topk(sel, k, dim=1).indices
    gate = torch.gather(score, 1, idx)
    if renorm:
        gate = gate / gate.sum(1, keepdim=True)
    out = torch.zeros_like(x)

    def mat(name, e, rows, cols):
        n = t[name].numel() // (1 if name.endswith("_sh") else E)
        return _decode(t[name][n * e:n * (e + 1)], ty).view(rows, cols)

    for e in range(E):
        tok, slot = torch.nonzero(idx == e, as_tuple=True)
        if tok.numel():
            y = _ffn(x[tok], mat("gate", e, f, d), mat("up", e, f, d), mat("down", e, d, f))
            out.index_add_(0, tok, y * gate[tok, slot].unsqueeze(1))
    fs = s.get("d_ff_shared", 0)
    if fs:
        out += _ffn(x, mat("gate_sh", 0, fs, d), mat("up_sh", 0, fs, d), mat("down_sh", 0, d, fs))
    return out
