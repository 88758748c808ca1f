"""What a user of this framework has it do, as cases that can be timed and checked.

The framework runs the decode step and the prompt pass of Llama-shaped models on
quantized weights: Q4_0 / Q5_0 / Q8_0 matrix-vector products with the work fused
around them, attention over an fp16 cache, the Q8_0 prefill GEMM on quantized
activations, attention over a prompt, and the reference-named calls on host
buffers.  The listed cases go from one small projection to four tokens of a 7B
model; draw() gives other sizes, layouts and block types of the same kinds.

Weights are N(0, 0.02^2) rows quantized to GGUF blocks, activations normal with
a few channels eight times larger (as a residual stream has them), caches N(0, 1).
"""

import ctypes
import math

import numpy as np
import torch

from asmllm_amd import native
from asmllm_amd.engine import STORIES_15M, DecodeEngine, LlamaShape

DEV = "cuda"
Q4, Q5, Q8 = native.Q4_0, native.Q5_0, native.Q8_0
EPS, THETA = 1e-5, 10000.0


def listed():
    return [
        # the k or v projection of a grouped-query layer: the smallest matvec a decode step has
        {"name": "matvec_q4_1024x4096", "kind": "matvec", "q": 4, "split": False, "M": 1024, "K": 4096},
        # a higher-precision projection at the size most weights of a 7B model have
        {"name": "matvec_q5_11008x4096", "kind": "matvec", "q": 5, "split": False, "M": 11008, "K": 4096},
        # the down projection cut over two ranks: K = 5504 is no multiple of 256
        {"name": "matvec_q8_4096x5504", "kind": "matvec", "q": 8, "split": False, "M": 4096, "K": 5504},
        # a decode FFN at the Llama-3 layer's sizes: RMSNorm, gate/up, SwiGLU, down
        {"name": "ffn_q4_14336", "kind": "ffn", "dim": 4096, "hidden": 14336},
        # decode attention of a grouped-query layer late in a long context
        {"name": "attn_gqa_8k", "kind": "attn", "heads": 32, "kv_heads": 8, "hd": 128, "max_ctx": 8192, "pos": 8000},
        # one head's attention over a prompt, fp32 as the reference's asm_attention has it
        {"name": "attention_1024x128", "kind": "prompt", "seq": 1024, "hd": 128},
        # a short prompt through one projection, weights as the GGUF file holds them
        {"name": "gemm_gguf_24", "kind": "gemm", "form": "gguf", "T": 24, "M": 4096, "K": 4096},
        # a ragged prompt through the down projection, the reference's split operands
        {"name": "gemm_split_200", "kind": "gemm", "form": "split", "T": 200, "M": 4096, "K": 11008},
        # a long prompt's chunk through gate or up, weights tiled once at load
        {"name": "gemm_tiled_512", "kind": "gemm", "form": "tiled", "T": 512, "M": 11008, "K": 4096},
        # the reference's own call on numpy buffers, as its Python runtime makes it
        {"name": "host_q4_4096x4096", "kind": "host", "q": 4, "M": 4096, "K": 4096, "threads": 4},
        # the reference's demo model, 32 greedy tokens from the start of a story
        {"name": "generate_15m", "kind": "generate", "dim": 288, "layers": 6, "heads": 6, "kv_heads": 6, "hidden": 768,
         "vocab": 32000, "q8_head": True, "max_ctx": 256, "pos": 0, "steps": 32},
        # four greedy tokens of a 7B model at context 2048
        {"name": "generate_7b", "kind": "generate", "dim": 4096, "layers": 32, "heads": 32, "kv_heads": 32,
         "hidden": 11008, "vocab": 32000, "q8_head": False, "max_ctx": 2176, "pos": 2044, "steps": 4},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "ffn", "attn", "attn", "prompt", "gemm", "gemm", "host", "generate"])
    if kind == "matvec":
        # projections of small and large models, whole or cut over ranks
        return {"kind": kind, "q": rng.choice([4, 4, 5, 8]), "split": rng.random() < 0.4,
                "M": _log(rng, 300, 33000), "K": _log(rng, 256, 14336, rng.choice([32, 64, 256, 256]))}
    if kind == "ffn":
        return {"kind": kind, "dim": _log(rng, 512, 8192, 256), "hidden": _log(rng, 1024, 16384, 64)}
    if kind == "attn":
        hd, kv = rng.choice([48, 64, 128, 128]), rng.choice([2, 4, 8, 8])
        max_ctx = _log(rng, 128, 16384)
        return {"kind": kind, "heads": kv * rng.choice([1, 2, 4, 4, 8]), "kv_heads": kv, "hd": hd, "max_ctx": max_ctx,
                "pos": rng.randrange(max_ctx // 2, max_ctx)}
    if kind == "prompt":
        return {"kind": kind, "seq": _log(rng, 64, 3000), "hd": rng.choice([48, 64, 80, 128])}
    if kind == "gemm":
        form = rng.choice(["gguf", "split", "tiled"])
        return {"kind": kind, "form": form, "T": _log(rng, 5, 600), "M": _log(rng, 500, 14336),
                "K": _log(rng, 512, 8192, 64)}
    if kind == "host":
        return {"kind": kind, "q": rng.choice([4, 8]), "M": _log(rng, 288, 8192), "K": _log(rng, 288, 8192, 32),
                "threads": rng.choice([1, 4, 8])}
    # small models of the same shape: few layers, so that rounding does not travel far
    hd, kv = rng.choice([48, 64, 128]), rng.choice([2, 3, 4, 8])
    heads = kv * rng.choice([1, 1, 2, 4])
    return {"kind": kind, "dim": hd * heads if hd * heads % 32 == 0 else 288, "layers": rng.randint(2, 6),
            "heads": heads if hd * heads % 32 == 0 else 6, "kv_heads": kv if hd * heads % 32 == 0 else 6,
            "hidden": _log(rng, 512, 4096, 64), "vocab": _log(rng, 2000, 33000), "q8_head": rng.random() < 0.5,
            "max_ctx": 512, "pos": rng.randrange(0, 450), "steps": rng.randint(8, 32)}


# ---- inputs ----------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _activations(g, *shape):
    """Normal rows with one channel in a hundred eight times larger."""
    x = _normal(g, *shape)
    hot = torch.rand(shape[-1], generator=g, device=DEV) < 0.01
    return torch.where(hot, 8 * x, x).contiguous()


def _half_bytes(d):
    return d.to(torch.float16).unsqueeze(-1).contiguous().view(torch.uint8)


def _quantize(w, q):
    """Rows to (d as fp16 [rows, nb], integer values [rows, nb, 32] before the offset is taken off)."""
    v = w.view(w.shape[0], -1, 32)
    if q == 8:
        d = v.abs().amax(-1) / 127
        return d.half(), torch.clamp(torch.round(v / d.clamp_min(1e-30).unsqueeze(-1)), -127, 127).to(torch.int16)
    z = 8 if q == 4 else 16
    top = torch.gather(v, 2, v.abs().argmax(-1, keepdim=True)).squeeze(-1)
    d = top / -z
    n = torch.floor(v / torch.where(d == 0, 1.0, d).unsqueeze(-1) + z + 0.5)
    return d.half(), torch.clamp(n, 0, 2 * z - 1).to(torch.int16)


def _weights(g, rows, K, q):
    """A weight matrix as its parts: {"d", "n"} (see _quantize), made a slice of rows at a time."""
    ds, ns = [], []
    step = max(1, (1 << 25) // K)
    for r in range(0, rows, step):
        d, n = _quantize(_normal(g, min(step, rows - r), K, std=0.02), q)
        ds.append(d)
        ns.append(n.to(torch.int8) if q == 8 else n.to(torch.uint8))
    return {"d": torch.cat(ds), "n": torch.cat(ns), "q": q}


def _planes(w):
    """The split layout's planes: qs (nibble pairs or int8), qh (Q5) and fp32 scales."""
    n, q = w["n"], w["q"]
    scales = w["d"].float().contiguous()
    if q == 8:
        return n.contiguous(), None, scales
    qs = (n[..., :16] & 15) | ((n[..., 16:] & 15) << 4)
    qh = None
    if q == 5:
        bit = (n >> 4).view(*n.shape[:2], 4, 8).to(torch.int32) << torch.arange(8, device=n.device, dtype=torch.int32)
        qh = bit.sum(-1).to(torch.uint8).contiguous()
    return qs.contiguous(), qh, scales


def _blocks(w):
    """GGUF blocks [rows, nb, 18 | 22 | 34]."""
    qs, qh, _ = _planes(w)
    parts = [_half_bytes(w["d"])] + ([qh] if qh is not None else []) + [qs.view(torch.uint8)]
    return torch.cat(parts, dim=-1).contiguous()


def _real(w):
    """The matrix in 64 bits."""
    z = {4: 8, 5: 16, 8: 0}[w["q"]]
    v = (w["n"].double() - z) * w["d"].double().unsqueeze(-1)
    return v.view(v.shape[0], -1)


def _interleaved(gate, up):
    """Gate and up rows in the order asmhip_matmul_swiglu reads them (groups of 8)."""
    H = gate["d"].shape[0]

    def mix(a, b):
        return torch.stack([a.view(H // 8, 8, *a.shape[1:]), b.view(H // 8, 8, *b.shape[1:])], 1).reshape(
            2 * H, *a.shape[1:])

    return {"d": mix(gate["d"], up["d"]), "n": mix(gate["n"], up["n"]), "q": gate["q"]}


def _inputs(case, seed):
    """The inputs of a case that has an exact() answer, as plain tensors."""
    g, k = _gen(seed), case["kind"]
    if k in ("matvec", "host"):
        return {"w": _weights(g, case["M"], case["K"], case["q"]), "x": _activations(g, case["K"])}
    if k == "ffn":
        d, h = case["dim"], case["hidden"]
        return {"x": _activations(g, d), "norm": 1 + 0.1 * _normal(g, d), "gate": _weights(g, h, d, 4),
                "up": _weights(g, h, d, 4), "down": _weights(g, d, h, 4)}
    if k == "attn":
        H, KV, hd, C = case["heads"], case["kv_heads"], case["hd"], case["max_ctx"]
        return {"qkv": _normal(g, (H + 2 * KV) * hd), "k": _normal(g, KV, C, hd).half(), "v": _normal(g, KV, C, hd).half()}
    if k == "prompt":
        return {n: _normal(g, case["seq"], case["hd"]) for n in ("q", "k", "v")}
    if k == "gemm":
        return {"w": _weights(g, case["M"], case["K"], 8), "x": _activations(g, case["T"], case["K"])}
    raise ValueError(k)


# ---- what a program holds before the call ---------------------------------------------------


def _empty(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device=DEV)


def prepare(case, seed):
    L, k = native.lib(), case["kind"]
    if k == "generate":
        shape = LlamaShape(dim=case["dim"], n_layers=case["layers"], n_heads=case["heads"], n_kv_heads=case["kv_heads"],
                           hidden_dim=case["hidden"], vocab=case["vocab"], eps=EPS, theta=THETA)
        if (case["dim"], case["layers"], case["hidden"]) == (STORIES_15M.dim, STORIES_15M.n_layers, STORIES_15M.hidden_dim):
            assert shape == STORIES_15M
        t = Q8 if case["q8_head"] else Q4
        eng = DecodeEngine(shape, max_ctx=case["max_ctx"], embed_type=t, output_type=t)
        eng.init_random(seed=int(seed) % 100003)
        # a serving program has its graphs before the first request
        eng.capture()
        return {"kind": k, "eng": eng, "token": int(seed) % case["vocab"], "pos": case["pos"], "steps": case["steps"]}

    v = _inputs(case, seed)
    s = {"kind": k, "case": dict(case), "L": L}
    if k == "matvec":
        M, K, q = case["M"], case["K"], case["q"]
        s.update(x=v["x"], y=_empty(M))
        if case["split"]:
            qs, qh, sc = _planes(v["w"])
            s["keep"] = (qs, qh, sc)
            ptrs = (qs, qh, sc) if q == 5 else (qs, sc)
            fn = {4: L.asmhip_matmul_q4_split, 5: L.asmhip_matmul_q5_split, 8: L.asmhip_matmul_q8_split}[q]
        else:
            b = _blocks(v["w"])
            s["keep"] = (b,)
            ptrs = (b,)
            fn = {4: L.asmhip_matmul_q4_0, 5: L.asmhip_matmul_q5_0, 8: L.asmhip_matmul_q8_0}[q]
        s["fn"], s["args"] = fn, [t.data_ptr() for t in ptrs] + [s["x"].data_ptr(), s["y"].data_ptr(), M, K]
    elif k == "ffn":
        s.update(x=v["x"], norm=v["norm"], gu=_blocks(_interleaved(v["gate"], v["up"])), down=_blocks(v["down"]),
                 h=_empty(case["hidden"]), work=_empty(2 * case["hidden"]), y=_empty(case["dim"]))
    elif k == "attn":
        H, hd, C = case["heads"], case["hd"], case["max_ctx"]
        s.update(qkv=v["qkv"], kc=v["k"], vc=v["v"], out=_empty(H, hd),
                 ws=_empty(max(1, int(L.asmhip_attention_decode_workspace(H, hd, C)))), table=_empty(C, hd),
                 pos=torch.full((1,), case["pos"], dtype=torch.int32, device=DEV))
        native.check(L.asmhip_rope_table(s["table"].data_ptr(), hd, C, ctypes.c_float(THETA), None))
    elif k == "prompt":
        s.update(q=v["q"], k=v["k"], v=v["v"], y=_empty(case["seq"], case["hd"]))
    elif k == "gemm":
        T, M, K = case["T"], case["M"], case["K"]
        s.update(x=v["x"], c=_empty(T, M))
        if case["form"] == "split":
            wq, _, ws = _planes(v["w"])
            s.update(wq=wq, ws=ws, aq=_empty(T, K, dtype=torch.int8), a_s=_empty(T, K // 32))
        else:
            b = _blocks(v["w"])
            if case["form"] == "tiled":
                t = _empty(int(L.asmhip_gemm_q8_0_tiled_weight_bytes(M, K)), dtype=torch.uint8)
                native.check(L.asmhip_gemm_q8_0_tile_weights(b.data_ptr(), t.data_ptr(), M, K, None))
                torch.cuda.synchronize()
                s.update(w=t, a=_empty(int(L.asmhip_gemm_q8_0_tiled_activation_bytes(T, K)), dtype=torch.uint8))
            else:
                s.update(w=b, a=_empty(T, K // 32, 34, dtype=torch.uint8))
    elif k == "host":
        qs, _, sc = _planes(v["w"])
        s.update(qs=qs.cpu().numpy(), sc=sc.cpu().numpy(), x=v["x"].cpu().numpy(), y=np.zeros(case["M"], np.float32))
        s["fn"] = L.asm_matmul_q4_mt if case["q"] == 4 else L.asm_matmul_q8_mt
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------------------------


def run(s):
    k = s["kind"]
    check = native.check
    if k == "generate":
        eng = s["eng"]
        tokens = eng.generate(s["token"], s["pos"], s["steps"])
        return {"tokens": np.array(tokens, np.int64), "logits": eng.logits.download(np.float32, (eng.shape.vocab,))}
    c, L = s["case"], s["L"]
    if k == "matvec":
        check(s["fn"](*s["args"], None))
        return s["y"]
    if k == "ffn":
        d, h = c["dim"], c["hidden"]
        check(L.asmhip_matmul_swiglu(Q4, s["gu"].data_ptr(), s["x"].data_ptr(), s["h"].data_ptr(), h, d,
                                     native.PRE_RMSNORM, s["norm"].data_ptr(), EPS, s["work"].data_ptr(), None))
        check(L.asmhip_matmul_fused(Q4, s["down"].data_ptr(), s["h"].data_ptr(), s["y"].data_ptr(), d, h,
                                    native.PRE_NONE, None, EPS, 0, None))
        return {"h": s["h"], "y": s["y"]}
    if k == "attn":
        check(L.asmhip_attention_decode_rope_table(s["qkv"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(),
                                                   s["ws"].data_ptr(), s["out"].data_ptr(), c["heads"], c["kv_heads"],
                                                   c["hd"], s["pos"].data_ptr(), c["max_ctx"], s["table"].data_ptr(),
                                                   None))
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    if k == "prompt":
        check(L.asmhip_attention(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["y"].data_ptr(), c["seq"],
                                 c["hd"], 1.0 / math.sqrt(c["hd"]), None))
        return s["y"]
    if k == "gemm":
        T, M, K = c["T"], c["M"], c["K"]
        if c["form"] == "split":
            check(L.asmhip_quantize_q8_split(s["x"].data_ptr(), s["aq"].data_ptr(), s["a_s"].data_ptr(), T, K, None))
            check(L.asmhip_gemm_q8_split(s["wq"].data_ptr(), s["ws"].data_ptr(), s["aq"].data_ptr(),
                                         s["a_s"].data_ptr(), s["c"].data_ptr(), T, M, K, None))
            return {"c": s["c"], "aq": s["aq"], "as": s["a_s"]}
        if c["form"] == "tiled":
            check(L.asmhip_quantize_q8_0_tiled(s["x"].data_ptr(), s["a"].data_ptr(), T, K, None))
            check(L.asmhip_gemm_q8_0_tiled(s["w"].data_ptr(), s["a"].data_ptr(), s["c"].data_ptr(), T, M, K, None))
        else:
            check(L.asmhip_quantize(Q8, s["x"].data_ptr(), s["a"].data_ptr(), T, K, None))
            check(L.asmhip_gemm_q8_0(s["w"].data_ptr(), s["a"].data_ptr(), s["c"].data_ptr(), T, M, K, None))
        return {"c": s["c"], "a": s["a"]}
    if k == "host":
        s["fn"](s["qs"].ctypes.data, s["sc"].ctypes.data, s["x"].ctypes.data, s["y"].ctypes.data, c["M"], c["K"],
                c["threads"])
        return s["y"]
    raise ValueError(k)


# ---- what a pass cannot do without ----------------------------------------------------------------

_BLOCK = {4: 18, 5: 22, 8: 34}
_SPLIT = {4: 20, 5: 24, 8: 36}


def work(case):
    k = case["kind"]
    if k in ("matvec", "host"):
        M, K, q = case["M"], case["K"], case["q"]
        per = (_SPLIT if k == "host" or case["split"] else _BLOCK)[q]
        return {"bytes": M * (K // 32) * per + 4 * K + 4 * M, "flops": 2 * M * K}
    if k == "ffn":
        d, h = case["dim"], case["hidden"]
        return {"bytes": 3 * h * d // 32 * 18 + 4 * (2 * d + 2 * h + d), "flops": 6 * h * d}
    if k == "attn":
        H, KV, hd, n = case["heads"], case["kv_heads"], case["hd"], case["pos"] + 1
        return {"bytes": 4 * KV * n * hd + 4 * (2 * H + 2 * KV) * hd, "flops": 4 * H * n * hd}
    if k == "prompt":
        s, hd = case["seq"], case["hd"]
        return {"bytes": 16 * s * hd, "flops": 4 * s * s * hd}
    if k == "gemm":
        T, M, K = case["T"], case["M"], case["K"]
        per = 36 if case["form"] == "split" else 34
        return {"bytes": M * (K // 32) * per + 4 * T * K + T * (K // 32) * per + 4 * T * M, "flops": 2 * T * M * K}
    d, h, n = case["dim"], case["hidden"], case["steps"]
    kv = d // case["heads"] * case["kv_heads"]
    per_layer = (d + 2 * kv + d + 2 * h) * d + d * h
    head = case["vocab"] * d
    weights = case["layers"] * per_layer * 18 // 32 + head * (34 if case["q8_head"] else 18) // 32
    ctx = sum(case["pos"] + i + 1 for i in range(n))
    return {"bytes": n * weights + case["layers"] * 4 * kv * ctx + n * 4 * case["vocab"],
            "flops": n * 2 * (case["layers"] * per_layer + head) + case["layers"] * 4 * d * ctx}


# ---- how far another correct implementation may be ----------------------------------------------------


def tolerance(case):
    """About four times what a correct path was seen to be off 64 bits, or, for whole
    engines, what two matvec kernels with differently ordered sums differ by."""
    k = case["kind"]
    if k in ("matvec", "host"):
        return {"rel": 6e-7, "max": 4e-6}  # fp32 sums: 1.3e-7, 6e-7 seen
    if k == "ffn":
        return {"rel": 1.2e-6, "max": 6e-6}  # two such sums and an exponential: 2.7e-7, 1e-6 seen
    if k == "attn":
        # fp32 softmax and sums: 2.5e-7, 1.5e-6 seen; the cache rows written are the same fp16 roundings
        return {"rel": 1e-6, "max": 6e-6}
    if k == "prompt":
        return {"rel": 4e-6, "max": 3e-5}  # the same over up to 3000 positions in one sum: 9e-7, 6e-6 seen
    if k == "gemm":
        return {"rel": 1.4e-6, "max": 1.2e-5}  # exact block dots, fp32 sums over blocks: 3.4e-7, 2.6e-6 seen
    # rounding travels through the layers, and through fp16 cache rows into later tokens: 9e-6, 3.8e-5 seen
    return {"rel": 4e-5, "max": 2e-4}


# ---- the same in 64 bits ---------------------------------------------------------------------------------


def _rotated(v, pos, hd):
    """Interleaved pairs rotated at pos, the angles in 64 bits."""
    i = torch.arange(hd // 2, device=v.device, dtype=torch.float32)
    e = torch.div(-2 * i, torch.full_like(i, hd)).double()  # the exponent is a 32-bit quotient by definition
    ang = pos * THETA**e
    a, b = v[..., 0::2], v[..., 1::2]
    return torch.stack([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1).reshape(v.shape)


def _q8_rows(x):
    """Q8_0 rows as the format's rule has them: d = amax / 127, q = rint(x * (127 / amax)), in fp32."""
    v = x.view(x.shape[0], -1, 32)
    amax = v.abs().amax(-1)
    # tensors on both sides of "/": a scalar on one side is turned into a product with a reciprocal
    full = torch.full_like(amax, 127.0)
    inv = torch.where(amax == 0, 0.0, torch.div(full, amax))
    n = torch.clamp(torch.round(v * inv.unsqueeze(-1)), -128, 127)
    return {"d": torch.div(amax, full).half(), "n": n.to(torch.int8), "q": 8}


def exact(case, seed):
    k = case["kind"]
    if k == "generate":
        return None
    v = _inputs(case, seed)
    if k in ("matvec", "host"):
        return _real(v["w"]) @ v["x"].double()
    if k == "ffn":
        x = v["x"].double()
        n = x / torch.sqrt((x * x).mean() + EPS) * v["norm"].double()
        g = _real(v["gate"]) @ n
        h = g / (1 + torch.exp(-g)) * (_real(v["up"]) @ n)
        return {"h": h, "y": _real(v["down"]) @ h}
    if k == "attn":
        H, KV, hd, pos = case["heads"], case["kv_heads"], case["hd"], case["pos"]
        qkv = v["qkv"].double()
        q = _rotated(qkv[: H * hd].view(H, hd), pos, hd)
        kk, vv = v["k"].double(), v["v"].double()
        kk[:, pos] = _rotated(qkv[H * hd : (H + KV) * hd].view(KV, hd), pos, hd).half().double()
        vv[:, pos] = qkv[(H + KV) * hd :].view(KV, hd).half().double()
        out = torch.empty(H, hd, dtype=torch.float64, device=DEV)
        for h in range(H):
            j = h // (H // KV)
            p = torch.softmax(kk[j, : pos + 1] @ q[h] / math.sqrt(hd), 0)
            out[h] = p @ vv[j, : pos + 1]
        return {"out": out, "k": None, "v": None}
    if k == "prompt":
        q, kk, vv = (v[n].double() for n in ("q", "k", "v"))
        return torch.softmax(q @ kk.t() / math.sqrt(case["hd"]), -1) @ vv
    if k == "gemm":
        return {"c": _real(_q8_rows(v["x"])) @ _real(v["w"]).t(), **{n: None for n in (("aq", "as") if case["form"] == "split" else ("a",))}}
    raise ValueError(k)
