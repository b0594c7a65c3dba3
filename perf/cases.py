"""The work this framework is used for, as cases to be timed: decode and prompt steps of every weight format it serves -- GGUF Q4_K_M,
16-bit safetensors, GPTQ 4-bit, a mixture of Q4_K experts over an e4m3 cache, and a layer-list model with recurrent state -- through
the models' public step functions, from one token behind a short context to a chunk of 4096 prompt tokens.

A model keeps the layer geometry of the benchmark (`bench.py`, `bench_legs.py`, `bench_hybrid.py`) and a quarter of its depth and of
its vocabulary, so that layers and output head keep their shares of a step; the experts' model keeps two layers (1.6 GB of experts).
Weights are random with the spread of a trained checkpoint's (a branch adds less than the stream it is added to)."""
import math
import random

import numpy as np
import torch

#: name -> hidden, heads, kv heads, head size, feed-forward, rotation base, norm epsilon, bias on q / k / v
GEOMETRY = {
    "1b": (2048, 16, 4, 128, 8192, 500000.0, 1e-5, False),
    "3b": (3072, 24, 8, 128, 8192, 500000.0, 1e-5, False),
    "7b": (3584, 28, 4, 128, 18944, 1000000.0, 1e-6, True),
    "8b": (4096, 32, 8, 128, 14336, 500000.0, 1e-5, False),
}
VOCAB, BLOCK, MAX_SEQ = 32000, 64, 16384
EXPERTS, TOP = 8, 2
GROUP = 128                                # GPTQ group
Q4K, Q6K = 12, 14                          # ggml type numbers
SPREAD = 0.012                             # of 16-bit weights


def case_of(family, mode, size, layers, batch, new, ctx, dtype="bf16", name=None):
    """batch sequences; decode: one new token each behind up to `ctx` tokens; prompt: `new` tokens in all, every sequence behind `ctx`"""
    c = {"family": family, "mode": mode, "size": size, "layers": layers, "batch": batch, "new": new, "ctx": ctx, "dtype": dtype}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a chat with a small model, the first words of an answer: launches and latency
        case_of("gguf", "decode", "1b", 8, 1, 1, 300, name="gguf_decode_small"),
        # one user, a long context: the headline workload of the benchmark
        case_of("gguf", "decode", "8b", 8, 1, 1, 4096, name="gguf_decode_1"),
        # a busy server: 32 sequences of unequal lengths
        case_of("gguf", "decode", "8b", 8, 32, 32, 4096, name="gguf_decode_32"),
        # a prompt of 2048 tokens
        case_of("gguf", "prompt", "8b", 8, 1, 2048, 0, name="gguf_prompt"),
        # 16-bit checkpoint, a few users
        case_of("bf16", "decode", "8b", 8, 8, 8, 3000, name="bf16_decode_8"),
        # three prompts of odd lengths admitted in one step
        case_of("bf16", "prompt", "8b", 8, 3, 3001, 0, name="bf16_prompt"),
        # 4-bit GPTQ, a moderate batch
        case_of("gptq", "decode", "7b", 7, 16, 16, 2500, name="gptq_decode_16"),
        # a prompt of ordinary length
        case_of("gptq", "prompt", "7b", 7, 1, 700, 0, name="gptq_prompt"),
        # mixture of experts, e4m3 cache, a busy server
        case_of("moe", "decode", "8b", 2, 32, 32, 4096, "fp8", name="moe_decode_32"),
        # the second chunk of a long prompt (chunked prefill)
        case_of("moe", "prompt", "8b", 2, 1, 4096, 4096, "fp8", name="moe_prompt_chunk"),
        # layer-list model with recurrent state: two prompts in one step, and a decoding batch
        case_of("hybrid", "prompt", "1b", 4, 2, 2100, 0, name="hybrid_prompt"),
        case_of("hybrid", "decode", "1b", 4, 8, 8, 2048, name="hybrid_decode_8"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    family = rng.choice(["gguf", "gguf", "bf16", "gptq", "moe", "hybrid"])
    mode = rng.choice(["decode", "prompt"])
    size = {"gptq": "7b", "moe": "8b"}.get(family) or rng.choice(["1b", "3b", "8b"] if family != "hybrid" else ["1b", "3b"])
    layers = {"gptq": 7, "moe": 2, "hybrid": 4}.get(family, 8)
    dtype = "fp8" if family == "moe" else rng.choice(["bf16", "bf16", "f32"]) if family == "hybrid" else "bf16"
    if mode == "decode":
        b = log(1, 8 if family == "hybrid" else 32)
        return case_of(family, mode, size, layers, b, b, log(64, 2048 if family == "hybrid" else 4096), dtype)
    new = log(17, 2048 if family in ("gguf", "hybrid") else 3000 if family == "bf16" else 700 if family == "gptq" else 4096)
    b = min(rng.choice([1, 1, 2, 3, 5]), max(1, new // 8))
    ctx = log(64, 4096) if family in ("gguf", "moe") and b == 1 and rng.random() < 0.3 else 0
    return case_of(family, mode, size, layers, b, new, ctx, dtype)


# ------------------------------------------------------------------------------------------------------------------- shapes of a case
def lengths(case):
    """-> (tokens cached before the pass, new tokens) per sequence"""
    r, n = random.Random("%(batch)d %(new)d %(ctx)d" % case), case["batch"]
    if case["mode"] == "decode":
        total = [case["ctx"]] + [r.randint(max(2, case["ctx"] // 16), case["ctx"]) for _ in range(n - 1)]
        return [t - 1 for t in total], [1] * n
    cuts = sorted(r.sample(range(1, case["new"]), n - 1)) if n > 1 else []
    return [case["ctx"]] * n, [b - a for a, b in zip([0] + cuts, cuts + [case["new"]])]


def blocks_of(case):
    return [-(-(a + b + 1) // BLOCK) for a, b in zip(*lengths(case))]      # the next token's place is there


def projections(case):
    """name -> (rows, columns) of one layer's matrices"""
    hid, H, G, D, ff = GEOMETRY[case["size"]][:5]
    return {"wq": (H * D, hid), "wk": (G * D, hid), "wv": (G * D, hid), "wo": (hid, H * D), "w1": (ff, hid), "w2": (hid, ff), "w3": (ff, hid)}


def type_of(case, name, layer):
    """the Q4_K_M mixture: output head Q6_K, value and down projections Q6_K on the layers that get more bits; experts' models all Q4_K"""
    n, n8 = case["layers"], case["layers"] // 8
    if name == "output":
        return Q6K
    if case["family"] == "gguf" and name in ("wv", "w2") and (layer < n8 or layer >= 7 * n8 or (layer - n8) % 3 == 2):
        return Q6K
    return Q4K


def hybrid_config(case):
    """windowed attention with a sink beside a gated delta rule, minGRU, the delta rule alone, and again both: the layer list of the benchmark"""
    hid, H, G, D, ff, base, eps, _ = GEOMETRY[case["size"]]
    att = {"dim": D, "heads": H, "kv_heads": G, "vdim": D, "scale": D ** -0.5, "mask": {"size": {"1b": 1024, "3b": 2048}[case["size"]]},
           "rot": {"base": base, "dims": D, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
    right = {"conv": 4, "dim": D, "heads": H, "kv_heads": H, "vdim": D}
    mlp = {"ff": ff, "kind": "dense", "limit": 7.0}
    both = {"type": "parallel", "mixer": {"left": att, "right": right, "left_scale": 1.0, "right_scale": 1.0}, "mlp": mlp}
    return {"architecture": "Sogodra", "norm": {"eps": eps}, "vocab": VOCAB, "width": hid,
            "layers": [both, {"type": "mingru", "mixer": {"width": 2 * hid}, "mlp": mlp}, {"type": "delta", "mixer": right, "mlp": mlp}, both]}


def hybrid_shapes(case, rank=64):
    cfg, sh = hybrid_config(case), {}
    W = cfg["width"]
    sh["embed"], sh["final.norm"], sh["head"] = (VOCAB, W), (W,), (VOCAB, W)

    def delta(p, c, low_rank):
        n = c["heads"] * c["dim"]
        for x in "qkv":
            sh[p + x], sh[p + x + ".conv"] = (n, W), (n, c["conv"])
        sh[p + "b"], sh[p + "A_log"], sh[p + "norm"], sh[p + "o"] = (c["heads"], W), (c["heads"],), (c["vdim"],), (W, n)
        if low_rank:
            sh[p + "a1"], sh[p + "a2"], sh[p + "dt_bias"], sh[p + "g1"], sh[p + "g2"] = (rank, W), (n, rank), (n,), (rank, W), (n, rank)
        else:
            sh[p + "a"], sh[p + "dt_bias"], sh[p + "g"] = (c["heads"], W), (c["heads"],), (n, W)
    for i, lc in enumerate(cfg["layers"]):
        p, m = "l%d." % i, lc["mixer"]
        if lc["type"] == "parallel":
            c, q = m["left"], p + "mix.left."
            sh[q + "q"], sh[q + "k"], sh[q + "v"] = (c["heads"] * c["dim"], W), (c["kv_heads"] * c["dim"], W), (c["kv_heads"] * c["vdim"], W)
            sh[q + "q.norm"], sh[q + "k.norm"], sh[q + "sink"], sh[q + "o"] = (c["dim"],), (c["dim"],), (c["heads"],), (W, c["heads"] * c["vdim"])
            delta(p + "mix.right.", m["right"], True)
        elif lc["type"] == "delta":
            delta(p + "mix.", m, False)
        else:
            w = m["width"]
            for x in "zxg":
                sh[p + "mix." + x] = (w, W)
            sh[p + "mix.z.b"], sh[p + "mix.x.b"], sh[p + "mix.o"] = (w,), (w,), (W, w)
        ff = lc["mlp"]["ff"]
        sh[p + "norm1"], sh[p + "norm2"] = (W,), (W,)
        sh[p + "mlp.gate"], sh[p + "mlp.up"], sh[p + "mlp.down"] = (ff, W), (ff, W), (W, ff)
    return sh


def work(case):
    old, new = lengths(case)
    T, n = sum(new), case["batch"]
    rows = T if case["mode"] == "decode" else n                        # rows of logits
    if case["family"] == "hybrid":
        cfg, sh = hybrid_config(case), hybrid_shapes(case)
        wide = 4 if case["dtype"] == "f32" else 2
        weights = sum(int(np.prod(s)) for k, s in sh.items() if k != "embed")
        layer = sum(int(np.prod(s)) for k, s in sh.items() if k not in ("embed", "head") and len(s) > 1)
        w = cfg["layers"][0]["mixer"]["left"]["mask"]["size"]
        hid, H, G, D = GEOMETRY[case["size"]][:4]
        pairs = sum(min(w, a + j + 1) for a, b in zip(old, new) for j in range(b))
        seen = sum(min(w - 1, a) + b for a, b in zip(old, new))
        state = n * (3 * H * D * D + 3 * 3 * 3 * H * D + 2 * hid) * 4
        return {"bytes": float(wide * (weights + 2 * 2 * G * D * seen + T * hid) + 2 * state + 4 * rows * VOCAB),
                "flops": float(2 * layer * T + 2 * VOCAB * hid * rows + 2 * 4 * D * H * pairs + 3 * T * H * 6 * D * D)}
    hid, H, G, D, ff = GEOMETRY[case["size"]][:5]
    bits = {"bf16": 16.0, "gptq": 4.0 + 16.0 / GROUP}
    weights = flops = 0.0
    used = min(EXPERTS, TOP * T) if case["family"] == "moe" else 1     # experts that some token selects (all of them from a few tokens on)
    for l in range(case["layers"]):
        for name, (r, k) in projections(case).items():
            ffn = name in ("w1", "w2", "w3") and case["family"] == "moe"
            per = bits.get(case["family"]) or (4.5 if type_of(case, name, l) == Q4K else 6.5625)
            weights += r * k * per / 8 * (used if ffn else 1)
            flops += 2.0 * r * k * T * (TOP if ffn else 1)
    weights += VOCAB * hid * (6.5625 if case["family"] in ("gguf", "moe") else 16.0) / 8
    flops += 2.0 * VOCAB * hid * rows
    pairs = sum(b * a + b * (b + 1) // 2 for a, b in zip(old, new))
    kv = sum(a + b for a, b in zip(old, new)) * 2 * G * D * case["layers"] * (1 if case["dtype"] == "fp8" else 2)
    return {"bytes": weights + kv + 4.0 * rows * VOCAB + 4.0 * T * hid, "flops": flops + 4.0 * D * H * pairs * case["layers"]}


def tolerance(case):
    """about four times what the step shows against 64 bits (measured over the listed and some eighty drawn cases); the 16-bit checkpoints'
    0.014 is what the design's rounding to bf16 behind every operator gives.  One step of e4m3 is an eighth."""
    if case["dtype"] == "f32":
        return {"rel": 1.2e-5, "max": 1e-4}
    if case["family"] == "moe":
        return {"rel": 0.03, "max": 0.4}
    return {"rel": {"gguf": 0.03, "bf16": 0.03, "gptq": 0.03, "hybrid": 0.02}[case["family"]], "max": 0.3}


# ------------------------------------------------------------------------------------------------------------------- values from a seed
class Source:
    """random tensors on the GPU, each from the seed and its own name: `prepare` and `exact` make the same ones in any order"""

    def __init__(self, seed):
        self.seed = int(seed)

    def gen(self, name):
        return torch.Generator(device="cuda").manual_seed((self.seed * 1000003 + sum((i + 1) * 131 * ord(c) for i, c in enumerate(name)) * 7919) & 0x7FFFFFFF)

    def normal(self, name, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=self.gen(name), device="cuda") * std + mean).to(dtype)

    def bytes(self, name, shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=self.gen(name))

    def quant(self, name, rows, k, kind):
        """GGUF blocks [rows, k / 256, 144 or 210] with random codes and sub-block scales, weights of spread 0.008"""
        n = 144 if kind == Q4K else 210
        b = self.bytes(name, (rows, k // 256, n))
        u = torch.rand((rows, k // 256, 1), generator=self.gen(name + ".d"), device="cuda") + 0.5

        def put(at, v):
            b[:, :, at:at + 2] = v.to(torch.float16).view(torch.uint8).view(rows, k // 256, 2)
        if kind == Q4K:
            put(0, 4e-5 * u)
            put(2, 3e-4 * u)
        else:
            put(208, 2.5e-6 * u * 4)
        return b


def tiles(b, kind):
    """GGUF blocks -> the 16-row x 256-column tiles that the library takes on the device"""
    nt, nkb = b.shape[0] // 16, b.shape[1]
    b = b.view(nt, 16, nkb, -1).transpose(1, 2)                        # [tile, k-block, row, bytes]
    if kind == Q4K:
        q = b[..., 16:].reshape(nt, nkb, 16, 2, 2, 4, 8).permute(0, 1, 3, 5, 2, 4, 6)
        return torch.cat([b[..., :16].reshape(nt, nkb, -1), q.reshape(nt, nkb, -1)], dim=2).contiguous().view(-1)
    ql = b[..., :128].reshape(nt, nkb, 16, 2, 2, 2, 4, 4).permute(0, 1, 3, 6, 2, 5, 4, 7)
    qh = b[..., 128:192].reshape(nt, nkb, 16, 4, 4, 4).permute(0, 1, 4, 2, 3, 5)
    parts = [b[..., 192:208], ql, qh, b[..., 208:210]]
    return torch.cat([p.reshape(nt, nkb, -1) for p in parts], dim=2).contiguous().view(-1)


def dequantised(b, kind):
    """GGUF blocks -> f64 [rows, k]"""
    def half(at):
        return b[:, :, at:at + 2].contiguous().view(torch.float16).double()
    rows, nkb = b.shape[:2]
    if kind == Q4K:
        s = b[:, :, 4:16].long()
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], dim=2)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], dim=2)
        qs = b[:, :, 16:].view(rows, nkb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], dim=3).reshape(rows, nkb, 8, 32)
        return ((half(0) * sc)[..., None] * q - (half(2) * mn)[..., None]).reshape(rows, -1)
    ql, qh = b[:, :, :128].view(rows, nkb, 2, 2, 32), b[:, :, 128:192].view(rows, nkb, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], dim=3)
    hi = torch.cat([(qh >> (2 * t)) & 3 for t in range(4)], dim=3)
    q = (lo | (hi << 4)).double() - 32
    sc = b[:, :, 192:208].contiguous().view(torch.int8).double().view(rows, nkb, 2, 4, 2, 1)
    return (half(208)[..., None, None, None] * (sc * q.view(rows, nkb, 2, 4, 2, 16))).reshape(rows, -1)


def gptq_codes(src, name, n, k):
    """(packed codes [k / 8, n] int32, scales [k / group, n] bf16): bell-shaped codes around 8, weights of spread 0.009"""
    c = (torch.randn((k // 8, 8, n), generator=src.gen(name), device="cuda") * 2.5 + 8.5).clamp_(0, 15.5).to(torch.int32)
    q = c[:, 0].clone()
    for i in range(1, 8):
        q |= c[:, i] << (4 * i)
    return q, (0.002 + 0.003 * torch.rand((k // GROUP, n), generator=src.gen(name + ".s"), device="cuda")).to(torch.bfloat16)


def weight64(case, src, name, layer, rows, k):
    """one projection as the model's format holds it, f64 [rows, k]"""
    key = "%d.%s" % (layer, name)
    if case["family"] == "bf16" or (case["family"] == "gptq" and name == "output"):
        return src.normal(key, (rows, k), SPREAD).double()
    if case["family"] == "gptq":
        q, s = gptq_codes(src, key, rows, k)
        c = torch.stack([(q >> (4 * i)) & 15 for i in range(8)], dim=1).view(k, rows).double() - 8
        return (c.view(k // GROUP, GROUP, rows) * s.double()[:, None]).view(k, rows).t()
    kind = type_of(case, name.split("#")[0], layer)
    return dequantised(src.quant(key, rows, k, kind), kind)


def norm_weight(src, name, n):
    return src.normal(name, (n,), 0.02, 1.0)


def embedding(case, src):
    hid = GEOMETRY[case["size"]][0]
    if case["family"] == "gguf":
        return src.normal("embed", (VOCAB, hid), 0.02, dtype=torch.float32)
    if case["family"] == "moe":                                        # a token carries what its two experts answer to
        u, r = experts(src, hid), torch.rand((VOCAB, EXPERTS), generator=src.gen("choice"), device="cuda").argsort(dim=1)
        return src.normal("embed", (VOCAB, hid), 0.3, dtype=torch.float32) + 0.2 * (u[r[:, 0]] + 0.9 * u[r[:, 1]])
    return src.normal("embed", (VOCAB, hid), 0.5)


def experts(src, hid):
    """the direction that every expert answers to: as in a trained router, the choice stands well clear of rounding"""
    return src.normal("experts", (EXPERTS, hid), dtype=torch.float32)


def router(src, layer, hid):
    return 0.0025 * experts(src, hid) + src.normal("%d.router" % layer, (EXPERTS, hid), 0.0005, dtype=torch.float32)


def hybrid_tensor(src, name, shape):
    last = name.split(".")[-1]
    if last.startswith("norm"):
        return norm_weight(src, name, shape[0])
    if name == "embed":
        return src.normal(name, shape)
    if name.endswith(".A_log"):
        return src.normal(name, shape, 0.5, -0.5)
    return src.normal(name, shape, 0.5 if last == "conv" else 0.3 if len(shape) == 1 else shape[-1] ** -0.5)


def cache_shape(case, which, blocks):
    G, D = GEOMETRY[case["size"]][2:4]
    x = 16 if case["dtype"] == "fp8" else 8
    return (blocks, G, D // x, BLOCK, x) if which == 0 else (blocks, G, D, BLOCK)


def cache_values(case, src, layer, which, blocks):
    """what earlier steps left in the pages; zeros where the pass starts from nothing"""
    shape = cache_shape(case, which, blocks)
    if case["mode"] == "prompt" and case["ctx"] == 0:
        t = torch.zeros(shape, dtype=torch.bfloat16, device="cuda")
    else:
        t = src.normal("kv%d.%d" % (layer, which), shape)
    return t.to(torch.float8_e4m3fn) if case["dtype"] == "fp8" else t


def inputs(case, src):
    """tokens of the pass and the block engine's step description, as numpy"""
    old, new = lengths(case)
    nb = blocks_of(case)
    order = torch.randperm(sum(nb), generator=src.gen("blocks"), device="cuda").cpu().numpy()
    bt, at = np.zeros((len(nb), max(nb)), np.uint32), 0
    for i, k in enumerate(nb):
        bt[i, :k] = order[at:at + k]
        at += k
    cu = np.concatenate([[0], np.cumsum(new)]).astype(np.uint32)
    seq = np.repeat(np.arange(len(new)), new)
    pos = np.concatenate([np.arange(a, a + b) for a, b in zip(old, new)]).astype(np.int64)
    tok = torch.randint(0, VOCAB, (int(cu[-1]),), generator=src.gen("tokens"), device="cuda").cpu().numpy()
    return {"input_ids": tok.astype(np.uint32), "positions": pos, "slot_mapping": bt[seq, pos // BLOCK].astype(np.int64) * BLOCK + pos % BLOCK,
            "block_tables": bt, "context_lens": np.asarray([a + b for a, b in zip(old, new)], np.uint32), "cu_seqlens_q": cu,
            "cu_seqlens_k": np.concatenate([[0], np.cumsum([a + b for a, b in zip(old, new)])]).astype(np.uint32),
            "max_seqlen_q": max(new), "max_context_len": max(a + b for a, b in zip(old, new))}


# ------------------------------------------------------------------------------------------------------------------- the models
class DeviceArray:
    """device memory that a model owns, as torch takes it; the model stays as long as a tensor over it does"""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": kind, "version": 2}


def view(owner, ptr, shape, dtype):
    kind = {torch.float32: "<f4", torch.bfloat16: "<i2", torch.float8_e4m3fn: "|u1"}[dtype]
    return torch.as_tensor(DeviceArray(owner, ptr, shape, kind), device="cuda").view(dtype)


def gguf_model(case, src):
    from candle_vllm_amd import model as M
    hid, H, G, D, ff, base, eps, _ = GEOMETRY[case["size"]]
    cfg = M.ModelDims(hidden=hid, n_layers=case["layers"], n_heads=H, n_kv_heads=G, head_dim=D, intermediate=ff, vocab=VOCAB, rms_eps=eps,
                      rope_theta=base, max_seq=MAX_SEQ, block_size=BLOCK)
    moe = case["family"] == "moe"
    if moe:
        cfg.n_expert, cfg.n_expert_used = EXPERTS, TOP
    m = M.GGUFLLaMa(cfg, max_batch=case["batch"], max_blocks_per_seq=max(blocks_of(case)), kv_layout=M.KV_PAGED_FP8 if case["dtype"] == "fp8" else M.KV_PAGED)

    def f32(layer, which, t):
        a = np.ascontiguousarray(t.float().cpu().numpy())
        M._check(M.lib.mi355_llama_set_f32(m.h, layer, which, a.ctypes.data, a.size), "set_f32")

    def matrix(layer, which, name, rows, k):
        kind = type_of(case, name, layer)
        t = tiles(src.quant("%d.%s" % (layer, name), rows, k, kind), kind)
        m._keep.append(t)
        M._check(M.lib.mi355_llama_set_qweight_tiles(m.h, layer, which, kind, t.data_ptr(), rows, k), "set_qweight_tiles")
    f32(-1, M.W_TOK_EMBD, embedding(case, src))
    f32(-1, M.W_OUTPUT_NORM, norm_weight(src, "norm", hid))
    matrix(-1, M.W_OUTPUT, "output", VOCAB, hid)
    slots = {"wq": M.W_WQ, "wk": M.W_WK, "wv": M.W_WV, "wo": M.W_WO, "w1": M.W_W1, "w2": M.W_W2, "w3": M.W_W3}
    for l in range(case["layers"]):
        f32(l, M.W_ATTN_NORM, norm_weight(src, "%d.n1" % l, hid))
        f32(l, M.W_FFN_NORM, norm_weight(src, "%d.n2" % l, hid))
        if moe:
            f32(l, 12, router(src, l, hid))
        for name, (r, k) in projections(case).items():
            if moe and name in ("w1", "w2", "w3"):
                for e in range(EXPERTS):
                    b = src.quant("%d.%s#%d" % (l, name, e), r, k, Q4K).cpu().numpy()
                    M._check(M.lib.mi355_llama_set_moe_expert(m.h, l, slots[name], e, Q4K, b.ctypes.data, r, k), "set_moe_expert")
            else:
                matrix(l, slots[name], name, r, k)
    return m, M.lib.mi355_llama_kv_ptr, M.lib.mi355_llama_logits_ptr


def dense_model(case, src):
    from types import SimpleNamespace
    from candle_vllm_amd import dense_model as DM
    hid, H, G, D, ff, base, eps, bias = GEOMETRY[case["size"]]
    cfg = SimpleNamespace(hidden=hid, n_layers=case["layers"], n_heads=H, n_kv_heads=G, head_dim=D, intermediate=ff, vocab=VOCAB, rms_eps=eps,
                          rope_theta=base, max_seq=MAX_SEQ, block_size=BLOCK, qkv_bias=bias, layer_norm=False, rotary_dim=0, kv_fp8=False)
    m = DM.DenseLlama(cfg, max_batch=case["batch"], max_blocks_per_seq=max(blocks_of(case)), kv_layout=DM.KV_PAGED)

    def put(layer, slot, t):
        DM._check(DM.lib.mi355_dense_set_weight_dev(m.h, layer, DM.W_SLOTS[slot], t.data_ptr(), t.numel()), slot)
        torch.cuda.synchronize()
    put(-1, "tok_embd", embedding(case, src))
    put(-1, "output_norm", norm_weight(src, "norm", hid))
    put(-1, "output", src.normal("-1.output", (VOCAB, hid), SPREAD))
    for l in range(case["layers"]):
        put(l, "attn_norm", norm_weight(src, "%d.n1" % l, hid))
        put(l, "ffn_norm", norm_weight(src, "%d.n2" % l, hid))
        for name, (r, k) in projections(case).items():
            key = "%d.%s" % (l, name)
            if case["family"] == "gptq":
                q, s = gptq_codes(src, key, r, k)
                m.set_gptq(l, name, q.cpu().numpy().view(np.uint32), s.float().cpu().numpy(), GROUP)
            else:
                put(l, name, src.normal(key, (r, k), SPREAD))
            if bias and name in ("wq", "wk", "wv"):
                put(l, "b" + name[1], src.normal(key + ".b", (r,), 0.1))
    return m, DM.lib.mi355_dense_kv_ptr, DM.lib.mi355_dense_logits_ptr


def hybrid_model(case, src, slots):
    from candle_vllm_amd import hybrid_model as hm
    cfg, shapes = hybrid_config(case), hybrid_shapes(case)
    spec = hm.SPECS[cfg["architecture"]](cfg, shapes)
    m = hm.HybridModel(spec, dtype="float32" if case["dtype"] == "f32" else "bfloat16", block_size=BLOCK, state_slots=slots)

    def put(layer, which, names):
        axis = 1 if which == hm.HW_OUT_PROJ and len(names) > 1 else 0
        ts = [hybrid_tensor(src, n, shapes[n]) if n else None for n in names]
        if which == hm.HW_IN_BIAS:
            rows = [shapes[n][0] for n in spec.slots[layer][hm.HW_IN_PROJ]]
            ts = [torch.zeros(r, dtype=torch.bfloat16, device="cuda") if t is None else t for t, r in zip(ts, rows)]
        t = torch.cat([x if axis else x.reshape(-1) for x in ts], dim=axis).contiguous()
        st = torch.cuda.current_stream().cuda_stream
        hm._check(hm.lib.mi355_hybrid_set_weight_dev(m.h, layer, which, t.data_ptr(), t.numel(), st), "set_weight_dev")
        torch.cuda.synchronize()
    for which, name in {hm.HW_EMBED: "embed", hm.HW_FINAL_NORM: "final.norm", hm.HW_HEAD: "head"}.items():
        put(-1, which, [name])
    for i, s in enumerate(spec.slots):
        for which, names in s.items():
            put(i, which, names)
    m.alloc_cache(sum(blocks_of(case)))
    floats = int(hm.lib.mi355_hybrid_state_floats_per_slot(m.h))
    return m, view(m, hm.lib.mi355_hybrid_state_ptr(m.h), (slots, floats), torch.float32)


def prepare(case, seed):
    src = Source(seed)
    meta = inputs(case, src)
    if case["family"] == "hybrid":
        n = case["batch"]
        m, state = hybrid_model(case, src, n)
        state.zero_()
        old, _ = lengths(case)
        for i in range(n if case["mode"] == "decode" else 0):          # the prompts that the decoding sequences stand behind
            one = dict(case, mode="prompt", batch=1, new=old[i], ctx=0)
            p = inputs(one, src)
            p["input_ids"] = history(src, i, old[i]).cpu().numpy().astype(np.uint32)
            p["block_tables"] = meta["block_tables"][i:i + 1]
            p["slot_mapping"] = p["block_tables"][0, p["positions"] // BLOCK].astype(np.int64) * BLOCK + p["positions"] % BLOCK
            m.step(p, [i])
        return {"case": case, "model": m, "meta": meta, "slots": list(range(n)), "state": state}
    m, kv_ptr, logits_ptr = (gguf_model if case["family"] in ("gguf", "moe") else dense_model)(case, src)
    blocks = sum(blocks_of(case))
    m.alloc_kv_cache(blocks)
    kv = []
    for l in range(case["layers"]):
        for which in (0, 1):
            t = cache_values(case, src, l, which, blocks)
            kv.append(view(m, kv_ptr(m.h, l, which), t.shape, t.dtype))
            kv[-1].copy_(t)
    if hasattr(m, "finalize"):
        m.finalize()
    s = {"case": case, "model": m, "meta": meta, "kv": kv}
    if case["mode"] == "decode":
        m.set_graph(True)
        s["stream"] = torch.cuda.Stream()
        torch.cuda.synchronize()
        s["logits_ptr"], s["capacity"] = logits_ptr, max(blocks_of(case)) * BLOCK
    torch.cuda.synchronize()
    return s


def run(state):
    """a decode step as the engine runs it after a change of the batch (inputs in, one step, tokens out), or one prompt step.  The sampled
    token is the largest logit's index; pages and recurrent state are returned as the model holds them."""
    case, m, meta = state["case"], state["model"], state["meta"]
    if case["family"] == "hybrid":
        return {"logits": m.step(meta, state["slots"]), "state": state["state"]}
    if case["mode"] == "decode":
        st = state["stream"].cuda_stream
        m.decode_begin(meta["input_ids"], meta["context_lens"], meta["block_tables"], state["capacity"], st)
        m.decode_step(st)
        m.read_tokens(st)
        if "logits" not in state:
            state["logits"] = view(m, state["logits_ptr"](m.h), (case["batch"], VOCAB), torch.float32)
        return {"logits": state["logits"], "kv": state["kv"]}
    if case["family"] in ("gguf", "moe"):
        return {"logits": m.forward_prefill(meta), "kv": state["kv"]}
    return {"logits": m.forward(meta, is_prefill=True), "kv": state["kv"]}


# ------------------------------------------------------------------------------------------------------------------- in 64 bits
def history(src, i, n):
    """the tokens that decoding sequence i of a recurrent model has behind it"""
    return torch.randint(0, VOCAB, (n,), generator=src.gen("history%d" % i), device="cuda")


def rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def attend(q, k, v, first, scale, window=0, sink=None):
    """q [T, H, d] at positions first .. ; k, v [S, G, d] at positions 0 ..  -> [T, H, vd]"""
    T, H, S, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    out = torch.empty((T, H, v.shape[2]), dtype=torch.float64, device=q.device)
    gap = torch.arange(first, first + T, device=q.device)[:, None] - torch.arange(S, device=q.device)[None, :]
    hide = (gap < 0) | (gap >= window) if window else gap < 0
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h] @ k[:, g].t() * scale).masked_fill_(hide, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].double().expand(T, 1)], dim=1)
        p = torch.softmax(s, dim=1)
        out[:, h] = p[:, :S] @ v[:, g]
    return out


def llama_exact(case, src):
    hid, H, G, D, ff, base, eps, bias = GEOMETRY[case["size"]]
    meta, (old, new) = inputs(case, src), lengths(case)
    blocks, pairs = sum(blocks_of(case)), case["family"] in ("gguf", "moe")
    pos = torch.from_numpy(meta["positions"]).cuda()
    slot = torch.from_numpy(meta["slot_mapping"]).cuda()
    ang = pos.double()[:, None] * base ** (-torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)[None]
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    T, x16 = len(pos), 16 if case["dtype"] == "fp8" else 8

    def rotate(t):
        a, b = (t[..., 0::2], t[..., 1::2]) if pairs else (t[..., :D // 2], t[..., D // 2:])
        u, w = a * cos - b * sin, b * cos + a * sin
        return torch.stack([u, w], dim=-1).flatten(-2) if pairs else torch.cat([u, w], dim=-1)

    def mul(t, name, layer, rows, k):
        return t @ weight64(case, src, name, layer, rows, k).t()
    x = embedding(case, src)[torch.from_numpy(meta["input_ids"].astype(np.int64)).cuda()].double()
    kv, P = [], projections(case)
    for l in range(case["layers"]):
        h = rms(x, norm_weight(src, "%d.n1" % l, hid), eps)
        q, k, v = (mul(h, n, l, *P[n]) + (src.normal("%d.%s.b" % (l, n), (P[n][0],), 0.1).double() if bias else 0.0) for n in ("wq", "wk", "wv"))
        q, k, v = rotate(q.view(T, H, D)), rotate(k.view(T, G, D)), v.view(T, G, D)
        if case["dtype"] == "fp8":                                     # the cache's format is part of what is asked for
            k, v = (t.float().to(torch.bfloat16).to(torch.float8_e4m3fn).double() for t in (k, v))
        kc = cache_values(case, src, l, 0, blocks).double().permute(0, 3, 1, 2, 4).reshape(blocks * BLOCK, G, D)
        vc = cache_values(case, src, l, 1, blocks).double().permute(0, 3, 1, 2).reshape(blocks * BLOCK, G, D)
        kc[slot], vc[slot] = k, v
        kv += [kc.view(blocks, BLOCK, G, D // x16, x16).permute(0, 2, 3, 1, 4).float(), vc.view(blocks, BLOCK, G, D).permute(0, 2, 3, 1).float()]
        y, at = [], 0
        for i, (a, b) in enumerate(zip(old, new)):
            rows = (torch.from_numpy(meta["block_tables"][i].astype(np.int64)).cuda()[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).view(-1)[:a + b]
            y.append(attend(q[at:at + b], kc[rows], vc[rows], a, D ** -0.5))
            at += b
        x = x + mul(torch.cat(y).reshape(T, H * D), "wo", l, *P["wo"])
        h = rms(x, norm_weight(src, "%d.n2" % l, hid), eps)
        if case["family"] == "moe":
            p = torch.softmax(h @ router(src, l, hid).double().t(), dim=1)
            top, ids = p.topk(TOP, dim=1)
            top = top / top.sum(1, keepdim=True)
            add = torch.zeros_like(x)
            for e in range(EXPERTS):
                t, j = (ids == e).nonzero(as_tuple=True)
                w = [weight64(case, src, "%s#%d" % (n, e), l, *P[n]).t() for n in ("w1", "w3", "w2")]
                add[t] += top[t, j][:, None] * ((torch.nn.functional.silu(h[t] @ w[0]) * (h[t] @ w[1])) @ w[2])
            x = x + add
        else:
            x = x + mul(torch.nn.functional.silu(mul(h, "w1", l, *P["w1"])) * mul(h, "w3", l, *P["w3"]), "w2", l, *P["w2"])
    if case["mode"] == "prompt":
        x = x[torch.from_numpy(meta["cu_seqlens_q"][1:].astype(np.int64) - 1).cuda()]
    return {"logits": mul(rms(x, norm_weight(src, "norm", hid), eps), "output", -1, VOCAB, hid), "kv": kv}


def hybrid_exact(case, src):
    cfg, shapes = hybrid_config(case), hybrid_shapes(case)
    eps, silu, sig = cfg["norm"]["eps"], torch.nn.functional.silu, torch.sigmoid
    W = {n: hybrid_tensor(src, n, s).double() for n, s in shapes.items()}

    def conv(x, w):
        taps = w.shape[1]
        xp = torch.cat([x.new_zeros((taps - 1, x.shape[1])), x])
        return silu(sum(w[:, i] * xp[i:i + len(x)] for i in range(taps)))

    def delta(p, c, h, low_rank):
        T, H, d, vd = len(h), c["heads"], c["dim"], c["vdim"]
        q, k, v = (conv(h @ W[p + n].t(), W[p + n + ".conv"]).view(T, H, -1) for n in "qkv")
        q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        beta, a = sig(h @ W[p + "b"].t()), -torch.exp(W[p + "A_log"])
        soft = torch.nn.functional.softplus
        if low_rank:
            g = torch.exp(a[:, None] * soft((h @ W[p + "a1"].t() @ W[p + "a2"].t() + W[p + "dt_bias"]).view(T, H, d), threshold=1e9))
            gate = sig(h @ W[p + "g1"].t() @ W[p + "g2"].t())
        else:
            g = torch.exp(a * soft(h @ W[p + "a"].t() + W[p + "dt_bias"], threshold=1e9))[..., None].expand(T, H, d)
            gate = silu(h @ W[p + "g"].t())
        S, o = h.new_zeros((H, d, vd)), h.new_empty((T, H, vd))
        g, kc, q = g[..., None].contiguous(), k[..., None].contiguous(), q.unsqueeze(2) * d ** -0.5
        kr = k.unsqueeze(2).contiguous()
        for t in range(T):
            S = S * g[t]
            S = torch.baddbmm(S, kc[t], beta[t][:, None, None] * (v[t].unsqueeze(1) - torch.bmm(kr[t], S)))
            o[t] = torch.bmm(q[t], S)[:, 0]
        return (rms(o, W[p + "norm"], eps) * gate.view(T, H, vd)).view(T, -1) @ W[p + "o"].t()

    def attention(p, c, h):
        T, H, G, d = len(h), c["heads"], c["kv_heads"], c["dim"]
        q, k, v = ((h @ W[p + n].t()).view(T, -1, d) for n in "qkv")
        q, k = rms(q, W[p + "q.norm"], eps), rms(k, W[p + "k.norm"], eps)
        r, sc = c["rot"], c["rot"]["scaling"]
        f = r["base"] ** (-torch.arange(0, r["dims"], 2, dtype=torch.float64, device="cuda") / r["dims"])
        turns = sc["original"] * f / (2 * math.pi)                     # turns over the original length
        mix = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        f = mix * f + (1 - mix) * f / sc["factor"]
        ang = torch.arange(T, dtype=torch.float64, device="cuda")[:, None] * f
        cos, sin = ang.cos()[:, None], ang.sin()[:, None]
        q, k = (torch.cat([t[..., :d // 2] * cos - t[..., d // 2:] * sin, t[..., d // 2:] * cos + t[..., :d // 2] * sin], dim=-1) for t in (q, k))
        return attend(q, k, v, 0, c["scale"], c["mask"]["size"], W[p + "sink"]).reshape(T, -1) @ W[p + "o"].t()

    def mingru(p, h):
        z, u = sig(h @ W[p + "z"].t() + W[p + "z.b"]), h @ W[p + "x"].t() + W[p + "x.b"]
        c, S, out = torch.where(u >= 0, u + 0.5, sig(u)), h.new_zeros(u.shape[1]), torch.empty_like(u)
        for t in range(len(h)):
            S = torch.lerp(S, c[t], z[t])
            out[t] = S
        return (out * silu(h @ W[p + "g"].t())) @ W[p + "o"].t()

    def forward(tokens):
        x = W["embed"][tokens]
        for i, lc in enumerate(cfg["layers"]):
            p, m = "l%d." % i, lc["mixer"]
            if lc["type"] == "parallel":
                y = attention(p + "mix.left.", m["left"], x) + delta(p + "mix.right.", m["right"], x, True)
            elif lc["type"] == "delta":
                y = delta(p + "mix.", m, x, False)
            else:
                y = mingru(p + "mix.", x)
            x = x + rms(y, W[p + "norm1"], eps)
            g, u, lim = x @ W[p + "mlp.gate"].t(), x @ W[p + "mlp.up"].t(), lc["mlp"]["limit"]
            g = g.clamp(max=lim)
            x = x + rms((g * sig(1.702 * g) * (u.clamp(-lim, lim) + 1)) @ W[p + "mlp.down"].t(), W[p + "norm2"], eps)
        return rms(x[-1:], W["final.norm"], eps) @ W["head"].t()
    meta, (old, _) = inputs(case, src), lengths(case)
    tok, cu, out = torch.from_numpy(meta["input_ids"].astype(np.int64)).cuda(), meta["cu_seqlens_q"], []
    for i in range(case["batch"]):
        t = tok[int(cu[i]):int(cu[i + 1])]
        out.append(forward(torch.cat([history(src, i, old[i]), t]) if case["mode"] == "decode" else t))
    return {"logits": torch.cat(out), "state": None}                    # the state pool's order is the model's own


def exact(case, seed):
    src = Source(seed)
    with torch.no_grad():
        return hybrid_exact(case, src) if case["family"] == "hybrid" else llama_exact(case, src)
