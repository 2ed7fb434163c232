"""Performance cases: the work that programs built on this framework give it, through its public entry points.

Every case is one pass of one path on the current stream, at a size a program meets in use: single small launches, the
row kernels, dense and odd-sized matrix products, block-scaled products, attention over a prompt and over a cache, a
mixture-of-experts product, the greedy LM head, and whole transformer blocks for one token and for a prompt.  ``listed()``
holds one representative of each, ``draw()`` spreads over the ranges they stand for.
"""
import math

import torch

from __graft_entry__ import load_package

ct = load_package()

EPS = 1e-6
HEAD_DIM = 128
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
MOST_GEMM_FLOPS = 2.0 * 8192 ** 3                        # no drawn matrix product costs more than the largest listed one
MOST_ATTENTION_FLOPS = 2.0 * 4 * 32 * 4096 * 4096 * 128  # no drawn attention costs more than the listed one


def listed():
    return [
        # the smallest call: a 64 KiB vector update, where the launch is the cost
        {"name": "saxpy_16k", "path": "saxpy", "n": 16384},
        # pre-attention norm of a large prompt batch (the row benchmark's shape)
        {"name": "rms_norm_16384x8192", "path": "rows", "op": "rms_norm", "rows": 16384, "n": 8192},
        # row softmax over an odd number of classes: rows that do not start on 16-byte boundaries
        {"name": "softmax_4000x5001", "path": "rows", "op": "softmax", "rows": 4000, "n": 5001},
        # the large square product of the GEMM benchmark, z += x . y
        {"name": "gemm_bf16_8192", "path": "gemm", "dtype": "bf16", "m": 8192, "n": 8192, "k": 8192, "accumulate": True},
        # logits of a batch of 200 tokens over a vocabulary with an odd number of entries
        {"name": "gemm_bf16_odd_vocabulary", "path": "gemm", "dtype": "bf16", "m": 200, "n": 50021, "k": 1024, "accumulate": False},
        # one transformer block on one new token with 4096 tokens in the cache
        {"name": "decode_block_4096", "path": "decode_block", "hidden": 4096, "kv_heads": 8, "group": 4, "inter": 14336, "ctx": 4096},
        # one transformer block on a prompt of ordinary, not round, length
        {"name": "prefill_block_1500", "path": "prefill_block", "hidden": 4096, "kv_heads": 8, "group": 4, "inter": 14336, "tokens": 1500, "start": 0},
        # causal attention of the benchmark configuration
        {"name": "attention_bf16_causal", "path": "attention", "dtype": "bf16", "batch": 4, "kv_heads": 32, "group": 1, "seq": 4096, "d": 128, "causal": True},
        # decode attention of a batch of long conversations
        {"name": "decode_attention_8x16384", "path": "decode_attention", "batch": 8, "kv_heads": 8, "group": 4, "d": 128, "ctx": 16384},
        # a block-scaled linear layer on a serving batch
        {"name": "linear_mxfp8_200", "path": "linear", "format": "mxfp8", "m": 200, "n": 14336, "k": 4096},
        # the expert product of a mixture-of-experts layer: 512 tokens, two experts each
        {"name": "moe_512", "path": "moe", "tokens": 512, "experts": 32, "top_k": 2, "n": 4096, "k": 4096},
        # greedy sampling of one token: LM head and argmax in one pass over the matrix
        {"name": "lm_head_128256", "path": "lm_head", "vocab": 128256, "k": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_multiple(rng, lo, hi, unit):
    return max(unit, _log(rng, lo, hi) // unit * unit)


def _block_dims(rng):
    hidden = _log_multiple(rng, 1024, 5120, 512)
    group = rng.choice([1, 2, 4, 8])
    heads = max(group, hidden // HEAD_DIM // group * group)
    return {"hidden": hidden, "kv_heads": heads // group, "group": group, "inter": int(hidden * rng.uniform(2.5, 4.0)) // 256 * 256}


def draw(rng):
    path = rng.choice(["saxpy", "rows", "gemm", "gemm", "decode_block", "prefill_block", "attention", "decode_attention", "linear", "moe", "lm_head"])
    if path == "saxpy":
        return {"path": path, "n": _log(rng, 1000, 1 << 24)}
    if path == "rows":
        n = _log(rng, 64, 16384)
        n = n if rng.random() < 0.3 else max(64, n // 64 * 64)
        return {"path": path, "op": rng.choice(["rms_norm", "add_rms_norm", "softmax"]), "rows": min(_log(rng, 1, 16384), 16384 * 8192 // n), "n": n}
    if path == "gemm":
        m, n, k = _log(rng, 1, 8192), _log(rng, 64, 16384), _log(rng, 64, 16384)
        if rng.random() < 0.67:
            n, k = max(64, n // 64 * 64), max(64, k // 64 * 64)
        m = max(1, min(m, int(MOST_GEMM_FLOPS / (2.0 * n * k))))
        dtype = rng.choice(["bf16", "bf16", "f16", "f16", "f32"])
        if dtype == "f32":                                # no matrix-core rate to match: the same range at a sixteenth of the work
            m, n, k = max(1, m // 2), max(64, n // 4), max(64, k // 2)
        return {"path": path, "dtype": dtype, "m": m, "n": n, "k": k, "accumulate": rng.random() < 0.3}
    if path == "decode_block":
        return {"path": path, **_block_dims(rng), "ctx": _log(rng, 16, 65536)}
    if path == "prefill_block":
        return {"path": path, **_block_dims(rng), "tokens": _log(rng, 16, 2048), "start": rng.choice([0, 0, _log(rng, 16, 8192)])}
    if path == "attention":
        c = {"path": path, "dtype": rng.choice(["bf16", "f16"]), "batch": _log(rng, 1, 8), "kv_heads": rng.choice([4, 8, 16, 32]),
             "group": rng.choice([1, 4]), "seq": _log(rng, 128, 8192), "d": rng.choice([64, 128, 128]), "causal": rng.random() < 0.7}
        while work(c)["flops"] > MOST_ATTENTION_FLOPS:
            c["seq"] = c["seq"] * 3 // 4
        return c
    if path == "decode_attention":
        batch = rng.choice([1, 1, _log(rng, 2, 32)])
        return {"path": path, "batch": batch, "kv_heads": rng.choice([4, 8]), "group": rng.choice([1, 2, 4, 8]), "d": rng.choice([64, 128]),
                "ctx": _log(rng, 256, 131072 // batch)}
    if path == "linear":
        return {"path": path, "format": rng.choice(["mxfp8", "nvfp4"]), "m": _log(rng, 1, 4096), "n": _log_multiple(rng, 512, 16384, 64),
                "k": _log_multiple(rng, 512, 8192, 128)}
    if path == "moe":
        return {"path": path, "tokens": _log(rng, 8, 4096), "experts": rng.choice([8, 16, 32, 64]), "top_k": rng.choice([1, 2, 4]),
                "n": _log_multiple(rng, 512, 8192, 256), "k": _log_multiple(rng, 512, 8192, 256)}
    return {"path": path, "vocab": _log(rng, 30000, 160000), "k": _log_multiple(rng, 1024, 8192, 512)}


# ---- inputs ------------------------------------------------------------------------------------------------------------
class _Make:
    """seeded inputs on the GPU"""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float16, std=1.0):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=self.g)

    def weight(self, k, n, dtype=torch.float16):
        return self.normal(k, n, dtype=dtype, std=k ** -0.5)

    def gain(self, n):
        return torch.empty(n, dtype=torch.float16, device="cuda").uniform_(0.5, 1.5, generator=self.g)

    def byte_codes(self, rows, cols, codes):
        """bytes drawn from a list of codes"""
        table = torch.tensor(codes, dtype=torch.uint8, device="cuda")
        return table[torch.randint(len(codes), (rows, cols), device="cuda", generator=self.g)]


def _empty(*shape, dtype=torch.float16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _gemm_tile(m, n):
    """256 x 256 tiles where they fill the chip's 256 compute units, smaller ones otherwise"""
    return [256, 256] if -(-m // 256) * -(-n // 256) >= 256 else [128, 128]


def _inv_freq(d):
    return (1.0 / 10000.0 ** (torch.arange(d // 2, dtype=torch.float32) / (d // 2))).cuda()


def _splits(batch, heads, ctx):
    """heads x splits about one workgroup per compute unit, at least 64 keys a split"""
    return max(1, min(256 // max(1, batch * heads), -(-ctx // 64)))


def _expert_rows(case):
    """how many of the tokens each expert receives: uneven, the same for every seed"""
    e, total = case["experts"], case["tokens"] * case["top_k"]
    share = [1.0 + (7 * g % 17) / 4.0 for g in range(e)]
    rows = [int(total * s / sum(share)) for s in share]
    for i in range(total - sum(rows)):
        rows[i % e] += 1
    return rows


def _descriptors(parts):
    metas = torch.zeros(len(parts), 8, dtype=torch.int32)
    for i, t in enumerate(parts):
        metas[i, 0], metas[i, 1], metas[i, 2] = t.shape[0], t.shape[1], t.stride(0)
    return torch.tensor([t.data_ptr() for t in parts], dtype=torch.int64).cuda(), metas.cuda()


def _block_weights(mk, case):
    h, nkv, inter = case["hidden"], case["kv_heads"], case["inter"]
    nq = nkv * case["group"]
    s = {"nq": nq, "nkv": nkv, "group": case["group"], "hidden": h, "inter": inter, "norm1": mk.gain(h), "norm2": mk.gain(h),
         "q_gain": mk.gain(HEAD_DIM), "k_gain": mk.gain(HEAD_DIM), "inv_freq": _inv_freq(HEAD_DIM), "scale": HEAD_DIM ** -0.5,
         "w_o": mk.weight(nq * HEAD_DIM, h), "w_gate": mk.weight(h, inter), "w_up": mk.weight(h, inter), "w_down": mk.weight(inter, h)}
    return s


def prepare(case, seed):
    mk, path = _Make(seed), case["path"]
    s = {"case": case}
    if path == "saxpy":
        s.update(x=mk.normal(case["n"], dtype=torch.float32), y=mk.normal(case["n"], dtype=torch.float32))
    elif path == "rows":
        r, n = case["rows"], case["n"]
        s.update(x=mk.normal(r, n), out=_empty(r, n), w=mk.gain(n))
        if case["op"] == "add_rms_norm":
            s.update(residual=mk.normal(r, n), residual_out=_empty(r, n))
    elif path == "gemm":
        m, n, k, dt = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
        s.update(x=mk.normal(m, k, dtype=dt), y=mk.weight(k, n, dtype=dt), tile=[64, 64] if dt == torch.float32 else _gemm_tile(m, n))
        s["z"] = mk.normal(m, n, dtype=dt) if case["accumulate"] else _empty(m, n, dtype=dt)
    elif path == "decode_block":
        s.update(_block_weights(mk, case))
        nq, nkv, h, ctx, inter = s["nq"], s["nkv"], s["hidden"], case["ctx"], s["inter"]
        max_seq = ctx + 1
        s.update(w_qkv=mk.weight(h, (nq + 2 * nkv) * HEAD_DIM), x=mk.normal(1, h), position=torch.tensor([ctx], dtype=torch.int32, device="cuda"),
                 k_cache=mk.normal(nkv, max_seq, HEAD_DIM), v_cache=mk.normal(nkv, max_seq, HEAD_DIM), normed=_empty(1, h),
                 qkv=_empty(1, (nq + 2 * nkv) * HEAD_DIM), q=_empty(nkv, s["group"], HEAD_DIM), att=_empty(nkv, s["group"], HEAD_DIM),
                 proj=_empty(1, h), normed2=_empty(1, h), residual=_empty(1, h), gate=_empty(1, inter), up=_empty(1, inter), act=_empty(1, inter),
                 down=_empty(1, h), out=_empty(1, h), splits=_splits(1, nkv, ctx + 1))
        ct.fmha_decode_gqa_noalloc_prepare(s["q"], s["k_cache"], s["v_cache"], ct.partition(s["att"], [1, s["group"], HEAD_DIM]), s["position"], s["splits"])
    elif path == "prefill_block":
        s.update(_block_weights(mk, case))
        nq, nkv, h, t, inter = s["nq"], s["nkv"], s["hidden"], case["tokens"], s["inter"]
        max_seq = case["start"] + t
        s.update(w_q=mk.weight(h, nq * HEAD_DIM), w_k=mk.weight(h, nkv * HEAD_DIM), w_v=mk.weight(h, nkv * HEAD_DIM), x=mk.normal(t, h),
                 k_cache=mk.normal(nkv, max_seq, HEAD_DIM), v_cache=mk.normal(nkv, max_seq, HEAD_DIM), normed=_empty(t, h),
                 q=_empty(t, nq * HEAD_DIM), k=_empty(t, nkv * HEAD_DIM), v=_empty(t, nkv * HEAD_DIM), q_rot=_empty(t, nq, HEAD_DIM),
                 att=_empty(t, nq, HEAD_DIM), proj=_empty(t, h), normed2=_empty(t, h), residual=_empty(t, h), gate=_empty(t, inter),
                 up=_empty(t, inter), act=_empty(t, inter), down=_empty(t, h), out=_empty(t, h))
    elif path == "attention":
        b, hk, g, n, d, dt = case["batch"], case["kv_heads"], case["group"], case["seq"], case["d"], DTYPES[case["dtype"]]
        s.update(q=mk.normal(b, hk * g, n, d, dtype=dt), k=mk.normal(b, hk, n, d, dtype=dt), v=mk.normal(b, hk, n, d, dtype=dt),
                 out=_empty(b * hk * g, n, d, dtype=dt), bm=256 if d == 128 and n > 128 else 128)
    elif path == "decode_attention":
        b, hk, g, d, ctx = case["batch"], case["kv_heads"], case["group"], case["d"], case["ctx"]
        splits = _splits(b, hk, ctx)
        if b == 1:
            s.update(q=mk.normal(hk, g, d), k=mk.normal(hk, ctx, d), v=mk.normal(hk, ctx, d), out=_empty(hk, g, d), splits=splits,
                     position=torch.tensor([ctx - 1], dtype=torch.int32, device="cuda"))
            ct.fmha_decode_gqa_noalloc_prepare(s["q"], s["k"], s["v"], ct.partition(s["out"], [1, g, d]), s["position"], splits)
        else:
            per = -(-ctx // splits) + 63
            per = per // 64 * 64
            splits = -(-ctx // per)
            s.update(q=mk.normal(b, hk, g, d), k=mk.normal(b, hk, ctx, d), v=mk.normal(b, hk, ctx, d), att=_empty(b, hk, g, splits, d),
                     lse=_empty(b, hk, g, splits, dtype=torch.float32), per=per, count=torch.tensor([ctx], dtype=torch.int32, device="cuda"))
    elif path == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        if case["format"] == "mxfp8":   # e4m3 values of both signs around one, power-of-two scales around one
            e4m3 = [sign | (e << 3) | f for sign in (0, 0x80) for e in range(3, 9) for f in range(8)]
            s.update(x=mk.byte_codes(m, k, e4m3), y=mk.byte_codes(n, k, e4m3), xs=mk.byte_codes(m, k // 32, range(124, 130)),
                     ys=mk.byte_codes(n, k // 32, range(118, 124)))
        else:                           # every pair of e2m1 values, e4m3 scales around one
            s.update(x=mk.byte_codes(m, k // 2, range(256)), y=mk.byte_codes(n, k // 2, range(256)), xs=mk.byte_codes(m, k // 16, range(48, 64)),
                     ys=mk.byte_codes(n, k // 16, range(24, 40)))
        s.update(z=_empty(m, n, dtype=torch.bfloat16), tile=_gemm_tile(m, n))
    elif path == "moe":
        rows, n, k = _expert_rows(case), case["n"], case["k"]
        a, c = mk.normal(sum(rows), k), _empty(sum(rows), n)     # tokens sorted by expert, one buffer
        b = [mk.weight(k, n) for _ in rows]
        s.update(a=a, b=b, c=c, a_tab=_descriptors(list(a.split(rows))), b_tab=_descriptors(b), c_tab=_descriptors(list(c.split(rows))),
                 tile=256 if sum(rows) > 128 * len(rows) else 128)
    else:
        blocks = -(-case["vocab"] // 64)
        s.update(w=mk.normal(case["vocab"], case["k"], std=case["k"] ** -0.5), hidden=mk.normal(1, case["k"]), block_max=_empty(blocks, dtype=torch.float32),
                 block_idx=_empty(blocks, dtype=torch.int32), token=_empty(1, dtype=torch.int32))
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------------
def _linear_f16(s, z, x, w):
    ct.gemm(ct.partition(s[z], _gemm_tile(s[z].shape[0], s[z].shape[1])), s[x], s[w], s[w].shape[0], accumulate=False)


def _block_tail(s):
    """everything behind the attention: output projection, second norm, gated MLP, second residual"""
    rows, h = s["x"].shape
    _linear_f16(s, "proj", "att2d", "w_o")
    ct.add_rms_norm_f16(s["x"], s["proj"], s["norm2"], ct.partition(s["normed2"], [1, h]), ct.partition(s["residual"], [1, h]), EPS)
    _linear_f16(s, "gate", "normed2", "w_gate")
    _linear_f16(s, "up", "normed2", "w_up")
    ct.silu_mul_2d_f16(ct.partition(s["act"], [1, 256]), s["gate"], s["up"])
    _linear_f16(s, "down", "act", "w_down")
    ct.add_2d_f16(ct.partition(s["out"], [1, 256]), s["residual"], s["down"])
    return s["out"], s["k_cache"], s["v_cache"]


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "saxpy":
        ct.saxpy(ct.partition(s["y"], [1024]), 0.5, s["x"])
        return s["y"]
    if path == "rows":
        out = ct.partition(s["out"], [1, case["n"]])
        if case["op"] == "rms_norm":
            ct.rms_norm_f16(s["x"], s["w"], out, EPS)
        elif case["op"] == "softmax":
            ct.softmax(s["x"], out)
        else:
            ct.add_rms_norm_f16(s["residual"], s["x"], s["w"], out, ct.partition(s["residual_out"], [1, case["n"]]), EPS)
            return s["out"], s["residual_out"]
        return s["out"]
    if path == "gemm":
        ct.gemm(ct.partition(s["z"], s["tile"]), s["x"], s["y"], case["k"], accumulate=case["accumulate"],
                generics=[case["dtype"], s["tile"][0], s["tile"][1], 1, case["k"]])
        return s["z"]
    if path == "decode_block":
        h, g = s["hidden"], s["group"]
        ct.rms_norm_f16(s["x"], s["norm1"], ct.partition(s["normed"], [1, h]), EPS)
        _linear_f16(s, "qkv", "normed", "w_qkv")
        ct.qk_norm_rope_kv_decode_raw_f16(s["qkv"], s["q_gain"], s["k_gain"], s["inv_freq"], s["q"], s["k_cache"], s["v_cache"], s["position"], EPS,
                                          s["nq"], s["nkv"])
        ct.fmha_decode_gqa_noalloc(s["q"], s["k_cache"], s["v_cache"], ct.partition(s["att"], [1, g, HEAD_DIM]), s["scale"], s["position"], s["splits"])
        s["att2d"] = s["att"].view(1, -1)
        return _block_tail(s)
    if path == "prefill_block":
        h, t, start = s["hidden"], case["tokens"], case["start"]
        ct.rms_norm_f16(s["x"], s["norm1"], ct.partition(s["normed"], [1, h]), EPS)
        for name in ("q", "k", "v"):
            _linear_f16(s, name, "normed", "w_" + name)
        heads = lambda name: s[name].view(t, -1, HEAD_DIM)
        ct.qk_norm_rope_kv_prefill_raw_f16(heads("q"), heads("k"), heads("v"), s["q_gain"], s["k_gain"], s["inv_freq"], s["q_rot"], s["k_cache"],
                                           s["v_cache"], EPS, start, t)
        ct.fmha_seq_f16(s["q_rot"], s["k_cache"], s["v_cache"], ct.partition(s["att"], [128, 1, HEAD_DIM]), s["scale"], s["group"], kv_len=start + t,
                        query_start=start, causal=True)
        s["att2d"] = s["att"].view(t, -1)
        return _block_tail(s)
    if path == "attention":
        ct.fmha(ct.partition(s["out"], [1, s["bm"], case["d"]]), s["q"], s["k"], s["v"], case["d"] ** -0.5, 0, case["group"], causal=case["causal"])
        return s["out"]
    if path == "decode_attention":
        if case["batch"] == 1:
            ct.fmha_decode_gqa_noalloc(s["q"], s["k"], s["v"], ct.partition(s["out"], [1, case["group"], case["d"]]), case["d"] ** -0.5, s["position"],
                                       s["splits"])
            return s["out"]
        ct.attention_decode_kernel_grouped_f16(s["q"], s["k"], s["v"], s["att"], s["lse"], case["d"] ** -0.5, s["count"], tile_n=64,
                                               kv_len_per_split=s["per"], query_group_tile_size=16)
        return s["att"], s["lse"]
    if path == "linear":
        f = ct.linear_tile_mxfp8 if case["format"] == "mxfp8" else ct.linear_tile_nvfp4
        f(ct.partition(s["z"], s["tile"]), s["x"], s["y"], s["xs"], s["ys"], 1.0)
        return s["z"]
    if path == "moe":
        (ap, am), (bp, bm), (cp, cm) = s["a_tab"], s["b_tab"], s["c_tab"]
        ct.group_gemm_f16_nt_desc(ap, bp, cp, am, bm, cm, case["experts"], generics=[s["tile"], s["tile"], 64, 256])
        return s["c"]
    ct.lm_head_argmax_blocks_f16(s["w"], s["hidden"], ct.partition(s["block_max"], [1]), ct.partition(s["block_idx"], [1]), case["vocab"])
    ct.argmax_reduce_blocks_to_u32(s["block_max"], s["block_idx"], ct.partition(s["token"], [1]), s["block_max"].numel())
    return s["block_max"], s["block_idx"], s["token"]


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
def _block_work(case, t, start):
    h, nkv, inter = case["hidden"], case["kv_heads"], case["inter"]
    nq = nkv * case["group"]
    weights = h * (nq + 2 * nkv) * HEAD_DIM + nq * HEAD_DIM * h + 3 * h * inter
    cache = 2 * nkv * (start + t) * HEAD_DIM
    pairs = t * start + t * (t + 1) // 2                   # (query, key) pairs under the causal mask
    return {"bytes": 2.0 * (weights + cache + 2 * t * h), "flops": 2.0 * t * weights + 4.0 * nq * HEAD_DIM * pairs}


def work(case):
    path = case["path"]
    if path == "saxpy":
        return {"bytes": 12.0 * case["n"], "flops": 2.0 * case["n"]}
    if path == "rows":
        per = {"rms_norm": 2, "softmax": 2, "add_rms_norm": 4}[case["op"]]
        return {"bytes": 2.0 * (per * case["rows"] * case["n"] + (case["n"] if case["op"] != "softmax" else 0)), "flops": 5.0 * case["rows"] * case["n"]}
    if path == "gemm":
        m, n, k, size = case["m"], case["n"], case["k"], 4 if case["dtype"] == "f32" else 2
        return {"bytes": float(size) * (m * k + k * n + m * n * (2 if case["accumulate"] else 1)), "flops": 2.0 * m * n * k}
    if path == "decode_block":
        return _block_work(case, 1, case["ctx"])
    if path == "prefill_block":
        return _block_work(case, case["tokens"], case["start"])
    if path == "attention":
        b, hk, g, n, d = case["batch"], case["kv_heads"], case["group"], case["seq"], case["d"]
        return {"bytes": 2.0 * b * hk * n * d * (2 * g + 2), "flops": 4.0 * b * hk * g * d * (n * (n + 1) // 2 if case["causal"] else n * n)}
    if path == "decode_attention":
        b, hk, g, d, ctx = case["batch"], case["kv_heads"], case["group"], case["d"], case["ctx"]
        return {"bytes": 2.0 * b * hk * d * (2 * ctx + 2 * g), "flops": 4.0 * b * hk * g * d * ctx}
    if path == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        per = 1.0 + 1 / 32 if case["format"] == "mxfp8" else 0.5 + 1 / 16
        return {"bytes": (m + n) * k * per + 2.0 * m * n, "flops": 2.0 * m * n * k}
    if path == "moe":
        rows = _expert_rows(case)
        used = sum(1 for r in rows if r)
        return {"bytes": 2.0 * (sum(rows) * (case["k"] + case["n"]) + used * case["k"] * case["n"]), "flops": 2.0 * sum(rows) * case["n"] * case["k"]}
    return {"bytes": 2.0 * case["vocab"] * case["k"], "flops": 2.0 * case["vocab"] * case["k"]}


def tolerance(case):
    """Four times the distance of each path from the same computation in float64, over the ranges above: one rounding of the
    result for the row kernels and the products (f16 2.1e-4, bf16 1.7e-3), a few for attention and a block; f32 sums of up to
    8192 terms; indices may differ where two logits are equal to the last bits."""
    path = case["path"]
    if path == "saxpy":
        return "exact"                                     # one fused multiply-add an element
    if path == "linear" or case.get("dtype") == "bf16":
        return {"rel": 1e-2, "max": 0.28} if path == "attention" else {"rel": 7e-3, "max": 2e-2}
    if case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 5e-5}
    if path in ("decode_block", "prefill_block"):
        return {"rel": 2e-3, "max": 2e-2}
    if path in ("attention", "decode_attention"):
        return {"rel": 1.2e-3, "max": 2e-2}
    if path == "lm_head":
        return {"rel": 1e-6, "max": 4e-6, "differ": 2e-3}
    return {"rel": 1e-3, "max": 2e-3}
