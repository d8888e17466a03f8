"""The attention hot path's measured workloads: what each case runs, its inputs, the work it
cannot do without and the accuracy it has to keep.

A case is a dict of plain values.  `family` names the call (or the few calls) a program makes;
the other entries are its sizes, element type and options:

  mha_decode      fp32 single-query MHA (kernel::mha_kernel_cu): the smallest call, one query
                  row over a short cache, bound by its own latency.
  decode_step     one token through the attention of every layer, replayed from a captured
                  graph with the position in device memory: per layer the Q/K norm + RoPE +
                  cache write, then the flash decode.  How a single conversation decodes.
  paged_decode    one query row per sequence over a paged KV pool: serving, with the ragged
                  lengths a batch of conversations has.
  prefill         causal GQA prefill of a prompt (start 0) or of a chunk behind a cached
                  prefix (start > 0), 16-bit.
  prefill_fp32    the same in fp32 (kernel::batched_mha_kernel_cu).
  prefill_layer   the attention of one layer over a prompt from the raw Q / K / V
                  projections: producer, prefill, wo projection.
  vision          the attention of one vision block: QKV split + 2-D rotary + transpose, then
                  bidirectional attention over packed images.
  qk_producer     per-head RMSNorm + RoPE of Q and K with the K / V cache writes, over a prompt.
  kv_write        K / V rows of a prefill batch stored to their slots of a paged pool.

Head counts are those of the models in this repository's tests and benchmark (32/8, 28/4 and
12/2 heads of 128, 12 heads of 64, 16 vision heads of 72).
"""
import math

import numpy as np
import torch

from orinmllm_amd import kernel as K

_TYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_EPS = 1e-6
_THETA = 1e6


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # One query of a 12-head fp32 model at position 255: the smallest call there is.
        {"name": "mha_decode_fp32", "family": "mha_decode", "dtype": "fp32", "q_heads": 12,
         "kv_heads": 12, "head_size": 64, "pos": 255, "capacity": 2048},
        # A conversation in its second page of text, Qwen3-8B heads, graph-captured step.
        {"name": "decode_step_fp16", "family": "decode_step", "dtype": "fp16", "layers": 16,
         "q_heads": 32, "kv_heads": 8, "head_size": 128, "pos": 1337, "capacity": 4096},
        # Serving: 32 conversations, lengths 512 to 4096.
        {"name": "paged_decode_b32_fp16", "family": "paged_decode", "dtype": "fp16", "batch": 32,
         "q_heads": 32, "kv_heads": 8, "head_size": 128, "min_len": 512, "max_len": 4096,
         "block": 16, "head_major": True},
        # A few long documents, 7 query heads per kv head, odd batch, token-major pool.
        {"name": "paged_decode_b5_bf16", "family": "paged_decode", "dtype": "bf16", "batch": 5,
         "q_heads": 28, "kv_heads": 4, "head_size": 128, "min_len": 2048, "max_len": 16000,
         "block": 32, "head_major": False},
        # A long prompt at once.
        {"name": "prefill_4096_fp16", "family": "prefill", "dtype": "fp16", "seq": 4096, "start": 0,
         "q_heads": 32, "kv_heads": 8, "head_size": 128},
        # A chunk of a long prompt behind its cached prefix, a small model's few heads.
        {"name": "prefill_chunk_bf16", "family": "prefill", "dtype": "bf16", "seq": 1000,
         "start": 2500, "q_heads": 12, "kv_heads": 2, "head_size": 128},
        # A short prompt: less than one block of queries per head.
        {"name": "prefill_137_fp16", "family": "prefill", "dtype": "fp16", "seq": 137, "start": 0,
         "q_heads": 32, "kv_heads": 8, "head_size": 128},
        # The fp32 attention type (kAttentionMHA) over a medium prompt.
        {"name": "prefill_fp32", "family": "prefill_fp32", "dtype": "fp32", "seq": 523, "start": 0,
         "q_heads": 28, "kv_heads": 4, "head_size": 128},
        # One layer's attention over an odd prompt, raw projections to wo.
        {"name": "prefill_layer_bf16", "family": "prefill_layer", "dtype": "bf16", "seq": 1531,
         "start": 0, "q_heads": 28, "kv_heads": 4, "head_size": 128, "fused": True},
        # Four images of different sizes through one vision block.
        {"name": "vision_bf16", "family": "vision", "dtype": "bf16", "heads": 16, "head_size": 72,
         "segments": "1024,731,1500,256"},
        # The producer of a long prompt.
        {"name": "qk_producer_fp16", "family": "qk_producer", "dtype": "fp16", "seq": 4096,
         "start": 0, "q_heads": 32, "kv_heads": 8, "head_size": 128},
        # A full prefill batch stored into a paged pool.
        {"name": "kv_write_bf16", "family": "kv_write", "dtype": "bf16", "rows": 16384,
         "kv_heads": 8, "head_size": 128, "block": 16, "head_major": True},
    ]


_GQA = [(32, 8), (28, 4), (12, 2)]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["mha_decode", "decode_step", "paged_decode", "paged_decode", "prefill",
                         "prefill", "prefill_fp32", "prefill_layer", "vision", "qk_producer",
                         "kv_write"])
    half = rng.choice(["fp16", "bf16"])
    hq, hkv = rng.choice(_GQA)
    if family == "mha_decode":
        hq, hkv, d = rng.choice([(12, 12, 64), (32, 8, 128), (28, 4, 128)])
        pos = _log_int(rng, 15, 4095)
        return {"family": family, "dtype": "fp32", "q_heads": hq, "kv_heads": hkv, "head_size": d,
                "pos": pos, "capacity": 4096}
    if family == "decode_step":
        capacity = rng.choice([2048, 4096, 8192])
        return {"family": family, "dtype": half, "layers": rng.randint(4, 16), "q_heads": hq,
                "kv_heads": hkv, "head_size": 128, "pos": _log_int(rng, 30, capacity - 1),
                "capacity": capacity}
    if family == "paged_decode":
        batch = _log_int(rng, 1, 64)
        longest = min(16384, 75000 // (batch * hkv) * 8)
        hi = _log_int(rng, 200, max(300, longest))
        return {"family": family, "dtype": half, "batch": batch, "q_heads": hq, "kv_heads": hkv,
                "head_size": 128, "min_len": max(1, int(hi * rng.uniform(0.1, 1.0))),
                "max_len": hi, "block": rng.choice([16, 32]),
                "head_major": rng.choice([True, False])}
    if family == "prefill":
        seq = _log_int(rng, 16, 4096)
        # the chunk and its prefix stay within the work of the longest listed prompt
        most = min(8192 - seq, int(2 ** 23 * 32 / hq / seq - seq / 2))
        start = 0 if rng.random() < 0.5 else _log_int(rng, 16, max(17, most))
        return {"family": family, "dtype": half, "seq": seq, "start": start, "q_heads": hq,
                "kv_heads": hkv, "head_size": rng.choice([128, 128, 64])}
    if family == "prefill_fp32":
        seq = _log_int(rng, 8, 480)
        start = 0 if rng.random() < 0.7 else rng.randint(1, 481 - seq)
        return {"family": family, "dtype": "fp32", "seq": seq, "start": start, "q_heads": hq,
                "kv_heads": hkv, "head_size": 128}
    if family == "prefill_layer":
        return {"family": family, "dtype": half, "seq": _log_int(rng, 16, 2048), "start": 0,
                "q_heads": hq, "kv_heads": hkv, "head_size": 128,
                "fused": rng.choice([True, False])}
    if family == "vision":
        n = rng.randint(1, 5)
        seg = [_log_int(rng, 64, 1536) for _ in range(n)]
        return {"family": family, "dtype": half, "heads": rng.choice([12, 16]),
                "head_size": rng.choice([72, 72, 64, 80]),
                "segments": ",".join(str(s) for s in seg)}
    if family == "qk_producer":
        return {"family": family, "dtype": half, "seq": _log_int(rng, 16, 4096),
                "start": rng.choice([0, 1000]), "q_heads": hq, "kv_heads": hkv, "head_size": 128}
    return {"family": family, "dtype": half, "rows": _log_int(rng, 16, 16384), "kv_heads": hkv,
            "head_size": 128, "block": rng.choice([16, 32]),
            "head_major": rng.choice([True, False])}


# ---------------------------------------------------------------- inputs

class _Inputs:
    """Tensors made on the GPU from the seed, in a fixed order."""

    def __init__(self, case, seed):
        self.type = _TYPES[case["dtype"]]
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(0x0A77 * 1000003 + seed)
        self.rng = np.random.default_rng(seed)

    def normal(self, *shape, scale=1.0, shift=0.0, dtype=None):
        x = torch.randn(*shape, device="cuda", generator=self.gen)
        if scale != 1.0 or shift != 0.0:
            x = x * scale + shift
        return x.to(dtype or self.type)

    def weight(self, d):  # RMSNorm weights: near one
        return self.normal(d, scale=0.1, shift=1.0)

    def rotated(self, rows, heads, d, start=0):
        """Q or K rows as the attention meets them: RMS-normalised, rotated."""
        x = torch.randn(rows, heads, d, device="cuda", generator=self.gen)
        x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + _EPS)
        c, s = _angles(rows, d, start, torch.float32)
        return _rotate(x, c[:, None], s[:, None]).reshape(rows, heads * d).to(self.type)


def _angles(rows, d, start, dtype):
    """cos / sin [rows, d / 2] of positions start .. start + rows - 1."""
    freq = 1.0 / _THETA ** (torch.arange(0, d // 2, device="cuda", dtype=torch.float64) * 2 / d)
    a = torch.arange(start, start + rows, device="cuda", dtype=torch.float64)[:, None] * freq
    return torch.cos(a).to(dtype), torch.sin(a).to(dtype)


def _rotate(x, c, s):
    lo, hi = x.chunk(2, -1)
    return torch.cat([c * lo - s * hi, c * hi + s * lo], -1)


def _tables(max_seq, d):
    """The fp32 sin / cos caches a program fills once."""
    sin = torch.empty(max_seq, d, device="cuda")
    cos = torch.empty_like(sin)
    K.sin_cos_cache_calc_cu(d, max_seq, sin, cos, _THETA)
    return sin, cos


def _draw_inputs(case, seed):
    i = _Inputs(case, seed)
    f = case["family"]
    d = case["head_size"]
    t = {}
    if f == "mha_decode":
        hq, hkv = case["q_heads"], case["kv_heads"]
        t["q"] = i.normal(hq * d)
        t["k"] = i.normal(1, case["capacity"], hkv * d)
        t["v"] = i.normal(1, case["capacity"], hkv * d)
    elif f == "decode_step":
        L, hq, hkv = case["layers"], case["q_heads"], case["kv_heads"]
        t["q"] = i.normal(L, hq * d)
        t["k"] = i.normal(L, hkv * d)
        t["v"] = i.normal(L, hkv * d)
        t["wq"], t["wk"] = i.weight(d), i.weight(d)
        t["k_cache"] = i.normal(L, case["capacity"], hkv * d)
        t["v_cache"] = i.normal(L, case["capacity"], hkv * d)
    elif f == "paged_decode":
        hkv, bs = case["kv_heads"], case["block"]
        lens = i.rng.integers(case["min_len"], case["max_len"] + 1, case["batch"]).astype(np.int32)
        lens[i.rng.integers(0, case["batch"])] = case["max_len"]
        nblk = (lens + bs - 1) // bs
        table = np.zeros((case["batch"], int(nblk.max())), np.int32)
        perm = i.rng.permutation(int(nblk.sum())).astype(np.int32)
        at = 0
        for b, n in enumerate(nblk):
            table[b, :n] = perm[at:at + n]
            at += n
        shape = (at, hkv, bs, d) if case["head_major"] else (at, bs, hkv, d)
        t["k"], t["v"] = i.normal(*shape), i.normal(*shape)
        t["q"] = i.normal(case["batch"], case["q_heads"], d)
        t["lens"], t["table"] = lens, table
    elif f in ("prefill", "prefill_fp32"):
        n = case["start"] + case["seq"]
        t["q"] = i.rotated(case["seq"], case["q_heads"], d, case["start"])
        t["k"] = i.rotated(n, case["kv_heads"], d)
        t["v"] = i.normal(n, case["kv_heads"] * d)
    elif f in ("prefill_layer", "qk_producer"):
        S, hq, hkv = case["seq"], case["q_heads"], case["kv_heads"]
        t["q"] = i.normal(S, hq * d)
        t["k"] = i.normal(S, hkv * d)
        t["v"] = i.normal(S, hkv * d)
        t["wq"], t["wk"] = i.weight(d), i.weight(d)
        if f == "prefill_layer":
            t["wo"] = i.normal(hq * d, hq * d, scale=(hq * d) ** -0.5)
    elif f == "vision":
        N = sum(_segments(case))
        t["qkv"] = i.normal(N, 3 * case["heads"] * d)
        # 2-D rotary: row and column angle of each patch, both halves of the head alike.
        pos = torch.randint(0, 48, (N, 2), device="cuda", generator=i.gen).float()
        freq = 1.0 / 1e4 ** (torch.arange(0, d // 4, device="cuda").float() * 4 / d)
        a = (pos[:, :, None] * freq).reshape(N, -1)
        a = torch.cat([a, a], -1)
        t["cos"], t["sin"] = a.cos().to(i.type), a.sin().to(i.type)
    else:
        n, hkv, bs = case["rows"], case["kv_heads"], case["block"]
        t["k"], t["v"] = i.normal(n, hkv, d), i.normal(n, hkv, d)
        nblk = (n + bs - 1) // bs
        perm = i.rng.permutation(nblk)
        at = np.arange(n)
        t["slots"] = (perm[at // bs] * bs + at % bs).astype(np.int32)
    return t


def _segments(case):
    return [int(x) for x in case["segments"].split(",")]


# ---------------------------------------------------------------- prepare

class _State:
    pass


_capture_stream = None  # the stream a program captures its step on


def prepare(case, seed):
    global _capture_stream
    st = _State()
    st.case = dict(case)
    st.__dict__.update(_draw_inputs(case, seed))
    f, d = case["family"], case["head_size"]
    if f == "mha_decode":
        st.out = torch.empty_like(st.q)
        st.score = torch.empty(case["q_heads"], case["capacity"], device="cuda")
    elif f == "decode_step":
        st.sin, st.cos = _tables(case["capacity"], d)
        st.q_step = torch.empty_like(st.q)  # the q projection writes here, the step rotates it
        st.out = torch.empty_like(st.q)
        st.pos = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
        if _capture_stream is None:
            _capture_stream = torch.cuda.Stream()
        K.reserve_decode_workspace(case["q_heads"], d, case["capacity"], _capture_stream)
        torch.cuda.synchronize()
        st.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st.graph, stream=_capture_stream):
            _decode_step(st)
    elif f == "paged_decode":
        st.out = torch.empty_like(st.q)
        st.max_len = int(st.lens.max())
        st.lens = torch.from_numpy(st.lens).cuda()
        st.table = torch.from_numpy(st.table).cuda()
        st.layout = K.KV_LAYOUT_HEAD_MAJOR if case["head_major"] else K.KV_LAYOUT_TOKEN_MAJOR
        n = K.decode_workspace_size(case["batch"], case["q_heads"], case["kv_heads"], d, st.max_len)
        st.workspace = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    elif f in ("prefill", "prefill_fp32"):
        st.out = torch.empty_like(st.q)
    elif f in ("prefill_layer", "qk_producer"):
        n = case["start"] + case["seq"]
        st.sin, st.cos = _tables(n, d)
        st.k_cache = torch.zeros(1, n, case["kv_heads"] * d, device="cuda", dtype=st.k.dtype)
        st.v_cache = torch.zeros_like(st.k_cache)
        st.q_rot = torch.empty_like(st.q)
        if f == "qk_producer":
            st.q_rot.copy_(st.q)
        else:
            st.attn = torch.empty_like(st.q)
            st.out = torch.empty_like(st.q)
    elif f == "vision":
        seg = _segments(case)
        st.cu = torch.tensor([0] + list(np.cumsum(seg)), dtype=torch.int32, device="cuda")
        st.longest = max(seg)
        N = sum(seg)
        st.qkv_t = [torch.empty(case["heads"], N, d, device="cuda", dtype=st.qkv.dtype)
                    for _ in range(3)]
        st.out = torch.empty(N, case["heads"] * d, device="cuda", dtype=st.qkv.dtype)
    else:
        n, hkv, bs = case["rows"], case["kv_heads"], case["block"]
        nblk = (n + bs - 1) // bs
        shape = (nblk, hkv, bs, d) if case["head_major"] else (nblk, bs, hkv, d)
        st.k_pool = torch.zeros(*shape, device="cuda", dtype=st.k.dtype)
        st.v_pool = torch.zeros_like(st.k_pool)
        st.slots = torch.from_numpy(st.slots).cuda()
        st.layout = K.KV_LAYOUT_HEAD_MAJOR if case["head_major"] else K.KV_LAYOUT_TOKEN_MAJOR
    return st


def _decode_step(st):
    c = st.case
    hq, hkv, d = c["q_heads"], c["kv_heads"], c["head_size"]
    for layer in range(c["layers"]):
        K.qk_norm_rope_cu(st.q_step[layer], st.k[layer], st.v[layer], st.wq, st.wk, st.sin, st.cos,
                          st.k_cache, st.v_cache, layer, c["capacity"], 0, 1, hq, hkv, d, _EPS,
                          pos_ptr=st.pos)
        K.flash_attention_decode_fp16_gpu_pos_cu(st.pos, hq, hkv, d, hq // hkv, layer,
                                                 c["capacity"], hkv * d, st.q_step[layer],
                                                 st.out[layer], st.k_cache, st.v_cache)


# ---------------------------------------------------------------- run

def run(st):
    c = st.case
    f, d = c["family"], c["head_size"]
    if f == "mha_decode":
        hq, hkv = c["q_heads"], c["kv_heads"]
        K.mha_kernel_cu(c["pos"], hq, 0, c["capacity"], hkv * d, hq // hkv, d, st.out, st.q,
                        st.score, st.k, st.v)
        return st.out
    if f == "decode_step":
        st.q_step.copy_(st.q)
        st.graph.replay()
        return st.out, st.k_cache, st.v_cache
    if f == "paged_decode":
        K.paged_decode_cu(st.q, st.k, st.v, st.out, st.table, st.lens, st.max_len,
                          workspace=st.workspace, layout=st.layout)
        return st.out
    if f == "vision":
        N = st.qkv.shape[0]
        q, k, v = st.qkv_t
        K.fused_split_rope_transpose_cu(st.qkv, st.cos, st.sin, q, k, v, N, c["heads"], d)
        K.vision_attention_varlen_cu(q, k, v, st.out, st.cu, st.longest, c["heads"], d)
        return st.out
    if f == "kv_write":
        K.kv_cache_write_paged(st.k, st.v, st.k_pool, st.v_pool, st.slots, layout=st.layout)
        return st.k_pool, st.v_pool
    S, start, hq, hkv = c["seq"], c["start"], c["q_heads"], c["kv_heads"]
    n = start + S
    if f == "prefill":
        K.flash_attention_prefill_cu(start, S, hq, hkv, d, hq // hkv, 0, n, hkv * d, st.q, st.out,
                                     st.k, st.v)
        return st.out
    if f == "prefill_fp32":
        K.batched_mha_kernel_cu(start, S, hq, 0, n, hq * d, hkv * d, hq // hkv, d, st.out, st.q,
                                None, st.k, st.v)
        return st.out
    if f == "qk_producer":
        # In place: a second call rotates rows that are already unit RMS.
        st.q_rot.copy_(st.q)
        K.qk_norm_rope_cu(st.q_rot, st.k, st.v, st.wq, st.wk, st.sin, st.cos, st.k_cache,
                          st.v_cache, 0, n, start, S, hq, hkv, d, _EPS)
        return st.q_rot, st.k_cache, st.v_cache
    if c["fused"]:
        K.qk_norm_rope_cu(None, st.k, st.v, None, st.wk, st.sin, st.cos, st.k_cache, st.v_cache, 0,
                          n, start, S, hq, hkv, d, _EPS)
        K.flash_attention_prefill_qk_norm_rope_cu(start, S, hq, hkv, d, hq // hkv, 0, n, hkv * d,
                                                  st.q, st.attn, st.k_cache, st.v_cache, st.wq,
                                                  st.sin, st.cos, _EPS)
    else:
        st.q_rot.copy_(st.q)
        K.qk_norm_rope_cu(st.q_rot, st.k, st.v, st.wq, st.wk, st.sin, st.cos, st.k_cache,
                          st.v_cache, 0, n, start, S, hq, hkv, d, _EPS)
        K.flash_attention_prefill_cu(start, S, hq, hkv, d, hq // hkv, 0, n, hkv * d, st.q_rot,
                                     st.attn, st.k_cache, st.v_cache)
    K.batched_matmul_kernel_cu(st.attn, st.wo, st.out, S)
    return st.out, st.k_cache, st.v_cache


# ---------------------------------------------------------------- work and tolerance

def work(case):
    f, d = case["family"], case["head_size"]
    e = 4 if case["dtype"] == "fp32" else 2
    if f == "kv_write":
        return {"bytes": 4 * case["rows"] * case["kv_heads"] * d * e + 4 * case["rows"], "flops": 0}
    if f == "vision":
        seg = _segments(case)
        H, N = case["heads"], sum(seg)
        # qkv, tables and the output; q / k / v between the two calls are the path's own
        # interface (head-major tensors): written once, read once.
        return {"bytes": (3 + 6 + 1) * N * H * d * e + 2 * N * d * e,
                "flops": 4 * d * H * sum(s * s for s in seg)}
    hq, hkv = case["q_heads"], case["kv_heads"]
    if f == "mha_decode":
        n = case["pos"] + 1
        return {"bytes": 2 * n * hkv * d * e + 2 * hq * d * e, "flops": 4 * n * hq * d}
    if f == "decode_step":
        L, n = case["layers"], case["pos"] + 1
        row = 2 * n * hkv * d + 4 * hq * d + 4 * hkv * d
        return {"bytes": L * row * e, "flops": L * 4 * n * hq * d}
    if f == "paged_decode":
        # the mean of the drawn lengths (uniform between the bounds, one at the maximum)
        total = case["max_len"] + (case["batch"] - 1) * (case["min_len"] + case["max_len"]) / 2
        return {"bytes": 2 * total * hkv * d * e + 2 * case["batch"] * hq * d * e,
                "flops": 4 * total * hq * d}
    S, n = case["seq"], case["start"] + case["seq"]
    producer = (2 * hq + 4 * hkv) * S * d * e + 2 * S * d * 4
    attention = {"bytes": (2 * S * hq + 2 * n * hkv) * d * e,
                 "flops": 4 * d * hq * sum(range(case["start"] + 1, n + 1))}
    if f == "qk_producer":
        # q_rot is a copy of the raw rows (read and written) that the producer then rotates in
        # place (read and written)
        return {"bytes": producer + 2 * S * hq * d * e, "flops": 0}
    if f == "prefill_layer":
        dim = hq * d
        return {"bytes": 4 * hkv * S * d * e + S * d * 8 + attention["bytes"] +
                (2 * S * dim + dim * dim) * e,
                "flops": attention["flops"] + 2 * S * dim * dim}
    return attention


def tolerance(case):
    # About four times the distance to float64 seen over the ranges.  fp32 (2.4e-7): sums in
    # another order.  16 bits: the output's own rounding and that of the softmax weights
    # (fp16 3.2e-4, bf16 1.7e-3), and in a layer or a vision block also that of the rows
    # between its calls (4.2e-4, 3.1e-3).
    if case["family"] == "kv_write":
        return "exact"
    if case["dtype"] == "fp32":
        return {"rel": 2e-6}
    if case["family"] in ("prefill_layer", "vision"):
        return {"rel": 1.7e-3 if case["dtype"] == "fp16" else 1.2e-2}
    return {"rel": 1.3e-3 if case["dtype"] == "fp16" else 6.6e-3}


# ---------------------------------------------------------------- exact

def _attend(q, k, v, last):
    """softmax(q k^T / sqrt(d)) v in float64 over one head: row i sees keys 0 .. last[i]."""
    out = torch.empty_like(q)
    keys = torch.arange(k.shape[0], device=q.device)
    kt = k.t().contiguous()
    for r in range(0, q.shape[0], 1024):
        s = q[r:r + 1024] @ kt / math.sqrt(q.shape[1])
        s.masked_fill_(keys[None] > last[r:r + 1024, None], -math.inf)
        out[r:r + 1024] = torch.softmax(s, -1) @ v
    return out


def _attend_heads(q, k, v, start, hq, hkv, d):
    """Causal attention in float64: q [S, hq * d] at positions start .., k / v [n, hkv * d]."""
    S, n = q.shape[0], k.shape[0]
    q, k, v = (x.double().view(x.shape[0], -1, d) for x in (q, k, v))
    out = torch.empty(S, hq, d, device="cuda", dtype=torch.float64)
    last = start + torch.arange(S, device="cuda")
    for h in range(hq):
        g = h // (hq // hkv)
        out[:, h] = _attend(q[:, h].contiguous(), k[:n, g].contiguous(), v[:n, g].contiguous(), last)
    return out.view(S, hq * d)


def _norm_rotate(x, heads, d, w, start):
    """RMSNorm and RoPE in float64 of rows [S, heads * d]."""
    S = x.shape[0]
    x = x.double().view(S, heads, d)
    x = x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + _EPS) * w.double()
    c, s = _angles(S, d, start, torch.float64)
    return _rotate(x, c[:, None], s[:, None]).reshape(S, heads * d)


def exact(case, seed):
    t = _draw_inputs(case, seed)
    f, d = case["family"], case["head_size"]
    if f == "kv_write":
        n, hkv, bs = case["rows"], case["kv_heads"], case["block"]
        nblk = (n + bs - 1) // bs
        out = []
        for x in (t["k"], t["v"]):
            pool = torch.zeros(nblk * bs, hkv, d, device="cuda", dtype=torch.float64)
            pool[torch.from_numpy(t["slots"]).long().cuda()] = x.double()
            pool = pool.view(nblk, bs, hkv, d)
            out.append(pool.transpose(1, 2).contiguous() if case["head_major"] else pool)
        return tuple(out)
    if f == "vision":
        H, seg = case["heads"], _segments(case)
        N = sum(seg)
        x = t["qkv"].double().view(N, 3, H, d)
        c, s = (t[z].double()[:, None] for z in ("cos", "sin"))
        lo, hi = x[:, :2].chunk(2, -1)
        c1, c2 = c[:, None].chunk(2, -1)
        s1, s2 = s[:, None].chunk(2, -1)
        qk = torch.cat([lo * c1 - hi * s1, lo * s2 + hi * c2], -1)
        out = torch.empty(N, H, d, device="cuda", dtype=torch.float64)
        at = 0
        for n in seg:
            last = torch.full((n,), n - 1, device="cuda")
            for h in range(H):
                q, k, v = (y[at:at + n, h].contiguous() for y in (qk[:, 0], qk[:, 1], x[:, 2]))
                out[at:at + n, h] = _attend(q, k, v, last)
            at += n
        return out.view(N, H * d)
    hq, hkv = case["q_heads"], case["kv_heads"]
    if f == "mha_decode":
        n = case["pos"] + 1
        return _attend_heads(t["q"][None], t["k"][0, :n], t["v"][0, :n], case["pos"], hq, hkv, d)[0]
    if f == "decode_step":
        pos = case["pos"]
        kc, vc = t["k_cache"].double(), t["v_cache"].double()
        out = []
        for layer in range(case["layers"]):
            q = _norm_rotate(t["q"][layer][None], hq, d, t["wq"], pos)
            kc[layer, pos] = _norm_rotate(t["k"][layer][None], hkv, d, t["wk"], pos)[0]
            vc[layer, pos] = t["v"][layer].double()
            out.append(_attend_heads(q, kc[layer, :pos + 1], vc[layer, :pos + 1], pos, hq, hkv, d)[0])
        return torch.stack(out), kc, vc
    if f == "paged_decode":
        out = []
        table = torch.from_numpy(t["table"]).long().cuda()
        for b, n in enumerate(t["lens"].tolist()):
            rows = []
            for pool in (t["k"], t["v"]):
                blocks = pool[table[b, :(n + case["block"] - 1) // case["block"]]]
                if case["head_major"]:
                    blocks = blocks.transpose(1, 2)
                rows.append(blocks.reshape(-1, hkv * d)[:n])
            out.append(_attend_heads(t["q"][b].reshape(1, -1), rows[0], rows[1], n - 1, hq, hkv, d))
        return torch.cat(out).view(-1, hq, d)
    if f in ("prefill", "prefill_fp32"):
        return _attend_heads(t["q"], t["k"], t["v"], case["start"], hq, hkv, d)
    start, n = case["start"], case["start"] + case["seq"]
    q = _norm_rotate(t["q"], hq, d, t["wq"], start)
    kc = torch.zeros(1, n, hkv * d, device="cuda", dtype=torch.float64)
    vc = torch.zeros_like(kc)
    kc[0, start:] = _norm_rotate(t["k"], hkv, d, t["wk"], start)
    vc[0, start:] = t["v"].double()
    if f == "qk_producer":
        return q, kc, vc
    attn = _attend_heads(q, kc[0], vc[0], start, hq, hkv, d)
    return attn @ t["wo"].double().t().contiguous(), kc, vc
