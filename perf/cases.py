"""The work a user of libbq has it do, as cases that can be timed and checked.

A case is one call (or one short call sequence) through the Python binding of
libbq (`bq.py`): the decode GEMVs, the multi-row verify GEMV, the prefill
GEMMs of every weight tier, a q8 producer over a prompt batch, and two whole
steps through the captured graph (one token, one prompt chunk).  Weights are
Gaussian(0, 0.02) encoded to GGUF Q5_K / Q6_K, activations Gaussian(0, 1) in
q8 rows, as in the benchmark.  Sizes are the benchmark's (hidden 3072, FF 9216,
QKV 5120, O 3072 x 4096, vocabulary 131072) and the reference engine's
(hidden 2560, FF 7168, prompt chunks of up to 512 rows).
"""
import ctypes
import importlib
import math

import torch

bq = importlib.import_module("bruce-engine_amd.bq")

Q5, Q6 = "q5k", "q6k"


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one small projection of one token: launch latency
        {"name": "gemv_3072x3072", "kind": "gemv", "type": Q5, "K": 3072, "N": 3072, "rows": 1},
        # the FFN of one token: fused quantize + gate + up, then silu*mul norm + down
        {"name": "ffn_token_3072", "kind": "ffn", "K": 3072, "FF": 9216},
        # speculative verify: five draft tokens through gate + up
        {"name": "verify5_gate_up", "kind": "verify", "K": 3072, "N": 9216, "parts": 2, "rows": 5},
        # the ragged end of a prompt
        {"name": "tail37_9216x3072", "kind": "prefill", "type": Q5, "rep": True, "K": 3072, "N": 9216, "parts": 1,
         "rows": 37},
        # the reference engine's full prompt chunk (512 rows) through its gate + up
        {"name": "chunk512_gate_up_2560", "kind": "prefill", "type": Q5, "rep": True, "K": 2560, "N": 7168,
         "parts": 2, "rows": 512},
        # a long prompt through one FFN projection
        {"name": "prefill2048_9216x3072", "kind": "prefill", "type": Q5, "rep": True, "K": 3072, "N": 9216,
         "parts": 1, "rows": 2048},
        # the largest call: 8192 tokens
        {"name": "prefill8192_9216x3072", "kind": "prefill", "type": Q5, "rep": True, "K": 3072, "N": 9216,
         "parts": 1, "rows": 8192},
        # weights kept as GGUF blocks only (no repack held), a ragged prompt
        {"name": "prefill1000_raw_3072x4096", "kind": "prefill", "type": Q5, "rep": False, "K": 4096, "N": 3072,
         "parts": 1, "rows": 1000},
        # the down projection (Q6_K) of a long prompt
        {"name": "prefill2048_down_q6k", "kind": "prefill", "type": Q6, "rep": True, "K": 9216, "N": 3072,
         "parts": 1, "rows": 2048},
        # the FFN's silu*mul -> norm -> q8 of a long prompt
        {"name": "silu_norm_q8_2048x9216", "kind": "producer", "op": "silu", "n": 9216, "rows": 2048},
        # one decoded token: 4 layers, final norm, Q6_K lm_head (fold = 2)
        {"name": "decode_step_4_layers", "kind": "step", "E": 3072, "A": 4096, "FF": 9216, "layers": 4, "rows": 1,
         "fold": 2, "vocab": 131072, "head": Q6},
        # a 512-row prompt chunk at the reference engine's sizes: 2 layers, Q8_0 head on the last row
        {"name": "chunk_step_512_2560", "kind": "step", "E": 2560, "A": 4096, "FF": 7168, "layers": 2, "rows": 512,
         "fold": 0, "vocab": 131072, "head": "q8s"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "ffn", "verify", "prefill", "prefill", "prefill", "prefill", "producer", "step", "step"])
    if kind == "gemv":
        return {"kind": kind, "type": rng.choice([Q5, Q6]), "K": 256 * rng.randint(8, 36), "N": 16 * _log_int(rng, 32, 640),
                "rows": 1}
    if kind == "ffn":
        return {"kind": kind, "K": 256 * rng.randint(8, 16), "FF": 256 * rng.randint(20, 48)}
    if kind == "verify":
        return {"kind": kind, "K": 256 * rng.randint(8, 16), "N": 16 * _log_int(rng, 64, 640), "parts": rng.randint(1, 4),
                "rows": rng.randint(2, 8)}
    if kind == "producer":
        return {"kind": kind, "op": rng.choice(["norm", "gate", "silu"]), "n": 32 * rng.randint(64, 320),
                "rows": _log_int(rng, 1, 2048)}
    if kind == "prefill":
        t = rng.choice([Q5, Q5, Q6])
        rep = True if t == Q6 else rng.random() < 0.7
        return {"kind": kind, "type": t, "rep": rep, "K": 512 * rng.randint(4, 18), "N": 128 * rng.randint(8, 72),
                "parts": 1 if t == Q6 else rng.randint(1, 2), "rows": _log_int(rng, 9, 2048)}
    rows = 1 if rng.random() < 0.5 else _log_int(rng, 2, 512)
    return {"kind": "step", "E": 512 * rng.randint(4, 6), "A": 512 * rng.randint(4, 8), "FF": 512 * rng.randint(10, 18),
            "layers": rng.randint(1, 3), "rows": rows, "fold": rng.randint(0, 2) if rows == 1 else 0,
            "vocab": 4096 * rng.randint(2, 16), "head": rng.choice([Q6, "q8s"])}


# ---------------------------------------------------------------------------
# inputs: GGUF encoders (torch, on the GPU) and q8 rows
# ---------------------------------------------------------------------------
def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(seed * 1009 + salt)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _rows_at_a_time(K):
    return max(1, (1 << 25) // K)


def _encode_q5k(w):
    """fp32 [n, K] -> GGUF Q5_K blocks, uint8 [n, K/256 * 176]."""
    n, K = w.shape
    v = w.reshape(n, K // 256, 8, 32)
    lo, hi = v.amin(-1), v.amax(-1)
    mn = torch.clamp(-lo, min=0)
    scale = (hi + mn) / 31
    dh, mh = (scale.amax(-1) / 63).half(), (mn.amax(-1) / 63).half()
    d, dmin = dh.float()[..., None], mh.float()[..., None]
    sc = torch.where(d > 0, torch.clamp(torch.ceil(scale / d), 0, 63), 0).int()
    m = torch.where(dmin > 0, torch.clamp(torch.ceil(mn / dmin), 0, 63), 0).int()
    ds, dm = (d * sc)[..., None], (dmin * m)[..., None]
    u = torch.where(ds > 0, torch.round((v + dm) / ds), 0).clamp(0, 31).to(torch.uint8)
    out = torch.zeros((n, K // 256, 176), dtype=torch.uint8, device=w.device)
    out[..., 0:2] = dh.contiguous().view(torch.uint8).reshape(n, K // 256, 2)
    out[..., 2:4] = mh.contiguous().view(torch.uint8).reshape(n, K // 256, 2)
    out[..., 4:8] = (sc[..., :4] | ((sc[..., 4:] >> 4) << 6)).to(torch.uint8)
    out[..., 8:12] = (m[..., :4] | ((m[..., 4:] >> 4) << 6)).to(torch.uint8)
    out[..., 12:16] = ((sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)).to(torch.uint8)
    for j in range(8):
        out[..., 16:48] |= (u[..., j, :] >> 4) << j
    out[..., 48:176] = ((u[..., 0::2, :] & 15) | ((u[..., 1::2, :] & 15) << 4)).reshape(n, K // 256, 128)
    return out.reshape(n, -1)


def _encode_q6k(w):
    """fp32 [n, K] -> GGUF Q6_K blocks, uint8 [n, K/256 * 210]."""
    n, K = w.shape
    v = w.reshape(n, K // 256, 16, 16)
    a = v.abs()
    top = torch.gather(v, -1, a.argmax(-1, keepdim=True))[..., 0]
    dh = (a.amax(-1) / 31).amax(-1).div(127).half()
    d = dh.float()[..., None]
    r = torch.where(d > 0, top / 31 / d, 0)
    sc = torch.clamp(torch.where(r < 0, torch.floor(r), torch.ceil(r)), -127, 127).int()
    s = (d * sc)[..., None]
    q = (torch.where(s != 0, torch.round(v / s), 0).clamp(-32, 31) + 32).to(torch.uint8).reshape(n, K // 256, 2, 4, 32)
    out = torch.zeros((n, K // 256, 210), dtype=torch.uint8, device=w.device)
    out[..., 0:128] = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4),
                                 (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -1).reshape(n, K // 256, 128)
    qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
    out[..., 128:192] = qh.reshape(n, K // 256, 64)
    out[..., 192:208] = sc.to(torch.int8).view(torch.uint8)
    out[..., 208:210] = dh.contiguous().view(torch.uint8).reshape(n, K // 256, 2)
    return out.reshape(n, -1)


def _blocks(g, kind, K, N):
    enc = _encode_q5k if kind == Q5 else _encode_q6k
    step = _rows_at_a_time(K)
    return torch.cat([enc(_randn(g, min(step, N - i), K) * 0.02) for i in range(0, N, step)])


def _weight(g, kind, K, N, rep):
    """(bq_weight, raw blocks): rep also holds the prefill repack (W144 + Dm / W160)."""
    raw = _blocks(g, kind, K, N)
    t = bq.TYPE_Q5_K if kind == Q5 else bq.TYPE_Q6_K
    if not rep:
        return bq.make_weight(raw, t, K, N), raw
    if kind == Q5:
        w144, dm = bq.repack_q5k(raw, K, N)
        return bq.make_weight(raw, t, K, N, rep=w144, rep_min=dm), raw
    return bq.make_weight(raw, t, K, N, rep=bq.repack_q6k(raw, K, N)), raw


def _q8(x):
    """q8 rows of fp32 [rows, K]: codes, group scales, code sums."""
    rows, K = x.shape
    v = x.reshape(rows, K // 32, 32)
    d = v.abs().amax(-1) * torch.tensor(1 / 127, dtype=torch.float32, device=x.device)
    inv = torch.where(d > 0, 1 / d, 0)
    q = torch.clamp(torch.round(v * inv[..., None]), -127, 127)
    return q.to(torch.int8).reshape(rows, K), d, q.sum(-1).int()


def _head_bf16(g, E, V):
    step = _rows_at_a_time(E)
    return torch.cat([(_randn(g, min(step, V - i), E) * 0.02).bfloat16() for i in range(0, V, step)])


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_gemv(c, seed):
    w, _ = _weight(_gen(seed, 1), c["type"], c["K"], c["N"], False)
    q = _q8(_randn(_gen(seed, 2), 1, c["K"]))
    return {"run": _run_gemv, "w": w, "q": q, "y": torch.empty((1, c["N"]), device="cuda")}


def _run_gemv(s):
    return bq.gemv(s["y"], s["w"], *s["q"])


def _ffn_vectors(seed, n):
    g = _gen(seed, 7)
    return [1 + 0.3 * _randn(g, n) for _ in range(2)]


def _prepare_ffn(c, seed):
    K, FF = c["K"], c["FF"]
    gate, up, down = (_weight(_gen(seed, i), t, k, n, False)[0]
                      for i, t, k, n in ((1, Q5, K, FF), (2, Q5, K, FF), (3, Q6, FF, K)))
    sg, su = _ffn_vectors(seed, FF)
    y = [torch.empty(n, device="cuda") for n in (FF, FF, K)]
    return {"run": _run_ffn, "gate": gate, "up": up, "down": down, "sg": sg, "su": su,
            "x": _randn(_gen(seed, 4), K), "y": y}


def _run_ffn(s):
    g, u, y = s["y"]
    bq.gemv_q8_fused([g, u], [s["gate"], s["up"]], s["x"])
    bq.gemv_norm_fused([y], [s["down"]], "silu", g, u, s["sg"], s["su"])
    return s["y"]


def _prepare_verify(c, seed):
    ws = [_weight(_gen(seed, i), Q5, c["K"], c["N"], False)[0] for i in range(c["parts"])]
    q = _q8(_randn(_gen(seed, 20), c["rows"], c["K"]))
    return {"run": _run_verify, "ws": ws, "q": q, "rows": c["rows"],
            "ys": [torch.empty((c["rows"], c["N"]), device="cuda") for _ in ws]}


def _run_verify(s):
    bq.verify_fused(s["ys"], s["ws"], s["rows"], *s["q"])
    return s["ys"]


def _prepare_prefill(c, seed):
    ws = [_weight(_gen(seed, i), c["type"], c["K"], c["N"], c["rep"])[0] for i in range(c["parts"])]
    q = _q8(_randn(_gen(seed, 20), c["rows"], c["K"]))
    return {"run": _run_prefill, "ws": ws, "q": q, "rows": c["rows"],
            "xdh": torch.empty((c["rows"], c["K"] // 32), dtype=torch.int16, device="cuda"),
            "ys": [torch.empty((c["rows"], c["N"]), device="cuda") for _ in ws]}


def _run_prefill(s):
    bq.gemm_b_fused(s["ys"], s["ws"], s["rows"], *s["q"], s["xdh"])
    return s["ys"]


def _producer_inputs(c, seed):
    g = _gen(seed, 1)
    a, b = (_randn(g, c["rows"], c["n"]) for _ in range(2))
    return a, b, *_ffn_vectors(seed, c["n"])


def _prepare_producer(c, seed):
    a, b, sg, su = _producer_inputs(c, seed)
    rows, n = c["rows"], c["n"]
    q = (torch.empty((rows, n), dtype=torch.int8, device="cuda"), torch.empty((rows, n // 32), device="cuda"),
         torch.empty((rows, n // 32), dtype=torch.int32, device="cuda"))
    args = {"norm": {"a": a}, "gate": {"a": a, "b": b, "c": sg}, "silu": {"a": a, "b": b, "c": sg, "d": su}}[c["op"]]
    return {"run": _run_producer, "op": c["op"], "rows": rows, "n": n, "args": args, "q": q}


def _run_producer(s):
    bq.norm_q8(s["op"], s["rows"], s["n"], q8=s["q"], **s["args"])
    return s["q"]


def _step_parts(c):
    """QKV parts of the step: q, k, gate, v (the V projection is Q6_K)."""
    return [(c["A"], Q5), (512, Q5), (c["A"], Q5), (512, Q6)]


def _step_inputs(c, seed):
    """The step's weights' raw blocks, vectors and token rows, in one order."""
    E, A, FF, R = c["E"], c["A"], c["FF"], c["rows"]
    layers = []
    for l in range(c["layers"]):
        g = _gen(seed, 100 + l)
        L = {"qkv": [(t, E, n, _blocks(g, t, E, n)) for n, t in _step_parts(c)],
             "o": (Q5, A, E, _blocks(g, Q5, A, E)), "gate": (Q5, E, FF, _blocks(g, Q5, E, FF)),
             "up": (Q5, E, FF, _blocks(g, Q5, E, FF)), "down": (Q6, FF, E, _blocks(g, Q6, FF, E)),
             "attn_out": _randn(g, R, A), "sgate": 1 + 0.3 * _randn(g, A), "sg": 1 + 0.3 * _randn(g, FF),
             "su": 1 + 0.3 * _randn(g, FF), "alpha_a": 0.5 + 0.2 * _randn(g, E), "alpha_f": 0.5 + 0.2 * _randn(g, E)}
        layers.append(L)
    g = _gen(seed, 99)
    head = _head_bf16(g, E, c["vocab"]) if c["head"] == "q8s" else _blocks(g, c["head"], E, c["vocab"])
    return layers, head, _randn(g, R, E)


def _prepare_step(c, seed):
    E, A, FF, R, V = c["E"], c["A"], c["FF"], c["rows"], c["vocab"]
    layers, head, emb = _step_inputs(c, seed)
    keep = [layers, head, emb]

    def weight(t, K, N, raw):
        rep = rmin = None
        if R > 1 and t == Q6:
            rep = bq.repack_q6k(raw, K, N)
        elif R > 8:
            rep, rmin = bq.repack_q5k(raw, K, N)
        w = bq.make_weight(raw, bq.TYPE_Q5_K if t == Q5 else bq.TYPE_Q6_K, K, N, rep=rep, rep_min=rmin)
        keep.append(w)
        return w

    f32 = lambda *shape: torch.empty(shape, device="cuda")
    top = max(E, A, FF)
    buf = {"x": f32(R, E), "x_alt": f32(E), "proj": f32(R, E), "ffn_g": f32(R, FF), "ffn_u": f32(R, FF),
           "logits": f32(R if R <= 8 else 1, V), "xq": torch.empty(R * top, dtype=torch.int8, device="cuda"),
           "xd": f32(R * top // 32), "xsum": torch.empty(R * top // 32, dtype=torch.int32, device="cuda"),
           "xdh": torch.empty(R * top // 32, dtype=torch.int16, device="cuda")}
    blocks = (bq.DecodeBlock * (2 * c["layers"]))()
    for l, L in enumerate(layers):
        a, f = blocks[2 * l], blocks[2 * l + 1]
        qkv = (bq.Weight * 4)(*[weight(*p) for p in L["qkv"]])
        outs = [f32(R, n) for n, _ in _step_parts(c)]
        ptrs = (ctypes.c_void_p * 4)(*[o.data_ptr() for o in outs])
        keep += [qkv, outs, ptrs]
        a.kind, a.alpha = bq.BLOCK_ATTN, L["alpha_a"].data_ptr()
        a.qkv, a.n_qkv, a.qkv_out = qkv, 4, ptrs
        a.attn_out, a.attn_gate = L["attn_out"].data_ptr(), outs[2].data_ptr()
        a.sgate, a.n_attn, a.o = L["sgate"].data_ptr(), A, ctypes.pointer(weight(*L["o"]))
        f.kind, f.alpha = bq.BLOCK_FFN, L["alpha_f"].data_ptr()
        f.gate, f.up, f.down = (ctypes.pointer(weight(*L[k])) for k in ("gate", "up", "down"))
        f.s_gate, f.s_up, f.n_ff = L["sg"].data_ptr(), L["su"].data_ptr(), FF
    blocks[-1].norm_after = 1
    s = bq.DecodeStep()
    s.n_blocks, s.blocks, s.n_embd, s.fold, s.rows, s.vocab = len(blocks), blocks, E, c["fold"], R, V
    for k in ("x", "x_alt", "xq", "xd", "xsum", "proj", "ffn_g", "ffn_u", "logits", "xdh"):
        setattr(s, k, buf[k].data_ptr())
    if c["head"] == "q8s":
        q8s = bq.quantize_q8s(head.view(torch.int16), E, V)
        keep.append(q8s)
        s.head_q8s = q8s.data_ptr()
    else:
        s.head = ctypes.pointer(weight(c["head"], E, V, head))
    if R > 8:
        n = max(bq.workspace_bytes(R, k, m) for k, m in ((E, 2 * A + 512), (E, 512), (A, E), (E, 2 * FF), (FF, E)))
        work = f32(max(n, 16) // 4)
        keep.append(work)
        s.work, s.work_bytes = work.data_ptr(), work.numel() * 4
    keep.append(blocks)
    return {"run": _run_step, "emb": emb, "buf": buf, "q": (buf["xq"], buf["xd"], buf["xsum"]), "rows": R, "E": E,
            "graph": bq.DecodeGraph(s), "keep": keep}


def _run_step(s):
    # the step's input: the tokens' embeddings, normalised into x and its q8 rows
    bq.norm_q8("norm", s["rows"], s["E"], out=s["buf"]["x"], a=s["emb"], q8=s["q"])
    s["graph"].launch()
    return {"logits": s["buf"]["logits"], "x": s["buf"]["x"]}


_PREPARE = {"gemv": _prepare_gemv, "ffn": _prepare_ffn, "verify": _prepare_verify, "prefill": _prepare_prefill,
            "producer": _prepare_producer, "step": _prepare_step}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _wbytes(t, K, N):
    return N * (K // 256) * (176 if t == Q5 else 210)


def _q8_bytes(rows, n):
    return rows * (n + n // 32 * 8)


def work(case):
    """Weights at their GGUF size, q8 or fp32 inputs read once, outputs written once."""
    c = case
    if c["kind"] in ("gemv", "verify", "prefill"):
        parts, t = c.get("parts", 1), c.get("type", Q5)
        return {"bytes": parts * (_wbytes(t, c["K"], c["N"]) + 4 * c["rows"] * c["N"]) + _q8_bytes(c["rows"], c["K"]),
                "flops": 2 * parts * c["rows"] * c["K"] * c["N"]}
    if c["kind"] == "ffn":
        K, FF = c["K"], c["FF"]
        return {"bytes": 2 * _wbytes(Q5, K, FF) + _wbytes(Q6, FF, K) + 4 * (K + 2 * FF + 2 * FF + K),
                "flops": 6 * K * FF}
    if c["kind"] == "producer":
        rows, n = c["rows"], c["n"]
        ins, vecs = {"norm": (1, 0), "gate": (2, 1), "silu": (2, 2)}[c["op"]]
        return {"bytes": 4 * n * (rows * ins + vecs) + _q8_bytes(rows, n), "flops": 10 * rows * n}
    E, A, FF, R, V = c["E"], c["A"], c["FF"], c["rows"], c["vocab"]
    mats = [(t, E, n) for n, t in _step_parts(c)] + [(Q5, A, E), (Q5, E, FF), (Q5, E, FF), (Q6, FF, E)]
    lr = R if R <= 8 else 1
    head = V * (E // 256) * 272 if c["head"] == "q8s" else _wbytes(c["head"], E, V)
    return {"bytes": c["layers"] * (sum(_wbytes(*m) for m in mats) + 4 * (R * A + A + 2 * FF + 2 * E)) + head
            + 4 * (2 * R * E + lr * V),
            "flops": 2 * (c["layers"] * R * sum(k * n for _, k, n in mats) + lr * E * V)}


def tolerance(case):
    """About four times the error measured against the same path in 64 bits."""
    c = case
    if c["kind"] == "producer":
        return {"rel": 1e-6, "max": 1e-5, "differ": 1e-4}
    if c["kind"] == "prefill":
        # W144 rounds the min term's operands to fp16 (6e-4); the other tiers sum in fp32 (4e-7)
        return {"rel": 2.5e-3 if c["rep"] and c["type"] == Q5 else 2e-6}
    if c["kind"] == "ffn":
        # one q8 code that rounds the other way moves a row by about 3e-4
        return {"rel": 1e-3}
    if c["kind"] == "step":
        # codes that round the other way in every layer; a prompt chunk has the fp16 min term
        # in front of them (1.3e-2 against 64 bits after two layers)
        return {"rel": 4e-3 if c["rows"] <= 8 else 1.5e-2}
    return {"rel": 1e-6}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _decode_q5k(raw, K):
    """GGUF Q5_K blocks -> float64 weights [n, K]."""
    n = raw.shape[0]
    b = raw.reshape(n, K // 256, 176)
    half = lambda x: x.contiguous().view(torch.float16).double()
    d, dmin = half(b[..., 0:2]), half(b[..., 2:4])
    s = b[..., 4:16].int()
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
    m = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
    qs = b[..., 48:176].reshape(n, K // 256, 4, 1, 32)
    u = torch.cat([qs & 15, qs >> 4], 3).reshape(n, K // 256, 8, 32)
    hi = torch.stack([(b[..., 16:48] >> j) & 1 for j in range(8)], 2)
    return ((d * sc)[..., None] * (u + 16 * hi) - (dmin * m)[..., None]).reshape(n, K)


def _decode_q6k(raw, K):
    """GGUF Q6_K blocks -> float64 weights [n, K]."""
    n = raw.shape[0]
    b = raw.reshape(n, K // 256, 210)
    ql = b[..., 0:128].reshape(n, K // 256, 2, 2, 32)
    qh = b[..., 128:192].reshape(n, K // 256, 2, 1, 32)
    q = torch.stack([(ql[..., u & 1, :] >> (4 * (u >> 1)) & 15) | (((qh[..., 0, :] >> (2 * u)) & 3) << 4)
                     for u in range(4)], 3)
    sc = b[..., 192:208].contiguous().view(torch.int8).double() * b[..., 208:210].contiguous().view(torch.float16).double()
    return (sc[..., None] * (q.double() - 32).reshape(n, K // 256, 16, 16)).reshape(n, K)


def _matmul(x, t, K, N, raw):
    """x [rows, K] float64 times the weight's rows."""
    dec = _decode_q5k if t == Q5 else _decode_q6k
    step = _rows_at_a_time(K)
    return torch.cat([x @ dec(raw[i:i + step], K).T for i in range(0, N, step)], 1)


def _dequant(q):
    return (q[0].double().reshape(*q[1].shape, 32) * q[1].double()[..., None]).reshape(q[0].shape)


def _q8_64(v):
    """q8 rows of float64 rows: codes, scales, code sums."""
    t = v.reshape(v.shape[0], -1, 32)
    d = t.abs().amax(-1) / 127
    q = torch.round(torch.where(d[..., None] > 0, t / d[..., None], 0))
    return q.reshape(v.shape), d, q.sum(-1)


def _through_q8(v):
    return _dequant(_q8_64(v))


def _norm(t):
    """t * l2_scale: (1 / sqrt(ss / n + eps / n)) * (1 / sqrt(n)) = 1 / sqrt(ss + eps)."""
    return t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)


def _silu_mul(g, u, sg, su):
    gv = g * sg.double()
    return gv / (1 + torch.exp(-gv)) * u * su.double()


def _gated(a, gate, sg):
    return a / (1 + torch.exp(-gate * sg.double()))


def exact(case, seed):
    c = case
    if c["kind"] == "gemv":
        raw = _blocks(_gen(seed, 1), c["type"], c["K"], c["N"])
        return _matmul(_dequant(_q8(_randn(_gen(seed, 2), 1, c["K"]))), c["type"], c["K"], c["N"], raw)
    if c["kind"] in ("verify", "prefill"):
        x = _dequant(_q8(_randn(_gen(seed, 20), c["rows"], c["K"])))
        t = c.get("type", Q5)
        return [_matmul(x, t, c["K"], c["N"], _blocks(_gen(seed, i), t, c["K"], c["N"])) for i in range(c["parts"])]
    if c["kind"] == "ffn":
        K, FF = c["K"], c["FF"]
        sg, su = _ffn_vectors(seed, FF)
        x = _dequant(_q8(_randn(_gen(seed, 4), K)[None]))
        g, u = (_matmul(x, Q5, K, FF, _blocks(_gen(seed, i), Q5, K, FF)) for i in (1, 2))
        t = _through_q8(_norm(_silu_mul(g, u, sg, su)))
        return [g[0], u[0], _matmul(t, Q6, FF, K, _blocks(_gen(seed, 3), Q6, FF, K))[0]]
    if c["kind"] == "producer":
        a, b, sg, su = _producer_inputs(c, seed)
        a, b = a.double(), b.double()
        t = {"norm": lambda: a, "gate": lambda: _gated(a, b, sg), "silu": lambda: _silu_mul(a, b, sg, su)}[c["op"]]()
        q, d, s = _q8_64(_norm(t))
        return q.to(torch.int8), d, s.int()
    layers, head, emb = _step_inputs(c, seed)
    x = _norm(emb.double())
    for i, L in enumerate(layers):
        _, K, N, raw = L["qkv"][2]
        gate = _matmul(_through_q8(x), Q5, K, N, raw)
        t = _through_q8(_norm(_gated(L["attn_out"].double(), gate, L["sgate"])))
        for p, alpha in ((_matmul(t, *L["o"]), L["alpha_a"]), (None, L["alpha_f"])):
            if p is None:
                xq = _through_q8(x)
                t = _through_q8(_norm(_silu_mul(_matmul(xq, *L["gate"]), _matmul(xq, *L["up"]), L["sg"], L["su"])))
                p = _matmul(t, *L["down"])
            a, b = _norm(x), _norm(p)
            x = _norm(a + (b - a) * alpha.double())
    x = _norm(x)
    xq = _through_q8(x if c["rows"] <= 8 else x[-1:])
    if c["head"] == "q8s":
        h = head.float().reshape(c["vocab"], -1, 32)
        d = h.abs().amax(-1) * torch.tensor(1 / 127, dtype=torch.float32, device=h.device)
        q = torch.round(h * torch.where(d > 0, 1 / d, 0)[..., None]).clamp(-127, 127)
        del h
        step = 16384
        logits = torch.cat([xq @ (q[i:i + step].double() * d[i:i + step].half().double()[..., None])
                            .reshape(-1, c["E"]).T for i in range(0, c["vocab"], step)], 1)
    else:
        logits = _matmul(xq, c["head"], c["E"], c["vocab"], head)
    return {"logits": logits, "x": x}
