"""The measured work of the quantised projections: what a model built on this library calls.

Kinds of case, each one pass over the public entry points of splosh_amd.runtime:

* ``projection`` -- one small eager call with every default (output and scratch made by the call):
  the latency of a single key or value projection of one token.
* ``layer`` -- the linear projections of one hybrid layer set on MLX affine q4 weights: attention
  q/k/v as one grouped call and o onto the fp32 residual, the gated-delta input, its two 48-row
  row-major a/b projections and its output, the MLP's fused gate+up and its down projection onto
  the residual. Above four rows the two residual projections also emit the next norm's operand.
* ``ends`` -- the two ends of the model on one q4 table: the embedding lookup of the rows' tokens,
  the bf16 operand from it, and the lm_head over the whole vocabulary.
* ``gguf_mlp`` -- the MLP on GGUF weights: gate and up projections to fp32, silu(gate) * up as the
  next operand, the down projection onto the fp32 residual (GGUF files mix types: the down
  projection of a K-quant file usually has a wider one).

Up to 64 rows (decode, draft and verify steps) a serving loop replays a captured HIP graph of its
layer, so the ``layer`` and ``gguf_mlp`` passes are one replay of the captured calls there; above
that (prefill) and for the other kinds the calls are made eagerly. Outputs and one shared scratch
are kept by the caller between passes, as an engine does, except in ``projection``.

Shapes are those of the library's benchmark workloads (hidden 5120, MLP 17408, vocabulary 248320)
and, in drawn cases, smaller ones of the same form.
"""
import math

import torch

from splosh_amd import runtime as rt

# GGUF type -> (ggml id, elements a block, bytes a block, byte offset of the fp16 scale, its size):
# random blocks with that scale give weights of about the size trained ones have.
GGUF = {
    "q4_k": (12, 256, 144, 0, 2.0e-4),
    "q5_k": (13, 256, 176, 0, 1.0e-4),
    "q6_k": (14, 256, 210, 208, 1.0e-4),
    "q8_0": (8, 32, 34, 0, 2.5e-4),
    "q3_k": (11, 256, 110, 108, 4.5e-4),
    "iq4_nl": (20, 32, 18, 0, 2.7e-4),
    "iq4_xs": (23, 256, 136, 0, 1.0e-4),
}
IQ4_VALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
AB_ROWS = 48  # outputs of the gated-delta a and b projections
LAYER = {"hidden": 5120, "q": 5120, "kv": 1024, "gdn_in": 12288, "gdn_out": 6144, "inter": 17408}


def listed():
    def layer(name, rows):
        return {"name": name, "kind": "layer", "rows": rows, **LAYER}

    def ends(name, rows):
        return {"name": name, "kind": "ends", "rows": rows, "hidden": 5120, "vocab": 248320}

    def gguf(name, rows, wide, down, rows32=False):
        return {"name": name, "kind": "gguf_mlp", "rows": rows, "hidden": 5120, "inter": 17408, "type": wide,
                "down": down, "rows32": rows32}

    return [
        # One key projection of one token: the smallest call, all latency.
        {"name": "projection_1", "kind": "projection", "rows": 1, "hidden": 5120, "outputs": 1024},
        # One token of plain decoding through a layer set, and through the vocabulary.
        layer("decode_layer_1", 1),
        ends("decode_ends_1", 1),
        # Eight drafted tokens of one session.
        layer("draft_layer_8", 8),
        # Eight sessions of eight drafted tokens verified together, and the logits of an odd batch.
        layer("verify_layer_64", 64),
        ends("verify_ends_37", 37),
        # A ragged prompt, and a whole prefill step.
        layer("prompt_layer_333", 333),
        layer("prefill_layer_2048", 2048),
        # GGUF files: decoding a Q5_K_M-like one, verifying a Q4_K_M-like one, a batch on Q8_0
        # (repacked once for batched calls), and prefill.
        gguf("gguf_decode_1", 1, "q5_k", "q6_k"),
        gguf("gguf_verify_24", 24, "q4_k", "q6_k"),
        gguf("gguf_batch_16", 16, "q8_0", "q8_0", True),
        gguf("gguf_prefill_1024", 1024, "q4_k", "q6_k"),
    ]


def _between(rng, low, high, step):
    """A multiple of `step` from low to high, even over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))) / step)) * step))


def _rows(rng):
    """1 to 2048 rows: decode, draft and verify, prompts; odd counts among them."""
    return rng.choice([1, rng.randint(1, 4), rng.randint(5, 32), rng.randint(33, 128),
                       _between(rng, 129, 2048, 1)])


def draw(rng):
    kind = rng.choice(["projection", "layer", "layer", "layer", "ends", "gguf_mlp", "gguf_mlp", "gguf_mlp"])
    if kind == "projection":
        return {"kind": kind, "rows": rng.randint(1, 4), "hidden": _between(rng, 1024, 5120, 64),
                "outputs": _between(rng, 128, 2048, 128)}
    hidden = _between(rng, 1536, 5120, 256)
    if kind == "ends":
        return {"kind": kind, "rows": rng.choice([1, rng.randint(1, 4), rng.randint(5, 64)]), "hidden": hidden,
                "vocab": _between(rng, 32768, 248320, 128)}
    if kind == "layer":
        return {"kind": kind, "rows": _rows(rng), "hidden": hidden, "q": _between(rng, 1536, 5120, 128),
                "kv": _between(rng, 256, 1024, 128), "gdn_in": _between(rng, 3072, 12288, 128),
                "gdn_out": _between(rng, 1536, 6144, 64), "inter": _between(rng, 4096, 17408, 128)}
    wide = rng.choice(sorted(GGUF))
    down = rng.choice([wide, "q6_k", "q8_0", "q5_k"])
    return {"kind": kind, "rows": min(_rows(rng), 1024), "hidden": hidden, "inter": _between(rng, 4096, 17408, 256),
            "type": wide, "down": down, "rows32": rng.random() < 0.5}


# ---- inputs, from the seed alone ----------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(seed * 1000 + salt)


def _q4(n, k, seed, salt):
    """(codes int32 [n * k / 8], scales, biases bf16 [n * k / 64]) in record order: codes of every
    value, biases that centre the weights, as a quantiser of trained weights leaves them."""
    gen = _gen(seed, salt)
    codes = torch.randint(-2**31, 2**31 - 1, (n * k // 8,), dtype=torch.int32, device="cuda", generator=gen)
    scales = 0.004 * (0.75 + 0.5 * torch.rand(n * k // 64, device="cuda", generator=gen))
    biases = -scales * (7.5 + 0.5 * torch.randn(n * k // 64, device="cuda", generator=gen))
    return codes, scales.to(torch.bfloat16), biases.to(torch.bfloat16)


def _q4_weight(n, k, seed, salt, order=rt.TILED128):
    codes, scales, biases = _q4(n, k, seed, salt)
    stride = 0 if order == rt.TILED128 else k // 8
    return rt.Q4Weight(codes, scales.view(torch.int16), biases.view(torch.int16), n, k, order, stride)


def _blocks(kind, n, k, seed, salt):
    """Native GGUF blocks [n, k / elements, bytes] (uint8)."""
    _, elems, size, at, mag = GGUF[kind]
    gen = _gen(seed, salt)
    raw = torch.randint(0, 256, (n * (k // elems), size), dtype=torch.uint8, device="cuda", generator=gen)
    fields = [(at, mag)] + ([(2, 15.5 * mag if kind == "q5_k" else 7.5 * mag)] if kind in ("q4_k", "q5_k") else [])
    for offset, value in fields:
        v = value * (0.75 + 0.5 * torch.rand(raw.shape[0], device="cuda", generator=gen))
        raw[:, offset:offset + 2] = v.to(torch.float16).view(torch.uint8).view(-1, 2)
    return raw.view(n, k // elems, size)


def _gguf_weight(kind, n, k, seed, salt, rows32):
    raw = _blocks(kind, n, k, seed, salt).reshape(-1)
    if kind == "q5_k":
        return rt.q5k_repack(raw, n, k)
    if kind == "q4_k":
        return rt.q4k_repack(raw, n, k)
    w = rt.GgufWeight(raw, GGUF[kind][0], n, k)
    return rt.gguf_repack_rows32(w) if rows32 else w


def _act(rows, k, seed, salt):
    return torch.randn(rows, k, device="cuda", generator=_gen(seed, salt)).to(torch.bfloat16)


def _residual(rows, n, seed, salt):
    return torch.randn(rows, n, device="cuda", generator=_gen(seed, salt))


def _norm(n, seed, salt):
    return (1 + 0.1 * torch.randn(n, device="cuda", generator=_gen(seed, salt))).to(torch.bfloat16)


def _tokens(case, seed):
    return torch.randint(0, case["vocab"], (case["rows"],), dtype=torch.int32, device="cuda", generator=_gen(seed, 2))


def _scratch(rows, shapes):
    need = max(rt.workspace_bytes(rows, n, k) for n, k in shapes)
    return torch.zeros(max(need, 1), dtype=torch.uint8, device="cuda")


def _layer_inputs(case, seed):
    m, h = case["rows"], case["hidden"]
    return {"x": _act(m, h, seed, 20), "attn": _act(m, case["q"], seed, 21), "gdn": _act(m, case["gdn_out"], seed, 22),
            "y": _act(m, h, seed, 23), "res": _residual(m, h, seed, 24), "norm": _norm(h, seed, 25)}


def _layer_shapes(case):
    h = case["hidden"]
    return {"wq": (case["q"], h), "wk": (case["kv"], h), "wv": (case["kv"], h), "wo": (h, case["q"]),
            "win": (case["gdn_in"], h), "wout": (h, case["gdn_out"]), "wgate": (case["inter"], h),
            "wup": (case["inter"], h), "wdown": (h, case["inter"])}


def prepare(case, seed):
    m, h = case["rows"], case["hidden"]
    bf16 = torch.bfloat16
    state = {"case": case}

    def empty(n, dtype=bf16):
        return torch.empty(m, n, dtype=dtype, device="cuda")

    if case["kind"] == "projection":
        state.update(w=_q4_weight(case["outputs"], h, seed, 1), x=_act(m, h, seed, 20))
        return state
    if case["kind"] == "ends":
        state.update(w=_q4_weight(case["vocab"], h, seed, 1), tokens=_tokens(case, seed),
                     embedded=empty(h, torch.float32), operand=empty(h),
                     sums=torch.empty(m, h // 64, device="cuda"), logits=empty(case["vocab"]),
                     scratch=_scratch(m, [(case["vocab"], h)]))
        return state
    if case["kind"] == "layer":
        shapes = _layer_shapes(case)
        for i, (name, (n, k)) in enumerate(shapes.items()):
            state[name] = _q4_weight(n, k, seed, i + 1)
        for i, name in enumerate(("wa", "wb")):
            state[name] = _q4_weight(AB_ROWS, h, seed, 40 + i, rt.ROW_MAJOR)
        state.update(_layer_inputs(case, seed))
        state["qkv"] = [empty(case["q"]), empty(case["kv"]), empty(case["kv"])]
        state.update(a=empty(AB_ROWS), b=empty(AB_ROWS), z=empty(case["gdn_in"]), g=empty(h),
                     act=empty(case["inter"]), h1=empty(h, torch.float32), h2=empty(h, torch.float32),
                     scratch=_scratch(m, list(shapes.values()) + [(AB_ROWS, h), (case["q"] + 2 * case["kv"], h)]))
    else:
        inter = case["inter"]
        state.update(wgate=_gguf_weight(case["type"], inter, h, seed, 1, case["rows32"]),
                     wup=_gguf_weight(case["type"], inter, h, seed, 2, case["rows32"]),
                     wdown=_gguf_weight(case["down"], h, inter, seed, 3, case["rows32"]),
                     x=_act(m, h, seed, 20), res=_residual(m, h, seed, 24),
                     gate=empty(inter, torch.float32), up=empty(inter, torch.float32), act=empty(inter),
                     sums=torch.empty(m, inter // 64, device="cuda"), out=empty(h, torch.float32),
                     scratch=_scratch(m, [(inter, h), (h, inter)]))
    if m <= 64:
        _calls(state)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outputs = _calls(state)
        state.update(graph=graph, outputs=outputs)
    return state


# ---- one pass -----------------------------------------------------------------------------------


def _residual_projection(s, w, a, out):
    """out = res + a w^T in fp32; above four rows with the next norm's operand."""
    if s["case"]["rows"] > 4:
        return rt.gemm_emit(w, a, s["norm"], out=out, residual=s["res"], workspace=s["scratch"])
    return (rt.gemm(w, a, out=out, residual=s["res"], workspace=s["scratch"]),)


def _calls(s):
    kind, ws = s["case"]["kind"], s.get("scratch")
    if kind == "projection":
        return rt.gemm(s["w"], s["x"])
    if kind == "ends":
        rt.embed(s["w"], s["tokens"], out=s["embedded"])
        rt.prepare_operand(s["embedded"], out=s["operand"], sums=s["sums"])
        rt.gemm(s["w"], s["operand"], out=s["logits"], workspace=ws)
        return {k: s[k] for k in ("embedded", "operand", "sums", "logits")}
    if kind == "layer":
        rt.gemm_group([s["wq"], s["wk"], s["wv"]], s["x"], outs=s["qkv"], workspace=ws)
        hidden = _residual_projection(s, s["wo"], s["attn"], s["h1"])
        rt.gemm(s["win"], s["x"], out=s["z"], workspace=ws)
        rt.gemm(s["wa"], s["x"], out=s["a"], workspace=ws)
        rt.gemm(s["wb"], s["x"], out=s["b"], workspace=ws)
        rt.gemm(s["wout"], s["gdn"], out=s["g"], workspace=ws)
        rt.mlp_in(s["wgate"], s["wup"], s["y"], out=s["act"], workspace=ws)
        out = _residual_projection(s, s["wdown"], s["act"], s["h2"])
        return {"qkv": s["qkv"], "o": hidden, "z": s["z"], "a": s["a"], "b": s["b"], "g": s["g"], "act": s["act"],
                "down": out}
    rt.gemm(s["wgate"], s["x"], out=s["gate"], workspace=ws)
    rt.gemm(s["wup"], s["x"], out=s["up"], workspace=ws)
    rt.silu_mul_operand(s["gate"], s["up"], out=s["act"], sums=s["sums"])
    rt.gemm(s["wdown"], s["act"], out=s["out"], residual=s["res"], workspace=ws)
    return {k: s[k] for k in ("gate", "up", "act", "sums", "out")}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return _calls(state)


# ---- what a pass cannot do without --------------------------------------------------------------


def _q4_bytes(n, k):
    return n * k // 2 + n * (k // 64) * 4


def work(case):
    m, h = case["rows"], case["hidden"]
    if case["kind"] == "projection":
        n = case["outputs"]
        return {"bytes": _q4_bytes(n, h) + 2 * m * (h + n), "flops": 2 * m * n * h}
    if case["kind"] == "ends":
        n = case["vocab"]
        # The embedded rows are read from the table and written as fp32 and bf16.
        return {"bytes": _q4_bytes(n, h) + m * _q4_bytes(1, h) + m * h * 6 + m * (h // 64) * 4 + 2 * m * n,
                "flops": 2 * m * n * h}
    if case["kind"] == "layer":
        shapes = list(_layer_shapes(case).values()) + [(AB_ROWS, h)] * 2
        weights = sum(_q4_bytes(n, k) for n, k in shapes)
        inputs = 2 * m * (2 * h + case["q"] + case["gdn_out"]) + 4 * m * h
        outputs = 2 * m * (case["q"] + 2 * case["kv"] + case["gdn_in"] + 2 * AB_ROWS + h + case["inter"]) + 8 * m * h
        if m > 4:
            outputs += 2 * (2 * m * h + 8 * m * (h // 64))
        return {"bytes": weights + inputs + outputs, "flops": 2 * m * sum(n * k for n, k in shapes)}
    inter = case["inter"]

    def size(kind, n, k):
        _, elems, block, _, _ = GGUF[kind]
        return n * (k // elems) * block

    weights = 2 * size(case["type"], inter, h) + size(case["down"], h, inter)
    return {"bytes": weights + m * (2 * h + 8 * inter + 2 * inter + 4 * (inter // 64) + 8 * h),
            "flops": 6 * m * inter * h}


def tolerance(case):
    # Weights enter the matrix cores as bf16 and most outputs are bf16, so a correct result is
    # about 1.7e-3 off in the 2-norm (three such roundings meet in the MLP's last output, 2.5e-3)
    # and its worst element about five times that.
    return {"rel": 8e-3, "max": 8e-2}


# ---- the same in 64 bits, in plain torch --------------------------------------------------------


def _untile(x, n, groups):
    """Record order [n / 128][group][128] to [n][group] (trailing axis kept)."""
    return x.view(n // 128, groups, 128, -1).transpose(1, 2).reshape(n, groups, -1)


def _q4_dense(n, k, seed, salt, tiled=True):
    codes, scales, biases = _q4(n, k, seed, salt)
    groups = k // 64
    if tiled:
        codes, scales, biases = (_untile(t, n, groups) for t in (codes, scales, biases))
    else:
        codes, scales, biases = codes.view(n, groups, 8), scales.view(n, groups, 1), biases.view(n, groups, 1)
    return codes, scales.double(), biases.double()


def _q4_rows(parts, r0, r1):
    """Rows [r0, r1) of a q4 weight in 64 bits."""
    codes, scales, biases = (t[r0:r1] for t in parts)
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((codes.unsqueeze(-1) >> shifts) & 15).reshape(codes.shape[0], codes.shape[1], 64)
    return (q.double() * scales + biases).reshape(codes.shape[0], -1)


def _product(a, rows, n, chunk=8192):
    """a @ w^T for a [m, k] in 64 bits; rows(r0, r1): rows of w in 64 bits."""
    return torch.cat([a @ rows(r, min(r + chunk, n)).t().contiguous() for r in range(0, n, chunk)], dim=1)


def _q4_product(a, n, k, seed, salt, tiled=True):
    parts = _q4_dense(n, k, seed, salt, tiled)
    return _product(a, lambda r0, r1: _q4_rows(parts, r0, r1), n)


def _half(raw, at):
    return raw[..., at:at + 2].contiguous().view(torch.float16).double()


def _gguf_rows(kind, raw):
    """Native blocks [n, blocks, bytes] as 64-bit weights [n, blocks * elements]."""
    n, nb = raw.shape[:2]
    b = raw.to(torch.int32)
    table = torch.tensor(IQ4_VALUES, dtype=torch.float64, device=raw.device)

    def signed(x):
        return torch.where(x > 127, x - 256, x).double()

    if kind == "q8_0":
        w = _half(raw, 0) * signed(b[..., 2:34])
    elif kind == "iq4_nl":
        q = b[..., 2:18]
        w = _half(raw, 0) * table[torch.cat([q & 15, q >> 4], dim=-1).long()]
    elif kind == "iq4_xs":
        high = b[..., 2] | (b[..., 3] << 8)
        groups = []
        for j in range(8):
            scale = ((b[..., 4 + j // 2] >> (4 * (j % 2))) & 15) | (((high >> (2 * j)) & 3) << 4)
            q = b[..., 8 + 16 * j:24 + 16 * j]
            groups.append((scale - 32).double().unsqueeze(-1) * table[torch.cat([q & 15, q >> 4], dim=-1).long()])
        w = _half(raw, 0) * torch.cat(groups, dim=-1)
    elif kind == "q6_k":
        groups = []
        for j in range(8):
            half, quarter = j // 4, j % 4
            low = b[..., 64 * half + 32 * (quarter % 2):64 * half + 32 * (quarter % 2) + 32] >> (4 * (quarter // 2))
            top = b[..., 128 + 32 * half:160 + 32 * half] >> (2 * quarter)
            scale = signed(b[..., 192 + 2 * j:194 + 2 * j]).repeat_interleave(16, dim=-1)
            groups.append(scale * (((low & 15) | ((top & 3) << 4)) - 32).double())
        w = _half(raw, 208) * torch.cat(groups, dim=-1)
    elif kind == "q3_k":
        groups = []
        for j in range(8):
            code = (b[..., 32 + 32 * (j // 4):64 + 32 * (j // 4)] >> (2 * (j % 4))) & 3
            code = code | (((b[..., 0:32] >> j) & 1) << 2)
            scales = []
            for i in (2 * j, 2 * j + 1):
                low = (b[..., 96 + i % 8] >> (4 * (i // 8))) & 15
                scales.append((low | (((b[..., 104 + i % 4] >> (2 * (i // 4))) & 3) << 4)) - 32)
            scale = torch.stack(scales, dim=-1).double().repeat_interleave(16, dim=-1)
            groups.append(scale * (code - 4).double())
        w = _half(raw, 108) * torch.cat(groups, dim=-1)
    else:  # q4_k, q5_k
        quants = 48 if kind == "q5_k" else 16
        d, dmin, sc = _half(raw, 0), _half(raw, 2), b[..., 4:16]
        groups = []
        for j in range(8):
            if j < 4:
                scale, least = sc[..., j] & 63, sc[..., j + 4] & 63
            else:
                scale = (sc[..., j + 4] & 15) | ((sc[..., j - 4] >> 6) << 4)
                least = (sc[..., j + 4] >> 4) | ((sc[..., j] >> 6) << 4)
            code = (b[..., quants + 32 * (j // 2):quants + 32 * (j // 2) + 32] >> (4 * (j % 2))) & 15
            if kind == "q5_k":
                code = code | (((b[..., 16:48] >> j) & 1) << 4)
            groups.append(d * scale.double().unsqueeze(-1) * code.double() - dmin * least.double().unsqueeze(-1))
        w = torch.cat(groups, dim=-1)
    return w.reshape(n, -1)


def _gguf_product(a, kind, n, k, seed, salt):
    raw = _blocks(kind, n, k, seed, salt)
    return _product(a, lambda r0, r1: _gguf_rows(kind, raw[r0:r1]), n, chunk=2048)


def _band_sums(x):
    return x.reshape(x.shape[0], -1, 64).sum(dim=-1)


def exact(case, seed):
    m, h = case["rows"], case["hidden"]
    if case["kind"] == "projection":
        return _q4_product(_act(m, h, seed, 20).double(), case["outputs"], h, seed, 1)
    if case["kind"] == "ends":
        parts = _q4_dense(case["vocab"], h, seed, 1)
        tokens = _tokens(case, seed).long()
        x = _q4_rows([t[tokens] for t in parts], 0, m)
        return {"embedded": x, "operand": x, "sums": _band_sums(x),
                "logits": _product(x, lambda r0, r1: _q4_rows(parts, r0, r1), case["vocab"])}
    if case["kind"] == "layer":
        shapes = _layer_shapes(case)
        salt = {name: i + 1 for i, name in enumerate(shapes)}
        ins = {k: v.double() for k, v in _layer_inputs(case, seed).items()}

        def proj(name, a):
            return _q4_product(a, *shapes[name], seed, salt[name])

        def residual(name, a):
            out = ins["res"] + proj(name, a)
            values = out * ins["norm"]
            return (out, values, _band_sums(values), _band_sums(out * out)) if m > 4 else (out,)

        gate = proj("wgate", ins["y"])
        act = gate * torch.sigmoid(gate) * proj("wup", ins["y"])
        a, b = (_q4_product(ins["x"], AB_ROWS, h, seed, 40 + i, tiled=False) for i in range(2))
        return {"qkv": [proj(n, ins["x"]) for n in ("wq", "wk", "wv")], "o": residual("wo", ins["attn"]),
                "z": proj("win", ins["x"]), "a": a, "b": b, "g": proj("wout", ins["gdn"]), "act": act,
                "down": residual("wdown", act)}
    inter = case["inter"]
    x, res = _act(m, h, seed, 20).double(), _residual(m, h, seed, 24).double()
    gate = _gguf_product(x, case["type"], inter, h, seed, 1)
    up = _gguf_product(x, case["type"], inter, h, seed, 2)
    act = gate * torch.sigmoid(gate) * up
    return {"gate": gate, "up": up, "act": act, "sums": _band_sums(act),
            "out": res + _gguf_product(act, case["down"], h, inter, seed, 3)}
