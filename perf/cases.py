"""Performance cases of the decoder KV-cache hot path: what a serving program has this library do.

Every case goes through the package's public entry points, on buffers laid out as such a program keeps them: KV planes,
block tables, rotary tables, weights and workspaces are made once (``prepare``), and a pass (``run``) is the call or the
calls of one step.  Kinds of work, and the ranges that ``draw`` takes its sizes from:

* ``decode``        one decode step of 1 to 18 caches of one length (a layer, or all layers of a step), 16 to 8192 rows;
* ``decode_batch``  one decode step of 2 to 256 sequences of different lengths (up to 32768 rows) in a paged pool;
* ``prefill``       rotary, range append and causal attention of a prompt of 16 to 4096 tokens;
* ``project``       the four linear projections of a decoder layer over 8 to 4096 prompt tokens;
* ``token_step``    a whole decoder token: 18 layers of GEMVs and decode attention and the LM head with its top-1,
                    replayed from a graph, 64 to 4096 rows of context;
* ``kv_move``       a prefix of 16 to 65536 rows moved into the paged cache and back;
* ``session``       the host-buffer session: begin, a few steps, finish, prefixes of 16 to 2048 rows.
"""

import math

import numpy as np
import torch

from __graft_entry__ import load_package

pvlc = load_package()

HEADS, KV, DIM, BLOCK = 16, 2, 128, 16
ROW = KV * DIM  # elements of one cache row of one plane
ROPE_BASE = 500000.0
LAYERS, HIDDEN, MLP, VOCAB = 18, 1024, 3072, 103424
# (input width, output width) of the projections of a layer: q|k|v, o, gate|up, down
PROJECTIONS = ((HIDDEN, HEADS * DIM + 2 * ROW), (HEADS * DIM, HIDDEN), (HIDDEN, 2 * MLP), (MLP, HIDDEN))


def listed():
    return [
        # the smallest call of a decode loop: one layer's attention of one sequence, on the f32 operands that its
        # projections wrote, query and key rotated in the call
        dict(name="decode_layer", kind="decode", layers=1, context=1157, io="f32", rotate_query=True),
        # the attention of a whole decode step: 18 caches of one length in one launch, fp16 operands
        dict(name="decode_step18", kind="decode", layers=18, context=2048, io="f16", rotate_query=False),
        # a small serving batch: pages in different states of recognition, ragged lengths, permuted block tables
        dict(name="decode_batch", kind="decode_batch", seqs=13, lo=90, hi=2010, io="f16"),
        # the largest batch: 256 sequences, log-uniform lengths up to 32768 rows
        dict(name="decode_long", kind="decode_batch", seqs=256, lo=1024, hi=32768, io="f16"),
        # a short prompt: a cropped line or table cell and its instruction
        dict(name="prefill_short", kind="prefill", tokens=211, io="f16", paged=False, positions=False),
        # an ordinary page: image tokens and the instruction, positions given, f32 operands of the projections, paged
        dict(name="prefill_page", kind="prefill", tokens=1157, io="f32", paged=True, positions=True),
        # the longest prompt: a dense page at full resolution
        dict(name="prefill_long", kind="prefill", tokens=4096, io="f16", paged=True, positions=False),
        # the projections of one layer over the ordinary page, and over the longest prompt
        dict(name="project_page", kind="project", rows=1157),
        dict(name="project_long", kind="project", rows=4096),
        # a whole decoder token from its graph
        dict(name="token_step", kind="token_step", context=2048),
        # a stored prefix taken into the paged cache and read back out of it
        dict(name="kv_move", kind="kv_move", tokens=5003),
        # the host-buffer session of the reference surface
        dict(name="session", kind="session", prefix=777, steps=4),
    ]


def _log(rng, lo, hi):
    """A whole number of lo..hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode_batch", "prefill", "prefill", "project", "project", "token_step", "kv_move", "session"])
    io = rng.choice(["f16", "f32"])
    if kind == "decode":
        return dict(kind=kind, layers=rng.choice([1, 1, 18, _log(rng, 2, 17)]), context=_log(rng, 16, 8192), io=io,
                    rotate_query=rng.random() < 0.5)
    if kind == "decode_batch":
        seqs = _log(rng, 2, 256)
        hi = min(_log(rng, 128, 32768), (1 << 21) // seqs)
        return dict(kind=kind, seqs=seqs, lo=_log(rng, max(16, hi // 32), hi), hi=hi, io=io)
    if kind == "prefill":
        return dict(kind=kind, tokens=_log(rng, 16, 4096), io=io, paged=rng.random() < 0.5, positions=rng.random() < 0.5)
    if kind == "project":
        return dict(kind=kind, rows=_log(rng, 8, 4096))
    if kind == "token_step":
        return dict(kind=kind, context=_log(rng, 64, 4096))
    if kind == "kv_move":
        return dict(kind=kind, tokens=_log(rng, 16, 65536))
    return dict(kind=kind, prefix=_log(rng, 16, 2048), steps=rng.randint(1, 8))


def _lengths(case):
    """Rows attended (after the append) by each sequence of a batch: evenly spread over the logarithm of lo..hi."""
    n, lo, hi = case["seqs"], case["lo"], case["hi"]
    return [min(hi, max(lo, int(round(lo * (hi / lo) ** ((i + 0.5) / n))))) for i in range(n)]


# ---------------------------------------------------------------------------
# Inputs, made from the seed alone (no library code), on the GPU
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, dtype=torch.float32, scale=1.0):
    x = torch.randn(*shape, generator=g, device="cuda", dtype=dtype)
    return x if scale == 1.0 else x.mul_(scale)


def _rope(rows):
    """cos and sin tables [rows][64] f32."""
    inv = ROPE_BASE ** (-torch.arange(0, DIM, 2, device="cuda", dtype=torch.float64) / DIM)
    angle = torch.arange(rows, device="cuda", dtype=torch.float64)[:, None] * inv[None, :]
    return angle.cos().float(), angle.sin().float()


def _blocks(tokens):
    return -(-tokens // BLOCK)


def _inputs(case, seed):
    g, kind, s = _gen(seed), case["kind"], {}
    operand = torch.float32 if case.get("io") == "f32" else torch.float16
    if kind in ("decode", "decode_batch"):
        if kind == "decode":
            n, cap = case["layers"], _blocks(case["context"] + 64)
            s["lens"] = [case["context"]] * n
            s["blocks"], s["row_blocks"], s["table"] = n * cap, cap, None
            rows = cap * BLOCK
        else:
            n, lens = case["seqs"], _lengths(case)
            order = torch.randperm(n, generator=g, device="cuda").tolist()
            s["lens"] = lens = [lens[i] for i in order]
            used = sum(_blocks(t) for t in lens)
            s["blocks"], s["row_blocks"] = used + 7, _blocks(case["hi"])
            ids = torch.randperm(s["blocks"], generator=g, device="cuda", dtype=torch.int32)
            s["table"] = torch.zeros(n, s["row_blocks"], dtype=torch.int32, device="cuda")
            at = 0
            for i, t in enumerate(lens):
                s["table"][i, :_blocks(t)] = ids[at:at + _blocks(t)]
                at += _blocks(t)
            rows = case["hi"]
        s["cos"], s["sin"] = _rope(rows)
        s["k"] = _normal(g, s["blocks"] * BLOCK * ROW, dtype=torch.float16)
        s["v"] = _normal(g, s["blocks"] * BLOCK * ROW, dtype=torch.float16)
        s["q"], s["nk"], s["nv"] = (_normal(g, n, h, DIM, dtype=operand) for h in (HEADS, KV, KV))
    elif kind == "prefill":
        n = case["tokens"]
        s["blocks"] = _blocks(n) + (5 if case["paged"] else 0)
        s["table"] = torch.randperm(s["blocks"], generator=g, device="cuda", dtype=torch.int32)[:_blocks(n)].contiguous() if case["paged"] else None
        s["rope_rows"] = n + 32
        s["positions"] = torch.arange(n, device="cuda", dtype=torch.int32) + 3 if case["positions"] else None
        s["cos"], s["sin"] = _rope(s["rope_rows"])
        s["k"] = _normal(g, s["blocks"] * BLOCK * ROW, dtype=torch.float16)
        s["v"] = _normal(g, s["blocks"] * BLOCK * ROW, dtype=torch.float16)
        s["q"], s["nk"], s["nv"] = (_normal(g, n, h, DIM, dtype=operand) for h in (HEADS, KV, KV))
    elif kind == "project":
        # activations: every row at its own scale, as after a layer's norms and gates
        s["x"] = [_normal(g, case["rows"], k) * torch.exp(_normal(g, case["rows"], 1)) for k, _ in PROJECTIONS]
        s["w"] = [_normal(g, n, k, dtype=torch.float16, scale=0.02) for k, n in PROJECTIONS]
        s["b"] = [_normal(g, n, scale=0.1) for _, n in PROJECTIONS]
    elif kind == "token_step":
        s["blocks"] = _blocks(case["context"] + 64)
        s["k"] = _normal(g, LAYERS, s["blocks"] * BLOCK * ROW, dtype=torch.float16)
        s["v"] = _normal(g, LAYERS, s["blocks"] * BLOCK * ROW, dtype=torch.float16)
        s["w"] = {name: _normal(g, LAYERS, rows, cols, dtype=torch.float16, scale=0.02) for name, rows, cols in (
            ("q", HEADS * DIM, HIDDEN), ("k", ROW, HIDDEN), ("v", ROW, HIDDEN), ("o", HIDDEN, HEADS * DIM),
            ("gate", MLP, HIDDEN), ("up", MLP, HIDDEN), ("down", HIDDEN, MLP))}
        s["head"] = _normal(g, VOCAB, HIDDEN, dtype=torch.float16, scale=0.02)
        s["x"] = _normal(g, HIDDEN)
        s["cos"], s["sin"] = _rope(case["context"] + 64)
    elif kind == "kv_move":
        n = case["tokens"]
        s["blocks"] = _blocks(n) + 9
        s["table"] = torch.randperm(s["blocks"], generator=g, device="cuda", dtype=torch.int32)[:_blocks(n)].contiguous()
        s["rows_k"], s["rows_v"] = (_normal(g, n, KV, DIM, dtype=torch.float16) for _ in range(2))
    else:  # session: host arrays
        r = np.random.default_rng(seed)
        s["capacity"] = case["prefix"] + case["steps"] + 11
        s["k"], s["v"] = (r.standard_normal((s["capacity"], KV, DIM), dtype=np.float32) for _ in range(2))
        s["steps"] = [tuple(r.standard_normal((h, DIM), dtype=np.float32) for h in (HEADS, KV, KV)) for _ in range(case["steps"])]
    return s


# ---------------------------------------------------------------------------
# What the program keeps, and one pass
# ---------------------------------------------------------------------------

def _workspace(nbytes):
    if not nbytes:
        return None
    w = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    pvlc.workspace_init(w, nbytes)
    return w


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = s["kind"] = case["kind"]
    f32 = s["f32"] = case.get("io") == "f32"
    if kind in ("decode", "decode_batch"):
        n = len(s["lens"])
        s["out"] = torch.empty(n, HEADS, DIM, device="cuda", dtype=s["q"].dtype)
        context = s["row_blocks"] * BLOCK if kind == "decode" else case["hi"]
        ragged = dict(block_tables=s["table"], cache_lens=torch.tensor([t - 1 for t in s["lens"]], dtype=torch.int32, device="cuda")) if kind == "decode_batch" else dict(uniform_cache_len=case["context"] - 1)
        nbytes = pvlc.decode_workspace_bytes(n, context)
        s["keep"] = ragged, _workspace(nbytes)
        operands = {} if f32 else dict(query=s["q"], new_key=s["nk"], new_value=s["nv"], out=s["out"])
        s["args"] = pvlc.paged_decode_args(
            num_seqs=n, num_blocks=s["blocks"], max_blocks_per_seq=s["row_blocks"], key_cache=s["k"], value_cache=s["v"],
            workspace=s["keep"][1], workspace_bytes=nbytes, max_context=context, rope_cos=s["cos"], rope_sin=s["sin"],
            rope_rows=s["cos"].shape[0], rotate_query=case.get("rotate_query", True),
            **{**dict(query=None, new_key=None, new_value=None, out=None), **operands}, **ragged)
    elif kind == "prefill":
        n = case["tokens"]
        s["out"] = torch.empty(n, HEADS, DIM, device="cuda", dtype=s["q"].dtype)
        s["error"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["ws_bytes"] = pvlc.prefill_workspace_bytes(n)
        s["ws"] = _workspace(s["ws_bytes"])
        s["tokens"] = n
    elif kind == "project":
        rows = s["rows"] = case["rows"]
        s["out"] = [torch.empty(rows, n, device="cuda") for _, n in PROJECTIONS]
        s["ws_bytes"] = max(pvlc.linear_projection_workspace_bytes(rows, k) for k, _ in PROJECTIONS)
        s["ws"] = torch.empty(s["ws_bytes"], dtype=torch.uint8, device="cuda")
    elif kind == "token_step":
        _prepare_token(case, s)
    elif kind == "kv_move":
        s["tokens"] = case["tokens"]
        s["k"], s["v"] = (torch.zeros(s["blocks"] * BLOCK * ROW, dtype=torch.float16, device="cuda") for _ in range(2))
        s["back_k"], s["back_v"] = torch.empty_like(s["rows_k"]), torch.empty_like(s["rows_v"])
    else:
        s["runtime"] = pvlc.NativeRuntime(0)
        s["descriptor"] = pvlc.DecoderKvSessionDescriptor(case["prefix"], s["capacity"], s["k"].ravel(), s["v"].ravel())
        s["step"] = [pvlc.DecoderKvSessionStep(*(x.ravel() for x in step)) for step in s["steps"]]
    return s


def _prepare_token(case, s):
    """The buffers of a decoder token and the graph that its loop replays."""
    cap = s["blocks"] * BLOCK
    s["qkv"] = torch.empty(LAYERS, HEADS * DIM + 2 * ROW, device="cuda")
    s["attn"] = torch.empty(LAYERS, HEADS * DIM, device="cuda")
    s["o"], s["gu"] = torch.empty(LAYERS, HIDDEN, device="cuda"), torch.empty(LAYERS, 2 * MLP, device="cuda")
    s["hidden"] = torch.empty(LAYERS, HIDDEN, device="cuda")
    s["logits"] = torch.empty(VOCAB, device="cuda")
    s["top"] = torch.zeros(2, dtype=torch.int32, device="cuda")
    top_bytes = pvlc.top1_workspace_bytes()
    top_ws = _workspace(top_bytes)
    nbytes = pvlc.decode_workspace_bytes(1, cap)
    ws = _workspace(nbytes)
    w, calls = s["w"], []
    for l in range(LAYERS):
        q, k, v = s["qkv"][l, :HEADS * DIM], s["qkv"][l, HEADS * DIM:HEADS * DIM + ROW], s["qkv"][l, HEADS * DIM + ROW:]
        members = pvlc.GemvMembers([(w["q"][l], q, HEADS * DIM), (w["k"][l], k, ROW), (w["v"][l], v, ROW)])
        mlp = pvlc.GemvMembers([(w["gate"][l], s["gu"][l, :MLP], MLP), (w["up"][l], s["gu"][l, MLP:], MLP)])
        args = pvlc.paged_decode_args(
            num_seqs=1, num_blocks=s["blocks"], max_blocks_per_seq=s["blocks"], key_cache=s["k"][l], value_cache=s["v"][l],
            query=None, new_key=None, new_value=None, out=None, workspace=ws, workspace_bytes=nbytes, max_context=cap,
            uniform_cache_len=case["context"] - 1, rope_cos=s["cos"], rope_sin=s["sin"], rope_rows=s["cos"].shape[0],
            rotate_query=True)
        calls.append((members, mlp, args, q, k, v))

    def token(stream):
        x = s["x"]
        for l, (members, mlp, args, q, k, v) in enumerate(calls):
            pvlc.gemv_group_f16(members, x, HIDDEN, stream)
            pvlc.paged_decode_f32io(args, q, k, v, s["attn"][l], stream)
            pvlc.gemv_f16(w["o"][l], s["attn"][l], s["o"][l], HIDDEN, HEADS * DIM, stream)
            pvlc.gemv_group_f16(mlp, s["o"][l], HIDDEN, stream)
            pvlc.gemv_f16(w["down"][l], s["gu"][l, :MLP], s["hidden"][l], HIDDEN, MLP, stream)
            x = s["hidden"][l]
        pvlc.lm_head_top1_f16(s["head"], x, s["logits"], VOCAB, HIDDEN, s["top"], top_ws, top_bytes, stream)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        token(side)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        token(torch.cuda.current_stream())
    s["keep"] = calls, ws, top_ws


def run(s):
    kind = s["kind"]
    if kind in ("decode", "decode_batch"):
        if s["f32"]:
            pvlc.paged_decode_f32io(s["args"], s["q"], s["nk"], s["nv"], s["out"])
        else:
            pvlc.paged_decode_f16(s["args"])
        return dict(out=s["out"], key_cache=s["k"], value_cache=s["v"])
    if kind == "prefill":
        call = pvlc.paged_prefill_f32io if s["f32"] else pvlc.paged_prefill_f16
        call(tokens=s["tokens"], num_blocks=s["blocks"], key_cache=s["k"], value_cache=s["v"], query=s["q"], key=s["nk"],
             value=s["nv"], out=s["out"], block_table=s["table"], rope_cos=s["cos"], rope_sin=s["sin"],
             rope_rows=s["rope_rows"], positions=s["positions"], error_word=s["error"], workspace=s["ws"],
             workspace_bytes=s["ws_bytes"])
        return dict(out=s["out"], key_cache=s["k"], value_cache=s["v"])
    if kind == "project":
        for x, w, b, out, (k, n) in zip(s["x"], s["w"], s["b"], s["out"], PROJECTIONS):
            pvlc.linear_projection_f16(x, w, b, out, s["rows"], k, n, s["ws"], s["ws_bytes"])
        return list(s["out"])
    if kind == "token_step":
        s["graph"].replay()
        return dict(hidden=s["hidden"], attention=s["attn"], logits=s["logits"], top=s["top"][:1],
                    top_logit=s["top"][1:].view(torch.float32), key_cache=s["k"], value_cache=s["v"])
    if kind == "kv_move":
        pvlc.kv_pack_f16(s["rows_k"], s["rows_v"], s["tokens"], s["k"], s["v"], s["blocks"], s["table"])
        pvlc.kv_unpack_f16(s["k"], s["v"], s["tokens"], s["back_k"], s["back_v"], s["blocks"], s["table"])
        return dict(key_cache=s["k"], value_cache=s["v"], keys=s["back_k"], values=s["back_v"])
    session = s["runtime"].begin_decoder_kv_session(s["descriptor"])
    out = [session.step(x).attention for x in s["step"]]
    snapshot = session.finish()
    return dict(attention=out, key_cache=snapshot.key_cache, value_cache=snapshot.value_cache)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what it gives
# ---------------------------------------------------------------------------

def _decode_bytes(t, f32):
    # keys and values once, the query and the new row in, the appended row and the output out
    return 1024 * (t - 1) + (2 * HEADS * DIM + 2 * ROW) * (4 if f32 else 2) + 1024


def work(case):
    kind, f32 = case["kind"], case.get("io") == "f32"
    if kind == "decode":
        return dict(bytes=case["layers"] * _decode_bytes(case["context"], f32), flops=8192 * case["layers"] * case["context"])
    if kind == "decode_batch":
        return dict(bytes=sum(_decode_bytes(t, f32) for t in _lengths(case)), flops=8192 * sum(_lengths(case)))
    if kind == "prefill":
        n = case["tokens"]
        return dict(bytes=n * ((2 * HEADS * DIM + 2 * ROW) * (4 if f32 else 2) + 1024), flops=8192 * n * (n + 1) // 2)
    if kind == "project":
        r = case["rows"]
        return dict(bytes=sum(4 * r * (k + n) + 2 * k * n + 4 * n for k, n in PROJECTIONS), flops=sum(2 * r * k * n for k, n in PROJECTIONS))
    if kind == "token_step":
        weights = LAYERS * sum(k * n for k, n in PROJECTIONS) + VOCAB * HIDDEN
        return dict(bytes=2 * weights + 4 * VOCAB + LAYERS * _decode_bytes(case["context"], True),
                    flops=2 * weights + 8192 * LAYERS * case["context"])
    if kind == "kv_move":
        return dict(bytes=4096 * case["tokens"], flops=0)
    t = case["prefix"] + case["steps"]
    return dict(bytes=4096 * t + sum(_decode_bytes(case["prefix"] + i + 1, True) for i in range(case["steps"])),
                flops=8192 * case["steps"] * t)


def tolerance(case):
    kind = case["kind"]
    if kind == "kv_move":
        return "exact"
    if kind in ("decode", "decode_batch", "prefill"):
        # against 64 bits, fp16 outputs show 2.5e-4 (their own rounding and that of the fp16 weights), f32 outputs 3e-7
        # to 6e-6 (a rotated key or query element that falls on the other side of its fp16 rounding)
        return dict(rel=2e-5, max=2e-3) if case["io"] == "f32" else dict(rel=1e-3, max=1e-2)
    if kind == "project":  # 3e-7 to 5e-7 against 64 bits
        return dict(rel=2e-6, max=1e-4)
    return dict(rel=2e-5, max=2e-3)


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _rotate(x, cos, sin):
    """Rotate-half of [..., heads, 128] at the rows' cos/sin [..., 64], in 64 bits."""
    x, cos, sin = x.double(), cos.double().unsqueeze(-2), sin.double().unsqueeze(-2)
    lo, hi = x[..., :64], x[..., 64:]
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)


def _stored(x):
    """What the fp16 cache (or an fp16 operand) holds of x, in 64 bits."""
    return x.half().double()


_SLOT = [(t & 3) | ((t & 4) << 1) | ((t & 8) >> 1) for t in range(BLOCK)]  # key slot of token t in a block


def _rows(k, v, ids):
    """Rows [blocks * 16][2][128] of the blocks `ids` of flat planes, in 64 bits."""
    kb = k.view(-1, KV, DIM // 8, BLOCK, 8)[ids][:, :, :, _SLOT]  # [block][head][chunk][token][8]
    vb = v.view(-1, KV, DIM, BLOCK)[ids]
    return (kb.permute(0, 3, 1, 2, 4).reshape(-1, KV, DIM).double(), vb.permute(0, 3, 1, 2).reshape(-1, KV, DIM).double())


def _put(k, v, ids, at, rows_k, rows_v):
    """Writes rows [n][2][128] at tokens `at` of the sequence whose blocks are `ids`."""
    b, t = ids[torch.div(at, BLOCK, rounding_mode="floor")].long(), at % BLOCK
    slot = torch.tensor(_SLOT, device=at.device)[t]
    k.view(-1, KV, DIM // 8, BLOCK, 8)[b, :, :, slot] = rows_k.to(k.dtype).view(-1, KV, DIM // 8, 8)
    v.view(-1, KV, DIM, BLOCK)[b, :, :, t] = rows_v.to(v.dtype)


def _attend(q, k, v):
    """[16][128] over rows [t][2][128]."""
    out = torch.empty_like(q)
    for g in range(KV):
        h = slice(g * HEADS // KV, (g + 1) * HEADS // KV)
        p = torch.softmax(q[h] @ k[:, g].t() / math.sqrt(DIM), -1)
        out[h] = p @ v[:, g].contiguous()
    return out


def _exact_decode(case, s):
    outs = []
    for i, t in enumerate(s["lens"]):
        ids = s["table"][i, :_blocks(t)].long() if s["table"] is not None else torch.arange(i * s["row_blocks"], i * s["row_blocks"] + _blocks(t), device="cuda")
        cos, sin = s["cos"][t - 1], s["sin"][t - 1]
        nk, nv = _stored(_rotate(s["nk"][i], cos, sin)), _stored(s["nv"][i])
        q = _stored(_rotate(s["q"][i], cos, sin)) if case.get("rotate_query", True) else _stored(s["q"][i])
        _put(s["k"], s["v"], ids, torch.tensor([t - 1], device="cuda"), nk[None], nv[None])
        k, v = _rows(s["k"], s["v"], ids)
        outs.append(_attend(q, k[:t], v[:t]))
    big = s["k"].numel() > 1 << 27  # (the planes of the largest batches are compared between runs only)
    return dict(out=torch.stack(outs), key_cache=None if big else s["k"], value_cache=None if big else s["v"])


def _exact_prefill(case, s):
    n = case["tokens"]
    pos = s["positions"].long() if s["positions"] is not None else torch.arange(n, device="cuda")
    cos, sin = s["cos"][pos], s["sin"][pos]
    q, k, v = _stored(_rotate(s["q"], cos, sin)), _stored(_rotate(s["nk"], cos, sin)), _stored(s["nv"])
    ids = s["table"].long() if s["table"] is not None else torch.arange(_blocks(n), device="cuda")
    _put(s["k"], s["v"], ids, torch.arange(n, device="cuda"), k, v)
    out = torch.empty_like(q)
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for h in range(HEADS):
        g = h * KV // HEADS
        scores = q[:, h] @ k[:, g].t() / math.sqrt(DIM)
        out[:, h] = torch.softmax(scores.masked_fill_(mask, -math.inf), -1) @ v[:, g].contiguous()
    return dict(out=out, key_cache=s["k"], value_cache=s["v"])


def _exact_token(case, s):
    t, x, w = case["context"], s["x"].double(), s["w"]
    ids, at = torch.arange(_blocks(t), device="cuda"), torch.tensor([t - 1], device="cuda")
    cos, sin = s["cos"][t - 1], s["sin"][t - 1]
    hidden, attention = [], []
    for l in range(LAYERS):
        q, k, v = (w[name][l].double() @ x for name in "qkv")
        q, nk = _stored(_rotate(q.view(HEADS, DIM), cos, sin)), _stored(_rotate(k.view(KV, DIM), cos, sin))
        _put(s["k"][l], s["v"][l], ids, at, nk[None], _stored(v.view(1, KV, DIM)))
        keys, values = _rows(s["k"][l], s["v"][l], ids)
        attention.append(_attend(q, keys[:t], values[:t]).view(-1))
        o = w["o"][l].double() @ attention[-1]
        x = w["down"][l].double() @ (w["gate"][l].double() @ o)
        hidden.append(x)
    logits = s["head"].double() @ x
    return dict(hidden=torch.stack(hidden), attention=torch.stack(attention), logits=logits, top=None,
                top_logit=logits.max().view(1), key_cache=s["k"], value_cache=s["v"])


def _exact_session(case, s):
    k, v = (torch.from_numpy(x.copy()) for x in (s["k"], s["v"]))
    outs, t = [], case["prefix"]
    for q, nk, nv in s["steps"]:
        k[t], v[t] = torch.from_numpy(nk), torch.from_numpy(nv)
        t += 1
        outs.append(_attend(_stored(torch.from_numpy(q)), _stored(k[:t]), _stored(v[:t])).view(-1))
    return dict(attention=outs, key_cache=k.double().view(-1), value_cache=v.double().view(-1))


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind in ("decode", "decode_batch"):
        return _exact_decode(case, s)
    if kind == "prefill":
        return _exact_prefill(case, s)
    if kind == "project":
        return [x.double() @ w.double().t() + b.double() for x, w, b in zip(s["x"], s["w"], s["b"])]
    if kind == "token_step":
        return _exact_token(case, s)
    if kind == "session":
        return _exact_session(case, s)
    return None  # kv_move: whole values
