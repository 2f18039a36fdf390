"""The calls that programs built on this framework make, at the sizes they make them: what a change of a kernel or
of the host path is timed on and compared over.

decide answers questions about a prompt: a constant prefix of 107 tokens is kept as a snapshot, a request of 276
(card), 603 (ticket) or 2,307 tokens (long document) runs behind it, a follow-up about a known state runs a few
dozen tokens, and each answer is read off the logits of a few candidate tokens at one row. The cases are the blocks
of that forward, each called through the kernel wrappers as a program that strings its own layers calls them, and
one whole request:

* ``mlp``: x = embed(ids); h = norm(x); x += SwiGLU(h·w_guᵀ)·w_downᵀ. with ``of`` the rows are gathered from a longer
  x of that many, as the pruned last layer does;
* ``gdn``: a Gated-DeltaNet decoder layer from the embedding on (in-projection, conv, recurrence from a carried
  state, gated norm, out-projection, MLP), returning x and the new recurrent and conv states;
* ``attn``: a gated attention decoder layer likewise, its rows at positions pos0.. behind cached keys, returning x
  and the caches;
* ``head``: gather of the answer rows, final norm and candidate logits;
* ``request``: host ids in, host logits out, through ``Model.logits`` on the snapshot route.

Each state has its own weights (three layers of 225 MB do not fit the 256 MB cache, so weights come from HBM as in
a forward through many layers).
"""

from __future__ import annotations

import math

import numpy as np
import torch

from decide_amd import hip
from decide_amd.forward import Model, ModelConfig
from decide_amd.kernels import Epilogue, Kernels

D, F = 2560, 9216  # hidden width, MLP width
VOCAB = 151936
LIN_N, LIN_Z, LIN_B, LIN_A = 12352, 8192, 12288, 12320  # w_in rows of a Gated-DeltaNet layer: qkv | z | b | a
ATT_N, ATT_GATE, ATT_K, ATT_V = 10240, 4096, 8192, 9216  # w_in rows of an attention layer: q | gate | k | v
NK, NV, DK = 16, 32, 128  # key heads, value heads, their width
NQ, NKV, HD, ROT = 16, 4, 256, 32  # query heads, key/value heads, their width, rotated pairs
CONV = 8192
PREFIX = 107  # tokens of decide's constant prompt prefix
EPS = 1e-6
CHUNK_MIN_T = 320  # rows from which a program calls conv and the chunked recurrence as one call
MAX_ROWS = 2307

REQ_LAYERS, REQ_VOCAB, REQ_CAND = 32, 248320, 62  # decide's own model and the most candidates it takes
REQ_COUNTS = (2, 8, 3, 62, 5, 20)  # candidates of a request's six answers


def listed():
    return [
        # the last layer's MLP over the 3 answer rows of a request: weight streaming and launches
        {"name": "mlp_answers", "kind": "mlp", "rows": 3, "of": 603},
        # the rows of a card request behind the snapshot (276 - 107)
        {"name": "mlp_card", "kind": "mlp", "rows": 169, "of": 0},
        # a whole ticket prompt: the shape of the benchmark's MLP block
        {"name": "mlp_ticket", "kind": "mlp", "rows": 603, "of": 0},
        # a long document's prompt in one chunk
        {"name": "mlp_long", "kind": "mlp", "rows": 2307, "of": 0},
        # a follow-up question about a cached state: a few dozen rows, token-by-token recurrence
        {"name": "gdn_followup", "kind": "gdn", "rows": 41},
        # a card request's rows: still the token-by-token recurrence
        {"name": "gdn_card", "kind": "gdn", "rows": 169},
        # a ticket and a long document: the chunked recurrence
        {"name": "gdn_ticket", "kind": "gdn", "rows": 603},
        {"name": "gdn_long", "kind": "gdn", "rows": 2307},
        # a ticket's rows behind the prefix's keys, and a long document's whole causal square
        {"name": "attn_ticket", "kind": "attn", "rows": 496, "pos0": 107},
        {"name": "attn_long", "kind": "attn", "rows": 2307, "pos0": 0},
        # as many answers with as many candidates as decide takes in one request
        {"name": "head_full", "kind": "head", "rows": 16, "cand": 62},
        # a whole card request through decide's 32 layers on the snapshot route, host to host
        {"name": "request_card", "kind": "request", "tokens": 276},
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "gdn", "gdn", "gdn", "attn", "attn", "head", "request"])
    if kind == "mlp":
        rows = _log_uniform(rng, 1, MAX_ROWS)
        return {"kind": kind, "rows": rows, "of": rng.randint(170, MAX_ROWS) if rows <= 16 else 0}
    if kind == "gdn":
        return {"kind": kind, "rows": _log_uniform(rng, 8, MAX_ROWS)}
    if kind == "attn":
        rows = _log_uniform(rng, 8, MAX_ROWS)
        room = MAX_ROWS - rows
        return {"kind": kind, "rows": rows, "pos0": rng.choice([0, min(PREFIX, room), rng.randint(0, room)])}
    if kind == "head":
        return {"kind": kind, "rows": rng.randint(1, 16), "cand": rng.randint(2, 62)}
    return {"kind": kind, "tokens": rng.randint(PREFIX + 16, 276)}


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, dtype=torch.float32, mean=0.0, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype).mul_(std).add_(mean)


def _ids(g, n, vocab=VOCAB):
    return torch.randint(0, vocab, (n,), generator=g, device="cuda", dtype=torch.int32)


def _mlp_weights(g):
    return {
        "post_norm": _normal(g, (D,), std=0.02),
        "w_gu": _normal(g, (2 * F, D), torch.float16, std=0.02),
        "w_down": _normal(g, (D, F), torch.float16, std=0.02),
    }


def _inputs(case, seed):
    """The tensors a program holds before the call, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "request":
        return _request_inputs(case, seed)
    rows = case["rows"]
    if kind == "head":
        return {
            "x": _normal(g, (603, D)),  # the residual rows after the last layer
            "table": _normal(g, (REQ_VOCAB, D), torch.bfloat16, std=0.02),
            "final_norm": _normal(g, (D,), std=0.02),
            "rowmap": torch.randperm(603, generator=g, device="cuda")[:rows].to(torch.int32),
            "cand": _ids(g, rows * case["cand"], REQ_VOCAB),
            "ncand": torch.full((rows,), case["cand"], device="cuda", dtype=torch.int32),
        }
    i = {"table": _normal(g, (VOCAB, D), torch.bfloat16, std=0.02), "ids": _ids(g, rows)}
    if kind == "mlp":
        i.update(_mlp_weights(g))
        if case["of"]:
            i["x_all"] = _normal(g, (case["of"], D))
            i["rowmap"] = torch.randperm(case["of"], generator=g, device="cuda")[:rows].to(torch.int32)
        return i
    i["in_norm"] = _normal(g, (D,), std=0.02)
    if kind == "gdn":
        i.update(
            w_in=_normal(g, (LIN_N, D), torch.float16, std=0.02),
            conv_w=_normal(g, (CONV, 4), std=0.3),
            a_log=_normal(g, (NV,), mean=0.5, std=0.5),
            dt_bias=_normal(g, (NV,), std=0.5),
            gnorm=_normal(g, (DK,), mean=1.0, std=0.02),
            conv_in=_normal(g, (3, CONV)),
            state_in=_normal(g, (NV, DK, DK), std=0.05),
        )
    else:
        i.update(
            w_in=_normal(g, (ATT_N, D), torch.float16, std=0.02),
            q_norm=_normal(g, (HD,), std=0.02),
            k_norm=_normal(g, (HD,), std=0.02),
            kc=_normal(g, (case["pos0"] + rows, NKV, HD), torch.float16),  # rows before pos0 are cached keys
            vc=_normal(g, (case["pos0"] + rows, NKV, HD), torch.float16),
            inv_freq=_inv_freq(),
            qpos=torch.arange(case["pos0"], case["pos0"] + rows, device="cuda", dtype=torch.int32),
        )
    i["w_out"] = _normal(g, (D, 4096), torch.float16, std=0.02)
    i.update(_mlp_weights(g))
    return i


def _inv_freq():
    return torch.tensor([1.0 / 1e7 ** (2 * i / 64.0) for i in range(ROT)], device="cuda", dtype=torch.float32)


def _request_inputs(case, seed):
    r = np.random.RandomState(int(seed) % (1 << 32))
    t = case["tokens"]
    rows = sorted(int(v) for v in r.choice(np.arange(PREFIX, t - 1), len(REQ_COUNTS) - 1, replace=False)) + [t - 1]
    return {
        "ids": [int(v) for v in r.randint(0, REQ_VOCAB, t)],
        "answers": [(row, [int(v) for v in r.randint(0, REQ_VOCAB, n)])
                    for row, n in zip(rows, REQ_COUNTS)],
    }


def _request_weights(seed):
    """(name, values) of every tensor of the request's model, in decide-weights-v1 names."""
    g = _gen(seed)
    yield "embed", _normal(g, (REQ_VOCAB, D), torch.bfloat16, std=0.02)
    yield "final_norm", _normal(g, (D,), std=0.02)
    for layer in range(REQ_LAYERS):
        attn = (layer + 1) % 4 == 0
        w = {"in_norm": _normal(g, (D,), std=0.02),
             "w_in": _normal(g, (ATT_N if attn else LIN_N, D), torch.float16, std=0.02),
             "w_out": _normal(g, (D, 4096), torch.float16, std=0.02)}
        if attn:
            w.update(q_norm=_normal(g, (HD,), std=0.02), k_norm=_normal(g, (HD,), std=0.02))
        else:
            w.update(conv_w=_normal(g, (CONV, 4), std=0.3), a_log=_normal(g, (NV,), mean=0.5, std=0.5),
                     dt_bias=_normal(g, (NV,), std=0.5), gnorm=_normal(g, (DK,), mean=1.0, std=0.02))
        w.update(_mlp_weights(g))
        for name, v in w.items():
            yield f"L{layer}.{name}", v


def prepare(case, seed):
    i = _inputs(case, seed)
    k = Kernels()
    s = {"case": case, "k": k, "stream": int(torch.cuda.current_stream().cuda_stream), "i": i}
    if case["kind"] == "request":
        model = Model(k.ctx, ModelConfig(REQ_LAYERS, REQ_VOCAB, 603, 16, REQ_CAND))
        for name, v in _request_weights(seed):
            ptr, n, _ = model.tensor(name)
            torch.cuda.current_stream().synchronize()
            hip.check(hip.rt().hipMemcpy(ptr, v.data_ptr(), v.numel() * v.element_size(), hip.D2D), name)
        k.gemm.warm_up(s["stream"], max_m=603)
        model.build_snapshot(s["stream"], i["ids"][:PREFIX])
        s["model"] = model
        return s
    rows = case["rows"]
    k.gemm.warm_up(s["stream"], max_m=max(rows, case.get("pos0", 0) + rows))

    def empty(*shape, dtype=torch.float32):
        return torch.empty(shape, device="cuda", dtype=dtype)

    b = s["b"] = {}
    if case["kind"] == "head":
        b.update(xs=empty(rows, D), logits=empty(rows, case["cand"]))
        return s
    b.update(x=empty(rows, D), h=empty(rows, D, dtype=torch.float16), mlp=empty(rows, F, dtype=torch.float16),
             iota=torch.arange(rows, device="cuda", dtype=torch.int32))
    if case["kind"] == "gdn":
        b.update(p=empty(rows, LIN_N), q=empty(rows, NK, DK), kk=empty(rows, NK, DK), v=empty(rows, NV, DK),
                 o=empty(rows, NV, DK), g=empty(rows, 4096, dtype=torch.float16), conv_out=empty(3, CONV),
                 state_out=empty(NV, DK, DK))
    if case["kind"] == "attn":
        b.update(p=empty(rows, ATT_N), qo=empty(rows, 4096, dtype=torch.float16),
                 g=empty(rows, 4096, dtype=torch.float16))
    return s


# ---- one pass ---------------------------------------------------------------------------------------------------
def _run_mlp(s, rows):
    """x += SwiGLU(h·w_guᵀ)·w_downᵀ for h = norm(x)."""
    k, st, i, b = s["k"], s["stream"], s["i"], s["b"]
    k.gemm.gemm(st, (b["h"], 0), (i["w_gu"], 0), (b["mlp"], 0), rows, 2 * F, D, D, D, F, Epilogue.SwigluF16)
    k.gemm.gemm(st, (b["mlp"], 0), (i["w_down"], 0), (b["x"], 0), rows, D, F, F, F, D, Epilogue.AddF32)


def _run_block(s):
    k, st, i, b, case = s["k"], s["stream"], s["i"], s["b"], s["case"]
    rows, kind = case["rows"], case["kind"]
    if case.get("of"):
        k.head.gather_rows_f32(st, (i["x_all"], 0), (i["rowmap"], 0), (b["x"], 0), rows, D)
    else:
        k.embed.embed(st, (i["ids"], 0), (i["table"], 0), (b["x"], 0), rows, D)
    first = i["post_norm"] if kind == "mlp" else i["in_norm"]
    k.norm.rmsnorm(st, (b["x"], 0), (first, 0), (b["h"], 0), (b["iota"], 0), rows, D, D, D, True, EPS)
    if kind == "mlp":
        _run_mlp(s, rows)
        return b["x"]
    n = LIN_N if kind == "gdn" else ATT_N
    k.gemm.gemm(st, (b["h"], 0), (i["w_in"], 0), (b["p"], 0), rows, n, D, D, D, n, Epilogue.StoreF32)
    if kind == "gdn":
        p, gates = (b["p"], 0), ((b["p"], 4 * LIN_A), (b["p"], 4 * LIN_B), (i["a_log"], 0), (i["dt_bias"], 0))
        if rows >= CHUNK_MIN_T:
            k.delta.conv_gated_delta_chunked(st, p, (i["conv_in"], 0), (i["conv_w"], 0), (b["q"], 0), *gates,
                                             (i["state_in"], 0), (b["state_out"], 0), (b["o"], 0), rows, n, n, True)
        else:
            k.conv.conv_silu_l2(st, p, (i["conv_in"], 0), (i["conv_w"], 0), (b["q"], 0), (b["kk"], 0), (b["v"], 0),
                                rows, n)
            k.delta.gated_delta(st, (b["q"], 0), (b["kk"], 0), (b["v"], 0), *gates, (i["state_in"], 0),
                                (b["state_out"], 0), (b["o"], 0), rows, n, True)
        k.conv.conv_state_update(st, p, (i["conv_in"], 0), (b["conv_out"], 0), rows, n)
        k.gnorm.gated_rmsnorm_silu(st, (b["o"], 0), (b["p"], 4 * LIN_Z), (i["gnorm"], 0), (b["g"], 0), rows, n)
        out = (b["x"], b["state_out"], b["conv_out"])
    else:
        k.rope.q_norm_rope(st, (b["p"], 0), (i["q_norm"], 0), (i["inv_freq"], 0), (i["qpos"], 0), (b["qo"], 0), rows,
                           n)
        k.rope.kv_norm_rope(st, (b["p"], 0), (i["k_norm"], 0), (i["inv_freq"], 0), (i["kc"], 0), (i["vc"], 0), rows,
                            n, ATT_K, ATT_V, case["pos0"])
        k.attn.attention(st, (b["qo"], 0), (i["kc"], 0), (i["vc"], 0), (b["p"], 0), (i["qpos"], 0), (b["g"], 0), rows,
                         n)
        out = (b["x"], i["kc"], i["vc"])
    k.gemm.gemm_add_rmsnorm(st, (b["g"], 0), (i["w_out"], 0), (b["x"], 0), rows, D, 4096, 4096, 4096, D,
                            (i["post_norm"], 0), (b["h"], 0), D, True, EPS)
    _run_mlp(s, rows)
    return out


def run(state):
    case, k, i = state["case"], state["k"], state["i"]
    if case["kind"] == "request":
        logits = state["model"].logits(state["stream"], i["ids"], i["answers"])
        return np.concatenate([np.array(v, np.float32) for v in logits])
    if case["kind"] == "head":
        b, st = state["b"], state["stream"]
        k.head.gather_rows_f32(st, (i["x"], 0), (i["rowmap"], 0), (b["xs"], 0), case["rows"], D)
        k.head.final_head(st, (b["xs"], 0), (i["final_norm"], 0), (i["table"], 0), (i["cand"], 0), (i["ncand"], 0),
                          (b["logits"], 0), case["rows"], D, case["cand"], EPS)
        return b["xs"], b["logits"]
    return _run_block(state)


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "head":
        r, c = case["rows"], case["cand"]
        return {"bytes": 4.0 * r * D * 2 + 2.0 * r * c * D + 4.0 * r * c, "flops": 2.0 * r * c * D}
    mlp = 3 * D * F
    lin, att = D * (LIN_N + 4096), D * (ATT_N + 4096)
    if kind == "request":
        rows = case["tokens"] - PREFIX
        n_att = REQ_LAYERS // 4
        n_lin = REQ_LAYERS - n_att
        weights = n_lin * (lin + mlp) + n_att * (att + mlp)
        states = n_lin * 2 * NV * DK * DK * 4
        last = D * (8192 + 4096) + mlp  # of the last layer, run for the answer rows only
        return {"bytes": 2.0 * weights + states + 2.0 * rows * D,
                "flops": 2.0 * rows * (weights - last) + 2.0 * len(REQ_COUNTS) * last + n_lin * rows * 6.0 * NV * DK * DK}
    rows = case["rows"]
    b = rows * D * (2 + 4)  # the embedding rows in, x out
    if kind == "mlp":
        if case["of"]:
            b = rows * D * 8
        return {"bytes": 2.0 * mlp + b, "flops": 2.0 * rows * mlp}
    if kind == "gdn":
        return {"bytes": 2.0 * (lin + mlp) + b + 2 * 4 * (NV * DK * DK + 3 * CONV),
                "flops": 2.0 * rows * (lin + mlp) + rows * 6.0 * NV * DK * DK}
    keys = rows * (case["pos0"] + (rows + 1) / 2.0)  # query-key pairs under the causal mask
    return {"bytes": 2.0 * (att + mlp) + b + 2.0 * 2 * NKV * HD * (case["pos0"] + rows),
            "flops": 2.0 * rows * (att + mlp) + 4.0 * keys * NQ * HD}


def tolerance(case):
    # four times what was measured between these calls and the same in 64 bits with the fp16 buffers' roundings (h, g,
    # the MLP's hidden, queries, caches): where a sum's last bits move a value across a rounding point, the products
    # behind it see that ulp
    return {"rel": {
        "mlp": 2.4e-4,  # 6e-5
        "gdn": 1.2e-3,  # 2.8e-4 (three products and the gated norm behind one another)
        "attn": 2.6e-3,  # 6.4e-4 (the probabilities enter their product as fp16)
        "head": 1e-6,  # 1.6e-7: fp32 sums of 2,560 products
        "request": 0.03,  # 7.4e-3: the same through 32 random-init layers
    }[case["kind"]]}


# ---- the same in 64 bits, nothing rounded on the way ----------------------------------------------------------------
def _mm(x, w, block=4096):
    return torch.cat([x @ w[n:n + block].double().t().contiguous() for n in range(0, w.shape[0], block)], 1)


def _rms(x, w, add_one=True):
    w = w.double() + 1.0 if add_one else w.double()
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_mlp(w, x):
    h = _rms(x, w["post_norm"])
    y = _mm(h, w["w_gu"]).view(len(x), F // 16, 2, 16)  # blocks of 16 gate rows, 16 up rows
    return x + _mm((_silu(y[:, :, 0]) * y[:, :, 1]).reshape(len(x), F), w["w_down"])


def _exact_gdn(w, x, conv_in, state):
    t = len(x)
    p = _mm(_rms(x, w["in_norm"]), w["w_in"])
    raw = torch.cat([conv_in.double(), p[:, :CONV]])
    y = _silu(sum(raw[j:j + t] * w["conv_w"][:, j].double() for j in range(4)))
    q, k = (y[:, o:o + NK * DK].view(t, NK, DK) for o in (0, NK * DK))
    q, k = (u * torch.rsqrt((u * u).sum(-1, keepdim=True) + 1e-6) for u in (q, k))
    q, k = ((u * f).repeat_interleave(NV // NK, 1).contiguous() for u, f in ((q, DK ** -0.5), (k, 1.0)))
    v = y[:, 2 * NK * DK:].reshape(t, NV, DK)
    a = torch.nn.functional.softplus(p[:, LIN_A:LIN_A + NV] + w["dt_bias"].double(), threshold=60.0)
    decay = torch.exp(-torch.exp(w["a_log"].double()) * a)
    beta = torch.sigmoid(p[:, LIN_B:LIN_B + NV])
    state, o = state.double().clone(), torch.empty(t, NV, DK, dtype=torch.float64, device=x.device)
    for s in range(t):  # state [head, value, key]
        state *= decay[s, :, None, None]
        d = (v[s] - (state * k[s, :, None, :]).sum(-1)) * beta[s, :, None]
        state += d[:, :, None] * k[s, :, None, :]
        o[s] = (state * q[s, :, None, :]).sum(-1)
    z = p[:, LIN_Z:LIN_Z + 4096].view(t, NV, DK)
    g = (_rms(o, w["gnorm"], add_one=False) * _silu(z)).reshape(t, 4096)
    return _exact_mlp(w, x + _mm(g, w["w_out"])), state, raw[t:t + 3].clone()


def _rope(u, w, pos):
    u = _rms(u, w)
    ang = (pos.float()[:, None] * _inv_freq()[None]).double()[:, None]  # the angle is an fp32 product by definition
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = u[..., :ROT], u[..., ROT:2 * ROT]
    return torch.cat([a * c - b * s, b * c + a * s, u[..., 2 * ROT:]], -1)


def _exact_attn(w, x, kc, vc, pos0, rows_out=None):
    """kc, vc: the caches' rows before pos0. rows_out: the rows to carry on with (all of them by default)."""
    t = len(x)
    pos = torch.arange(pos0, pos0 + t, device=x.device)
    p = _mm(_rms(x, w["in_norm"]), w["w_in"])
    kc = torch.cat([kc, _rope(p[:, ATT_K:ATT_V].view(t, NKV, HD), w["k_norm"], pos)])
    vc = torch.cat([vc, p[:, ATT_V:].reshape(t, NKV, HD)])
    if rows_out is not None:
        x, p, pos = x[rows_out], p[rows_out], pos[rows_out]
        t = len(x)
    q = _rope(p[:, :ATT_GATE].view(t, NQ, HD), w["q_norm"], pos)
    hidden = torch.arange(len(kc), device=x.device)[None] > pos[:, None]
    o = torch.empty(t, NQ, HD, dtype=torch.float64, device=x.device)
    for h in range(NQ):
        sc = q[:, h].contiguous() @ kc[:, h // 4].t().contiguous() / 16.0
        o[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), -1) @ vc[:, h // 4].contiguous()
    g = o.reshape(t, 4096) * torch.sigmoid(p[:, ATT_GATE:ATT_K])
    return _exact_mlp(w, x + _mm(g, w["w_out"])), kc, vc


def _exact_head(x, final_norm, table, cand):
    return torch.einsum("rd,rcd->rc", _rms(x, final_norm).cpu(), table[cand.long()].double().cpu())


def _exact_request(case, seed):
    i = _request_inputs(case, seed)
    ids = torch.tensor(i["ids"], device="cuda")
    rows = torch.tensor([r for r, _ in i["answers"]], device="cuda")
    table = final_norm = x = None
    w, layer = {}, 0
    for name, v in _request_weights(seed):
        if name == "embed":
            table, x = v, v[ids].double()
            continue
        if name == "final_norm":
            final_norm = v
            continue
        w[name.split(".")[1]] = v
        if not name.endswith("w_down"):
            continue
        if (layer + 1) % 4:
            x = _exact_gdn(w, x, torch.zeros(3, CONV, device="cuda"), torch.zeros(NV, DK, DK, device="cuda"))[0]
        else:
            none = torch.empty(0, NKV, HD, dtype=torch.float64, device="cuda")
            x = _exact_attn(w, x, none, none, 0, rows if layer == REQ_LAYERS - 1 else None)[0]
        w, layer = {}, layer + 1
    return torch.cat([_exact_head(x[r:r + 1], final_norm, table, torch.tensor([c], device="cuda"))[0]
                      for r, (_, c) in enumerate(i["answers"])])


def exact(case, seed):
    kind = case["kind"]
    if kind == "request":
        return _exact_request(case, seed)
    i = _inputs(case, seed)
    if kind == "head":
        xs = i["x"][i["rowmap"].long()].double()
        return xs, _exact_head(xs, i["final_norm"], i["table"], i["cand"].view(case["rows"], case["cand"]))
    x = (i["x_all"][i["rowmap"].long()] if case.get("of") else i["table"][i["ids"].long()]).double()
    if kind == "mlp":
        return _exact_mlp(i, x)
    if kind == "gdn":
        return _exact_gdn(i, x, i["conv_in"], i["state_in"])
    before = case["pos0"]
    return _exact_attn(i, x, i["kc"][:before].double(), i["vc"][:before].double(), before)
