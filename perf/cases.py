"""The workloads by which this library's speed is measured: what an inference engine asks of it, through its C ABI.

A case is one kind of call with its sizes:

  norm    rmsnorm of some tokens' hidden rows fused with their Q8_0 and Q8_K blocks (es_hip_rmsnorm_prepare_dev)
  ffn     the dense SwiGLU FFN of some tokens, layer after layer (es_hip_dense_ffn_dev)
  model   a decode step's products: per layer norm, q/k/v, output projection, norm and FFN, then the final norm and the head
  plan    a prepared batch of every layer's FFN matrices at once (es_hip_plan_*)
  head    the output head against some activations (es_hip_matvec_multi_dev)
  moe     device-routed MoE layers from the router's logits (es_hip_moe_ctx_*), optionally with the attention projections
  host    the engine's two job queues per FFN over host activations and outputs (es_hip_run_jobs_host)

listed() holds the named cases, draw() gives more of the same ranges, prepare() makes what a program holds before the call
(weights, activations, plans, contexts), run() is one pass, exact() the same results from plain torch in 64 bits.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "stream-_amd"))
import es_hip_quant as E  # noqa: E402

LIB = None
HEAD_ROWS = 151936


def lib():
    global LIB
    if LIB is None:
        LIB = E.Lib()
        if not LIB.available():
            raise RuntimeError(LIB.last_error())
    return LIB


# ---- the cases -------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one token's hidden row between two products of a decode step: the smallest call of the library, all latency
        dict(name="norm_t1", kind="norm", rows=1, cols=2048),
        # the same for a prompt chunk
        dict(name="norm_t512", kind="norm", rows=512, cols=2048),
        # batch-1 decode of a 0.5B model's FFNs in Q4_0 (896 wide, not a multiple of 256), 24 layers of small products
        dict(name="ffn_q4_0_t1", kind="ffn", gate="Q4_0", up="Q4_0", down="Q4_0", n=896, ff=4864, tokens=1, layers=24),
        # batch-1 decode of a whole 1B model: 16 layers in Q4_K and the Q6_K head, every product of the token in order
        dict(name="model_q4k_t1", kind="model", wtype="Q4_K", n=2048, kv=512, ff=8192, layers=16, head_rows=HEAD_ROWS, tokens=1),
        # every FFN matrix of 38 layers as one prepared batch at one token: weight streaming alone (1.08 GB)
        dict(name="plan_q4k_t1", kind="plan", wtype="Q4_K", n=2048, ff=8192, layers=38, tokens=1),
        # reading a prompt: a dense FFN over 512 tokens
        dict(name="ffn_q4k_t512", kind="ffn", gate="Q4_K", up="Q4_K", down="Q4_K", n=2048, ff=8192, tokens=512, layers=1),
        # reading a prompt in the engine's batches of 64 tokens with the usual mixed file (Q6_K down projections)
        dict(name="ffn_mixed_t64", kind="ffn", gate="Q4_K", up="Q4_K", down="Q6_K", n=2048, ff=8192, tokens=64, layers=4),
        # a ragged prompt chunk through a low-bit mixed file
        dict(name="ffn_q3k_q5k_t333", kind="ffn", gate="Q3_K", up="Q3_K", down="Q5_K", n=2048, ff=8192, tokens=333, layers=1),
        # the head of a 64-sequence decode batch
        dict(name="head_q6k_t64", kind="head", wtype="Q6_K", rows=HEAD_ROWS, cols=1024, tokens=64),
        # MoE prompt reading: 64 experts, top 8, 128 tokens, every expert used
        dict(name="moe_q2k_t128", kind="moe", gate="Q2_K", up="Q2_K", down="Q2_K", n=2048, ff=1024, experts=64, k=8, norm_topk=False,
             tokens=128, layers=4, attn=False),
        # MoE decode batch of 32 sequences with mixed formats and the Q5_0 attention projections
        dict(name="moe_mixed_t32", kind="moe", gate="Q4_K", up="Q4_K", down="Q6_K", n=2048, ff=768, experts=128, k=8, norm_topk=True,
             tokens=32, layers=3, attn=True),
        # MoE decode of a single sequence: 8 experts of 128 a layer, 12 layers
        dict(name="moe_mixed_t1", kind="moe", gate="Q4_K", up="Q4_K", down="Q6_K", n=2048, ff=768, experts=128, k=8, norm_topk=True,
             tokens=1, layers=12, attn=False),
    ]


def _log(rng, lo, hi, step=1):
    """a whole multiple of step in [lo, hi], spread evenly over its logarithm"""
    v = int(round(lo * (hi / lo) ** rng.random() / step)) * step
    return max(lo, min(hi, v))


DENSE_MIXES = [("Q4_K", "Q4_K", "Q4_K"), ("Q4_K", "Q4_K", "Q6_K"), ("Q3_K", "Q3_K", "Q5_K"), ("Q5_K", "Q5_K", "Q5_K"),
               ("Q2_K", "Q2_K", "Q3_K"), ("Q4_0", "Q4_0", "Q4_0"), ("Q8_0", "Q8_0", "Q8_0"), ("Q5_0", "Q5_0", "Q5_0"),
               ("Q6_K", "Q6_K", "Q6_K")]
MOE_MIXES = [("Q2_K", "Q2_K", "Q2_K"), ("Q4_K", "Q4_K", "Q6_K"), ("Q4_K", "Q4_K", "Q4_K")]


def draw(rng):
    kind = rng.choice(["norm", "ffn", "ffn", "ffn", "model", "plan", "head", "moe", "moe", "moe", "host"])
    if kind == "norm":
        return dict(kind=kind, rows=_log(rng, 1, 512), cols=_log(rng, 768, 8192, 32))
    if kind == "ffn":
        g, u, d = rng.choice(DENSE_MIXES)
        step = 32 if E.BLOCK_ELEMS[E.TYPES[g]] == 32 else 256
        n, tokens = _log(rng, 768, 4096, step), _log(rng, 1, 512)
        ff = _log(rng, 1024, 8192, step)
        return dict(kind=kind, gate=g, up=u, down=d, n=n, ff=ff, tokens=tokens, layers=rng.randint(1, 8 if tokens <= 16 else 2))
    if kind == "model":
        n = rng.choice([1024, 1536, 2048])
        return dict(kind=kind, wtype=rng.choice(["Q4_K", "Q5_K", "Q6_K"]), n=n, kv=256 * rng.randint(1, 4),
                    ff=_log(rng, 2048, 8192, 256), layers=rng.randint(2, 12), head_rows=_log(rng, 32000, HEAD_ROWS),
                    tokens=_log(rng, 1, 8))
    if kind == "plan":
        return dict(kind=kind, wtype=rng.choice(["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0"]), n=_log(rng, 1024, 4096, 256),
                    ff=_log(rng, 2048, 8192, 256), layers=rng.randint(4, 32), tokens=rng.randint(1, 4))
    if kind == "head":
        return dict(kind=kind, wtype=rng.choice(["Q6_K", "Q6_K", "Q8_0"]), rows=_log(rng, 32000, HEAD_ROWS), cols=_log(rng, 768, 2048, 256),
                    tokens=_log(rng, 1, 64))
    if kind == "host":
        return dict(kind=kind, wtype=rng.choice(["Q4_K", "Q4_0", "Q6_K"]), n=_log(rng, 1024, 2048, 256), ff=_log(rng, 2048, 8192, 256),
                    tokens=_log(rng, 1, 64))
    g, u, d = rng.choice(MOE_MIXES)
    tokens = _log(rng, 1, 128)
    return dict(kind="moe", gate=g, up=u, down=d, n=_log(rng, 1024, 2048, 256), ff=_log(rng, 512, 1024, 256),
                experts=rng.choice([16, 32, 60, 64, 128]), k=rng.choice([2, 4, 6, 8]), norm_topk=rng.random() < 0.5, tokens=tokens,
                layers=rng.randint(1, 6 if tokens <= 8 else 2), attn=False)


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _weights(g, name, rows, cols):
    """random blocks [rows, nb, block bytes]: uniform codes, weights around zero of standard deviation about cols^-1/2, the
    min terms of the K-quants near the codes' middle as a quantizer of centred weights leaves them"""
    t = E.TYPES[name]
    nb, bb = cols // E.BLOCK_ELEMS[t], E.BLOCK_BYTES[t]
    n = rows * nb * bb
    w = torch.empty((n + 3) // 4, dtype=torch.int32, device="cuda").random_(-2**31, 2**31, generator=g).view(torch.uint8)[:n]
    w = w.view(rows, nb, bb)
    u = 0.75 + 0.5 * torch.rand((rows, nb), device="cuda", generator=g)
    sd = cols ** -0.5
    # standard deviation of a weight at block scale 1
    unit = {"Q4_0": 4.6, "Q5_0": 9.2, "Q8_0": 74.0, "Q2_K": 1.1 * 9, "Q3_K": 2.3 * 18, "Q4_K": 4.6 * 32, "Q5_K": 9.2 * 32,
            "Q6_K": 18.5 * 74}[name]
    d = (sd / unit * u)

    def half(pos, v):
        w[:, :, pos:pos + 2] = v.to(torch.float16).view(torch.uint8).view(rows, nb, 2)

    if name in ("Q4_0", "Q5_0", "Q8_0"):
        half(0, d)
    elif name in ("Q4_K", "Q5_K"):   # each sub-block's 6-bit min code equals its scale code
        half(0, d)
        half(2, d * (7.5 if name == "Q4_K" else 15.5))
        w[:, :, 8:12] = w[:, :, 4:8]
        w[:, :, 12:16] = (w[:, :, 12:16] & 15) * 17
    elif name == "Q2_K":             # scale nibble = min nibble
        w[:, :, 0:16] = (w[:, :, 0:16] & 15) * 17
        half(80, d)
        half(82, d * 1.5)
    elif name == "Q3_K":
        half(108, d)
    else:
        half(208, d)
    return w


def _ptr(t):
    return t.data_ptr()


def _blocks(t, x):
    """x [T, cols] fp32 -> the activation blocks weights of type t take, [T, bytes]"""
    T, cols = x.shape
    out = torch.zeros((T, E.act_bytes(t, cols)), dtype=torch.uint8, device="cuda")
    k = E.BLOCK_ELEMS[t] == 256
    lib().act_prepare_dev(_ptr(x), 0, T, cols, None if k else _ptr(out), 0, _ptr(out) if k else None, 0)
    return out


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _zeros(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def _ffn_layer(g, c):
    return {"g": _weights(g, c["gate"], c["ff"], c["n"]), "u": _weights(g, c["up"], c["ff"], c["n"]),
            "d": _weights(g, c["down"], c["n"], c["ff"])}


def _inputs(c, seed):
    """the tensors of a case, from the seed alone (shared by prepare and exact)"""
    g = _gen(seed)
    k = c["kind"]
    if k == "norm":
        return {"x": _randn(g, c["rows"], c["cols"]) * 3.0, "w": 1.0 + 0.1 * _randn(g, c["cols"])}
    if k == "ffn":
        return {"layers": [_ffn_layer(g, c) for _ in range(c["layers"])],
                "x": [_randn(g, c["tokens"], c["n"]) for _ in range(c["layers"])]}
    if k == "model":
        t, n, kv, ff = c["wtype"], c["n"], c["kv"], c["ff"]
        ls = []
        for _ in range(c["layers"]):
            ls.append({"n1": 1.0 + 0.1 * _randn(g, n), "q": _weights(g, t, n, n), "k": _weights(g, t, kv, n), "v": _weights(g, t, kv, n),
                       "o": _weights(g, t, n, n), "n2": 1.0 + 0.1 * _randn(g, n), "g": _weights(g, t, ff, n),
                       "u": _weights(g, t, ff, n), "d": _weights(g, t, n, ff)})
        return {"layers": ls, "nf": 1.0 + 0.1 * _randn(g, n), "head": _weights(g, "Q6_K", c["head_rows"], n),
                "x": _randn(g, c["layers"] + 1, c["tokens"], n)}
    if k in ("plan", "host"):
        t, n, ff = c["wtype"], c["n"], c["ff"]
        mix = dict(gate=t, up=t, down=t, n=n, ff=ff)
        return {"layers": [_ffn_layer(g, mix) for _ in range(c.get("layers", 1))], "x": _randn(g, c["tokens"], n),
                "h": _randn(g, c["tokens"], ff)}
    if k == "head":
        return {"w": _weights(g, c["wtype"], c["rows"], c["cols"]), "x": _randn(g, c["tokens"], c["cols"])}
    ne, n, ff = c["experts"], c["n"], c["ff"]
    ls = []
    for _ in range(c["layers"]):
        l = {"g": _weights(g, c["gate"], ne * ff, n), "u": _weights(g, c["up"], ne * ff, n), "d": _weights(g, c["down"], ne * n, ff),
             "logits": _randn(g, c["tokens"], ne), "x": _randn(g, c["tokens"], n)}
        if c["attn"]:
            l["attn"] = [_weights(g, "Q5_0", r, n) for r in (4096, 512, 512)]
        ls.append(l)
    return {"layers": ls}


class _Registered:
    """host weights kept registered (resident on the device) while the state lives"""

    def __init__(self, arrays):
        self.arrays = arrays
        for a in arrays:
            lib().register(a)

    def __del__(self):
        for a in self.arrays:
            lib().unregister(a)


def _host_blocks(t, x):
    """[T, nblocks] records in host memory"""
    b = _blocks(t, x).cpu().numpy()
    return np.ascontiguousarray(b.reshape(x.shape[0], -1, E.ACT_BYTES[t]))


def prepare(case, seed):
    c, L = case, lib()
    s = {"case": c, "in": _inputs(c, seed)}
    i, k = s["in"], c["kind"]
    if k == "norm":
        r, n = c["rows"], c["cols"]
        s["xn"], s["q80"] = _zeros(r, n), torch.zeros((r, n // 32 * 36), dtype=torch.uint8, device="cuda")
        s["q8k"] = torch.zeros((r, n // 256 * 292), dtype=torch.uint8, device="cuda") if n % 256 == 0 else None
    elif k == "ffn":
        T, n, ff = c["tokens"], c["n"], c["ff"]
        s["xb"] = [_blocks(E.TYPES[c["gate"]], x) for x in i["x"]]
        s["gu"], s["hq"] = _zeros(T, 2 * ff), torch.zeros((T, E.act_bytes(E.TYPES[c["down"]], ff)), dtype=torch.uint8, device="cuda")
        s["out"] = [_zeros(T, n) for _ in i["x"]]
    elif k == "model":
        T, n, kv, ff, t = c["tokens"], c["n"], c["kv"], c["ff"], E.TYPES[c["wtype"]]
        s["xb"] = torch.zeros((T, E.act_bytes(t, n)), dtype=torch.uint8, device="cuda")
        s["qb"] = torch.zeros_like(s["xb"])
        s["q"], s["kk"], s["v"] = _zeros(T, n), _zeros(c["layers"], T, kv), _zeros(c["layers"], T, kv)
        s["h"], s["o"] = _zeros(c["layers"], T, n), _zeros(T, n)
        s["gu"], s["hq"] = _zeros(T, 2 * ff), torch.zeros((T, E.act_bytes(t, ff)), dtype=torch.uint8, device="cuda")
        s["logits"] = _zeros(T, c["head_rows"])
        s["qkv"] = []
        for j, l in enumerate(i["layers"]):
            jobs = [dict(type=t, rows=m.shape[0], cols=n, W=_ptr(m), act=_ptr(s["xb"]), astride=s["xb"].stride(0), nb=T, y=_ptr(y),
                         ystride=m.shape[0]) for m, y in ((l["q"], s["q"]), (l["k"], s["kk"][j]), (l["v"], s["v"][j]))]
            s["qkv"].append(L.plan(jobs))
    elif k == "plan":
        T, t = c["tokens"], E.TYPES[c["wtype"]]
        xb, hb = _blocks(t, i["x"]), _blocks(t, i["h"])
        s["keep"], s["y"], jobs = (xb, hb), {}, []
        for m, rows in (("g", c["ff"]), ("u", c["ff"]), ("d", c["n"])):
            s["y"][m] = _zeros(c["layers"], T, rows)
        for j, l in enumerate(i["layers"]):
            for name, a, cols in (("g", xb, c["n"]), ("u", xb, c["n"]), ("d", hb, c["ff"])):
                m, y = l[name], s["y"][name][j]
                jobs.append(dict(type=t, rows=m.shape[0], cols=cols, W=_ptr(m), act=_ptr(a), astride=a.stride(0), nb=T, y=_ptr(y),
                                 ystride=m.shape[0]))
        s["plan"] = L.plan(jobs)
    elif k == "head":
        s["xb"], s["y"] = _blocks(E.TYPES[c["wtype"]], i["x"]), _zeros(c["tokens"], c["rows"])
    elif k == "host":
        T, n, ff, t = c["tokens"], c["n"], c["ff"], E.TYPES[c["wtype"]]
        W = [i["layers"][0][m].cpu().numpy() for m in "gud"]
        s["reg"] = _Registered(W)
        x, h = _host_blocks(t, i["x"]), _host_blocks(t, i["h"])
        s["gu"], s["out"] = np.zeros((T, 2 * ff), np.float32), np.zeros((T, n), np.float32)
        s["q1"] = L.host_jobs([(t, W[0], ff, n, x, s["gu"][:, :ff]), (t, W[1], ff, n, x, s["gu"][:, ff:])])
        s["q2"] = L.host_jobs([(t, W[2], n, ff, h, s["out"])])
    else:
        T, ne, n, ff, kk = c["tokens"], c["experts"], c["n"], c["ff"], c["k"]
        types = [E.TYPES[c[m]] for m in ("gate", "up", "down")]
        s["xb"] = [_blocks(types[0], l["x"]) for l in i["layers"]]
        s["ctx"], s["out"], s["plans"], s["ya"], s["xa"] = [], [], [], [], []
        for j, l in enumerate(i["layers"]):
            sizes = [E.row_bytes(types[0], n) * ff, E.row_bytes(types[1], n) * ff, E.row_bytes(types[2], ff) * n]
            experts = [{m: _ptr(l[m[0]]) + e * z for m, z in zip(("gate", "up", "down"), sizes)} for e in range(ne)]
            args = E.MoeArgs(*types, n, ff, experts, np.full(T, kk), np.zeros((T, kk)), np.zeros((T, kk)))
            s["ctx"].append(L.moe_ctx(args, T, kk))
            s["out"].append((_zeros(T, n), torch.zeros((T, kk), dtype=torch.int32, device="cuda"), _zeros(T, kk)))
            if c["attn"]:
                xa = _blocks(E.Q5_0, l["x"])
                ya = [_zeros(T, m.shape[0]) for m in l["attn"]]
                s["xa"].append(xa)
                s["ya"].append(ya)
                s["plans"].append(L.plan([dict(type=E.Q5_0, rows=m.shape[0], cols=n, W=_ptr(m), act=_ptr(xa), astride=xa.stride(0), nb=T,
                                               y=_ptr(y), ystride=m.shape[0]) for m, y in zip(l["attn"], ya)]))
    return s


# ---- one pass --------------------------------------------------------------------------------------------------------
def run(s):
    c, i, L = s["case"], s["in"], lib()
    k = c["kind"]
    if k == "norm":
        q8k = s["q8k"]
        L.rmsnorm_prepare_dev(_ptr(i["x"]), 0, _ptr(i["w"]), 1e-5, c["rows"], c["cols"], _ptr(s["xn"]), 0, _ptr(s["q80"]), 0,
                              None if q8k is None else _ptr(q8k), 0)
        return [s["xn"], s["q80"]] + ([] if q8k is None else [q8k])
    if k == "ffn":
        t = [E.TYPES[c[m]] for m in ("gate", "up", "down")]
        for l, xb, out in zip(i["layers"], s["xb"], s["out"]):
            L.dense_ffn_dev(t[0], _ptr(l["g"]), t[1], _ptr(l["u"]), t[2], _ptr(l["d"]), c["n"], c["ff"], c["tokens"], _ptr(xb),
                            xb.stride(0), _ptr(s["gu"]), _ptr(s["hq"]), _ptr(out), c["n"])
        return s["out"]
    if k == "model":
        # the attention itself and the residual adds are the engine's: the output projection takes the q rows here, and each
        # layer (and the head) starts from hidden rows of its own
        T, n, t = c["tokens"], c["n"], E.TYPES[c["wtype"]]
        xb, qb, astr = _ptr(s["xb"]), _ptr(s["qb"]), s["xb"].stride(0)
        o, q = _ptr(s["o"]), _ptr(s["q"])
        for l, plan, x, h in zip(i["layers"], s["qkv"], i["x"], s["h"]):
            L.rmsnorm_prepare_dev(_ptr(x), 0, _ptr(l["n1"]), 1e-5, T, n, None, 0, None, 0, xb, 0)
            plan.run()
            L.act_prepare_dev(q, 0, T, n, None, 0, qb, 0)
            L.matvec_multi_dev(t, _ptr(l["o"]), n, 0, n, qb, astr, T, o, n)
            L.rmsnorm_prepare_dev(o, 0, _ptr(l["n2"]), 1e-5, T, n, None, 0, None, 0, xb, 0)
            L.dense_ffn_dev(t, _ptr(l["g"]), t, _ptr(l["u"]), t, _ptr(l["d"]), n, c["ff"], T, xb, astr, _ptr(s["gu"]), _ptr(s["hq"]),
                            _ptr(h), n)
        L.rmsnorm_prepare_dev(_ptr(i["x"][-1]), 0, _ptr(i["nf"]), 1e-5, T, n, None, 0, None, 0, xb, 0)
        L.matvec_multi_dev(E.Q6_K, _ptr(i["head"]), n, 0, c["head_rows"], xb, astr, T, _ptr(s["logits"]), c["head_rows"])
        return {"logits": s["logits"], "k": s["kk"], "v": s["v"], "h": s["h"]}
    if k == "plan":
        s["plan"].run()
        return s["y"]
    if k == "head":
        xb = s["xb"]
        L.matvec_multi_dev(E.TYPES[c["wtype"]], _ptr(i["w"]), c["cols"], 0, c["rows"], _ptr(xb), xb.stride(0), c["tokens"], _ptr(s["y"]),
                           c["rows"])
        return s["y"]
    if k == "host":
        for (arr, _), n in ((s["q1"], 2), (s["q2"], 1)):
            L._check(L._L.es_hip_run_jobs_host(arr, n))
        return [s["gu"], s["out"]]
    for j, l in enumerate(i["layers"]):
        if s["plans"]:
            s["plans"][j].run()
        out, sel, w = s["out"][j]
        xb = s["xb"][j]
        s["ctx"][j].run_logits(c["tokens"], _ptr(l["logits"]), 0, c["norm_topk"], _ptr(xb), xb.stride(0), _ptr(out), c["n"], _ptr(sel), _ptr(w))
    return {"moe": s["out"], "attn": s["ya"]}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def work(case):
    c, k = case, case["kind"]

    def mat(t, rows, cols, T):
        """(bytes, operations) of one product: weights, activation blocks in, outputs out"""
        t = E.TYPES[t]
        return E.row_bytes(t, cols) * rows + E.act_bytes(t, cols) * T + 4 * rows * T, 2 * rows * cols * T

    if k == "norm":
        r, n = c["rows"], c["cols"]
        return {"bytes": r * (8 * n + n // 32 * 36 + (n // 256 * 292 if n % 256 == 0 else 0)) + 4 * n, "flops": 4 * r * n}
    if k == "ffn":
        parts = [mat(c["gate"], c["ff"], c["n"], c["tokens"]), mat(c["up"], c["ff"], c["n"], c["tokens"]),
                 mat(c["down"], c["n"], c["ff"], c["tokens"])] * c["layers"]
        # gate and up share their activation rows, and the float gate|up rows need not leave the chip
        dup = (E.act_bytes(E.TYPES[c["up"]], c["n"]) + 8 * c["ff"]) * c["tokens"] * c["layers"]
        return {"bytes": sum(p[0] for p in parts) - dup, "flops": sum(p[1] for p in parts)}
    if k == "model":
        t, n, kv, ff, T = c["wtype"], c["n"], c["kv"], c["ff"], c["tokens"]
        one = [mat(t, n, n, T), mat(t, kv, n, T), mat(t, kv, n, T), mat(t, n, n, T), mat(t, ff, n, T), mat(t, ff, n, T), mat(t, n, ff, T)]
        head = mat("Q6_K", c["head_rows"], n, T)
        return {"bytes": c["layers"] * sum(p[0] for p in one) + head[0], "flops": c["layers"] * sum(p[1] for p in one) + head[1]}
    if k in ("plan", "host"):
        t, n, ff, T = c["wtype"], c["n"], c["ff"], c["tokens"]
        parts = [mat(t, ff, n, T), mat(t, ff, n, T), mat(t, n, ff, T)] * c.get("layers", 1)
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if k == "head":
        b, f = mat(c["wtype"], c["rows"], c["cols"], c["tokens"])
        return {"bytes": b, "flops": f}
    T, ne, n, ff, kk = c["tokens"], c["experts"], c["n"], c["ff"], c["k"]
    used = ne * (1 - (1 - kk / ne) ** T)   # experts that a random routing reads
    per = E.row_bytes(E.TYPES[c["gate"]], n) * ff + E.row_bytes(E.TYPES[c["up"]], n) * ff + E.row_bytes(E.TYPES[c["down"]], ff) * n
    b = used * per + T * (E.act_bytes(E.TYPES[c["gate"]], n) + 4 * n + 4 * ne)
    f = 2 * T * kk * 3 * n * ff
    if c["attn"]:
        parts = [mat("Q5_0", r, n, T) for r in (4096, 512, 512)]
        b, f = b + sum(p[0] for p in parts), f + sum(p[1] for p in parts)
    return {"bytes": b * c["layers"], "flops": f * c["layers"]}


def tolerance(case):
    # Products of 8-bit integers are exact, their float sums over a row's blocks in 32 bits (a few 1e-7 from 64 bits). Where a
    # result is quantized again inside the call (FFN and MoE layers), a last-bit difference before a rounding moves an 8-bit
    # value by one step; a whole model's layer does so four times in a row.
    k = case["kind"]
    if k == "norm":
        return {"rel": 1e-6, "differ": 0.0}
    if k in ("plan", "head", "host"):
        return {"rel": 4e-6}
    if k == "model":
        return {"rel": 5e-3}
    return {"rel": 2.5e-3, "differ": 0.0}


# ---- the same results in 64 bits ---------------------------------------------------------------------------------------
def _half(w, pos):
    return w[..., pos:pos + 2].contiguous().view(torch.float16)[..., 0].double()


def _decode(name, w):
    """blocks [rows, nb, bytes] -> weights [rows, cols] in 64 bits (the GGUF block formats)"""
    rows, nb = w.shape[0], w.shape[1]
    if name in ("Q4_0", "Q5_0"):
        off = 2 if name == "Q4_0" else 6
        qs = w[..., off:off + 16].to(torch.int32)
        q = torch.cat([qs & 15, qs >> 4], -1)
        if name == "Q5_0":
            qh = w[..., 2:6].to(torch.int32)
            bits = torch.stack([(qh >> b) & 1 for b in range(8)], -1).reshape(rows, nb, 32)
            q = q + 16 * bits
        v = (q - (8 if name == "Q4_0" else 16)).double() * _half(w, 0)[..., None]
    elif name == "Q8_0":
        v = w[..., 2:34].contiguous().view(torch.int8).double() * _half(w, 0)[..., None]
    elif name in ("Q4_K", "Q5_K"):
        s = w[..., 4:16].to(torch.int32)
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
        off = 16 if name == "Q4_K" else 48
        qs = w[..., off:off + 128].to(torch.int32).reshape(rows, nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 3).reshape(rows, nb, 8, 32)
        if name == "Q5_K":
            qh = w[..., 16:48].to(torch.int32)
            q = q + 16 * torch.stack([(qh >> j) & 1 for j in range(8)], 2)
        v = (_half(w, 0)[..., None] * sc)[..., None] * q - (_half(w, 2)[..., None] * mn)[..., None]
    elif name == "Q6_K":
        ql = w[..., 0:128].to(torch.int32).reshape(rows, nb, 2, 2, 32)
        qh = w[..., 128:192].to(torch.int32).reshape(rows, nb, 2, 32)
        parts = [(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | (((qh >> 2) & 3) << 4),
                 (ql[..., 0, :] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 1, :] >> 4) | ((qh >> 6) << 4)]
        q = torch.stack(parts, 3).reshape(rows, nb, 16, 16) - 32
        sc = w[..., 192:208].contiguous().view(torch.int8).double()
        v = (_half(w, 208)[..., None] * sc)[..., None] * q
    elif name == "Q2_K":
        s = w[..., 0:16].to(torch.int32)
        qs = w[..., 16:80].to(torch.int32).reshape(rows, nb, 2, 32)
        q = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], 3).reshape(rows, nb, 16, 16)
        v = (_half(w, 80)[..., None] * (s & 15))[..., None] * q - (_half(w, 82)[..., None] * (s >> 4))[..., None]
    else:   # Q3_K
        hm = w[..., 0:32].to(torch.int32)
        qs = w[..., 32:96].to(torch.int32).reshape(rows, nb, 2, 32)
        lo = torch.stack([(qs >> (2 * j)) & 3 for j in range(4)], 3)                                   # [.., half, j, 32]
        hi = torch.stack([torch.stack([(hm >> (4 * n + j)) & 1 for j in range(4)], 2) for n in range(2)], 2)
        q = (lo + 4 * hi - 4).reshape(rows, nb, 16, 16)
        s = w[..., 96:108].to(torch.int32)
        low = torch.cat([s[..., 0:8] & 15, s[..., 0:8] >> 4], -1)
        top = torch.cat([(s[..., 8:12] >> (2 * j)) & 3 for j in range(4)], -1)
        v = (_half(w, 108)[..., None] * ((low | (top << 4)) - 32))[..., None] * q
    return v.double().reshape(rows, -1)


def _quant(name, x):
    """x [T, cols] -> what its activation blocks for weights of this format stand for, in 64 bits. A 32-bit x is quantized
    in 32 bits as the library's inputs are, a 64-bit one in 64."""
    if E.BLOCK_ELEMS[E.TYPES[name]] == 256:
        b = x.reshape(x.shape[0], -1, 256)
        amax = b.abs().amax(-1, keepdim=True)
        q = torch.where(amax > 0, torch.round(b * (127.0 / amax)).clamp(-127, 127), torch.zeros_like(b))
        d = amax / 127.0
    else:
        b = x.reshape(x.shape[0], -1, 32)
        d = b.abs().amax(-1, keepdim=True) / 127.0
        v = b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
        q = torch.trunc(torch.where(v < 0, v - 0.5, v + 0.5))
    return (q.double() * d.double()).reshape(x.shape[0], -1)


def _product(name, w, a, chunk=16384):
    """w blocks against activations a [T, cols] in 64 bits, some rows at a time"""
    return torch.cat([a @ _decode(name, w[r:r + chunk]).T for r in range(0, w.shape[0], chunk)], 1)


def _ffn64(types, g, u, d, a):
    gate, up = _product(types[0], g, a), _product(types[1], u, a)
    return _product(types[2], d, _quant(types[2], gate / (1.0 + torch.exp(-gate)) * up))


def _norm64(x, w):
    x = x.double()
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + float(np.float32(1e-5))) * w.double()


def exact(case, seed):
    c, k = case, case["kind"]
    i = _inputs(c, seed)
    if k == "norm":
        return [_norm64(i["x"], i["w"])] + [None] * (2 if c["cols"] % 256 == 0 else 1)
    if k == "ffn":
        t = (c["gate"], c["up"], c["down"])
        return [_ffn64(t, l["g"], l["u"], l["d"], _quant(t[0], x)) for l, x in zip(i["layers"], i["x"])]
    if k == "model":
        t, ks, vs, hs = c["wtype"], [], [], []
        for l, x in zip(i["layers"], i["x"]):
            a = _quant(t, _norm64(x, l["n1"]))
            ks.append(_product(t, l["k"], a))
            vs.append(_product(t, l["v"], a))
            o = _product(t, l["o"], _quant(t, _product(t, l["q"], a)))
            hs.append(_ffn64((t, t, t), l["g"], l["u"], l["d"], _quant(t, _norm64(o, l["n2"]))))
        return {"logits": _product("Q6_K", i["head"], _quant("Q6_K", _norm64(i["x"][-1], i["nf"]))), "k": torch.stack(ks),
                "v": torch.stack(vs), "h": torch.stack(hs)}
    if k == "plan":
        t = c["wtype"]
        a, h = _quant(t, i["x"]), _quant(t, i["h"])
        return {m: torch.stack([_product(t, l[m], h if m == "d" else a) for l in i["layers"]]) for m in "gud"}
    if k == "head":
        return _product(c["wtype"], i["w"], _quant(c["wtype"], i["x"]))
    if k == "host":
        t, l = c["wtype"], i["layers"][0]
        a, h = _quant(t, i["x"]), _quant(t, i["h"])
        return [torch.cat([_product(t, l["g"], a), _product(t, l["u"], a)], 1), _product(t, l["d"], h)]
    t, T, n, ff, kk = (c["gate"], c["up"], c["down"]), c["tokens"], c["n"], c["ff"], c["k"]
    moe, attn = [], []
    for l in i["layers"]:
        p = torch.softmax(l["logits"].double(), -1)
        w, sel = torch.topk(p, kk, -1)
        if c["norm_topk"]:
            w = w / w.sum(-1, keepdim=True).clamp_min(2.0 ** -14)
        a = _quant(t[0], l["x"])
        out = torch.zeros((T, n), dtype=torch.float64, device="cuda")
        for e in sorted(set(sel.reshape(-1).tolist())):
            at, j = torch.nonzero(sel == e, as_tuple=True)
            y = _ffn64(t, l["g"][e * ff:(e + 1) * ff], l["u"][e * ff:(e + 1) * ff], l["d"][e * n:(e + 1) * n], a[at])
            out[at] += w[at, j][:, None] * y
        moe.append((out, None, w))
        if c["attn"]:
            aa = _quant("Q5_0", l["x"])
            attn.append([_product("Q5_0", m, aa) for m in l["attn"]])
    return {"moe": moe, "attn": attn}
