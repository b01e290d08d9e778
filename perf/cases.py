"""The workloads this library's performance is measured on: quantized MoE
layers, dense quantized products and whole-model calls, each through its
public entry point (llm.c_amd/hipmoe.py, llm.c_amd/hiplm.py over the C ABI of
include/hip_moe.h and include/hip_lm.h).

Shapes are those of bench.py and of the tests: the OLMoE-1B-7B and
Mixtral-8x7B layers and models, and the tests' reduced ones.  Weights are
N(0, 0.02) in GGUF blocks of each type, activations N(0, 1), routers N(0,
0.02) fp32, token ids uniform.

Calls pass no stream: they run on the library's own stream, in call order,
as every caller without a stream of its own has them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "llm.c_amd"))
import hiplm  # noqa: E402
import hipmoe  # noqa: E402

TYPES = {"q8_0": hipmoe.Q8_0, "q4_0": hipmoe.Q4_0, "q4_k": hipmoe.Q4_K, "q6_k": hipmoe.Q6_K}
KQUANT = ("q4_k", "q6_k")
# E, EI, NE, topk, renorm
SHAPES = {
    "olmoe": (2048, 1024, 64, 8, 0),
    "mixtral": (4096, 14336, 8, 2, 1),
    "olmoe_small": (1024, 512, 64, 8, 0),
    "mixtral_small": (2048, 1024, 8, 2, 1),
}
# heads, kv heads, vocabulary, rope theta
MODELS = {
    "olmoe": (16, 16, 50304, 1e4),
    "mixtral": (32, 8, 32000, 1e6),
    "olmoe_small": (8, 8, 512, 1e4),
    "mixtral_small": (16, 4, 512, 1e6),
}
CONTEXT = 1024


def _layer(shape, gate, down, T, bias=False, host=False, name=None):
    return dict(({"name": name} if name else {}), kind="layer", shape=shape, gate=gate,
                down=down, T=T, bias=bias, host=host)


def _dense(wtype, N, K, T, add, name=None):
    return dict(({"name": name} if name else {}), kind="dense", wtype=wtype, N=N, K=K, T=T,
                add=add)


def _model(shape, wtype, layers, seqs, prompt, steps, name=None):
    return dict(({"name": name} if name else {}), kind="model", shape=shape, wtype=wtype,
                layers=layers, seqs=seqs, prompt=prompt, steps=steps)


def listed():
    return [
        # one generated token through the C drop-in for moe_ffn: host buffers, synchronous
        _layer("olmoe", "q8_0", "q8_0", 1, host=True, name="olmoe_q8_t1_host"),
        # one generated token of the large model, activations on the device
        _layer("mixtral", "q4_0", "q4_0", 1, name="mixtral_q4_t1"),
        # sixty-four sequences served together: every expert a handful of tokens
        _layer("mixtral", "q4_0", "q4_0", 64, name="mixtral_q4_t64"),
        # a 512-token prompt with a router that loads its experts unevenly
        _layer("olmoe", "q4_0", "q4_0", 512, bias=True, name="olmoe_q4_t512_skew"),
        # a Q4_K_M file: one generated token, a prompt of ordinary length, and
        # the large model's prompt
        _layer("olmoe", "q4_k", "q6_k", 1, name="olmoe_q4km_t1"),
        _layer("olmoe", "q4_k", "q6_k", 301, name="olmoe_q4km_t301"),
        _layer("mixtral", "q4_k", "q6_k", 200, name="mixtral_q4km_t200"),
        # the lm_head of one generated token
        _dense("q8_0", 50304, 2048, 1, "none", name="dense_q8_lm_head_t1"),
        # q/k/v of a prompt's rows
        _dense("q4_0", 6144, 4096, 333, "none", name="dense_q4_qkv_t333"),
        # the output product of a Q4_K_M prompt with its residual
        _dense("q4_k", 4096, 4096, 77, "full", name="dense_q4k_out_t77"),
        # a 512-token prompt, then four generated tokens, two full layers and the head
        _model("olmoe", "q8_0", 2, 1, 512, 4, name="olmoe_prompt512_decode4"),
        # sixteen sequences in lockstep: their prompts, then four tokens each
        _model("mixtral", "q4_0", 1, 16, 64, 4, name="mixtral_lockstep16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    """Another case of the listed ones' ranges."""
    kind = rng.choice(("layer", "layer", "layer", "dense", "dense", "model"))
    if kind == "layer":
        shape = rng.choice(("olmoe", "olmoe", "mixtral", "olmoe_small", "mixtral_small"))
        gate, down = rng.choice((("q8_0", "q8_0"), ("q4_0", "q4_0"), ("q4_k", "q6_k"),
                                 ("q4_k", "q4_k"), ("q6_k", "q6_k")))
        most = 200 if shape == "mixtral" else 512 if gate in KQUANT else 2048
        T = _log_int(rng, 1, most)
        return _layer(shape, gate, down, T, bias=rng.random() < 0.3, host=rng.random() < 0.2)
    if kind == "dense":
        wtype = rng.choice(tuple(TYPES))
        N, K = rng.choice(((6144, 2048), (2048, 2048), (6144, 4096), (4096, 4096),
                           (rng.randrange(300, 5000), 1024)) +
                          (((4096, 14336),) if wtype in KQUANT else ()))
        T = _log_int(rng, 1, 512)
        if rng.random() < 0.2:
            N, K = rng.choice(((50304, 2048), (32000, 4096)))
            T = _log_int(rng, 1, 16)
        return _dense(wtype, N, K, T, rng.choice(("none", "row", "full")))
    shape = rng.choice(("olmoe", "olmoe_small", "mixtral_small"))
    seqs = rng.choice((1, 1, rng.randrange(2, 17)))
    return _model(shape, rng.choice(("q8_0", "q4_0")), rng.choice((1, 2)), seqs,
                  _log_int(rng, 2, 512 // seqs), rng.randrange(1, 5))


# --------------------------------------------------------------------------
# inputs, made on the GPU from the seed
# --------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _f16(v):
    """fp32 [...] -> its f16 bytes [..., 2]"""
    return v.half().contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _pack(x, wtype):
    """Rows of values x [rows, cols] as GGUF blocks: uint8 [rows, bytes]."""
    rows = x.shape[0]
    if wtype in ("q8_0", "q4_0"):
        b = x.reshape(rows, -1, 32)
        d = b.abs().amax(-1) / (127 if wtype == "q8_0" else 7)
        q = torch.round(b / d.clamp_min(1e-30)[..., None]).to(torch.int8)
        if wtype == "q4_0":
            q = (q + 8).clamp(0, 15).to(torch.uint8)
            q = q[..., :16] | (q[..., 16:] << 4)
        return torch.cat([_f16(d), q.view(torch.uint8)], -1).reshape(rows, -1)
    if wtype == "q4_k":
        b = x.reshape(rows, -1, 8, 32)
        lo = b.amin(-1).clamp_max(0)
        s, m = (b.amax(-1) - lo) / 15, -lo
        d, dm = s.amax(-1) / 63, m.amax(-1) / 63
        sc = torch.round(s / d[..., None]).clamp(0, 63)
        mn = torch.round(m / dm[..., None]).clamp(0, 63)
        es, em = (sc * d[..., None])[..., None], (mn * dm[..., None])[..., None]
        q = torch.round((b + em) / es).clamp(0, 15).to(torch.uint8)
        q = q.reshape(rows, -1, 4, 2, 32)
        qs = (q[..., 0, :] | (q[..., 1, :] << 4)).reshape(rows, -1, 128)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        p = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6),
                       mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                       (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
        return torch.cat([_f16(d), _f16(dm), p, qs], -1).reshape(rows, -1)
    b = x.reshape(rows, -1, 16, 16)
    at = b.abs().argmax(-1, keepdim=True)
    s = -b.gather(-1, at)[..., 0] / 32
    top = s.gather(-1, s.abs().argmax(-1, keepdim=True))[..., 0]
    d = -top / 128
    sc = torch.round(s / d[..., None]).clamp(-128, 127)
    es = sc * d[..., None]
    es = torch.where(es == 0, torch.full_like(es, 1e30), es)
    u = (torch.round(b / es[..., None]).clamp(-32, 31) + 32).to(torch.uint8)
    u = u.reshape(rows, -1, 2, 4, 32)  # c, g, l
    low, high = u & 15, u >> 4
    ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4),
                    low[..., 1, :] | (low[..., 3, :] << 4)], -1).reshape(rows, -1, 128)
    qh = (high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) |
          (high[..., 3, :] << 6)).reshape(rows, -1, 64)
    return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _f16(d)], -1).reshape(rows, -1)


def _matrix(g, wtype, rows, cols):
    """A random matrix in blocks on the GPU, about 2^27 values at a time."""
    step = max(1, (1 << 27) // cols)
    return torch.cat([_pack(torch.randn(min(step, rows - r), cols, generator=g, device="cuda")
                            .mul_(0.02), wtype) for r in range(0, rows, step)])


def _moe_weights(g, shape, gate, down):
    E, EI, NE, _, _ = SHAPES[shape]
    return dict(router=torch.randn(NE, E, generator=g, device="cuda").mul_(0.02),
                gate=_matrix(g, gate, NE * EI, E).reshape(NE, -1),
                up=_matrix(g, gate, NE * EI, E).reshape(NE, -1),
                down=_matrix(g, down, NE * E, EI).reshape(NE, -1))


def _layer_inputs(case, seed):
    g = _gen(seed)
    E, _, NE, _, _ = SHAPES[case["shape"]]
    w = _moe_weights(g, case["shape"], case["gate"], case["down"])
    x = torch.randn(case["T"], E, generator=g, device="cuda")
    bias = torch.randn(NE, generator=g, device="cuda") if case["bias"] else None
    return w, x, bias


def _dense_inputs(case, seed):
    g = _gen(seed)
    w = _matrix(g, case["wtype"], case["N"], case["K"])
    x = torch.randn(case["T"], case["K"], generator=g, device="cuda")
    add = None
    if case["add"] != "none":
        shape = (case["N"],) if case["add"] == "row" else (case["T"], case["N"])
        add = torch.randn(*shape, generator=g, device="cuda")
    return w, x, add


def _model_inputs(case, seed):
    """The model's tensors on the GPU (hiplm's dict layout) and its ids."""
    g = _gen(seed)
    E, EI, NE, K, _ = SHAPES[case["shape"]]
    H, KH, V, theta = MODELS[case["shape"]]
    wt = case["wtype"]
    olmoe = case["shape"].startswith("olmoe")

    def norm(n):
        return 1 + 0.1 * torch.randn(n, generator=g, device="cuda")
    md = dict(arch="olmoe" if olmoe else "mixtral", layers=case["layers"], E=E, H=H, KH=KH, V=V,
              NE=NE, K=K, EI=EI, wtype=TYPES[wt], theta=theta, window=0,
              token_embd=_matrix(g, wt, V, E), output=_matrix(g, wt, V, E), output_norm=norm(E),
              blk=[])
    for _ in range(case["layers"]):
        b = _moe_weights(g, case["shape"], wt, wt)
        b.update(q=_matrix(g, wt, H * 128, E), k=_matrix(g, wt, KH * 128, E),
                 v=_matrix(g, wt, KH * 128, E), o=_matrix(g, wt, E, H * 128),
                 attn_norm=norm(E), ffn_norm=norm(E))
        if olmoe:
            b.update(q_norm=norm(E), k_norm=norm(E))
        md["blk"].append(b)
    n = case["prompt"] + case["steps"]
    ids = torch.randint(0, V, (case["seqs"], n), generator=g, device="cuda")
    return md, ids


def _host(v):
    return np.ascontiguousarray(v.cpu().numpy())


def _moe_type(gate, down):
    return TYPES[gate] | (TYPES[down] << 8 if down != gate else 0)


def prepare(case, seed):
    if case["kind"] == "layer":
        w, x, bias = _layer_inputs(case, seed)
        E, EI, NE, K, renorm = SHAPES[case["shape"]]
        L = hipmoe.MoeLayer(_host(w["router"]), _host(w["gate"]), _host(w["up"]),
                            _host(w["down"]), _moe_type(case["gate"], case["down"]), E, EI, NE,
                            K, renorm)
        if case["host"]:
            return dict(case=case, layer=L, x=_host(x), bias=None if bias is None else _host(bias))
        T = case["T"]
        st = dict(case=case, layer=L, x=x, bias=bias, out=torch.empty(T, E, device="cuda"),
                  ids=torch.empty(T, K, dtype=torch.int32, device="cuda"),
                  w=torch.empty(T, K, device="cuda"))
        torch.cuda.synchronize()
        return st
    if case["kind"] == "dense":
        w, x, add = _dense_inputs(case, seed)
        m = hipmoe.QMat(_host(w).reshape(-1), TYPES[case["wtype"]], case["N"], case["K"])
        st = dict(case=case, mat=m, x=x, add=add,
                  out=torch.empty(case["T"], case["N"], device="cuda"))
        torch.cuda.synchronize()
        return st
    md, ids = _model_inputs(case, seed)
    md = {k: _host(v) if torch.is_tensor(v) else v for k, v in md.items()}
    md["blk"] = [{k: _host(v) for k, v in b.items()} for b in md["blk"]]
    M = hiplm.LmModel(md, CONTEXT)
    st = dict(case=case, model=M, ids=_host(ids).astype(np.int32))
    if case["seqs"] > 1:
        st["batch"] = hiplm.LmBatch(M, case["seqs"])
    return st


def run(state):
    case = state["case"]
    if case["kind"] == "layer":
        L = state["layer"]
        if case["host"]:
            return L.ffn(state["x"], state["bias"])
        bias = state["bias"]
        L.ffn_dev(state["x"].data_ptr(), state["out"].data_ptr(), case["T"],
                  None if bias is None else bias.data_ptr(), state["ids"].data_ptr(),
                  state["w"].data_ptr())
        return state["out"], state["ids"], state["w"]
    if case["kind"] == "dense":
        add = state["add"]
        state["mat"].mul_dev(state["x"].data_ptr(), case["T"], state["out"].data_ptr(),
                             None if add is None else add.data_ptr(),
                             0 if add is None else add.numel())
        return state["out"]
    ids, n = state["ids"], case["prompt"]
    logits = []
    if case["seqs"] > 1:  # the prompts, then given tokens in lockstep
        B = state["batch"]
        B.reset()
        B.generate(ids[:, :n], 0)
        for s in range(case["steps"]):
            logits.append(B.decode(ids[:, n + s])[1])
        return logits
    M = state["model"]
    M.reset()
    logits.append(M.prefill(ids[0, :n])[1])
    for s in range(case["steps"]):
        logits.append(M.decode(int(ids[0, n + s]))[1])
    return logits


# --------------------------------------------------------------------------
# what a pass cannot do without, and the tolerances
# --------------------------------------------------------------------------

def _moe_work(shape, gate, down, T):
    E, EI, NE, K, _ = SHAPES[shape]
    touched = NE * (1 - (1 - K / NE) ** T)
    per = 2 * EI * hipmoe.row_bytes(TYPES[gate], E) + E * hipmoe.row_bytes(TYPES[down], EI)
    return (touched * per + NE * E * 4 + 2 * T * E * 4 + 2 * T * K * 4,
            T * K * 6 * E * EI + 2 * T * NE * E)


def work(case):
    if case["kind"] == "layer":
        b, f = _moe_work(case["shape"], case["gate"], case["down"], case["T"])
        return {"bytes": b, "flops": f}
    if case["kind"] == "dense":
        N, K, T = case["N"], case["K"], case["T"]
        add = {"none": 0, "row": N, "full": T * N}[case["add"]]
        return {"bytes": N * hipmoe.row_bytes(TYPES[case["wtype"]], K) + 4 * (T * K + T * N + add),
                "flops": 2 * T * N * K}
    E = SHAPES[case["shape"]][0]
    H, KH, V, _ = MODELS[case["shape"]]
    wt, S, L = case["wtype"], case["seqs"], case["layers"]
    row = hipmoe.row_bytes(TYPES[wt], E)
    attn = 2 * (H + KH) * 128 * row  # q, k, v, o (H * 128 = E)
    nbytes = flops = 0

    def forward(rows, past):
        """rows new rows a sequence after `past` cached ones; the head on one row each"""
        mb, mf = _moe_work(case["shape"], wt, wt, S * rows)
        keys = rows * past + rows * (rows + 1) / 2
        kv = 2 * S * KH * 128 * 4 * (past + 2 * rows)
        return (L * (mb + attn + kv) + V * row + S * (rows * row + V * 4),
                L * (mf + 2 * S * rows * 2 * (H + KH) * 128 * E + 4 * S * H * 128 * keys) +
                2 * S * V * E)
    for rows, past in [(case["prompt"], 0)] + [(1, case["prompt"] + s)
                                               for s in range(case["steps"])]:
        b, f = forward(rows, past)
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def _grouped(shape, gate, T):
    """Whether the layer's products take f16 operands (the documented grouped path)."""
    _, _, NE, K, _ = SHAPES[shape]
    return gate not in KQUANT and 4 * T * K > 3 * NE


def tolerance(case):
    if case["kind"] == "layer":
        if case["gate"] in KQUANT:  # equal to the reference's bit for bit by contract
            return "exact"
        if _grouped(case["shape"], case["gate"], case["T"]):  # f16 operands: 5e-4 seen
            return {"rel": 2e-3}
        return {"rel": 4e-6}  # fp32 dots: 1e-6 seen
    if case["kind"] == "dense":
        return "exact" if case["wtype"] in KQUANT else {"rel": 4e-6}
    return {"rel": 2e-3}  # a layer on f16 operands: 5e-4 seen


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------

def _d16(b):
    return b.contiguous().view(torch.float16).double()


def _unpack(b, wtype):
    """Blocks uint8 [rows, bytes] -> float64 [rows, cols]"""
    rows = b.shape[0]
    if wtype == "q8_0":
        b = b.reshape(rows, -1, 34)
        return (_d16(b[..., :2]) * b[..., 2:].view(torch.int8).double()).reshape(rows, -1)
    if wtype == "q4_0":
        b = b.reshape(rows, -1, 18)
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        return (_d16(b[..., :2]) * q).reshape(rows, -1)
    if wtype == "q4_k":
        b = b.reshape(rows, -1, 144)
        p = b[..., 4:16]
        sc = torch.cat([p[..., :4] & 63, (p[..., 8:] & 15) | ((p[..., :4] >> 6) << 4)], -1)
        mn = torch.cat([p[..., 4:8] & 63, (p[..., 8:] >> 4) | ((p[..., 4:8] >> 6) << 4)], -1)
        q = b[..., 16:].reshape(rows, -1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 3).reshape(rows, -1, 8, 32).double()
        s, m = _d16(b[..., :2]) * sc.double(), _d16(b[..., 2:4]) * mn.double()
        return (s[..., None] * q - m[..., None]).reshape(rows, -1)
    b = b.reshape(rows, -1, 210)
    ql = b[..., :128].reshape(rows, -1, 2, 2, 32)
    qh = b[..., 128:192].reshape(rows, -1, 2, 32)
    low = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4,
                       ql[..., 1, :] >> 4], 3)
    high = torch.stack([(qh >> (2 * g)) & 3 for g in range(4)], 3)
    q = (low | (high << 4)).reshape(rows, -1, 16, 16).double() - 32
    s = _d16(b[..., 208:]) * b[..., 192:208].contiguous().view(torch.int8).double()
    return (s[..., None] * q).reshape(rows, -1)


def _q8k(x):
    """Rows of fp32 values as their Q8_K encoding represents them, in float64."""
    b = x.float().reshape(x.shape[0], -1, 256)
    top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    inv = torch.where(top == 0, torch.zeros_like(top), -127.0 / top)
    v = (inv * b).double()
    q = (torch.floor(v.abs() + 0.5) * v.sign()).clamp_max(127)
    d = torch.where(inv == 0, torch.zeros_like(inv), 1.0 / inv).double()
    return (d * q).reshape(x.shape[0], -1)


def _route64(logits, k, renorm):
    """softmax and the reference's insertion top-k, which starts from k
    copies of expert 0: the experts ranked before expert 0 take slots, the
    others all stay expert 0's (as long as expert 0 is among the k)."""
    p = torch.softmax(logits, -1)
    rows, n = p.shape
    order = torch.sort(p, dim=-1, descending=True, stable=True).indices
    rank = torch.empty_like(order).scatter_(1, order, torch.arange(n, device=p.device)
                                            .expand(rows, n).contiguous())
    r0 = rank[:, :1]
    slot = torch.arange(k - 1, -1, -1, device=p.device)[None]  # rank held by slot s
    ids = torch.where(slot < r0, order[:, :k].flip(1), torch.zeros_like(order[:, :k]))
    w = p.gather(1, ids)
    return ids, w / w.sum(-1, keepdim=True) if renorm else w


def _moe64(x, w, shape, gate, down, bias):
    _, _, NE, K, renorm = SHAPES[shape]
    x = x.double()
    logits = x @ w["router"].double().T
    ids, wt = _route64(logits if bias is None else logits + bias.double(), K, renorm)
    xq = _q8k(x) if gate in KQUANT else x
    out = torch.zeros_like(x)
    for e in range(NE):
        t, s = torch.nonzero(ids == e, as_tuple=True)
        if t.numel() == 0:
            continue
        rows = xq[t]
        g = rows @ _unpack_rows(w["gate"][e], gate, x.shape[1]).T
        u = rows @ _unpack_rows(w["up"][e], gate, x.shape[1]).T
        h = g / (1 + torch.exp(-g)) * u
        out.index_add_(0, t, (h @ _unpack_rows(w["down"][e], down, h.shape[1]).T) *
                       wt[t, s][:, None])
    return out, wt


def _unpack_rows(b, wtype, cols):
    return _unpack(b.reshape(-1, hipmoe.row_bytes(TYPES[wtype], cols)), wtype)


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double()


def _rope64(x, theta):
    """x [S, n, heads, 128]: consecutive pairs turned by position * frequency."""
    n = x.shape[1]
    f = theta ** (-torch.arange(0, 128, 2, device=x.device, dtype=torch.float64) / 128)
    a = torch.arange(n, device=x.device, dtype=torch.float64)[:, None] * f
    c, s = torch.cos(a)[None, :, None], torch.sin(a)[None, :, None]
    y = torch.empty_like(x)
    y[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * s
    y[..., 1::2] = x[..., 0::2] * s + x[..., 1::2] * c
    return y


def _model64(case, md, ids):
    """Logits of the rows from the prompt's last on (a lockstep batch: after it)."""
    E = SHAPES[case["shape"]][0]
    H, KH, V, theta = MODELS[case["shape"]]
    wt, (S, n) = case["wtype"], ids.shape
    first = case["prompt"] - (1 if S == 1 else 0)
    mask = torch.ones(n, n, device="cuda", dtype=torch.bool).triu(1)
    h = _unpack(md["token_embd"][ids.reshape(-1)], wt).reshape(S, n, E)
    for b in md["blk"]:
        x = _rms64(h, b["attn_norm"])
        q, k, v = (x @ _unpack(b[c], wt).T for c in "qkv")
        if "q_norm" in b:
            q, k = _rms64(q, b["q_norm"]), _rms64(k, b["k_norm"])
        q = _rope64(q.reshape(S, n, H, 128), theta)
        k = _rope64(k.reshape(S, n, KH, 128), theta).repeat_interleave(H // KH, 2)
        v = v.reshape(S, n, KH, 128).repeat_interleave(H // KH, 2)
        o = torch.empty_like(q)
        for s in range(S):
            for i in range(H):
                p = (q[s, :, i] @ k[s, :, i].T.contiguous()) / math.sqrt(128)
                o[s, :, i] = torch.softmax(p.masked_fill(mask, -math.inf), -1) @ v[s, :, i]
        h = h + o.reshape(S, n, H * 128) @ _unpack(b["o"], wt).T
        y, _ = _moe64(_rms64(h, b["ffn_norm"]).reshape(S * n, E), b, case["shape"], wt, wt, None)
        h = h + y.reshape(S, n, E)
    head = _unpack(md["output"], wt)
    return [_rms64(h[:, i] if S > 1 else h[0, i], md["output_norm"]) @ head.T
            for i in range(first, n)]


def exact(case, seed):
    """run()'s outputs in 64 bits (expert ids, whole numbers, left out)."""
    if case["kind"] == "layer":
        w, x, bias = _layer_inputs(case, seed)
        out, wt = _moe64(x, w, case["shape"], case["gate"], case["down"], bias)
        return out, None, wt
    if case["kind"] == "dense":
        w, x, add = _dense_inputs(case, seed)
        out = (_q8k(x) if case["wtype"] in KQUANT else x.double()) @ _unpack(w, case["wtype"]).T
        return out if add is None else out + add.double()
    return _model64(case, *_model_inputs(case, seed))
