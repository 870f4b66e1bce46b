"""The calls that are timed when this library's speed is compared.

Every case is one call of the MoE expert path as a serving program makes it:

* ``logits``: a routed layer with everything in device memory, router logits
  in, layer output out (``moe_forward_logits_dev``: softmax top-k router);
* ``ids``: the reference's own router (sigmoid scores with a selection bias)
  followed by the layer over its ids (``route_sigmoid_topk_dev`` then
  ``moe_forward_dev``);
* ``host``: the reference's host-buffer call (``expert_group_reduce``): one
  row of x per (token, expert) in host memory, the combined output back.

A case names the layer (E experts, hidden D, intermediate I), the batch (S
tokens, top k), the weight format (QT format code and group size), the
activation scale group (0: per row, the reference's mode; 32: per 32 elements)
and how the router logits are drawn (``normal``, or ``zipf`` for skewed expert
popularity). Weights, scales, tokens and logits have the distributions of
``peregrine_amd/synth.py``; they are made on the GPU.
"""
import math

import numpy as np
import torch

from peregrine_amd import hip, qt

DEV = "cuda:0"
ROUTED_SCALE = 2.5   # the sigmoid router's factor on its renormalised weights


def listed():
    i4, i4g, i8, i8g = qt.FMT_I4, qt.FMT_I4G, qt.FMT_I8, qt.FMT_I8G
    mid = dict(E=160, D=5120, I=1536, k=8)    # the 160-expert layer of bench.py
    big = dict(E=256, D=6144, I=2048, k=8)    # its 256-expert layer
    return [
        # the smallest call: one resident expert, one token (a shared expert, or a lane that holds one of them)
        dict(name="one_expert_1tok", call="logits", E=1, D=5120, I=1536, k=1, S=1, fmt=i4g, gs=32, ga=32, route="normal"),
        # decode of one stream, grouped scales
        dict(name="decode_1tok", call="logits", S=1, fmt=i4g, gs=32, ga=32, route="normal", **mid),
        # decode of one stream as the reference runs it: its router, per-row int4, per-row activations
        dict(name="decode_1tok_rowscale", call="ids", S=1, fmt=i4, gs=0, ga=0, route="normal", **mid),
        # a handful of streams decoded together
        dict(name="decode_5tok", call="logits", S=5, fmt=i4g, gs=32, ga=32, route="normal", **mid),
        # batched decode with skewed expert popularity (groups of 1 to about 40 rows)
        dict(name="decode_64tok", call="logits", S=64, fmt=i4g, gs=32, ga=32, route="zipf", **mid),
        # a long prompt, grouped scales
        dict(name="prefill_2048tok", call="logits", S=2048, fmt=i4g, gs=32, ga=32, route="zipf", **mid),
        # a prompt of odd length as the reference runs it (per-row int4, per-row activations)
        dict(name="prefill_1777tok_rowscale", call="ids", S=1777, fmt=i4, gs=0, ga=0, route="zipf", **mid),
        # the large layer, every expert read, int4 and int8 weights
        dict(name="large_512tok_int4", call="logits", S=512, fmt=i4g, gs=32, ga=32, route="normal", **big),
        dict(name="large_512tok_int8", call="logits", S=512, fmt=i8g, gs=32, ga=32, route="normal", **big),
        # the reference's own call at decode: host rows in, host row out
        dict(name="host_1tok_rowscale", call="host", S=1, fmt=i4, gs=0, ga=0, route="normal", **mid),
        # the same call over a small batch with coarse groups
        dict(name="host_24tok_g128", call="host", S=24, fmt=i4g, gs=128, ga=0, route="zipf", **mid),
        # a small layer whose sizes fit no tile, int8 per row
        dict(name="small_ragged_300tok_int8", call="logits", E=60, D=1000, I=712, k=6, S=300, fmt=i8, gs=0, ga=0,
             route="zipf"),
    ]


FORMATS = [(qt.FMT_I4, 0), (qt.FMT_I4G, 32), (qt.FMT_I4G, 64), (qt.FMT_I4G, 128), (qt.FMT_I8, 0), (qt.FMT_I8G, 32)]


def draw(rng):
    def log_uniform(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def width(lo, hi):   # layer widths: usually a multiple of 64, sometimes anything
        v = log_uniform(lo, hi)
        return max(64, v // 64 * 64) if rng.random() < 0.6 else v

    call = rng.choice(["logits", "logits", "logits", "ids", "host"])
    E = log_uniform(8, 256)
    fmt, gs = rng.choice(FORMATS)
    c = dict(call=call, E=E, D=width(512, 6144), I=width(256, 2048), k=rng.randint(1, min(8, E)),
             S=log_uniform(1, 64 if call == "host" else 2048), fmt=fmt, gs=gs, ga=rng.choice([0, 32]),
             route=rng.choice(["normal", "zipf"]))
    # no more arithmetic than the longest listed prompt
    c["S"] = max(1, min(c["S"], int(2048 * 8 * 5120 * 1536 / (c["k"] * c["D"] * c["I"]))))
    return c


# ---------------------------------------------------------------- inputs

def _gen(seed, part):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1_000_003 + part) & 0x7FFFFFFFFFFFFFFF)
    return g


def _expert_raw(case, seed, e):
    """QT bytes and scales of one expert's gate, up and down, in device memory."""
    g = _gen(seed, 16 + e)
    out = []
    for o, i in ((case["I"], case["D"]), (case["I"], case["D"]), (case["D"], case["I"])):
        if case["fmt"] in (qt.FMT_I4, qt.FMT_I4G):
            q = torch.randint(0, 256, (o, (i + 1) // 2), dtype=torch.uint8, device=DEV, generator=g)
        else:
            q = torch.randint(-127, 128, (o, i), dtype=torch.int8, device=DEV, generator=g)
        ng = -(-i // case["gs"]) if case["gs"] else 1
        sc = torch.empty((o, ng), device=DEV).log_normal_(math.log(0.01), 0.5, generator=g)
        out.append((q, sc, o, i))
    return out


def _tokens(case, seed):
    return torch.randn((case["S"], case["D"]), device=DEV, generator=_gen(seed, 1))


def _logits(case, seed):
    S, E = case["S"], case["E"]
    g = _gen(seed, 2)
    if case["route"] == "normal":
        return torch.randn((S, E), device=DEV, generator=g)
    p = 1.0 / torch.arange(1, E + 1, device=DEV, dtype=torch.float64) ** 1.1
    p = p[torch.randperm(E, device=DEV, generator=g)]
    u = torch.rand((S, E), device=DEV, generator=g, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    return (torch.log(p / p.sum()) - torch.log(-torch.log(u))).float()


def _bias(case, seed):
    return 0.01 * torch.randn((case["E"],), device=DEV, generator=_gen(seed, 3))


def _softmax_route(logits, k):
    v, ids = torch.sort(logits, dim=1, descending=True, stable=True)
    return ids[:, :k], torch.softmax(v[:, :k].double(), dim=1)


def _sigmoid_route(logits, bias, k):
    s = torch.sigmoid(logits.double())
    ids = torch.sort(s + bias.double(), dim=1, descending=True, stable=True)[1][:, :k]
    w = torch.gather(s, 1, ids)
    return ids, w / (w.sum(1, keepdim=True) + 1e-20) * ROUTED_SCALE


def _host_rows(case, seed):
    """The host call's grouping: experts in first-seen order, their rows in
    token order, the token and the weight of each row."""
    ids, w = _softmax_route(_logits(case, seed), case["k"])
    ids, w = ids.cpu().numpy(), w.float().cpu().numpy()
    order = list(dict.fromkeys(ids.reshape(-1).tolist()))
    tok, slot, rows = [], [], []
    for e in order:
        t, j = np.nonzero(ids == e)
        tok.append(t)
        slot.append(j)
        rows.append(len(t))
    tok, slot = np.concatenate(tok), np.concatenate(slot)
    return order, rows, tok, w[tok, slot].astype(np.float32)


_ready = False


def _init():
    global _ready
    if not _ready:
        torch.cuda.init()
        if hip.init([0]) != 1:
            raise RuntimeError("hip.init failed")
        _ready = True


def _upload(case, seed, which):
    experts = []
    for e in which:
        raw = _expert_raw(case, seed, e)
        torch.cuda.synchronize()
        t = [hip.upload_tensor_dev(0, q.data_ptr(), sc.data_ptr(), case["fmt"], i, o, case["gs"]) for q, sc, o, i in raw]
        experts.append(hip.GpuExpert(t[0], t[1], t[2], case["D"], case["I"]))
    return experts


def prepare(case, seed):
    _init()
    S, D, E, k = case["S"], case["D"], case["E"], case["k"]
    st = dict(case=case)
    if case["call"] == "host":
        order, rows, tok, rw = _host_rows(case, seed)
        st["experts"] = _upload(case, seed, order)
        st["rows"] = rows
        st["x"] = np.ascontiguousarray(_tokens(case, seed).cpu().numpy()[tok])
        st["rw"] = rw
        st["layout"] = hip.ReduceLayout.build(tok, S)
        hip.set_act_group(case["ga"])
        return st
    st["set"] = hip.ExpertSet(_upload(case, seed, range(E)))
    st["x"], st["logits"] = _tokens(case, seed), _logits(case, seed)
    if case["call"] == "ids":
        st["bias"] = _bias(case, seed)
    st["ids"] = torch.zeros((S, k), dtype=torch.int32, device=DEV)
    st["w"] = torch.zeros((S, k), device=DEV)
    st["out"] = torch.zeros((S, D), device=DEV)
    torch.cuda.synchronize()
    return st


def run(st):
    c = st["case"]
    if c["call"] == "host":
        return {"out": hip.expert_group_reduce(st["experts"], st["rows"], st["x"], c["D"], st["layout"], st["rw"], c["S"])}
    x, ids, w, out = st["x"].data_ptr(), st["ids"].data_ptr(), st["w"].data_ptr(), st["out"].data_ptr()
    if c["call"] == "ids":
        hip.route_sigmoid_topk_dev(0, st["logits"].data_ptr(), st["bias"].data_ptr(), c["S"], c["E"], c["k"], ids, w,
                                   routed_scale=ROUTED_SCALE)
        hip.moe_forward_dev(st["set"], x, c["S"], ids, w, c["k"], out, c["ga"])
    else:
        hip.moe_forward_logits_dev(st["set"], x, c["S"], st["logits"].data_ptr(), c["k"], ids, w, out, c["ga"])
    return {"out": st["out"], "ids": st["ids"], "weights": st["w"]}


def _distinct(case):
    """Experts that a batch is expected to touch."""
    E, S, k = case["E"], case["S"], case["k"]
    if case["route"] == "normal":
        return E * (1.0 - (1.0 - k / E) ** S)
    p = 1.0 / np.arange(1, E + 1) ** 1.1
    p /= p.sum()
    return min(float(E), max(float(k), float(np.sum(1.0 - (1.0 - p) ** (S * k)))))


def work(case):
    D, I, S, k = case["D"], case["I"], case["S"], case["k"]
    wb = 0.5 if case["fmt"] in (qt.FMT_I4, qt.FMT_I4G) else 1.0
    weights = 3 * D * I * wb
    if case["gs"]:
        scales = 4 * (2 * I * -(-D // case["gs"]) + D * -(-I // case["gs"]))
    else:
        scales = 4 * (2 * I + D)
    rows_in = S * k if case["call"] == "host" else S
    moved = _distinct(case) * (weights + scales) + 4 * (rows_in + S) * D + 4 * S * case["E"] + 8 * S * k
    return {"bytes": float(moved), "flops": float(2 * 3 * S * k * D * I)}


def tolerance(case):
    # The sums are exact integers and 32-bit floats, but the intermediate row
    # is quantised to 8 bits again: a sum in another order moves a few of its
    # codes by one. Measured against 64 bits: 2e-7 to 3e-7 where no code moves,
    # 2e-4 to 4.3e-4 where some do.
    return {"rel": 2e-3, "max": 2e-2, "differ": 1e-3}


# ---------------------------------------------------------------- 64 bits

def _quant(x, ga):
    """int8 codes times their scale, in 64 bits: one scale per row, or per ga elements."""
    n, K = x.shape
    if ga:
        pad = -K % ga
        v = torch.nn.functional.pad(x, (0, pad)).reshape(n, -1, ga)
    else:
        v = x.reshape(n, 1, K)
    s = (v.abs().amax(dim=2, keepdim=True) / 127.0).clamp_min(1e-12)
    return (torch.round(v / s) * s).reshape(n, -1)[:, :K]


def _dequant(case, q, sc, i):
    if case["fmt"] in (qt.FMT_I4, qt.FMT_I4G):
        v = torch.stack((q & 15, q >> 4), dim=2).reshape(q.shape[0], -1)[:, :i].double() - 8.0
    else:
        v = q.double()
    gs = case["gs"] or i
    return v * sc.double().repeat_interleave(gs, dim=1)[:, :i]


def _expert_rows(case, seed, e, x):
    (g, u, d) = [_dequant(case, q, sc, i) for q, sc, _, i in _expert_raw(case, seed, e)]
    a, b = x @ g.T, x @ u.T
    return _quant(a / (1.0 + torch.exp(-a)) * b, case["ga"]) @ d.T


def exact(case, seed):
    torch.cuda.init()
    x = _quant(_tokens(case, seed).double(), case["ga"])
    out = torch.zeros_like(x)
    if case["call"] == "host":
        order, rows, tok, rw = _host_rows(case, seed)
        at = 0
        for e, n in zip(order, rows):
            t = torch.from_numpy(tok[at:at + n]).to(DEV)
            y = _expert_rows(case, seed, e, x[t]) * torch.from_numpy(rw[at:at + n]).to(DEV).double()[:, None]
            out.index_add_(0, t, y)
            at += n
        return {"out": out.cpu().numpy()}
    logits = _logits(case, seed)
    if case["call"] == "ids":
        ids, w = _sigmoid_route(logits, _bias(case, seed), case["k"])
    else:
        ids, w = _softmax_route(logits, case["k"])
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        out.index_add_(0, t, _expert_rows(case, seed, e, x[t]) * w[t, j][:, None])
    return {"out": out, "ids": ids.to(torch.int32), "weights": w}
