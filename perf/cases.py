"""The work this framework's users have it do, as measured cases.

The framework is the int8 product path of a FastConformer TDT speech
recognizer: quantize + int8 product on host pointers (the drop-in backend),
the same on device pointers, the whole encoder layer, the attention's float
part, the decoder's token steps and its greedy search. A frame is 80 ms of
audio, so 384 frames are the longest segment the recognizer cuts long audio
into (30.72 s), 750 a minute, 7500 ten minutes in one piece. The model's
shapes: d_model 1024, 8 heads, feed-forward 4096, 9 depthwise taps; prediction
network and joint 640 wide, 2 LSTM layers, 1024 tokens and the blank, 5
durations. The encoder quantizes in blocks of 32 inputs (its default) or 64
(its fast mode), the joint and the decoder whole rows.

Every output is compared exactly: the path's contract is the scalar
reference's bits, so any other correct implementation of it has the same.
"""
import math
import random

import numpy as np
import torch

import libpktito_amd as pk
from libpktito_amd import synth

D_MODEL, HEADS, FF, TAPS = 1024, 8, 4096, 9
PRED, LSTMS, JOINT, VOCAB, N_DUR = 640, 2, 640, 1024, 5
DURATIONS = [0, 1, 2, 3, 4]
MAX_SYMBOLS = 10
EPS = 1e-5

# the layer's matrices, (rows, cols)
LAYER_SHAPES = {"ff1_up": (FF, D_MODEL), "ff1_down": (D_MODEL, FF), "ff2_up": (FF, D_MODEL),
                "ff2_down": (D_MODEL, FF), "q": (D_MODEL, D_MODEL), "k": (D_MODEL, D_MODEL),
                "v": (D_MODEL, D_MODEL), "pos": (D_MODEL, D_MODEL), "o": (D_MODEL, D_MODEL),
                "pw1": (2 * D_MODEL, D_MODEL), "pw2": (D_MODEL, D_MODEL)}


def listed():
    return [
        # the decoder driven from the host over a run of eight known labels (rescoring, forced alignment):
        # each a prediction and a joint, the smallest calls there are
        {"name": "token_steps_8", "kind": "tokens", "steps": 8},
        # the greedy search of the longest segment in one call
        {"name": "search_384", "kind": "search", "T": 384, "scale": 2.0},
        # a few frames against a deep matrix: weights streamed once, with the split's workspace
        {"name": "product_16_deep", "kind": "product", "M": 16, "K": 4096, "N": 1024, "qb": 0, "packed": False,
         "add": False, "bias": False, "work": True},
        # the joint's encoder half of a segment: whole rows, bias, row-major
        {"name": "joint_frames_384", "kind": "product", "M": 384, "K": 1024, "N": 640, "qb": 0, "packed": False,
         "add": False, "bias": True, "work": False},
        # fast mode's pointwise product of an odd segment, packed activations
        {"name": "product_333_qb64", "kind": "product", "M": 333, "K": 1024, "N": 2048, "qb": 64, "packed": True,
         "add": False, "bias": False, "work": False},
        # eight segments of 12 to 60 s against one matrix in one launch
        {"name": "grouped_8_segments", "kind": "grouped", "segments": 8, "lo": 150, "hi": 750, "lengths": 2024,
         "K": 1024, "N": 4096},
        # the host-pointer drop-in the recognizer's backend table calls: feed-forward up at the longest segment
        {"name": "dropin_384", "kind": "dropin", "M": 384, "K": 1024, "N": 4096, "qb": 32},
        # whole encoder layers: a short utterance in fast mode, the longest segment, a minute
        {"name": "layer_137_qb64", "kind": "layer", "T": 137, "qb": 64},
        {"name": "layer_384_qb32", "kind": "layer", "T": 384, "qb": 32},
        {"name": "layer_750_qb32", "kind": "layer", "T": 750, "qb": 32},
        # the attention alone over two minutes of audio, an odd length
        {"name": "attention_1499", "kind": "attention", "T": 1499},
        # ten minutes in one piece: a layer's quantizes and products over whole rows, the headline's chain
        {"name": "chain_7500", "kind": "chain", "M": 7500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tokens", "search", "product", "product", "product", "grouped", "dropin", "layer", "layer",
                       "layer", "attention", "chain"])
    if kind == "tokens":
        return {"kind": kind, "steps": 2 * rng.randint(1, 16)}
    if kind == "search":
        return {"kind": kind, "T": _log(rng, 20, 384), "scale": round(rng.uniform(1.5, 3.0), 2)}
    if kind == "product":
        K, N = rng.choice([(1024, 1024), (1024, 4096), (4096, 1024), (1024, 2048), (1024, 640), (640, 1040)])
        qb = rng.choice([0, 32, 64])
        return {"kind": kind, "M": _log(rng, 1, 3000), "K": K, "N": N, "qb": qb, "packed": rng.random() < 0.5,
                "add": rng.random() < 0.3, "bias": rng.random() < 0.3, "work": rng.random() < 0.3}
    if kind == "grouped":
        lo = _log(rng, 16, 300)
        K, N = rng.choice([(1024, 1024), (1024, 4096), (1024, 2048), (4096, 1024)])
        return {"kind": kind, "segments": rng.randint(2, 16), "lo": lo, "hi": lo + rng.randint(1, 450),
                "lengths": rng.randrange(1 << 30), "K": K, "N": N}
    if kind == "dropin":
        K, N = rng.choice([(1024, 1024), (1024, 4096), (4096, 1024), (1024, 640)])
        return {"kind": kind, "M": _log(rng, 1, 750), "K": K, "N": N, "qb": rng.choice([0, 32, 64])}
    if kind == "layer":
        return {"kind": kind, "T": _log(rng, 12, 1500), "qb": rng.choice([32, 64])}
    if kind == "attention":
        return {"kind": kind, "T": _log(rng, 12, 2000)}
    return {"kind": kind, "M": _log(rng, 400, 7500)}


# ---------------------------------------------------------------- inputs --

def _segment_lengths(case):
    r = random.Random(case["lengths"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["segments"])]


def _normal(g, *shape):
    return g.standard_normal(shape, dtype=np.float32)


def _matrix(g, rows, cols, gain=1.0):
    """int8 uniform in [-127, 127], row-major, and its row scales: small enough that a product of inputs of
    order 1 has outputs of order 1."""
    w = g.integers(-127, 128, size=(rows, cols), dtype=np.int8)
    s = (g.uniform(0.5, 1.5, rows) * (gain / (73.0 * math.sqrt(cols)))).astype(np.float32)
    return w, s


def _inputs(case, seed):
    """The case's inputs as host arrays, from the seed alone: matrices row-major."""
    g = np.random.Generator(np.random.PCG64(seed))
    kind = case["kind"]
    if kind in ("product", "dropin"):
        M, K, N = case["M"], case["K"], case["N"]
        return {"x": _normal(g, M, K), "w": _matrix(g, N, K),
                "bias": _normal(g, N) if case.get("bias") else None,
                "old": _normal(g, M, N) if case.get("add") else None}
    if kind == "grouped":
        return {"x": [_normal(g, t, case["K"]) for t in _segment_lengths(case)],
                "w": _matrix(g, case["N"], case["K"])}
    if kind == "attention":
        T = case["T"]
        return {"q": _normal(g, T, D_MODEL), "k": _normal(g, T, D_MODEL), "v": _normal(g, T, D_MODEL),
                "p": _normal(g, 2 * T - 1, D_MODEL), "u": 0.1 * _normal(g, D_MODEL),
                "b": 0.1 * _normal(g, D_MODEL)}
    if kind in ("layer", "chain"):
        T = case["T"] if kind == "layer" else case["M"]
        i = {"x": _normal(g, T, D_MODEL), "ape": _normal(g, 2 * T - 1, D_MODEL)}
        for n, (rows, cols) in LAYER_SHAPES.items():
            i[n] = _matrix(g, rows, cols, 0.5 if n.endswith("down") else 1.0)
        if kind == "layer":
            for n in synth.LAYER_VECTORS:
                i[n] = ((1.0 if n.endswith("nw") else 0.0) + 0.1 * _normal(g, D_MODEL)).astype(np.float32)
            i["bias_u"], i["bias_v"] = 0.1 * _normal(g, D_MODEL), 0.1 * _normal(g, D_MODEL)
            i["dw"], i["dw_b"] = 0.3 * _normal(g, D_MODEL, TAPS), 0.1 * _normal(g, D_MODEL)
        return i
    n_out = VOCAB + 1 + N_DUR
    n_pad = (n_out + 15) // 16 * 16
    i = {"embed": 0.5 * _normal(g, VOCAB + 1, PRED), "jpred": _matrix(g, JOINT, PRED),
         "jpred_b": 0.1 * _normal(g, JOINT), "jout": _matrix(g, n_pad, JOINT), "jout_b": 0.1 * _normal(g, n_pad)}
    i["jout"][0][n_out:] = 0
    i["jout_b"][n_out:] = 0
    # speech: about four tokens a second, few frames with two of them
    i["jout_b"][VOCAB] += 4.0
    i["jout_b"][VOCAB + 1:n_out] += np.array([-4.0, 0.0, 0.5, 0.5, 0.5], dtype=np.float32)
    for l in range(LSTMS):
        i[f"wx{l}"], i[f"wh{l}"] = _matrix(g, 4 * PRED, PRED), _matrix(g, 4 * PRED, PRED)
        i[f"b{l}"] = 0.1 * _normal(g, 4 * PRED)
    frames = case["T"] if kind == "search" else case["steps"]
    i["f"] = np.float32(case.get("scale", 2.0)) * _normal(g, frames, JOINT)
    i["h"], i["c"] = np.tanh(_normal(g, LSTMS, PRED)), _normal(g, LSTMS, PRED)
    i["labels"] = [int(v) for v in g.integers(0, VOCAB, size=case.get("steps", 1))]
    return i


class _State(dict):
    """What a program holds between calls; its uploaded matrices are released with it."""

    def __del__(self):
        for m in self.get("release", []):
            m.release()


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda() if a is not None else None


def _upload(ws):
    w, s = ws
    return pk.Q8Matrix(synth.pack_q8(w), s)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    pk.init()
    i = _inputs(case, seed)
    kind = case["kind"]
    s = _State(case=case)
    if kind == "product":
        M, K, N = case["M"], case["K"], case["N"]
        qb = case["qb"] or K
        s["m"] = _upload(i["w"])
        s["release"] = [s["m"]]
        s.update(x=_dev(i["x"]), bias=_dev(i["bias"]), old=_dev(i["old"]), out=_empty(M, N),
                 d=_empty(M, K // qb), q=_empty(pk.packed_bytes(K, M) if case["packed"] else M * K, dtype=torch.int8),
                 work=torch.zeros(pk.gemm_workspace(N), dtype=torch.uint8, device="cuda") if case["work"] else None)
    elif kind == "grouped":
        K, N = case["K"], case["N"]
        s["m"] = _upload(i["w"])
        s["release"] = [s["m"]]
        s["segs"] = [(_dev(x), _empty(*x.shape, dtype=torch.int8), _empty(x.shape[0]), _empty(x.shape[0], N))
                     for x in i["x"]]
    elif kind == "dropin":
        M, K, N = case["M"], case["K"], case["N"]
        qb = case["qb"] or K
        s["m"] = _upload(i["w"])
        s["release"] = [s["m"]]
        s.update(x=i["x"].reshape(-1), q=np.empty(M * K, np.int8), d=np.empty(M * (K // qb), np.float32),
                 out=np.empty(M * N, np.float32))
        s["act"] = pk.make_act(s["q"], s["d"], K, qb, M)
    elif kind == "attention":
        s.update({n: _dev(a) for n, a in i.items()})
        s["o"] = _empty(case["T"], D_MODEL)
        s["ws"] = _empty(pk.attention_workspace(case["T"], HEADS), dtype=torch.uint8)
    elif kind == "layer":
        T, qb = case["T"], case["qb"]
        w = {"D": D_MODEL, "H": HEADS, "F": FF, "K": TAPS, "eps": EPS}
        for n in LAYER_SHAPES:
            w[n], w[n + "_s"] = synth.pack_q8(i[n][0]), i[n][1]
        for n in synth.LAYER_VECTORS + ("bias_u", "bias_v", "dw", "dw_b"):
            w[n] = i[n]
        s["layer"] = pk.DeviceLayer(w, torch)
        s["release"] = [s["layer"]]
        R = 2 * T - 1
        s["ape_qp"], s["ape_d"] = _empty(pk.packed_bytes(D_MODEL, R), dtype=torch.int8), _empty(R, D_MODEL // qb)
        pk.quantize_packed_dev(None, s["ape_qp"], s["ape_d"], _dev(i["ape"]), D_MODEL, R, D_MODEL, qb=qb)
        s["ws"] = _empty(s["layer"].workspace(T, qb), dtype=torch.uint8)
        s["x0"], s["x"] = _dev(i["x"]), _empty(T, D_MODEL)
    elif kind == "chain":
        M, R = case["M"], 2 * case["M"] - 1
        s["m"] = {n: _upload(i[n]) for n in LAYER_SHAPES}
        s["release"] = list(s["m"].values())
        s["x0"], s["x"] = _dev(i["x"]), _empty(M, D_MODEL)
        s["u"], s["u2"] = _empty(M, FF), _empty(M, 2 * D_MODEL)
        s["qo"], s["ko"], s["vo"], s["po"] = (_empty(t, D_MODEL) for t in (M, M, M, R))
        s["qp"], s["qd"] = _empty(pk.packed_bytes(FF, M), dtype=torch.int8), _empty(M)
        s["ape_qp"], s["ape_d"] = _empty(pk.packed_bytes(D_MODEL, R), dtype=torch.int8), _empty(R)
        pk.quantize_packed_dev(None, s["ape_qp"], s["ape_d"], _dev(i["ape"]), D_MODEL, R, D_MODEL)
    else:
        w = {"P": PRED, "L": LSTMS, "J": JOINT, "V": VOCAB, "n_dur": N_DUR}
        for n, a in i.items():
            if isinstance(a, tuple):
                w[n], w[n + "_s"] = synth.pack_q8(a[0]), a[1]
            else:
                w[n] = a
        s["dec"] = pk.DeviceDecoder(w, torch)
        s["release"] = [s["dec"]]
        s.update(f=_dev(i["f"]), labels=i["labels"])
        if kind == "search":
            s["h"] = s["c"] = torch.zeros(LSTMS, PRED, device="cuda")
        else:
            s["h"], s["c"] = _dev(i["h"]), _dev(i["c"])
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ runs --

def _chain(s):
    """A layer's products over whole rows in the encoder's order: x += down(up(x)), q, k, v and the positions in
    one launch, x += o(v), x += pw2(pw1(x)) (the first half of pw1's columns, as after its gate), x += down(up(x));
    each product's input quantized into packed activations."""
    M, m, x, u, qp, qd = s["case"]["M"], s["m"], s["x"], s["u"], s["qp"], s["qd"]

    def quantize(a, n, xs):
        pk.quantize_packed_dev(None, qp, qd, a, n, M, xs)

    def product(out, name, n, add):
        pk.gemm_q8_packed_dev(out, out.shape[1], m[name], 0, m[name].rows, m[name].dev_scales, None, qp, qd, n, M, add)

    x.copy_(s["x0"])
    quantize(x, D_MODEL, D_MODEL)
    product(u, "ff1_up", D_MODEL, 0)
    quantize(u, FF, FF)
    product(x, "ff1_down", FF, 1)
    quantize(x, D_MODEL, D_MODEL)
    jobs = [(s[o], D_MODEL, m[n], 0, D_MODEL, m[n].dev_scales, None, qp, qd, D_MODEL, M, 0)
            for n, o in (("q", "qo"), ("k", "ko"), ("v", "vo"))]
    jobs.append((s["po"], D_MODEL, m["pos"], 0, D_MODEL, m["pos"].dev_scales, None, s["ape_qp"], s["ape_d"], D_MODEL,
                 2 * M - 1, 0))
    pk.gemm_q8_batch_dev(jobs)
    quantize(s["vo"], D_MODEL, D_MODEL)
    product(x, "o", D_MODEL, 1)
    quantize(x, D_MODEL, D_MODEL)
    product(s["u2"], "pw1", D_MODEL, 0)
    quantize(s["u2"], D_MODEL, 2 * D_MODEL)
    product(x, "pw2", D_MODEL, 1)
    quantize(x, D_MODEL, D_MODEL)
    product(u, "ff2_up", D_MODEL, 0)
    quantize(u, FF, FF)
    product(x, "ff2_down", FF, 1)
    return [x, s["qo"], s["ko"], s["vo"], s["po"]]


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "product":
        M, K, N = case["M"], case["K"], case["N"]
        qb = case["qb"] or K
        if s["old"] is not None:
            s["out"].copy_(s["old"])
        if case["packed"]:
            pk.quantize_packed_dev(None, s["q"], s["d"], s["x"], K, M, K, qb=qb)
            pk.gemm_q8_packed_dev(s["out"], N, s["m"], 0, N, s["m"].dev_scales, s["bias"], s["q"], s["d"], K, M,
                                  case["add"], qb=qb, work=s["work"])
        else:
            pk.quantize_dev(s["q"], s["d"], s["x"], K, qb, M, K)
            pk.gemm_q8_dev(s["out"], N, s["m"], 0, N, None, s["bias"], s["q"], s["d"], K, qb, M, case["add"],
                           ws_ptr=s["m"].dev_scales, work=s["work"])
        return s["out"]
    if kind == "grouped":
        K, N = case["K"], case["N"]
        for x, q, d, _ in s["segs"]:
            pk.quantize_dev(q, d, x, K, K, x.shape[0], K)
        pk.gemm_q8_grouped_dev(s["m"], 0, N, s["m"].dev_scales, None,
                               [(out, N, q, d, K, K, x.shape[0]) for x, q, d, out in s["segs"]], 0)
        return [out for _, _, _, out in s["segs"]]
    if kind == "dropin":
        pk.quantize(s["act"], s["x"], case["K"])
        pk.gemm_q8(s["out"], case["N"], s["m"].q, s["m"].s, None, case["N"], s["act"], 0)
        return [s["q"], s["d"], s["out"]]
    if kind == "attention":
        pk.attention_dev(s["o"], s["q"], s["k"], s["v"], s["p"], s["u"], s["b"], case["T"], D_MODEL, HEADS, s["ws"])
        return s["o"]
    if kind == "layer":
        s["x"].copy_(s["x0"])
        s["layer"].run(s["x"], case["T"], s["ape_qp"], s["ape_d"], case["qb"], s["ws"])
        return s["x"]
    if kind == "chain":
        return _chain(s)
    dec = s["dec"]
    dec.set_state(s["h"], s["c"])
    if kind == "tokens":
        for t, label in enumerate(s["labels"]):
            dec.predict(label)
            dec.joint(s["f"][t])
        h, c = dec.state()
        return [dec.logit, dec.tok_dur, h, c]
    # the search's tokens (a segment's buffer of them, as the call fills it), and the logits of its first step
    toks = dec.search(s["f"], case["T"], VOCAB, DURATIONS, MAX_SYMBOLS)
    dec.predict(VOCAB)
    dec.joint(s["f"][0])
    out = np.full((case["T"] * MAX_SYMBOLS, 3), -1, dtype=np.int32)
    out[:len(toks)] = np.array(toks, dtype=np.int32).reshape(-1, 3)
    return [out, dec.logit]


# ---------------------------------------------------------- work, bounds --

def _product_work(M, K, N, add=False):
    return 4 * M * K + N * K + 4 * N + 4 * M * N * (2 if add else 1), 2 * M * K * N


def _layer_products(T):
    flops = sum(2 * T * r * c for n, (r, c) in LAYER_SHAPES.items() if n != "pos")
    return flops + 2 * (2 * T - 1) * D_MODEL * D_MODEL, sum(r * c + 4 * r for r, c in LAYER_SHAPES.values())


def work(case):
    kind = case["kind"]
    if kind in ("product", "dropin"):
        b, f = _product_work(case["M"], case["K"], case["N"], case.get("add"))
    elif kind == "grouped":
        b, f = _product_work(sum(_segment_lengths(case)), case["K"], case["N"])
    elif kind == "attention":
        T = case["T"]
        b, f = 4 * D_MODEL * (4 * T + 2 * T - 1), 3 * 2 * T * T * D_MODEL
    elif kind == "layer":
        T = case["T"]
        f, wb = _layer_products(T)
        b = wb + 4 * D_MODEL * 2 * T + (2 * T - 1) * (D_MODEL + 4 * D_MODEL // case["qb"])
        f += 3 * 2 * T * T * D_MODEL + 2 * T * D_MODEL * TAPS
    elif kind == "chain":
        M = case["M"]
        f, wb = _layer_products(M)
        b = wb + 4 * D_MODEL * (M + 4 * M + 2 * M - 1) + (2 * M - 1) * (D_MODEL + 4)
    else:
        per = 2 * LSTMS * 4 * PRED * PRED + JOINT * PRED + (VOCAB + 1 + N_DUR) * JOINT
        # a search makes about one prediction and one joint every two frames
        n = case["steps"] if kind == "tokens" else max(1, case["T"] // 2)
        b, f = per + 4 * JOINT * (n if kind == "tokens" else case["T"]), 2 * per * n
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    return "exact"


# ----------------------------------------------------------- 64-bit values --

def _w64(ws, dev):
    w, s = ws
    return torch.from_numpy(w).to(dev).double() * torch.from_numpy(s).to(dev).double()[:, None]


def _quantized(x, qb):
    """x's rows quantized in blocks of qb inputs and scaled back."""
    b = x.reshape(x.shape[0], -1, qb)
    amax = b.abs().amax(-1, keepdim=True)
    d = amax / 127.0
    q = torch.where(amax > 0, torch.round(b * (127.0 / amax.clamp_min(1e-300))), torch.zeros_like(b))
    return (q * d).reshape(x.shape)


def _attention64(q, k, v, p, u, b):
    T = q.shape[0]
    dk = D_MODEL // HEADS
    idx = (T - 1 - torch.arange(T, device=q.device))[:, None] + torch.arange(T, device=q.device)[None, :]
    out = torch.empty_like(q)
    for h in range(HEADS):
        c = slice(h * dk, (h + 1) * dk)
        qu, qv = q[:, c] + u[c], q[:, c] + b[c]
        s = qu @ k[:, c].T.contiguous()
        s += torch.gather(qv @ p[:, c].T.contiguous(), 1, idx)
        out[:, c] = torch.softmax(s / math.sqrt(dk), -1) @ v[:, c].contiguous()
    return out


def _norm64(x, w, b):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + EPS) * w + b


def _layer64(i, case, dev):
    t = {n: torch.from_numpy(a).to(dev).double() for n, a in i.items() if not isinstance(a, tuple)}
    w = {n: _w64(a, dev) for n, a in i.items() if isinstance(a, tuple)}
    qb, x, T = case["qb"], t["x"], case["T"]

    def product(a, name):
        return _quantized(a, qb) @ w[name].T.contiguous()

    def ff(x, f):
        h = product(_norm64(x, t[f + "_nw"], t[f + "_nb"]), f + "_up")
        return x + product(h * torch.sigmoid(h), f + "_down")

    x = ff(x, "ff1")
    a = _norm64(x, t["att_nw"], t["att_nb"])
    o = _attention64(product(a, "q"), product(a, "k"), product(a, "v"), product(t["ape"], "pos"), t["bias_u"],
                     t["bias_v"])
    x = x + product(o, "o")
    u = product(_norm64(x, t["conv_nw"], t["conv_nb"]), "pw1")
    g = torch.nn.functional.pad(u[:, :D_MODEL] * torch.sigmoid(u[:, D_MODEL:]), (0, 0, TAPS // 2, TAPS // 2))
    c = t["dw_b"] + sum(g[j:j + T] * t["dw"][:, j] for j in range(TAPS))
    x = x + product(c * torch.sigmoid(c), "pw2")
    return _norm64(ff(x, "ff2"), t["out_nw"], t["out_nb"])


def _chain64(i, dev):
    x, ape = (torch.from_numpy(i[n]).to(dev).double() for n in ("x", "ape"))

    def product(a, name):
        return _quantized(a, a.shape[1]) @ _w64(i[name], dev).T.contiguous()

    x = x + product(product(x, "ff1_up"), "ff1_down")
    q, k, v, p = product(x, "q"), product(x, "k"), product(x, "v"), product(ape, "pos")
    x = x + product(v, "o")
    x = x + product(product(x, "pw1")[:, :D_MODEL].contiguous(), "pw2")
    x = x + product(product(x, "ff2_up"), "ff2_down")
    return [x, q, k, v, p]


def _tokens64(i, labels, h, c, dev):
    w = {n: _w64(a, dev) for n, a in i.items() if isinstance(a, tuple)}
    t = {n: torch.from_numpy(a).to(dev).double() for n, a in i.items() if isinstance(a, np.ndarray)}
    h, c = [a.double() for a in h], [a.double() for a in c]

    def gemv(x, name):
        return w[name] @ _quantized(x[None], x.shape[0])[0]

    for s, label in enumerate(labels):
        x = t["embed"][label]
        for l in range(LSTMS):
            g = gemv(x, f"wx{l}") + t[f"b{l}"] + gemv(h[l], f"wh{l}")
            gi, gf, gu, go = g.reshape(4, PRED)
            c[l] = torch.sigmoid(gf) * c[l] + torch.sigmoid(gi) * torch.tanh(gu)
            h[l] = x = torch.sigmoid(go) * torch.tanh(c[l])
        gp = gemv(x, "jpred") + t["jpred_b"]
        logit = gemv(torch.relu(t["f"][s] + gp), "jout") + t["jout_b"]
    return logit, torch.stack(h), torch.stack(c)


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    i = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("product", "dropin"):
        x = torch.from_numpy(i["x"]).to(dev).double()
        out = _quantized(x, case["qb"] or case["K"]) @ _w64(i["w"], dev).T.contiguous()
        if i["bias"] is not None:
            out = out + torch.from_numpy(i["bias"]).to(dev).double()
        if i["old"] is not None:
            out = out + torch.from_numpy(i["old"]).to(dev).double()
        return out if kind == "product" else [None, None, out.reshape(-1).cpu().numpy()]
    if kind == "grouped":
        w = _w64(i["w"], dev).T.contiguous()
        return [_quantized(torch.from_numpy(x).to(dev).double(), case["K"]) @ w for x in i["x"]]
    if kind == "attention":
        t = {n: torch.from_numpy(a).to(dev).double() for n, a in i.items()}
        return _attention64(t["q"], t["k"], t["v"], t["p"], t["u"], t["b"])
    if kind == "layer":
        return _layer64(i, case, dev)
    if kind == "chain":
        return _chain64(i, dev)
    if kind == "tokens":
        h, c = torch.from_numpy(i["h"]).to(dev), torch.from_numpy(i["c"]).to(dev)
        logit, h, c = _tokens64(i, i["labels"], h, c, dev)
        return [logit, None, h, c]
    z = torch.zeros(LSTMS, PRED, device=dev)
    return [None, _tokens64(i, [VOCAB], z, z, dev)[0]]
