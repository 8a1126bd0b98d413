"""The work that the MoE block's users have it do, as measurable cases.

An engine that decodes with this library makes one call per layer and token;
one that serves several streams makes calls of a few to some tens of tokens;
prompts come in chunks of up to a few thousand.  Layers are in the 4-bit group
format or come from GGUF files.  All cases go through dismoen.MoEBlock, one
block per process with each layer in a slot of its own, as a program keeps it.

A case is a dict of plain values:
  kind     "block"  forward_device: router, experts, shared expert, combine on
                    device buffers (bf16-valued activations)
           "host"   forward_into: the same on the caller's host arrays
           "norm"   forward_port_moe_norm_device: RMSNorm, block and residual
                    (the port block's MoE section; fp32 activations)
           "stack"  forward_stack_device: `layers` such sections in sequence
           "gguf"   forward_gguf_device: a layer of a GGUF file, fp32
                    activations
  tokens   tokens per call
  hidden, experts, top_k, inter, inter_sh   the layer's shape
  layers   stack depth (1 elsewhere)
  group    weights per scale of the 4-bit format
  skew     exponent of the Zipf popularity of the experts (0: even)
  residual whether the call adds a residual (block, host, gguf)
  type     GGML type of the experts: "q3_k", "q4_k", "q8_0" ("" elsewhere)
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "disk-streaming-moe-engine_amd"))
from dismoen import MoEBlock, gguf, synth  # noqa: E402

EPS = 1e-6
TYPES = {"q3_k": (11, 256, 114), "q4_k": (12, 256, 144), "q8_0": (8, 32, 34)}
QWEN36 = synth.CONFIG_QWEN36
TOY = synth.CONFIG_TOY


def _case(kind, tokens, shape, name=None, layers=1, group=32, skew=0.0, residual=False, type=""):
    c = {"kind": kind, "tokens": tokens, "hidden": shape["hidden"],
         "experts": shape["num_experts"], "top_k": shape["top_k"], "inter": shape["inter"],
         "inter_sh": shape["inter_sh"], "layers": layers, "group": group, "skew": skew,
         "residual": residual, "type": type}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one layer of batch-1 decode of the small test model: launches and latency only
        _case("block", 1, TOY, "toy decode"),
        # one layer of batch-1 decode, the headline benchmark
        _case("block", 1, QWEN36, "decode"),
        # the same through host arrays: the call a compiled engine makes per layer and token
        _case("host", 1, QWEN36, "decode, host arrays"),
        # a whole token's MoE sections, all 40 layers of the model
        _case("stack", 1, QWEN36, "decode, 40 layers", layers=40),
        # a few streams decoded together
        _case("block", 8, QWEN36, "batch 8", residual=True),
        # some tens of streams, or speculative tokens, with the layer's norm
        _case("norm", 32, QWEN36, "batch 32 with norm", group=128),
        # a short prompt or a large decode batch, a ragged size
        _case("block", 131, QWEN36, "131 tokens"),
        # a prompt chunk with skewed expert popularity, the benchmark's prefill
        _case("block", 2048, QWEN36, "prefill 2048", skew=1.1),
        # a ragged prompt tail through the port block's MoE section
        _case("norm", 1533, QWEN36, "prefill 1533 with norm"),
        # batch-1 decode of a GGUF layer
        _case("gguf", 1, QWEN36, "gguf q3_k decode", type="q3_k"),
        # a decode batch on a GGUF layer
        _case("gguf", 24, QWEN36, "gguf q4_k batch 24", residual=True, type="q4_k"),
        # a prompt chunk on a GGUF layer
        _case("gguf", 2048, QWEN36, "gguf q3_k prefill 2048", residual=True, type="q3_k"),
    ]


def draw(rng):
    kind = rng.choice(["block", "block", "norm", "gguf", "gguf", "gguf", "host", "stack"])
    shape = dict(QWEN36)
    if rng.random() < 0.5:  # another layer shape: rows of whole and of broken 256-weight blocks
        shape = {"hidden": 128 * rng.randint(2, 16), "num_experts": rng.randint(9, 256),
                 "top_k": rng.randint(1, 8), "inter": 128 * rng.randint(1, 4),
                 "inter_sh": 128 * rng.randint(1, 4)}
    tokens = round(math.exp(rng.uniform(0.0, math.log(2048.0))))
    if kind == "host":
        tokens = min(tokens, 1 + tokens % 64)
    layers = 1
    if kind == "stack":
        tokens = min(tokens, 1 + tokens % 16)
        layers = rng.randint(2, 12)
    return _case(kind, tokens, shape, layers=layers,
                 group=rng.choice([32, 64, 128]) if kind != "gguf" else 32,
                 skew=rng.choice([0.0, 1.1]) if kind in ("block", "gguf") and tokens > 64 else 0.0,
                 residual=rng.random() < 0.5 if kind in ("block", "host", "gguf") else False,
                 type=rng.choice(sorted(TYPES)) if kind == "gguf" else "")


# ---- inputs -----------------------------------------------------------------
def _dims(case):
    return (case["hidden"], case["experts"], case["top_k"], case["inter"], case["inter_sh"])


def _activations(case, seed):
    """x and the residual (or None) on the GPU: N(0, 1), rounded to bf16
    values where the program's activations are bf16, feature 0 = 1 where the
    router carries a popularity bias in its column 0."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)
    n = (case["tokens"], case["hidden"])
    x = torch.randn(n, generator=g, device="cuda")
    if case["kind"] in ("block", "host"):
        x = x.to(torch.bfloat16).float()
    res = torch.randn(n, generator=g, device="cuda") if case["residual"] else None
    if case["skew"]:
        x[:, 0] = 1.0
    return x, res


def _weights4(case, seed, layer):
    """One layer in the 4-bit format: field name -> device tensor."""
    H, E, K, I, Ish = _dims(case)
    w = synth.make_layer_device(H, E, K, I, Ish, case["group"], seed * 1009 + layer)
    if case["skew"]:
        bias = torch.from_numpy(synth.zipf_router_bias(E, case["skew"], seed)).cuda()
        w["router_bf16"].view(E, H)[:, 0] = bias.to(torch.bfloat16).view(torch.int16)
    return w


def _gamma(case, seed, layer):
    g = np.random.default_rng([seed, layer, 3])
    return (1.0 + 0.1 * g.standard_normal(case["hidden"])).astype(np.float32)


def _payloads(case, seed):
    """A GGUF layer's raw bytes: router (Q8_0), shared gate (F32) and the
    experts' gate, up and down, the shared expert's last."""
    H, E, K, I, Ish = _dims(case)
    t = TYPES[case["type"]][0]
    rng = np.random.default_rng([seed, 5])
    router = synth.gguf_payload(rng, 8, E * H, 1.4e-5)
    if case["skew"]:  # the popularity bias: the first block of each row holds it in code 0
        blocks = np.frombuffer(router, np.uint8).reshape(E, H // 32, 34).copy()
        bias = synth.zipf_router_bias(E, case["skew"], seed)
        d = np.abs(bias) / 127.0 + 1e-4
        blocks[:, 0, 0:2] = d.astype(np.float16).view(np.uint8).reshape(E, 2)
        blocks[:, 0, 2:] = 0
        blocks[:, 0, 2] = np.round(bias / d).astype(np.int8).view(np.uint8)
        router = blocks.tobytes()
    gate = (rng.standard_normal(H) * 0.02).astype("<f4").tobytes()
    experts = synth.gguf_payload(rng, t, 3 * H * (E * I + Ish), 1.4e-5 if t == 8 else 1e-4)
    return router, gate, experts


def _split(case, raw):
    """[(gate, up, down)] of the experts' bytes, the shared expert's last."""
    H, E, K, I, Ish = _dims(case)
    _, bs, bpb = TYPES[case["type"]]
    out, at = [], 0
    for n in [I * H] * E + [Ish * H]:
        b = n // bs * bpb
        out.append(tuple(raw[at + i * b:at + (i + 1) * b] for i in range(3)))
        at += 3 * b
    return out


def _upload_gguf(blk, slot, case, seed):
    H, E, K, I, Ish = _dims(case)
    t = TYPES[case["type"]][0]
    router, gate, raw = _payloads(case, seed)
    ts = [("blk.0.ffn_gate_exps.weight", [H, E], 8, router)]
    for e, parts in enumerate(_split(case, memoryview(raw))):
        names = [f"blk.0.ffn_{k}.{e}.weight" if e < E else f"blk.0.ffn_shared_{k}.weight"
                 for k in ("gate", "up", "down")]
        n = I if e < E else Ish
        for name, dims, part in zip(names, ([H, n], [H, n], [n, H]), parts):
            ts.append((name, dims, t, part))
    ts.append(("blk.0.shared_gate.weight", [H], 0, gate))
    fd, path = tempfile.mkstemp(suffix=".gguf")
    os.close(fd)
    try:
        gguf.write_gguf(path, ts)
        with gguf.parse_gguf_index(path) as index:
            blk.upload_layer_gguf(slot, _dims(case), index)
    finally:
        os.unlink(path)


# ---- the program ------------------------------------------------------------
_block = None
_slots = set()


def _the_block():
    global _block
    if _block is None:
        _block = MoEBlock(0)
    return _block


class State:
    """The layers of one case in slots of their own, its inputs and outputs."""

    def __init__(self, case, seed):
        self.case, self.blk = case, _the_block()
        T, L = case["tokens"], case["layers"]
        H, E, K, I, Ish = _dims(case)
        first = 0
        while any(s in _slots for s in range(first, first + L)):
            first += 1
        self.first, self.mine = first, list(range(first, first + L))
        _slots.update(self.mine)
        self.x, self.res = _activations(case, seed)
        if case["kind"] == "gguf":
            _upload_gguf(self.blk, first, case, seed)
        for l in self.mine if case["kind"] != "gguf" else []:
            w = _weights4(case, seed, l - first)
            torch.cuda.synchronize()  # drawn on torch's stream, read on the block's
            self.blk.upload_layer_device(l, _dims(case), {k: v.data_ptr() for k, v in w.items()},
                                         case["group"])
            self.blk.sync()
            if case["kind"] in ("norm", "stack"):
                self.blk.set_layer_norm(l, _gamma(case, seed, l - first))
        rows = T * L if case["kind"] == "stack" else T
        self.y = torch.empty((T, H), device="cuda")
        self.ids = torch.empty((rows, K), dtype=torch.int32, device="cuda")
        self.probs = torch.empty((rows, K), device="cuda")
        self.shg = torch.empty(T, device="cuda")
        if case["kind"] == "host":
            self.x, self.res, self.y, self.ids, self.probs, self.shg = (
                None if t is None else t.cpu().numpy()
                for t in (self.x, self.res, self.y, self.ids, self.probs, self.shg))
        torch.cuda.synchronize()

    def __del__(self):
        for s in self.mine:
            if self.case["kind"] == "gguf":
                self.blk.free_layer_gguf(s)
            else:
                self.blk.free_layer(s)
        _slots.difference_update(self.mine)


def prepare(case, seed):
    return State(case, seed)


def run(s):
    blk, T, kind = s.blk, s.case["tokens"], s.case["kind"]
    if kind == "host":
        blk.forward_into(s.first, s.x, T, s.y, s.ids, s.probs, s.shg, s.res)
        return {"y": s.y, "ids": s.ids, "probs": s.probs, "shared_gate": s.shg}
    x, y, ids, probs = s.x.data_ptr(), s.y.data_ptr(), s.ids.data_ptr(), s.probs.data_ptr()
    res = s.res.data_ptr() if s.res is not None else None
    if kind == "stack":
        blk.forward_stack_device(x, s.first, s.case["layers"], T, y, EPS, ids, probs)
        return {"y": s.y, "ids": s.ids, "probs": s.probs}
    if kind == "gguf":
        blk.forward_gguf_device(s.first, x, T, y, ids, probs, res)
        return {"y": s.y, "ids": s.ids, "probs": s.probs}
    if kind == "norm":
        blk.forward_port_moe_norm_device(s.first, x, T, y, EPS, ids, probs, s.shg.data_ptr())
    else:
        blk.forward_device(s.first, x, T, y, ids, probs, s.shg.data_ptr(), res)
    return {"y": s.y, "ids": s.ids, "probs": s.probs, "shared_gate": s.shg}


# ---- what a pass cannot do without --------------------------------------------
def work(case):
    H, E, K, I, Ish = _dims(case)
    T, L = case["tokens"], case["layers"]
    # distinct experts of T tokens with K of E each, drawn evenly
    used = E * (1.0 - (1.0 - K / E) ** T)
    if case["kind"] == "gguf":
        _, bs, bpb = TYPES[case["type"]]
        per = bpb / bs
        router = E * H * 34 / 32 + H * 4
    else:
        per = 0.5 + 2.0 / case["group"]
        router = (E + 1) * H * 2
    weights = 3 * H * (used * I + Ish) * per + router
    norm = 4 * H if case["kind"] in ("norm", "stack") else 0
    rows = T * H * 4 * (3 if case["residual"] else 2) + T * (K * 8 * L + 4)
    flops = 2 * T * (3 * H * (K * I + Ish) + (E + 1) * H)
    return {"bytes": L * (weights + norm) + rows, "flops": L * flops}


def tolerance(case):
    # 4-bit layers carry activations as pairs of bf16 values (16 bits); over
    # a stack of layers such differences travel, and may decide a close
    # choice of experts.  GGUF layers are 32-bit throughout.
    if case["kind"] == "stack":
        return {"rel": 2e-4, "max": 4e-3, "differ": 0.01}
    if case["kind"] == "gguf":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 4e-5, "max": 1e-3}


# ---- the same in 64 bits --------------------------------------------------------
def _codes4(packed, n):
    b = packed[: n // 2].to(torch.int16)
    q = torch.stack((b & 15, b >> 4), 1).reshape(-1)
    return torch.where(q > 7, q - 16, q)


def _matrix4(scales, packed, at, rows, cols, group):
    """Rows `at` .. of a flat 4-bit tensor: bf16(scale * code), in 64 bits."""
    n, o = rows * cols, at * cols
    s = scales[o // group:(o + n) // group].view(torch.float16).float()
    q = _codes4(packed[o // 2:(o + n) // 2], n).float().view(-1, group)
    return (s[:, None] * q).to(torch.bfloat16).double().view(rows, cols)


def _matrix_gguf(case, part, rows, cols):
    t, bs, bpb = TYPES[case["type"]]
    b = torch.frombuffer(bytearray(part), dtype=torch.uint8).cuda().view(-1, bpb)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    u = b.double()
    if t == 8:  # fp16 d, 32 signed codes
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif t == 11:  # 32 bytes of high bits, 64 of low pairs, 16 scales (+ 32), fp16 d
        i = torch.arange(256, device="cuda")
        hi = (b[:, i // 8] >> (i % 8)) & 1
        lo = (b[:, 32 + i // 4] >> (2 * (i % 4))) & 3
        w = half(112) * (u[:, 96 + i // 16] - 32.0) * ((hi * 4 + lo).double() - 4.0)
    else:  # fp16 d and dmin, 12 bytes of 6-bit scales and mins, 128 of code pairs
        j = torch.arange(8, device="cuda")
        q, lo4 = b[:, 4:16], j < 4
        jj = j.clamp(max=3)
        kk = (j - 4).clamp(min=0)
        sc = torch.where(lo4, q[:, jj] & 63, (q[:, j] & 15) | ((q[:, kk] >> 6) << 4))
        mn = torch.where(lo4, q[:, jj + 4] & 63, (q[:, j] >> 4) | ((q[:, j] >> 6) << 4))
        i = torch.arange(256, device="cuda")
        code = b[:, 16 + (i // 32) * 16 + i % 16]
        code = torch.where(i % 32 < 16, code & 15, code >> 4)
        w = half(0) * sc[:, i // 32].double() * code.double() - half(2) * mn[:, i // 32].double()
    return w.reshape(rows, cols)


def _swiglu(x, gate, up, down):
    return (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T


def _moe(case, x, router, shgate, expert):
    """(y, probs, gate) of the block without residual; expert(e) gives the
    three matrices of expert e, of the shared one for e = E."""
    E, K = case["experts"], case["top_k"]
    probs, ids = torch.topk(torch.softmax(x @ router.T, 1), K, 1)
    gate = torch.sigmoid(x @ shgate)
    y = gate[:, None] * _swiglu(x, *expert(E))
    for e in torch.unique(ids).tolist():
        t, k = torch.nonzero(ids == e, as_tuple=True)
        y[t] += probs[t, k][:, None] * _swiglu(x[t], *expert(e))
    return y, probs, gate


def exact(case, seed):
    H, E, K, I, Ish = _dims(case)
    if case["layers"] * case["tokens"] > 4096:
        return None
    x, res = _activations(case, seed)
    x = x.double()
    out = {"ids": None}
    if case["kind"] == "gguf":
        router, gate, raw = _payloads(case, seed)
        parts = _split(case, memoryview(raw))

        def expert(e):
            n = I if e < E else Ish
            return tuple(_matrix_gguf(case, p, r, c)
                         for p, r, c in zip(parts[e], (n, n, H), (H, H, n)))

        w = _matrix_gguf(dict(case, type="q8_0"), router, E, H)
        g = torch.from_numpy(np.frombuffer(gate, np.float32).copy()).cuda().double()
        y, out["probs"], _ = _moe(case, x, w, g, expert)
    else:
        y, probs = x, []
        for l in range(case["layers"]):
            w = _weights4(case, seed, l)
            G = case["group"]

            def expert(e):
                if e == E:
                    m = _matrix4(w["sh_gu_scales"], w["sh_gu_packed"], 0, 2 * Ish, H, G)
                    return m[:Ish], m[Ish:], _matrix4(w["sh_d_scales"], w["sh_d_packed"], 0, H,
                                                      Ish, G)
                m = _matrix4(w["gu_scales"], w["gu_packed"], e * 2 * I, 2 * I, H, G)
                return m[:I], m[I:], _matrix4(w["d_scales"], w["d_packed"], e * H, H, I, G)

            xn = y
            if case["kind"] in ("norm", "stack"):
                gamma = torch.from_numpy(_gamma(case, seed, l)).cuda().double()
                xn = y * torch.rsqrt((y * y).mean(1, keepdim=True) + EPS) * gamma
            r, p, gate = _moe(case, xn, w["router_bf16"].view(torch.bfloat16).double().view(E, H),
                              w["shgate_bf16"].view(torch.bfloat16).double(), expert)
            y = y + r if case["kind"] in ("norm", "stack") else r
            probs.append(p)
        out["probs"] = torch.cat(probs)
        if case["kind"] != "stack":
            out["shared_gate"] = gate
    out["y"] = y if res is None else y + res.double()
    return out
