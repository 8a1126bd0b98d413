"""GGUF layers with many tokens per call (from 256 on, experts in Q3_K, Q4_K
or Q8_0 with hidden, inter and inter_sh multiples of 128): the experts'
products on the matrix cores, integer codes in f16 against activations in
three f16 parts.

Reference: the reference's composition on the dequantized weights in float64
(ids and probabilities of the oracle, which must match bit for bit).  Bar: the
relative 2-norm error of a token's output stays below 2e-6.  The parts hold
an activation exactly, the longest chain of fp32 additions is 2048 / 32
matrix instructions for each of the three parts, and random rounding over n
additions grows as sqrt(n) 2^-24 = 14 * 6e-8 = 8.3e-7 per product; those of
gate, up and down are independent: sqrt(3) * 8.3e-7 = 1.5e-6."""
import json

import numpy as np
import pytest

from dismoen import DismoenError, gguf, synth

pytestmark = pytest.mark.gpu
BAR = 2e-6


def _upload(block, tmp_path, slot, dims, ty, mutate=None):
    H, E, K, I, Ish = dims
    ts = synth.make_gguf_moe_layer(H, E, I, Ish, seed=slot, expert_type=ty)
    # logits near one, so that several experts carry weight
    ts[0] = (*ts[0][:3], synth.gguf_payload(np.random.default_rng(slot), 8, E * H, 1.4e-5))
    p = str(tmp_path / f"mm{slot}.gguf")
    gguf.write_gguf(p, mutate(ts) if mutate else ts)
    g = gguf.parse_gguf_index(p)
    block.upload_layer_gguf(slot, dims, g)
    return g


def _reference(oracle, g, dims, x, ids, probs, shg):
    """The block without residual in float64 for the given routing."""
    H, E, K, I, Ish = dims

    def deq(name, rows, cols):
        t = g.tensors[g.tensor_map["blk.0." + name]]
        return oracle.dequant_gguf(t.dtype, g.read_raw("blk.0." + name),
                                   t.num_elements).astype(np.float64).reshape(rows, cols)

    def ffn(v, gate, up, down, n):
        a, b = v @ deq(gate, n, H).T, v @ deq(up, n, H).T
        with np.errstate(over="ignore"):
            return (a / (1.0 + np.exp(-a)) * b) @ deq(down, H, n).T

    x = x.astype(np.float64)
    y = shg.astype(np.float64)[:, None] * ffn(x, "ffn_shared_gate.weight", "ffn_shared_up.weight",
                                              "ffn_shared_down.weight", Ish)
    for e in np.unique(ids):
        t, k = np.nonzero(ids == e)
        y[t] += probs[t, k].astype(np.float64)[:, None] * ffn(
            x[t], *(f"ffn_{w}.{e}.weight" for w in ("gate", "up", "down")), I)
    return y


def _check(block, oracle, g, slot, dims, x):
    H, E, K, I, Ish = dims
    T = x.shape[0]
    res = np.random.default_rng(T).standard_normal((T, H)).astype(np.float32)
    y, ids, probs, shg = block.forward_port_moe_gguf(x, None, slot, T)
    yr, ids2, _, _ = block.forward_port_moe_gguf(x, res, slot, T)
    t = g.tensors[g.tensor_map["blk.0.ffn_gate_exps.weight"]]
    w = oracle.dequant_gguf(t.dtype, g.read_raw("blk.0.ffn_gate_exps.weight"), t.num_elements)
    rid, rp = oracle.router_forward(x, w, T, H, E, K, layer=slot)
    assert np.array_equal(ids, rid) and np.array_equal(ids2, rid)
    assert np.array_equal(probs.view(np.uint32), rp.view(np.uint32))
    ref = _reference(oracle, g, dims, x, ids, probs, shg)
    err = np.linalg.norm(y - ref, axis=1) / np.maximum(np.linalg.norm(ref, axis=1), 1e-300)
    print(f"T={T} worst token {err.max():.2e}", flush=True)
    assert err.max() < BAR, (int(err.argmax()), err.max())
    # the residual is added last
    assert np.array_equal(yr.view(np.uint32), (y + res).view(np.uint32))
    return y, ids


@pytest.mark.parametrize("ty", [11, 12, 8])
@pytest.mark.parametrize("slot,dims,T", [
    (60, (128, 2, 1, 128, 128), 256),     # two stages a product; several full units of an expert
    (61, (640, 9, 3, 384, 128), 257),     # rows of broken 256-weight blocks; partial row blocks
    (62, (256, 70, 5, 256, 384), 300),    # units of about 21 tokens: two column tiles
    (63, (2048, 16, 8, 512, 512), 333),   # the Qwen3.6 shape
])
def test_against_float64(block, oracle, tmp_path, ty, slot, dims, T):
    g = _upload(block, tmp_path, slot, dims, ty)
    x = np.random.default_rng(T + ty).standard_normal((T, dims[0])).astype(np.float32)
    _, ids = _check(block, oracle, g, slot, dims, x)
    n = np.bincount(ids.reshape(-1), minlength=dims[1])
    print("tokens per expert", n.min(), n.max(), flush=True)
    block.free_layer_gguf(slot)


@pytest.mark.parametrize("ty", [11, 12, 8])
def test_unit_sizes(block, oracle, tmp_path, ty):
    """Experts with 1 to 129 tokens: every number of column tiles (one to three
    and units of 48 for Q8_0, one, two and four and units of 64 else) and the
    sizes on either side of each."""
    sizes = [1, 15, 16, 17, 32, 33, 47, 48, 49, 63, 64, 65, 81, 97, 129]
    n = len(sizes)
    dims = (256, n, 1, 128, 128)

    def route(ts):  # expert e's logit is x[e]
        blocks = np.zeros((n, 8, 34), np.uint8)
        blocks[:, :, 0:2] = np.array([1.0], np.float16).view(np.uint8)
        for e in range(n):
            blocks[e, 0, 2 + e] = 1
        return [(*ts[0][:3], blocks.tobytes())] + ts[1:]

    g = _upload(block, tmp_path, 64, dims, ty, route)
    rng = np.random.default_rng(5)
    owner = rng.permutation(np.repeat(np.arange(n), sizes))
    x = rng.standard_normal((owner.size, 256)).astype(np.float32)
    x[np.arange(owner.size), owner] = 6.0
    x[:, :n] = np.minimum(x[:, :n], 6.0)
    _, ids = _check(block, oracle, g, 64, dims, x)
    assert np.array_equal(np.bincount(ids.reshape(-1), minlength=n), sizes)
    block.free_layer_gguf(64)


@pytest.mark.parametrize("ty", [11, 12])
def test_rows_of_any_scale(block, oracle, tmp_path, ty):
    """Rows whose values lie near 1e-30, 1e-4 and 1e4 and rows that hold one
    large value among small ones: each row has its own power of two.  (The
    tiny rows' h is below fp32's range in the reference too; the bar is on
    the others and a zero row gives zeros.)"""
    dims = (256, 12, 4, 128, 256)
    g = _upload(block, tmp_path, 65, dims, ty)
    rng = np.random.default_rng(9)
    x = rng.standard_normal((264, 256)).astype(np.float32)
    x[0:40] *= np.float32(1e-4)
    x[40:80] *= np.float32(1e4)
    x[80:120, 3] = 3e4
    x[120:160] *= rng.choice(np.float32([1e-6, 1.0, 1e3]), (40, 256))
    y, _ = _check(block, oracle, g, 65, dims, x)
    x[5] = 0.0
    x[6] *= np.float32(1e-26)
    y2, _, _, _ = block.forward_port_moe_gguf(x, None, 65, 264)
    assert not y2[5].any() and np.isfinite(y2).all()
    keep = np.arange(264) // 2 != 3
    keep[5] = False
    assert np.array_equal(y[keep], y2[keep])
    block.free_layer_gguf(65)


def _encode(ty, codes, d):
    """A payload whose weight i is d[block of i] * codes[i] (fp16 d; Q3_K codes
    -4 .. 3, Q4_K 0 .. 15 without mins, Q8_0 -127 .. 127)."""
    bs, n = (32, 34) if ty == 8 else (256, 114 if ty == 11 else 144)
    q = np.asarray(codes).reshape(-1, bs)
    raw = np.zeros((q.shape[0], n), np.uint8)
    half = np.broadcast_to(d, q.shape[0]).astype("<f2").view(np.uint8).reshape(-1, 2)
    if ty == 8:
        raw[:, :2], raw[:, 2:] = half, q.astype(np.int8).view(np.uint8)
    elif ty == 11:
        u = (q + 4).astype(np.uint8)
        raw[:, :32] = np.packbits(u >> 2, axis=1, bitorder="little")
        raw[:, 32:96] = ((u & 3).reshape(-1, 64, 4) << np.array([0, 2, 4, 6])).sum(2)
        raw[:, 96:112], raw[:, 112:] = 33, half
    else:
        raw[:, :2], raw[:, 4:16] = half, 1
        u = q.astype(np.uint8).reshape(-1, 8, 2, 16)
        raw[:, 16:] = (u[:, :, 0] | u[:, :, 1] << 4).reshape(-1, 128)
    return raw.tobytes()


@pytest.mark.parametrize("ty", [11, 12, 8])
def test_every_bit_of_an_activation(block, oracle, tmp_path, ty):
    """gate = x0 + x1 where x1 is -x0 but for its last bits, up = x2: the
    difference is exact in fp32, and the outputs keep the bar only if the last
    bit of every activation counts."""
    dims, T = (256, 4, 2, 128, 128), 256

    def f(ts):
        gate, up = np.zeros((128, 256), int), np.zeros((128, 256), int)
        gate[:, :2] = 1
        up[:, 2] = 1
        return [(n, d, t, _encode(ty, gate if "gate" in n else up, 1.0))
                if n.split(".")[2] in ("ffn_gate", "ffn_up", "ffn_shared_gate", "ffn_shared_up")
                else (n, d, t, raw) for n, d, t, raw in ts]

    g = _upload(block, tmp_path, 68, dims, ty, f)
    rng = np.random.default_rng(21)
    x = rng.standard_normal((T, 256)).astype(np.float32)
    x[:, 0] = rng.uniform(1, 2, T).astype(np.float32)
    x[:, 1] = -(x[:, 0].view(np.int32) + rng.integers(1, 9, T).astype(np.int32)).view(np.float32)
    _check(block, oracle, g, 68, dims, x)
    block.free_layer_gguf(68)


@pytest.mark.parametrize("ty", [11, 12, 8])
def test_values_far_below_the_rows_largest(block, oracle, tmp_path, ty):
    """x5 is 2^26 times the others where every weight is zero, and h7 2^20
    times the others where every down weight is: the small values alone make
    the outputs."""
    dims, T = (256, 4, 2, 128, 128), 256
    lo, hi = {11: (-4, 4), 12: (0, 16), 8: (-127, 128)}[ty]
    rng = np.random.default_rng(22)

    def f(ts):
        out = []
        for n, dm, t, raw in ts:
            k = n.split(".")[2]
            if k == "shared_gate":
                w = np.frombuffer(raw, "<f4").copy()
                w[5] = 0
                raw = w.tobytes()
            elif k == "ffn_gate_exps":
                w = np.frombuffer(raw, np.uint8).reshape(4, 8, 34).copy()
                w[:, 0, 2 + 5] = 0
                raw = w.tobytes()
            elif k in ("ffn_down", "ffn_shared_down"):
                c = rng.integers(lo, hi, (256, 128))
                c[:, 7] = 0
                raw = _encode(ty, c, 2.0 ** -6)
            elif k.startswith("ffn"):
                c = rng.integers(lo, hi, (128, 256))
                c[:, 5] = 0
                d = np.full((128, 256 // (32 if ty == 8 else 256)), 2.0 ** (-11 if ty == 8 else -7))
                if "up" in k:
                    d[7] *= 2.0 ** 20
                raw = _encode(ty, c, d.reshape(-1))
            out.append((n, dm, t, raw))
        return out

    g = _upload(block, tmp_path, 69, dims, ty, f)
    x = rng.standard_normal((T, 256)).astype(np.float32)
    x[:, 5] *= np.float32(2.0 ** 26)
    _check(block, oracle, g, 69, dims, x)
    block.free_layer_gguf(69)


def test_more_tokens_than_one_launch_combines(block, oracle, tmp_path):
    """65537 tokens: the combine splits at 65535; rows on either side of the
    split against float64, and the same bits as in a call of their own of 256
    tokens."""
    dims, T = (128, 4, 2, 128, 128), 65537
    g = _upload(block, tmp_path, 67, dims, 11)
    x = np.random.default_rng(11).standard_normal((T, 128)).astype(np.float32)
    y, ids, probs, shg = block.forward_port_moe_gguf(x, None, 67, T)
    y2, ids2, _, _ = block.forward_port_moe_gguf(x[-256:], None, 67, 256)
    assert np.array_equal(ids[-256:], ids2)
    assert np.array_equal(y[-256:].view(np.uint32), y2.view(np.uint32))
    rows = np.array([0, 65534, 65535, 65536])
    ref = _reference(oracle, g, dims, x[rows], ids[rows], probs[rows], shg[rows])
    err = np.linalg.norm(y[rows] - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert err.max() < BAR, err
    block.free_layer_gguf(67)


def test_errors(block, tmp_path):
    """The texts of the other forms: a non-finite activation, an infinite
    super-scale in a shared and in a routed expert."""
    dims, T = (256, 8, 2, 128, 128), 300
    x = np.random.default_rng(1).standard_normal((T, 256)).astype(np.float32)
    _upload(block, tmp_path, 66, dims, 11)
    bad = x.copy()
    bad[299, 7] = np.inf
    with pytest.raises(DismoenError) as ei:
        block.forward_port_moe_gguf(bad, None, 66, T)
    assert json.loads(str(ei.value))["error_type"] == "ACT_LOAD_FAILED"
    block.forward_port_moe_gguf(x, None, 66, T)  # and recovers

    def inf_scale(name):
        def f(ts):
            i = [k for k, t in enumerate(ts) if t[0] == "blk.0." + name][0]
            raw = bytearray(ts[i][3])
            raw[112:114] = b"\x00\x7c"
            return ts[:i] + [(*ts[i][:3], bytes(raw))] + ts[i + 1:]
        return f

    for name, detail in (("ffn_shared_up.weight", "non-finite in up projection"),
                         ("ffn_shared_down.weight", "non-finite in down projection"),
                         ("ffn_gate.3.weight", "non-finite in gate projection")):
        _upload(block, tmp_path, 66, dims, 11, inf_scale(name))
        texts = []
        for n in (T, 255):  # the matrix-core form and the form below it
            with pytest.raises(DismoenError) as ei:
                block.forward_port_moe_gguf(x[:n], None, 66, n)
            texts.append(str(ei.value))
        assert texts[0] == texts[1] and json.loads(texts[0])["detail"] == detail
    block.free_layer_gguf(66)


def test_closed_contexts_keep_nothing(tmp_path):
    """A context's buffers go with it, those of the column sums (12 MB here)
    among them."""
    import torch
    from dismoen import MoEBlock
    dims, T = (2048, 2, 1, 512, 512), 16384
    x = np.zeros((T, 2048), np.float32)
    free = []
    for _ in range(4):
        b = MoEBlock(0)
        _upload(b, tmp_path, 0, dims, 12)
        b.forward_port_moe_gguf(x, None, 0, T)
        b.close()
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
    assert free[0] - free[-1] < 8 << 20, free


def _both_forms(block, slot, x):
    """Outputs of one call, and of calls below the matrix-core form."""
    T = x.shape[0]
    y = block.forward_port_moe_gguf(x, None, slot, T)[0]
    z = np.concatenate([block.forward_port_moe_gguf(x[i:i + 128], None, slot, x[i:i + 128].shape[0])[0]
                        for i in range(0, T, 128)])
    return y, z


def test_records_declined(block, tmp_path):
    dims = (256, 8, 2, 128, 128)
    p = str(tmp_path / "l.gguf")
    gguf.write_gguf(p, synth.make_gguf_moe_layer(256, 8, 128, 128, seed=70, expert_type=11))
    x = np.random.default_rng(3).standard_normal((300, 256)).astype(np.float32)
    with gguf.parse_gguf_index(p) as g:
        for records in (True, False):
            block.upload_layer_gguf(70, dims, g, records=records)
            y, z = _both_forms(block, 70, x)
            assert np.array_equal(y, z) != records
    block.free_layer_gguf(70)


def test_records_make_room(block, tmp_path):
    """With the device's memory all but full, an upload takes the records of
    another layer, not those a captured graph uses; that layer's calls run in
    the form of fewer tokens, and the graph's replays are right."""
    import torch
    dims, T = (2048, 32, 2, 512, 512), 256
    p = str(tmp_path / "l.gguf")
    gguf.write_gguf(p, synth.make_gguf_moe_layer(2048, 32, 512, 512, seed=71, expert_type=11))
    x = np.random.default_rng(4).standard_normal((T, 2048)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    yd = torch.zeros_like(xd)
    fill, s, graph = [], torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with gguf.parse_gguf_index(p) as g:
        for slot in (71, 72):
            block.upload_layer_gguf(slot, dims, g)
            y, z = _both_forms(block, slot, x)
            assert not np.array_equal(y, z)
        block.forward_gguf_device(72, xd.data_ptr(), T, yd.data_ptr())  # (its buffers)
        torch.cuda.synchronize()
        block.set_stream(s.cuda_stream)
        try:
            with torch.cuda.graph(graph, stream=s):
                block.forward_gguf_device(72, xd.data_ptr(), T, yd.data_ptr())
        finally:
            block.set_stream(None)
        block.sync()
        try:
            left = 24 << 20  # a payload is 47 MB, its records 71 MB
            while (free := torch.cuda.mem_get_info()[0]) > left + (8 << 20) and len(fill) < 40:
                fill.append(torch.empty(min(free - left, 32 << 30), dtype=torch.uint8, device="cuda"))
            print("free", free >> 20, "MB", flush=True)
            block.upload_layer_gguf(73, dims, g)
        finally:
            fill.clear()
            torch.cuda.empty_cache()
    for slot in (71, 73):  # taken back; not made
        y1, z1 = _both_forms(block, slot, x)
        assert np.array_equal(y1, z) and np.array_equal(z1, z), slot
    for _ in range(3):
        yd.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(yd.cpu().numpy(), y)
        assert np.array_equal(_both_forms(block, 72, x)[0], y)
    del graph
    for slot in (71, 72, 73):
        block.free_layer_gguf(slot)
