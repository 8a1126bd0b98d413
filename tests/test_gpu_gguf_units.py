"""GGUF layers, several tokens grouped by expert: every token's outputs are
those of its own single-token call, bit for bit, at the unit sizes and shapes
where the grouped kernels branch (units of 1 .. 8 tokens, rows past a wave's
share, rows that start inside a block, partial chunks of a row)."""
import numpy as np
import pytest

from dismoen import gguf, synth

pytestmark = pytest.mark.gpu


# (hidden, experts, top_k, inter, inter_sh), tokens
SHAPES = [
    ((1040, 6, 2, 48, 80), 60),      # 20 tokens per expert: units of eight and their remainders
    ((1040, 64, 2, 48, 80), 60),     # units of four, most of one or two tokens
    ((2048, 9, 3, 640, 128), 9),     # two chunks in every row, a few tokens
    ((256, 16, 4, 128, 512), 130),   # a quarter of a wave's chunk per row
    # without the blocked kernels: grouped from 128 tokens
    ((264, 6, 2, 64, 96), 130),      # rows of eight weights per lane, units of eight
    ((264, 80, 1, 64, 96), 130),     # and of four
    ((2304, 6, 2, 64, 64), 130),     # hidden above 2048
    ((256, 6, 2, 1088, 128), 130),   # inter above 1024: blocked gate/up, down not
]


def _tensors(dims, ty):
    """A layer with experts of type ty (BF16, 30: the high halves of F32)."""
    H, E, K, I, Ish = dims
    ts = synth.make_gguf_moe_layer(H, E, I, Ish, seed=ty + H, expert_type=0 if ty == 30 else ty)
    if ty != 30:
        return ts
    return [(n, d, 30, np.frombuffer(raw, np.uint16)[1::2].tobytes())
            if t == 0 and "ffn_" in n else (n, d, t, raw) for n, d, t, raw in ts]


@pytest.mark.parametrize("ty", [11, 12, 8, 30, 0])
@pytest.mark.parametrize("dims,T", SHAPES)
def test_same_bits_as_single_tokens(block, tmp_path, ty, dims, T):
    H = dims[0]
    p = str(tmp_path / "layer.gguf")
    gguf.write_gguf(p, _tensors(dims, ty))
    with gguf.parse_gguf_index(p) as g:
        block.upload_layer_gguf(24, dims, g)
    x = synth.make_activations(np.random.default_rng(ty), (T, H))
    res = synth.make_activations(np.random.default_rng(ty + 1), (T, H))
    y, ids, probs, shg = block.forward_port_moe_gguf(x, res, 24, T)
    for t in range(T):
        y1, i1, p1, s1 = block.forward_port_moe_gguf(x[t:t + 1], res[t:t + 1], 24, 1)
        assert np.array_equal(ids[t], i1[0]) and np.array_equal(probs[t], p1[0]), t
        assert shg[t] == s1[0], t
        assert np.array_equal(y[t].view(np.uint32), y1[0].view(np.uint32)), t
