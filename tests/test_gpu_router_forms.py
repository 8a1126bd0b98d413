"""The routers of many tokens at the sizes where each form runs: ids and
probabilities of every token, shared gates of a sample, bit-exact against the
oracle.  256 CUs: the matrix-core router splits an expert group's chains over
four waves while tiles (of 16 tokens) x (ceil(E / 16) + 1) workgroups fit them,
takes four waves of 16 experts while tiles x (ceil(E / 64) + 1) do, and eight
beyond; the lane-chain router holds two rows per lane from 131072 logits on."""
import numpy as np
import pytest

from dismoen import synth

pytestmark = pytest.mark.gpu


def _check(block, oracle, slot, H, E, K, x):
    T = x.shape[0]
    L = synth.make_layer(H, E, K, 128, 128, seed=H + E)
    block.upload_layer(slot, L)
    _, ids, probs, shg = block.forward_arrays(slot, x, T)
    w = synth.bf16_bits_to_f32(L.router_bf16).reshape(E, H)
    ido, po = oracle.router_forward(x, w, T, H, E, K)
    assert np.array_equal(ids, ido)
    assert np.array_equal(probs.view(np.uint32), po.view(np.uint32))
    sample = np.unique(np.linspace(0, T - 1, 9).astype(int))
    _, _, _, so = oracle.moe_layer_q4(L, x[sample], len(sample))
    assert np.array_equal(shg[sample].view(np.uint32), so.view(np.uint32))
    block.free_layer(slot)


@pytest.mark.parametrize("H,E,T", [
    (384, 40, 70),       # split; experts and rounds (3) short of the group's and the ring's
    (640, 200, 288),     # split, the last size
    (384, 40, 1100),     # four waves, one partial wave of experts; 3 rounds on a ring of 4
    (640, 200, 304),     # four waves, a partial last column; 5 rounds
    (2048, 256, 301),    # four waves, the Qwen3.6 shape, a ragged tile
    (2048, 256, 816),    # four waves, the last size
    (2048, 256, 833),    # eight waves, the first size
    (384, 40, 2100),     # eight waves, five of them without experts (the gate's among them)
    (640, 200, 901),     # eight waves, a partial second column; an odd number of rounds
])
def test_matrix_core_router(block, oracle, H, E, T):
    x = synth.make_activations(np.random.default_rng(T), (T, H))
    _check(block, oracle, 75, H, E, 4, x)


@pytest.mark.parametrize("H", [256, 512, 1024, 2048])
@pytest.mark.parametrize("E,T", [
    (200, 652),     # one row, the last size
    (200, 661),     # two rows; the last block's second rows past row E; a ragged last pass
    (33, 4001),     # two rows, one live wave in the last block
])
def test_lane_chain_router(block, oracle, H, E, T):
    x = np.random.default_rng(T).standard_normal((T, H)).astype(np.float32)
    _check(block, oracle, 76, H, E, 4, x)
