"""The grouped expert kernels at the unit sizes where they branch: one, two
and four column tiles and the edges between them, several units of one
expert, a unit's remainder, a partial last block of output rows, and the
shortest reduction, with activations that are bf16 values and that are not.

Bar: max-abs-err <= 1e-3 x RMS of the oracle's fp32 SwiGLU on the same
bf16-rounded weights (the outputs' bar everywhere; the activations enter with
16 bits, 2^-17 of the value per product)."""
import numpy as np
import pytest

from conftest import tol_check
from dismoen import synth
from test_gpu_units import oracle_expert

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 129]


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("H,I,Ish", [(128, 128, 128), (384, 256, 128)])
def test_unit_sizes(block, oracle, H, I, Ish, fp32):
    L = synth.make_layer(hidden=H, num_experts=len(SIZES), top_k=1, inter=I, inter_sh=Ish, seed=H)
    block.upload_layer(25, L)
    rng = np.random.default_rng(H + fp32)
    ids = rng.permutation(np.repeat(np.arange(len(SIZES)), SIZES)).astype(np.int32)
    T = ids.size
    x = synth.make_activations(rng, (T, H))
    if fp32:
        x = (x * np.float32(1 + 2.0 ** -10)).astype(np.float32)
    out, sh = block.experts_forward(x, ids[:, None], 25, T, with_shared=True)
    for e in range(len(SIZES)):
        rows = ids == e
        err, rms, ok = tol_check(out[rows, 0], oracle_expert(oracle, L, e, x[rows]))
        assert ok, (SIZES[e], err, rms)
    err, rms, ok = tol_check(sh, oracle_expert(oracle, L, -1, x))
    assert ok, (err, rms)
