"""A call captured into a graph after an eager call of more tokens: its buffers
are there already (an allocation would fail the capture), on both sides of the
sizes where the work units change.  Replays with eager calls between."""
import numpy as np
import pytest

from dismoen import MoEBlock, gguf, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,eager,captured", [
    ("q4", 33, 32), ("q4", 64, 9),
    (11, 256, 255), (11, 300, 257), (11, 256, 31),
])
def test_captured_after_a_larger_call(tmp_path, kind, eager, captured):
    import torch
    H, E, K, I = 256, 16, 4, 128
    b = MoEBlock(0)  # without buffers of other calls
    if kind == "q4":
        b.upload_layer(0, synth.make_layer(H, E, K, I, I, seed=5))
        call = b.forward_device
    else:
        p = str(tmp_path / "l.gguf")
        gguf.write_gguf(p, synth.make_gguf_moe_layer(H, E, I, I, seed=5, expert_type=kind))
        with gguf.parse_gguf_index(p) as g:
            b.upload_layer_gguf(0, (H, E, K, I, I), g)
        call = b.forward_gguf_device
    x = torch.randn((eager, H), generator=torch.Generator().manual_seed(eager)).bfloat16().float()
    xd, yd = x.cuda(), torch.zeros((eager, H), device="cuda")
    ids = torch.zeros((eager, K), dtype=torch.int32, device="cuda")
    probs = torch.zeros((eager, K), device="cuda")
    shg = torch.zeros(eager, device="cuda")

    def run(T, y):
        args = (0, xd.data_ptr(), T, y.data_ptr(), ids.data_ptr(), probs.data_ptr())
        call(*args, shg.data_ptr()) if kind == "q4" else call(*args)

    # (a first GGUF call without shared-gate output makes that buffer too)
    run(eager, yd)
    b.sync()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    out = torch.zeros((captured, H), device="cuda")
    torch.cuda.synchronize()
    b.set_stream(s.cuda_stream)
    try:
        with torch.cuda.graph(g, stream=s):
            run(captured, out)
    finally:
        b.set_stream(None)
    b.sync()
    ref = torch.zeros_like(out)
    run(captured, ref)
    b.sync()
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), ref.cpu().numpy())
        run(eager, yd)
        b.sync()
    del g
    b.close()
