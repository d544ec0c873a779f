"""The device memory a layer's prefill buffers take (k3x_moe_layer_reserve)."""
import pytest

import synth
from gpu_util import say, synth_layer

pytestmark = pytest.mark.gpu


def test_reserve_bytes(torch, k3x):
    """2048 tokens of a layer with the K2 layer's widths and few experts: per (token, slot) the
    activations (inter floats), an output row (hidden floats) and the MXFP8 codes and scales
    (hidden bytes and a 32nd), per token two rows (hidden floats: x's and the shared expert's)
    and the shared activations; 5% for the index tables and the allocator's rounding.  fp32
    rows of every (token, slot) in place of the codes would pass it by a third."""
    H, I, K, T = 7168, 2048, 8, 2048
    L = synth.Layer(H=H, E=16, K=K, I=I, seed=3)
    layer = synth_layer(k3x, L)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    layer.reserve(T)
    used = before - torch.cuda.mem_get_info()[0]
    want = T * (K * (I * 4 + H * 4 + H * 33 // 32) + 2 * H * 4 + I * 4)
    say(f"  reserved {used} bytes, {want} for the rows")
    assert 0 < used < 1.05 * want
    layer.close()
