"""The routed prefill GEMMs at the edges of their tile classes: layers whose tokens all choose
every expert (top-k of all experts), so that each expert's segment has exactly T rows, at T
around the classes' limits (16, 32, 48, 64, 96 rows a tile) and past one column block; widths
whose quads do not fill a super-quad or a row block; K2 and latent forms, fp32 and bf16 rows,
with and without a shared expert.  Against the oracle (ko_moe): relative L2 below 2e-5, the
activations' 2^-17 (hi + lo) on each of the three products and fp32 sums of up to 640 terms
(640 x 2^-24 = 4e-5 at worst, their square root in practice)."""
import numpy as np
import pytest

import synth
from gpu_util import bank_layer, dev_forward, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["k2", "k2-noshared", "latent"])
@pytest.mark.parametrize("bf16", [False, True])
def test_tile_class_edges(torch, k3x, form, bf16):
    kw = dict(H=640, E=4, K=4, I=384, seed=17)
    if form == "latent":
        L = synth.Layer(latent=384, latent_norm=1, n_shared=2, situ_b1=4.0, situ_b2=25.0,
                        routed_scale=1.0, **kw)
    else:
        L = synth.Layer(n_shared=0 if form == "k2-noshared" else 1, **kw)
    layer = bank_layer(k3x, L)
    for T in (9, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 193):
        x = L.x(T, bf16=bf16, stream_sub=170 + T)
        o, oi, ow, _ = L.oracle_moe(x)
        out, idx, wt = dev_forward(torch, k3x, layer, x, bf16=bf16)
        err = synth.rel_l2(out, o)
        say(f"  {form} bf16={bf16} T={T}: rel_l2 {err:.2e}")
        assert np.array_equal(idx, oi)
        assert err < 2e-5
    layer.close()


def test_one_expert_takes_every_token(torch, k3x):
    """The most uneven call: one expert with every token's first slot, the others spread (a
    segment of many column blocks beside many of a few rows)."""
    L = synth.Layer(H=256, E=64, K=2, I=256, seed=18)
    L.bias[:] = 0.0
    L.bias[5] = 3.0
    layer = bank_layer(k3x, L)
    T = 500
    x = L.x(T, bf16=True, stream_sub=18)
    o, oi, ow, _ = L.oracle_moe(x)
    out, idx, wt = dev_forward(torch, k3x, layer, x, bf16=True)
    assert (oi[:, 0] == 5).all() and np.array_equal(idx, oi)
    assert synth.rel_l2(out, o) < 2e-5
    layer.close()


@pytest.mark.parametrize("E,K,T,H,I,bf16", [(1, 1, 17, 256, 256, False), (3, 2, 9, 128, 256, True),
                                            (2, 2, 16, 128, 128, False), (5, 1, 93, 384, 128, False),
                                            (4, 1, 33, 128, 128, True)])
def test_few_experts(torch, k3x, E, K, T, H, I, bf16):
    """Calls whose launch grids, rounded up to the XCDs, exceed the tile table: the table is
    held against the tiles themselves."""
    L = synth.Layer(H=H, E=E, K=K, I=I, seed=19)
    layer = bank_layer(k3x, L)
    x = L.x(T, bf16=bf16, stream_sub=19)
    o, oi, _, _ = L.oracle_moe(x)
    out, idx, _ = dev_forward(torch, k3x, layer, x, bf16=bf16)
    assert np.array_equal(idx, oi)
    assert synth.rel_l2(out, o) < 2e-5
    layer.close()
