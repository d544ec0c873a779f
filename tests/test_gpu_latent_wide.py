"""LatentMoE layers whose latent width is above the hidden size: in prefill the routed rows
(latent floats each) and the shared expert's rows (hidden floats each) share one buffer and
are written on two streams; decode calls of one to eight tokens beside them.  On the library's shared expert (bf16 rows, 2 * n_shared * inter
<= hidden) and on the framework's own, in the exact and the MXFP8 mode, against the oracle
(ko_moe, ko_moe_mx).  Relative L2 below 2e-5, the activations' 2^-17 (hi + lo) on each of the
five products and fp32 sums of up to 768 terms (their square root times 2^-24 in practice)."""
import numpy as np
import pytest

import synth
from gpu_util import bank_layer, dev_forward, say
from test_gpu_mx import check_mx

pytestmark = pytest.mark.gpu

SHAPES = [(128, 768, 128, 2), (256, 384, 128, 1)]        # hidden, latent, inter, n_shared


def wide_layer(H, LT, I, NS):
    return synth.Layer(H=H, E=8, K=3, I=I, n_shared=NS, latent=LT, latent_norm=1, situ_b1=4.0,
                       situ_b2=25.0, routed_scale=1.0, seed=23)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("H,LT,I,NS", SHAPES)
def test_latent_above_hidden(torch, k3x, H, LT, I, NS, bf16):
    L = wide_layer(H, LT, I, NS)
    layer = bank_layer(k3x, L)
    for T in (1, 2, 5, 8, 9, 40, 200):
        x = L.x(T, bf16=bf16, stream_sub=T)
        o, oi, _, _ = L.oracle_moe(x)
        out, idx, _ = dev_forward(torch, k3x, layer, x, bf16=bf16)
        err = synth.rel_l2(out, o)
        say(f"  H={H} latent={LT} shared={NS} bf16={bf16} T={T}: rel_l2 {err:.2e}")
        assert np.array_equal(idx, oi)
        assert err < 2e-5
    layer.close()


@pytest.mark.parametrize("H,LT,I,NS", SHAPES)
def test_latent_above_hidden_mx(torch, k3x, H, LT, I, NS):
    L = wide_layer(H, LT, I, NS)
    layer = bank_layer(k3x, L)
    layer.set_prefill_mode(k3x.K3X_PREFILL_MXFP8)
    for T in (9, 200):
        x = L.x(T, bf16=True, stream_sub=T)
        o, oi, _, _ = L.oracle_moe_mx(x)
        out, idx, _ = dev_forward(torch, k3x, layer, x, bf16=True)
        assert np.array_equal(idx, oi)
        check_mx(out, o, f"MXFP8, H={H} latent={LT} T={T}")
    layer.close()
