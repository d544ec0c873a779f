"""Prefill calls below four rows an expert, where one tile class serves every expert: the edge
of one column block and several, for an expert that every token chooses beside many of a few
rows and many of none (200 experts, top 4).  K2 and latent form, fp32 and bf16 rows, exact and
MXFP8 mode, against the oracle.  Relative L2 below 2e-5 in the exact mode, the activations'
2^-17 (hi + lo) on each product and fp32 sums of up to 384 terms."""
import numpy as np
import pytest

import synth
from gpu_util import bank_layer, dev_forward, say
from test_gpu_mx import check_mx

pytestmark = pytest.mark.gpu
E, K = 200, 4


def busy_layer(form):
    kw = dict(H=256, E=E, K=K, I=384, seed=29)
    if form == "latent":
        L = synth.Layer(latent=128, latent_norm=1, n_shared=1, situ_b1=4.0, situ_b2=25.0,
                        routed_scale=1.0, **kw)
    else:
        L = synth.Layer(**kw)
    L.bias[:] = 0.0
    L.bias[7] = 3.0
    return L


# tokens: one column block of the busy expert (16 fp32 or latent, 32 bf16 and MXFP8 rows), one
# row past it, past two, four and six; all below 4 E / K = 200
TOKENS = (9, 16, 17, 32, 33, 65, 97, 199)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("form", ["k2", "latent"])
def test_one_class(torch, k3x, form, bf16):
    L = busy_layer(form)
    layer = bank_layer(k3x, L)
    for T in TOKENS:
        assert T * K < 4 * E
        x = L.x(T, bf16=bf16, stream_sub=290 + T)
        o, oi, _, _ = L.oracle_moe(x)
        assert (oi[:, 0] == 7).all()
        out, idx, _ = dev_forward(torch, k3x, layer, x, bf16=bf16)
        err = synth.rel_l2(out, o)
        say(f"  {form} bf16={bf16} T={T}: rel_l2 {err:.2e}")
        assert np.array_equal(idx, oi)
        assert err < 2e-5
    layer.close()


@pytest.mark.parametrize("form", ["k2", "latent"])
def test_one_class_mx(torch, k3x, form):
    L = busy_layer(form)
    layer = bank_layer(k3x, L)
    layer.set_prefill_mode(k3x.K3X_PREFILL_MXFP8)
    for T in (9, 32, 33, 65, 199):
        x = L.x(T, bf16=True, stream_sub=290 + T)
        o, oi, _, _ = L.oracle_moe_mx(x)
        out, idx, _ = dev_forward(torch, k3x, layer, x, bf16=True)
        assert np.array_equal(idx, oi)
        check_mx(out, o, f"MXFP8 {form} T={T}")
    layer.close()
