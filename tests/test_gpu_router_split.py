"""The prefill router over split K (k3x_moe_route past 8 tokens and every prefill call):
experts and weights bit for bit the oracle's (k3_router, k3_ops.c:1624-1719), at the edges of
its tiles (32 experts, 16 or 32 tokens), of its segments (fewer 64-element chunks than waves,
uneven ones) and of its parts, on rows that its bound proves and rows that it does not.
Renorm off and scale 1: the weights are the sigmoid scores themselves."""
import numpy as np
import pytest

import oracle_lib as ol
import synth
from gpu_util import layer_cfg, say

pytestmark = pytest.mark.gpu


def oracle_routes(L, x):
    T, H = x.shape
    ri = np.empty((T, L.K), np.int32)
    rw = np.empty((T, L.K), np.float32)
    for t in range(T):
        xt = np.ascontiguousarray(x[t])
        ol.oracle().ko_router(ol.ptr(ri[t], ol.I32P), ol.ptr(rw[t], ol.F32P),
                              ol.ptr(xt, ol.F32P), ol.ptr(L.gate, ol.F32P),
                              ol.ptr(L.bias, ol.F32P), H, L.E, L.K, L.renorm, L.routed_scale)
    return ri, rw


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("H,E,K,T", [
    (128, 33, 1, 9),          # two chunks for four waves; parts would not fit: one part
    (384, 32, 4, 16),         # one expert tile, one token tile of 16
    (640, 97, 8, 17),         # ten chunks over uneven segments, a token past the tile
    (2176, 130, 6, 33),       # 34 chunks, several parts
    (7168, 384, 8, 40),       # the K2 router, eight parts
    (7168, 896, 16, 70),      # the K3 router
    (1024, 1000, 2, 1600),    # more tiles than workgroups wanted: one part
])
def test_split_router_bitwise(torch, k3x, H, E, K, T, bf16):
    say(f"case: split router H={H} E={E} K={K} T={T} bf16={bf16}")
    L = synth.Layer(H=H, E=E, K=K, I=128, n_shared=0, seed=91, renorm=0, routed_scale=1.0)
    p = H // 2
    L.gate[:, p + 1] = L.gate[:, p]
    x = L.x(T, bf16=bf16, stream_sub=91)
    # a pair that cancels but first rounds away low bits of the sums it meets (2^28: some
    # logits of the row are proven, others not), rows of zeros (logits of exactly 0: every
    # score ties), of one large element, of tiny elements, and of infinities and NaN
    for t in range(0, T, 5):
        x[t, p], x[t, p + 1] = 2.0 ** 28, -(2.0 ** 28)
    x[1] = 0.0
    x[2] = 0.0
    x[2, H - 1] = 2.0 ** 20
    x[3] *= 2.0 ** -100
    x[4, 0] = np.inf
    x[6, 0], x[6, H - 1] = np.inf, -np.inf
    x[7, 5] = np.nan
    layer = k3x.MoELayer.from_bank(layer_cfg(k3x, L), L.gate, L.bias, [L.expert(0)] * E)
    xt = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    xt = xt.to(torch.bfloat16) if bf16 else xt
    idx = torch.full((T, K), -7, dtype=torch.int32, device="cuda")
    wt = torch.full((T, K), -7.0, dtype=torch.float32, device="cuda")
    layer.route(idx.data_ptr(), wt.data_ptr(), xt.data_ptr(), T,
                k3x.K3X_BF16 if bf16 else k3x.K3X_F32, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ri, rw = oracle_routes(L, x)
    bad = np.nonzero((idx.cpu().numpy() != ri).any(1))[0]
    assert bad.size == 0, (bad[:8], idx.cpu().numpy()[bad[:2]], ri[bad[:2]])
    # the weights: each selected pair's chain in double (accumulate adds in order), rounded to
    # float, then the device's sigmoid: exp in double rounded once.  (The oracle's scores go
    # through the host's expf, which is not correctly rounded: a pair in a few thousand is one
    # unit in the last place away.)
    with np.errstate(invalid="ignore", over="ignore"):
        for t in range(T):
            terms = L.gate[ri[t]].astype(np.float64) * x[t].astype(np.float64)
            f = np.add.accumulate(terms, axis=1)[:, -1].astype(np.float32)
            s = np.float32(1) / (np.float32(1) + np.exp(-f.astype(np.float64)).astype(np.float32))
            want = np.where(np.isnan(f), np.float32(0), s)
            got = wt[t].cpu().numpy()
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (t, got, want)
    assert np.abs(wt.cpu().numpy() - rw).max() <= 2.0 ** -23
    layer.close()


@pytest.mark.parametrize("E,K", [(200, 8), (100, 64), (64, 64), (896, 16)])
@pytest.mark.parametrize("T", [1, 3, 20])
def test_equal_choices(torch, k3x, E, K, T):
    """More equal choices than the selection's list holds, K up to every expert: rows of
    zeros (every score 0.5) over biases of a few values, the lower index first; a row of
    N(0, 1) beside them."""
    say(f"case: equal choices E={E} K={K} T={T}")
    L = synth.Layer(H=256, E=E, K=K, I=128, n_shared=0, seed=92)
    L.bias[:] = np.where(np.arange(E) % 3 == 1, 0.25, 0.0).astype(np.float32)
    L.bias[E - 1] = -np.inf
    x = L.x(T, bf16=False, stream_sub=92)
    x[: max(1, T - 1)] = 0.0
    layer = k3x.MoELayer.from_bank(layer_cfg(k3x, L), L.gate, L.bias, [L.expert(0)] * E)
    xt = torch.from_numpy(x).cuda()
    out = torch.empty_like(xt)
    idx = torch.full((T, K), -7, dtype=torch.int32, device="cuda")
    wt = torch.full((T, K), -7.0, dtype=torch.float32, device="cuda")
    layer.forward(out.data_ptr(), xt.data_ptr(), T, k3x.K3X_F32, 0, idx.data_ptr(), wt.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    layer.check()
    ri, rw = oracle_routes(L, x)
    assert np.array_equal(idx.cpu().numpy(), ri)
    assert np.abs(wt.cpu().numpy() - rw).max() <= 2.0 ** -22
    layer.close()
