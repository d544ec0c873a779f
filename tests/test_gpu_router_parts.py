"""The prefill router at sizes past one tile a CU, where a tile's K goes to one to four
workgroups (k3x_moe_route): experts bit for bit the oracle's (k3_router, k3_ops.c:1624-1719)
and weights bit for bit the sigmoid of the reference's chain.  Every third row carries a pair
that cancels but first rounds away low bits of the sums it meets: the bound cannot prove those
rows' logits, and the test counts the selected ones whose float any sum over K segments gets
wrong, so only the chain gives the weights."""
import numpy as np
import pytest

import synth
from gpu_util import layer_cfg, say
from test_gpu_router_split import oracle_routes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,K,T,parts", [
    (1024, 384, 8, 1500, 4), (768, 384, 8, 1700, 3), (1024, 384, 8, 1000, 2),
    (1024, 896, 16, 300, 4), (512, 128, 4, 2048, 1), (256, 896, 16, 600, 1),
])
def test_router_parts_bitwise(torch, k3x, H, E, K, T, parts):
    say(f"case: router H={H} E={E} K={K} T={T}, {parts} parts")
    L = synth.Layer(H=H, E=E, K=K, I=128, n_shared=0, seed=93, renorm=0, routed_scale=1.0)
    p = H // 2
    L.gate[:, p + 1] = L.gate[:, p]
    x = L.x(T, bf16=True, stream_sub=93)
    # 2^36 times a weight of 0.02 is about 2^30, whose double steps of 2^-22 round away more
    # than the last bit of a float logit near 1: an order that lets the pair meet another sum
    # gives another float, for all but a few
    x[::3, p], x[::3, p + 1] = 2.0 ** 36, -(2.0 ** 36)
    layer = k3x.MoELayer.from_bank(layer_cfg(k3x, L), L.gate, L.bias, [L.expert(0)] * E)
    xt = torch.from_numpy(x).cuda().to(torch.bfloat16)
    idx = torch.full((T, K), -7, dtype=torch.int32, device="cuda")
    wt = torch.full((T, K), -7.0, dtype=torch.float32, device="cuda")
    layer.route(idx.data_ptr(), wt.data_ptr(), xt.data_ptr(), T, k3x.K3X_BF16,
                torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ri, _ = oracle_routes(L, x)
    assert np.array_equal(idx.cpu().numpy(), ri)
    got = wt.cpu().numpy()
    wrong = 0
    for t in range(T):
        terms = L.gate[ri[t]].astype(np.float64) * x[t].astype(np.float64)
        f = np.add.accumulate(terms, axis=1)[:, -1].astype(np.float32)
        s = np.float32(1) / (np.float32(1) + np.exp(-f.astype(np.float64)).astype(np.float32))
        assert np.array_equal(got[t].view(np.uint32), s.view(np.uint32)), (t, got[t], s)
        if t % 3 == 0:
            seg = terms.reshape(K, 4, -1).sum(axis=2).sum(axis=1).astype(np.float32)
            wrong += int((seg != f).sum())
    say(f"  selected logits that four segments' sums get wrong: {wrong}")
    assert wrong >= T // 10
    layer.close()
