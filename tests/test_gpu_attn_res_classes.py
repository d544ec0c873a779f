"""k3x_attn_res's launch classes (rows a call, row length, aligned or not) against the oracle."""
import numpy as np
import pytest

import synth
from gpu_util import say
from oracle_lib import F32P, oracle, ptr

pytestmark = pytest.mark.gpu
EPS = 1e-5


@pytest.mark.parametrize("T,n,nb,shift", [
    (1, 2560, 1, 1), (1, 2561, 0, 0), (2, 2688, 3, 1), (256, 129, 2, 0),   # a row a CU
    (257, 132, 3, 0), (300, 3600, 1, 0), (300, 2049, 2, 0), (512, 512, 9, 0),
    (513, 4, 0, 0), (513, 257, 3, 0), (520, 1028, 5, 0), (600, 2048, 1, 0), (513, 2052, 1, 0),
])
def test_attn_res_launch_classes(torch, k3x, T, n, nb, shift):
    say(f"case: attn_res T={T} n={n} nb={nb}, bases {4 * shift} bytes off 16")
    rng = np.random.default_rng(T + n + nb)
    maxb = nb + 1
    blocks = (rng.standard_normal((T, maxb, n)) * rng.uniform(0.2, 5, (T, maxb, 1))).astype(np.float32)
    pref = rng.standard_normal((T, n)).astype(np.float32)
    fold = (rng.standard_normal(n) * 0.05).astype(np.float32)
    want = np.empty_like(pref)
    for t in range(T):
        src = np.ascontiguousarray(np.concatenate([blocks[t, :nb], pref[t:t + 1]]), np.float32)
        oracle().ko_attn_res(ptr(want[t], F32P), ptr(src, F32P), ptr(fold, F32P), nb + 1, n, EPS)

    def dev(a):
        d = torch.empty(a.size + 4, dtype=torch.float32, device="cuda")
        d[shift:shift + a.size] = torch.from_numpy(a.ravel()).cuda()
        return d

    bd, pd, fd, hd = dev(blocks), dev(pref), dev(fold), dev(np.zeros_like(pref))
    h, b, p, f = (d.data_ptr() + 4 * shift for d in (hd, bd, pd, fd))
    k3x.attn_res(h, b, maxb, nb, p, f, n, T, EPS, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = hd[shift:shift + pref.size].cpu().numpy().reshape(T, n)
    # a weight may be one unit in its last place from the oracle's (its exp is the host's expf)
    r = np.linalg.norm((got - want).astype(np.float64), axis=1)
    assert (r < 2.0 ** -22 * np.linalg.norm(want.astype(np.float64), axis=1)).all()
    if nb == 0:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
