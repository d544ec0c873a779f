"""k3x_attn_res at the edges of its forms: row lengths around the loads' pieces (a
multiple of 4 or not, one piece, one float4 past a step of 3584 floats), unaligned rows,
one source up to the most it takes (more sources than two waves each cover at once),
against the oracle's (k3_attn_res, k3_ops.c:1722-1753)."""
import numpy as np
import pytest

import synth
from gpu_util import say
from oracle_lib import F32P, oracle, ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nb,shift", [(4, 0, 0), (128, 1, 0), (130, 2, 0), (3584, 7, 0),
                                        (3588, 8, 0), (7168, 15, 0), (7168, 5, 1), (512, 63, 0)])
def test_attn_res_forms(torch, k3x, n, nb, shift):
    say(f"case: attn_res n={n} nb={nb}, bases {4 * shift} bytes off 16")
    T, maxb, eps = 3, nb + 1, 1e-5
    rng = np.random.default_rng(n + nb)
    blocks = (rng.standard_normal((T, maxb, n)) * rng.uniform(0.2, 5, (T, maxb, 1))).astype(np.float32)
    pref = rng.standard_normal((T, n)).astype(np.float32)
    fold = (rng.standard_normal(n) * 0.05).astype(np.float32)
    want = np.empty_like(pref)
    for t in range(T):
        src = np.ascontiguousarray(np.concatenate([blocks[t, :nb], pref[t:t + 1]]), np.float32)
        oracle().ko_attn_res(ptr(want[t], F32P), ptr(src, F32P), ptr(fold, F32P), nb + 1, n, eps)

    def dev(a):
        d = torch.empty(a.size + 4, dtype=torch.float32, device="cuda")
        d[shift:shift + a.size] = torch.from_numpy(a.ravel()).cuda()
        return d

    bd, pd, fd, hd = dev(blocks), dev(pref), dev(fold), dev(np.zeros_like(pref))
    h, b, p, f = (d.data_ptr() + 4 * shift for d in (hd, bd, pd, fd))
    k3x.attn_res(h, b, maxb, nb, p, f, n, T, eps, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = hd[shift:shift + pref.size].cpu().numpy().reshape(T, n)
    # the softmax's exp is rounded once from double, the oracle's is the host's expf: a
    # weight may be one unit in its last place away, every other bit is the oracle's
    assert synth.rel_l2(got, want) < 2.0 ** -22
    if nb == 0:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
