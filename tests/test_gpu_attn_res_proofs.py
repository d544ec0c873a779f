"""k3x_attn_res's proofs of a key's float: keys steered to within a chosen distance of the
midpoint of two floats, so that the first bound (sum |p|) fails and the second (the partial
sums' magnitudes) holds, or both fail and only the reference's chain (k3_ops.c:1738-1741)
decides.  The outputs bit for bit the float64 evaluation of the reference's steps: chains by
np.add.accumulate, exp in double rounded once."""
import math

import numpy as np
import pytest

from gpu_util import say

pytestmark = pytest.mark.gpu
EPS = 1e-5


def terms(v, fold):
    """The products of v's key in double (exact), v normalised as the reference does."""
    v64 = v.astype(np.float64)
    ss = np.add.accumulate(v64 * v64)[-1]
    inv = np.float32(1.0 / math.sqrt(ss / v.size + float(np.float32(EPS))))
    return (v * inv).astype(np.float64) * fold.astype(np.float64), (v * inv).astype(np.float64)


def chain(p):
    return np.float32(np.add.accumulate(p)[-1])


def tree(p):
    """The kernel's order for rows of whole 512-float pieces: float4s dealt to 128 lanes, four
    sums a lane, the waves' trees, the two halves."""
    a = np.add.accumulate(p.reshape(-1, 128, 4), axis=0)[-1]
    s = (a[:, 0] + a[:, 1]) + (a[:, 2] + a[:, 3])
    s = s.reshape(2, 64)
    for off in (32, 16, 8, 4, 2, 1):
        s = s + s[:, np.arange(64) ^ off]
    return np.float32(s[0, 0] + s[1, 0])


def bounds(p):
    """The kernel's two bounds of a key, with sum |p| as it is."""
    n, ap = p.size, np.abs(p).sum()
    first = (n + n // 128 + 16) * 2.0 ** -53 * ap
    return first, (np.abs(np.add.accumulate(p)).sum() + 2 * (n // 512 + 16) * ap) * 2.0 ** -53


def steer(v, fold, at, off):
    """fold with the three columns of `at` set so that v's key lies off(bounds) past a midpoint
    of two floats, to about 1e-20."""
    fold = fold.copy()
    fold[at] = 0.0
    p, vi = terms(v, fold)
    key = np.float32(math.fsum(p))
    mid = (float(key) + float(np.nextafter(key, np.float32(np.inf)))) / 2.0
    d = off(bounds(p))
    for c in at:
        r = math.fsum([mid, d] + list(-p))
        fold[c] = np.float32(r / vi[c])
        p[c] = vi[c] * float(fold[c])
    return fold


@pytest.mark.parametrize("T", [1, 300, 520])
@pytest.mark.parametrize("n", [1024, 2048, 7168])
def test_attn_res_key_proofs(torch, k3x, T, n):
    rng = np.random.default_rng(n)
    kinds = {"second proof": 0, "chain": 0}
    differ = 0
    for trial in range(12):
        v = rng.standard_normal(n).astype(np.float32)
        w = rng.standard_normal(n).astype(np.float32)
        fold = (rng.standard_normal(n) * 0.05).astype(np.float32)
        at = [3, n // 2, n - 2]
        v[at] = (1.0, -1.5, 0.75)
        if trial % 3 == 0:                       # between the bounds, either side
            s = 1.0 if trial % 2 else -1.0
            fold = steer(v, fold, at, lambda b: s * math.sqrt(b[0] * b[1]))
        else:                                    # on the midpoint
            fold = steer(v, fold, at, lambda b: 0.0)
        p, _ = terms(v, fold)
        k = np.float64(math.fsum(p))
        lo = np.float32(k)
        nb_ = np.nextafter(lo, np.float32(np.inf if float(lo) < k else -np.inf))
        dist = abs(k - (float(lo) + float(nb_)) / 2.0)
        b1, b2 = bounds(p)
        assert dist < b1
        kinds["second proof" if dist > 1.5 * b2 else "chain"] += 1
        differ += chain(p) != tree(p)
        # the reference's steps with the chains' keys
        src = [v, w]
        sc = np.array([chain(terms(s_, fold)[0]) for s_ in src], np.float32)
        e = np.exp((sc - sc.max()).astype(np.float64)).astype(np.float32)
        z = float(e[0]) + float(e[1])
        pr = (e.astype(np.float64) / z).astype(np.float32)
        want = np.zeros(n, np.float32)
        for s_, q in zip(src, pr):
            want = want + q * s_
        bd = torch.from_numpy(v).cuda().repeat(T, 1).contiguous()
        pd = torch.from_numpy(w).cuda().repeat(T, 1).contiguous()
        fd = torch.from_numpy(fold).cuda()
        hd = torch.empty_like(pd)
        k3x.attn_res(hd.data_ptr(), bd.data_ptr(), 1, 1, pd.data_ptr(), fd.data_ptr(), n, T, EPS,
                     torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = hd.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), np.broadcast_to(want, got.shape).view(np.uint32)), trial
    say(f"  n={n}: {kinds}, keys whose float the kernel's order alone gets wrong: {differ}")
    # teeth: both outcomes are met, and a bound too small would let a wrong float through
    assert kinds["second proof"] >= 3 and kinds["chain"] >= 6 and differ >= 2
