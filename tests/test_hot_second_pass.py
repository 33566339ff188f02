"""The second scatter pass where its workgroups are shared by the buckets' sizes (GPU
tests): the partition of relations whose tuples pile up in one bucket or are missing from
most, at the edges of that sharing, and the time of the pass under a hot key."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu

MUL = np.uint32(0x9E3779B1)


def keys(n, hot, seed):
    """hot: the part of the tuples with one key."""
    rng = np.random.default_rng(seed)
    k = rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    k[rng.random(n) < hot] = 77
    return k


@pytest.mark.parametrize("n,kw", [
    (16_384, dict(radix_bits=8, pass1_bits=3)),        # one chunk: one workgroup a bucket
    (16_385, dict(radix_bits=8, pass1_bits=3)),        # two chunks: one workgroup more to share
    (50_001, dict(radix_bits=8, pass1_bits=3)),
    (500_003, dict(radix_bits=8, pass1_bits=1)),
    (500_003, dict(radix_bits=12, pass1_bits=6)),      # one bucket per lane
    (900_001, dict(radix_bits=13, pass1_bits=7)),      # two buckets per lane
    (1_500_007, dict(radix_bits=15, pass1_bits=9)),    # eight per lane
    (1_500_007, dict(radix_bits=15, pass1_bits=4)),    # 2048-way second pass
    (1_500_007, dict(radix_bits=10, pass1_bits=5, scatter_wg=512)),
    (8_000_009, dict(radix_bits=10)),
])
@pytest.mark.parametrize("hot", [0.0, 0.5, 0.999, 1.0])
def test_partition(gpu_ctx, n, kw, hot):
    import torch
    bits = kw["radix_bits"]
    key = keys(n, hot, n)
    val = np.arange(n, dtype=np.uint32)
    dk, dv = (torch.from_numpy(a.view(np.int32)).cuda() for a in (key, val))
    ok, ov = torch.empty_like(dk), torch.empty_like(dv)
    st = torch.empty((1 << bits) + 1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    print(f"[hot second pass] n={n} hot={hot} {kw}", flush=True)
    gpu_ctx.partition(bj.default_params(r_size=n, s_size=n, inputs_on_device=1, **kw), dk, dv, n, ok, ov, st)
    ok, ov, st = ok.cpu().numpy().view(np.uint32), ov.cpu().numpy().view(np.uint32), st.cpu().numpy()
    bucket = (ok * MUL) >> np.uint32(32 - bits)
    assert np.array_equal(st, np.concatenate([[0], np.cumsum(np.bincount((key * MUL) >> np.uint32(32 - bits),
                                                                        minlength=1 << bits))]))
    assert np.all(np.diff(bucket.astype(np.int64)) >= 0)     # in its bucket's range, as the counts agree
    assert np.array_equal(np.sort(ov), val) and np.array_equal(key[ov], ok)   # every tuple once


def test_rows_and_time_under_a_hot_key(gpu_ctx):
    """3M x 4.5M with half of S on one key: 32 workgroups share its bucket, about 17 tiles
    each against four to five without it (eight had 69), so at most some 4.5 times the time."""
    import torch
    n_r, n_s = 3_000_017, 4_500_007
    ms = {}
    for hot in (0, n_s // 2):
        rng = np.random.default_rng(hot)
        rk = np.arange(n_r, dtype=np.uint32) * np.uint32(2654435761)
        sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
        sk[:n_s // 10] = rk[rng.integers(0, n_r, n_s // 10)]
        sk[n_s - hot:] = rk[5]
        host = (rk, np.arange(n_r, dtype=np.uint32), rng.permutation(sk), np.arange(n_s, dtype=np.uint32))
        dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
        torch.cuda.synchronize()
        p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, collect_phase_times=1)
        t = []
        for _ in range(7):
            res = gpu_ctx.join(p, *dev)
            t.append(res.kernels()["scatter2_r"] + res.kernels()["scatter2_s"])
        ms[hot] = sorted(t)[3]
        n, k, a, b = O.cpu_join(*host)
        assert res.match_count == n and np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), O.sort_rows(k, a, b))
    print(f"[hot second pass] {ms}", flush=True)
    assert ms[n_s // 2] < 6.0 * ms[0], ms
