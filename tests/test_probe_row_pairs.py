"""Rows of several probe rounds of one work item (GPU tests): every number of rounds
from one to six, ragged at both ends of a round, with empty, sparse and full rounds
in every order, and the same cut off by the row capacity."""
import itertools

import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu

INV = pow(0x9E3779B1, -1, 2**32)  # of the radix hash's multiplier


def _keys(bucket, low, bits):
    """The keys whose hash has `bucket` on top and `low` below."""
    h = (np.uint64(bucket) << np.uint64(32 - bits)) | low.astype(np.uint64)
    return (h * np.uint64(INV) & np.uint64(0xFFFFFFFF)).astype(np.uint32)


@pytest.mark.parametrize("tile", [4096, 8192])
@pytest.mark.parametrize("rounds", range(1, 7))
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_rows_of_consecutive_rounds(gpu_ctx, tile, rounds, edge):
    import torch
    bits, n_b = 9, 1500            # 512 sub-buckets: one work item each
    per = tile * 5 // 8            # probe keys of a round
    rng = np.random.default_rng(rounds * 10 + edge)
    rk, sk = [], []
    # one sub-bucket per order of round densities
    for sb, kinds in enumerate(itertools.product((0.0, 0.1, 0.9), repeat=min(rounds, 3))):
        low = rng.choice(1 << 23, n_b + per, replace=False)
        rk.append(_keys(sb, low[:n_b], bits))
        miss = _keys(sb, low[n_b:], bits)
        n = rounds * per + edge
        hit = rng.random(n) < np.repeat(np.resize(kinds, rounds + 1), per)[:n]
        sk.append(np.where(hit, rk[-1][rng.integers(0, n_b, n)], miss[rng.integers(0, per, n)]))
    rk, sk = np.concatenate(rk), np.concatenate(sk)
    host = (rk, rng.permutation(rk.size).astype(np.uint32), sk, np.arange(sk.size, dtype=np.uint32))
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    print(f"[row pairs] tile={tile} rounds={rounds} edge={edge} |S|={sk.size}", flush=True)
    n, k, a, b = O.cpu_join(*host)
    expect = O.sort_rows(k, a, b)
    for scale in (1.0, 0.2):
        p = bj.default_params(r_size=rk.size, s_size=sk.size, inputs_on_device=1, radix_bits=bits, tile=tile,
                              answer_scale=scale)
        res = gpu_ctx.join(p, *dev)
        assert res.match_count == n
        got = O.sort_rows(*gpu_ctx.rows_to_host(res))
        if not res.truncated:
            assert np.array_equal(got, expect)
        else:  # as many rows as fit, all of the join, none twice (S's value is its row)
            assert len(got) == res.capacity and len(np.unique(got[:, 2])) == len(got)
            assert np.array_equal(got, expect[np.isin(expect[:, 2], got[:, 2])])
