"""The join without a partition (small build sides), through the C ABI (GPU
tests): rows bit-exact against the oracle at the edges of its LDS table chunks
and rounds, both build sides, with and without the filter; the same survivors as
the partitioned join with the same filter."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


def join(ctx, host, dev, **kw):
    p = bj.default_params(r_size=len(host[0]), s_size=len(host[2]), inputs_on_device=1, **kw)
    res = ctx.join(p, *dev)
    return res, O.sort_rows(*ctx.rows_to_host(res))


def to_dev(a):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a, np.uint32).view(np.int32)).cuda()
    return t if t.numel() else torch.zeros(1, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("n_r,n_s,dup", [
    (1, 1, 1), (1, 5000, 1), (0, 100, 1), (100, 0, 1),
    (8191, 1023, 1), (8192, 1025, 1), (8193, 5119, 1),   # one table chunk, then two; S one round or more
    (8192, 3_000_001, 1),                                # long slices of S
    (16_385, 70_000, 1), (200_003, 300_001, 1),
    (300_001, 9000, 1),                                  # S is the build side
    (6000, 40_000, 3), (20_000, 9000, 2),                # duplicate keys
])
@pytest.mark.parametrize("bf", [0, 1])
def test_direct_rows(gpu_ctx, n_r, n_s, dup, bf):
    import torch
    rng = np.random.default_rng(n_r * 7 + n_s)
    rk = (np.arange(n_r, dtype=np.uint32) // np.uint32(dup)) * np.uint32(2654435761) + np.uint32(5)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    if n_r and n_s:
        hit = rng.random(n_s) < 0.6
        sk[hit] = rk[rng.integers(0, n_r, int(hit.sum()))]
    rv, sv = np.arange(n_r, dtype=np.uint32) * 3, np.arange(n_s, dtype=np.uint32) + 7
    host = (rk, rv, sk, sv)
    dev = [to_dev(a) for a in host]
    torch.cuda.synchronize()
    print(f"[direct] |R|={n_r} |S|={n_s} dup={dup} bf={bf}", flush=True)
    kw = dict(use_bf=bf, bf_bits_per_key=10.0, num_hashes=3, answer_scale=4.0)
    res, rows = join(gpu_ctx, host, dev, **kw)
    assert res.kernels()["hist_r"] == 0.0 and res.kernels()["scatter1_s"] == 0.0   # nothing was partitioned
    n, k, a, b = O.cpu_join(*host)
    assert res.match_count == n and res.truncated == 0
    assert np.array_equal(rows, O.sort_rows(k, a, b))
    # the partitioned join of the same relations: the same rows and survivors
    part, prows = join(gpu_ctx, host, dev, radix_bits=6, bf_stage=1 if bf else 0, **kw)
    assert part.s_survivors == res.s_survivors and np.array_equal(prows, rows)
