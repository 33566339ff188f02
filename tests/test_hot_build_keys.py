"""Small joins whose build side is dominated by one key (GPU tests): the join without a
partition gives up there and the relations are joined by partitions after all, with
every row once, in bj_join and in bj_join_noalloc, with and without the filter, whole
and cut off by the row capacity; below that the join stays without a partition."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu

HOT = np.uint32(77)


def relations(n_r, n_s, hot_r, hot_s):
    """hot_r, hot_s: tuples of R and of S with the hot key."""
    rng = np.random.default_rng(n_r + hot_r + hot_s)
    rk = np.arange(n_r, dtype=np.uint32) * np.uint32(2654435761) + np.uint32(1)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    sk[:n_s // 10] = rk[rng.integers(max(hot_r, 1), n_r, n_s // 10)]
    rk[:hot_r] = HOT
    sk[n_s - hot_s:] = HOT
    host = (rng.permutation(rk), np.arange(n_r, dtype=np.uint32), rng.permutation(sk), np.arange(n_s, dtype=np.uint32))
    return host


@pytest.mark.parametrize("n_r,n_s,hot_r,hot_s,by_partitions", [
    (300_000, 200_000, 1, 60_000, True),      # S is the build side
    (300_000, 200_000, 0, 180_000, True),     # its hot key has no match
    (200_000, 300_000, 100_000, 2, True),     # R is the build side
    (20_001, 20_003, 19_000, 1, True),        # three chunks
    (300_000, 200_000, 1, 5_000, False),      # about 200 copies in a chunk
    (8192, 100_000, 8000, 1, False),          # one chunk: the partitioned join's table would be the same
])
@pytest.mark.parametrize("bf", [0, 1])
def test_hot_key_on_the_build_side(gpu_ctx, n_r, n_s, hot_r, hot_s, by_partitions, bf):
    import torch
    host = relations(n_r, n_s, hot_r, hot_s)
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    print(f"[hot build] |R|={n_r} |S|={n_s} hot={hot_r},{hot_s} bf={bf}", flush=True)
    n, k, a, b = O.cpu_join(*host)
    expect = O.sort_rows(k, a, b)
    kw = dict(r_size=n_r, s_size=n_s, inputs_on_device=1, use_bf=bf, bf_bits_per_key=10.0, num_hashes=3)
    for timing in (0, 1):
        p = bj.default_params(answer_scale=2.0, collect_phase_times=timing, **kw)
        for _ in range(2):
            res = gpu_ctx.join(p, *dev)
            assert res.match_count == n and not res.truncated
            assert np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), expect)
    if not (bf and hot_s == 180_000):   # (the filter drops that S side's hot key)
        assert (res.kernels()["hist_r"] > 0.0) == by_partitions, res.kernels()
    assert res.phases()["total"] >= sum(res.kernels()[x] for x in ("hist_r", "probe"))
    part = gpu_ctx.join(bj.default_params(answer_scale=2.0, radix_bits=6, bf_stage=1 if bf else 0, **kw), *dev)
    assert part.s_survivors == res.s_survivors
    # into the caller's arrays, whole and with room for half the rows
    out = [torch.empty(n + 1, dtype=torch.int32, device="cuda") for _ in range(3)]
    for cap in (n + 1, n // 2):
        res = gpu_ctx.join_noalloc(bj.default_params(**kw), *dev, *out, cap)
        assert res.match_count == n and res.rows_written == min(n, cap) and res.truncated == (cap < n)
        rows = O.sort_rows(*(t[:res.rows_written].cpu().numpy().view(np.uint32) for t in out))
        if cap > n:
            assert np.array_equal(rows, expect)
        else:
            assert len(np.unique(rows, axis=0)) == cap and np.isin(rows[:, 2], expect[:, 2]).all()
