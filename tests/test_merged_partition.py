"""R and S partitioned by the same launches, the probe planned in the second pass,
and finely sliced probe sides of few sub-buckets (GPU tests): rows against the
oracle, and the allocation-free join at sizes where only one set of partition
buffers fits its scratch array."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


def inputs(n_r, n_s, match, seed, hot=0):
    rng = np.random.default_rng(seed)
    rk = rng.permutation(n_r).astype(np.uint32) * np.uint32(2654435761) + np.uint32(11)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    hit = rng.random(n_s) < match
    sk[hit] = rk[rng.integers(0, n_r, int(hit.sum()))]
    sk[:hot] = rk[0]
    return rk, np.arange(n_r, dtype=np.uint32), sk, np.arange(n_s, dtype=np.uint32)


def to_dev(host):
    import torch
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    return dev


@pytest.mark.parametrize("n_r,n_s,kw", [
    (1, 70_000, dict(radix_bits=3)),                                   # one chunk against several
    (70_000, 1, dict(radix_bits=9)),
    (50_000, 60_000, dict(radix_bits=7)),                              # one pass on both sides
    (50_000, 60_000, dict(radix_bits=12, pass1_bits=2, s_pass1_bits=9)),
    (50_000, 60_000, dict(radix_bits=12, pass1_bits=12 - 1, s_pass1_bits=12 - 11)),
    (300_000, 200_000, dict(radix_bits=15)),
    (300_000, 200_000, dict(radix_bits=10, pass1_bits=10)),            # one pass on R only: not merged
    (60_000, 90_000, dict(radix_bits=9, use_bf=1, bf_stage=2)),
    (60_000, 90_000, dict(radix_bits=9, use_bf=1, bf_stage=2, s_pass1_bits=9)),
    (60_000, 90_000, dict(radix_bits=9, use_bf=1, bf_stage=2, scatter_wg=512)),
    (20_000, 3_000_001, dict(radix_bits=1)),                           # few sub-buckets, long probe sides
    (3_000_001, 20_000, dict(radix_bits=2)),
    (20_000, 3_000_001, dict(radix_bits=3, tile=4096)),
])
@pytest.mark.parametrize("hot", [0, 20_000])
def test_merged_rows(gpu_ctx, n_r, n_s, kw, hot):
    host = inputs(n_r, n_s, 0.3, n_r + n_s, min(hot, n_s))
    dev = to_dev(host)
    print(f"[merged] |R|={n_r} |S|={n_s} hot={hot} {kw}", flush=True)
    n, k, a, b = O.cpu_join(*host)
    for times in (0, 1):
        p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, collect_phase_times=times, **kw)
        res = gpu_ctx.join(p, *dev)
        assert res.match_count == n
        assert np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), O.sort_rows(k, a, b))
    ks = res.kernels()
    assert min(ks["hist_r"], ks["hist_s"], ks["scatter1_r"], ks["scatter1_s"], ks["probe"]) > 0
    assert res.phases()["total"] >= ks["probe"]


def test_noalloc_without_room_for_both(gpu_ctx):
    import torch
    n = 9_000_000          # one set of partition buffers fits 256 MiB, S's own beside it does not
    host = inputs(n, n, 0.1, 5)
    dev = to_dev(host)
    outs = [torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    p = bj.default_params(r_size=n, s_size=n, inputs_on_device=1)
    res = gpu_ctx.join_noalloc(p, *dev, *outs, n)
    m = res.rows_written
    k, a, b = (t[:m].cpu().numpy().view(np.uint32) for t in outs)
    rk, _, sk, _ = host
    assert m == res.match_count and np.array_equal(rk[a], k) and np.array_equal(sk[b], k)
    assert np.array_equal(np.sort(b), np.nonzero(np.isin(sk, rk))[0].astype(np.uint32))
