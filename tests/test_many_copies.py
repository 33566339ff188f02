"""Build keys with many copies (GPU tests): their rows whole and cut off by the row
capacity in every kernel form, and the time of rows that are written and of rows past
the capacity, which are counted only."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


def relations(n_r, n_s, copies, match, seed):
    rng = np.random.default_rng(seed)
    rk = (np.arange(n_r, dtype=np.uint32) // np.uint32(copies)) * np.uint32(2654435761)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    hit = rng.random(n_s) < match
    sk[hit] = rk[rng.integers(0, n_r, int(hit.sum()))]
    return rng.permutation(rk), np.arange(n_r, dtype=np.uint32), sk, np.arange(n_s, dtype=np.uint32)


def to_dev(host):
    import torch
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    return dev


@pytest.mark.parametrize("kw", [dict(), dict(radix_bits=1), dict(radix_bits=1, tile=4096), dict(radix_bits=6)])
@pytest.mark.parametrize("n_r,n_s,copies,match", [
    (3000, 3000, 12, 1.0), (3000, 3000, 24, 1.0), (3000, 3000, 25, 1.0),   # about the runs that the wave reads
    (3000, 3000, 50, 1.0),
    (8000, 2500, 63, 0.3), (8000, 2500, 64, 0.3), (8000, 2500, 65, 0.3), (8000, 2500, 129, 0.3),   # steps of a run
    (8000, 2500, 4000, 0.01),
    (40_000, 30_000, 100, 0.05),
    (3000, 70_000, 20, 0.3),         # long probe sides
])
def test_rows(gpu_ctx, kw, n_r, n_s, copies, match):
    import torch
    host = relations(n_r, n_s, copies, match, n_r + copies)
    dev = to_dev(host)
    n, k, a, b = O.cpu_join(*host)
    expect = O.sort_rows(k, a, b)
    print(f"[copies] {n_r}x{n_s} copies={copies} rows={n} {kw}", flush=True)
    for cap in (n, n - 1, n // 2, 1000, 1):
        out = [torch.full((cap,), -1, dtype=torch.int32, device="cuda") for _ in range(3)]
        torch.cuda.synchronize()
        p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, **kw)
        res = gpu_ctx.join_noalloc(p, *dev, *out, cap)
        assert res.match_count == n and res.rows_written == min(n, cap)
        rows = O.sort_rows(*(t[:res.rows_written].cpu().numpy().view(np.uint32) for t in out))
        if cap >= n:
            assert np.array_equal(rows, expect)
        else:   # distinct rows of the join
            place = rows[:, 1].astype(np.uint64) << np.uint64(32) | rows[:, 2]
            assert len(np.unique(place)) == cap
            assert np.array_equal(host[0][rows[:, 1]], rows[:, 0]) and np.array_equal(host[2][rows[:, 2]], rows[:, 0])


def probe_ms(ctx, dev, n_r, n_s, scale):
    p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, answer_scale=scale, collect_phase_times=1)
    res = [ctx.join(p, *dev) for _ in range(5)]
    return sorted(r.kernels()["probe"] for r in res)[2], res[0]


def test_time_of_rows_past_the_capacity(gpu_ctx):
    """10 rows per S tuple and room for one: the rest is counted in less than the time of writing them."""
    n = 7_000_000
    host = relations(n, n, 50, 0.2, 1)
    dev = to_dev(host)
    whole, res = probe_ms(gpu_ctx, dev, n, n, 10.5)
    assert not res.truncated
    cut, res = probe_ms(gpu_ctx, dev, n, n, 1.0)
    print(f"[copies] whole {whole:.3f} ms, cut {cut:.3f}", flush=True)
    assert res.truncated and cut < 0.7 * whole


def test_time_of_many_copies(gpu_ctx):
    """15M rows of keys with a thousand copies against 20M rows of one each: within five times as long."""
    n_r, n_s = 6000, 20_000_000
    one, res = probe_ms(gpu_ctx, to_dev(relations(n_r, n_s, 1, 1.0, 2)), n_r, n_s, 1.0)
    assert res.match_count > 19_000_000
    n_s = 300_000
    many, res = probe_ms(gpu_ctx, to_dev(relations(n_r, n_s, 1000, 0.05, 3)), n_r, n_s, 52.0)
    print(f"[copies] one {one:.3f} ms, many {many:.3f} for {res.match_count} rows", flush=True)
    assert not res.truncated and res.match_count > 14_000_000 and many < 5 * one
