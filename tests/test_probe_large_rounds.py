"""Probe rounds with more rows than the LDS stage (GPU tests): one row per match,
a few duplicates per key, and more duplicates than a wave's share of the stage
holds for one key group; whole and cut off by the row capacity."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(), dict(radix_bits=2), dict(radix_bits=2, tile=4096)])
@pytest.mark.parametrize("dup", [1, 2, 5, 40])
@pytest.mark.parametrize("cut", [False, True])
def test_rows_of_large_rounds(gpu_ctx, kw, dup, cut):
    import torch
    rng = np.random.default_rng(dup)
    n_r, n_s = 8000, 30_011
    rk = (np.arange(n_r, dtype=np.uint32) // np.uint32(dup)) * np.uint32(2654435761)
    rv = rng.permutation(n_r).astype(np.uint32)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    hit = rng.random(n_s) < 0.7
    sk[hit] = rk[rng.integers(0, n_r, int(hit.sum()))]
    sv = np.arange(n_s, dtype=np.uint32)
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in (rk, rv, sk, sv)]
    torch.cuda.synchronize()
    print(f"[large rounds] dup={dup} cut={cut} {kw}", flush=True)
    scale = 1.0 if cut and dup > 1 else dup + 1.0
    p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, answer_scale=scale, **kw)
    res = gpu_ctx.join(p, *dev)
    n, k, a, b = O.cpu_join(rk, rv, sk, sv)
    assert res.match_count == n and res.truncated == (n > res.capacity)
    got = O.sort_rows(*gpu_ctx.rows_to_host(res))
    expect = O.sort_rows(k, a, b)
    if not res.truncated:
        assert np.array_equal(got, expect)
    else:
        # rows_written distinct rows of the join
        assert len(got) == res.capacity
        as_set = {tuple(r) for r in expect.tolist()}
        assert len({tuple(r) for r in got.tolist()} & as_set) == len(got)
