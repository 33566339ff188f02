"""Both filter kernels at the edges of their tiles and sub-bucket scans (GPU tests):
the filter after S's first pass with up to 64, 512 and 2048 sub-buckets per bucket
and the filter before the partition keep the same tuples, and the rows are the
oracle's."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [3, 4, 5])
@pytest.mark.parametrize("n_s", [1, 4095, 4097, 100_003, 3_000_001])
def test_filter_forms_agree(gpu_ctx, n_s, k):
    import torch
    n_r = 30_000
    rng = np.random.default_rng(n_s + k)
    rk = (np.arange(n_r, dtype=np.uint32) + np.uint32(k)) * np.uint32(2654435761)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    hit = rng.random(n_s) < 0.3
    sk[hit] = rk[rng.integers(0, n_r, int(hit.sum()))]
    rv, sv = rng.permutation(n_r).astype(np.uint32), np.arange(n_s, dtype=np.uint32)
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in (rk, rv, sk, sv)]
    torch.cuda.synchronize()
    n, a, b, c = O.cpu_join(rk, rv, sk, sv)
    expect = O.sort_rows(a, b, c)
    kept = set()
    for stage, s_pass1 in ((1, -1), (2, 8), (2, 4), (2, 3), (2, 2)):
        print(f"[filter tiles] |S|={n_s} k={k} stage={stage} s_pass1={s_pass1}", flush=True)
        p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, use_bf=1, bf_bits_per_key=10.0,
                              num_hashes=k, radix_bits=13, bf_stage=stage, s_pass1_bits=s_pass1)
        res = gpu_ctx.join(p, *dev)
        assert res.match_count == n
        assert np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), expect)
        kept.add(int(res.s_survivors))
    assert len(kept) == 1 and n <= kept.pop() <= n_s
