"""Dealing the probe's work items to its workgroups (GPU tests): item counts below,
at and above one claim per workgroup, with empty and sliced sub-buckets between."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hot", [0, 60_000])
@pytest.mark.parametrize("bits", [2, 8, 9, 10, 11, 12])   # 4 .. 4096 sub-buckets
@pytest.mark.parametrize("tile", [4096, 8192])            # twice the workgroups at 4096
def test_items_all_probed_once(gpu_ctx, bits, tile, hot):
    import torch
    rng = np.random.default_rng(bits * 10_000 + tile)
    n_r, n_s = 12_000, 120_000
    rk = rng.integers(0, 2**32, n_r, dtype=np.uint64).astype(np.uint32)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    sk[::3] = rk[rng.integers(0, n_r // 2, sk[::3].size)]
    sk[:hot] = rk[7]
    host = (rk, np.arange(n_r, dtype=np.uint32), sk, np.arange(n_s, dtype=np.uint32))
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    print(f"[items] bits={bits} tile={tile} hot={hot}", flush=True)
    n, k, a, b = O.cpu_join(*host)
    for times in (0, 1):
        p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, radix_bits=bits, tile=tile,
                              collect_phase_times=times)
        res = gpu_ctx.join(p, *dev)
        assert res.match_count == n
        assert np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), O.sort_rows(k, a, b))
