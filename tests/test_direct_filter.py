"""The filter of an unpartitioned R with equal keys or few blocks (GPU tests): the same
survivors and rows as the partitioned join's filter, and built no slower than that one,
which gathers the bits of a block on chip (one atomic in memory per key took 13 times as
long for 100K equal keys)."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_r,n_s,equal,kw", [
    (100_000, 300_000, 1.0, dict(bf_bits_per_key=10.0)),
    (200_000, 300_000, 0.5, dict(bf_bits_per_key=10.0)),
    (200_001, 300_000, 0.0, dict(num_bits=256)),        # four 64-bit blocks
    (2_500_000, 8000, 1.0, dict(bf_bits_per_key=10.0)),
    (255, 5000, 0.5, dict(bf_bits_per_key=10.0)),       # one workgroup's keys less one, and one more
    (257, 5000, 0.0, dict(bf_bits_per_key=14.0)),
])
def test_filter_of_equal_keys(gpu_ctx, n_r, n_s, equal, kw):
    import torch
    rng = np.random.default_rng(n_r)
    rk = np.arange(n_r, dtype=np.uint32) * np.uint32(2654435761) + np.uint32(1)
    hot = int(n_r * equal)
    rk[:hot] = 77
    rng.shuffle(rk)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    once = rk[rk != 77]
    if len(once):
        sk[:n_s // 10] = once[rng.integers(0, len(once), n_s // 10)]
    sk[sk == 77] = 78
    host = (rk, np.arange(n_r, dtype=np.uint32), sk, np.arange(n_s, dtype=np.uint32))
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    print(f"[direct filter] |R|={n_r} equal={equal} {kw}", flush=True)
    n, k, a, b = O.cpu_join(*host)
    expect = O.sort_rows(k, a, b)
    seen = {}
    for stage in (0, 1):   # the library's choice; the filter stage given: partitioned
        p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, use_bf=1, num_hashes=3, bf_stage=stage,
                              collect_phase_times=1, **kw)
        ms = []
        for _ in range(5):
            res = gpu_ctx.join(p, *dev)
            ms.append(res.kernels()["bf_build"])
        seen[stage] = (res.s_survivors, sorted(ms)[2])
        assert res.match_count == n and np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), expect)
    assert seen[0][0] == seen[1][0]
    if equal == 1.0 or "num_bits" in kw:
        assert seen[0][1] < seen[1][1], seen
