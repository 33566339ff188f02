"""The scatter's tiles, carries and bucket scans at their edges (GPU tests): every
fan-out form (one wave, the whole workgroup with one, two or four buckets per
thread), relation sizes around whole tiles, uniform and single-bucket keys."""
import numpy as np
import pytest

import brigjoin as bj

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wg", [512, 1024])
@pytest.mark.parametrize("pass1,bits", [(1, 1), (1, 2), (6, 7), (7, 7), (8, 9), (10, 12), (11, 11), (4, 15)])
@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 8193, 65_536, 123_457])
def test_partition_tile_edges(gpu_ctx, n, pass1, bits, wg):
    import torch
    rng = np.random.default_rng(n + bits)
    key = rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    key[: n // 3] = key[-1]                                   # a third of the tuples in one bucket
    val = rng.permutation(n).astype(np.uint32)
    dk, dv = (torch.from_numpy(a.view(np.int32)).cuda() for a in (key, val))
    ok, ov = torch.empty_like(dk), torch.empty_like(dv)
    st = torch.zeros((1 << bits) + 1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    print(f"[tile edges] n={n} pass1={pass1} bits={bits} wg={wg}", flush=True)
    p = bj.default_params(radix_bits=bits, pass1_bits=pass1, scatter_wg=wg)
    gpu_ctx.partition(p, dk, dv, n, ok, ov, st)
    hk, hv = (t.cpu().numpy().view(np.uint32) for t in (ok, ov))
    start = st.cpu().numpy()

    def bucket(k):
        return (((k.astype(np.uint64) * 0x9E3779B1) & 0xFFFFFFFF) >> np.uint64(32 - bits)).astype(np.int64)

    at = np.empty(n, np.int64)
    at[val] = np.arange(n)
    assert np.array_equal(np.sort(hv), np.arange(n, dtype=np.uint32))      # a permutation
    assert np.array_equal(hk, key[at[hv]])                                 # keys travel with their values
    assert np.array_equal(np.diff(start), np.bincount(bucket(key), minlength=1 << bits))
    b = bucket(hk)
    pos = np.arange(n)
    assert np.all((start[b] <= pos) & (pos < start[b + 1]))
