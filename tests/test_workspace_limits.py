"""What a join, a join without allocation and a request need of device memory: figures
that were once enough stay enough (few radix bits have many chunks and need no fine
slices besides; a request keeps the histograms of 32K-tuple chunks)."""
import numpy as np
import pytest

import brigjoin as bj
import oracle as O


@pytest.mark.parametrize("n_r,n_s,bits,tile,enough", [
    (110_130_328, 249_003_751, 1, 4096, 2_895_529_720),   # (2 983 220 216 with 256 slices of every chunk)
    (99_285_756, 132_661_284, 1, 4096, None),
    (50_000_000, 50_000_000, 3, 8192, None),
])
def test_work_items_of_few_radix_bits(n_r, n_s, bits, tile, enough):
    p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, radix_bits=bits, tile=tile)
    if enough is None:
        # both relations in one pass, at most 1 MB of histograms and offsets, and 16 bytes
        # an item, 16 slices of both sides' chunks
        enough = (n_r + n_s) * 8 + (1 << 20) + 16 * (16 * ((n_r + n_s) // tile + 2**bits) + 16)
    plan = bj.plan(p)
    assert plan.workspace_bytes - 12 * plan.capacity <= enough


@pytest.mark.gpu
def test_noalloc_of_one_radix_bit(gpu_ctx):
    """268 179 456 bytes of the 268 435 456, before its items were cut into 256 slices."""
    import torch
    n_r, n_s = 9_004_187, 24_385_346
    rng = np.random.default_rng(3)
    rk = np.arange(n_r, dtype=np.uint32) * np.uint32(2654435761)
    sk = rng.integers(0, 2**32, n_s, dtype=np.uint64).astype(np.uint32)
    dev = [torch.from_numpy(a.view(np.int32)).cuda()
           for a in (rk, np.arange(n_r, dtype=np.uint32), sk, np.arange(n_s, dtype=np.uint32))]
    out = [torch.empty(n_s // 100, dtype=torch.int32, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    print(f"[workspace] noalloc {n_r} x {n_s}", flush=True)
    p = bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, radix_bits=1, tile=8192)
    res = gpu_ctx.join_noalloc(p, *dev, *out, n_s // 100)
    row = (sk.astype(np.uint64) * pow(2654435761, -1, 2**32) & 0xFFFFFFFF)   # R's row of a key, if below n_r
    hit = np.nonzero(row < n_r)[0]
    assert res.match_count == len(hit) == res.rows_written
    k, a, b = (t[:len(hit)].cpu().numpy().view(np.uint32) for t in out)
    order = np.argsort(b)
    assert np.array_equal(b[order], hit) and np.array_equal(a[order], row[hit]) and np.array_equal(k[order], sk[hit])


@pytest.mark.gpu
def test_request_that_just_fits():
    import torch
    n_r, n_s = 2_000_000, 8_000_000
    enough = 192_750_080 + 3 * 32_000_000   # its S side, and its rows
    rk, rv = O.gen_r(3, n_r)
    m = n_s // 10
    sk, sv = O.gen_s(3, 4, n_r, n_s, m)
    dev = [torch.from_numpy(x.view(np.int32)).cuda() for x in (rk, rv, sk, sv)]
    torch.cuda.synchronize()
    with bj.Server(0, arena_bytes=enough) as server:
        rel = server.add_relation(dev[0], dev[1], n_r)
        assert server.request_bytes(rel, n_s) <= enough
        print(f"[workspace] request {server.request_bytes(rel, n_s)} of {enough}", flush=True)
        done = server.wait(server.submit(rel, dev[2], dev[3], n_s))
        assert done.match_count == m == done.rows_written
        k, a, b = server.rows_to_host(done)
        assert np.array_equal(rk[a], k) and np.array_equal(sk[b], k) and len(np.unique(b)) == m
