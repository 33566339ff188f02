"""Rows of consecutive probe rounds of one work item, at the round lengths that the
kernels have (GPU tests): items of one to six rounds that end a key before, at and a
key after a round, with rounds without matches, staged rounds and rounds with more rows
than the stage in every order, whole and cut off by the row capacity.  The lengths come
from the launcher's source, so that they follow it."""
import itertools
import os
import re

import numpy as np
import pytest

import brigjoin as bj

pytestmark = pytest.mark.gpu

INV = pow(0x9E3779B1, -1, 2**32)  # of the radix hash's multiplier
SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "brig-join_amd", "csrc", "bj_kernels.hip")


def rounds_of_kernels():
    """{(tile, whether the probe sides are long): probe keys of a round}, and from which mean size they are long."""
    with open(SRC) as f:
        src = f.read()
    value = {}
    for decl in re.findall(r"constexpr (?:int|uint64_t) (PROBE_\w+ = \d+(?:, PROBE_\w+ = \d+)*);", src):
        value.update((n, int(v)) for n, v in re.findall(r"(PROBE_\w+) = (\d+)", decl))
    per = {}
    for cond, block, cap, items in re.findall(r"if \((tile == \d+[^)]*)\) BJ_PROBE\((\d+), (\d+), (\w+),", src):
        per[int(cap), "long_probe" in cond] = int(block) * value[items]
    assert set(per) == {(8192, True), (8192, False), (4096, False)}, per
    return per, value["PROBE_LONG"]


PER, LONG = rounds_of_kernels()


def test_the_listed_lengths_are_the_kernels():
    assert PER[8192, False] < PER[8192, True] <= LONG


def keys(bucket, low, bits):
    """The keys whose hash has `bucket` on top and `low` below."""
    h = (np.uint64(bucket) << np.uint64(32 - bits)) | low.astype(np.uint64)
    return (h * np.uint64(INV) & np.uint64(0xFFFFFFFF)).astype(np.uint32)


def check(ctx, tile, bits, per, rounds, edge, items_of_bucket, buckets):
    """buckets sub-buckets of items_of_bucket items, each of rounds * per + edge probe keys."""
    import torch
    n_b, n = 1500, rounds * per + edge
    rng = np.random.default_rng(rounds * 100 + edge * 10 + tile + bits)
    orders = list(itertools.product((0.0, 0.1, 0.9), repeat=min(rounds, 4)))
    rk, sk, row = [], [], []
    for sb in range(buckets):
        low = rng.choice(1 << min(23, 32 - bits), n_b + per, replace=False)
        r, miss = keys(sb, low[:n_b], bits), keys(sb, low[n_b:], bits)
        for i in range(items_of_bucket):
            kinds = np.resize(orders[(sb * items_of_bucket + i) % len(orders)], rounds + 1)
            hit = rng.random(n) < np.repeat(kinds, per)[:n]
            at = rng.integers(0, n_b, n)
            sk.append(np.where(hit, r[at], miss[rng.integers(0, per, n)]))
            row.append(np.where(hit, at + sb * n_b, -1))
        rk.append(r)
    rk, sk, row = np.concatenate(rk), np.concatenate(sk), np.concatenate(row)
    dev = [torch.from_numpy(a.view(np.int32)).cuda()
           for a in (rk, np.arange(rk.size, dtype=np.uint32), sk, np.arange(sk.size, dtype=np.uint32))]
    torch.cuda.synchronize()
    print(f"[rounds] tile={tile} bits={bits} per={per} rounds={rounds} edge={edge} |S|={sk.size}", flush=True)
    hits = np.nonzero(row >= 0)[0]
    for cap in (hits.size, hits.size // 3):
        out = [torch.full((max(cap, 1),), -1, dtype=torch.int32, device="cuda") for _ in range(3)]
        torch.cuda.synchronize()
        p = bj.default_params(r_size=rk.size, s_size=sk.size, inputs_on_device=1, radix_bits=bits, tile=tile)
        res = ctx.join_noalloc(p, *dev, *out, cap)
        assert res.match_count == hits.size and res.rows_written == cap
        k, a, b = (t[:cap].cpu().numpy().view(np.uint32) for t in out)
        assert len(np.unique(b)) == cap and np.array_equal(a, row[b]) and np.array_equal(k, sk[b])
        if cap == hits.size:
            assert np.array_equal(np.sort(b), hits)


@pytest.mark.parametrize("tile", [4096, 8192])
@pytest.mark.parametrize("rounds", range(1, 7))
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_rounds(gpu_ctx, tile, rounds, edge):
    bits, per = 9, PER[tile, False]   # 512 sub-buckets, one work item each
    assert rounds * per + edge <= 65536 and 81 * (rounds * per + 1) >> bits < LONG
    check(gpu_ctx, tile, bits, per, rounds, edge, 1, 3**min(rounds, 4))


@pytest.mark.parametrize("rounds", range(1, 6))
@pytest.mark.parametrize("edge", [-1, 0, 1])
def test_long_rounds(gpu_ctx, rounds, edge):
    # two sub-buckets, their probe sides cut into the 256 slices of few sub-buckets
    per = PER[8192, True]
    assert 256 * (rounds * per + edge) >= LONG and rounds * per + edge <= 65536
    check(gpu_ctx, 8192, 1, per, rounds, edge, 256, 2)
