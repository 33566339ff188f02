"""What a user of the join has it do, as cases that can be timed.

A case is one call (or one burst of calls) through the Python binding of the C
ABI: a single join, a join into the caller's arrays, a join of host relations in
chunks of S, a batch of joins, a burst of requests against resident relations.

Rows come back from a join in no defined order, so every case puts them into
columns, as a consumer does that materialises late: S's value of a matching tuple
is its place in the result (`slot`), and the row's key and R value are stored
there.  With R keys that occur `dup` times, a matching S tuple owns `dup` places.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "brig-join_amd"))
import brigjoin as bj  # noqa: E402

DEV = "cuda:0"
CHUNK = 1 << 26  # tuples generated at a time


def _join(name, n_r, n_s, every, **kw):
    """every: one S tuple in so many has a match.  dup: copies of every R key.  keys: "mixed" (spread over 32 bits)
    or "ids" (R sorted by a dense id).  zipf: matching S keys follow a Zipf law (exponent about 1) over R."""
    c = dict(name=name, kind="join", n_r=n_r, n_s=n_s, every=every, dup=1, keys="mixed", zipf=False, use_bf=0,
             bf_bits_per_key=0.0, num_hashes=-1, partition_size=-1, radix_bits=-1, s_chunks=1,
             collect_phase_times=0)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: a lookup of a couple of thousand keys (latency and launches only)
        _join("lookup_1500_2000", 1500, 2000, 3),
        # a small join with the filter and the default phase times, the sizes of the smoke run
        _join("small_200k_300k_bf", 200_000, 300_000, 10, use_bf=1, bf_bits_per_key=10.0, num_hashes=3,
              collect_phase_times=1),
        # a small dimension table against a long fact table, every fact row matches
        _join("dimension_6k_20m", 6001, 20_000_003, 1),
        # device-resident relations joined without allocation into the caller's arrays (serving loops)
        _join("into_arrays_3m_4500k", 3_000_017, 4_500_007, 4, kind="into"),
        # the benchmark's 16M join without a filter
        _join("join16m_nobf", 16_000_000, 16_000_000, 10, partition_size=1024),
        # every R key four times: more than one row per match
        _join("dups_9m_24m", 9_000_004, 24_000_001, 5, dup=4),
        # two large ragged tables on a dense sorted id, no filter, a quarter of S matches
        _join("ids_100m_130m", 100_000_007, 130_000_001, 4, keys="ids"),
        # the benchmark's headline join: 640M tuples on each side, filter, 10% match
        _join("join640m_bf10", 640_000_000, 640_000_000, 10, use_bf=1, bf_bits_per_key=10.0, num_hashes=3,
              partition_size=512, radix_bits=14),
        # the benchmark's skewed join: long S, Zipf-distributed matches, 1% match
        _join("join64m_1280m_zipf", 64_000_000, 1_280_000_000, 100, zipf=True, use_bf=1, bf_bits_per_key=12.0,
              num_hashes=4),
        # relations in (pinned) host memory, S copied and joined in chunks
        _join("host_10m_40m_chunks4", 10_000_000, 40_000_000, 10, kind="host", s_chunks=4, use_bf=1,
              bf_bits_per_key=10.0, num_hashes=3),
        # many joins of uneven sizes as one captured launch sequence
        dict(name="batch_40_64k_4m", kind="batch", joins=40, r_lo=65_536, r_hi=4_194_304, every=6),
        # a burst of requests of uneven sizes against resident relations
        dict(name="serve_3x8_16m_64m", kind="serve", relations=3, r_lo=16_000_000, r_hi=64_000_000, requests=8,
             s_lo=1_000_000, s_hi=32_000_000, every=10),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["join"] * 6 + ["into", "host", "batch", "serve"])
    every = rng.choice([1, 2, 3, 5, 8, 10, 20, 50, 100])
    if kind == "batch":
        lo = _log_uniform(rng, 20_000, 500_000)
        return dict(kind=kind, joins=rng.randint(4, 48), r_lo=lo, r_hi=lo * rng.randint(2, 30), every=max(2, every))
    if kind == "serve":
        r_lo = _log_uniform(rng, 1_000_000, 30_000_000)
        s_lo = _log_uniform(rng, 100_000, 4_000_000)
        return dict(kind=kind, relations=rng.randint(1, 3), r_lo=r_lo, r_hi=r_lo * rng.randint(1, 4),
                    requests=rng.randint(2, 10), s_lo=s_lo, s_hi=s_lo * rng.randint(2, 8), every=max(2, every))
    if kind == "into":
        n_r, ratio = _log_uniform(rng, 1000, 4_000_000), rng.uniform(0.3, 1.5)
    elif kind == "host":
        n_r, ratio = _log_uniform(rng, 10_000, 12_000_000), rng.uniform(0.5, 4.0)
    else:
        n_r, ratio = _log_uniform(rng, 1000, 640_000_000), math.exp(rng.uniform(math.log(0.3), math.log(30.0)))
    n_s = int(min(max(1000, n_r * ratio), 1_280_000_000))
    if n_r + n_s > 1_280_000_000:
        n_s = 1_280_000_000 - n_r
    # the rows are a limited part of the work: at most about 64M of them
    every = max(every, -(-n_s // 64_000_000))
    dup = rng.choice([1, 1, 1, 2, 4]) if n_s // every <= 16_000_000 else 1
    n_r = max(dup, n_r - n_r % dup)
    c = _join("", n_r, n_s, every, kind=kind, dup=dup, keys=rng.choice(["mixed", "mixed", "ids"]),
              zipf=dup == 1 and rng.random() < 0.15, collect_phase_times=rng.choice([0, 0, 1]))
    del c["name"]
    if rng.random() < 0.5:
        bits = rng.choice([6.0, 8.0, 10.0, 12.0, 14.0])
        c.update(use_bf=1, bf_bits_per_key=bits, num_hashes=rng.choice([-1, 2, 3, 4, 5]))
    if kind == "host":
        c["s_chunks"] = rng.choice([1, 2, 3, 4])
    return c


# ---------------------------------------------------------------- inputs
def _mix(x, salt):
    """A bijection on 32-bit words (int32 tensors, wrapping arithmetic)."""
    x = x + salt
    x = (x ^ ((x >> 16) & 0xFFFF)) * 0x7FEB352D
    x = (x ^ ((x >> 15) & 0x1FFFF)) * -2073254261
    return x ^ ((x >> 16) & 0xFFFF)


def _key(index, c, salt):
    """The key of key index `index` (int32 or int64 below 2^31 + 2^31)."""
    x = index.to(torch.int32)
    return x if c["keys"] == "ids" else _mix(x, salt)


def _salts(seed):
    return [((seed * 0x9E3779B1 + i * 0x85EBCA6B + 0x165667B1) % 0x7FFFFFFF) for i in range(3)]


def _make_r(c, seed):
    n, dup = c["n_r"], c["dup"]
    salt = _salts(seed)[0]
    key = torch.empty(n, dtype=torch.int32, device=DEV)
    for at in range(0, n, CHUNK):
        m = min(CHUNK, n - at)
        i = torch.arange(at, at + m, dtype=torch.int64, device=DEV)
        if dup > 1:
            # the copies of a key lie apart: row i holds key index i mod (n / dup)
            i = i % (n // dup)
        key[at:at + m] = _key(i, c, salt)
    return key, torch.arange(n, dtype=torch.int32, device=DEV)


def _make_s(c, seed, first_slot=0, s_seed=None):
    """In every group of `every` tuples one matches, at a place that the seed decides."""
    n, g, kinds = c["n_s"], c["every"], c["n_r"] // c["dup"]
    salt, pick, place = _salts(seed)
    if s_seed is not None:
        _, pick, place = _salts(s_seed)
    key = torch.empty(n, dtype=torch.int32, device=DEV)
    val = torch.empty(n, dtype=torch.int32, device=DEV)
    whole = n // g * g
    for at in range(0, n, CHUNK):
        m = min(CHUNK, n - at)
        j = torch.arange(at, at + m, dtype=torch.int32, device=DEV)
        group = torch.div(j, g, rounding_mode="floor")
        hit = (((_mix(group, place) & 0x7FFFFFFF) % g) == j - group * g) & (j < whole)
        u = (_mix(group, pick).to(torch.float64) + 2147483648.5) / 4294967296.0
        if c["zipf"]:
            u = torch.exp(u * math.log(kinds + 1.0)) - 1.0
        else:
            u = u * kinds
        index = torch.where(hit, u.to(torch.int64).clamp_(0, kinds - 1), j.to(torch.int64) + c["n_r"])
        key[at:at + m] = _key(index, c, salt)
        val[at:at + m] = torch.where(hit, group + first_slot, j)
    return key, val


def _rows(c):
    return c["n_s"] // c["every"] * c["dup"]


def _geometric(lo, hi, n):
    return [int(lo * (hi / lo) ** (i / max(1, n - 1))) for i in range(n)]


def _parts(c):
    """The single joins that a batch or a burst consists of: (relation, plain join) pairs."""
    base = _join("", 1, 1, c["every"])
    if c["kind"] == "batch":
        sizes = _geometric(c["r_lo"], c["r_hi"], c["joins"])
        return [(i, dict(base, n_r=n + i % 7, n_s=int(n * (1 + (i * 5 % 13) / 4.0)) + i % 11))
                for i, n in enumerate(sizes)]
    rels = _geometric(c["r_lo"], c["r_hi"], c["relations"])
    sizes = _geometric(c["s_lo"], c["s_hi"], c["requests"])
    return [(i % len(rels), dict(base, n_r=rels[i % len(rels)] + i % len(rels), n_s=n + i)) for i, n in enumerate(sizes)]


_open = {}


def _context():
    """The program's one context and the stream that its joins and its own work run on."""
    if not _open:
        _open["stream"] = torch.cuda.Stream()
        _open["ctx"] = bj.Context(0)
        _open["ctx"].set_stream(_open["stream"].cuda_stream)
    return _open["ctx"], _open["stream"]


def _params(c):
    return bj.default_params(r_size=c["n_r"], s_size=c["n_s"], use_bf=c["use_bf"],
                             bf_bits_per_key=c["bf_bits_per_key"], num_hashes=c["num_hashes"],
                             partition_size=c["partition_size"], radix_bits=c["radix_bits"],
                             s_chunks=c["s_chunks"], collect_phase_times=c["collect_phase_times"],
                             answer_scale=float(c["dup"]), inputs_on_device=0 if c["kind"] == "host" else 1)


def _inputs(case, seed):
    """[(relation, join, R, S)] of a case's joins; S's slots follow each other."""
    if case["kind"] not in ("batch", "serve"):
        return [(0, case, _make_r(case, seed), _make_s(case, seed))]
    got, made, slot = [], {}, 0
    for i, (rel, c) in enumerate(_parts(case)):
        if rel not in made:
            made[rel] = _make_r(c, seed * 64 + rel)
        got.append((rel, c, made[rel], _make_s(c, seed * 64 + rel, slot, s_seed=seed * 64 + 17 + i)))
        slot += _rows(c)
    return got


def prepare(case, seed):
    ctx, stream = _context()
    kind = case["kind"]
    got = _inputs(case, seed)
    torch.cuda.synchronize()
    state = dict(case=case, ctx=ctx, stream=stream, rows=sum(_rows(c) for _, c, _, _ in got))
    if kind == "batch":
        specs = [bj.join_spec(*r, *s, r_size=c["n_r"], s_size=c["n_s"]) for _, c, r, s in got]
        state.update(inputs=got, batch=bj.Batch(ctx, specs))
    elif kind == "serve":
        server = bj.Server(0, arena_bytes=64 * sum(c["n_s"] for _, c, _, _ in got) + (64 << 20))
        ids = {}
        for rel, c, r, _ in got:
            if rel not in ids:
                ids[rel] = server.add_relation(r[0], r[1], c["n_r"])
        state.update(server=server, requests=[(ids[rel], s[0], s[1], c["n_s"]) for rel, c, _, s in got])
    else:
        (_, c, r, s), = got
        if kind == "host":
            r, s = ([torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t) for t in x] for x in (r, s))
        state.update(params=_params(c), r=r, s=s)
        if kind == "into":
            state["out"] = [torch.empty(max(1, state["rows"]), dtype=torch.int32, device=DEV) for _ in range(3)]
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------- one pass
class _DeviceArray:
    """int32 values in device memory that the library owns."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i4", data=(ptr, False), version=3)


def _columns_of(res):
    n = res.rows_written
    if n == 0:
        return [torch.empty(0, dtype=torch.int32, device=DEV)] * 3
    return [torch.as_tensor(_DeviceArray(p, n), device=DEV) for p in (res.key, res.r_val, res.s_val)]


def _slots(c, r_val, s_val):
    if c.get("dup", 1) == 1:
        return s_val.long()
    copy = torch.div(r_val, c["n_r"] // c["dup"], rounding_mode="floor")
    return torch.add(copy, s_val, alpha=c["dup"]).long()


def _place(state, count, key, r_val, s_val):
    slot = _slots(state["case"], r_val, s_val)
    out = torch.full((2, state["rows"]), -1, dtype=torch.int32, device=DEV)
    out[0].scatter_(0, slot, key)
    out[1].scatter_(0, slot, r_val)
    return dict(count=count, rows=out)


def run(state):
    kind = state["case"]["kind"]
    with torch.cuda.stream(state["stream"]):
        if kind == "batch":
            outs, _ = state["batch"].run()
            cols = [torch.cat(x) for x in zip(*(_columns_of(o) for o in outs))]
            return _place(state, sum(o.match_count for o in outs), *cols)
        if kind == "serve":
            server = state["server"]
            ids = [server.submit(*q) for q in state["requests"]]
            done = [server.wait(i) for i in ids]
            cols = [torch.cat(x) for x in zip(*(_columns_of(d) for d in done))]
            state["stream"].synchronize()  # the rows are copied: their memory goes back
            for i in ids:
                server.release(i)
            return _place(state, sum(d.match_count for d in done), *cols)
        if kind == "into":
            res = state["ctx"].join_noalloc(state["params"], *state["r"], *state["s"], *state["out"],
                                            state["out"][0].numel())
            cols = [t[:res.rows_written] for t in state["out"]]
        else:
            res = state["ctx"].join(state["params"], *state["r"], *state["s"])
            cols = _columns_of(res)
        return _place(state, res.match_count, *cols)


# ---------------------------------------------------------------- yardsticks
def work(case):
    """Every input tuple (8 bytes) read once, every row (12 bytes) written once."""
    if case["kind"] not in ("batch", "serve"):
        parts = [(0, case)]
    else:
        parts = _parts(case)
    tuples = sum({rel: c["n_r"] for rel, c in parts}.values()) + sum(c["n_s"] for _, c in parts)
    return dict(bytes=8 * tuples + 12 * sum(_rows(c) for _, c in parts), flops=0)


def exact(case, seed):
    """The same columns from a sorted R and a binary search (whole numbers: equal, not near)."""
    got = _inputs(case, seed)
    n = sum(_rows(c) for _, c, _, _ in got)
    out = torch.full((2, n), -1, dtype=torch.int32, device=DEV)
    count = 0
    for _, c, (rk, rv), (sk, sv) in got:
        key, order = torch.sort(rk)
        val = rv[order]
        del order
        for at in range(0, c["n_s"], CHUNK // 2):
            k, v = sk[at:at + CHUNK // 2], sv[at:at + CHUNK // 2]
            p = torch.searchsorted(key, k, out_int32=True)
            for d in range(c["dup"]):
                q = (p + d).clamp_(max=c["n_r"] - 1).long()
                hit = (key[q] == k) & (p + d < c["n_r"])
                r = val[q[hit]]
                slot = _slots(c, r, v[hit])
                out[0][slot] = k[hit]
                out[1][slot] = r
                count += int(hit.sum())
    return dict(count=count, rows=out)
