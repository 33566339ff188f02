"""Branches whose condition is a wave's own vote: the waves of a workgroup may take
different ways there, so no barrier of the workgroup lies inside (CPU test on the kernel
sources), and probe rounds whose waves do take different ways (GPU test)."""
import glob
import os
import re

import numpy as np
import pytest

import brigjoin as bj
import oracle as O

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "brig-join_amd", "csrc")
BARRIERS = ("__syncthreads", "block_exclusive_scan")


def _close(s, at, pair):
    """The index after the bracket that closes the one at s[at]."""
    depth = 0
    for i in range(at, len(s)):
        depth += (s[i] == pair[0]) - (s[i] == pair[1])
        if depth == 0:
            return i + 1
    raise AssertionError("unbalanced source")


def _arm(s, at):
    """A statement or block from s[at] on: (text, index after it)."""
    while s[at].isspace():
        at += 1
    end = _close(s, at, "{}") if s[at] == "{" else s.index(";", at) + 1
    return s[at:end], end


def per_wave_arms(src):
    src = re.sub(r"//[^\n]*", "", src)
    votes = set(re.findall(r"\bbool\s+(\w+)\s*=[^;]*__ballot", src))
    for m in re.finditer(r"\bif\s*(?:constexpr\s*)?\(", src):
        end = _close(src, m.end() - 1, "()")
        cond = src[m.end() - 1:end]
        if "__ballot" not in cond and not votes & set(re.findall(r"\w+", cond)):
            continue
        text, end = _arm(src, end)
        yield cond, text
        rest = src[end:].lstrip()
        if rest.startswith("else"):
            yield cond, _arm(src, src.index("else", end) + 4)[0]


def test_the_rule_sees_both_arms():
    bad = "if (__ballot(x) == 0ull) { a(); } else { b(); __syncthreads(); }"
    assert [any(b in t for b in BARRIERS) for _, t in per_wave_arms(bad)] == [False, True]
    assert list(per_wave_arms("const bool v = __ballot(x) != 0; if (v) y(); __syncthreads();")) == [("(v)", "y();")]


@pytest.mark.parametrize("name", sorted(os.path.basename(p) for p in glob.glob(CSRC + "/*.h") + glob.glob(CSRC + "/*.hip")))
def test_no_barrier_in_a_wave_branch(name):
    with open(os.path.join(CSRC, name)) as f:
        for cond, text in per_wave_arms(f.read()):
            assert not any(b in text for b in BARRIERS), (name, cond)


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(), dict(radix_bits=2), dict(radix_bits=2, tile=4096)])
@pytest.mark.parametrize("twice", [0, 1, 40])
@pytest.mark.parametrize("n_s", [40_000, 300_000])
def test_rounds_of_both_forms(gpu_ctx, kw, twice, n_s):
    """Every S tuple matches and few R keys occur twice: large rounds in which no wave, one
    wave or several waves have a key with two matches (300K: rounds of 4 keys a thread)."""
    import torch
    rng = np.random.default_rng(twice)
    n_r = 8000
    rk = np.arange(n_r, dtype=np.uint32) * np.uint32(2654435761)
    rk[n_r - twice:] = rk[:twice]
    host = (rk, rng.permutation(n_r).astype(np.uint32), rk[rng.integers(0, n_r, n_s)], np.arange(n_s, dtype=np.uint32))
    dev = [torch.from_numpy(a.view(np.int32)).cuda() for a in host]
    torch.cuda.synchronize()
    print(f"[both forms] twice={twice} |S|={n_s} {kw}", flush=True)
    res = gpu_ctx.join(bj.default_params(r_size=n_r, s_size=n_s, inputs_on_device=1, answer_scale=2.0, **kw), *dev)
    n, k, a, b = O.cpu_join(*host)
    assert res.match_count == n and not res.truncated
    assert np.array_equal(O.sort_rows(*gpu_ctx.rows_to_host(res)), O.sort_rows(k, a, b))
