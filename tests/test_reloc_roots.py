"""The two-level interval index at the edges of its parts: root entries that
answer themselves, whose range holds one leaf (4 intervals), all seven (28) and one more (a tree of
lines: 29, 60, 61, 900, 901), starts on the fences' unit and off it, one, two and
256 entries more or less, a gap before every interval and none, both policies.
On the CPU the host build and one lane's search against the oracle's binary
search, and on the GPU the device build against the host build, entry for entry
and line for line, and k_reloc's searches by waves, through this index and
through the index of root lines, against the oracle's, bit for bit."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import oracle
from foundry_amd._lib import FoundryError
from foundry_amd.restore import RelocPlan, relocate_words_static

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "_build")
CHECK = os.path.join(NATIVE, "reloc_roots_check")
BUILD_CHECK = os.path.join(NATIVE, "roots_build_check")


def _run_of(rng, at, count, unit, gap):
    """count intervals of a few units each from `at`, abutting or with gaps."""
    size = unit * rng.integers(1, 4, count).astype(np.uint64)
    step = size + (unit * rng.integers(1, 3, count).astype(np.uint64) if gap else np.uint64(0))
    lo = np.uint64(at) + np.cumsum(step, dtype=np.uint64) - step
    return lo, lo + size


def _table(kind, rng):
    """Runs of the given lengths of small intervals, spread over a wide span."""
    base = 0x7F0000000000
    if kind == "one":
        lo, hi = np.array([base], np.uint64), np.array([base + 12345], np.uint64)
    elif kind in ("aligned", "unaligned", "bytes"):
        unit = {"aligned": 256, "unaligned": 24, "bytes": 1}[kind]
        parts = []
        at = base
        for rep in range(3):
            for count in (1, 3, 4, 5, 27, 28, 29, 30, 60, 61, 900, 901):
                parts.append(_run_of(rng, at, count, unit, gap=rep != 1))
                at = int(parts[-1][1][-1]) + int(rng.integers(1, 64)) * (1 << 22)
                at -= at % unit if kind == "aligned" else 0
        lo, hi = (np.concatenate(x) for x in zip(*parts))
    elif kind == "crowded":  # thousands under one entry beside one interval far away
        lo, hi = _run_of(rng, base, 20000, 256, gap=False)
        lo, hi = np.append(lo, np.uint64(base + (1 << 45))), np.append(hi, np.uint64(base + (1 << 45) + 4096))
    else:  # n intervals of 100 kB or so; "wide": of up to 64 MB
        n = int(kind.split("-")[0])
        size = 256 * (1 + np.exp(rng.uniform(0, 12.5 if "wide" in kind else 7, n))).astype(np.uint64)
        hi = np.uint64(base) + np.cumsum(size, dtype=np.uint64)
        lo = hi - size
    n = len(lo)
    nlo = np.uint64(1 << 44) + rng.permutation(n).astype(np.uint64) * np.uint64(1 << 27)
    edges = np.concatenate([lo - np.uint64(1), lo, lo + np.uint64(1), hi - np.uint64(1), hi, hi + np.uint64(1)])
    inside = lo[0] + rng.integers(0, int(hi[-1] - lo[0]) + 2, 20001).astype(np.uint64)
    return lo, hi, nlo, np.concatenate([edges, inside, np.array([0, (1 << 64) - 1], np.uint64)])


KINDS = ["one", "2", "5", "aligned", "unaligned", "bytes", "crowded", "1021", "2048", "2049", "40000", "300-wide", "4096-wide"]


@pytest.mark.parametrize("kind", KINDS)
def test_host_build_and_search(tmp_path, kind):
    lo, hi, nlo, words = _table(kind, np.random.default_rng(KINDS.index(kind)))
    t, w, o = (str(tmp_path / f) for f in ("t.bin", "w.bin", "o.bin"))
    words.tofile(w)
    for policy in (0, 1):
        np.concatenate([np.array([len(lo), policy], np.uint64), lo, hi, nlo]).tofile(t)
        p = subprocess.run([CHECK, t, w, o], capture_output=True, text=True, timeout=60)
        assert p.returncode == 0, p.stderr
        shape = json.loads(p.stdout)
        assert kind not in ("aligned", "1021", "40000") or (shape["exact"] and shape["flat"] > 0), shape
        assert kind != "bytes" or not shape["exact"], shape
        assert kind == "one" or shape["direct"] > 0, shape
        assert shape["bad_pairs"] == 0, shape
        assert kind not in ("aligned", "unaligned", "bytes", "crowded") or shape["deep"] > 0, shape
        np.testing.assert_array_equal(np.fromfile(o, np.uint64), oracle.relocate_words(words, lo, hi, nlo, policy))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_device_build_and_search(cuda, kind):
    lo, hi, nlo, words = _table(kind, np.random.default_rng(KINDS.index(kind)))
    print(f"[case] two-level index: {kind}, {len(lo)} intervals, {len(words)} words", flush=True)
    d_in = cuda.from_numpy(words.view(np.int64)).to("cuda")
    for policy in (0, 1):
        want = oracle.relocate_words(words, lo, hi, nlo, policy)
        plan = RelocPlan(lo, hi, nlo, policy)
        for start in (0, 1):  # 16-byte aligned words, and 8-byte aligned ones
            d_out = cuda.zeros_like(d_in)
            plan.relocate(d_in.data_ptr() + 8 * start, d_out.data_ptr() + 8 * start, len(words) - start)
            cuda.cuda.synchronize()
            np.testing.assert_array_equal(d_out.cpu().numpy().view(np.uint64)[start:], want[start:])
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [k for k in KINDS if k != "one"])
def test_search_through_root_lines(cuda, kind):
    """k_reloc's search through an index of root lines (relocate_words_static)
    over the same tables, the words shuffled so that the lookups of a wave end
    in leaves, under one fence line and under several at once: in one small call
    and in one of over a million words."""
    rng = np.random.default_rng(KINDS.index(kind))
    lo, hi, nlo, words = _table(kind, rng)
    print(f"[case] root lines: {kind}, {len(lo)} intervals, {len(words)} words", flush=True)
    words = rng.permutation(words)
    for n in (len(words), (1 << 20) + 4097):
        w = np.resize(words, n)
        d_in = cuda.from_numpy(w.view(np.int64)).to("cuda")
        for policy in (0, 1):
            d_out = cuda.zeros_like(d_in)
            relocate_words_static(lo, hi, nlo, d_in.data_ptr(), d_out.data_ptr(), n, policy)
            cuda.cuda.synchronize()
            np.testing.assert_array_equal(d_out.cpu().numpy().view(np.uint64),
                                          oracle.relocate_words(w, lo, hi, nlo, policy, threads=8))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_device_build_equals_the_host_build(cuda, tmp_path, kind):
    """Every root entry and line that the index kernels place is the host
    build's (roots_build_check runs both)."""
    lo, hi, nlo, _ = _table(kind, np.random.default_rng(KINDS.index(kind)))
    print(f"[case] device build of the two-level index: {kind}, {len(lo)} intervals", flush=True)
    t = str(tmp_path / "t.bin")
    for policy in (0, 1):
        np.concatenate([np.array([len(lo), policy], np.uint64), lo, hi, nlo]).tofile(t)
        p = subprocess.run([BUILD_CHECK, t], capture_output=True, text=True, timeout=60)
        assert p.returncode == 0, (p.returncode, p.stderr)
        got = json.loads(p.stdout)
        assert got["device_lines"] == got["lines"] and got["bad_roots"] == got["bad_lines"] == 0, got
        assert kind not in ("crowded", "40000") or got["lines"] > 1000, got


@pytest.mark.gpu
@pytest.mark.parametrize("n", [32768, 32769, 70001])
def test_tables_at_fault_are_refused_with_their_first_fault(cuda, n):
    """Tables of 32768 intervals and fewer are checked on the host, larger
    ones on the device: the same faults, each at the table's ends and between
    two workgroups' shares, with the same message; the whole table passes."""
    print(f"[case] refused tables of {n} intervals", flush=True)
    lo = np.uint64(1 << 40) + np.uint64(4096) * np.arange(n, dtype=np.uint64)
    hi = lo + np.uint64(4096)
    RelocPlan(lo, hi, lo).close()
    for at in (0, 1, 255, 256, n - 1):
        h = hi.copy()
        h[at] = lo[at]
        with pytest.raises(FoundryError, match=f"interval {at} is empty"):
            RelocPlan(lo, h, lo)
        if at:
            h = hi.copy()
            h[at - 1] += np.uint64(1)
            with pytest.raises(FoundryError, match=f"intervals {at - 1} and {at} overlap"):
                RelocPlan(lo, h, lo)
    h = hi.copy()
    h[-1] = np.uint64((1 << 64) - 1)
    with pytest.raises(FoundryError, match=f"interval {n - 1} ends at 2"):
        RelocPlan(lo, h, lo)
    h[-1] = lo[0] + np.uint64(1 << 54)
    with pytest.raises(FoundryError, match="span more than 2"):
        RelocPlan(lo, h, lo)
    with pytest.raises(FoundryError, match="policy"):
        RelocPlan(lo, hi, lo, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("intervals", [2, 64, 1000, 40000])
def test_restore_by_a_crowded_table(cuda, intervals):
    """An archive's allocations under one root entry (another one lies 2^45
    bytes away), so that every search of the template and search passes descends
    a tree, in batches of a few words and of many: the oracle's restore."""
    from foundry_amd import synth
    from foundry_amd.restore import Archive
    from tests.parity import assert_restore_parity

    print(f"[case] restore by a crowded table of {intervals} intervals", flush=True)
    s = synth.SynthArchive(synth.preset(2, num_graphs=12, num_groups=3, nodes_per_graph=200, num_intervals=intervals,
                                        diff_lo=0.1, diff_hi=0.1, pointer_frac=0.4, seed=0x5EEDC0 + intervals))
    lo, hi, nlo = (np.asarray(a) for a in s.intervals())
    far = np.uint64(int(lo[0]) + (1 << 45))
    table = np.append(lo, far), np.append(hi, far + np.uint64(4096)), np.append(nlo, np.uint64(1 << 46))
    for policy in (0, 1):
        arch = Archive.from_synth(s)
        arch.set_relocation(*table, policy=policy)
        arch.restore()
        assert_restore_parity(arch, oracle.Restore(s.images(), table, policy=policy, threads=4))
        arch.close()


@pytest.mark.skipif(torch.cuda.is_available(), reason="there is a device")
def test_large_tables_at_fault_without_a_device():
    """A table that the device would check (more than 32768 intervals) is
    checked on the host where there is none: its fault is what is reported."""
    n = 40000
    lo = np.uint64(1 << 40) + np.uint64(4096) * np.arange(n, dtype=np.uint64)
    hi = lo + np.uint64(4096)
    hi[n // 2] = lo[n // 2]
    with pytest.raises(FoundryError, match=f"interval {n // 2} is empty"):
        RelocPlan(lo, hi, lo)
    with pytest.raises(FoundryError, match="hipMalloc"):
        RelocPlan(lo, lo + np.uint64(4096), lo)


_FIRST_TABLES = """
import numpy as np, torch
import oracle
from foundry_amd.restore import RelocPlan
rng = np.random.default_rng(9)
d = None
for k, (n, busy) in enumerate([(300_000, False), (300_000, False), (40_000, True), (300_000, False), (10, True)]):
    size = rng.integers(1, 64, n).astype(np.uint64) * np.uint64(256)
    hi = np.uint64(1 << 44) + np.cumsum(size, dtype=np.uint64)
    lo = hi - size
    nlo = rng.permutation(n).astype(np.uint64) << np.uint64(20)
    words = np.concatenate([lo, hi, hi - np.uint64(1)])
    d_in = torch.from_numpy(words.view(np.int64)).cuda()
    d_out = torch.zeros_like(d_in)
    torch.cuda.synchronize()
    if busy:
        torch.cuda._sleep(50_000_000)
    plan = RelocPlan(lo, hi, nlo)
    plan.relocate(d_in.data_ptr(), d_out.data_ptr(), len(words))
    torch.cuda.synchronize()
    assert np.array_equal(d_out.cpu().numpy().view(np.uint64), oracle.relocate_words(words, lo, hi, nlo, 0)), (k, n)
    plan.close()
    print("table", k, n, "same", flush=True)
"""


@pytest.mark.gpu
def test_first_tables_of_a_process():
    """A process's first table is copied from where it lies, later ones go
    through the staging slots (several rounds of them here), on the null stream
    or, with work queued there, on the stage's own: each relocates as the
    oracle does."""
    print("[case] the first tables of a process", flush=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", _FIRST_TABLES], cwd=root, capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.count("same") == 5, (p.returncode, p.stdout, p.stderr)
