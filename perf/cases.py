"""The work that a program has this framework do, as cases that can be timed and compared.

A case is a dict of plain values.  `listed()` names twelve, `draw(rng)` gives
one more of the same ranges, `prepare(case, seed)` makes what a program holds
before the call, `run(state)` is one pass through the public entry points, and
`work`, `tolerance` and `exact` say what a pass cannot do without, how close
its outputs have to be (exactly: they are whole numbers) and what plain torch
makes of the same inputs.

Kinds of case, after what a LOAD does and what a program does with a loaded
archive afterwards:

  restore   Archive.restore of an archive whose images are in HBM
  load      Archive.open from files, set_relocation, restore, groups
  switch    Archive.switch_sequence over a restored archive
  replay    GroupGraph.replay of graphs of a restored archive
  reloc     RelocPlan.relocate of packed words in HBM
  plan      RelocPlan built from a table, one relocation with it
  static    relocate_words_static, several buffers by one table

The results of a restore, a load or a switch are the archive's own device
buffers: the framework's programs build and run graphs from them there and do
not copy them to the host.  `run` returns them as lists that read them out,
whole, when they are looked at (padded with zeros to a size that does not
depend on the seed).
"""
import os
import tempfile

import numpy as np
import torch

from foundry_amd import synth
from foundry_amd.graph import GroupGraph, Registry
from foundry_amd.restore import Archive, RelocPlan, relocate_words_static

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# The code object whose kernel takes any node's params and does nothing with them.
PROBE_CO = os.path.join(ROOT, "tests", "native", "_build", "probe.co")

REGION_BASE = 0x7F0000000000  # where the saved allocations lay
NEW_BASE = 0x7E0000000000     # where they lie now

# An archive with no special nodes: what the other archive cases start from.
PLAIN = {"groups": 1, "min_blob": 32, "max_blob": 1024, "params": 16, "pointers": 0.25, "diff": 0.03, "run_bytes": 0,
         "grid_pct": 20, "memset_pct": 0, "memcpy_pct": 0, "event_pct": 0, "extra_pct": 0, "layout_pct": 0,
         "ragged": False, "intervals": 40000, "inclusive": False}


def _archive(kind, graphs, nodes, **over):
    return {"kind": kind, "graphs": graphs, "nodes": nodes, **PLAIN, **over}


def listed():
    return [
        # The smallest archive in use: 64 graphs of one topology, 120 nodes each, the whole region moved as one
        # interval.  Launches and latency count.
        {"name": "restore_small", **_archive("restore", 64, 120, min_blob=64, max_blob=512, params=8, pointers=0.3,
                                              diff=0.05, grid_pct=0, intervals=1)},
        # A decode server's capture list: 256 batch sizes of a 48-layer model, 40k saved allocations.
        {"name": "restore_decode", **_archive("restore", 256, 1200, groups=4)},
        # Mixture-of-experts graphs: large descriptor arrays, memset and memcpy nodes, differences in runs.
        {"name": "restore_moe", **_archive("restore", 64, 3000, groups=8, max_blob=4096, params=40, diff=0.1,
                                            run_bytes=256, memset_pct=10, memcpy_pct=5)},
        # Everything that a capture may hold: params that are not whole words, argument buffers, events, layouts and
        # grids that follow the batch size; an odd node count; the inclusive policy.
        {"name": "restore_mixed", **_archive("restore", 48, 1237, groups=3, diff=0.05, grid_pct=20, memset_pct=8,
                                              memcpy_pct=4, event_pct=4, extra_pct=20, layout_pct=5, ragged=True,
                                              intervals=4096, inclusive=True)},
        # A whole cold LOAD of a smaller capture list, from files to groups.
        {"name": "load_files", **_archive("load", 64, 1200, groups=2)},
        # Sustained graph switching on the largest graphs (5000 nodes), the override scatter alone.
        {"name": "switch_sequence", **_archive("switch", 64, 5000, groups=8, min_blob=64, max_blob=3064, diff=0.04),
         "steps": 2000},
        # A serving loop that replays graphs of two groups, mostly its hot batch sizes.
        {"name": "replay_steps", **_archive("replay", 24, 300, groups=2), "steps": 12},
        # One moved region (the most common relocation), a decode archive's params.
        {"name": "reloc_region", "kind": "reloc", "words": 20523776, "intervals": 1, "pointers": 0.25,
         "inclusive": False},
        # The same params by a table of 40k allocations.
        {"name": "reloc_decode", "kind": "reloc", "words": 20523777, "intervals": 40000, "pointers": 0.25,
         "inclusive": False},
        # 1 GiB of words by a table of 2M allocations.
        {"name": "reloc_heavy", "kind": "reloc", "words": 1 << 27, "intervals": 2000000, "pointers": 0.4,
         "inclusive": False},
        # A LOAD that learns where its allocations lie now and relocates once.
        {"name": "plan_once", "kind": "plan", "words": 4000000, "intervals": 200000, "pointers": 0.25,
         "inclusive": False},
        # A serving loop that may not allocate: graphs' params by a small table, one call each.
        {"name": "static_calls", "kind": "static", "words": 30011, "intervals": 1000, "pointers": 0.25,
         "inclusive": False, "steps": 8},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_archive(rng, kind, graphs, nodes, param_bytes):
    g = _log(rng, *graphs)
    n = _log(rng, *nodes)
    mixed = rng.random() < 0.35
    moe = not mixed and rng.random() < 0.35
    top = 8 * _log(rng, 16, 512 if moe else 128)
    top = max(64, min(top, 8 * int(param_bytes / (4.0 * g * n))))
    c = _archive(kind, g, n, groups=rng.randint(1, max(1, min(16, g // 4))), min_blob=8 * rng.randint(1, 6), max_blob=top,
                 params=rng.randint(4, 40 if moe else 16), pointers=rng.choice([0.1, 0.25, 0.4]),
                 diff=rng.choice([0.01, 0.03, 0.05, 0.1]), run_bytes=256 if moe else 0,
                 intervals=_log(rng, 1, 40000))
    if kind == "replay":
        c["max_blob"] = min(c["max_blob"], 1024)
        return c
    if moe or mixed:
        c.update(memset_pct=10, memcpy_pct=5)
    if mixed:
        c.update(event_pct=4, extra_pct=rng.choice([0, 10, 40]), layout_pct=rng.choice([0, 5]),
                 ragged=rng.random() < 0.6, inclusive=rng.random() < 0.5)
    return c


def draw(rng):
    kind = rng.choice(["restore", "restore", "restore", "load", "switch", "replay", "reloc", "reloc", "plan", "static"])
    if kind == "restore":
        return _draw_archive(rng, kind, (8, 256), (40, 3500), 3.5e8)
    if kind == "load":
        return _draw_archive(rng, kind, (4, 64), (40, 2000), 5e7)
    if kind == "switch":
        return {**_draw_archive(rng, kind, (8, 96), (100, 5000), 2e8), "steps": _log(rng, 50, 2000)}
    if kind == "replay":
        return {**_draw_archive(rng, kind, (4, 32), (20, 400), 2e7), "steps": rng.randint(2, 12)}
    c = {"kind": kind, "pointers": rng.choice([0.1, 0.25, 0.4]), "inclusive": rng.random() < 0.3}
    if kind == "reloc":
        return {**c, "words": _log(rng, 1000, 1 << 26), "intervals": _log(rng, 1, 2000000)}
    if kind == "plan":
        return {**c, "words": _log(rng, 1000, 1 << 24), "intervals": _log(rng, 1, 400000)}
    return {**c, "words": _log(rng, 100, 1 << 20), "intervals": _log(rng, 1, 20000), "steps": rng.randint(2, 8)}


# ---- archives --------------------------------------------------------------


class _OnDevice(list):
    """Results that stay in the archive's device buffers; read out when iterated."""

    def __init__(self, read):
        super().__init__()
        self._read = read

    def __iter__(self):
        return iter(self._read())


def _whole(arrays, dtype, size):
    """The arrays end to end, then zeros up to `size`, which the case alone gives (what a seed draws is smaller)."""
    out = np.zeros(size, dtype)
    at = 0
    for a in arrays:
        a = np.ascontiguousarray(a).view(dtype)
        out[at:at + a.size] = a
        at += a.size
    return out if dtype == np.int64 else out.astype(np.int64)


def _graph_words(case):
    """No graph's param image holds more words: every node's largest blob, each of its params padded to a word."""
    return case["nodes"] * (case["max_blob"] // 8 + (case["params"] if case["ragged"] else 0))


def _read_restore(arch, case):
    graphs, n = range(arch.num_graphs), case["graphs"]
    words = n * _graph_words(case)
    nodes = n * (case["nodes"] + 8)
    return [arch.groups().astype(np.int64), arch.status().astype(np.int64), arch.digests().view(np.int64),
            arch.override_offsets().view(np.int64), arch.param_bytes().view(np.int64),
            _whole((arch.param_image(g) for g in graphs), np.int64, words),
            _whole((arch.overrides(g) for g in graphs), np.int64, 2 * int(2 * case["diff"] * words) + 1024),
            _whole((arch.node_words(g) for g in graphs), np.int32, nodes),
            _whole((arch.node_flags(g) for g in graphs), np.uint8, nodes),
            _whole((arch.node_pointers(g) for g in graphs), np.int64, 2 * nodes)]


def _read_live(arch, case, templates):
    live = [arch.live(t) for t in templates]
    n = case["groups"]
    return [_whole((w for w, _, _ in live), np.int64, n * _graph_words(case)),
            _whole((s for _, s, _ in live), np.int32, n * (case["nodes"] + 8)),
            np.array([c for _, _, c in live], np.int64)]


def _synthesise(case, seed, sink_hash=0):
    p = synth.preset(
        2, num_graphs=case["graphs"], num_groups=case["groups"], nodes_per_graph=case["nodes"],
        min_blob_bytes=case["min_blob"], max_blob_bytes=case["max_blob"], max_params=case["params"],
        ragged=int(case["ragged"]), extra_style_pct=case["extra_pct"], memset_pct=case["memset_pct"],
        memcpy_pct=case["memcpy_pct"], event_pct=case["event_pct"], grid_bs_pct=case["grid_pct"],
        layout_var_pct=case["layout_pct"], run_min_bytes=64 if case["run_bytes"] else 0,
        run_max_bytes=case["run_bytes"], pointer_frac=case["pointers"], diff_lo=case["diff"] / 2,
        diff_hi=case["diff"] * 1.5, seed=(0x5EED0000 + 7919 * seed) & 0xFFFFFFFFFFFF, num_intervals=case["intervals"],
        sink_hash=sink_hash)
    if not case["run_bytes"]:
        p.diff_lo = p.diff_hi = case["diff"]
    return synth.SynthArchive(p)


class _Archive:
    """A restored archive and what a program keeps beside it; closed with its last reference."""

    def __init__(self, case, seed):
        self.case, self.kind = dict(case), case["kind"]
        self.registry, self.graphs = None, {}
        sink = 0
        if self.kind == "replay":
            self.registry = Registry()
            sink = self.registry.add_file(PROBE_CO)
        s = _synthesise(case, seed, sink)
        self.table = s.intervals()
        self.policy = int(case["inclusive"])
        self.arch = None
        if self.kind == "load":
            self.folder = tempfile.TemporaryDirectory()
            self.paths = s.write_dir(self.folder.name)
            return
        self.arch = Archive.from_synth(s)
        self.arch.set_relocation(*self.table, policy=self.policy)
        stream = torch.cuda.current_stream()
        self.arch.restore(stream)
        # The first read settles the restore's scratch, as in every program.
        self.template_of = self.arch.groups(stream)
        self.templates = [int(t) for t in np.unique(self.template_of)]
        if self.kind == "switch":
            self.targets = synth.switch_sequence(seed + 1, case["graphs"], case["steps"])
            self.arch.switch_sequence(self.targets[:1], stream)
        if self.kind == "replay":
            for t in self.templates:
                self.graphs[t] = GroupGraph(self.arch, t, self.registry, stream)
            # Three hot batch sizes of each group take four steps of five.
            rng = np.random.default_rng(seed + 2)
            hot = [int(g) for t in self.templates for g in np.flatnonzero(self.template_of == t)[:3]]
            self.targets = [int(rng.choice(hot)) if rng.random() < 0.8 else int(rng.integers(case["graphs"]))
                            for _ in range(case["steps"])]

    def __del__(self):
        for g in getattr(self, "graphs", {}).values():
            g.close()
        if getattr(self, "arch", None) is not None:
            self.arch.close()
        if getattr(self, "registry", None) is not None:
            self.registry.close()


def _run_archive(a):
    stream = torch.cuda.current_stream()
    if a.kind == "restore":
        a.arch.restore(stream)
        return _OnDevice(lambda: _read_restore(a.arch, a.case))
    if a.kind == "load":
        arch = Archive.open(a.paths)
        arch.set_relocation(*a.table, policy=a.policy)
        arch.restore(stream)
        template_of = arch.groups(stream)
        return [template_of.astype(np.int64), _OnDevice(lambda: _read_restore(arch, a.case))]
    if a.kind == "switch":
        a.arch.switch_sequence(a.targets, stream)
    else:
        for g in a.targets:
            a.graphs[int(a.template_of[g])].replay(g, stream)
    return _OnDevice(lambda: _read_live(a.arch, a.case, a.templates))


# ---- packed words ----------------------------------------------------------


def _table(rng, n):
    """n allocations that tile a region, sizes log-uniform over 256 B to 64 MiB in 256-byte granules, and their new
    places: the same allocations in another order from NEW_BASE.  One interval: a 4 GiB region moved whole."""
    if n == 1:
        lo = np.array([REGION_BASE], np.uint64)
        return lo, lo + np.uint64(1 << 32), np.array([NEW_BASE + (rng.integers(1, 64) << 21)], np.uint64)
    size = np.exp(rng.uniform(np.log(256.0), np.log(64.0 * 2**20), n))
    size = 256 * (1 + (size * min(1.0, 100e3 / size.mean()) / 256).astype(np.uint64))  # about 100 kB each at most
    hi = np.uint64(REGION_BASE) + np.cumsum(size, dtype=np.uint64)
    lo = hi - size
    order = rng.permutation(n)
    new_lo = np.empty(n, np.uint64)
    new_lo[order] = np.uint64(NEW_BASE) + np.cumsum(size[order], dtype=np.uint64) - size[order]
    return lo, hi, new_lo


def _words(rng, table, n, pointers):
    """n packed param words on the GPU: pointers uniform over the allocations and inside each, 1% of them on an
    allocation's edges; the rest pairs of random 32-bit numbers."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(rng.integers(1 << 62)))
    lo = torch.from_numpy(table[0].view(np.int64)).to(dev)
    hi = torch.from_numpy(table[1].view(np.int64)).to(dev)
    out = torch.empty(n, dtype=torch.int64, device=dev)
    step = 1 << 24
    for at in range(0, n, step):
        m = min(step, n - at)
        u = torch.rand(m, device=dev, generator=gen, dtype=torch.float64)
        i = torch.randint(0, len(lo), (m,), device=dev, generator=gen)
        v = torch.rand(m, device=dev, generator=gen, dtype=torch.float64)
        l, h = lo[i], hi[i]
        p = l + ((v * (h - l).double()).long().clamp(min=0) & ~7)
        edge = torch.stack([l, h - 1, h, l - 1])
        e = torch.randint(0, 4, (m,), device=dev, generator=gen)
        on_edge = torch.rand(m, device=dev, generator=gen) < 0.01
        p = torch.where(on_edge, edge.gather(0, e[None])[0], p)
        other = torch.randint(-(1 << 62), 1 << 62, (m,), device=dev, generator=gen)
        out[at:at + m] = torch.where(u < pointers, p, other)
    return out


class _Words:
    def __init__(self, case, seed):
        rng = np.random.default_rng([seed, 77])
        self.kind, self.policy = case["kind"], int(case["inclusive"])
        self.table = _table(rng, case["intervals"])
        self.inputs = [_words(rng, self.table, case["words"], case["pointers"])
                       for _ in range(case.get("steps", 1))]
        self.outputs = [torch.empty_like(w) for w in self.inputs]
        self.plan = RelocPlan(*self.table, policy=self.policy) if self.kind == "reloc" else None


def _run_words(s):
    stream = torch.cuda.current_stream()
    plan = RelocPlan(*s.table, policy=s.policy) if s.kind == "plan" else s.plan
    for w, o in zip(s.inputs, s.outputs):
        if s.kind == "static":
            relocate_words_static(*s.table, w.data_ptr(), o.data_ptr(), w.numel(), policy=s.policy, stream=stream)
        else:
            plan.relocate(w.data_ptr(), o.data_ptr(), w.numel(), stream)
    if s.kind == "plan":
        stream.synchronize()  # the plan goes with this pass: its index is in use until here
        plan.close()
    return s.outputs


# ---- the interface ---------------------------------------------------------


def _of_words(case):
    return case["kind"] in ("reloc", "plan", "static")


def prepare(case, seed):
    return _Words(case, seed) if _of_words(case) else _Archive(case, seed)


def run(state):
    return _run_words(state) if isinstance(state, _Words) else _run_archive(state)


def work(case):
    """Bytes that a pass cannot do without, from the sizes that the case asks for."""
    if _of_words(case):
        return {"bytes": 16.0 * case["words"] * case.get("steps", 1) + 24.0 * case["intervals"], "flops": 0.0}
    nodes = case["graphs"] * case["nodes"]
    kernels = nodes * (100 - case["memset_pct"] - case["memcpy_pct"] - case["event_pct"]) / 100
    params = kernels * (case["min_blob"] + case["max_blob"]) / 2
    records = 16.0 * case["diff"] * params / 8 * (1 - case["groups"] / case["graphs"])
    # A node entry and its dependency; a kernel's name and its param entries.
    image = nodes * 176.0 + kernels * (20 + 4 * (case["params"] + 1)) + params
    if case["kind"] == "restore":
        return {"bytes": image + params + records, "flops": 0.0}
    if case["kind"] == "load":  # files to HBM, then the restore
        return {"bytes": 2 * image + params + records, "flops": 0.0}
    # A switch reads the old and the new graph's records and writes as many words.
    per_step = 2 * 24.0 * case["diff"] * params / 8 / case["graphs"]
    if case["kind"] == "replay":  # and launches a node's params each
        per_step += params / case["graphs"]
    return {"bytes": per_step * case["steps"], "flops": 0.0}


def tolerance(case):
    """Addresses, counts and param bytes: whole numbers, the same bit for bit."""
    return "exact"


def exact(case, seed):
    """Relocated words by a binary search in plain torch; the other kinds have no form in plain torch."""
    if not _of_words(case):
        return None
    s = _Words({**case, "kind": "words"}, seed)
    lo, hi, new_lo = (torch.from_numpy(a.view(np.int64)).cuda() for a in s.table)
    out = []
    for w in s.inputs:
        i = torch.searchsorted(lo, w, right=True) - 1
        j = i.clamp(min=0)
        inside = (i >= 0) & ((w <= hi[j]) if s.policy else (w < hi[j]))
        out.append(torch.where(inside, w - lo[j] + new_lo[j], w))
    return out
