"""Switch sequences by tiles (k_switch_seq) at the edges of their splits:
templates of less than a 1024-word tile, a tile more or less than full and
many, words differing in none, some and nearly all of a tile (more records than
a workgroup has threads), one group and more groups than one launch holds,
more switches than one launch holds, layouts and descriptors that differ,
no-op switches, and sequences again after single switches and after another
restore.  Every template's live words, node sources and current graph equal
the oracle's after each sequence."""
import threading

import numpy as np
import pytest

import graph_cases as GC
from foundry_amd import synth
from tests.parity import gpu_and_oracle

pytestmark = pytest.mark.gpu


def _same_live(arch, ref, templates):
    for t in templates:
        w, src, cur = arch.live(t)
        w2, src2, cur2 = ref.live(t)
        assert cur == cur2, (t, cur, cur2)
        assert np.array_equal(w, w2), f"template {t}: {np.flatnonzero(w != w2)[:8]}"
        assert np.array_equal(src, src2), f"template {t}: node sources"


@pytest.mark.parametrize("graphs,groups,nodes,blob,diff,layout,steps", [
    (6, 1, 1, 64, 0.5, 0, 40),           # a few words
    (6, 2, 16, 512, 0.05, 0, 40),        # 1024 words a graph or a little less
    (6, 2, 17, 512, 0.05, 0, 40),        # and a little more
    (12, 3, 300, 700, 0.0, 0, 100),      # no words differ
    (12, 3, 300, 700, 0.03, 10, 300),    # layouts and descriptors
    (8, 2, 60, 2048, 0.95, 0, 60),       # most words: more records than threads
    (80, 40, 20, 256, 0.1, 5, 400),      # more groups than a launch holds
    (10, 1, 50, 256, 0.1, 0, 1500),      # more switches than a launch holds
])
def test_sequences_against_the_oracle(cuda, graphs, groups, nodes, blob, diff, layout, steps):
    print(f"[case] {steps} switches: {graphs} graphs x {nodes} nodes, {groups} groups, diff {diff}", flush=True)
    s = synth.SynthArchive(synth.preset(
        2, num_graphs=graphs, num_groups=groups, nodes_per_graph=nodes, min_blob_bytes=blob, max_blob_bytes=blob,
        max_params=8, diff_lo=diff, diff_hi=diff, layout_var_pct=layout, num_intervals=64, seed=0x5E9 + steps + nodes))
    arch, ref = gpu_and_oracle(s)
    of = arch.groups()
    templates = sorted(set(int(t) for t in of))
    seq = [int(g) for g in synth.switch_sequence(steps, graphs, steps)]
    seq[3:6] = [seq[2]] * 3  # no-op switches
    for part in (seq[: steps // 2], seq[steps // 2:]):
        arch.switch_sequence(part)
        for g in part:
            ref.switch(g)
        _same_live(arch, ref, templates)
    arch.switch(int(seq[0]))  # a single switch in between
    ref.switch(int(seq[0]))
    arch.switch_sequence(seq)
    for g in seq:
        ref.switch(g)
    _same_live(arch, ref, templates)
    arch.restore()  # the tables of the restore before are not this one's
    arch.groups()
    _, again = gpu_and_oracle(s)
    arch.switch_sequence(seq)
    for g in seq:
        again.switch(g)
    _same_live(arch, again, templates)
    arch.close()


def test_captured_sequence(cuda):
    """A sequence under stream capture enqueues kernels only, with its tables
    there (a longer sequence ran before) and without (it ran none): replays
    scatter what the eager sequence does."""
    s = synth.SynthArchive(synth.preset(2, num_graphs=8, num_groups=2, nodes_per_graph=40, num_intervals=64))
    for tables in (False, True):
        print(f"[case] captured switch sequence, tables {'built' if tables else 'missing'}", flush=True)
        arch, ref = gpu_and_oracle(s)
        templates = sorted(set(int(t) for t in arch.groups()))
        if tables:
            warm = [int(g) for g in synth.switch_sequence(1, 8, 40)]
            arch.switch_sequence(warm)
            for g in warm:
                ref.switch(g)
        seq = [int(g) for g in synth.switch_sequence(2, 8, 40)]
        cuda.cuda.synchronize()
        stream = cuda.cuda.Stream()
        graph = cuda.cuda.CUDAGraph()
        with cuda.cuda.graph(graph, stream=stream):
            arch.switch_sequence(seq, stream)
        for g in seq:
            ref.switch(g)
        for _ in range(3):  # the scatters leave the same live words from any state they left before
            graph.replay()
            cuda.cuda.synchronize()
            _same_live(arch, ref, templates)
        arch.close()


def _restored():
    s = synth.SynthArchive(synth.preset(2, num_graphs=12, num_groups=2, nodes_per_graph=60, num_intervals=64))
    arch, ref = gpu_and_oracle(s)
    templates = sorted(set(int(t) for t in arch.groups()))  # the restore's results are read here
    return arch, ref, templates


def test_first_sequence_waits_for_nothing(cuda):
    """The first sequence after a restore, which builds the tables, returns
    while the work queued on its stream before it is still running; a sequence
    on another stream, of the other group, comes behind the tables."""
    print("[case] first switch sequence behind a running kernel, and one on another stream", flush=True)
    arch, ref, templates = _restored()
    of = arch.groups()
    own = [[int(g) for g in np.flatnonzero(of == t)] for t in templates]
    first, second = (own[k][1:] * 8 for k in range(2))
    a, b = cuda.cuda.Stream(), cuda.cuda.Stream()
    with cuda.cuda.stream(a):
        cuda.cuda._sleep(100_000_000)
        slept = cuda.cuda.Event()
        slept.record(a)
    arch.switch_sequence(first, a)
    running = not slept.query()
    arch.switch_sequence(second, b)
    running_after = not slept.query()
    cuda.cuda.synchronize()
    assert running and running_after
    for g in first + second:
        ref.switch(g)
    _same_live(arch, ref, templates)
    arch.close()


def test_first_sequence_beside_a_capture_on_another_thread(cuda):
    """A thread's sequence, the first after a restore, on its own stream while
    another thread captures in the global mode: it runs, and the capture stays
    whole."""
    print("[case] first switch sequence while another thread captures", flush=True)
    arch, ref, templates = _restored()
    seq = [int(g) for g in synth.switch_sequence(3, 12, 40)]
    own, cap, graph = cuda.cuda.Stream(), cuda.cuda.Stream(), cuda.cuda.CUDAGraph()
    x = cuda.zeros(1000, device="cuda")
    failed = []

    def switches():
        try:
            arch.switch_sequence(seq, own)
        except Exception as e:  # reported below, once the capture has ended
            failed.append(e)

    cuda.cuda.synchronize()
    with cuda.cuda.graph(graph, stream=cap, capture_error_mode="global"):
        x.add_(1)
        t = threading.Thread(target=switches)
        t.start()
        t.join()
        x.add_(1)
    assert not failed, failed
    own.synchronize()
    for g in seq:
        ref.switch(g)
    _same_live(arch, ref, templates)
    for k in (1, 2, 3):
        graph.replay()
        cuda.cuda.synchronize()
        assert x.eq(2.0 * k).all()
    arch.close()


@pytest.mark.parametrize("graphs,groups,nodes,blob", [
    (8, 2, 40, 256),      # all tiles on the GPU together
    (9, 3, 5000, 1600),   # 2930 tiles, two rounds of them: layers for short sequences
])
def test_short_sequences_with_tables(cuda, graphs, groups, nodes, blob):
    """Sequences on either side of the rule that chooses layers or tiles, one
    after another on an archive whose tables are built: each leaves the live
    words that the oracle's switches leave, whichever kernel it took."""
    print(f"[case] short sequences: {graphs} graphs x {nodes} nodes, {groups} groups", flush=True)
    s = synth.SynthArchive(synth.preset(
        2, num_graphs=graphs, num_groups=groups, nodes_per_graph=nodes, min_blob_bytes=blob, max_blob_bytes=blob,
        max_params=8, diff_lo=0.03, diff_hi=0.03, num_intervals=64, seed=0x5E9A + nodes))
    arch, ref = gpu_and_oracle(s)
    of = arch.groups()
    own = [[int(g) for g in np.flatnonzero(of == t)] for t in sorted(set(int(t) for t in of))]
    for layers in (40, 1, 2, 3, 4, 12, 1, 16):
        seq = [m[(k + layers) % len(m)] for k in range(layers) for m in own]
        arch.switch_sequence(seq)
        for g in seq:
            ref.switch(g)
        _same_live(arch, ref, [m[0] for m in own])
    arch.close()


def test_sequences_in_the_serving_layout(cuda):
    """A sequence that builds the tables, then a group graph on one group (the
    archive packs its records and images, so the tables are another layout's),
    sequences of the other groups and of all, and after the group graph another
    restore and the first sequence again."""
    from foundry_amd.graph import GroupGraph, Registry

    print("[case] switch sequences before, in and after the serving layout", flush=True)
    reg = Registry()
    s = synth.SynthArchive(synth.preset(2, num_graphs=12, num_groups=3, nodes_per_graph=80, num_intervals=64,
                                        diff_lo=0.1, diff_hi=0.1, sink_hash=reg.add_file(GC.PROBE_CO)))
    arch, ref = gpu_and_oracle(s)
    of = arch.groups()
    templates = sorted(set(int(t) for t in of))
    seq = [int(g) for g in synth.switch_sequence(5, 12, 60)]
    others = [g for g in seq if of[g] != templates[0]]
    assert len(others) >= 16

    def run(targets, against):
        arch.switch_sequence(targets)
        for g in targets:
            against.switch(g)
        _same_live(arch, against, templates)

    run(seq, ref)
    gg = GroupGraph(arch, templates[0], reg, cuda.cuda.current_stream())
    assert arch.info()["serving_layout"] == 1
    ref.switch(templates[0])  # a new group graph is its template
    run(others, ref)
    run(seq, ref)  # the bound group's switches go through its group graph
    run(others[::-1], ref)
    gg.close()
    arch.restore()
    assert arch.info()["serving_layout"] == 0
    _, again = gpu_and_oracle(s)
    run(seq, again)
    arch.close()
    reg.close()
