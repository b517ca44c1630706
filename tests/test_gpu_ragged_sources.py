"""Ragged-word sources (k_aux): sixteen lanes take a node's param entries in
batches of sixteen, sixteen nodes per step of a 256-node chunk.  Archives at
the edges of those splits -- one node, a step more or less than full, a chunk
more or less than full; one param, a batch more or less than full, several
batches -- with ragged params and arg buffers, against the oracle bit for
bit.  The first restore of such an archive finds ragged nodes without the
array and runs again with it; the second has it from the start."""
import pytest

from foundry_amd import synth
from tests.parity import assert_restore_parity, gpu_and_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("params", [1, 15, 16, 17, 33, 48])
@pytest.mark.parametrize("nodes", [1, 15, 17, 255, 257])
def test_ragged_sources_at_the_edges(cuda, nodes, params):
    print(f"[case] ragged sources: {nodes} nodes, up to {params} params", flush=True)
    s = synth.SynthArchive(synth.preset(
        2, num_graphs=5, num_groups=2, nodes_per_graph=nodes, min_blob_bytes=8, max_blob_bytes=max(64, 24 * params),
        max_params=params, ragged=1, extra_style_pct=25, memset_pct=5, layout_var_pct=10, diff_lo=0.1, diff_hi=0.1,
        num_intervals=64, seed=0x5EED7000 + 64 * nodes + params))
    arch, ref = gpu_and_oracle(s)
    assert_restore_parity(arch, ref)
    arch.restore()
    assert_restore_parity(arch, ref)
    arch.close()
