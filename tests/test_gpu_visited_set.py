"""Both forms of the traversal's visited set, bit for bit against the oracle:
one bit per cell-local id up to the largest cell that takes it, the hash
table one point above that and where a long list's table outgrows the bits."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,grid,L", [(65536, [1, 1], 40), (65537, [1, 1], 40), (9000, [2, 2], 700),
                                      (1100, [4, 4], 1200)])
def test_visited_set_matches_oracle(N, grid, L):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] visited set N={N} grid={grid} L={L}", flush=True)
    Q, R, K = 24, 16, 10
    vec = synth.uniform_int_vectors(N, 64, 600)
    att = synth.uniform_attrs(N, 2, 610)
    ix = synth.build_index(vec, att, grid, R, 1, 0, device="hip")
    qv = synth.uniform_int_vectors(Q, 64, 620)
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 0.2, 1.0, 630), 640)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    dev = synth.open_device_index(ix)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    b.mark_cells(0.0)
    ids, dists, _ = b.search(L=L, K=K, entry_points=ent)
    cells, counts, little, _ = b.get_cells()
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"])
    oids, odist, octr = O.search(qv, lo, hi, cells, counts, little, ent, L)
    assert np.array_equal(ids, oids)
    assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    assert np.array_equal(b.get_counters(), octr)
    b.close()
    dev.close()
