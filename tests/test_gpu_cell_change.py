"""The traversal's move from one cell to the next, bit for bit against the
oracle: every number of cross edges (up to two take the parallel route, more
the slot-by-slot one), cells smaller than the 128 slots, lists shorter than
the 64 candidates that feed them, and repeated points, whose cross edges
coincide."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,N,L", [(1, 700, 40), (2, 700, 130), (3, 700, 64), (4, 2500, 100), (2, 2500, 10),
                                   (1, 2500, 300)])
def test_cell_change_matches_oracle(E, N, L):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] cell change E={E} N={N} L={L}", flush=True)
    Q, R, K, grid = 48, 16, 10, [3, 4]
    vec = synth.uniform_int_vectors(N, 64, 500 + E)
    vec[N // 2:N // 2 + 60] = vec[:60]               # equal points in other cells
    att = synth.uniform_attrs(N, 2, 510 + E, hi=1000)
    ix = synth.build_index(vec, att, grid, R, E, 8, seed=9)
    qv = synth.uniform_int_vectors(Q, 64, 520 + E)
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 0.1, 1.0, 530), 540, hi=1000)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    dev = synth.open_device_index(ix)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    b.mark_cells(0.0)
    b.order_cells(4)
    ids, dists, _ = b.search(L=L, K=K, entry_points=ent)
    cells, counts, little, _ = b.get_cells()
    assert counts.max() > 4
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"])
    oids, odist, octr = O.search(qv, lo, hi, cells, counts, little, ent, L)
    assert np.array_equal(ids, oids)
    assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    assert np.array_equal(b.get_counters(), octr)
    b.close()
    dev.close()
