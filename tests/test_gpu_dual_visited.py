"""The dual-channel traversal with both forms of its visited set (a bit per
row up to as many queries as the chip holds with them, the hash table beyond)
and with one and two cross edges to choose the partner from, bit for bit
against the oracle."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


# 250k rows take 31488 bytes of bits: four waves of L = 40 per CU, 1024 queries
# on 256 CUs; one more goes to the hash table.
@pytest.mark.parametrize("N,E,L,R,Q", [(2048, 1, 16, 16, 16), (2049, 2, 40, 32, 16), (250000, 2, 40, 16, 1024),
                                       (250000, 2, 40, 16, 1025)])
def test_dual_visited_set_matches_oracle(N, E, L, R, Q):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] dual visited set N={N} E={E} L={L} R={R} Q={Q}", flush=True)
    K = 10
    grid = [2, 3] if N < 10000 else [4, 4]
    vec = synth.uniform_int_vectors(N, 64, 700)
    att = synth.uniform_attrs(N, 2, 710)
    ix = synth.build_index(vec, att, grid, R, E, 0, device="hip")
    qv = synth.uniform_int_vectors(Q, 64, 720)
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 0.1, 1.0, 730), 740)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    dev = synth.open_device_index(ix)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], L)
    b.mark_cells(0.0)
    ids, dists, st = b.search(L=L, K=K, entry_points=ent, channels=2)
    cells, counts, little, _ = b.get_cells()
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"])
    orc.set_channels(2)
    try:
        oids, odist, octr = O.search(qv, lo, hi, cells, counts, little, ent, L)
    finally:
        orc.set_channels(1)
    assert st.q_traverse == Q
    assert np.array_equal(ids, oids)
    assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    assert np.array_equal(b.get_counters(), octr)
    b.close()
    dev.close()
