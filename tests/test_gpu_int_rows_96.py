"""Integer-valued fp32 rows at 96 dimensions, which the fp32 matrix-core route
holds as they are and the int8 route pads: integer queries take the int8
route, non-integer ones the fp32 route, small batches of either the gather
kernel, bit for bit against the oracle."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frac,Q,K,mfma", [(0.0, 60, 10, 0), (0.0, 700, 10, 1), (0.0, 700, 16, 1), (0.25, 30, 10, 0),
                                           (0.25, 1000, 10, 2), (0.25, 1000, 11, 0)])
def test_int_rows_96_match_oracle(frac, Q, K, mfma):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] int rows 96 frac={frac} Q={Q} K={K}", flush=True)
    N, D, R, L = 14001, 96, 16, 32
    vec, qv = synth.uniform_int_vectors(N, D, 60), synth.uniform_int_vectors(Q, D, 61) + np.float32(frac)
    vec[N // 2] = vec[7]
    att = synth.uniform_attrs(N, 2, 62)
    ix = synth.build_index(vec, att, [3, 2], R, 1, 0, device="hip")
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 0.002, 1.0, 63), 64)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    dev = synth.open_device_index(ix)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    b.mark_cells(1.0)
    cells, counts, little, _ = b.get_cells()
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"])
    oids, odist, _ = O.search(qv, lo, hi, cells, counts, little, ent, L, K=K)
    for _ in range(3):   # eager, captured, replayed
        ids, dists, st = b.search(L=L, K=K, entry_points=ent)
        assert st.bf_mfma == mfma
        assert np.array_equal(ids, oids)
        assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    b.close()
    dev.close()
