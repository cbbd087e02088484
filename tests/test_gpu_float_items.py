"""The float matrix-core brute force with items of whole sub-cells, which large
batches over even sub-cells take, bit for bit against the oracle."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


# some 160 sub-cells of 63 tiles each times 91 query groups: above 14000 items
@pytest.mark.parametrize("rows,D", [("f32", 64), ("f16", 64), ("f16", 96)])
def test_whole_items_match_oracle(rows, D):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] whole items rows={rows} D={D}", flush=True)
    N, Q, R, L, K = 161_000, 5800, 8, 32, 10
    vec, qv = synth.gaussian_unit_vectors(N, D, 50), synth.gaussian_unit_vectors(Q, D, 51)
    att = synth.uniform_attrs(N, 2, 52)
    ix = synth.build_index(vec, att, [16, 10], R, 1, 0, device="hip")
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 1e-5, 1e-3, 53), 54)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    lo[5], hi[5] = 0, 10**6
    half = rows == "f16"
    dev = synth.open_device_index(ix, vec_dtype=gf.VEC_F16 if half else gf.VEC_F32)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    b.mark_cells(1.0)
    cells, counts, little, _ = b.get_cells()
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"],
                        vec_f16=orc.f2h(vec) if half else None)
    oids, odist, _ = O.search(orc.f2h(qv) if half else qv, lo, hi, cells, counts, little, ent, L, K=K)
    for _ in range(3):   # eager, captured, replayed
        ids, dists, st = b.search(L=L, K=K, entry_points=ent)
        assert st.bf_mfma == 2
        assert np.array_equal(ids, oids)
        assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    b.close()
    dev.close()
