"""One batch at a padded dimension under prefilters in turn: the matrix-core
route at 1, by size at 0.3, the gather kernel at 0.05 for the few narrow
queries it sends to the brute force, bit for bit against the oracle each
time."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,Q,routes", [("int", 700, (1, 0, 0)), ("int", 2000, (1, 1, 0)), ("f32", 700, (2, 0, 0)),
                                           ("f32", 3000, (2, 2, 0)), ("f16", 1400, (2, 0, 0))])
def test_padded_route_by_prefilter(rows, Q, routes):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] padded route rows={rows} Q={Q}", flush=True)
    N, D, R, L, K = 14001, 104 if rows == "f16" else 100, 16, 32, 10
    make = synth.uniform_int_vectors if rows == "int" else synth.gaussian_unit_vectors
    vec, qv = make(N, D, 80), make(Q, D, 81)
    att = synth.uniform_attrs(N, 2, 82)
    ix = synth.build_index(vec, att, [3, 2], R, 1, 0, device="hip")
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 0.01, 0.5, 83), 84)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    half = rows == "f16"
    dev = synth.open_device_index(ix, vec_dtype=gf.VEC_F16 if half else gf.VEC_F32)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"],
                        vec_f16=orc.f2h(vec) if half else None)
    want = {}
    for _ in range(3):   # eager, then captured anew at every change of route
        for prefilter, route in zip((1.0, 0.3, 0.05), routes):
            b.mark_cells(prefilter)
            if prefilter not in want:
                cells, counts, little, _ = b.get_cells()
                want[prefilter] = O.search(orc.f2h(qv) if half else qv, lo, hi, cells, counts, little, ent, L, K=K)
            ids, dists, st = b.search(L=L, K=K, entry_points=ent)
            oids, odist, _ = want[prefilter]
            assert st.bf_mfma == route
            assert np.array_equal(ids, oids)
            assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    b.close()
    dev.close()
