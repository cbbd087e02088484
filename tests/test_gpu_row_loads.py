"""The traversal's and the gather brute force's row and attribute loads at the
sizes where they can go wrong: attribute counts around the 16-byte loads (the
last rows' loads reach into the array's padding) and dimensions whose chunks
do not fill the lanes (the idle lanes repeat a chunk), bit for bit against the
oracle."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu

GRIDS = {1: [4], 3: [2, 2, 1], 4: [2, 1, 2, 1], 5: [2, 1, 1, 1, 2], 8: [2, 1, 1, 1, 1, 1, 1, 2]}


@pytest.mark.parametrize("a,rows,D", [(1, "f32", 100), (3, "f32", 36), (4, "f16", 104), (5, "u8", 112),
                                      (8, "f32", 260), (8, "f16", 24)])
def test_row_loads_match_oracle(a, rows, D):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] row loads a={a} rows={rows} D={D}", flush=True)
    N, Q, R, K = 1501, 40, 16, 10
    vec = synth.uniform_int_vectors(N, D, 300 + a)
    if rows != "u8":
        vec = (vec - 100.0) / np.float32(64.0)
    att = synth.uniform_attrs(N, a, 310 + a, hi=200)
    ix = synth.build_index(vec, att, GRIDS[a], R, 2, 8, seed=7)
    qv = synth.uniform_int_vectors(Q, D, 320 + a)
    if rows != "u8":
        qv = (qv - 100.0) / np.float32(64.0)
    sel = synth.log_uniform(Q, 0.05, 0.9, 330 + a)
    lo, hi = synth.ranges_for_selectivity(Q, a, sel, 340 + a, hi=200)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    dt = {"f32": gf.VEC_F32, "f16": gf.VEC_F16, "u8": gf.VEC_U8}[rows]
    dev = synth.open_device_index(ix, vec_dtype=dt)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    half = rows == "f16"
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"],
                        vec_f16=orc.f2h(vec) if half else None, u8=rows == "u8")
    for prefilter, L in ((0.0, 33), (0.2, 64)):
        b.mark_cells(prefilter)
        b.order_cells(4)
        ids, dists, st = b.search(L=L, K=K, entry_points=ent)
        cells, counts, little, _ = b.get_cells()
        oids, odist, octr = O.search(orc.f2h(qv) if half else qv, lo, hi, cells, counts, little, ent, L)
        assert np.array_equal(ids, oids)
        assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
        if prefilter == 0.0:
            assert np.array_equal(b.get_counters(), octr)
    b.close()
    dev.close()
