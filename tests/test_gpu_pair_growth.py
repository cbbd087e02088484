"""Queries that reach every one of some 120 sub-cells of several chunks each,
bit for bit against the oracle: a batch of them, whose (query, sub-cell chunk)
pairs fit the first lists, and one whose every tenth query, the ones that size
the lists, is narrow, so that the pairs outgrow them and the first search runs
its brute force again in larger ones."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", ["int", "f32", "f16"])
def test_pair_lists_grow_over_chunks(rows):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] pair growth rows={rows}", flush=True)
    N, D, Q, R, L, K = 120_000, 64, 320, 8, 32, 10
    make = synth.uniform_int_vectors if rows == "int" else synth.gaussian_unit_vectors
    vec, qv = make(N, D, 40), make(Q, D, 41)
    att = synth.uniform_attrs(N, 2, 42)
    ix = synth.build_index(vec, att, [2, 2], R, 1, 0, device="hip")
    dt = {"f32": gf.VEC_F32, "f16": gf.VEC_F16, "int": gf.VEC_F32}[rows]
    half = rows == "f16"
    dev = synth.open_device_index(ix, vec_dtype=dt)
    ent = gf.entry_points(N, ix["P"], R)
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"],
                        vec_f16=orc.f2h(vec) if half else None)
    for every_tenth in (1.0, 0.002):
        sel = np.where(np.arange(Q) % 10 == 0, every_tenth, 1.0)
        lo, hi = synth.ranges_for_selectivity(Q, 2, sel, 43)
        lo, hi = lo.astype(np.float32), hi.astype(np.float32)
        b = dev.batch(qv, lo, hi)
        b.mark_cells(1.0)
        cells, counts, little, _ = b.get_cells()
        oids, odist, _ = O.search(orc.f2h(qv) if half else qv, lo, hi, cells, counts, little, ent, L, K=K)
        for _ in range(3):   # eager (grown), captured, replayed
            ids, dists, st = b.search(L=L, K=K, entry_points=ent)
            assert st.bf_mfma == (1 if rows == "int" else 2)
            assert np.array_equal(ids, oids)
            assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
        b.close()
    dev.close()
