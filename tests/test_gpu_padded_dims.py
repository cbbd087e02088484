"""The matrix-core brute force at dimensions that its records pad with zeros:
just above a supported dimension, just below one, and odd chunk counts, for
each row type, bit for bit against the oracle; the batch sizes on either side
of the line below which the gather kernel runs."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,D,Q,mfma", [("f32", 68, 700, 2), ("f32", 100, 700, 2), ("f32", 252, 500, 2),
                                           ("f32", 100, 60, 0), ("f16", 72, 800, 2), ("f16", 136, 700, 2),
                                           ("f16", 264, 500, 2), ("int", 4, 800, 1), ("int", 100, 700, 1),
                                           ("int", 200, 300, 1), ("int", 100, 60, 0), ("u8", 80, 700, 1),
                                           ("u8", 240, 600, 1)])
def test_padded_dims_match_oracle(rows, D, Q, mfma):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] padded dims rows={rows} D={D} Q={Q}", flush=True)
    N, R, L, K = 14001, 16, 32, 10
    ints = rows in ("int", "u8")
    make = synth.uniform_int_vectors if ints else synth.gaussian_unit_vectors
    vec, qv = make(N, D, 800 + D), make(Q, D, 810 + D)
    vec[N // 2] = vec[7]
    att = synth.uniform_attrs(N, 3 if D % 3 else 2, 820)
    a = att.shape[1]
    ix = synth.build_index(vec, att, [3, 2, 1][:a], R, 1, 0, device="hip")
    lo, hi = synth.ranges_for_selectivity(Q, a, synth.log_uniform(Q, 0.002, 1.0, 830), 840)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    lo[0], hi[0] = 5, 4
    dt = {"f32": gf.VEC_F32, "f16": gf.VEC_F16, "int": gf.VEC_F32, "u8": gf.VEC_U8}[rows]
    dev = synth.open_device_index(ix, vec_dtype=dt)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    b.mark_cells(1.0)
    cells, counts, little, _ = b.get_cells()
    half = rows == "f16"
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"],
                        vec_f16=orc.f2h(vec) if half else None, u8=rows == "u8")
    oids, odist, _ = O.search(orc.f2h(qv) if half else qv, lo, hi, cells, counts, little, ent, L, K=K)
    for _ in range(3):   # eager, captured, replayed
        ids, dists, st = b.search(L=L, K=K, entry_points=ent)
        assert st.bf_mfma == mfma
        assert np.array_equal(ids, oids)
        assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    b.close()
    dev.close()
