"""The matrix-core brute force with its sub-cells' tiles in even chunks per
item: one tile more or less than a chunk, a sub-cell that is one chunk, the
last chunk shorter, and the batch sizes of each chunk length, bit for bit
against the oracle."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


# sub-cells of about 1024 points (N / their number below 1536): their tiles
# are ceil(n / 16), in chunks of at most 16 or 32 (int8), 48 (float rows).
@pytest.mark.parametrize("rows,N,grid,Q", [("int", 16 * 16, [1, 1], 70), ("int", 16 * 16 + 1, [1, 1], 130),
                                           ("int", 2 * 1500 - 7, [2, 1], 300), ("int", 33 * 16 * 6, [3, 2], 900),
                                           ("u8", 161000, [16, 10], 8100), ("f32", 48 * 16, [1, 1], 200),
                                           ("f32", 49 * 16, [1, 1], 200), ("f32", 6 * 1533, [3, 2], 700),
                                           ("f16", 4 * (48 * 16 + 1), [2, 2], 500)])
def test_item_chunks_match_oracle(rows, N, grid, Q):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] item chunks rows={rows} N={N} Q={Q}", flush=True)
    D, R, L, K = 64, 16, 32, 10
    ints = rows in ("int", "u8")
    make = synth.uniform_int_vectors if ints else synth.gaussian_unit_vectors
    vec, qv = make(N, D, 900 + Q), make(Q, D, 910 + Q)
    att = synth.uniform_attrs(N, 2, 920)
    ix = synth.build_index(vec, att, grid, R, 1, 0, device="hip")
    sel = synth.log_uniform(Q, 1e-5, 1e-3, 930) if N > 100000 else synth.log_uniform(Q, 0.002, 1.0, 930)
    lo, hi = synth.ranges_for_selectivity(Q, 2, sel, 940)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    half = rows == "f16"
    dt = {"f32": gf.VEC_F32, "f16": gf.VEC_F16, "int": gf.VEC_F32, "u8": gf.VEC_U8}[rows]
    dev = synth.open_device_index(ix, vec_dtype=dt)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    b.mark_cells(1.0)
    cells, counts, little, _ = b.get_cells()
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"],
                        vec_f16=orc.f2h(vec) if half else None, u8=rows == "u8")
    oids, odist, _ = O.search(orc.f2h(qv) if half else qv, lo, hi, cells, counts, little, ent, L, K=K)
    for _ in range(3):   # eager, captured, replayed
        ids, dists, st = b.search(L=L, K=K, entry_points=ent)
        assert st.bf_mfma == (1 if ints else 2)
        assert np.array_equal(ids, oids)
        assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
    b.close()
    dev.close()
