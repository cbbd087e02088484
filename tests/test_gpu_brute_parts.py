"""The gather brute force in parts, bit for bit against the oracle: one query
(every part a few rows, some none), queries of very different reach, more
queries than the launch has parts for (one wave each), and the one-call entry
point, whose scratch holds the parts."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q,K,N", [(1, 10, 1501), (3, 64, 90), (33, 1, 1501), (40, 20, 9000), (4500, 5, 700)])
def test_brute_parts_match_oracle(Q, K, N):
    import garfield_amd as gf
    from oracle import oracle as orc
    print(f"[case] brute parts Q={Q} K={K} N={N}", flush=True)
    R, L = 16, 64
    vec = synth.gaussian_unit_vectors(N, 52, 700)     # no matrix-core route at this width
    vec[N // 2] = vec[0]                              # equal distances
    att = synth.uniform_attrs(N, 2, 710, hi=500)
    ix = synth.build_index(vec, att, [2, 3], R, 1, 0)
    qv = synth.gaussian_unit_vectors(Q, 52, 720)
    lo, hi = synth.ranges_for_selectivity(Q, 2, synth.log_uniform(Q, 0.002, 1.0, 730), 740, hi=500)
    lo, hi = lo.astype(np.float32), hi.astype(np.float32)
    if Q > 1:
        lo[0], hi[0] = 0, 499
        lo[1], hi[1] = 5, 4
    dev = synth.open_device_index(ix)
    b = dev.batch(qv, lo, hi)
    ent = gf.entry_points(N, ix["P"], R)
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"])
    for prefilter in (1.0, 0.1):
        b.mark_cells(prefilter)
        cells, counts, little, _ = b.get_cells()
        oids, odist, octr = O.search(qv, lo, hi, cells, counts, little, ent, L, K=K)
        for _ in range(3):   # eager, captured, replayed
            ids, dists, _ = b.search(L=L, K=K, entry_points=ent)
            assert np.array_equal(ids, oids)
            assert np.array_equal(dists.view(np.uint32), odist.view(np.uint32))
            assert np.array_equal(b.get_counters(), octr)
        nids, ndist = gf.search_noalloc(dev, qv, lo, hi, prefilter, L=L, K=K, entry_points=ent)
        assert np.array_equal(nids, oids)
        assert np.array_equal(ndist.view(np.uint32), odist.view(np.uint32))
    b.close()
    dev.close()
