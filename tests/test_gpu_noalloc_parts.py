"""gf_search_noalloc on both sides of the batch size from which its scratch no
longer holds the arrays of the brute force in parts: the largest batch it
takes (one wave a query) and a smaller one (parts), both with a few brute-force
queries among empty ones, against the oracle."""
import numpy as np
import pytest

from garfield_amd import synth

pytestmark = pytest.mark.gpu


def test_noalloc_without_room_for_parts():
    import garfield_amd as gf
    from oracle import oracle as orc
    N, D, R, L, K = 3001, 52, 16, 64, 64
    vec = synth.gaussian_unit_vectors(N, D, 90)
    att = synth.uniform_attrs(N, 2, 91, hi=500)
    ix = synth.build_index(vec, att, [2, 3], R, 1, 0)
    dev = synth.open_device_index(ix)
    ent = gf.entry_points(N, ix["P"], R)
    O = orc.OracleIndex(ix["vectors"], ix["attrs"], ix["global_pid"], ix["P"], ix["cell_graphs"], ix["cross"])
    most = 65536
    qv = np.zeros((most, D), np.float32)
    lo, hi = np.full((most, 2), 5, np.float32), np.full((most, 2), 4, np.float32)   # empty
    real = np.arange(20) * 97
    qv[real] = synth.gaussian_unit_vectors(real.size, D, 92)
    l, h = synth.ranges_for_selectivity(real.size, 2, synth.log_uniform(real.size, 0.02, 1.0, 93), 94, hi=500)
    lo[real], hi[real] = l, h
    assert real[-1] < 2000

    def fits(n):
        try:
            return gf.search_noalloc(dev, qv[:n], lo[:n], hi[:n], 1.0, L=L, K=K, entry_points=ent)
        except gf.GarfieldError as e:
            assert "scratch" in str(e)
            return None
    a, z = 2000, most          # a fits, z does not
    assert fits(a) and not fits(z)
    while z - a > 1:
        m = (a + z) // 2
        a, z = (m, z) if fits(m) else (a, m)
    b = dev.batch(qv[real], lo[real], hi[real])
    b.mark_cells(1.0)
    cells, counts, little, _ = b.get_cells()
    oids, odist, _ = O.search(qv[real], lo[real], hi[real], cells, counts, little, ent, L, K=K)
    b.close()
    # the parts' arrays take 4096 K keys: 2 MiB, more than a query's room
    for n in (a, a * 7 // 8):
        print(f"[case] noalloc parts Q={n}", flush=True)
        ids, dist = fits(n)
        assert np.array_equal(ids[real], oids)
        assert np.array_equal(dist[real].view(np.uint32), odist.view(np.uint32))
        rest = np.setdiff1d(np.arange(n), real)
        assert (ids[rest] == orc.SENTINEL).all()
    dev.close()
