"""Graph optimisation over groups of cells: the second step's scratch held so
small that the cells run in several groups (each alone, some together, one
larger than the limit, empty cells at the cuts), bit for bit against the
oracle and the ungrouped call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[700, 0, 1500, 40, 0, 0, 300, 900], [0, 60, 1200, 0], [33, 35, 34]])
def test_groups_match_oracle(sizes):
    import garfield_amd as gf
    from oracle import oracle
    I, R, P = 32, 16, len(sizes)
    rng = np.random.default_rng(sum(sizes))
    gp = rng.permutation(np.repeat(np.arange(P), sizes)).astype(np.uint32)
    v = rng.integers(0, 256, (gp.size, 64)).astype(np.uint8)
    knn, _, _ = gf.build_graphs(v, gp, P, I, 1)
    want = oracle.optimize_graphs(knn, np.array(sizes), R)
    for max_pairs in (None, 0, 34 * R, 1000 * R, 1500 * R - 1, 1500 * R, 2200 * R):
        print(f"[case] graph groups sizes={sizes} max_pairs={max_pairs}", flush=True)
        out, _ = gf.optimize_graphs(knn, sizes, R, max_pairs=max_pairs)
        assert np.array_equal(out, want)
