"""The search by groups of targets at the sizes where it changes: below and
above the 64 sources it starts at, the source counts that it takes whole and
the first ones it gathers, partial blocks, groups and waves, the neighbour
counts at which the row slots change; and the clouds that drive its radius:
copies of a point beyond a row's slots, lattices (every distance tied), tight
clusters beside a thin background, targets outside the sources' box. Indices
and distances equal the oracle's brute-force order bit for bit, in both
geometries."""
import numpy as np
import pytest

from conftest import grid_points

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dtk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import datatransferkit_amd as d

    return d


def check(dtk, oracle_lib, src, tgt, k, geometry):
    print(f"groups: {len(src)} -> {len(tgt)}, k={k}, {geometry}", flush=True)
    idx, dist = dtk.knn(torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda(), k,
                        geometry=geometry, with_distances=True)
    gi, gd = oracle_lib.knn(src, tgt, k, geometry=0 if geometry == "float" else 1)
    assert np.array_equal(idx.cpu().numpy(), gi)
    assert np.array_equal(dist.cpu().numpy().view(np.uint64),
                          np.ascontiguousarray(gd).view(np.uint64))


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("n_src", [63, 64, 65, 192, 193, 256, 257, 511, 513, 4097, 33001])
def test_source_counts(dtk, oracle_lib, geometry, n_src):
    rng = np.random.default_rng(n_src)
    src, tgt = rng.random((n_src, 3)), 1.4 * rng.random((1027, 3)) - 0.2
    for k in (1, 8, 20, 42, 43):
        check(dtk, oracle_lib, src, tgt, k, geometry)


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("n_tgt", [1, 15, 17, 63, 65, 8193, 70001])
def test_target_counts(dtk, oracle_lib, geometry, n_tgt):
    rng = np.random.default_rng(n_tgt)
    src, tgt = rng.random((3001, 3)), rng.random((n_tgt, 3))
    for k in (9, 21, 64):
        check(dtk, oracle_lib, src, tgt, k, geometry)


@pytest.mark.parametrize("geometry", ["float", "double"])
def test_hard_clouds(dtk, oracle_lib, geometry):
    rng = np.random.default_rng(5)
    lattice = grid_points((20, 20, 20), (0, 0, 0)) / 19.0
    flat = rng.random((6000, 3)) * np.array([1.0, 1.0, 0.0])
    line = rng.random((6000, 3)) * np.array([1.0, 0.0, 0.0])
    copies = np.repeat(rng.random((60, 3)), 150, axis=0)
    cluster = np.concatenate([0.5 + 1e-4 * rng.standard_normal((8000, 3)),
                              rng.random((300, 3))])
    for src in (lattice, flat, line, copies, cluster):
        near = src[rng.integers(0, len(src), 700)]
        tgt = np.concatenate([near, near + 1e-5 * rng.standard_normal(near.shape),
                              rng.random((400, 3)), 30 * rng.random((50, 3))])
        for k in (4, 10, 32, 64):
            check(dtk, oracle_lib, src, tgt, k, geometry)
