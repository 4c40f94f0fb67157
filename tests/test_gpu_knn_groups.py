"""The search by groups of targets at the sizes where it changes: below and
above the 64 sources it starts at, the source counts that it takes whole and
the first ones it gathers, partial blocks, the neighbour counts at which the
row slots change; and the clouds that drive its radius: copies of a point
beyond a row's slots, lattices (every distance tied), tight clusters beside a
thin background, targets outside the sources' box. A wave takes fewer targets
where a launch has few (one below 8,192), so these clouds run again at target
counts that fill waves and groups, with a partial last wave, alone and in a
batch. Indices and distances equal the oracle's brute-force order bit for bit,
in both geometries."""
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


def hard_sources(rng):
    lattice = grid_points((20, 20, 20), (0, 0, 0)) / 19.0
    flat = rng.random((6000, 3)) * np.array([1.0, 1.0, 0.0])
    line = rng.random((6000, 3)) * np.array([1.0, 0.0, 0.0])
    copies = np.repeat(rng.random((60, 3)), 150, axis=0)
    cluster = np.concatenate([0.5 + 1e-4 * rng.standard_normal((8000, 3)),
                              rng.random((300, 3))])
    return {"lattice": lattice, "flat": flat, "line": line, "copies": copies,
            "cluster": cluster}


def hard_targets(rng, src, n):
    """About n targets: sources, points beside sources, in the box, beyond it."""
    near = src[rng.integers(0, len(src), 3 * n // 8)]
    return np.concatenate([near, near + 1e-5 * rng.standard_normal(near.shape),
                           rng.random((n // 5, 3)), 30 * rng.random((n // 40 + 1, 3))])


@pytest.mark.parametrize("geometry", ["float", "double"])
def test_hard_clouds(dtk, oracle_lib, geometry):
    rng = np.random.default_rng(5)
    for src in hard_sources(rng).values():
        tgt = hard_targets(rng, src, 1850)
        for k in (4, 10, 32, 64):
            check(dtk, oracle_lib, src, tgt, k, geometry)


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("cloud", ["lattice", "flat", "line", "copies", "cluster"])
def test_hard_clouds_in_full_groups(dtk, oracle_lib, cloud, geometry):
    """64 targets a wave from 524,288 targets on for k <= 16, 32 from 262,144
    for larger k: waves and groups of every kind of target, finished together,
    in part or one by one."""
    rng = np.random.default_rng(9)
    src = hard_sources(rng)[cloud]
    for n, ks in ((550_000, (1, 4, 10)), (280_000, (20, 32, 64))):
        tgt = hard_targets(rng, src, n)
        assert len(tgt) > (524_288 if ks[0] == 1 else 262_144) and len(tgt) % 64
        sample = rng.permutation(len(tgt))[:3000]
        d_src, d_tgt = torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda()
        for k in ks:
            print(f"full groups: {cloud} {len(src)} -> {len(tgt)}, k={k}, {geometry}", flush=True)
            idx, dist = dtk.knn(d_src, d_tgt, k, geometry=geometry, with_distances=True)
            gi, gd = oracle_lib.knn(src, tgt[sample], k,
                                    geometry=0 if geometry == "float" else 1)
            assert np.array_equal(idx.cpu().numpy()[sample], gi)
            assert np.array_equal(dist.cpu().numpy()[sample].view(np.uint64),
                                  np.ascontiguousarray(gd).view(np.uint64))


@pytest.mark.parametrize("k", [10, 33])
@pytest.mark.parametrize("geometry", ["float", "double"])
def test_hard_clouds_in_a_batch(dtk, k, geometry):
    """Problems of hard clouds, small clouds and clouds of other scales in the
    waves of one batch: each equals its own operator."""
    rng = np.random.default_rng(12)
    clouds = list(hard_sources(rng).values())
    clouds += [rng.random((n, 3)) * s for n, s in ((70, 1.0), (200, 1e-7), (300, 1e6), (k, 1.0))]
    probs = []
    for i in range(27):
        src = clouds[i % len(clouds)]
        n = int(rng.integers(9000, 15000)) if i else 170_000
        probs.append((torch.as_tensor(src).cuda(),
                      torch.as_tensor(hard_targets(rng, src, n) * np.abs(src).max()).cuda()))
    print(f"hard batch k={k} {geometry} {sum(len(t) for _, t in probs)}", flush=True)
    batch = dtk.MovingLeastSquaresBatch([(s, t, "constant", k) for s, t in probs],
                                        geometry=geometry)
    xs = [torch.as_tensor(rng.random(len(s))).cuda() for s, _ in probs]
    ys = [torch.zeros(len(t), dtype=torch.float64, device="cuda") for _, t in probs]
    batch.rebuild()
    batch.apply(xs, ys)
    for (s, t), x, y in zip(probs, xs, ys):
        op = dtk.MovingLeastSquaresOperator(s, t, basis="constant", k=k, geometry=geometry)
        assert torch.equal(op.apply(x, torch.empty_like(y)), y)


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("scale", [1e-9, 1e-7, 1.0, 1e6])
def test_small_clouds_of_any_scale(dtk, oracle_lib, scale, geometry):
    """Clouds that a wave takes whole, in other units: no row is left to the
    tree search (its first threshold was a distance of 1)."""
    rng = np.random.default_rng(4)
    for n_src in (64, 192, 200, 256):
        src, tgt = scale * rng.random((n_src, 3)), scale * rng.random((3000, 3))
        d_src, d_tgt = torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda()
        for k in (1, 3, 16, 40):
            print(f"scale {scale} {n_src} k={k} {geometry}", flush=True)
            op = dtk.MovingLeastSquaresOperator(d_src, d_tgt, basis="constant", k=k,
                                                geometry=geometry)
            assert op.stats()["n_stack_overflow"] == 0
            gi, _ = oracle_lib.knn(src, tgt, k, geometry=0 if geometry == "float" else 1)
            assert np.array_equal(op.graph()[1].cpu().numpy(), gi)


TIED = {
    # counts around a cell's centre: 8, 32, 56, ...; around a node: 1, 7, 19, 27
    "cells": (lambda n: (grid_points((n, n, n), (0, 0, 0)),
                         grid_points((n - 1, n - 1, n - 1), (0.5, 0.5, 0.5))), (8, 10, 16, 20)),
    "nodes": (lambda n: (grid_points((n, n, n), (0, 0, 0)),) * 2, (8, 10, 16, 20)),
    # a spacing that rounds: the same shells a few units of rounding thick
    "rounded": (lambda n: (grid_points((n, n, n), (0, 0, 0)) / (n + 0.7),
                           grid_points((n - 1, n - 1, n - 1), (0.5, 0.5, 0.5)) / (n + 0.7)),
                (10, 16, 20)),
    # every node eight times, as the corners of hexahedra give them
    "copies": (lambda n: (np.repeat(grid_points((n // 2,) * 3, (0, 0, 0)), 8, axis=0),
                          grid_points((n // 2 - 1,) * 3, (0.5, 0.5, 0.5))), (1, 10, 32, 64)),
}


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("n", [12, 64])
@pytest.mark.parametrize("cloud", list(TIED))
def test_tied_distances_stay_in_the_groups(dtk, oracle_lib, cloud, n, geometry):
    """Where the number of sources within a distance jumps over the row's
    slots no threshold fits them; the rows are finished all the same, none is
    left to the tree search."""
    make, ks = TIED[cloud]
    src, tgt = make(n)
    rng = np.random.default_rng(n)
    src = np.ascontiguousarray(src[rng.permutation(len(src))])
    sample = rng.permutation(len(tgt))[:4000]
    d_src, d_tgt = torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda()
    for k in ks:
        print(f"ties: {cloud} {len(src)} -> {len(tgt)}, k={k}, {geometry}", flush=True)
        op = dtk.MovingLeastSquaresOperator(d_src, d_tgt, basis="constant", k=k,
                                            geometry=geometry)
        assert op.stats()["n_stack_overflow"] == 0
        gi, gd = oracle_lib.knn(src, tgt[sample], k, geometry=0 if geometry == "float" else 1)
        idx, dist = dtk.knn(d_src, d_tgt, k, geometry=geometry, with_distances=True)
        assert np.array_equal(idx.cpu().numpy()[sample], gi)
        assert np.array_equal(dist.cpu().numpy()[sample].view(np.uint64),
                              np.ascontiguousarray(gd).view(np.uint64))
        assert np.array_equal(op.graph()[1].cpu().numpy(), idx.cpu().numpy())


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("box", [(1, 1e-2, 1e-4), (1e-4, 1, 1e-2), (3e-9, 3e-5, 3e-7)])
def test_thin_boxes_stay_in_the_groups(dtk, oracle_lib, box, geometry):
    """Clouds much thinner in some directions: the curve's cells are cubes
    (the grid is as wide as the longest side), so that groups of its points
    stay round and are finished without the tree search."""
    rng = np.random.default_rng(8)
    src, tgt = rng.random((60_000, 3)) * np.array(box), rng.random((30_000, 3)) * np.array(box)
    d_src, d_tgt = torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda()
    sample = rng.permutation(len(tgt))[:2000]
    for k in (1, 10, 64):
        print(f"thin box {box} k={k} {geometry}", flush=True)
        op = dtk.MovingLeastSquaresOperator(d_src, d_tgt, basis="constant", k=k,
                                            geometry=geometry)
        assert op.stats()["n_stack_overflow"] == 0
        gi, _ = oracle_lib.knn(src, tgt[sample], k, geometry=0 if geometry == "float" else 1)
        assert np.array_equal(op.graph()[1].cpu().numpy()[sample], gi)


def outside(rng, n, where):
    """Targets of the unit box: inside it, beside it, in a box around it."""
    t = rng.random((n, 3))
    if where == "beside":
        t[:, 0] += 2.0
    return 3.0 * t - 1.0 if where == "around" else t


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("where", ["beside", "around"])
def test_targets_outside_cost_no_more_than_their_tree_search(dtk, oracle_lib, where, geometry):
    """No radius that holds k sources holds few more for a target far outside
    the sources' box; gathered one at a time such targets took 10 to 20 times
    the query of targets inside. They go to the tree search at once: at most 6
    times (1.8 to 3 measured), with the oracle's rows."""
    rng = np.random.default_rng(11)
    src, n = rng.random((300_000, 3)), 300_000
    sample = rng.permutation(n)[:2000]
    d_src = torch.as_tensor(src).cuda()

    def query(tgt, k):
        ops = [dtk.MovingLeastSquaresOperator(d_src, torch.as_tensor(tgt).cuda(),
                                              basis="constant", k=k, geometry=geometry)
               for _ in range(4)]
        return ops[0], min(op.stats()["ms_knn_query"] for op in ops)

    for k in (1, 10, 24):
        print(f"outside: {where} k={k} {geometry}", flush=True)
        tgt = outside(rng, n, where)
        _, inside = query(outside(rng, n, "inside"), k)
        op, ms = query(tgt, k)
        print(f"  {inside:.3f} ms inside, {ms:.3f} {where}", flush=True)
        gi, _ = oracle_lib.knn(src, tgt[sample], k, geometry=0 if geometry == "float" else 1)
        assert np.array_equal(op.graph()[1].cpu().numpy()[sample], gi)
        assert ms <= 6 * inside


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("n_tgt", [1, 65, 300, 513, 9000, 140_001])
@pytest.mark.parametrize("k", [1, 4, 9, 10, 17, 32, 33, 64])
def test_rows_left_to_the_tree_search(dtk, oracle_lib, k, n_tgt, geometry):
    """Clouds whose rows the groups leave (more sources at one distance than
    a wave holds), at list lengths from one row to more than the lanes of the
    launch over the list, for every form of the tree search."""
    rng = np.random.default_rng(k)
    near = rng.standard_normal((900, 3))
    src = np.concatenate([np.repeat([[0.5, 0.5, 0.5]], 700, axis=0),
                          4.0 * near / np.linalg.norm(near, axis=1)[:, None]])
    unique = 0.5 + 1e-3 * rng.standard_normal((min(n_tgt, 500), 3))
    tgt = unique[np.arange(n_tgt) % len(unique)]
    print(f"left rows: k={k} n={n_tgt} {geometry}", flush=True)
    op = dtk.MovingLeastSquaresOperator(torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda(),
                                        basis="constant", k=k, geometry=geometry)
    assert op.stats()["n_stack_overflow"] == n_tgt
    idx, dist = dtk.knn(torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda(), k,
                        geometry=geometry, with_distances=True)
    gi, gd = oracle_lib.knn(src, unique, k, geometry=0 if geometry == "float" else 1)
    at = np.arange(n_tgt) % len(unique)
    assert np.array_equal(idx.cpu().numpy(), gi[at])
    assert np.array_equal(dist.cpu().numpy().view(np.uint64),
                          np.ascontiguousarray(gd)[at].view(np.uint64))
    assert np.array_equal(op.graph()[1].cpu().numpy(), gi[at])


def test_nearest_with_many_targets_needs_no_rows(dtk):
    """The nearest source alone is found without rows, a gather for a whole
    wave: well below the query of a few neighbours (0.6 to 0.7 of it measured,
    the same time when it took rows)."""
    rng = np.random.default_rng(2)
    src = torch.as_tensor(rng.random((3000, 3))).cuda()
    tgt = torch.as_tensor(rng.random((400_000, 3))).cuda()

    def query(k):
        return min(dtk.MovingLeastSquaresOperator(src, tgt, basis="constant", k=k)
                   .stats()["ms_knn_query"] for _ in range(12))

    one, four = query(1), query(4)
    print(f"nearest {one:.3f} ms, four nearest {four:.3f} ms", flush=True)
    assert one <= 0.85 * four
