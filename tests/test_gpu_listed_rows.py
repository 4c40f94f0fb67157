"""Truncated rows that the Cholesky setup lists are solved by rotating the
moments first and forming the eigenvectors from the kept tangents afterwards.
They equal the general eigen-solver's bit for bit, with its truncated set,
sweeps and convergence, over list lengths at the edges of a tile and beyond
one tile a block, with the sweeps capped below convergence and uncapped, in
both truncations and precisions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def dtk():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import datatransferkit_amd as d

    return d


def _plane(rng, n):
    p = rng.random((n, 3))
    p[:, 2] = 0.25  # moments in z are exactly zero: every row is truncated
    return p


@pytest.mark.parametrize("basis,m,k", [("linear", 4, 8), ("quadratic", 10, 21)])
@pytest.mark.parametrize("n", [1, 63, 65, 2000, 132_000])
def test_truncated_rows_equal_the_eigen_solver(dtk, basis, m, k, n):
    rng = np.random.default_rng(n + m)
    src, tgt = _plane(rng, 3000), _plane(rng, n)
    d_src, d_tgt = torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda()
    for precision in ("fp64", "fp32_bulk"):
        for truncation, sweeps in (("absolute", 0), ("absolute", 2), ("relative", 0)):
            print(f"listed rows {basis} n={n} {precision} {truncation} {sweeps}", flush=True)
            kw = dict(basis=basis, k=k, rbf="wendland0", precision=precision,
                      truncation=truncation, rcond=1e-13, max_rotations=sweeps)
            a = dtk.MovingLeastSquaresOperator(d_src, d_tgt, solver="cholesky", **kw)
            b = dtk.MovingLeastSquaresOperator(d_src, d_tgt, solver="cyclic", **kw)
            sa, sb = a.stats(), b.stats()
            assert sa["n_eigen_fallback"] == n
            for key in ("n_underdetermined", "n_unconverged", "total_rotations"):
                assert sa[key] == sb[key], key
            assert sa["n_underdetermined"] == n
            ca, cb = a.graph()[2], b.graph()[2]
            assert torch.equal(ca.view(torch.int32), cb.view(torch.int32))


@pytest.mark.parametrize("precision", ["fp64", "fp32_bulk"])
@pytest.mark.parametrize("n", [700, 60_000, 1_000_000])
@pytest.mark.parametrize("spacing", [1e-2, 7e-3])
def test_few_truncated_rows_among_others(dtk, precision, n, spacing):
    """10 neighbours for 10 unknowns: about half of the rows are listed and a
    part of those truncated (a few a wave at the larger spacing, more at the
    smaller), so waves leave them to the second pass. The truncated rows have
    the eigen-solver's bits, and every row the same bits among half of the
    targets as among all."""
    rng = np.random.default_rng(n)
    side = spacing * n ** (1 / 3)
    src, tgt = (torch.as_tensor(side * rng.random((n, 3))).cuda() for _ in range(2))
    kw = dict(basis="quadratic", k=10, rbf="wendland2", precision=precision)

    def build(t, solver):
        op = dtk.MovingLeastSquaresOperator(src, t, solver=solver, **kw)
        return op.stats(), op.graph()[2].view(torch.int32).reshape(t.shape[0], -1)

    sa, ca = build(tgt, "cholesky")
    sb, cb = build(tgt, "cyclic")
    _, half = build(tgt[: n // 2].contiguous(), "cholesky")
    print(f"few truncated {precision} n={n} {spacing}: {sa['n_eigen_fallback']} listed, "
          f"{sa['n_underdetermined']} truncated", flush=True)
    assert sa["n_eigen_fallback"] > sa["n_underdetermined"] == sb["n_underdetermined"] > 0
    assert sa["n_unconverged"] == sb["n_unconverged"]
    assert int((ca == cb).all(dim=1).sum()) >= sa["n_underdetermined"]
    assert torch.equal(ca[: n // 2], half)
