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
