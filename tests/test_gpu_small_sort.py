"""Searches whose sorts run in one launch, at the edges of its sizes (keys a
thread, the last size and the first beyond it) and with sources and targets of
different ones: rows equal the oracle's, in both geometries, from the
operator (which takes every output of the sort) and from the search alone."""
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


@pytest.mark.parametrize("geometry", ["float", "double"])
@pytest.mark.parametrize("n_src,n_tgt", [
    (1, 1), (64, 63), (2047, 2049), (2048, 65), (4096, 4097), (8193, 8192), (8192, 8192), (8192, 8193),
    (12289, 900), (700, 12289)])
def test_small_sorts(dtk, oracle_lib, geometry, n_src, n_tgt):
    rng = np.random.default_rng(n_src + n_tgt)
    src, tgt = rng.random((n_src, 3)), rng.random((n_tgt, 3))
    src[n_src // 2:] = np.round(src[n_src // 2:], 2)  # equal codes among them
    k = min(7, n_src)
    print(f"small sorts {n_src} -> {n_tgt} {geometry}", flush=True)
    gi, _ = oracle_lib.knn(src, tgt, k, geometry=0 if geometry == "float" else 1)
    d_src, d_tgt = torch.as_tensor(src).cuda(), torch.as_tensor(tgt).cuda()
    idx = dtk.knn(d_src, d_tgt, k, geometry=geometry)
    assert np.array_equal(idx.cpu().numpy(), gi)
    op = dtk.MovingLeastSquaresOperator(d_src, d_tgt, basis="constant", k=k,
                                        geometry=geometry)
    _, idx, c = op.graph()
    assert np.array_equal(idx.cpu().numpy(), gi)
    x = rng.random(n_src)
    y = torch.zeros(n_tgt, dtype=torch.float64, device="cuda")
    op.apply(torch.as_tensor(x).cuda(), y)
    ref = (c.cpu().numpy() * x[gi]).sum(axis=1)
    # a sum of k positive terms of total weight 1, in another order
    assert np.abs(y.cpu().numpy() - ref).max() <= k * np.finfo(float).eps
