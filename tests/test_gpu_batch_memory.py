"""Device memory that a batch's rebuild graph holds for the scratch of its
listed rows: one share for all of its groups, of 6 kept sweeps and one more
(2,048 blocks of 64 rows, 45 rotations, 7 regions of 8 bytes: 330 MB, and 9 MB
of spare regions), not one for each basis."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_rebuild_graph_keeps_one_scratch():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import datatransferkit_amd as dtk

    rng = np.random.default_rng(6)
    n, rows = 300, 1000  # 150,000 rows of each basis: the scratch's full size
    ns, nt = [400] * n, [rows] * n
    src = torch.as_tensor(rng.random((sum(ns), 3))).cuda()
    tgt = torch.as_tensor(rng.random((sum(nt), 3))).cuda()
    basis = ["linear", "quadratic"] * (n // 2)

    def kept(solver):
        dtk.release_cached_memory()
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        op = dtk.MovingLeastSquaresBatch.from_concatenated(
            src, tgt, ns, nt, basis, [16] * n, precision="fp32_bulk", solver=solver)
        op.rebuild()
        torch.cuda.synchronize()
        dtk.release_cached_memory()
        held = before - torch.cuda.mem_get_info()[0]
        del op
        return held

    for solver in ("cyclic", "cholesky"):
        kept(solver)  # (what the runtime keeps from the first ones)
    more = kept("cholesky") - kept("cyclic")
    print(f"scratch of the listed rows kept: {more / 2**20:.0f} MiB", flush=True)
    # 315 MiB, the lists of the rows and the rounding of the blocks
    assert more <= 340 * 2**20
