"""Grouping at the edges of its waves' segments (64 routes, 1,024 with one route per thread and two),
of its tiles and of the expert range, exact against a stable sort; also with every route on one
expert (the largest per-wave count)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 1984, 2047, 2048, 2049, 3072, 20001])
@pytest.mark.parametrize("E", [1, 513, 1024])
def test_group_edges(n, E):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import ops
    rng = np.random.default_rng(n)
    for sel in (rng.integers(0, E, size=(n, 1)), np.full((n, 1), E - 1), rng.integers(-1, min(E, 3), size=(n, 1))):
        sel = sel.astype(np.int32)
        counts, offsets, pairs, rows = [t.cpu().numpy() for t in ops.group(torch.from_numpy(sel).cuda(), E)]
        idx = np.nonzero((sel.ravel() >= 0) & (sel.ravel() < E))[0]
        want = idx[np.argsort(sel.ravel()[idx], kind="stable")]
        np.testing.assert_array_equal(counts, np.bincount(sel.ravel()[idx], minlength=E))
        np.testing.assert_array_equal(offsets, np.concatenate([[0], np.cumsum(counts)]))
        np.testing.assert_array_equal(pairs[:len(want)], want)
        np.testing.assert_array_equal(rows[:len(want)], want)
