"""Short prefill entries (gate/up with the mid in one launch) at the edges of its tiles: entries of
1 to 64 rows, one chunk pair of k and several, the rates whose weight steps differ in form."""
import numpy as np
import pytest

import oracle as O
from test_gpu_moe import oracle_layer, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

COUNTS = (1, 2, 15, 16, 17, 32, 33, 47, 48, 49, 63, 64)  # rows of each expert; the shared one's: 6 x 64 + 3


@pytest.mark.parametrize("H,Ie,bgu,cb", [(128, 128, 4, "mul1"), (384, 256, 3, "mul1"), (256, 128, 8, "mul1"),
                                         (256, 384, 1.5, "mul1"), (640, 128, 5, "mcg"), (128, 256, 6, "3inst")])
def test_entry_rows(H, Ie, bgu, cb):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import synth
    E, k, M = len(COUNTS), 1, sum(COUNTS)
    plan = synth.device_moe_layer(77, E=E, H=H, Ie=Ie, topk=k, bits_gu=bgu, bits_d=4, codebook=cb)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((M, H)).astype(np.float16)
    lg = rng.standard_normal((M, E + 1)).astype(np.float32)
    lg[np.arange(M), rng.permutation(np.repeat(np.arange(E), COUNTS))] = 9.0
    y = plan(torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda(), mode=2).cpu().numpy()
    rs, rw = O.route(lg, E, k)
    np.testing.assert_array_equal(np.bincount(rs.ravel(), minlength=E), COUNTS)
    ref = oracle_layer(plan, x, rs, rw)
    assert rel_l2(y, ref) <= 1e-3  # the layer tests' bounds
    assert np.abs(y - ref).max() <= 2e-3 * np.abs(ref).max()
