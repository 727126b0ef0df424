"""Long prefill calls with fp32 activations (more than 4,096 compact rows: one wave transforms a
whole row, several 128-blocks in flight): bitwise the fp16 path on the rounded activations."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,E,H,I,topk", [(779, 24, 2048, 128, 7), (1121, 16, 1792, 128, 6), (700, 16, 640, 128, 6)])
def test_fp32_prefill_equals_fp16(M, E, H, I, topk):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import CX_MOE_PREFILL, synth
    plan = synth.device_moe_layer(3, E, H, I, topk)
    rng = np.random.default_rng(M)
    x = torch.from_numpy(rng.standard_normal((M, H)).astype(np.float32)).cuda()
    lg = torch.from_numpy(rng.standard_normal((M, E + 1)).astype(np.float32)).cuda()
    want = plan(x.half(), lg, mode=CX_MOE_PREFILL)
    for _ in range(3):
        got = plan(x, lg, mode=CX_MOE_PREFILL)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
