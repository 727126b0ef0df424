"""The tall prefill GEMM (forced by its switch) at the edges of its tiles: entries of 1 to 192 rows (one
body for each number of 16-row blocks), experts of more than one entry, K of 4 steps and more, the rates
whose weight copies differ in form, every codebook, gate and up with the mid in one workgroup and plane by
plane.  Bitwise the register-blocked form on the same calls, which sums in the same order."""
import numpy as np
import pytest

import oracle as O
from test_gpu_moe import oracle_layer, rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# Rows of each expert; the shared one's entries: 12 x 192 + 151.
COUNTS = (0, 1, 15, 16, 17, 32, 33, 48, 64, 65, 80, 81, 97, 112, 113, 128, 129, 145, 160, 161, 177, 191, 192, 193, 205)


@pytest.mark.parametrize("H,Ie,bgu,bd,cb", [(128, 128, 4, 4, "mul1"), (384, 256, 3, 5, "mul1"), (256, 128, 1.5, 2.5, "mul1"),
                                            (640, 128, 8, 6, "mul1"), (256, 384, 1, 7, "mul1"), (256, 128, 2, 8, "mcg"),
                                            (128, 256, 5, 4, "3inst"), (256, 256, 3.5, 3, "mul1")])
@pytest.mark.parametrize("seq", ["1", "0"])
def test_tall_entries(monkeypatch, H, Ie, bgu, bd, cb, seq):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import synth
    E, M = len(COUNTS), sum(COUNTS)
    monkeypatch.setenv("CX_TALL_SEQMID", seq)
    plans = []
    for form in ("1", "0"):
        monkeypatch.setenv("CX_PREFILL_GEMM", form)
        plans.append(synth.device_moe_layer(7, E=E, H=H, Ie=Ie, topk=1, bits_gu=bgu, bits_d=bd, codebook=cb))
    rng = np.random.default_rng(6)
    x = rng.standard_normal((M, H)).astype(np.float16)
    lg = rng.standard_normal((M, E + 1)).astype(np.float32)
    lg[np.arange(M), rng.permutation(np.repeat(np.arange(E), COUNTS))] = 9.0
    xd, ld = torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda()
    tall, short = [p(xd, ld, mode=2) for p in plans]
    assert torch.equal(tall.view(torch.int32), short.view(torch.int32))
    if seq == "1":
        rs, rw = O.route(lg, E, 1)
        np.testing.assert_array_equal(np.bincount(rs.ravel(), minlength=E), COUNTS)
        ref = oracle_layer(plans[0], x, rs, rw)
        y = tall.cpu().numpy()
        assert rel_l2(y, ref) <= 1e-3  # the layer tests' bounds
        assert np.abs(y - ref).max() <= 2e-3 * np.abs(ref).max()


@pytest.mark.parametrize("cb,idle", [("mcg", True), ("3inst", True), ("mul1", False)])
def test_tall_not_on_an_idle_chip(monkeypatch, cb, idle):
    # 8 experts of more than 96 rows, I = 256: 22 gate/up workgroups of the tall form.  In the mcg and 3inst
    # codebooks the register-blocked form runs, in a workspace no larger than the tall form's.
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import CX_MOE_PREFILL, synth
    monkeypatch.delenv("CX_PREFILL_GEMM", raising=False)
    make = lambda: synth.device_moe_layer(9, E=8, H=256, Ie=256, topk=2, codebook=cb)
    plan = make()
    monkeypatch.setenv("CX_PREFILL_GEMM", "1")
    tall = make()
    M = 500
    assert (plan.workspace_size(M, CX_MOE_PREFILL) < tall.workspace_size(M, CX_MOE_PREFILL)) == idle
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(M, 256, device="cuda", generator=g).half()
    lg = torch.randn(M, 9, device="cuda", generator=g)
    a, b = plan(x, lg, mode=CX_MOE_PREFILL), tall(x, lg, mode=CX_MOE_PREFILL)
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))
