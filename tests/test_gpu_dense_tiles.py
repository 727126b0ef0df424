"""Router linear over more than 64 rows (DenseTileKernel and, for rows that are not 16-byte aligned
or widths that are no multiple of 64, DenseMfmaKernel) against a binary64 product."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# One chunk of 64 k, odd chunk counts, 48- to 96-output tiles with 1-output remainders, row tiles of
# 1 to 64 rows in grids that are no multiple of 8, padded and unaligned rows.
@pytest.mark.parametrize("M,I,Ot,pad", [
    (65, 64, 1, 0), (127, 128, 49, 0), (192, 192, 65, 8), (577, 320, 97, 0), (300, 2048, 513, 0), (1100, 2048, 257, 24),
    (70, 96, 33, 0), (201, 160, 100, 0), (130, 64, 70, 1), (99, 256, 17, 3), (2113, 64, 81, 0),
])
@pytest.mark.parametrize("dt", ["float32", "float16"])
def test_dense_tiles(M, I, Ot, pad, dt):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(M + I)
    W = torch.randn(Ot, I, device="cuda", generator=g).half()
    xb = torch.randn(M, I + pad, device="cuda", generator=g).to(getattr(torch, dt))
    x = xb[:, :I]
    yb = torch.full((M, Ot + 5), 7.0, device="cuda")
    ops.dense_linear(W, x, y=yb[:, :Ot])
    xs = x.half().double()  # rounded to fp16, as the kernel does
    ref, bound = xs @ W.double().t(), xs.abs() @ W.double().abs().t()
    # fp32 sums of exact products: at most I roundings of 2^-24 relative to the sum of magnitudes.
    assert torch.all((yb[:, :Ot].double() - ref).abs() <= I * 2.0**-24 * bound + 1e-30)
    assert torch.all(yb[:, Ot:] == 7.0)
