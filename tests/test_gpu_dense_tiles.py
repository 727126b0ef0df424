"""Router linear over more than 64 rows (DenseTileKernel and, for rows that are not 16-byte aligned
or widths that are no multiple of 64, DenseMfmaKernel) against a binary64 product."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# One chunk of 64 k, odd chunk counts, 48-output tiles with remainders, row tiles of 1 to 64 rows in
# grids that are no multiple of 8, padded and unaligned rows; fewer than 8 row tiles of many outputs
# (spread over the XCDs).
@pytest.mark.parametrize("M,I,Ot,pad", [
    (65, 64, 1, 0), (127, 128, 49, 0), (192, 192, 65, 8), (577, 320, 97, 0), (300, 2048, 513, 0), (1100, 2048, 257, 24),
    (70, 96, 33, 0), (201, 160, 100, 0), (130, 64, 70, 1), (99, 256, 17, 3), (2113, 64, 81, 0),
    (65, 128, 1585, 0), (384, 192, 2049, 8), (17, 64, 1600, 0),
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


def tile_width(M, O, dt):
    """Blocks of 16 outputs per workgroup, as the launcher chooses them for DenseTileKernel."""
    mt, ob, rows = -(-M // 64), -(-O // 16), 8 if dt == "float32" else 4
    return min((3, 4, 5, 6), key=lambda n: (-(-(mt * -(-ob // n)) // 256) * (rows + n), -n))


# Every tile width (their copies split over the waves, waits and LDS differ), each with a part block and
# a part tile of outputs and with whole ones, one chunk of 64 k and several; up to 64 rows where I is a
# multiple of 64 and not of 256.
@pytest.mark.parametrize("M,I,Ot,width", [
    (2048, 64, 512, 4), (1990, 128, 500, 4), (2600, 64, 600, 4), (2048, 128, 513, 5), (2048, 64, 577, 5), (1000, 320, 1041, 5),
    (2600, 192, 513, 6), (1111, 128, 1217, 6), (9, 896, 513, 3), (33, 1920, 70, 3), (64, 896, 49, 3), (1, 1920, 33, 3),
])
@pytest.mark.parametrize("dt", ["float32", "float16"])
def test_dense_tile_widths(M, I, Ot, width, dt):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import ops
    assert tile_width(M, Ot, dt) == width
    g = torch.Generator(device="cuda")
    g.manual_seed(M + I + Ot)
    W = torch.randn(Ot, I, device="cuda", generator=g).half()
    x = torch.randn(M, I, device="cuda", generator=g).to(getattr(torch, dt))
    yb = torch.full((M + 1, Ot + 5), 7.0, device="cuda")
    ops.dense_linear(W, x, y=yb[:M, :Ot])
    xs = (x if dt == "float32" and M <= 8 else x.half()).double()  # up to 8 fp32 rows: fp32 products
    ref, bound = xs @ W.double().t(), xs.abs() @ W.double().abs().t()
    # fp32 sums: at most I roundings of the products and I of the sums, 2^-24 each.
    assert torch.all((yb[:M, :Ot].double() - ref).abs() <= 2 * I * 2.0**-24 * bound + 1e-30)
    assert torch.all(yb[:, Ot:] == 7.0) and torch.all(yb[M] == 7.0)


# x as columns [off, off + I) of a wider matrix, up to its last column: the storage ends where x does,
# and NaN stands in every other column.  DenseTileKernel, DenseSplitKernel (up to 64 rows, I a multiple of
# 256), DenseMfmaKernel (the others), DenseGemvKernel (fp32, up to 8 rows).
@pytest.mark.parametrize("M,I,Ot,off", [
    (8192, 2048, 70, 128), (65, 64, 33, 8), (130, 192, 513, 64), (64, 2048, 33, 64), (17, 256, 49, 8), (9, 512, 17, 4),
    (70, 96, 33, 32), (300, 160, 65, 8), (33, 64, 20, 1), (5, 256, 40, 4),
])
@pytest.mark.parametrize("dt", ["float32", "float16"])
def test_dense_offset_view(M, I, Ot, off, dt):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import ops
    g = torch.Generator(device="cuda")
    g.manual_seed(M + I + off)
    W = torch.randn(Ot, I, device="cuda", generator=g).half()
    xb = torch.full((M, off + I), float("nan"), device="cuda", dtype=getattr(torch, dt))
    xb[:, off:] = torch.randn(M, I, device="cuda", generator=g).to(xb.dtype)
    x = xb[:, off:]
    y = ops.dense_linear(W, x)
    xs = (x if dt == "float32" and M <= 8 else x.half()).double()  # up to 8 fp32 rows: fp32 products
    ref, bound = xs @ W.double().t(), xs.abs() @ W.double().abs().t()
    # fp32 sums: at most I roundings of the products and I of the sums, 2^-24 each.
    assert torch.all((y.double() - ref).abs() <= 2 * I * 2.0**-24 * bound + 1e-30)
