"""Linears over many rows (Exl3GemmRowsKernel): bitwise the few-row path on slices of the rows."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# Shapes that take the many-row GEMM: uneven K splits (60, 20 and 52 steps), 1 to 8 K segments
# (sums parked in the workspace), half-bit rates (weights copied every second chunk), entries in
# plain and in XCD order, 1 to 8 row blocks per entry, last entries of every size.
@pytest.mark.parametrize("I,Ot,bits,cb,rows", [
    (2048, 4096, 4, "mul1", (300, 2047)), (1920, 5120, 3, "mul1", (193, 1025)), (640, 12288, 2.5, "mul1", (129, 777)),
    (4096, 2048, 5, "mcg", (1290,)), (1664, 8192, 3.5, "mul1", (255,)), (8192, 1024, 6, "mul1", (2033,)),
    (1024, 16384, 8, "3inst", (65, 400)), (512, 24576, 1.5, "mul1", (96, 129)), (3072, 6144, 7, "mul1", (511,)),
    (2048, 8192, 1, "3inst", (201,)), (2048, 8192, 2, "mul1", (1111,)), (256, 512, 3, "mul1", (81, 192)),
])
def test_rows_linear_equals_few_row_path(I, Ot, bits, cb, rows):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import synth
    g = torch.Generator(device="cuda")
    g.manual_seed(I + Ot)
    lin = synth.device_linear(g, I, Ot, bits, codebook=cb)
    for M in rows:
        x = torch.randn(M, I, device="cuda", generator=g)
        x = x if M % 2 else x.half()
        for yt in (torch.float32, torch.float16):
            want = torch.cat([lin(x[r:r + 48].contiguous(), yt) for r in range(0, M, 48)])
            got = lin(x, yt)
            it = torch.int32 if yt == torch.float32 else torch.int16
            assert torch.equal(got.view(it), want.view(it)), (M, yt)


def test_rows_group_equals_single_calls():
    # A group at many rows: jobs of two rates and very different widths, padded outputs.
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import ops, synth
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    lins = [synth.device_linear(g, 2048, o, 4) for o in (4096, 512, 640)] + [synth.device_linear(g, 1024, 256, 3)]
    M = 1003
    xs = [torch.randn(M, lin.in_features, device="cuda", generator=g) for lin in lins]
    ys = [torch.full((M, lin.out_features + 64), 3.0, device="cuda") for lin in lins]
    ops.linear_group([(lin, x, y) for lin, x, y in zip(lins, xs, ys)])
    for lin, x, y in zip(lins, xs, ys):
        want = torch.cat([lin(x[r:r + 48].contiguous()) for r in range(0, M, 48)])
        assert torch.equal(y[:, :lin.out_features].view(torch.int32), want.view(torch.int32))
        assert torch.all(y[:, lin.out_features:] == 3.0)
