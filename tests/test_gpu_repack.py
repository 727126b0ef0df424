"""Loader repack: checkpoint tile order to column-pair order, exact, with 16-byte aligned and unaligned
pointers, the smallest and odd tile sizes, and more rows of tiles than one pass of the grid."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("I,O,k2", [(128, 128, 2), (384, 640, 3), (256, 1152, 7), (2048, 4096, 8), (1152, 128, 16),
                                    (16 * 4 * 65535 + 64 * 5, 128, 2)])
@pytest.mark.parametrize("shift", [0, 2, 4])  # int16 elements past a 16-byte boundary; 4-byte alignment is required
def test_repack(I, O, k2, shift):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from exl3moe import check, lib, ptr, stream_ptr
    I = -(-I // 128) * 128
    A, B, n = I // 16, O // 16, 8 * k2
    size = A * B * n
    g = torch.Generator(device="cuda").manual_seed(3)
    src = torch.randint(-32768, 32768, (size + 8,), dtype=torch.int16, device="cuda", generator=g)[shift:shift + size]
    out = torch.zeros(size + 8, dtype=torch.int16, device="cuda")
    dst = out[shift:shift + size]
    check("cx_exl3_repack", lib().cx_exl3_repack(ptr(src), I, O, k2, ptr(dst), stream_ptr(None)))
    want = src.view(A, B // 2, 2 * n).transpose(0, 1).reshape(-1)
    assert torch.equal(dst, want)
    assert not out[:shift].any() and not out[shift + size:].any()
