"""The streaming forms of quantize and dequantize at the edges of what they take: widths round one
lane's run and the widest row, row counts round the rows of a wave and of its turn, inputs off the
16-byte grid (which the general form takes). Bytes and values exact, as the other tests of the two."""
import numpy as np
import pytest

import oracle

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FORMATS = [(2, False, 0), (4, False, 0), (8, False, 0), (8, True, 0), (4, False, 1), (8, False, 1), (2, False, 1)]
OUT = [(0, torch.float32, torch.int32, np.int32), (1, torch.float16, torch.int16, np.int16), (5, torch.bfloat16, torch.int16, np.int16)]


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    import fbgemm_amd.ops as o
    return o


@pytest.mark.parametrize("bits,sb_float,layout", FORMATS)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_quantize(ops, dtype, bits, sb_float, layout):
    for n, cols in enumerate((8, 16, 24, 40, 72, 120, 264, 504, 512, 520)):
        for rows in (1, 7, 64, 129, 1025):
            rng = np.random.default_rng(10 * cols + rows)
            x = rng.normal(size=(rows, cols)).astype(dtype)
            x[rng.random(x.shape) < 0.2] *= 0  # zeros of both signs
            x[rows // 2] = np.abs(x[rows // 2])
            x[rows // 3] = -np.abs(x[rows // 3])
            want = oracle.quantize_rowwise(x, bits, sb_float, layout)
            d = torch.from_numpy(x).cuda()
            assert (ops.quantize_rowwise(d, bits, sb_float, layout).cpu().numpy() == want).all(), (cols, rows)
            if n % 3 == 0:  # one element off the 16-byte grid
                off = torch.empty(rows * cols + 1, dtype=d.dtype, device="cuda")[1:].view(rows, cols)
                off.copy_(d)
                assert (ops.quantize_rowwise(off, bits, sb_float, layout).cpu().numpy() == want).all(), (cols, rows)


@pytest.mark.parametrize("bits,sb_float,layout", FORMATS)
@pytest.mark.parametrize("out_ty,dtype,bits_dtype,np_bits", OUT)
def test_dequantize(ops, out_ty, dtype, bits_dtype, np_bits, bits, sb_float, layout):
    for n, cols in enumerate((4, 8, 16, 24, 40, 48, 100, 128, 264, 2056, 65536, 65544)):
        for rows in (1, 3, 255, 1030) if cols < 2000 else (1, 3):
            rng = np.random.default_rng(10 * cols + rows)
            pad = (n % 3) * 4 + (1 if n == 3 else 0)  # n == 3: rows off the dword grid
            stride = oracle.quantized_row_bytes(cols, bits, sb_float, layout) + pad
            q = rng.integers(0, 256, size=(rows, stride), dtype=np.uint8)
            at = 0 if layout else (cols * bits + 7) // 8
            pair = np.stack([rng.uniform(1e-3, 1, rows), rng.uniform(-3, 3, rows)], 1).astype(np.float32 if sb_float else np.float16)
            q[:, at:at + pair.view(np.uint8).shape[1]] = pair.view(np.uint8)
            want = oracle.dequantize_rowwise(q, cols, bits, sb_float, layout, out_ty).view(np_bits)
            got = ops.dequantize_rowwise(torch.from_numpy(q).cuda(), cols, bits, sb_float, layout, dtype)
            assert (got.cpu().view(bits_dtype).numpy() == want).all(), (cols, rows)
