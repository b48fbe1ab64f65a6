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
def test_quantize_quads(ops, bits, sb_float, layout):
    """The widths where lanes hold two quads of an fp32 row in streams long enough (below: those), and their neighbours;
    rows off the dword grid; padded rows."""
    for cols in (56, 64, 72, 120, 128, 136, 248, 256):
        for rows in (1, 15, 16, 17, 130):
            rng = np.random.default_rng(100 * cols + rows)
            x = rng.normal(size=(rows, cols)).astype(np.float32)
            x[rng.random(x.shape) < 0.1] *= 0
            x[rows // 2, cols // 2:] = np.abs(x[rows // 2, cols // 2:]) + 9  # extremes in the one and in the other quad
            want = oracle.quantize_rowwise(x, bits, sb_float, layout)
            d = torch.from_numpy(x).cuda()
            assert (ops.quantize_rowwise(d, bits, sb_float, layout).cpu().numpy() == want).all(), (cols, rows)
            for pad in (1, 8):
                out = torch.full((rows, want.shape[1] + pad), 7, dtype=torch.uint8, device="cuda")
                ops.quantize_rowwise(d, bits, sb_float, layout, out=out)
                assert (out[:, :-pad].cpu().numpy() == want).all() and bool((out[:, -pad:] == 7).all()), (cols, rows, pad)


@pytest.mark.parametrize("bits,sb_float,layout", FORMATS)
def test_quantize_quads_of_long_streams(ops, bits, sb_float, layout):
    """The same at the sizes from which rows that use every lane are held as quads (2^20 elements), one row fewer, and a
    last group of one row and of all but one; zeros of both signs as the extremes of either quad."""
    for cols in (64, 128, 256, 512):
        for rows in ((1 << 20) // cols - 1, (1 << 20) // cols, (1 << 20) // cols + 1, (1 << 20) // cols + 16 * 512 // cols - 1):
            rng = np.random.default_rng(cols + rows)
            x = np.abs(rng.normal(size=(rows, cols))).astype(np.float32)
            x[rng.random(x.shape) < 0.05] *= 0
            x[rng.random(x.shape) < 0.02] = -0.0
            want = oracle.quantize_rowwise(x, bits, sb_float, layout)
            for pad in (1, 8):
                out = torch.full((rows, want.shape[1] + pad), 7, dtype=torch.uint8, device="cuda")
                ops.quantize_rowwise(torch.from_numpy(x).cuda(), bits, sb_float, layout, out=out)
                assert (out[:, :-pad].cpu().numpy() == want).all() and bool((out[:, -pad:] == 7).all()), (cols, rows, pad)


@pytest.mark.parametrize("bits,sb_float,layout", FORMATS)
@pytest.mark.parametrize("dtype,cols", [(torch.float16, 200), (torch.float16, 64), (torch.float32, 32)])
def test_quantize_four_groups(ops, dtype, cols, bits, sb_float, layout):
    """Streams of more than 2^26 elements take four row groups at a time: the bytes of their parts, which take two."""
    x = torch.randn((1 << 26) // cols + 19, cols, device="cuda", generator=torch.Generator("cuda").manual_seed(cols)).to(dtype)
    got = ops.quantize_rowwise(x, bits, sb_float, layout)
    assert torch.equal(got, torch.cat([ops.quantize_rowwise(part, bits, sb_float, layout) for part in x.split(x.size(0) // 3 // 8 * 8)]))


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


def special_rows(cols, dtype):
    """Rows whose extremes or elements are not ordinary numbers, and rows of one value."""
    rng = np.random.default_rng(cols)
    rows = rng.normal(size=(24, cols)).astype(dtype)
    inf, nan, big = np.inf, np.nan, np.finfo(dtype).max
    for r, (at, v) in enumerate([(0, nan), (cols // 2, nan), (cols - 1, nan), (0, inf), (cols - 1, inf), (0, -inf), (cols // 2, -inf),
                                 (slice(None), nan), (slice(None), inf), (slice(None), -inf), (slice(None), 0.0), (slice(None), -0.0),
                                 (slice(None), 1.25), (slice(None), -3.0), (0, big), (cols - 1, -big)]):
        rows[r, at] = v
    rows[16, 0], rows[16, -1] = inf, -inf
    rows[17, 0], rows[17, -1] = big, -big
    rows[18, 1], rows[18, -1] = nan, inf
    rows[19] *= dtype(np.finfo(dtype).tiny)          # subnormal ranges
    rows[20] = np.finfo(dtype).smallest_subnormal
    rows[21, :] = 0.0
    rows[21, 3] = nan                                # a zero extreme: the search with positions
    rows[22] = np.abs(rows[22])
    rows[22, ::2] = -0.0
    return rows


@pytest.mark.parametrize("bits,sb_float,layout", FORMATS)
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_quantize_special_values(ops, dtype, bits, sb_float, layout):
    """The bytes of the general form, which takes the same rows one element off the 16-byte grid; those of
    the oracle where a row and its range are finite."""
    for cols in (8, 40, 128, 512):
        x = special_rows(cols, dtype)
        d = torch.from_numpy(x).cuda()
        off = torch.empty(x.size + 1, dtype=d.dtype, device="cuda")[1:].view(x.shape)
        off.copy_(d)
        got = ops.quantize_rowwise(d, bits, sb_float, layout).cpu().numpy()
        assert (got == ops.quantize_rowwise(off, bits, sb_float, layout).cpu().numpy()).all(), cols
        with np.errstate(over="ignore", invalid="ignore"):
            finite = np.isfinite(x).all(1) & np.isfinite(x.astype(np.float32).max(1) - x.astype(np.float32).min(1))
            if not sb_float:  # the pair is stored in fp16
                finite &= np.isfinite(x.astype(np.float16)).all(1) & (x.astype(np.float32).max(1) - x.astype(np.float32).min(1) < 6e4)
        assert finite.sum() >= 6
        assert (got[finite] == oracle.quantize_rowwise(x[finite], bits, sb_float, layout)).all(), cols


@pytest.mark.parametrize("bits,sb_float,layout", FORMATS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_dequantize_special_values(ops, dtype, bits, sb_float, layout):
    """Scales and biases that are infinite, no numbers, zero or subnormal: the bits of the general form, which
    takes the same rows off the dword grid."""
    pair_type = np.float32 if sb_float and not layout else np.float16
    special = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, np.finfo(pair_type).max, np.finfo(pair_type).smallest_subnormal, 0.5], pair_type)
    rows = len(special) ** 2
    for cols in (8, 40, 128):
        rng = np.random.default_rng(cols)
        data = (cols * bits + 7) // 8
        stride = oracle.quantized_row_bytes(cols, bits, sb_float, layout)
        q = rng.integers(0, 256, size=(rows, stride), dtype=np.uint8)
        at = 0 if layout else data
        pair = np.ascontiguousarray(np.stack(np.meshgrid(special, special), -1).reshape(rows, 2))
        q[:, at:at + pair.view(np.uint8).shape[1]] = pair.view(np.uint8)
        off = torch.empty(rows, stride + 1, dtype=torch.uint8, device="cuda")
        off[:, :stride] = torch.from_numpy(q).cuda()
        got = ops.dequantize_rowwise(torch.from_numpy(q).cuda(), cols, bits, sb_float, layout, dtype)
        want = ops.dequantize_rowwise(off, cols, bits, sb_float, layout, dtype)
        as_int = torch.int32 if dtype == torch.float32 else torch.int16
        assert torch.equal(got.view(as_int), want.view(as_int)), cols
