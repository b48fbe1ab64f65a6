"""The burst kernel (a workgroup per bag and 256 columns) at the sizes where it can go wrong: windows
of columns that end inside a 16-byte piece, rows at every alignment, bags around its staging sizes,
both numbers of waves, and the line where its rule hands over to the other kernels. Bit for bit."""
import numpy as np
import pytest

import helpers as H
import test_spmdm_gpu as S
import test_tbe_gpu as TB
from helpers import BF16, FP16, FP32, INT2, INT4, INT8

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    import fbgemm_amd.ops as o
    return o


@pytest.fixture
def burst():
    import fbgemm_amd
    lib = fbgemm_amd.lib()
    yield lib.fbgemm_amd_set_burst
    lib.fbgemm_amd_set_burst(-1)


# around one lane's 4 columns, a 16-byte piece of every type, the window of 256 columns, several windows
DIMS = [1, 3, 4, 5, 7, 8, 10, 16, 20, 31, 33, 63, 65, 100, 128, 255, 256, 257, 260, 300, 511, 516, 1000]
# around the 8 rows of a turn, the staged 64 / 256 entries, several stagings
LENS = [0, 1, 7, 8, 9, 31, 63, 64, 65, 130, 255, 256, 257, 520]


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("ty", [INT8, INT4, INT2, FP16, FP32, BF16])
def test_single_table(ops, oracle, burst, ty, waves):
    burst(waves)
    for i, dim in enumerate(DIMS):
        D = (dim + {INT4: 1, INT2: 3}.get(ty, 0)) // {INT4: 2, INT2: 4}.get(ty, 1) * {INT4: 2, INT2: 4}.get(ty, 1)
        for sbl in (True, False):
            rng = np.random.default_rng(1000 * ty + 10 * dim + sbl)
            rows, pad = 300, [0, 0, 1, 3, 12][(i + sbl) % 5]
            elem = max(1, H.BITS[ty] // 8)
            stride = H.default_stride_bytes(ty, D, sbl) + pad * elem
            table, _ = H.make_table(rng, ty, rows, D, sbl, stride_bytes=stride)
            lens = rng.permutation(LENS)
            off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
            idx = rng.integers(0, rows, size=int(off[-1])).astype([np.int64, np.int32][i % 2])
            if not sbl:
                idx[rng.random(len(idx)) < 0.1] = -1
            positional = i % 3 == 2
            w = rng.normal(size=max(LENS) if positional else len(idx)).astype(np.float32) if i % 3 else None
            S.check_case(ops, oracle, ty=ty, D=D, table=table, idx=idx, off_or_len=off, w=w, normalize=i % 2 == 0,
                         out_ty=[FP32, FP16, BF16][i % 3], positional=positional, use_offsets=True,
                         output_stride=-1 if i % 2 else D + 3, input_stride=stride // elem if pad else -1, sbl=sbl,
                         data_size=rows, output_size=len(lens), what=f"burst {waves}: ty={ty} D={D} trailer={sbl} pad={pad}")


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("align", [1, 4, 16])
def test_table_batched(ops, oracle, burst, waves, align):
    burst(waves)
    rng = np.random.default_rng(align)
    specs = [(50 + 10 * i, D, ty) for i, (D, ty) in enumerate(
        (D, ty) for ty in (INT8, INT4, INT2, FP16, FP32) for D in (4, 12, 36, 52, 100, 256, 300))]
    weights, wo, _ = TB.build_weights(rng, specs, align)
    B = 5
    lens = rng.choice(LENS[:9], size=len(specs) * B)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = np.concatenate([rng.integers(0, specs[t][0], size=int(lens[t * B:(t + 1) * B].sum())) for t in range(len(specs))])
    idx = idx.astype(np.int64)
    idx[rng.random(len(idx)) < 0.1] = -1
    psw = rng.normal(size=len(idx)).astype(np.float32)
    for pooling, out_ty, w in ((0, FP16, psw), (1, FP32, None), (0, BF16, psw)):
        got, want = TB.run_both(ops, oracle, weights, wo, specs, idx, off, pooling, w, out_ty, align)
        H.assert_same_bits(got, want, f"burst {waves}: align={align} pooling={pooling} out={out_ty}")


@pytest.mark.parametrize("waves", [1, 4])
def test_rejected_inputs(ops, oracle, burst, waves):
    """What the other kernels reject is rejected here, with the first position in index order."""
    burst(waves)
    rng = np.random.default_rng(5)
    D, rows = 300, 40
    table, _ = H.make_table(rng, INT8, rows, D, True)
    lens = np.array([3, 70, 0, 400, 5])
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    good = rng.integers(0, rows, size=int(off[-1])).astype(np.int64)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    kern = ops.generate_embedding_spmdm(ops.INT8, D, False, False)

    def bits(idx, offsets, index_size):
        st = ops.Status()
        out = torch.empty(len(lens) * D, device="cuda")
        kern(len(lens), index_size, rows, cu(table), cu(idx), cu(offsets), None, out, status=st)
        return st.read()

    assert bits(good, off, len(good)) == (0, -1)
    bad = good.copy()
    bad[[20, 300, 470]] = [rows, -1, 1 << 40]
    assert bits(bad, off, len(bad)) == (ops.ERR_INDEX_OUT_OF_RANGE, 20)
    assert bits(good, off, len(good) - 1)[0] & ops.ERR_BAG_OVERRUN
    down = off.copy()
    down[2] = 1
    assert bits(good, down, len(good))[0] & ops.ERR_NEGATIVE_LENGTH
    assert bits(good, off, len(good) + 1)[0] == ops.ERR_LENGTH_MISMATCH


@pytest.mark.parametrize("bags", [4095, 4097, 8192, 8193, 16384, 16385])
def test_both_sides_of_the_line(ops, oracle, bags):
    """The rule's own choice just below, at and above the numbers of bags where it changes."""
    rng = np.random.default_rng(bags)
    D, rows = 20, 500
    table, _ = H.make_table(rng, INT4, rows, D, True)
    lens = rng.integers(20, 33, size=bags)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    idx = rng.integers(0, rows, size=int(off[-1])).astype(np.int32)
    S.check_case(ops, oracle, ty=INT4, D=D, table=table, idx=idx, off_or_len=off, w=None, normalize=False, out_ty=FP32,
                 positional=False, use_offsets=True, output_stride=-1, input_stride=-1, sbl=True, data_size=rows,
                 output_size=bags, what=f"{bags} bags")


@pytest.mark.parametrize("avg", [95, 96, 255])
def test_whole_bags_in_the_tolerance_grade_mode(ops, avg):
    """Bags that the burst kernel takes whole in place of segments, on both sides of the length from which
    they get four waves, one bag much longer than the others: exact, so the bits of the exact mode."""
    rng = np.random.default_rng(avg)
    D, rows, bags = 64, 500, 600
    table, _ = H.make_table(rng, INT4, rows, D, True)
    lens = np.full(bags, avg - 10)
    lens[17] += 10 * bags
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    idx = cu(rng.integers(0, rows, size=int(off[-1])).astype(np.int32))
    kern = ops.generate_embedding_spmdm_nbit(4, D, False, False)
    outs = [torch.empty(bags, D, device="cuda") for _ in range(2)]
    for out, mode in zip(outs, (ops.ACC_EXACT, ops.ACC_FAST)):
        assert kern(bags, len(idx), rows, cu(table), idx, cu(off), None, out, accumulate=mode)
    H.assert_same_bits(outs[1].cpu().numpy(), outs[0].cpu().numpy(), f"{avg} entries per bag")
