"""The lookup on the matrix cores: unweighted bags of 4- and 8-bit rows in the tolerance-grade mode, against sums in 64
bits. A bag of n rows is 2 n additions (elements and biases) and three roundings more; each is at most one unit of 2^-23 of
what has been summed, so an fp32 result is within (2 n + 3) 2^-23 of the sum of the terms' magnitudes, and a 16-bit one
half a unit of its own more."""
import numpy as np
import pytest

from helpers import BF16, FP16, FP32, INT2, INT4, INT8

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ALIGN = 16
TORCH = {FP32: torch.float32, FP16: torch.float16, BF16: torch.bfloat16}
HALF_UNIT = {FP32: 0.0, FP16: 2.0 ** -11, BF16: 2.0 ** -8}


@pytest.fixture
def fwd():
    """A forward whose launch neither the burst kernel nor the narrow lanes take, whatever its size."""
    import fbgemm_amd
    import fbgemm_amd.ops as ops
    lib = fbgemm_amd.lib()
    lib.fbgemm_amd_set_narrow_below_waves(0)

    def run(specs, weights, offs, idx, off, out_ty, pooling=0, index=np.int64, status=None):
        T = len(specs)
        D = np.concatenate([[0], np.cumsum([s[1] for s in specs])]).astype(np.int32)
        cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
        return ops.int_nbit_split_embedding_codegen_lookup_function(
            cu(weights), torch.zeros(0, dtype=torch.uint8, device="cuda"), cu(np.zeros(T, np.int32)), cu(offs),
            cu(np.array([s[2] for s in specs], np.uint8)), cu(D), int(D[-1]), 512, 512, 512, 512, 512,
            cu(idx.astype(index)), cu(off.astype(index)), pooling, None, out_ty, row_alignment=ALIGN,
            accumulate=ops.ACC_FAST, **({} if status is None else {"status": status}))
    yield run
    lib.fbgemm_amd_set_narrow_below_waves(-1)


def row_bytes(D, ty):
    return (4 + D * {INT8: 8, INT4: 4, INT2: 2}[ty] // 8 + ALIGN - 1) // ALIGN * ALIGN


def tables(rng, specs, scale=(1e-3, 5e-2), bias=(-1.0, 1.0)):
    """(all rows' bytes, where each table starts, per table the integers, scales and biases)."""
    parts, offs, views, at = [], [], [], 0
    for rows, D, ty in specs:
        t = rng.integers(0, 256, size=(rows, row_bytes(D, ty)), dtype=np.uint8)
        sb = np.stack([rng.uniform(*scale, rows), rng.uniform(*bias, rows)], 1).astype(np.float16)
        t[:, :4] = sb.view(np.uint8)
        data = t[:, 4:4 + row_bytes(D, ty)]
        per = {INT8: 1, INT4: 2, INT2: 4}[ty]
        bits = 8 // per
        q = np.stack([(data >> (bits * k)) & (2 ** bits - 1) for k in range(per)], -1).reshape(rows, -1)[:, :D]
        views.append((q.astype(np.float64), sb[:, 0].astype(np.float64), sb[:, 1].astype(np.float64)))
        offs.append(at)
        at += t.size
        parts.append(t.reshape(-1))
    return np.concatenate(parts), np.array(offs, np.int64), views


def check(got, specs, views, idx, off, B, out_ty, pooling=0):
    got = got.float().cpu().numpy().astype(np.float64)
    col = 0
    for t, (rows, D, ty) in enumerate(specs):
        q, s, b = views[t]
        for bag in range(B):
            i = idx[off[t * B + bag]:off[t * B + bag + 1]]
            n, i = len(i), i[(i >= 0) & (i < rows)]
            terms = q[i] * s[i, None]
            want, size = (terms + b[i, None]).sum(0), (np.abs(terms) + np.abs(b[i, None])).sum(0)
            if pooling and n:
                want, size = want / n, size / n
            bound = (2 * len(i) + 3) * 2.0 ** -23 * size + HALF_UNIT[out_ty] * np.abs(want) + (2.0 ** -25 if out_ty == FP16 else 0)
            err = np.abs(got[bag, col:col + D] - want)
            assert (err <= bound).all(), (t, bag, n, float((err / np.maximum(bound, 1e-300)).max()))
        col += D


@pytest.mark.parametrize("D,ty", [(128, INT4), (256, INT4), (64, INT8), (128, INT8)])
@pytest.mark.parametrize("B", [1, 7, 8, 9, 65])
def test_matrix_lookup_every_width(fwd, D, ty, B):
    """Bags around the blocks of 16 and stages of 64 entries, bags that do not fill a wave, pruned rows."""
    rng = np.random.default_rng(D * 100 + ty * 10 + B)
    specs = [(400, D, ty), (1, D, ty), (77, 32, INT2), (90, 64, INT4)]  # two of them for other kernels
    weights, offs, views = tables(rng, specs)
    edges = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200]
    lens = rng.choice(edges, size=len(specs) * B)
    lens[0] = [0, 1, 64, 129, 16][B % 5]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = np.concatenate([rng.integers(0, s[0], int(lens[t * B:(t + 1) * B].sum())) for t, s in enumerate(specs)]).astype(np.int64)
    idx[rng.random(len(idx)) < 0.05] = -1
    for out_ty, pooling, index in ((FP32, 0, np.int64), (FP16, 1, np.int32), (BF16, 0, np.int32), (FP32, 1, np.int64)):
        check(fwd(specs, weights, offs, idx, off, out_ty, pooling, index), specs, views, idx, off, B, out_ty, pooling)


def test_matrix_lookup_keeps_a_bags_infinities_to_itself(fwd):
    """Scales and biases that are infinite, denormal or zero, beside bags of ordinary rows."""
    rng = np.random.default_rng(3)
    specs = [(64, 256, INT4), (64, 128, INT8)]
    weights, offs, views = tables(rng, specs)
    B = 11
    for t, (rows, D, ty) in enumerate(specs):
        w = weights[offs[t]:offs[t] + rows * row_bytes(D, ty)].reshape(rows, -1)
        for r, (s, b) in enumerate([(np.inf, 0), (1, -np.inf), (np.nan, 1), (2.0 ** -24, 2.0 ** -24), (65504, -65504), (0, 0)]):
            sb = np.array([s, b], np.float16)
            w[r, :4] = sb.view(np.uint8)
            views[t][1][r], views[t][2][r] = float(sb[0]), float(sb[1])
    off = (np.arange(2 * B + 1) * 5).astype(np.int64)
    idx = rng.integers(6, 64, size=2 * B * 5).astype(np.int64)
    for t in range(2):  # bags 0 .. 2 hold one row each that is not finite; 3 .. 5 nothing but denormals, large ones, zeros
        for r in range(3):
            idx[off[t * B + r] + 2] = r
        for r in range(3, 6):
            idx[off[t * B + r]:off[t * B + r + 1]] = r
    got = fwd(specs, weights, offs, idx, off, FP32)
    col = 0
    for t, (rows, D, ty) in enumerate(specs):
        q, s, b = views[t]
        block = got[:, col:col + D].cpu().numpy()
        zero = q[0] == 0  # infinity times zero
        assert np.isnan(block[0][zero]).all() and (block[0][~zero] == np.inf).all()
        assert (block[1] == -np.inf).all() and np.isnan(block[2]).all()
        assert np.isfinite(block[3:]).all()
        finite = [(v[0], np.where(np.isfinite(v[1]), v[1], 0), np.where(np.isfinite(v[2]), v[2], 0)) for v in views]
        col += D
    keep = got.clone()
    keep[:3] = 0
    idx0 = idx.copy()
    off0 = off.copy()
    for t in range(2):
        idx0[off[t * B]:off[t * B + 3]] = -1
    check(keep, specs, finite, idx0, off0, B, FP32)


def test_matrix_lookup_reports_what_it_rejects(fwd):
    """Indices outside their table add nothing and the first is reported; offsets that are not in order cost their bag."""
    from fbgemm_amd import ops
    rng = np.random.default_rng(4)
    specs, B = [(50, 256, INT4), (60, 128, INT4)], 20
    weights, offs, views = tables(rng, specs)
    lens = rng.integers(10, 30, size=2 * B)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = rng.integers(0, 50, size=int(off[-1])).astype(np.int64)
    idx[[37, 200]] = [50, -2]
    st = ops.Status()
    check(fwd(specs, weights, offs, idx, off, FP32, status=st), specs, views, idx, off, B, FP32)
    assert st.read() == (1, 37)
    st.clear()
    bad = off.copy()
    bad[5] = off[6] + 3  # bag 4 longer, bag 5 negative; bags 0 .. 3 and 6 .. are as they were
    got = fwd(specs, weights, offs, idx % 50, bad, FP32, status=st)
    assert st.read()[0] == 8
    ref = fwd(specs, weights, offs, idx % 50, off, FP32)
    assert torch.equal(got[5, :256], torch.zeros_like(got[5, :256]))
    keep = [i for i in range(B) if i not in (4, 5)]
    # (a bag pooled on its own is summed in other groups of 16)
    assert torch.allclose(got[keep], ref[keep], rtol=1e-5, atol=1e-5)
    st.clear()
    over = off.copy()
    over[-1] += 7
    fwd(specs, weights, offs, idx % 50, over, FP32, status=st)
    assert st.read()[0] == 2


@pytest.mark.parametrize("D,ty", [(128, INT4), (256, INT4), (64, INT8), (128, INT8)])
def test_matrix_lookup_of_many_bags(fwd, D, ty):
    """So many bags that a wave pools sixteen, the last of a table fewer; bags of 0 .. 5 entries and some of 150."""
    rng = np.random.default_rng(D + ty)
    T, B, rows = 5, 53001, 300
    specs = [(rows, D, ty)] * T
    weights, offs, views = tables(rng, specs)
    lens = rng.integers(0, 6, size=T * B)
    lens[rng.integers(0, T * B, size=2000)] = 150
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = rng.integers(0, rows, size=int(off[-1])).astype(np.int64)
    got = fwd(specs, weights, offs, idx, off, FP32).double()
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    bag = torch.repeat_interleave(torch.arange(T * B, device="cuda"), dev(lens))
    for t, (q, s, b) in enumerate(views):
        lo, hi = off[t * B], off[(t + 1) * B]
        i, where = dev(idx[lo:hi]), bag[lo:hi] - t * B
        q, s, b = dev(q), dev(s)[:, None], dev(b)[:, None]
        want, size = (torch.zeros(B, D, dtype=torch.float64, device="cuda").index_add_(0, where, x[i]) for x in (q * s + b, q * s + b.abs()))
        n = dev(lens[t * B:(t + 1) * B]).double()[:, None]
        err = (got[:, t * D:(t + 1) * D] - want).abs()
        assert bool((err <= (2 * n + 3) * 2.0 ** -23 * size).all())


@pytest.mark.parametrize("beside", [False, True])
def test_matrix_lookup_replays_from_a_graph(fwd, beside):
    """Captured on a stream the plan has not met, alone and with 2-bit tables on the side stream; every replay against the
    eager forward, with eager work of the same plan between the replays."""
    from fbgemm_amd import ops
    rng = np.random.default_rng(9)
    specs = [(500, 128, INT8)] * 3 + ([(300, 32, INT2)] if beside else [])
    weights, offs, _ = tables(rng, specs)
    T, B = len(specs), 700
    L = -(-(1 << 21) // (T * B)) if beside else 20  # the side stream belongs to forwards that order their bags
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    D = np.concatenate([[0], np.cumsum([s[1] for s in specs])]).astype(np.int32)
    meta = (dev(weights), torch.zeros(0, dtype=torch.uint8, device="cuda"), dev(np.zeros(T, np.int32)), dev(offs), dev(np.array([s[2] for s in specs], np.uint8)), dev(D))
    off = dev((np.arange(T * B + 1) * L).astype(np.int64))
    idx = torch.zeros(T * B * L, dtype=torch.int64, device="cuda")
    st = ops.Status()
    call = lambda: ops.int_nbit_split_embedding_codegen_lookup_function(
        *meta, int(D[-1]), 512, 512, 512, 512, 512, idx, off, 0, None, BF16, row_alignment=ALIGN, status=st, accumulate=ops.ACC_FAST)
    call()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            captured = call()
    torch.cuda.synchronize()
    for _ in range(4):
        idx.copy_(dev(rng.integers(0, 300, size=idx.numel())))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(call(), captured)
        torch.cuda.synchronize()
    assert st.read() == (0, -1)
