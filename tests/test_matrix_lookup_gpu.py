"""The lookup on the matrix cores: unweighted bags of 4- and 8-bit rows in the tolerance-grade mode, against sums in 64
bits. A bag of n rows is 2 n additions (elements and biases) and three roundings more; each is at most one unit of 2^-23 of
what has been summed, so an fp32 result is within (2 n + 3) 2^-23 of the sum of the terms' magnitudes, and a 16-bit one
half a unit of its own more.

All tables that the kernel takes in one forward have one row type and width; tables of other kinds are pooled beside it from
2^21 lookups on. Every forward here asks the plan whether the kernel has taken it."""
import numpy as np
import pytest

from helpers import BF16, FP16, FP32, INT2, INT4, INT8

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ALIGN = 16
HALF_UNIT = {FP32: 0.0, FP16: 2.0 ** -11, BF16: 2.0 ** -8}
WIDTHS = [(128, INT4), (256, INT4), (64, INT8), (128, INT8)]


def cu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


class Forward:
    """A plan over the tables in the tolerance-grade mode, and forwards of it."""

    def __init__(self, specs, weights, offs):
        import fbgemm_amd.ops as ops
        D = np.concatenate([[0], np.cumsum([s[1] for s in specs])]).astype(np.int32)
        self.total_D = int(D[-1])
        # weights, unified-memory weights, placements, offsets, types, D offsets
        self.meta = (cu(weights), torch.zeros(0, dtype=torch.uint8, device="cuda"), cu(np.zeros(len(specs), np.int32)), cu(offs),
                     cu(np.array([s[2] for s in specs], np.uint8)), cu(D))
        w, uvm, place, offs, tys, D = self.meta
        self.plan = ops.TbePlan(offs, tys, D, place, w.numel(), 0, ALIGN)
        self.plan.set_accumulate(ops.ACC_FAST)

    def taken(self):
        import fbgemm_amd
        return fbgemm_amd.lib().fbgemm_amd_tbe_plan_matrix_forwards(self.plan.handle)

    def __call__(self, idx, off, out_ty, pooling=0, status=None):
        import fbgemm_amd.ops as ops
        before = self.taken()
        out = ops.int_nbit_split_embedding_codegen_lookup_function(
            *self.meta, self.total_D, 512, 512, 512, 512, 512, idx, off, pooling, None, out_ty, row_alignment=ALIGN, plan=self.plan, status=status)
        assert self.taken() == before + 1, "another kernel"
        return out


@pytest.fixture(autouse=True)
def neither_burst_nor_narrow():
    """A forward's launch goes neither to the burst kernel nor to the narrow lanes, whatever its size."""
    import fbgemm_amd
    lib = fbgemm_amd.lib()
    lib.fbgemm_amd_set_narrow_below_waves(0)
    yield
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


def check(got, specs, views, idx, off, B, out_ty, pooling=0, bags=None):
    """Every bag (or those of `bags` in each table) against the sums in 64 bits; bags may overlap, and a bag that ends in
    front of its start has no entries."""
    idx, off = torch.as_tensor(idx).cuda(), torch.as_tensor(off).cuda()
    col = 0
    for t, ((rows, D, ty), view) in enumerate(zip(specs, views)):
        q, s, b = (cu(v) for v in view)
        first = off[t * B:(t + 1) * B]
        n = (off[t * B + 1:(t + 1) * B + 1] - first).clamp(min=0)
        bag = torch.repeat_interleave(torch.arange(B, device="cuda"), n)
        entry = torch.arange(bag.numel(), device="cuda") - (n.cumsum(0) - n)[bag] + first[bag]
        i = idx[entry]
        here = (i >= 0) & (i < rows)
        i, bag = i[here], bag[here]
        terms, add = (q * s[:, None])[i], b[i][:, None]
        zero = torch.zeros(B, D, dtype=torch.float64, device="cuda")
        want, size = zero.index_add(0, bag, terms + add), zero.index_add(0, bag, terms.abs() + add.abs())
        n = n.double()[:, None]
        if pooling:
            want, size = want / n.clamp(min=1), size / n.clamp(min=1)
        bound = (2 * n + 3) * 2.0 ** -23 * size + HALF_UNIT[out_ty] * want.abs() + (2.0 ** -25 if out_ty == FP16 else 0)
        err = (got[:, col:col + D].double() - want).abs()
        bad = ~(err <= bound)
        if bags is not None:
            bad = bad[bags]
        assert not bool(bad.any()), (t, bad.nonzero()[0].tolist(), float((err / bound.clamp(min=1e-300)).max()))
        col += D


@pytest.mark.parametrize("D,ty", WIDTHS)
@pytest.mark.parametrize("B", [1, 7, 8, 9, 65])
def test_matrix_lookup_every_width(D, ty, B):
    """Bags around the blocks of 16 and stages of 64 entries, bags that do not fill a wave, pruned rows."""
    rng = np.random.default_rng(D * 100 + ty * 10 + B)
    specs = [(400, D, ty), (1, D, ty), (77, D, ty)]
    weights, offs, views = tables(rng, specs)
    fwd = Forward(specs, weights, offs)
    edges = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200]
    lens = rng.choice(edges, size=len(specs) * B)
    lens[0] = [0, 1, 64, 129, 16][B % 5]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = np.concatenate([rng.integers(0, s[0], int(lens[t * B:(t + 1) * B].sum())) for t, s in enumerate(specs)]).astype(np.int64)
    idx[rng.random(len(idx)) < 0.05] = -1
    for index in (np.int64, np.int32):
        for out_ty in (FP32, FP16, BF16):
            for pooling in (0, 1):
                got = fwd(cu(idx.astype(index)), cu(off.astype(index)), out_ty, pooling)
                check(got, specs, views, idx, off, B, out_ty, pooling)


@pytest.mark.parametrize("D,ty", WIDTHS)
def test_matrix_lookup_keeps_a_bags_infinities_to_itself(D, ty):
    """Scales and biases that are infinite, denormal or zero, beside bags of ordinary rows."""
    rng = np.random.default_rng(3)
    specs = [(64, D, ty)] * 2
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
    got = Forward(specs, weights, offs)(cu(idx), cu(off), FP32)
    for t, (q, s, b) in enumerate(views):
        block = got[:, t * D:(t + 1) * D].cpu().numpy()
        zero = q[0] == 0  # infinity times zero
        assert np.isnan(block[0][zero]).all() and (block[0][~zero] == np.inf).all()
        assert (block[1] == -np.inf).all() and np.isnan(block[2]).all()
        assert np.isfinite(block[3:]).all()
    check(got, specs, views, idx, off, B, FP32, bags=slice(3, None))


@pytest.mark.parametrize("D,ty", WIDTHS)
def test_matrix_lookup_reports_what_it_rejects(D, ty):
    """Indices outside their table add nothing and the first is reported; offsets that are not in order cost their bag."""
    from fbgemm_amd import ops
    rng = np.random.default_rng(4)
    specs, B = [(50, D, ty), (60, D, ty)], 20
    weights, offs, views = tables(rng, specs)
    fwd = Forward(specs, weights, offs)
    lens = rng.integers(10, 30, size=2 * B)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = rng.integers(0, 50, size=int(off[-1])).astype(np.int64)
    idx[[37, 200, 201]] = [50, -2, -(1 << 63)]
    st = ops.Status()
    check(fwd(cu(idx), cu(off), FP32, status=st), specs, views, idx, off, B, FP32)
    assert st.read() == (1, 37)
    st.clear()
    idx[37] = 0
    fwd(cu(idx), cu(off), FP32, status=st)
    assert st.read() == (1, 200)
    st.clear()
    idx = idx % 50
    bad = off.copy()
    bad[5] = off[6] + 3  # bag 4 longer, bag 5 negative; the wave's bags are pooled one by one
    got = fwd(cu(idx), cu(bad), FP32, status=st)
    assert st.read()[0] == 8
    check(got, specs, views, idx, bad, B, FP32)
    st.clear()
    over = off.copy()
    over[-1] += 7
    got = fwd(cu(idx), cu(over), FP32, status=st)
    assert st.read()[0] == 2
    over[-1] = over[-2]  # the last bag adds nothing
    check(got, specs, views, idx, over, B, FP32)


@pytest.mark.parametrize("D,ty", WIDTHS)
def test_matrix_lookup_of_many_bags(D, ty):
    """So many bags that a wave pools sixteen, the last of a table fewer; bags of 0 .. 5 entries and some of 150."""
    rng = np.random.default_rng(D + ty)
    T, B, rows = 5, 53001, 300
    specs = [(rows, D, ty)] * T
    weights, offs, views = tables(rng, specs)
    fwd = Forward(specs, weights, offs)
    lens = rng.integers(0, 6, size=T * B)
    lens[rng.integers(0, T * B, size=2000)] = 150
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = rng.integers(0, rows, size=int(off[-1])).astype(np.int64)
    for out_ty in (FP32, BF16):
        check(fwd(cu(idx), cu(off), out_ty), specs, views, idx, off, B, out_ty)


@pytest.mark.parametrize("D,ty", WIDTHS)
@pytest.mark.parametrize("beside", [1, 6])
def test_matrix_lookup_beside_other_tables(D, ty, beside):
    """From 2^21 lookups on, tables that the kernel does not take are pooled beside it: few 2-bit ones, whose bags are not
    ordered then, and so many that they are; their columns between the others'."""
    rng = np.random.default_rng(D + beside)
    specs = [(300, 32, INT2), (300, D, ty), (200, 64, INT2), (100, D, ty), (50, 36, INT2), (50, 28, INT2), (9, 32, INT2), (200, 64, INT2)]
    specs = specs[:4] + specs[4:3 + beside] if beside > 1 else specs[1:2] + specs[:1] + specs[3:4]
    T = len(specs)
    weights, offs, views = tables(rng, specs)
    fwd = Forward(specs, weights, offs)
    B = 1500
    lens = rng.integers(0, 2 * (-(-(1 << 21) // (T * B))) + 100, size=T * B)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = np.concatenate([rng.integers(-1, s[0], int(lens[t * B:(t + 1) * B].sum())) for t, s in enumerate(specs)]).astype(np.int64)
    assert len(idx) >= 1 << 21
    for out_ty, pooling in ((FP32, 0), (FP16, 1)):
        check(fwd(cu(idx), cu(off), out_ty, pooling), specs, views, idx, off, B, out_ty, pooling)


@pytest.mark.parametrize("beside", [False, True])
def test_matrix_lookup_replays_from_a_graph(beside):
    """Captured on a stream the plan has not met, alone and with 2-bit tables on the side stream; every replay against the
    eager forward and the sums in 64 bits, with eager work of the same plan between the replays."""
    from fbgemm_amd import ops
    rng = np.random.default_rng(9)
    specs = [(500, 128, INT8)] * 3 + ([(300, 32, INT2)] if beside else [])
    weights, offs, views = tables(rng, specs)
    fwd = Forward(specs, weights, offs)
    T, B = len(specs), 700
    L = -(-(1 << 21) // (T * B)) if beside else 20  # the side stream belongs to forwards that order their bags
    off = cu((np.arange(T * B + 1) * L).astype(np.int64))
    idx = torch.zeros(T * B * L, dtype=torch.int64, device="cuda")
    st = ops.Status()
    call = lambda: fwd(idx, off, BF16, status=st)
    call()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            captured = call()
    torch.cuda.synchronize()
    for _ in range(4):
        idx.copy_(cu(rng.integers(0, 300, size=idx.numel())))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(call(), captured)
        torch.cuda.synchronize()
        check(captured, specs, views, idx, off, B, BF16)
    assert st.read() == (0, -1)
