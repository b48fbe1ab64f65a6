"""The module's forward with its check in the lookup's own kernels against the check and the forward as two calls: the
same bits and the same warning count, for every kernel that such a forward can take, over indices and offsets that
are in order, repaired and refused."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# row types and widths of the tables, bags per table, entries per bag: the burst kernel with one wave and four, in several
# windows of columns; the lean kernel, ordered and not; its instance for wide 4-bit rows; the general kernel with wide
# lanes and several column passes; both in one launch
SHAPES = {
    "burst": ([("int4", 64), ("int8", 128), ("fp16", 256), ("int2", 32)], 40, 20),
    "burst windows": ([("int8", 300), ("fp32", 520)], 33, 90),
    "lean": ([("int4", 64), ("int8", 128), ("fp16", 64)], 16_000, 4),
    "lean ordered": ([("int4", 64), ("int8", 64)], 16_000, 68),
    "wide": ([("int4", 256)] * 2, 9000, 122),
    "general": ([("int2", 36), ("fp8", 20), ("int8", 100), ("fp32", 20)], 6000, 6),
    "passes": ([("fp32", 1500)], 5000, 4),
    "both": ([("int4", 64), ("fp32", 12), ("int8", 128), ("int2", 52)], 6000, 8),
}


def make(case, pruned, mode, rng, indices_dtype=torch.int32, entries=()):
    from fbgemm_amd import module as M
    tables, B, avg = SHAPES[case]
    specs = [("", int(rng.integers(200, 900)), d, M.SparseType(ty), M.EmbeddingLocation.DEVICE) for ty, d in tables]
    m = M.IntNBitTableBatchedEmbeddingBagsCodegen(specs, bounds_check_mode=M.BoundsCheckMode(mode), output_dtype=M.SparseType.FP32,
                                                  pooling_mode=M.PoolingMode.MEAN, fp8_exponent_bits=4, fp8_exponent_bias=7,
                                                  indices_dtype=indices_dtype)
    m.quantize_and_assign([torch.from_numpy(rng.normal(size=(n, d)).astype(np.float32)) for _, n, d, _, _ in specs])
    logical = [n for _, n, _, _, _ in specs]
    if pruned:  # not all tables, and entries beyond the physical rows and below -1 among the mappings'
        maps = [None if t % 3 == 2 else torch.from_numpy(rng.integers(-1, n + 2, size=2 * n) - 3 * (rng.random(2 * n) < 0.01))
                for t, n in enumerate(logical)]
        for k, entry in enumerate(entries):
            maps[0][3 + k::17] = entry
        m.set_index_remappings([None if a is None else a.cuda() for a in maps])
        logical = [n if a is None else 2 * n for n, a in zip(logical, maps)]
    lens = rng.integers(0, 2 * avg + 1, size=len(tables) * B)
    off = np.concatenate([[0], np.cumsum(lens)])
    idx = np.concatenate([rng.integers(0, n, size=int(off[(t + 1) * B] - off[t * B])) for t, n in enumerate(logical)])
    return m, idx, off


def apart(m, idx, off, psw):
    from fbgemm_amd import ops
    maps = (m.original_rows_per_table, m._feature_remap_array, m._feature_remap_offsets) if m.index_remappings_array.numel() else (None,) * 3
    warning = torch.full((1,), 5, dtype=torch.int64, device="cuda")
    i, o = ops.check_remap_indices(m.rows_per_table, idx, off, m.bounds_check_mode_int, warning, psw, *maps)
    out = ops.int_nbit_split_embedding_codegen_lookup_function(
        m.weights_dev, m.weights_uvm, m.weights_placements, m.weights_offsets, m.weights_tys, m.D_offsets, m.total_D, m.max_int2_D,
        m.max_int4_D, m.max_int8_D, m.max_float16_D, m.max_float32_D, i, o, int(m.pooling_mode), psw, m.output_dtype,
        row_alignment=m.row_alignment, max_float8_D=m.max_float8_D, fp8_exponent_bits=4, fp8_exponent_bias=7)
    return out, int(warning)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("pruned", [False, True])
@pytest.mark.parametrize("case", SHAPES)
def test_same_as_check_and_forward(case, pruned, dtype):
    from fbgemm_amd import ops
    rng = np.random.default_rng(len(case) + 2 * pruned)
    for mode in (1, 2):
        m, idx, off = make(case, pruned, mode, rng)
        taken = not pruned or case in ("burst", "burst windows", "lean", "lean ordered", "wide")
        for what in ("good", "indices", "offsets", "last", "first", "weighted"):
            i2, o2 = idx.copy(), off.copy()
            if what in ("indices", "weighted"):
                hit = rng.random(len(i2)) < 0.02
                i2[hit] = rng.choice([-1, -2, -(1 << 31), 1000, 1 << 30], size=int(hit.sum()))
            elif what == "offsets":
                o2[rng.integers(1, len(o2) - 1, size=3)] += 40
            elif what == "last":
                o2[-1] += rng.choice([-1, 2])
            elif what == "first":
                o2[0] = rng.choice([-3, 1])
            cu = lambda a: torch.from_numpy(a).cuda().to(dtype)
            psw = torch.rand(len(idx), device="cuda") if what == "weighted" else None
            args = (cu(i2), cu(o2), psw)
            before = [a.clone() for a in args[:2]]
            want, count = apart(m, *args)
            calls = []
            run = ops.checked_lookup
            try:
                ops.checked_lookup = lambda *a: calls.append(run(*a)) or calls[-1]
                for _ in range(2):  # the second time the counter is not what the first has found
                    m._apart_left, m._apart_for = 0, -1
                    m.bounds_check_warning.fill_(77)
                    got = m(*args)
                    assert torch.equal(got.view(torch.int32), want.view(torch.int32)), (what, mode)
                    assert int(m.bounds_check_warning) == (count if mode == 1 else 77), (what, mode)
            finally:
                ops.checked_lookup = run
            assert all(torch.equal(a, b) for a, b in zip(args, before))
            in_order = bool(o2[0] >= 0 and (np.diff(o2) >= 0).all() and o2[-1] == len(idx))
            assert [(out is None, repair) for out, repair in calls] == [(not (taken and in_order), taken and not in_order)] * 2, (what, mode)


def in_the_kernels(m, *args):
    """A forward that has to be made in the lookup's own kernels."""
    from fbgemm_amd import ops
    run, calls = ops.checked_lookup, []
    try:
        ops.checked_lookup = lambda *a: calls.append(run(*a)) or calls[-1]
        out = m(*args)
    finally:
        ops.checked_lookup = run
    assert [c[0] is out for c in calls] == [True]
    return out


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("case,pruned", [(c, p) for c in ("lean", "lean ordered", "wide") for p in (False, True)] + [("both", False)])
def test_waves_that_cannot_be_prescaled_count_once(case, pruned, dtype):
    """Scales and weights that send a wave of the lean kernels to its row-at-a-time loop, which every lane of a bag walks,
    with indices outside the tables among them: still the same bits and the same count."""
    import fbgemm_amd
    rng = np.random.default_rng(7)
    m, idx, off = make(case, pruned, 1, rng)
    for (_, rows, _, ty, _), (_, head) in zip(m.embedding_specs, m.split_embedding_weights()):
        if not ty.is_float():  # a few rows whose scale (or bias) is no number
            head[3], head[rows // 2] = (torch.tensor(h, dtype=torch.float16).view(torch.uint8).cuda() for h in ([np.inf, 1.0], [np.nan, np.inf]))
    hit = rng.random(len(idx)) < 0.02
    idx[hit] = rng.choice([-2, 1000, 1 << 30], size=int(hit.sum()))
    huge = torch.rand(len(idx), device="cuda")
    huge[::977] = 2.0 ** 120
    huge[::1999] = float("inf")
    idx, off = (torch.from_numpy(a).cuda().to(dtype) for a in (idx, off))
    lib = fbgemm_amd.lib()
    try:
        for wide4 in (0, 2) if case == "wide" else (-1,):  # both lean kernels of wide 4-bit rows
            lib.fbgemm_amd_set_wide4(wide4)
            for psw in (None, huge):
                want, count = apart(m, idx, off, psw)
                m.bounds_check_warning.fill_(77)
                assert torch.equal(in_the_kernels(m, idx, off, psw).view(torch.int32), want.view(torch.int32))
                assert int(m.bounds_check_warning) == count > 0
    finally:
        lib.fbgemm_amd_set_wide4(-1)


IN_KERNELS = [(c, p) for c in SHAPES for p in (False, True) if not p or c in ("burst", "burst windows", "lean", "lean ordered", "wide")]


@pytest.mark.parametrize("case,pruned", IN_KERNELS)
def test_lowest_value_of_an_index(case, pruned):
    """No value of an index, or of a mapping's entry, is anything but an index: the lowest is outside its table like any other."""
    rng = np.random.default_rng(11)
    low = -(1 << 63)
    m, idx, off = make(case, pruned, 1, rng, torch.int64, (low, low + 1))
    hit = rng.random(len(idx)) < 0.02
    idx[hit] = rng.choice([low, low + 1, -1], size=int(hit.sum()))
    idx, off = torch.from_numpy(idx).cuda(), torch.from_numpy(off).cuda()
    want, count = apart(m, idx, off, None)
    assert torch.equal(in_the_kernels(m, idx, off).view(torch.int32), want.view(torch.int32))
    assert int(m.bounds_check_warning) == count > 0


@pytest.mark.parametrize("case", [c for c, p in IN_KERNELS if p])
def test_entries_wider_than_the_indices(case):
    """A mapping of 64-bit entries under 32-bit indices: what does not fit them is cut, as the check of its own cuts it."""
    m, idx, off = make(case, True, 1, np.random.default_rng(13), torch.int64, ((1 << 32) - 1, (1 << 32) + 3, 1 << 31, (1 << 40) + 10_000))
    idx, off = torch.from_numpy(idx).cuda().int(), torch.from_numpy(off).cuda().int()
    want, count = apart(m, idx, off, None)
    assert torch.equal(in_the_kernels(m, idx, off).view(torch.int32), want.view(torch.int32))
    assert int(m.bounds_check_warning) == count > 0


@pytest.mark.parametrize("case", ["burst", "lean", "wide", "general", "both"])
def test_lowest_value_of_an_index_is_reported(case):
    """The same in a forward that does not check."""
    from fbgemm_amd import ops
    m, idx, off = make(case, False, 0, np.random.default_rng(12))
    at = len(idx) // 3
    idx[at] = -(1 << 63)
    st = ops.Status()
    ops.int_nbit_split_embedding_codegen_lookup_function(
        m.weights_dev, m.weights_uvm, m.weights_placements, m.weights_offsets, m.weights_tys, m.D_offsets, m.total_D, m.max_int2_D,
        m.max_int4_D, m.max_int8_D, m.max_float16_D, m.max_float32_D, torch.from_numpy(idx).cuda(), torch.from_numpy(off).cuda(), 0, None,
        m.output_dtype, row_alignment=m.row_alignment,
        max_float8_D=m.max_float8_D, fp8_exponent_bits=4, fp8_exponent_bias=7, status=st)
    assert st.read() == (ops.ERR_INDEX_OUT_OF_RANGE, at)


def test_counts_and_apart_forwards():
    """What a forward that had to be repaired leaves behind: some forwards in two calls, then one again, on any stream."""
    rng = np.random.default_rng(0)
    m, idx, off = make("burst", False, 1, rng)
    idx, off = torch.from_numpy(idx).cuda(), torch.from_numpy(off).cuda()
    want, _ = apart(m, idx, off, None)
    bad, bad_off = idx.clone(), off.clone()
    bad[7:27] = 10_000
    bad_off[-1] += 1
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for k in range(140):
        with torch.cuda.stream(side if k % 3 else torch.cuda.current_stream()):
            if k == 30:
                m(idx, bad_off)
                assert int(m.bounds_check_warning) == 1 and m._apart_left == 64
            elif k % 7 == 0:
                m(bad, off)
                assert int(m.bounds_check_warning) == 20, k
            else:
                assert torch.equal(m(idx, off), want) and int(m.bounds_check_warning) == 0, k
    assert m._apart_left == 0
    # a row count of nothing, and one that the weights have no room for: what the two calls make of them
    bad = torch.full_like(idx, 950)
    m.rows_per_table[1] = 0
    want, count = apart(m, bad, off, None)
    assert torch.equal(m(bad, off), want) and int(m.bounds_check_warning) == count
    m.rows_per_table[1], m._apart_left = 1 << 20, 0
    errors = []
    for f in (lambda: apart(m, bad, off, None), lambda: m(bad, off)):
        with pytest.raises(RuntimeError) as e:
            f()
        errors.append(str(e.value))
    assert errors[0] == errors[1]


def test_refusals_are_not_for_ever():
    """A forward that the kernels do not check says little about others of its batch size: not where it was captured or its
    arguments were wrong, and where the mapping or the plan's arithmetic was why, not once that has changed."""
    from fbgemm_amd import ops
    rng = np.random.default_rng(5)
    m, idx, off = make("lean", False, 1, rng)
    idx, off = torch.from_numpy(idx).cuda(), torch.from_numpy(off).cuda()
    want, _ = apart(m, idx, off, None)
    assert torch.equal(in_the_kernels(m, idx, off), want)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            assert m._checked_forward(m._buffers, idx, off, None, False, len(m.embedding_specs)) is None
            torch.zeros(8, device="cuda")  # a graph of something
    torch.cuda.synchronize()
    assert torch.equal(in_the_kernels(m, idx, off), want)
    with pytest.raises(RuntimeError):
        m(idx, off, torch.ones(len(idx) - 1, device="cuda"))
    assert torch.equal(in_the_kernels(m, idx, off), want)
    plan = ops._plan_for(m.weights_dev, m.weights_uvm, m.weights_placements, m.weights_offsets, m.weights_tys, m.D_offsets, m.row_alignment)
    tried, run = [], ops.checked_lookup
    try:
        ops.checked_lookup = lambda *a: tried.append(run(*a)) or tried[-1]
        plan.set_accumulate(ops.ACC_FAST)
        for _ in range(10):
            m(idx, off)
        assert len(tried) == 1 and tried[0][0] is None
        plan.set_accumulate(ops.ACC_EXACT)
        for _ in range(60):
            assert torch.equal(m(idx, off), want)
        assert len(tried) == 6 and all(c[0] is not None for c in tried[1:])
    finally:
        ops.checked_lookup = run
    m, idx, off = make("both", True, 1, rng)
    idx, off = torch.from_numpy(idx % 200).cuda(), torch.from_numpy(off).cuda()
    m(idx, off)
    m.set_index_remappings([None] * len(m.embedding_specs))
    assert torch.equal(in_the_kernels(m, idx, off), apart(m, idx, off, None)[0])
