"""The one-pass bounds check and pruned-row mapping against the operators it stands for, run one after
the other: exact, over table and batch counts around its workgroups of 256 bags and its three ways of
carrying the running maximum, with broken offsets, indices and mappings."""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    import fbgemm_amd.ops as o
    return o


def one_after_the_other(ops, rows, indices, offsets, mode, warning, logical, remap, remap_offsets):
    indices, offsets = indices.clone(), offsets.clone()
    if remap is not None:
        ops.bounds_check_indices(logical, indices, offsets, mode, warning)
        indices = ops.pruned_array_lookup(indices, offsets, remap, remap_offsets)
    ops.bounds_check_indices(rows, indices, offsets, mode, warning)
    return indices, offsets


#                       one bag, one table's window, several tables in a window, B = 1, one launch at most, a kernel
#                       more, maxima of the second level, more of those than a workgroup reads itself
SHAPES = [(1, 1, 40), (1, 255, 9), (1, 256, 9), (1, 257, 9), (9, 32, 20), (70, 1, 15), (300, 1, 3), (16, 256, 12), (17, 241, 30),
          (3, 3000, 12), (2, 4104, 3), (2, 100_000, 2), (2, 530_000, 1), (2, 4_300_000, 1)]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("mapped", [None, torch.int32, torch.int64])
@pytest.mark.parametrize("mode", [1, 2])
def test_same_as_the_operators(ops, mode, mapped, dtype):
    cu = lambda a, dt=None: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt or torch.int64)
    for n, (T, B, avg) in enumerate(SHAPES):
        rng = np.random.default_rng(100 * n + mode)
        rows = rng.integers(1, 500, size=T)
        logical = rows.copy()
        remap = remap_offsets = None
        if mapped is not None:
            has = rng.random(T) < 0.8
            has[0] = True
            logical = np.where(has, 2 * rows, rows)
            sizes = np.where(has, 2 * rows, 0)
            remap_offsets = np.concatenate([[0], np.cumsum(sizes)])
            remap = np.concatenate([rng.integers(-1, rows[t] + 1, size=sizes[t]) for t in range(T)])  # rows[t]: not a row
            remap[rng.random(len(remap)) < 0.01] = -7
        lens = rng.integers(0, 2 * avg + 1, size=T * B)
        off = np.concatenate([[0], np.cumsum(lens)])
        N = int(off[-1])
        idx = np.concatenate([rng.integers(0, logical[t], size=int(off[(t + 1) * B] - off[t * B])) for t in range(T)])
        for what in ("good", "indices", "offsets", "last", "first"):
            i2, o2 = idx.copy(), off.copy()
            if what == "indices" and N:
                where = rng.random(N) < 0.05
                i2[where] = rng.choice([-1, -2, 1000, 1 << 30], size=int(where.sum()))
            elif what == "offsets":
                where = rng.random(len(o2)) < 0.02
                o2[where] += rng.integers(-50, 50, size=int(where.sum()))
            elif what == "last":
                o2[-1] += 3
            elif what == "first":
                o2[0] = N + 5 if n % 2 else min(3, N)
            if what != "good" and n >= len(SHAPES) - 2 and what != "offsets":
                continue
            args = (cu(rows), cu(i2, dtype), cu(o2, dtype), mode)
            more = (cu(logical), None, None) if remap is None else (cu(logical), cu(remap, mapped), cu(remap_offsets))
            w0, w1 = torch.full((1,), 77, device="cuda"), torch.full((1,), 77, device="cuda")
            wi, wo = one_after_the_other(ops, *args, w0, *more)
            for _ in range(2):  # the library's counters are zero again after the first
                before = [t.clone() for t in args[1:3]]
                gi, go = ops.check_remap_indices(*args, w1, None, *more)
                tag = f"T={T} B={B} {what} mapped={mapped} {dtype}"
                assert torch.equal(go, wo), tag
                start = int(wo[0])
                assert torch.equal(gi[start:], wi[start:]), tag
                assert torch.equal(w0, w1), (tag, int(w0), int(w1))
                assert all(torch.equal(a, b) for a, b in zip(before, args[1:3])), tag


#                               one launch at most, two launches, the running maxima made by a launch of their own
@pytest.mark.parametrize("bags", [(512, 3000, 4096), (9000, 6000, 20_000), (8_600_000, 8_500_000, 5000)])
def test_streams_and_captured_calls(ops, bags):
    """Calls of one thread on several streams and from a graph that is replayed beside them, each with
    offsets and indices of its own, leave what each of them leaves alone, and nothing for a later call."""
    rng = np.random.default_rng(bags[0])
    cu = lambda a: torch.from_numpy(a).cuda()
    T = 8
    calls, want = [], []
    for n, total in enumerate(bags):
        lens = rng.integers(0, 2 * (n + 1) + 1, size=total)
        off = np.concatenate([[0], np.cumsum(lens)])
        idx = rng.integers(0, 100, size=int(off[-1]))
        idx[rng.choice(len(idx), 37 + n, replace=False)] = 100
        broken = rng.random(total + 1) < 0.01
        off[broken] += rng.integers(-20, 20, size=int(broken.sum()))  # what the running maximum repairs
        rows = torch.full((T,), 100, dtype=torch.int64, device="cuda")
        calls.append((rows, cu(idx), cu(off), 1))
        w = torch.zeros(1, dtype=torch.int64, device="cuda")
        want.append((*one_after_the_other(ops, *calls[-1], w, None, None, None), w))
    failures = []

    def turns():  # a thread of its own: it has called nothing before
        try:
            streams = [torch.cuda.Stream() for _ in bags]
            warnings = [torch.full((1,), -1, dtype=torch.int64, device="cuda") for _ in bags]
            call = lambda k: ops.check_remap_indices(*calls[k], warnings[k])
            torch.cuda.synchronize()
            for k, s in enumerate(streams):
                with torch.cuda.stream(s):
                    call(k)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=streams[2]):
                captured = call(2)
            for turn in range(20):
                outs = []
                for k, s in enumerate(streams[:2]):
                    with torch.cuda.stream(s):
                        outs.append(call(k))
                graph.replay()
                torch.cuda.synchronize()
                for k, o in enumerate(outs + [captured]):
                    start = int(want[k][1][0])
                    assert torch.equal(o[1], want[k][1]), (turn, k)
                    assert torch.equal(o[0][start:], want[k][0][start:]), (turn, k)
                    assert int(warnings[k]) == int(want[k][2]), (turn, k)
                for w in warnings:
                    w.fill_(-1)
                captured[1].fill_(0)
                torch.cuda.synchronize()
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    t = threading.Thread(target=turns)
    t.start()
    t.join()
    assert not failures, failures


def order_preserving(rng, rows, keep):
    """A mapping of `rows` logical rows that numbers the kept ones in order, and how many it keeps."""
    kept = rng.random(rows) < keep
    return np.where(kept, np.cumsum(kept) - 1, -1), int(kept.sum())


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("mapped", [torch.int32, torch.int64])
def test_compact_mappings(ops, mapped, dtype):
    """Tables with order-preserving mappings (around the 32 rows of a record: none kept, all kept, some), others and
    none side by side: the compact form answers as the arrays do."""
    rng = np.random.default_rng(8)
    cu = lambda a, dt=torch.int64: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt)
    maps, rows, logical = [], [], []
    for n in (1, 31, 32, 33, 64, 255, 1000, 8191, 8193, 40_000):
        for keep in (0.0, 0.5, 1.0):
            m, kept = order_preserving(rng, n, keep)
            maps.append(m)
            rows.append(max(kept - (n % 2), 0))  # odd ones: the last kept row lies outside the table
            logical.append(n)
    for n in (50, 300):
        maps += [rng.integers(-1, n, size=n), np.zeros(0, np.int64)]
        rows += [n, n]
        logical += [n, n]
    T = len(maps)
    rows, logical = cu(rows), cu(logical)
    offs = cu(np.concatenate([[0], np.cumsum([len(m) for m in maps])]))
    remap = cu(np.concatenate(maps), mapped)
    ranks = ops.RankRecords(remap, offs)
    assert ranks.handle is not None
    for B, avg in ((1, 40), (300, 7)):
        lens = rng.integers(0, 2 * avg, size=T * B)
        off = np.concatenate([[0], np.cumsum(lens)])
        idx = rng.integers(-2, int(logical.max()) + 40, size=int(off[-1]))
        idx = np.where(rng.random(len(idx)) < 0.9, idx % np.repeat(logical.cpu().numpy(), lens.reshape(T, B).sum(1)), idx)
        for mode in (1, 2):
            args = (rows, cu(idx, dtype), cu(off, dtype), mode)
            w0, w1 = torch.zeros(1, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
            want = one_after_the_other(ops, *args, w0, logical, remap, offs)
            got = ops.check_remap_indices(*args, w1, None, logical, remap, offs, ranks)
            assert all(torch.equal(g, w) for g, w in zip(got, want)) and torch.equal(w0, w1), (B, mode)


@pytest.mark.parametrize("edited", [False, True])
def test_module_follows_its_mappings(edited):
    """A pruned module's forward after its mappings have been edited in place, set anew, and in copies and saved
    modules; and a captured check that was handed the compact form of earlier contents."""
    import copy
    import io

    from fbgemm_amd import module as M
    rng = np.random.default_rng(2)
    rows, D, B = 400, 32, 64
    m = M.IntNBitTableBatchedEmbeddingBagsCodegen([("", rows, D, M.SparseType.INT8, M.EmbeddingLocation.DEVICE)] * 2,
                                                  bounds_check_mode=M.BoundsCheckMode.WARNING, output_dtype=M.SparseType.FP32)
    m.fill_random_weights()
    for _, sb in m.split_embedding_weights():
        sb.view(torch.float16).copy_(torch.rand(rows, 2, device="cuda").half())
    mapping = lambda: torch.from_numpy(order_preserving(rng, 2 * rows, 0.4)[0]).cuda()
    off = torch.arange(2 * B + 1, dtype=torch.int64, device="cuda") * 5
    idx = torch.from_numpy(rng.integers(0, 2 * rows, size=10 * B)).cuda()
    plain = copy.deepcopy(m)

    def check(mod, maps):
        flat = torch.cat(maps).to(idx.device)
        where = torch.cat([idx[:5 * B], idx[5 * B:] + 2 * rows])
        want = plain(flat[where].to(torch.int64), off)
        for _ in range(3):
            assert torch.equal(mod(idx, off), want)

    maps = [mapping(), mapping()]
    m.set_index_remappings(maps)
    check(m, maps)
    maps = [mapping(), mapping()]
    m.index_remappings_array.copy_(torch.cat(maps))
    check(m, maps)
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    for other in (copy.deepcopy(m), torch.load(buf, weights_only=False)):
        check(other, maps)
        changed = [maps[1], maps[0]]
        other.index_remappings_array.copy_(torch.cat(changed))
        check(other, changed)
        check(m, maps)
    # a graph reads the array: it sees what is written there between its replays; compact forms of the contents at the
    # capture and of those before the last edit, which a capture right behind that edit leaves aside
    graph, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        ranks = [M.ops.RankRecords(m._feature_remap_array, m._feature_remap_offsets)]
        call = lambda: M.ops.check_remap_indices(m.rows_per_table, idx, off, 1, m.bounds_check_warning, None, m.original_rows_per_table,
                                                 m._feature_remap_array, m._feature_remap_offsets, ranks[0])
        call()
        if edited:
            maps = [mapping(), mapping()]
            m.index_remappings_array.copy_(torch.cat(maps))
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            out, _ = call()
    for maps in ([mapping(), mapping()], [mapping(), mapping()]):
        m.index_remappings_array.copy_(torch.cat(maps))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        flat = torch.cat(maps)
        assert torch.equal(out, torch.where(flat < rows, flat, 0)[torch.cat([idx[:5 * B], idx[5 * B:] + 2 * rows])])
        check(m, maps)


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("write", ["data", "dlpack", "replay"])
def test_module_sees_writes_without_a_version(write, mode):
    """What writes the mappings without raising the tensor's version (``.data``, another view of the memory, a graph that
    refreshes them, as collectives and kernels of the caller's do too) is seen by the next checked forward, also after
    forwards on unchanged mappings."""
    from fbgemm_amd import module as M
    rng = np.random.default_rng(5)
    rows, D, B = 300, 32, 64
    m = M.IntNBitTableBatchedEmbeddingBagsCodegen([("", rows, D, M.SparseType.INT8, M.EmbeddingLocation.DEVICE)] * 2,
                                                  bounds_check_mode=M.BoundsCheckMode(mode), output_dtype=M.SparseType.FP32)
    m.fill_random_weights()
    for _, sb in m.split_embedding_weights():
        sb.view(torch.float16).copy_(torch.rand(rows, 2, device="cuda").half())
    off = torch.arange(2 * B + 1, dtype=torch.int64, device="cuda") * 5
    idx = torch.from_numpy(rng.integers(0, 2 * rows, size=10 * B)).cuda()
    where = torch.cat([idx[:5 * B], idx[5 * B:] + 2 * rows])
    plain = M.IntNBitTableBatchedEmbeddingBagsCodegen([("", rows, D, M.SparseType.INT8, M.EmbeddingLocation.DEVICE)] * 2,
                                                      bounds_check_mode=M.BoundsCheckMode(mode), output_dtype=M.SparseType.FP32)
    plain.initialize_weights()
    plain.weights_dev.copy_(m.weights_dev)
    maps = lambda: [torch.from_numpy(order_preserving(rng, 2 * rows, 0.4)[0]).cuda() for _ in range(2)]
    first = maps()
    m.set_index_remappings(first)
    array = m.index_remappings_array
    fresh = torch.cat(first).to(array.dtype)
    if write == "replay":
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            array.copy_(fresh)
        torch.cuda.synchronize()
    for turn in range(3):
        if turn:
            fresh.copy_(torch.cat(maps()))
            version = array._version
            {"data": lambda: array.data.copy_(fresh), "dlpack": lambda: torch.from_dlpack(array).copy_(fresh),
             "replay": lambda: graph.replay()}[write]()
            assert array._version == version
        for _ in range(3):
            assert torch.equal(m(idx, off), plain(fresh[where].to(torch.int64), off)), turn
