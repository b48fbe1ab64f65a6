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
