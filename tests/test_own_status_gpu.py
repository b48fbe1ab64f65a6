"""Calls that wait for their result share a status block per thread that is clear between them: a
rejected call must not be seen by the next one, nor a call that failed on its way."""
import threading
import time

import numpy as np
import pytest

import helpers as H
from helpers import INT8

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("no_bag", [False, True])
def test_rejected_accepted_in_turn(no_bag):
    assert torch.cuda.is_available(), "these tests need the GPU"
    from fbgemm_amd import ops
    rng = np.random.default_rng(3)
    D, rows, nb = 32, 50, 20
    table, _ = H.make_table(rng, INT8, rows, D, True)
    table = torch.from_numpy(table).cuda()
    good = torch.from_numpy(rng.integers(0, rows, size=nb).astype(np.int64)).cuda()
    bad = good.clone()
    bad[7] = rows
    off = torch.arange(nb + 1, dtype=torch.int32, device="cuda")
    kern = ops.generate_embedding_spmdm_with_strides(ops.INT8, D, False, False, no_bag=no_bag)
    failures = []

    def turns():
        try:
            out = torch.empty(nb, D, device="cuda")
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    assert kern(nb, nb, rows, table, good, off, None, out) is True
                    assert kern(nb, nb, rows, table, bad, off, None, out) is False
                    with pytest.raises(RuntimeError):  # refused on the host, after the block was handed out
                        kern(nb, nb, -1, table, good, off, None, out)
                    assert kern(0, 0, rows, table, good, off, None, out) is True
                    assert kern(0, nb, rows, table, good, off, None, out) is no_bag
                torch.cuda.current_stream().synchronize()
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=turns) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    turns()
    assert not failures, failures


def single_table_calls():
    """A good and a bad launch of a single-table lookup into a status block, and the same as waiting calls."""
    assert torch.cuda.is_available(), "these tests need the GPU"
    from fbgemm_amd import ops
    rng = np.random.default_rng(9)
    D, rows, nb = 32, 50, 20
    table, _ = H.make_table(rng, INT8, rows, D, True)
    table = torch.from_numpy(table).cuda()
    good = torch.from_numpy(rng.integers(0, rows, size=nb).astype(np.int64)).cuda()
    bad = good.clone()
    bad[7] = rows
    off = torch.arange(nb + 1, dtype=torch.int32, device="cuda")
    out = torch.empty(nb, D, device="cuda")
    kern = ops.generate_embedding_spmdm_with_strides(ops.INT8, D, False, False)
    return ops, lambda idx, st=None, bags=nb: kern(bags, nb, rows, table, idx, off, None, out, status=st), good, bad


def test_own_block_cleared_by_its_user():
    """status_clear on the block of status_begin clears it and leaves what makes it report."""
    ops, call, good, bad = single_table_calls()
    from fbgemm_amd import _lib
    for reported in (False, True):
        st = ops._OwnStatus()
        if reported:
            call(bad, st)
        ops.check(_lib.lib().fbgemm_amd_status_clear(st.ptr, ops._stream()))
        assert st.read() == (0, -1)
        assert call(good) is True and call(bad) is False and call(good) is True
        st = ops._OwnStatus()
        ops.check(_lib.lib().fbgemm_amd_status_clear(st.ptr, ops._stream()))
        call(bad, st)
        assert st.read() == (ops.ERR_INDEX_OUT_OF_RANGE, 7)
        assert call(good) is True and call(bad) is False


def test_no_bags_but_indices():
    """No bags but indices is an error that is known without a kernel; it is reported like any other."""
    ops, call, good, bad = single_table_calls()
    for _ in range(2):
        st = ops._OwnStatus()
        call(good, st, bags=0)
        assert st.read() == (ops.ERR_LENGTH_MISMATCH, -1)
        assert call(good) is True and call(bad) is False
    st = ops.Status()
    call(bad, st)
    call(good, st, bags=0)
    assert st.read() == (ops.ERR_INDEX_OUT_OF_RANGE | ops.ERR_LENGTH_MISMATCH, 7)


def test_first_call_of_a_thread_beside_a_capture(oracle):
    """A thread's first waiting call makes its status block. That waits for nothing but itself, also while
    another thread captures (in the mode that lets other threads wait); and a block that an ended thread
    leaves is taken over the same way."""
    assert torch.cuda.is_available(), "these tests need the GPU"
    from fbgemm_amd import ops
    from test_tbe_gpu import build_weights
    rng = np.random.default_rng(4)
    D, rows, B = 32, 50, 40
    weights, wo, _ = build_weights(rng, [(rows, D, INT8)], 16)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    meta = (cu(weights), torch.zeros(0, dtype=torch.uint8, device="cuda"), cu(np.zeros(1, np.int32)), cu(wo),
            cu(np.array([INT8], np.uint8)), cu(np.array([0, D], np.int32)))
    idx, off = cu(rng.integers(0, rows, size=3 * B).astype(np.int64)), cu(np.arange(B + 1, dtype=np.int64) * 3)
    call = lambda: ops.int_nbit_split_embedding_codegen_lookup_function(
        *meta, D, 0, 0, D, 0, 0, idx, off, ops.POOL_NONE, None, ops.FP32, row_alignment=16)
    want = call()
    torch.cuda.synchronize()
    got, failures = [], []

    def first():
        try:
            with torch.cuda.stream(streams.pop()):
                got.append(call())
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    for turn in range(2):  # a block of its own, then perhaps the one the first thread left
        streams = [torch.cuda.Stream() for _ in range(2)]
        x = torch.ones(100, device="cuda")
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.Stream(), capture_error_mode="thread_local"):
            y = x * 2
            threads = [threading.Thread(target=first) for _ in range(2)]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
            z = y + 1
        assert not failures, failures
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert bool((z == 3).all())
            x.fill_(1)
        assert len(got) == 2 * (turn + 1) and all(torch.equal(g, want) for g in got)


@pytest.mark.parametrize("products", [0, 40])
def test_waiting_call_behind_other_work(products):
    """A waiting call returns when its stream has come to its end, also where that takes longer than the host
    watches for it (40 products of 4096 x 4096 floats are tens of milliseconds): an event recorded before the call is
    over, and what the last of the work before it wrote is there for a kernel and for a copy of another stream."""
    ops, call, good, bad = single_table_calls()
    x = torch.ones(4096, 4096, device="cuda") / 4096
    product, y, other = torch.empty_like(x), torch.zeros_like(x), torch.cuda.Stream()
    host = torch.empty(x.shape, pin_memory=True)
    torch.cuda.synchronize()
    for turn in range(1, 4):
        for _ in range(products):
            torch.mm(x, x, out=product)
        y.fill_(turn)
        before = torch.cuda.Event()
        before.record()
        assert call(good) is True
        # the event's signal is written before the word the call waits for, by another unit: far less than a product apart
        until = time.perf_counter() + 1e-4
        while not before.query() and time.perf_counter() < until:
            pass
        assert before.query()
        with torch.cuda.stream(other):
            host.copy_(y, non_blocking=True)
            assert bool((y == turn).all())
            other.synchronize()
        assert bool((host == turn).all())
        assert call(bad) is False
