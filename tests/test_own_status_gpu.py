"""Calls that wait for their result share a status block per thread that is clear between them: a
rejected call must not be seen by the next one, nor a call that failed on its way."""
import threading

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
