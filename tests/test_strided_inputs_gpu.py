"""Operators whose inputs are strided vectors: the same as for contiguous ones. Sizes are such that the
copies of two inputs would fit the same memory, which the allocator hands out again as soon as one is
given up."""
import numpy as np
import pytest

import helpers as H
import test_tbe_gpu as TB
from helpers import FP16, INT4

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    assert torch.cuda.is_available(), "these tests need the GPU"
    import fbgemm_amd.ops as o
    return o


def strided(t):
    out = torch.zeros(3 * t.numel(), dtype=t.dtype, device=t.device)
    out[::3] = t
    return out[::3]


T, B, D, ROWS = 3, 40, 64, 300


def inputs():
    rng = np.random.default_rng(1)
    weights, wo, _ = TB.build_weights(rng, [(ROWS, D, INT4)] * T, 16)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    meta = (cu(weights), torch.zeros(0, dtype=torch.uint8, device="cuda"), cu(np.zeros(T, np.int32)), cu(wo), cu(np.full(T, INT4, np.uint8)),
            cu(np.arange(T + 1, dtype=np.int32) * D))
    offsets = cu(np.arange(T * B + 1, dtype=np.int64))  # one entry per bag: as many indices as bags
    indices = cu(rng.integers(0, ROWS, size=T * B))
    return meta, indices, offsets, cu(rng.normal(size=T * B).astype(np.float32))


@pytest.mark.parametrize("pooling,weighted", [(0, False), (0, True), (1, False), (1, True), (2, False)])
def test_lookup(ops, pooling, weighted):
    meta, indices, offsets, weights = inputs()
    call = lambda i, o, w: ops.int_nbit_split_embedding_codegen_lookup_function(
        *meta, T * D, 0, D, 0, 0, 0, i, o, pooling, w, FP16, row_alignment=16)
    want = call(indices, offsets, weights if weighted else None)
    for _ in range(3):
        got = call(strided(indices), strided(offsets), strided(weights) if weighted else None)
        H.assert_same_bits(got.cpu().view(torch.int16).numpy().view(np.uint16), want.cpu().view(torch.int16).numpy().view(np.uint16), "strided")


def test_index_operators(ops):
    _, indices, offsets, weights = inputs()
    rng = np.random.default_rng(2)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    remap = cu(rng.integers(-1, ROWS, size=T * ROWS).astype(np.int32))
    remap_offsets = cu(np.arange(T + 1, dtype=np.int64) * ROWS)
    tables = cu(np.repeat(np.arange(T, dtype=np.int32), B))
    for _ in range(3):
        assert torch.equal(ops.pruned_array_lookup(strided(indices), strided(offsets), strided(remap), strided(remap_offsets)),
                           ops.pruned_array_lookup(indices, offsets, remap, remap_offsets))
        assert torch.equal(ops.pruned_array_lookup_from_row_idx(strided(indices), strided(tables), strided(remap), strided(remap_offsets)),
                           ops.pruned_array_lookup_from_row_idx(indices, tables, remap, remap_offsets))
        got = ops.compressed_indices_remap(strided(indices), strided(remap), strided(offsets), strided(weights))
        want = ops.compressed_indices_remap(indices, remap, offsets, weights)
        n = int(want[1][-1])
        assert torch.equal(got[1], want[1]) and all(torch.equal(got[k][:n], want[k][:n]) for k in (0, 2))


def test_inplace_update(ops):
    meta, _, _, _ = inputs()
    rng = np.random.default_rng(3)
    cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    row = ops.padded_row_size_in_bytes(D, INT4, 16)
    n = T * B
    rows = cu(rng.permutation(ROWS)[:n].astype(np.int64))
    tables = cu(rng.integers(0, T, size=n).astype(np.int32))
    offs = cu(np.arange(n, dtype=np.int64) * row)
    data = cu(rng.integers(0, 256, size=n * row, dtype=np.uint8))
    a, b = meta[0].clone(), meta[0].clone()
    ops.emb_inplace_update(a, *meta[1:], data, tables, rows, offs, row_alignment=16)
    ops.emb_inplace_update(b, *meta[1:], strided(data), strided(tables), strided(rows), strided(offs), row_alignment=16)
    assert torch.equal(a, b) and not torch.equal(a, meta[0])
