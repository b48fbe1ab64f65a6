"""Caffe2-style lengths: the prefix sum over runs of several workgroups, around their sizes."""
import numpy as np
import pytest

import helpers as H
import test_spmdm_gpu as S
from helpers import FP32, INT8

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("bags", [1, 1023, 1024, 1025, 9 * 1024 + 1, 256 * 1024, 256 * 1024 + 1, 3 * 256 * 1024 + 77])
def test_lengths(oracle, bags, dtype):
    from fbgemm_amd import ops
    rng = np.random.default_rng(bags)
    rows, D = 64, 4
    table, _ = H.make_table(rng, INT8, rows, D, True)
    lens = rng.integers(0, 4, size=bags).astype(dtype)
    idx = rng.integers(0, rows, size=int(lens.sum())).astype(np.int32)
    assert S.check_case(ops, oracle, ty=INT8, D=D, table=table, idx=idx, off_or_len=lens, w=None, normalize=False, out_ty=FP32,
                        positional=False, use_offsets=False, output_stride=-1, input_stride=-1, sbl=True, data_size=rows,
                        output_size=bags, what=f"{bags} lengths")


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("bags", [1, 2, 64, 65, 256, 257, 1024, 1025, 4095, 4096, 4097])
def test_lengths_added_up_by_the_burst_kernel(oracle, bags, waves, dtype):
    """Around the loads in flight per thread of either workgroup size and the most bags it is done for, over two windows of columns;
    a sum of lengths that is not the number of indices is reported."""
    import fbgemm_amd
    from fbgemm_amd import ops
    rng = np.random.default_rng(bags * waves)
    rows, D = 64, 300
    table, _ = H.make_table(rng, INT8, rows, D, True)
    lens = rng.integers(0, 4, size=bags).astype(dtype)
    lens[-1] += 1
    idx = rng.integers(0, rows, size=int(lens.sum())).astype(np.int32)
    lib = fbgemm_amd.lib()
    lib.fbgemm_amd_set_burst(waves)
    try:
        for cut, fine in ((0, True), (1, False)):
            assert S.check_case(ops, oracle, ty=INT8, D=D, table=table, idx=idx[:len(idx) - cut], off_or_len=lens, w=None, normalize=True,
                                out_ty=FP32, positional=False, use_offsets=False, output_stride=-1, input_stride=-1, sbl=True, data_size=rows,
                                output_size=bags, what=f"{bags} lengths, {waves} waves") == fine
    finally:
        lib.fbgemm_amd_set_burst(-1)
