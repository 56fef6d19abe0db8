"""Block copies at the lines between their forms: narrow blocks as a list or in
row windows.  Integer-valued entries and dyadic factors make every result
exact, so all comparisons are for equality; the padding of the operands is NaN
and dst's must stay so."""
import pytest

from test_transform_tiles_gpu import matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.5, 0.0), (2.0, 0.5)])
@pytest.mark.parametrize("rows,cols,pad_src,pad_dst,off_src,off_dst", [
    (1, 16511, 0, 1, 0, 0), (1, 16512, 1, 0, 0, 1), (3, 16767, 0, 0, 1, 0), (3, 16769, 0, 0, 0, 1),   # narrow: windows, list
    (48, 22527, 1, 0, 0, 0), (48, 22528, 0, 1, 0, 0), (49, 22656, 0, 0, 0, 1), (64, 24576, 0, 1, 0, 0), (65, 24704, 0, 0, 1, 1),
    (2, 1, 0, 0, 0, 0), (255, 1, 0, 3, 0, 1), (511, 3, 1, 1, 0, 0), (1040, 3, 0, 1, 0, 0),            # waves without rows
])
def test_copy_forms_at_their_lines(handle, rows, cols, pad_src, pad_dst, off_src, off_dst, alpha, beta):
    import torch
    src, dst = matrix(rows, cols, pad_src, off_src, 1), matrix(rows, cols, pad_dst, off_dst, 2)
    want = alpha * src[:, :rows] + (beta * dst[:, :rows] if beta else 0.0)
    if not beta:
        dst[:, :rows] = float("nan")   # must not be read
    handle.block_transform("N", rows, cols, alpha, src.data_ptr(), src.stride(0), beta, dst.data_ptr(), dst.stride(0))
    torch.cuda.synchronize()
    assert torch.equal(dst[:, :rows], want)
    assert torch.isnan(dst[:, rows:]).all()
