"""Block copies at the lines between their forms: narrow blocks as a list or in
row windows, cached and streamed loads, with and without reading dst, from
matrices and from the block lists of a layout multiply.  Integer-valued entries
and dyadic factors make every result exact, so all comparisons are for
equality; the padding of the operands is NaN and dst's must stay so."""
import pytest

from test_transform_tiles_gpu import matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.5, 0.0), (2.0, 0.5)])
@pytest.mark.parametrize("rows,cols,pad_src,pad_dst,off_src,off_dst", [
    (1, 16511, 0, 1, 0, 0), (1, 16512, 1, 0, 0, 1), (3, 16767, 0, 0, 1, 0), (3, 16769, 0, 0, 0, 1),   # narrow: windows, list
    (48, 22527, 1, 0, 0, 0), (48, 22528, 0, 1, 0, 0), (49, 22656, 0, 0, 0, 1), (64, 24576, 0, 1, 0, 0), (65, 24704, 0, 0, 1, 1),
    (500, 41999, 0, 1, 0, 0), (1025, 20489, 1, 0, 0, 1), (300, 70000, 0, 0, 0, 0),                    # 21 * 10^6 elements
    (383, 88773, 0, 0, 1, 0), (384, 88542, 1, 1, 0, 0), (2000, 17001, 0, 1, 0, 1), (24, 1416667, 0, 0, 0, 1),   # 34
    (380, 100000, 0, 0, 1, 0), (380, 100001, 1, 1, 0, 0), (384, 100000, 0, 0, 0, 0), (384, 100001, 1, 0, 0, 0), (2000, 19001, 0, 1, 0, 1), (24, 1583334, 0, 0, 0, 1),   # 38
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


@pytest.mark.parametrize("m,n,beta", [(4584, 4584, 0.5), (5832, 5832, 0.5), (6169, 6169, 0.0), (60, 640000, 0.0)])
def test_block_lists_beyond_the_cache(handle, m, n, beta):
    """C past 21, 34 and 38 * 10^6 elements in device blocks of a layout multiply; the last one's lines are shared."""
    import torch
    k, size = 2, (m + 2) // 3
    A, B, C0 = matrix(m, k, 0, 0, 3), matrix(k, n, 0, 0, 4), matrix(m, n, 0, 0, 5)
    cuts = []
    for t, rows, cols in ((A, m, k), (B, k, n), (C0, m, n)):
        cuts.append([])
        for r in range(0, rows, size):
            for c in range(0, cols, (n + 2) // 3):
                b = t[c:c + (n + 2) // 3, r:r + size].contiguous()
                cuts[-1].append((b, r, c))
    blocks = [[(b.data_ptr(), b.shape[1], r, c, b.shape[1], b.shape[0]) for b, r, c in blk] for blk in cuts]
    torch.cuda.synchronize()
    handle.dgemm_layout("N", "N", m, n, k, 2.0, blocks[0], blocks[1], beta, blocks[2])
    want = 2.0 * (B[:, :1] * A[:1] + B[:, 1:] * A[1:]) + (beta * C0 if beta else 0.0)
    for b, r, c in cuts[2]:
        assert torch.equal(b, want[c:c + b.shape[0], r:r + b.shape[1]])
