"""The forms of the block transform at their edges: streamed and cached copies,
narrow blocks, large transposes in shifted and in whole-line windows, and the
block lists of a layout multiply.  Integer-valued entries and dyadic factors
make every result exact, so all comparisons are for equality; the padding of
the operands is NaN and dst's must stay so."""
import pytest

pytestmark = pytest.mark.gpu


def matrix(rows, cols, pad, offset, seed):
    """Column-major rows x cols view with `pad` NaN rows below, `offset` elements into its allocation."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    ld = rows + pad
    buf = torch.full((cols * ld + offset,), float("nan"), dtype=torch.float64, device="cuda")
    full = buf[offset:].view(cols, ld)
    full[:, :rows] = torch.randint(-1000, 1000, (cols, rows), device="cuda", generator=g).double()
    return full


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.5, 0.0), (2.0, 0.5)])
@pytest.mark.parametrize("op,rows,cols,pad_src,pad_dst,off_src,off_dst", [
    ("N", 1, 1, 0, 0, 0, 0), ("N", 1023, 70, 1, 0, 1, 0), ("N", 1025, 65, 0, 3, 0, 1),   # cached, without and with shift
    ("N", 4099, 4097, 0, 2, 1, 1), ("N", 4096, 4096, 0, 0, 0, 0),                        # streamed
    ("N", 1, 1048577, 0, 1, 0, 1), ("N", 255, 4200, 2, 0, 0, 1), ("N", 256, 4096, 0, 0, 0, 0),   # narrow
    ("N", 1, (1 << 23) + 1, 0, 1, 0, 0), ("N", 3, (1 << 24) - 1, 1, 0, 1, 1),             # narrow, cut in pieces
    ("T", 1024, 19532, 1, 0, 0, 1), ("T", 5001, 4003, 0, 1, 1, 0), ("T", 19532, 1024, 0, 0, 0, 0),   # shifted
    ("T", 4096, 16384, 0, 0, 0, 0), ("T", 4111, 16401, 15, 1, 0, 0),                    # whole lines
    ("T", 2601, 8501, 1, 0, 1, 0), ("T", 1040, 30802, 0, 0, 0, 0), ("T", 1040, 30702, 0, 0, 0, 0),   # part tiles; dst in whole lines
])
def test_transform_forms(handle, op, rows, cols, pad_src, pad_dst, off_src, off_dst, alpha, beta):
    import torch
    src = matrix(*((rows, cols) if op == "N" else (cols, rows)), pad_src, off_src, 1)
    dst = matrix(rows, cols, pad_dst, off_dst, 2)
    x = src[:, :rows] if op == "N" else src[:, :cols].t()
    want = alpha * x + (beta * dst[:, :rows] if beta else 0.0)
    if not beta:
        dst[:, :rows] = float("nan")   # must not be read
    handle.block_transform(op, rows, cols, alpha, src.data_ptr(), src.stride(0), beta, dst.data_ptr(), dst.stride(0))
    torch.cuda.synchronize()
    assert torch.equal(dst[:, :rows], want)
    assert torch.isnan(dst[:, rows:]).all()


def cut(t, rows, cols, size):
    """Blocks of a column-major (cols, ld) tensor, each in an allocation of its own with an odd leading dimension."""
    import torch
    out = []
    for c in range(0, cols, size):
        for r in range(0, rows, size):
            nr, nc = min(size, rows - r), min(size, cols - c)
            b = torch.full((nc, nr + 1 - nr % 2 + 1), float("nan"), dtype=torch.float64, device="cuda")
            b[:, :nr] = t[c:c + nc, r:r + nr]
            out.append((b, r, c, nr, nc))
    return out


@pytest.mark.parametrize("ta,tb,m,n,k,size", [("N", "N", 601, 333, 257, 67), ("T", "N", 100, 95, 71, 9),
                                              ("N", "T", 300, 1200, 40, 300), ("T", "T", 17, 40, 33, 1)])
def test_layout_of_many_device_blocks(handle, ta, tb, m, n, k, size):
    """More blocks than one launch takes, down to single elements, against the product of the whole matrices."""
    import torch
    A = matrix(*((m, k) if ta == "N" else (k, m)), 0, 0, 3)
    B = matrix(*((k, n) if tb == "N" else (n, k)), 0, 0, 4)
    C0 = matrix(m, n, 0, 0, 5)
    cuts = [cut(A, A.shape[1], A.shape[0], size), cut(B, B.shape[1], B.shape[0], size), cut(C0, m, n, size)]
    torch.cuda.synchronize()
    a, b, c = ([(t.data_ptr(), t.stride(0), r, col, nr, nc) for t, r, col, nr, nc in blk] for blk in cuts)
    handle.dgemm_layout(ta, tb, m, n, k, 2.0, a, b, 0.5, c)
    want = C0.clone()
    handle.dgemm(ta, tb, m, n, k, 2.0, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), 0.5, want.data_ptr(), m)
    torch.cuda.synchronize()
    for t, r, col, nr, nc in cuts[2]:
        assert torch.equal(t[:, :nr], want[col:col + nc, r:r + nr])
        assert torch.isnan(t[:, nr:]).all()
