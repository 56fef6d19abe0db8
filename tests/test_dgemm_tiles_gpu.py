"""The direct-LDS DGEMM tiles at their edges: every tile shape of the automatic
choice against the register-staged kernel (tile configuration 1), which sums
k in the same order, so the results must be equal bit for bit; NaN in the
padding of the operands must not leak and nothing outside C may change."""
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k) by the tile the automatic choice takes
SHAPES = [
    (1, 1, 1), (1, 33, 16), (33, 1, 17), (31, 32, 15), (100, 97, 129), (33, 65, 1),   # 32 x 32
    (627, 2133, 101),                                                                  # 64 x 32
    (1009, 1023, 2001), (1283, 1391, 229), (2671, 967, 45),                            # 64 x 64, one to three per CU
    (1985, 2001, 333), (2417, 4007, 4001),                                             # 64 x 128
    (3967, 3969, 3001),                                                                # 128 x 128
]


def tensor(rows, cols, pad, seed):
    """Column-major rows x cols matrix with `pad` NaN rows below it, as a (cols, rows + pad) tensor."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.full((cols, rows + pad), float("nan"), dtype=torch.float64, device="cuda")
    t[:, :rows] = torch.rand((cols, rows), dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    return t


@pytest.mark.parametrize("pads", [(0, 0, 0), (1, 3, 1), (2, 1, 2)])
@pytest.mark.parametrize("ta,tb", [("T", "N"), ("N", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tiles_equal_register_staged_kernel(handle, m, n, k, ta, tb, pads):
    import torch
    import cosma_amd as ca
    A = tensor(*((m, k) if ta == "N" else (k, m)), pads[0], 1)
    B = tensor(*((k, n) if tb == "N" else (n, k)), pads[1], 2)
    C0 = tensor(m, n, pads[2], 3)
    out = []
    try:
        for cfg in (0, 1):
            ca.set_dgemm_tuning(cfg, 0)
            for beta in (0.0, -0.5):
                C = C0.clone()
                if beta == 0.0:
                    C[:, :m] = float("nan")
                handle.dgemm(ta, tb, m, n, k, 1.25, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), beta,
                             C.data_ptr(), C.stride(0))
                torch.cuda.synchronize()
                assert torch.isnan(C[:, m:]).all()
                out.append(C[:, :m].clone())
    finally:
        ca.set_dgemm_tuning(0, 0)
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3])
    assert not torch.isnan(out[0]).any() and not torch.isnan(out[1]).any()


def test_odd_extent_reads_nothing_behind_the_operand(handle):
    """The last element of an odd row-contiguous operand is the last of its
    allocation: with NaN right behind it (and in the 16-byte load's reach)
    the result stays finite and equals the product of a copy elsewhere."""
    import torch
    m, n, k = 65, 33, 48
    g = torch.Generator(device="cuda").manual_seed(5)
    buf = torch.full((m * k + 64,), float("nan"), dtype=torch.float64, device="cuda")
    buf[:m * k] = torch.rand(m * k, dtype=torch.float64, device="cuda", generator=g)
    B = torch.rand((n, k), dtype=torch.float64, device="cuda", generator=g)
    copy = torch.zeros_like(buf)
    copy[:m * k] = buf[:m * k]
    res = []
    for A in (buf, copy):
        C = torch.zeros((n, m), dtype=torch.float64, device="cuda")
        handle.dgemm("N", "N", m, n, k, 1.0, A.data_ptr(), m, B.data_ptr(), k, 0.0, C.data_ptr(), m)
        torch.cuda.synchronize()
        res.append(C)
    assert torch.isfinite(res[0]).all() and torch.equal(res[0], res[1])
