"""Host products with the default tiles, whose resident schedule cuts them finer:
extents around the cuts' thresholds and uneven last tiles, against the
device-resident product of the same operands.  Both are within gemm_bound(k) of
the exact product (k-panels only add roundings of C that the bound covers)."""
import pytest

from helpers import gemm_bound

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pin", [True, False])
@pytest.mark.parametrize("ta,tb,m,n,k,beta", [
    ("N", "N", 767, 768, 1791, 0.0), ("T", "N", 1792, 1793, 769, 0.5), ("N", "T", 2815, 1025, 3333, -1.0),
    ("T", "T", 3841, 2817, 1300, 0.0), ("T", "N", 600, 500, 6001, 0.5),   # the last: C too small to be cut
])
def test_default_tiles(handle, ta, tb, m, n, k, beta, pin):
    import torch
    g = torch.Generator(device="cuda").manual_seed(9)

    def matrix(r, c, pad):
        return torch.rand((c, r + pad), dtype=torch.float64, device="cuda", generator=g) * 2 - 1

    def host(t):
        h = torch.empty(t.shape, dtype=torch.float64, pin_memory=pin)
        h.copy_(t)
        return h

    A = matrix(*((m, k) if ta == "N" else (k, m)), 3)
    B = matrix(*((k, n) if tb == "N" else (n, k)), 0)
    C = matrix(m, n, 1)
    hA, hB, hC = host(A), host(B), host(C)
    handle.dgemm(ta, tb, m, n, k, 1.5, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), beta, C.data_ptr(), m + 1)
    torch.cuda.synchronize()
    handle.dgemm_host(ta, tb, m, n, k, 1.5, hA.data_ptr(), A.stride(0), hB.data_ptr(), B.stride(0), beta,
                      hC.data_ptr(), m + 1)
    want = C.cpu()
    diff = (hC - want)[:, :m].norm() / want[:, :m].norm()
    assert diff <= 2 * gemm_bound(k)
    assert torch.equal(hC[:, m], want[:, m])


def test_finer_tiles_keep_to_the_memory_limit():
    """The limit admits one slot of the whole C, not the four of 1024 x 1024 that need 8 MB more: those are
    allocated (here: refused) only once the limit is lifted."""
    import torch
    import cosma_amd as ca
    m, n, k = 1793, 1793, 64
    h = ca.Handle(0)
    A, B, C = (torch.rand(s, dtype=torch.float64).pin_memory() for s in ((k, m), (n, k), (n, m)))
    want = 1.5 * (B @ A) + 0.5 * C

    def product():
        h.dgemm_host("N", "N", m, n, k, 1.5, A.data_ptr(), m, B.data_ptr(), k, 0.5, C.data_ptr(), m)
        assert h.last_mode() == 1

    h.set_memory_limit(8 * (m * k + k * n + 2 * m * n))
    product()
    assert (C - want).norm() / want.norm() <= 2 * gemm_bound(k)
    h.set_memory_limit(0)
    ca.fail_allocations(0, 1)
    try:
        with pytest.raises(ca.CosmaAmdError) as e:
            product()
        assert e.value.status == 3
    finally:
        ca.fail_allocations(0, 0)
