"""The INT8 residue products at the edges of their 256 x 256 tiles and 128-byte
k-steps, for short and for wide sums (k > 32768), against the BF16 residue
products, which run another kernel: both are exact, so the split-precision
results must be equal bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (255, 257, 256), (256, 256, 257), (513, 16, 127), (300, 520, 1000),
                                   (17, 260, 33000)])
def test_int8_products_equal_bf16_products(handle, m, n, k, ta, tb):
    import torch
    import cosma_amd as ca
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    A = torch.randn(*((k, m) if ta == "N" else (m, k)), dtype=torch.float64, device="cuda", generator=g)
    B = torch.randn(*((n, k) if tb == "N" else (k, n)), dtype=torch.float64, device="cuda", generator=g)
    out = []
    for method in (ca.OZAKI_MODULI, ca.OZAKI_MODULI_BF16):
        C = torch.full((n, m), float("nan"), dtype=torch.float64, device="cuda")
        info = handle.dgemm_ozaki(ta, tb, m, n, k, 1.0, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), 0.0,
                                  C.data_ptr(), m, method=method, count=16)
        torch.cuda.synchronize()
        assert info["method"] == method
        out.append(C)
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])


def test_int8_products_of_planes_beyond_the_last_level_cache(handle):
    """Planes of more than 384 Mi elements take another INT8 kernel: just past that line, with ragged tiles."""
    import torch
    import cosma_amd as ca
    m, n, k = 257, 12300, 32768
    assert (m + n) * k > 384 << 20
    g = torch.Generator(device="cuda").manual_seed(11)
    A = torch.randn(m, k, dtype=torch.float64, device="cuda", generator=g)   # op(A) = A^T: rows contiguous in k
    B = torch.randn(n, k, dtype=torch.float64, device="cuda", generator=g)
    out = []
    for method in (ca.OZAKI_MODULI, ca.OZAKI_MODULI_BF16):
        C = torch.full((n, m), float("nan"), dtype=torch.float64, device="cuda")
        info = handle.dgemm_ozaki("T", "N", m, n, k, 1.0, A.data_ptr(), k, B.data_ptr(), k, 0.0, C.data_ptr(), m,
                                  method=method, count=16)
        torch.cuda.synchronize()
        assert info["method"] == method
        out.append(C)
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])
