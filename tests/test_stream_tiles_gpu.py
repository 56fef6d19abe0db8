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


TILES_OF = """
import torch, sys
import cosma_amd as ca
h = ca.Handle(0)
def call(kinds, m, n, k, beta):
    put = {"d": lambda t: t.cuda(), "p": lambda t: t.pin_memory(), "g": lambda t: t}
    A, B, C = (put[x](torch.zeros(s, dtype=torch.float64)) for x, s in zip(kinds, ((k, m), (n, k), (n, m))))
    print("call", kinds, m, n, k, beta, file=sys.stderr, flush=True)
    h.dgemm_host("N", "N", m, n, k, 1.0, A.data_ptr(), m, B.data_ptr(), k, beta, C.data_ptr(), m)
for beta in (0.0, 0.5):
    for kinds in ("ppp", "gpp", "pgp", "ppg", "ddg", "ddp"):
        call(kinds, 1800, 1800, 1800, beta)
    call("ddg", 8192, 8192, 64, beta)
    call("dgp", 1500, 7000, 1200, beta)
    call("gdp", 1500, 7000, 1200, beta)
"""


def test_pageable_blocks_stay_large_enough_for_the_packing_threads():
    """The traced tiles of host products: 1800^3 is cut in 2 x 2 tiles of C unless an operand is pageable (its blocks
    of 1024^2 would be packed by two threads).  Pageable operands whose blocks keep 16 MB or their size are cut,
    unless beta != 0 has a pageable C packed on its way up too."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", TILES_OF], cwd=root, capture_output=True, text=True, timeout=100,
                       env={**os.environ, "COSMA_AMD_TRACE": "1"})
    assert r.returncode == 0, r.stderr[-2000:]
    tiles, got = {}, None
    for line in r.stderr.splitlines():
        if line.startswith("call "):
            got = tuple(line.split()[1:])
            tiles[got] = 0
        elif line.startswith("[cosma_amd] tile ("):
            tiles[got] += 1
    want = {}
    for beta in ("0.0", "0.5"):
        for kinds in ("ppp", "gpp", "pgp", "ppg", "ddg", "ddp"):
            want[kinds, "1800", "1800", "1800", beta] = 1 if "g" in kinds else 4
        want["ddg", "8192", "8192", "64", beta] = 16 if beta == "0.0" else 4
        for kinds in ("dgp", "gdp"):   # B in blocks of 1200 x 1792, A in one
            want[kinds, "1500", "7000", "1200", beta] = 4
    assert tiles == want
