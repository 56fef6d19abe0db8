"""Grouped DGEMM kernels of one common transpose, mixed transposes and plans
with a leading dimension beyond the direct-LDS kernels, in every tile
configuration: each problem must equal its own cosma_amd_dgemm call bit for
bit, with NaN in the operands' padding and C's padding untouched."""
import pytest

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (16, 17, 16), (33, 64, 15), (64, 65, 32), (65, 33, 47), (97, 129, 1), (128, 128, 96), (130, 31, 0),
        (200, 150, 33), (31, 300, 64), (257, 5, 130)]


def tensor(rows, cols, pad, g):
    import torch
    t = torch.full((cols, rows + pad), float("nan"), dtype=torch.float64, device="cuda")
    t[:, :rows] = torch.rand((cols, rows), dtype=torch.float64, device="cuda", generator=g) * 2 - 1
    return t


def problems(trans, pad):
    import torch
    g = torch.Generator(device="cuda").manual_seed(7)
    out = []
    for i, (m, n, k) in enumerate(DIMS):
        ta, tb = trans[i % len(trans)]
        A = tensor(*((m, k) if ta == "N" else (k, m)), pad * (i % 3), g)
        B = tensor(*((k, n) if tb == "N" else (n, k)), pad * (i % 2), g)
        out.append((ta, tb, m, n, k, (1.0, -1.5)[i % 2], A, B, (0.0, 0.5)[i % 2], tensor(m, n, pad * (i % 4), g)))
    return out


def args(p, C):
    ta, tb, m, n, k, alpha, A, B, beta, _ = p
    return (ta, tb, m, n, k, alpha, A.data_ptr(), max(1, A.stride(0)), B.data_ptr(), max(1, B.stride(0)), beta,
            C.data_ptr(), C.stride(0))


def check(handle, probs, cfgs):
    import torch
    import cosma_amd as ca
    want = [p[9].clone() for p in probs]
    for p, C in zip(probs, want):
        handle.dgemm(*args(p, C))
    for cfg in cfgs:
        got = [p[9].clone() for p in probs]
        plan = ca.Grouped(handle, [args(p, C) for p, C in zip(probs, got)], tile_config=cfg)
        for grid in (0, 3, 1 << 20):   # the default, persistent workgroups with many tiles each, one per tile
            for p, C in zip(probs, got):
                C.copy_(p[9])
            plan.set_config(cfg, grid)
            plan.run()
            torch.cuda.synchronize()
            for p, C, W in zip(probs, got, want):
                assert torch.equal(C[:, :p[2]], W[:, :p[2]]), (cfg, grid, p[:5])
                assert torch.isnan(C[:, p[2]:]).all()
        plan.close()


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("trans", [["NN"], ["TN"], ["NT"], ["TT"], ["NN", "TN", "NT", "TT"]], ids="-".join)
def test_grouped_tiles(handle, trans, pad):
    check(handle, problems(trans, pad), (1, 2, 3, 4, 5))


def test_leading_dimension_beyond_the_lane_offsets(handle):
    import torch
    g = torch.Generator(device="cuda").manual_seed(8)
    probs = problems(["NN"], 0)
    m, n, k, ld = 40, 3, 50, (1 << 22) + 2
    B = torch.zeros((n, ld), dtype=torch.float64, device="cuda")
    B[:, :k] = torch.rand((n, k), dtype=torch.float64, device="cuda", generator=g)
    probs.append(("N", "N", m, n, k, 1.0, tensor(m, k, 0, g), B, 0.0, tensor(m, n, 0, g)))
    check(handle, probs, (1, 2, 3, 4, 5))


def test_tuned_choice_is_not_taken_over_by_other_kernels(handle):
    """A plan beyond the direct-LDS kernels runs others under the same configuration numbers: what tuning found for
    the same shapes within their limits is not its choice."""
    import torch
    import cosma_amd as ca
    m, count, ld = 16, 20000, (1 << 22) + 2
    A = torch.rand((m, m), dtype=torch.float64, device="cuda")
    B = torch.zeros((m, ld), dtype=torch.float64, device="cuda")
    C = torch.zeros(count * m * m, dtype=torch.float64, device="cuda")

    def plan(ldb, cfg=0):
        return ca.Grouped(handle, [("N", "N", m, m, m, 1.0, A.data_ptr(), m, B.data_ptr(), ldb if i == 0 else m, 0.0,
                                    C.data_ptr() + 8 * i * m * m, m) for i in range(count)], tile_config=cfg)

    first = plan(m)
    first.tune()
    assert plan(m).info() == first.info()
    assert plan(ld).info() == plan(ld, 1).info()   # the default: 64 x 64 with its default grid
