"""The split's reduction of integers above 2^50 (ozaki.hpp: moduli_residues16),
restated with the same FP64 operations: reduced modulo the product of a group
of moduli first, every value must be an exact integer below 2^48 and give the
symmetric residue of each modulus.  The FMAs are exact (integers below 2^53),
so plain integers stand in for them."""
import random

MODULI = [256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193, 191, 181, 179, 173]
GROUP = 6


def residue(x, m):
    q = round(float(x) * (1.0 / m))       # rint of the FP64 product: ties to even
    r = x - m * q
    return (r + 128) % 256 - 128          # the byte that is stored


def test_group_reduction_gives_symmetric_residues():
    rng = random.Random(1)
    for P in range(51, 59):
        top = 1 << P
        cases = [top, -top, top - (1 << (P - 53) if P > 53 else 1), 0, 1, -1]
        cases += [int(float(rng.randrange(-top, top + 1))) for _ in range(3000)]   # FP64 integers
        for first in range(0, len(MODULI), GROUP):
            group = MODULI[first:first + GROUP]
            M = 1
            for m in group:
                M *= m
            assert M < 1 << 48 and float(M) == M
            near = [k * M + d for k in (1, -1, (top // M) // 2) for d in (M // 2, -(M // 2), 0, 1)]
            for x in cases + [int(float(v)) for v in near if abs(v) <= top]:
                q = round(float(x) * (1.0 / float(M)))
                y = x - M * q
                assert abs(y) < 1 << 48 and float(y) == y
                for m in group:
                    want = x % m
                    want = want - m if want > (m - 1) // 2 else want
                    assert residue(y, m) == want, (P, x, m)


def test_the_header_holds_the_constants_checked_here():
    import os
    import re
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    text = open(os.path.join(root, "cosma_amd", "csrc", "ozaki.hpp")).read()
    moduli = re.search(r"kModuli\[20\] = \{([^}]*)\}", text).group(1)
    assert [int(x) for x in moduli.split(",")] == MODULI
    assert int(re.search(r"constexpr int MOD_GROUP = (\d+);", text).group(1)) == GROUP
    assert int(re.search(r"constexpr int MAX_P = (\d+);", text).group(1)) == 58   # the largest P above
