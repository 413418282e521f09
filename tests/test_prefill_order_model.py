"""Host model of the block order of the prefill tile launches (pf_block_of and pf_padded in promoe_amd/csrc/moe_prefill.hip):
every block of both classes is taken exactly once, and no XCD (workgroup index modulo 8) gets more of a class than an even
share and, in the order of runs, one run."""
import os
import re

import pytest

_SRC = " ".join(open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "promoe_amd", "csrc",
                                  "moe_prefill.hip")).read().split())
DEAL = int(re.search(r"#define PF_DEAL (\d+)", _SRC).group(1))


def test_the_model_is_the_source():
    for ln in ("const int q = even && blocks < 8 * PF_DEAL ? 8 : 8 * PF_DEAL; return (blocks + q - 1) / q * q;",
               "xcd = (xcd - (n0 + PF_DEAL - 1) / PF_DEAL) & 7;",
               "const int i = pb >> 3, first = i / PF_DEAL * (8 * PF_DEAL), j = i % PF_DEAL;",
               "int b = first + xcd * PF_DEAL + j;", "if (EVEN && n_real - first < 8 * PF_DEAL) {",
               "const int each = (n_real - first + 7) >> 3; if (j >= each) return false; b = first + xcd * each + j;"):
        assert ln in _SRC, ln


def _order(even, n_shared, n_routed, n_routed_max):
    """[(class, block, XCD)] of a launch: class 0 = shared (all blocks in use), 1 = routed (n_routed of n_routed_max)."""
    padded = []
    for n in (n_shared, n_routed_max):
        q = 8 if even and n < 8 * DEAL else 8 * DEAL
        padded.append(-(-n // q) * q)
    out = []
    for blk in range(sum(padded)):
        ci = int(blk >= padded[0])
        pb = blk - padded[0] if ci else blk
        n = (n_shared, n_routed)[ci]
        xcd = pb & 7
        if not even and ci:
            xcd = (xcd - -(-n_shared // DEAL)) & 7
        i = pb >> 3
        first, j = i // DEAL * 8 * DEAL, i % DEAL
        b = first + xcd * DEAL + j
        if even and n - first < 8 * DEAL:
            each = (n - first + 7) >> 3
            if j >= each:
                continue
            b = first + xcd * each + j
        if b < n:
            out.append((ci, b, blk & 7))
    return out


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("n_shared", [0, 1, 7, 8, 9, 24, 40, 44, 63, 64, 65, 72, 88, 128, 352, 1000])
@pytest.mark.parametrize("n_routed,n_max", [(0, 0), (0, 8), (1, 16), (7, 9), (40, 40), (63, 64), (480, 496), (1000, 2000)])
def test_every_block_once_and_evenly(even, n_shared, n_routed, n_max):
    order = _order(even, n_shared, n_routed, n_max)
    for ci, n in enumerate((n_shared, n_routed)):
        mine = [(b, x) for c, b, x in order if c == ci]
        assert sorted(b for b, _ in mine) == list(range(n))
        per = [sum(1 for _, x in mine if x == k) for k in range(8)]
        assert max(per) <= -(-n // 8) + (0 if even else DEAL)
