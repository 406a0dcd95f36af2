"""k_router_exact_small: the adding wave and the producing waves meet at the
same number of barriers for every row length.  The producers take one per chunk
they are rounded up to; the adding wave's come from three loops, modelled here
with the main loop's condition taken from the source."""
import re

import pytest

from cpubrrr_amd.build import CSRC

SRC = (CSRC / "moe_grouped.hip").read_text()
KERNEL = SRC[SRC.index("void k_router_exact_small"):SRC.index("void k_router_transpose")]


@pytest.mark.parametrize("chunk", [64, 128])
def test_same_barriers(chunk):
    cond, = re.findall(r"for \(; (.*); k \+= 3\) \{", KERNEL)
    assert "if (k + j + 1 < nch) arrive();" in KERNEL and "for (k += 4; k < nch; k++) arrive();" in KERNEL
    cond = compile(cond, "main loop", "eval")
    ahead = int(re.search(r"kPcSteps = (\d+)", SRC)[1]) // chunk
    B = chunk // 32
    for d in range(32, 8192 + 32, 32):
        nch = -(-d // (ahead * chunk)) * ahead
        nb, k, met, summed = d // 32, 0, 1, 0
        while eval(cond, {}, {"B": B, "k": k, "nb": nb, "nch": nch}):
            k, met, summed = k + 3, met + 3, summed + 3 * B
        for j in range(3):
            summed += sum(B * (k + j) + m < nb for m in range(B))
            met += k + j + 1 < nch
        met += max(0, nch - (k + 4))
        assert (met, summed) == (nch, nb), f"d={d}: {met} barriers against {nch}, {summed} of {nb} blocks"
