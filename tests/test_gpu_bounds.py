"""Where a kernel's arithmetic, addressing or launch rule has a bound: calls
on both sides of it, against the oracle or plain torch."""
import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

AA = "ARNDCQEGHILKMFPSTWYV"


def rand_seq(rng, n, alphabet=AA):
    return "".join(rng.choice(list(alphabet), int(n)))


@pytest.mark.parametrize("L", [744, 745, 2978, 2979, 3000, 3300])
def test_backtrack_16bit_cells(orc, dev, L):
    """The definition's cells are 16 bits: scores around and past 2^15 (11 a
    residue) wrap in the kernel where they wrap in the oracle."""
    from sseqs_amd.sw import sw_affine_backtrack
    announce(f"backtrack 16-bit cells L={L}")
    rng = np.random.default_rng(L)
    query = "W" * L
    tg = ["W" * L, "W" * (L // 2) + rand_seq(rng, 5) + "W" * (L - L // 2 - 5), rand_seq(rng, L), "W" * (L - 7)]
    for o, e in ((11, 1), (3, 0)):
        _, _, got = sw_affine_backtrack(query, tg, o, e)
        for t, g in zip(tg, got):
            assert g == orc.backtrack(query, t, o, e), (len(t), o, e)
