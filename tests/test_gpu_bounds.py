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


@pytest.mark.parametrize("M", [1, 61, 64, 65, 190])
def test_wgrad_not_finite(dev, M):
    """Infinities and NaN in the last rows of X and in the four rows past them
    reach the taps that read them and no other: the rows of the last stage past
    M add nothing.  dU has no zeros, so 0 x infinity comes from nowhere else."""
    from sseqs_amd._lib import call, stream_of
    announce(f"wgrad not finite M={M}")
    rng = np.random.default_rng(M)
    X = rng.integers(-4, 5, (M + 8, 64)).astype(np.float32)
    dU = rng.integers(1, 5, (M, 64)).astype(np.float32)  # small whole numbers: every sum is exact
    for i, row in enumerate((M + 3, M + 4, M + 7)):  # rows M - 1, M and M + 3 of the sequence
        X[row, 8 * i], X[row, 8 * i + 1] = np.inf, np.nan
    tX = torch.from_numpy(X).to(dev).to(torch.bfloat16)
    tU = torch.from_numpy(dU).to(dev).to(torch.bfloat16)
    dW = torch.zeros(9 * 64, 64, device=dev)
    call("sseqs_enc_wgrad", tX.data_ptr() + 8 * 64, 64, tU.data_ptr(), 64, M, dW.data_ptr(), stream_of(tX.device))
    with np.errstate(invalid="ignore"):
        for t in range(9):
            want = (X[t:t + M, :, None].astype(np.float64) * dU[:, None, :]).sum(0)
            assert np.array_equal(dW[64 * t:64 * t + 64].double().cpu().numpy(), want, equal_nan=True), t
