"""Edges of the size rules that choose between kernels, against the oracle.

Integer results must be equal; prefilter scores lie within the oracle's
stated tolerance (orc.corr_tol)."""
import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu

AA = "ARNDCQEGHILKMFPSTWYV"


def rand_seq(rng, n, alphabet=AA):
    return "".join(rng.choice(list(alphabet), int(n)))


@pytest.mark.parametrize("Lq,n", [(1, 1), (31, 3), (32, 4), (33, 5), (992, 15), (993, 16), (1024, 17), (1025, 17)])
def test_ascii_sw_packed_edges(orc, dev, Lq, n):
    """ASCII targets on the packed 16-bit kernel and past it (1024 residues,
    gap parameters of 16000): counts around the four targets of a wave and
    the sixteen of a block, targets around the 256 staged rows, an empty one,
    and the largest score there is."""
    from sseqs_amd import ops
    announce(f"ascii sw Lq={Lq} n={n}")
    rng = np.random.default_rng(10 * Lq + n)
    query = "W" * Lq
    lens = [255, 0, 256, 257, 1, 513, Lq]
    tg = [("W" * L if i % 2 else rand_seq(rng, L, AA + "XBZ*-")) for i, L in enumerate(lens)]
    a = np.frombuffer(("@".join(tg) + "@").encode(), np.uint8).copy()
    P = np.nonzero(a == 64)[0].astype(np.int32)
    gi = (np.arange(n) % P.size).astype(np.int32)
    qc = orc.encode_query_sw(query)
    t = [torch.from_numpy(x).to(dev) for x in (qc, gi, a, P)]
    for o, e in ((11, 1), (16000, 16000), (16001, 1)):
        assert np.array_equal(ops.sw_cuda_affine(*t, o, e).cpu().numpy(), orc.sw_affine(qc, gi, a, P, o, e)), (o, e)
    for gap in (-1, -16000, -16001):
        got = ops.sw_cuda_blosum62(*t, gap_penalty_param=gap).cpu().numpy()
        assert np.array_equal(got, orc.sw_linear(qc, gi, a, P, gap)), gap
