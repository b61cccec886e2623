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


SEL_N = 1 << 22  # scores from which few of them are selected from a sample's guess


@pytest.mark.parametrize("n,k,dtype,kind", [
    (SEL_N, SEL_N // 64, "f32", "normal"), (SEL_N, SEL_N // 64 + 1, "f32", "normal"),
    (SEL_N - 1, 1000, "f32", "normal"), (SEL_N + 16384 + 257, 1, "f32", "normal"),
    (SEL_N + 4097, 5000, "f32", "special"), (SEL_N + 3, 5000, "f16", "normal"),
    (SEL_N + 1, 777, "f16", "special"), (SEL_N + 2, 5000, "i32", "normal"),
    (SEL_N, 4096, "i32", "ties"), (SEL_N, 4096, "f32", "equal"), (SEL_N + 5, 20000, "f32", "rising"),
    (SEL_N, 30000, "f32", "bunched")])
def test_topk_sampled(dev, n, k, dtype, kind):
    """Top-k of a sample's guess around the sizes that choose it: ties, NaN
    and infinities, scores whose sample misleads (all the largest within one
    stretch), an address that is not aligned, sorted output, and the same
    indices from the entry point without a workspace."""
    from sseqs_amd import _lib, ops
    announce(f"topk n={n} k={k} {dtype} {kind}")
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal(n + 1).astype(np.float32) * 8 + 21
    if kind == "special":
        x[::97] = np.nan
        x[5::1013] = np.inf
        x[7::1013] = -np.inf
        x[9::11] = -0.0
    elif kind == "ties":
        x = np.where(x > 33, 5, -5).astype(np.float32)
    elif kind == "equal":
        x[:] = 3.5
    elif kind == "rising":
        x.sort()
    elif kind == "bunched":
        x[1_000_001:1_000_001 + k + 7] += 1000
    v = x.astype(np.float16) if dtype == "f16" else x.astype(np.int32) if dtype == "i32" else x
    full = torch.from_numpy(v).to(dev)
    for off in (0, 1):  # aligned, and one score past it
        y = v[off:off + n].astype(np.float32)
        # (score desc, index asc), -0 below +0, NaN last: order of the bits
        b = y.view(np.uint32)
        key = np.where(b >> 31 == 1, ~b, b | np.uint32(0x80000000))
        key = np.where(np.isnan(y), 0, key).astype(np.int64)
        want = np.argsort(-key, kind="stable")[:k]
        s = full[off:off + n]
        assert np.array_equal(ops.topk_indices(s, k, sorted=False).cpu().numpy(), np.sort(want))
        if k <= 16384:
            assert np.array_equal(ops.topk_indices(s, k, sorted=True).cpu().numpy(), want)
        out = torch.empty(k, dtype=torch.int64, device=dev)
        _lib.call("sseqs_topk_noalloc", s.data_ptr(), ops._DT[s.dtype], n, k, 0, out.data_ptr(),
                  _lib.stream_of(dev))
        assert np.array_equal(out.cpu().numpy(), np.sort(want))
