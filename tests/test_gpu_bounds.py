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


@pytest.mark.parametrize("N,Lq", [(128, 60), (256, 200), (512, 400), (1024, 560), (1024, 1000), (2048, 1700)])
def test_prefilter_packed_alignment(orc, dev, N, Lq):
    """A packed stream at any address: the ring kernel's copies start at the
    16-byte granule that holds its first byte, and the band kernel's sizes take
    it too.  Sequences back to back and scattered, spans that hold '@', the
    stream's last symbol in the last byte."""
    from sseqs_amd import ops
    from sseqs_amd._lib import call, ptr, stream_of
    announce(f"prefilter alignment N={N} Lq={Lq}")
    rng = np.random.default_rng(N + Lq)
    query = rand_seq(rng, Lq)
    A, B = orc.weighted_luts(query, 4)
    qrev = orc.encode_query_rev(query)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
    lens = np.sort(np.array([0, 1, 31, 32, 33, N // 2, N - 31, N - 1, N] + list(rng.integers(1, N + 1, 40)), np.int32))
    lutB = torch.cat([t(B).reshape(-1), torch.zeros(1, device=dev)])
    for gap in (1, 40 * N):
        off = np.concatenate([[0], np.cumsum(lens + gap)[:-1]]).astype(np.int32)
        flat = np.full(int(off[-1] + lens[-1]), 64, np.uint8)
        for o, n in zip(off, lens):
            flat[o:o + n] = np.frombuffer((query * (N // Lq + 1)).encode(), np.uint8)[:n] if n % 3 else \
                rng.choice(np.frombuffer((AA + "XB").encode(), np.uint8), n)
        spans = flat.copy()
        for o, n in zip(off, lens):
            if n > 2:
                spans[o + n // 2] = 64
        for name, sym in (("sseqs_db_prefilter", flat), ("sseqs_db_prefilter_spans", spans)):
            want = orc.corr(qrev, A, B, 4, sym.tobytes(), off, lens, N, N)
            tol = orc.corr_tol(qrev, A, B, 4, sym.tobytes(), off, lens, N, N, want)
            packed = ops.compress(t(sym))
            keep = [t(off.astype(np.int64)), t(lens), t(qrev), t(A)]
            for lead in (0, 1, 4, 8, 13):
                buf = torch.zeros(16 + lead + packed.numel() + 64, dtype=torch.uint8, device=dev)
                at = buf[16 + lead:]
                at[:packed.numel()] = packed
                assert at.data_ptr() % 16 == lead
                out = torch.full((lens.size,), -7.0, dtype=torch.float32, device=dev)
                call(name, ptr(at), ptr(keep[0]), ptr(keep[1]), 0, lens.size, ptr(keep[2]), Lq, ptr(keep[3]),
                     ptr(lutB), 21, 4, N, N, ptr(out), stream_of(dev))
                assert (np.abs(out.cpu().numpy() - want) <= tol).all(), (name, gap, lead)


@pytest.mark.parametrize("bits", [5, 11, 12, 13, 17, 21, 22, 23, 28])
def test_topk_sample_guard(dev, bits):
    """The guess of the sampled select is dropped (P, the fifth word of the
    state behind the histogram, is 0) when more than an eighth of the scores
    reach it, whatever the digits of the sample's key range, and kept when
    they do not; the indices are the same either way."""
    from sseqs_amd import _lib
    announce(f"topk sample guard bits={bits}")
    n, k = 1 << 22, 10000
    g = torch.Generator(device=dev).manual_seed(bits)
    base = torch.randint(0, 1 << (bits - 1), (n,), generator=g, device=dev, dtype=torch.int32)
    top = (1 << bits) - 1
    few = torch.rand(n, generator=g, device=dev) < 0.01
    for share, kept in ((0.01, True), (0.3, False)):
        tied = torch.rand(n, generator=g, device=dev) < share
        x = torch.where(tied, torch.full_like(base, top - 1), base)
        x[few & tied] = top  # some above the tie, fewer than k
        ws = torch.zeros(_lib.load().sseqs_topk_ws_bytes(n), dtype=torch.uint8, device=dev)
        out = torch.empty(k, dtype=torch.int64, device=dev)
        _lib.call("sseqs_topk", x.data_ptr(), _lib.I32, n, k, 0, out.data_ptr(), ws.data_ptr(), ws.numel(),
                  _lib.stream_of(dev))
        P = int(ws[2048 * 4:2048 * 4 + 32].view(torch.int32)[4].item())
        assert (P != 0) == kept, (share, P)
        want = torch.sort(torch.sort(x, descending=True, stable=True).indices[:k]).values
        assert torch.equal(out, want)


@pytest.mark.parametrize("dtype,n,ratio", [
    ("f32", 1 << 22, 400), ("f32", 5999999, 400), ("f32", 6000000, 64), ("f16", 1 << 22, 128), ("f16", 5999996, 128),
    ("f16", 6000004, 64), ("i32", 1 << 22, 64), ("i32", 6000000, 64)])
def test_topk_sample_line(dev, dtype, n, ratio):
    """The largest selection that takes a sample's guess (P, the fifth word of
    the state, is not 0) and one more, for the types and lengths that choose it;
    the same indices either way."""
    from sseqs_amd import _lib, ops
    announce(f"topk sample line {dtype} n={n}")
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.randn(n, generator=g, device=dev) * 8 + 21
    x = x.half() if dtype == "f16" else (x * 1000).int() if dtype == "i32" else x
    order = torch.sort(x, descending=True, stable=True).indices
    for k, sampled in ((n // ratio, True), (n // ratio + 1, False)):
        ws = torch.zeros(_lib.load().sseqs_topk_ws_bytes(n), dtype=torch.uint8, device=dev)
        out = torch.empty(k, dtype=torch.int64, device=dev)
        _lib.call("sseqs_topk", x.data_ptr(), ops._DT[x.dtype], n, k, 0, out.data_ptr(), ws.data_ptr(), ws.numel(),
                  _lib.stream_of(dev))
        P = int(ws[2048 * 4:2048 * 4 + 32].view(torch.int32)[4].item())
        assert (P != 0) == sampled, (k, P)
        assert torch.equal(out, torch.sort(order[:k]).values)


@pytest.mark.parametrize("dtype", ["f16", "f32", "i32"])
def test_topk_segments_uncut(dev, dtype):
    """Segments that the instance with a list does not cut, next to ones that
    it does: short ones, selections too large for the list, an empty one, all of
    a segment, begins of any alignment."""
    from sseqs_amd import ops
    announce(f"topk_segments uncut {dtype}")
    rng = np.random.default_rng(4)
    segs = [(1, 1), (127, 127), (128, 128), (129, 128), (5000, 200), (8191, 8191), (8192, 4000), (8193, 150),
            (32767, 160), (32768, 160), (0, 0), (100003, 30000), (300007, 20000), (281000, 1405), (70001, 70001)]
    n = np.array([s[0] for s in segs])
    k = np.array([s[1] for s in segs])
    begin = np.concatenate([[1], 1 + np.cumsum(n + 1)[:-1]])
    flat = np.round(rng.normal(21.0, 4.0, int(n.sum() + n.size + 1)) * 8) / 8  # ties
    flat = flat.astype({"f16": np.float16, "f32": np.float32, "i32": np.int32}[dtype])
    for drop in ((0, 0), (1, 2)):
        got, base = ops.topk_segments(torch.from_numpy(flat).to(dev), begin, n, k, drop_front=drop[0],
                                      drop_back=drop[1])
        got = got.cpu().numpy()
        for j, (nj, kj) in enumerate(segs):
            x = flat[begin[j]: begin[j] + nj].astype(np.float64)
            want = np.sort(np.argsort(-x, kind="stable")[:kj])[drop[0]: max(drop[0], kj - drop[1])]
            assert np.array_equal(got[base[j]: base[j] + want.size], want), (segs[j], drop)


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1023, 1025, 16383, 16384, 16385, 16384 + 1024, 3 * 16384 + 257])
@pytest.mark.parametrize("dtype", ["f16", "f32", "i32"])
def test_topk_last_tile(dev, dtype, n):
    """The count and write passes end with the scores: lengths around their
    steps of 256 and 1024 in the last tile of 16384, aligned and one score past
    an aligned address, few and all of them selected, with ties."""
    from sseqs_amd import ops
    announce(f"topk last tile {dtype} n={n}")
    g = torch.Generator(device=dev).manual_seed(n)
    full = torch.round(torch.randn(n + 1, generator=g, device=dev) * 40)
    full = full.half() if dtype == "f16" else full.int() if dtype == "i32" else full
    for lead in (0, 1):
        x = full[lead:lead + n]
        order = torch.sort(x, descending=True, stable=True).indices
        for k in sorted({1, (n + 3) // 4, n}):
            assert torch.equal(ops.topk_indices(x, k, sorted=False), torch.sort(order[:k]).values), (lead, k)


@pytest.mark.parametrize("M,cin,cout", [(64, 64, 64), (128, 128, 256), (64 * 9 + 1, 64, 64), (64 * 64, 64, 128),
                                        (64 * 333, 128, 256), (64 * 1400, 64, 64)])
def test_gradient_sums_exact(dev, M, cin, cout):
    """Weight, bias and embedding gradients of small whole numbers, whose fp32
    sums are exact in any order: one lost or doubled row or stage shows.  Row
    counts of one slice, of a few stages each and of many blocks."""
    from sseqs_amd._lib import call, stream_of
    announce(f"exact gradient sums M={M} cin={cin} cout={cout}")
    g = torch.Generator(device=dev).manual_seed(M + cin + cout)
    small = lambda *s: torch.randint(-3, 4, s, generator=g, device=dev)  # noqa: E731
    X = torch.zeros(M + 8, cin, device=dev)
    X[4:-4] = small(M, cin)
    dU = small(M, cout).float()
    tX, tU, st = X.to(torch.bfloat16), dU.to(torch.bfloat16), stream_of(X.device)
    assert 9 * M < 2 ** 23  # the largest sum there can be, and the start of 3
    dW = torch.full((9 * cin, cout), 3.0, device=dev)
    call("sseqs_enc_wgrad", tX.data_ptr() + 8 * cin, cin, tU.data_ptr(), cout, M, dW.data_ptr(), st)
    for t in range(9):
        want = X[t:t + M].double().T @ dU.double() + 3
        assert torch.equal(dW[t * cin:(t + 1) * cin].double(), want), t
    db = torch.full((cout,), 3.0, device=dev)
    call("sseqs_enc_bias_grad", tU.data_ptr(), cout, M, db.data_ptr(), st)
    assert torch.equal(db.double(), dU.double().sum(0) + 3)
    code = torch.randint(0, 22, (M,), generator=g, device=dev).to(torch.uint8)
    dx = small(M, 64).float()
    dE = torch.full((22, 64), 3.0, device=dev)
    call("sseqs_enc_embed_grad", code.data_ptr(), M, dx.data_ptr(), dE.data_ptr(), st)
    want = torch.zeros(22, 64, dtype=torch.float64, device=dev).index_add_(0, code.long(), dx.double())
    want[20:] = 0
    assert torch.equal(dE.double(), want + 3)


@pytest.mark.parametrize("nseq,most", [(1, 70), (511, 40), (512, 17), (513, 17), (1056, 40), (2048, 9), (4095, 20),
                                       (4096, 20), (70000, 3)])
def test_pool_gradient_split(dev, nseq, most):
    """The pool's gradient for the numbers of sequences that choose its blocks
    per sequence, past the grid's 65536 blocks too, equals that of 256 sequences
    at a time bit for bit: every row of every sequence, no row between them."""
    from sseqs_amd._lib import call, stream_of
    announce(f"pool gradient nseq={nseq}")
    g = torch.Generator(device=dev).manual_seed(nseq)
    lens = torch.randint(0, most + 1, (nseq,), generator=g, device=dev)
    lens[-1] = most
    row0 = 4 + torch.cumsum(lens + 2, 0) - (lens + 2)
    M = int((row0[-1] + lens[-1] + 4).item())
    e = torch.nn.functional.normalize(torch.randn(nseq, 256, generator=g, device=dev), dim=1)
    de = torch.randn(nseq, 256, generator=g, device=dev)
    zn = torch.rand(nseq, generator=g, device=dev) + 0.5
    U = torch.randn(M, 256, generator=g, device=dev).to(torch.bfloat16)
    tl = lens.to(torch.int32)
    out, want = (torch.full((M, 256), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
    grad = lambda a, b, t: call("sseqs_enc_pool_grad", de[a:].data_ptr(), e[a:].data_ptr(), zn[a:].data_ptr(),  # noqa: E731
                                U.data_ptr(), row0[a:].data_ptr(), tl[a:].data_ptr(), b - a, t.data_ptr(),
                                stream_of(e.device))
    grad(0, nseq, out)
    for a in range(0, nseq, 256):  # the most blocks a sequence, against 64 bits in test_encoder_pool_gradient_rows
        grad(a, min(a + 256, nseq), want)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("Lq", [640, 641, 672, 673, 768, 769, 896, 897, 928, 929, 1023, 1024])
def test_ascii_affine_stripes(orc, dev, Lq):
    """Affine SW of ASCII targets at the stripe widths around which the packed
    kernel's registers change."""
    from sseqs_amd import ops
    announce(f"ascii affine stripes Lq={Lq}")
    rng = np.random.default_rng(Lq)
    query = rand_seq(rng, Lq, AA + "X")
    tg = [query, query[Lq // 3:] + rand_seq(rng, 40), "", rand_seq(rng, 300, AA + "XB*"), query[:200][::-1], "W" * 700,
          query[: Lq // 2] + rand_seq(rng, 31) + query[Lq // 2 + 7:]] * 3
    a = np.frombuffer(("@".join(tg) + "@").encode(), np.uint8).copy()
    P = np.nonzero(a == 64)[0].astype(np.int32)
    gi = np.arange(P.size, dtype=np.int32)
    qc = orc.encode_query_sw(query)
    t = [torch.from_numpy(x).to(dev) for x in (qc, gi, a, P)]
    for o, e in ((11, 1), (0, 0), (3, 7)):
        assert np.array_equal(ops.sw_cuda_affine(*t, o, e).cpu().numpy(), orc.sw_affine(qc, gi, a, P, o, e)), (o, e)


@pytest.mark.parametrize("sign", [1, -1])
def test_encoder_gelu_every_float(dev, sign):
    """The tiled kernels' GELU equals the general kernel's for every normal fp32
    number: the upper seven bits of the mantissa come as a product with 1, the
    lower sixteen as a bias, and the sum is exact.  (Subnormal numbers and
    infinities: test_encoder_gelu_rounding.)"""
    from sseqs_amd._lib import call, stream_of
    announce(f"gelu of every float, sign {sign}")
    M, N = 128, 1 << 16
    A = torch.zeros(M + 8, 64, dtype=torch.bfloat16, device=dev)
    Bt = torch.zeros(N, 576, dtype=torch.bfloat16, device=dev)
    Bt[:, 4 * 64] = 1  # the row itself, channel 0
    mask = torch.ones(M, dtype=torch.uint8, device=dev)
    U, Y, Z = (torch.empty(M * N + 8, dtype=torch.bfloat16, device=dev) for _ in range(3))
    hi = torch.arange(128, device=dev, dtype=torch.int64) << 16
    low = torch.arange(N, device=dev, dtype=torch.int64)
    neg = -2 ** 31 if sign < 0 else 0
    st = stream_of(A.device)
    bad = torch.zeros((), dtype=torch.int64, device=dev)
    for e in range(1, 255):  # the exponent's field
        head = ((e << 23) | hi) + neg
        A[4:-4, 0] = head.to(torch.int32).view(torch.float32).to(torch.bfloat16)
        one = torch.tensor([(e << 23) + neg], device=dev).to(torch.int32).view(torch.float32)
        bias = (((e << 23) | low) + neg).to(torch.int32).view(torch.float32) - one
        for out, shift in ((Y, 0), (Z, 2)):  # 2: not 16-byte aligned, the general kernel
            call("sseqs_enc_conv", A.data_ptr() + 8 * 64, 64, Bt.data_ptr(), M, N, 576, bias.data_ptr(), mask.data_ptr(),
                 U.data_ptr() if shift == 0 else None, out.data_ptr() + 2 * shift, None, None, 0, st)
        bad += (Y[:M * N].view(torch.int16) != Z[2:M * N + 2].view(torch.int16)).sum()
        x = (head[:, None] + low[None, :]).to(torch.int32).view(torch.float32)
        if e in (1, 100, 127, 254):  # the numbers are the ones meant
            assert torch.equal(U[:M * N].view(M, N).view(torch.int16), x.to(torch.bfloat16).view(torch.int16)), e
    assert int(bad) == 0


@pytest.mark.parametrize("N,Lq", [(64, 50), (128, 100), (256, 200), (512, 400), (1024, 700), (2048, 1500)])
@pytest.mark.parametrize("mt", [None, "1"])
def test_prefilter_without_band(orc, dev, monkeypatch, N, Lq, mt):
    """SSEQS_CORR_NO_BAND takes every rank-4 size to the dense kernels (m-tiles
    per pass capped by SSEQS_CORR_MT) and the ASCII operator to the general one:
    scores within the tolerance, and the kernels' names say so."""
    from sseqs_amd import ops
    from sseqs_amd._lib import call, ptr, stream_of
    from sseqs_amd.search import prefilter_kernel_name
    announce(f"prefilter without band N={N} Lq={Lq} mt={mt}")
    monkeypatch.setenv("SSEQS_CORR_NO_BAND", "1")
    if mt:
        monkeypatch.setenv("SSEQS_CORR_MT", mt)
    passes = min(N // 64, 4 if N <= 512 else 8)
    assert prefilter_kernel_name(Lq, 4, N) == f"k_corr_db4<{1 if mt else passes}>"
    rng = np.random.default_rng(N + Lq)
    query = rand_seq(rng, Lq)
    A, B = orc.weighted_luts(query, 4)
    qrev = orc.encode_query_rev(query)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
    lens = np.sort(np.array([1, 15, 16, 17, N // 2, N - 1, N] + list(rng.integers(1, N + 1, 70)), np.int32))
    off = np.concatenate([[0], np.cumsum(lens + 1)[:-1]]).astype(np.int32)
    flat = np.full(int(off[-1] + lens[-1] + 1), 64, np.uint8)
    for o, n in zip(off, lens):
        flat[o:o + n] = np.frombuffer((query * (N // Lq + 1)).encode(), np.uint8)[:n] if n % 3 else \
            rng.choice(np.frombuffer((AA + "XB").encode(), np.uint8), n)
    want = orc.corr(qrev, A, B, 4, flat.tobytes(), off, lens, N, N)
    tol = orc.corr_tol(qrev, A, B, 4, flat.tobytes(), off, lens, N, N, want)
    packed = torch.cat([ops.compress(t(flat)), torch.zeros(64, dtype=torch.uint8, device=dev)])
    keep = [t(off.astype(np.int64)), t(lens), t(qrev), t(A), torch.cat([t(B).reshape(-1), torch.zeros(1, device=dev)])]
    for name in ("sseqs_db_prefilter", "sseqs_db_prefilter_spans"):
        out = torch.empty(lens.size, dtype=torch.float32, device=dev)
        call(name, ptr(packed), ptr(keep[0]), ptr(keep[1]), 0, lens.size, ptr(keep[2]), Lq, ptr(keep[3]), ptr(keep[4]),
             21, 4, N, N, ptr(out), stream_of(dev))
        assert (np.abs(out.cpu().numpy() - want) <= tol).all(), name
    scores = torch.zeros(lens.size, dtype=torch.float16, device=dev)
    ops.warp_corr(scores, keep[2], keep[3], t(B), t(flat), t(off), keep[1], 4, Lq, N, N,
                  torch.zeros(1, dtype=torch.float16, device=dev))
    assert (np.abs(scores.float().cpu().numpy() - want) <= tol).all()


def test_topk_segments_captured(dev):
    """The segmented select that cuts long segments, captured in a graph: the
    same indices on every replay, with eager work between the replays."""
    from sseqs_amd import _lib
    announce("topk_segments captured")
    g = torch.Generator(device=dev).manual_seed(9)
    n, k, nseg = 50000, 300, 6
    x = torch.randn(nseg * n, generator=g, device=dev).half()
    begin = torch.arange(nseg, device=dev) * n
    base = torch.arange(nseg, device=dev) * k
    nn, kk = (torch.full((nseg,), v, dtype=torch.int32, device=dev) for v in (n, k))
    out = torch.zeros(nseg * k, dtype=torch.int64, device=dev)
    call = lambda: _lib.call("sseqs_topk_segments", x.data_ptr(), _lib.F16, begin.data_ptr(), nn.data_ptr(),  # noqa: E731
                             kk.data_ptr(), base.data_ptr(), nseg, k, 0, 0, 0, 0, out.data_ptr(), _lib.stream_of(dev))
    want = lambda: torch.cat([torch.sort(torch.sort(s, descending=True, stable=True).indices[:k]).values  # noqa: E731
                              for s in x.view(nseg, n)])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for i in range(3):
        x.copy_(torch.randn(nseg * n, generator=g, device=dev).half())
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want()), i
