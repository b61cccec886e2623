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


RING_SHAPES = [(128, 40), (128, 100), (256, 60), (256, 150), (256, 250), (512, 120), (512, 200), (512, 300),
               (512, 500), (1024, 90), (1024, 350), (1024, 450), (1024, 560), (1024, 690), (1024, 820),
               (1024, 1000), (1024, 1500), (2048, 200), (2048, 1100), (2048, 1400), (2048, 1700), (2048, 2000)]


@pytest.mark.parametrize("N,Lq", RING_SHAPES)
def test_rank4_ring(orc, dev, N, Lq):
    """Every shape of the rank-4 ring kernel on an ASCII batch: segments of
    every kind of length (empty, one, chunk edges, the whole N, past it), any
    byte inside them, in order and scattered over the batch (slots, and no
    stage), batches at odd addresses, one segment alone; and on packed spans
    that hold '@'."""
    from sseqs_amd import ops
    from sseqs_amd._lib import call, ptr, stream_of
    announce(f"ring N={N} Lq={Lq}")
    rng = np.random.default_rng(7 * N + Lq)
    query = rand_seq(rng, Lq)
    A, B = orc.weighted_luts(query, 4)
    qrev = orc.encode_query_rev(query)
    t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
    edges = [0, 1, 31, 32, 33, N // 2, N - 32, N - 31, N - 1, N, N + 5]
    lens = np.array(edges + list(rng.integers(1, N + 1, 60)), np.int32)
    for order in ("sorted", "shuffled", "scattered"):
        ln = np.sort(lens) if order == "sorted" else rng.permutation(lens).astype(np.int32)
        gap = 40 * N if order == "scattered" else 1
        off = np.concatenate([[0], np.cumsum(ln + gap)[:-1]]).astype(np.int32)
        letters = np.frombuffer((AA * 20 + "XBZ*-@").encode(), np.uint8)
        flat = letters[rng.integers(0, letters.size, int(off[-1] + ln[-1] + 1))].copy()
        for o, n in zip(off, ln):  # homologous stretches, and bytes that are no letters
            if n > 40:
                q = np.frombuffer(query.encode(), np.uint8)[: int(n)]
                flat[o:o + q.size] = q
            flat[o + int(rng.integers(0, n)) if n else 0] = rng.choice([0, 255, 64, 42, 1])
        maxlen = int(ln.max()) if order != "shuffled" else max(1, N - 40)
        want = orc.corr(qrev, A, B, 4, flat.tobytes(), off, ln, maxlen, N)
        tol = orc.corr_tol(qrev, A, B, 4, flat.tobytes(), off, ln, maxlen, N, want)
        for lead, sel in ((0, slice(None)), (5, slice(None)), (0, slice(3, 4))):
            f = torch.cat([torch.zeros(lead, dtype=torch.uint8, device=dev), t(flat)])[lead:]
            scores = torch.zeros(ln[sel].size, dtype=torch.float16, device=dev)
            ops.warp_corr(scores, t(qrev), t(A), t(B), f, t(off[sel]), t(ln[sel]), 4, Lq, maxlen, N,
                          torch.zeros(1, dtype=torch.float16, device=dev))
            got = scores.float().cpu().numpy()
            assert (np.abs(got - want[sel]) <= tol[sel]).all(), (order, lead)
        # the same symbols packed, as spans that may hold '@' (5 bits hold letters only)
        sym = np.where((flat >= 64) & (flat < 96), flat, 64).astype(np.uint8)
        want = orc.corr(qrev, A, B, 4, sym.tobytes(), off, ln, maxlen, N)
        tol = orc.corr_tol(qrev, A, B, 4, sym.tobytes(), off, ln, maxlen, N, want)
        packed = torch.cat([ops.compress(t(sym)), torch.zeros(64, dtype=torch.uint8, device=dev)])
        out = torch.empty(ln.size, dtype=torch.float32, device=dev)
        lutB = torch.cat([t(B).reshape(-1), torch.zeros(1, device=dev)])
        keep = [t(off.astype(np.int64)), t(ln), t(qrev), t(A), lutB]
        call("sseqs_db_prefilter_spans", ptr(packed), ptr(keep[0]), ptr(keep[1]), 0, ln.size, ptr(keep[2]), Lq,
             ptr(keep[3]), ptr(keep[4]), 21, 4, N, maxlen, ptr(out), stream_of(dev))
        assert (np.abs(out.cpu().numpy() - want) <= tol).all(), order


@pytest.mark.parametrize("Lq", [1, 2, 127, 128, 129, 255, 257, 744, 745, 900])
def test_backtrack_edges(orc, dev, Lq):
    """Alignments around the strips of 128 query rows, the blocks of eight
    steps and the lengths and gap parameters that choose tagged cells: related
    targets with indels, unrelated ones, non-residues, empty ones and the
    largest score there is."""
    from sseqs_amd.sw import sw_affine_backtrack
    announce(f"backtrack edges Lq={Lq}")
    rng = np.random.default_rng(Lq)
    query = rand_seq(rng, Lq, AA + "XB")
    tg = ["W" * 3 + query[5:], query[: Lq // 2] + rand_seq(rng, 9) + query[Lq // 2 + 3:], "", "X" * 7]
    for T in (1, 6, 7, 8, 9, 120, 121, 127, 128, 129, 136, 743, 744, 745, 800):
        part = list(rand_seq(rng, T))
        a = int(rng.integers(0, max(1, Lq - T // 2)))
        piece = query[a: a + T // 2]
        part[T // 4: T // 4 + len(piece)] = piece
        tg.append("".join(part)[:T])
    for q, targets, gaps in ((query, tg, ((11, 1), (0, 0), (1024, 1024), (1025, 3), (-1, 1))),
                             ("W" * Lq, ["W" * 900, "W" * 744, "W" * 8], ((11, 1),)),
                             (query, tg[:10], ((11, 1), (3, 0)))):
        for o, e in gaps:
            _, _, got = sw_affine_backtrack(q, targets, o, e)
            for t, g in zip(targets, got):
                assert g == orc.backtrack(q, t, o, e), (len(t), o, e)


@pytest.mark.parametrize("M,cin,N", [(128, 64, 128), (256, 128, 64), (640, 256, 128), (128 * 251, 128, 256),
                                     (128 * 497, 64, 64), (128 * 481, 256, 128), (128 * 995, 128, 128)])
def test_encoder_conv_tiles(dev, M, cin, N):
    """The convolution's tiled kernels equal its general one (reached by an
    output that is not aligned) bit for bit, for every epilogue, around the
    row counts of their tiles and of the rule between them; both lie within
    bf16's rounding of a product in 64 bits."""
    from sseqs_amd._lib import call, stream_of
    announce(f"conv M={M} cin={cin} N={N}")
    g = torch.Generator(device=dev).manual_seed(M + cin + N)
    bf = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)  # noqa: E731
    A = torch.zeros(M + 8, cin, dtype=torch.bfloat16, device=dev)
    A[4:-4] = bf(M, cin)
    Bt, bias = bf(N, 9 * cin) * (9 * cin) ** -0.5, torch.randn(N, generator=g, device=dev)
    mask = (torch.rand(M, generator=g, device=dev) < 0.9).to(torch.uint8)
    up = bf(M * N + 4)
    rows = torch.arange(0, M, max(1, M // 257), device=dev)
    win = torch.stack([A[rows + t] for t in range(9)], 1).reshape(rows.numel(), -1).double()
    C = win @ Bt.double().T
    m = mask[rows, None].double()
    for epi in (0, 1, 2):
        outs = []
        for shift in (0, 2):  # elements: 4 bytes off in bf16, 8 in fp32
            U, Y = (torch.full((M * N + 8,), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
            Yf = torch.full((M * N + 8,), 7.0, device=dev)
            call("sseqs_enc_conv", A.data_ptr() + 8 * cin, cin, Bt.data_ptr(), M, N, 9 * cin,
                 bias.data_ptr() if epi == 0 else None, mask.data_ptr(),
                 U.data_ptr() + 2 * shift if epi == 0 else None, Y.data_ptr() + 2 * shift if epi < 2 else None,
                 up.data_ptr() if epi == 1 else None, Yf.data_ptr() + 4 * shift if epi == 2 else None, epi,
                 stream_of(A.device))
            for t in (U, Y, Yf):  # nothing before the output or past its end
                assert (t[:shift] == 7).all() and (t[M * N + shift:] == 7).all()
            outs.append([t[shift:M * N + shift].clone() for t in (U, Y, Yf)])
        for a, b in zip(*outs):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), epi
        U, Y, Yf = (t.view(M, N)[rows].double() for t in outs[0])
        if epi == 0:
            want = C + bias.double()
            assert (U - want).abs().max() <= 2.0 ** -8 * want.abs().max()
            want = torch.nn.functional.gelu(want, approximate="tanh") * m
            assert (Y - want).abs().max() <= 2.0 ** -8 * want.abs().max()
        elif epi == 1:
            x = up[:M * N].view(M, N)[rows].double().requires_grad_()
            gelu = torch.nn.functional.gelu(x, approximate="tanh")
            want = C * torch.autograd.grad(gelu.sum(), x)[0] * m
            assert (Y - want).abs().max() <= 2.0 ** -8 * want.abs().max()
        else:
            assert (Yf - C * m).abs().max() <= 2.0 ** -16 * C.abs().max()


@pytest.mark.parametrize("M,cin,cout", [(1, 64, 64), (63, 64, 128), (64, 128, 64), (65, 128, 256), (1025, 64, 64),
                                        (32769, 128, 128), (128 * 700, 128, 256)])
def test_encoder_gradient_sums(dev, M, cin, cout):
    """Weight, bias and embedding gradients around their stages (64 rows, 1024
    rows, 128 rows) against sums in 64 bits, added to what is there; the bias
    gradient also from an odd element's address."""
    from sseqs_amd._lib import call, stream_of
    announce(f"gradient sums M={M} cin={cin} cout={cout}")
    g = torch.Generator(device=dev).manual_seed(M + cin + cout)
    X = torch.zeros(M + 8, cin, dtype=torch.bfloat16, device=dev)
    X[4:-4] = torch.randn(M, cin, generator=g, device=dev)
    flat = torch.randn(M * cout + 1, generator=g, device=dev).to(torch.bfloat16)
    st = stream_of(X.device)
    for shift in (0, 1):
        dU = flat[shift: M * cout + shift].view(M, cout).double()
        db = torch.full((cout,), 3.0, device=dev)
        call("sseqs_enc_bias_grad", flat.data_ptr() + 2 * shift, cout, M, db.data_ptr(), st)
        # fp32 sums of M terms: M 2^-24 of the sum of absolute values is a bound on the rounding
        tol = M * 2.0 ** -24 * dU.abs().sum(0).max() + 1e-6
        assert (db.double() - 3 - dU.sum(0)).abs().max() <= tol
    dU = flat[: M * cout].view(M, cout).double()
    dW = torch.full((9 * cin, cout), 3.0, device=dev)
    call("sseqs_enc_wgrad", X.data_ptr() + 8 * cin, cin, flat.data_ptr(), cout, M, dW.data_ptr(), st)
    for t in range(9):
        x = X[t: t + M].double()
        want, tol = x.T @ dU, (x.abs().T @ dU.abs()).max() * M * 2.0 ** -24 + 1e-6
        assert (dW[t * cin:(t + 1) * cin].double() - 3 - want).abs().max() <= tol, t
    code = torch.randint(0, 22, (M,), generator=g, device=dev).to(torch.uint8)
    dx = torch.randn(M, 64, generator=g, device=dev)
    dE = torch.full((22, 64), 3.0, device=dev)
    call("sseqs_enc_embed_grad", code.data_ptr(), M, dx.data_ptr(), dE.data_ptr(), st)
    want = torch.zeros(22, 64, dtype=torch.float64, device=dev).index_add_(0, code.long(), dx.double())
    want[20:] = 0
    assert (dE.double() - 3 - want).abs().max() <= M * 2.0 ** -24 * dx.abs().double().sum(0).max() + 1e-6


def test_encoder_pool_gradient_rows(dev):
    """The pool's gradient on sequences of 0 to 70 rows (groups of eight rows
    over eight blocks), rows outside them untouched."""
    from sseqs_amd._lib import call, stream_of
    announce("pool gradient rows")
    g = torch.Generator(device=dev).manual_seed(5)
    lens = [0, 1, 7, 8, 9, 63, 64, 65, 70]
    row0 = torch.tensor(np.cumsum([4] + [n + 4 for n in lens[:-1]]), dtype=torch.int64, device=dev)
    M = int(row0[-1]) + lens[-1] + 4
    e = torch.nn.functional.normalize(torch.randn(len(lens), 256, generator=g, device=dev), dim=1)
    de = torch.randn(len(lens), 256, generator=g, device=dev)
    zn = torch.rand(len(lens), generator=g, device=dev) + 0.5
    U = torch.randn(M, 256, generator=g, device=dev).to(torch.bfloat16)
    tl = torch.tensor(lens, dtype=torch.int32, device=dev)
    out = torch.full((M, 256), 7.0, dtype=torch.bfloat16, device=dev)
    call("sseqs_enc_pool_grad", de.data_ptr(), e.data_ptr(), zn.data_ptr(), U.data_ptr(), row0.data_ptr(),
         tl.data_ptr(), len(lens), out.data_ptr(),
         stream_of(e.device))
    torch.cuda.synchronize()
    want = torch.full((M, 256), 7.0, dtype=torch.float64, device=dev)
    x = U.double().requires_grad_()
    gg = torch.autograd.grad(torch.nn.functional.gelu(x, approximate="tanh").sum(), x)[0]
    for s, n in enumerate(lens):
        dz = (de[s].double() - e[s].double() * (e[s].double() @ de[s].double())) / zn[s].double() / max(n, 1)
        want[row0[s]: row0[s] + n] = dz * gg[row0[s]: row0[s] + n]
    # fp32 steps before one rounding to bf16: half a unit of 2^-8, and room for the cancellation in dz
    assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("dtype", ["f16", "f32", "i32"])
@pytest.mark.parametrize("sorted_", [False, True])
def test_topk_segments_cut(dev, dtype, sorted_):
    """Segments around the length (32768) and the counts that choose the cut
    to a list: random, equal, rising and bunched scores (a sample that
    misleads), NaN and infinities, begins of any alignment."""
    from sseqs_amd import ops
    announce(f"topk_segments cut {dtype} sorted={sorted_}")
    rng = np.random.default_rng(3)
    segs = [(n, k, kind) for n in (32767, 32768, 32769 + 512, 70001, 400003) for k in (1, 163, n // 200, 1600, 2049)
            for kind in ("normal", "special")]
    segs += [(50000, 300, "equal"), (50000, 300, "rising"), (50000, 300, "bunched"), (281001, 1405, "ties")]
    parts = []
    for n, k, kind in segs:
        x = rng.normal(21.0, 2.5, n)
        if kind == "equal":
            x[:] = 3.0
        elif kind == "rising":
            x = np.arange(n) / 64.0
        elif kind == "bunched":
            x[1000:1400] += 50.0
        elif kind == "ties":
            x = np.round(x)
        elif kind == "special" and dtype != "i32":
            x[::7], x[3::50], x[5::9] = np.nan, np.inf, -np.inf
        parts.append(x)
    n = np.array([p.size for p in parts])
    begin = np.concatenate([[1], 1 + np.cumsum(n + 1)[:-1]])  # a score between segments
    flat = np.full(int(n.sum() + n.size + 1), 7.0)
    for b, p in zip(begin, parts):
        flat[b: b + p.size] = p
    flat = flat.astype({"f16": np.float16, "f32": np.float32, "i32": np.int32}[dtype])
    k = np.minimum([s[1] for s in segs], 4096)
    got, base = ops.topk_segments(torch.from_numpy(flat).to(dev), begin, n, k, sorted=sorted_)
    got = got.cpu().numpy()
    for j in range(len(segs)):
        x = flat[begin[j]: begin[j] + n[j]].astype(np.float64)
        if dtype != "i32":
            x = np.where(np.isnan(x), -np.inf, np.where(x == -np.inf, -1e300, x))
        want = np.argsort(-x, kind="stable")[: k[j]]
        assert np.array_equal(got[base[j]: base[j] + k[j]], want if sorted_ else np.sort(want)), segs[j]


def test_encoder_gelu_rounding(dev):
    """The tiled kernels' GELU equals the general kernel's on 2^21 values (all
    magnitudes, both signs, the steep range densely) as bias of zero products,
    on rows with and without a mask: no bf16 differs, infinities included."""
    from sseqs_amd._lib import call, stream_of
    announce("gelu rounding")
    g = torch.Generator(device=dev).manual_seed(11)
    bits = torch.randint(-2 ** 31, 2 ** 31, (1 << 20,), generator=g, device=dev, dtype=torch.int64).to(torch.int32)
    vals = torch.cat([bits.view(torch.float32), torch.rand(1 << 20, generator=g, device=dev) * 14 - 9])
    vals = torch.where(torch.isnan(vals), torch.full_like(vals, -float("inf")), vals)
    N, M = 1 << 15, 128
    A = torch.zeros(M + 8, 64, dtype=torch.bfloat16, device=dev)
    Bt = torch.zeros(N, 576, dtype=torch.bfloat16, device=dev)
    mask = (torch.arange(M, device=dev) % 5 != 0).to(torch.uint8)
    for bias in vals.view(-1, N):
        out = []
        for shift in (0, 2):
            Y = torch.empty(M * N + 8, dtype=torch.bfloat16, device=dev)
            call("sseqs_enc_conv", A.data_ptr() + 8 * 64, 64, Bt.data_ptr(), M, N, 576, bias.data_ptr(),
                 mask.data_ptr(), None, Y.data_ptr() + 2 * shift, None, None, 0, stream_of(A.device))
            out.append(Y[shift: M * N + shift])
        a, b = (y.view(torch.int16) for y in out)
        assert torch.equal(torch.isnan(out[0]), torch.isnan(out[1]))
        assert bool(((a == b) | torch.isnan(out[0])).all())


@pytest.mark.parametrize("n", [1, 39, 64, 16384, 16385, 8192 * 16384 // 64 + 7])
def test_packed_stream_without_tail(orc, dev, n):
    """compress and from_packed on streams around the chunks of 32 symbols and
    the index's tiles: bytes equal to the oracle's, no byte of the output left
    as it was allocated, runs as numpy finds them."""
    from sseqs_amd import ops
    from sseqs_amd.db import SeqDB
    announce(f"packed stream n={n}")
    rng = np.random.default_rng(n)
    a = rng.integers(65, 91, n).astype(np.uint8)
    a[rng.random(n) < 0.02] = 64
    a[0] = 65
    torch.full((1 << 20,), 255, dtype=torch.uint8, device=dev)  # what the allocator hands out again
    packed = ops.compress(torch.from_numpy(a).to(dev))
    assert np.array_equal(packed.cpu().numpy(), orc.xbit_pack(a))
    db = SeqDB.from_packed(packed, n)
    d = np.diff(np.concatenate([[0], (a != 64).astype(np.int8), [0]]))
    off, end = np.nonzero(d == 1)[0], np.nonzero(d == -1)[0]
    order = np.argsort(end - off, kind="stable")
    assert np.array_equal(db.seq_off.cpu().numpy(), off[order])
    assert np.array_equal(db.seq_len.cpu().numpy(), (end - off)[order])
    tail = db.packed[(n * 5 + 7) // 8:]
    assert tail.numel() >= 64 and not bool(tail.any())
