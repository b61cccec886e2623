"""Timed cases of the framework's public entry points.

A case is a dict of plain values; ``prepare`` makes what a program holds before the call (database, query,
selection, weights), ``run`` is one pass through the public entry points, ``work`` the bytes and operations the
pass cannot do without, and ``exact`` the floating outputs in 64 bits from plain torch.

The kinds, and what each stands for:

* ``sw``       ``sseqs.sw(query, targets)``: scoring a list of target strings, from host strings to scores.
* ``align``    ``sw_affine_backtrack``: the alignments of a search's hits, host strings to host rows (the a3m stage).
* ``ops``      the extension operators on one ASCII batch, as a program written against ``xbit``, ``conv`` and ``sw``
               calls them: unpack, prefilter of every segment, linear SW of a 1/200 selection, affine SW of a tenth.
* ``targets``  ``sw.sw_cuda_affine`` or ``sw.sw_cuda_blosum62`` over a large selection of an unpacked batch.
* ``batches``  ``batch_search``: the cascade that ``msa()`` runs by default over the resident database.
* ``search``   ``global_search`` + ``backtrack_hits``: the whole-database cascade with its alignments.
* ``prefilter``  ``prefilter_scores`` of every database sequence.
* ``topk``     ``topk_indices``: the candidate selection (fp32 prefilter scores, fp16 proposal scores, int32 SW scores).
* ``table``    ``EmbeddingTable``: the encoder over every database sequence, to the FP8 table.
* ``train``    forward, losses and backward of one encoder training step.
* ``ingest``   packing a stream of sequences and indexing it (``xbit.compress``, ``SeqDB.from_packed``).
* ``sweep``    ``MultiSearch`` with the learned proposal: several queries of mixed lengths in one sweep.
"""
import math
from types import SimpleNamespace

import numpy as np
import torch

import sseqs_amd
from sseqs_amd import learned, ops, synth
from sseqs_amd._lib import call, ptr, stream_of
from sseqs_amd.db import SeqDB
from sseqs_amd.multi import MultiSearch
from sseqs_amd.query import prepare as prepare_query
from sseqs_amd.search import (BacktrackWorkspace, backtrack_hits, batch_search, global_search,
                              prefilter_scores)
from sseqs_amd.sw import sw_affine_backtrack

DEV = "cuda"


def listed():
    return [
        # the smallest call: a handful of designed sequences against one query
        {"name": "sw_32", "kind": "sw", "q_len": 120, "n": 32},
        # the alignments behind one a3m file: the default msa() keeps two hits of each 50 MB batch, and
        # a large database has some hundreds of batches
        {"name": "align_1420", "kind": "align", "q_len": 250, "n": 1420},
        # one 50 MB batch of a length-ordered database file through the extension operators
        {"name": "ops_batch", "kind": "ops", "q_len": 200, "n": 261000, "median": 305},
        # a wide selection of such a batch rescored with affine gaps through the operator
        {"name": "targets_40k", "kind": "targets", "q_len": 350, "n": 40000, "linear": False},
        # the default msa() search: 20 M sequences in 50 MB batches
        {"name": "batches_20M", "kind": "batches", "q_len": 200, "n": 20000000},
        # the whole-database cascade at the headline's query length, hits aligned
        {"name": "search_20M", "kind": "search", "q_len": 200, "n": 20000000, "top": 100000, "hits": 4096},
        # the prefilter of a long query (two thirds of the batched workload's queries pass 350 residues)
        {"name": "prefilter_900", "kind": "prefilter", "q_len": 900, "n": 4000000},
        # the candidate selection at full database size
        {"name": "topk_200M", "kind": "topk", "n": 200000000, "k": 100000, "dtype": "f32", "sorted": False},
        # the encoder over a database part, to the FP8 table (embedding is done once for each database)
        {"name": "table_30k", "kind": "table", "n": 30000},
        # one training step of the encoder: 32 queries with 32 targets each, as the training program takes them
        {"name": "train_32x32", "kind": "train", "queries": 32, "pairs": 32},
        # a quarter of the 1 GB chunk in which database files are read
        {"name": "ingest_250MB", "kind": "ingest", "n": 1400000, "sorted": True},
        # a serving sweep: 16 queries of mixed lengths with the learned proposal
        {"name": "sweep_16", "kind": "sweep", "queries": 16, "n": 2000000, "top": 20000, "hits": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sw", "align", "ops", "targets", "batches", "search", "prefilter", "prefilter", "topk",
                       "topk", "table", "train", "ingest", "sweep"])
    if kind == "sw":
        return {"kind": kind, "q_len": _log_int(rng, 20, 1200), "n": _log_int(rng, 1, 4000)}
    if kind == "align":
        return {"kind": kind, "q_len": _log_int(rng, 30, 700), "n": _log_int(rng, 1, 2000)}
    if kind == "ops":
        return {"kind": kind, "q_len": _log_int(rng, 30, 900), "n": _log_int(rng, 3000, 260000),
                "median": _log_int(rng, 60, 300)}
    if kind == "targets":
        return {"kind": kind, "q_len": _log_int(rng, 30, 1300), "n": _log_int(rng, 300, 40000),
                "linear": rng.random() < 0.4}
    if kind == "batches":
        return {"kind": kind, "q_len": _log_int(rng, 50, 600), "n": _log_int(rng, 300000, 15000000)}
    if kind == "search":
        return {"kind": kind, "q_len": _log_int(rng, 50, 600), "n": _log_int(rng, 300000, 12000000),
                "top": _log_int(rng, 8000, 100000), "hits": _log_int(rng, 64, 4096)}
    if kind == "prefilter":
        return {"kind": kind, "q_len": _log_int(rng, 30, 1500), "n": _log_int(rng, 50000, 3000000)}
    if kind == "topk":
        n = _log_int(rng, 2000, 200000000)
        k = min(n, 500000, _log_int(rng, max(1, n // 20000), max(2, n // 8)))
        return {"kind": kind, "n": n, "k": k, "dtype": rng.choice(["f32", "f32", "f16", "i32"]),
                "sorted": k <= 4096 and rng.random() < 0.6}
    if kind == "table":
        return {"kind": kind, "n": _log_int(rng, 100, 25000)}
    if kind == "train":
        return {"kind": kind, "queries": _log_int(rng, 8, 64), "pairs": rng.randint(8, 32)}
    if kind == "ingest":
        return {"kind": kind, "n": _log_int(rng, 5000, 1300000), "sorted": rng.random() < 0.7}
    return {"kind": "sweep", "queries": rng.randint(2, 24), "n": _log_int(rng, 200000, 1500000),
            "top": _log_int(rng, 4000, 16000), "hits": _log_int(rng, 64, 2048)}


# ------------------------------------------------------------- inputs --

def _query(length, seed, qid=0):
    return synth.make_query(int(length), qid, seed=1_000_003 * (int(seed) % 1_000_003) + 17)


def _db(n, queries, seed, hom_period=8):
    return SeqDB.synthetic(int(n), queries, seed=int(seed), device=DEV, hom_period=hom_period)


def _homologs(db, n, seed, width=500):
    """n strings of a database: its homologs first (the hits of a search), cut at `width` as hits are."""
    hom = torch.nonzero(db.extra["hom_query"] >= 0).flatten()
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    ids = hom[torch.randperm(hom.numel(), generator=g, device=DEV)[:n]]
    return db.strings(ids, width)


def _batch(case, seed):
    """An unpacked batch in length order, as the operators see it, and a query."""
    query = _query(case["q_len"], seed)
    if case["kind"] == "ops":
        g = synth.generate_db(case["n"], [query], seed=seed, device=DEV, hom_period=50,
                              median=float(case["median"]), sigma=0.02)
    else:
        g = synth.generate_db(case["n"], [query], seed=seed, device=DEV, hom_period=8)
    s = SimpleNamespace(kind=case["kind"], query=query, q=prepare_query(query, device=DEV), packed=g.packed,
                        n_syms=g.n_syms, off=g.seq_off.to(torch.int32), len=g.seq_len,
                        ends=(g.seq_off + g.seq_len).to(torch.int32))
    s.maxlen = int(g.seq_len.max().item())
    return s


def _corr_size(q_len, length):
    return min(max(1 << (max(q_len, length, 1) - 1).bit_length(), 16), 2048)


def _train_inputs(case, seed):
    rng = np.random.default_rng(seed)
    nq, pairs = case["queries"], case["pairs"]
    lens = rng.integers(50, 1001, size=nq)
    queries = [_query(L, seed, i) for i, L in enumerate(lens)]
    db = _db(40 * nq * pairs, queries, seed, hom_period=2)
    hq = db.extra["hom_query"].cpu().numpy()
    ids, y, own = [], [], []
    for i in range(nq):
        hom = np.nonzero(hq == i)[0]
        h = rng.choice(hom, size=min(pairs // 2, hom.size), replace=False)
        b = rng.choice(np.nonzero(hq < 0)[0], size=pairs - h.size, replace=False)
        ids.append(np.concatenate([h, b]))
        y.append(np.concatenate([rng.uniform(0.1, 0.9, h.size), rng.uniform(0.0, 0.05, b.size)]))
        own.append(np.concatenate([np.full(h.size, 4.0), np.ones(b.size)]))
    P = np.zeros((nq, nq * pairs), np.float32)
    for i in range(nq):
        w = np.exp((y[i] - y[i].max()) / 0.1)
        P[i, i * pairs:(i + 1) * pairs] = w / w.sum()
    return SimpleNamespace(queries=queries, db=db, ids=np.concatenate(ids).astype(np.int64), nq=nq,
                           nt=nq * pairs, y=np.concatenate(y).astype(np.float32),
                           w=np.concatenate(own).astype(np.float32), P=P)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sw":
        query = _query(case["q_len"], seed)
        db = _db(max(64, 4 * case["n"]), [query], seed, hom_period=2)
        return SimpleNamespace(kind=kind, query=query, targets=_homologs(db, case["n"], seed, 1000))
    if kind == "align":
        query = _query(case["q_len"], seed)
        db = _db(max(64, 4 * case["n"]), [query], seed, hom_period=2)
        return SimpleNamespace(kind=kind, query=query, targets=_homologs(db, case["n"], seed))
    if kind == "ops":
        s = _batch(case, seed)
        n = case["n"]
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        pick = torch.randperm(n, generator=g, device=DEV)[: max(1, n // 200)]
        s.good = torch.sort(pick).values.to(torch.int32)
        s.good2 = s.good[torch.randperm(s.good.numel(), generator=g, device=DEV)[: max(1, n // 2000)]].contiguous()
        s.N = _corr_size(case["q_len"], s.maxlen)
        s.rfft = torch.zeros(1, dtype=torch.float16, device=DEV)
        return s
    if kind == "targets":
        s = _batch(case, seed)
        s.ascii = ops.decompress(s.packed, s.n_syms, 0)
        s.good = torch.arange(case["n"], dtype=torch.int32, device=DEV)
        s.linear = case["linear"]
        return s
    if kind in ("batches", "search", "prefilter"):
        query = _query(case["q_len"], seed)
        db = _db(case["n"], [query], seed)
        s = SimpleNamespace(kind=kind, query=query, q=prepare_query(query, device=DEV), db=db)
        db.length_ranges(case["q_len"])
        if kind == "batches":
            db.batch_plan(50_000_000)
        if kind == "search":
            s.top, s.hits = case["top"], case["hits"]
            s.ws = BacktrackWorkspace(case["hits"], case["q_len"], 500, db.device)
        return s
    if kind == "topk":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        x = torch.randn(case["n"], generator=g, device=DEV)
        if case["dtype"] == "f16":      # proposal scores: 256 * cosine
            x = (x * 18.0).to(torch.float16)
        elif case["dtype"] == "i32":    # affine scores of candidates
            x = (x * 9.0 + 42.0).clamp_(min=0).to(torch.int32)
        else:                           # prefilter scores
            x = x * 2.5 + 21.0
        return SimpleNamespace(kind=kind, x=x, k=case["k"], sorted=case["sorted"])
    if kind == "table":
        db = _db(case["n"], [_query(300, seed, i) for i in range(4)], seed)
        return SimpleNamespace(kind=kind, enc=learned.Encoder.load(device=DEV), db=db)
    if kind == "train":
        t = _train_inputs(case, seed)
        enc = learned.Encoder.load(device=DEV)
        qcode, qmask, qrows = enc.rows_of_strings(t.queries)
        tcode, tmask, trows = enc.rows_of_db(t.db, t.ids)
        rows = learned.Rows(qrows.M + trows.M, torch.cat([qrows.row0, trows.row0 + qrows.M]),
                            torch.cat([qrows.length, trows.length]),
                            np.concatenate([qrows.row0_h, trows.row0_h + qrows.M]),
                            np.concatenate([qrows.len_h, trows.len_h]))
        dev = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
        enc.g = torch.zeros_like(enc.p)
        return SimpleNamespace(kind=kind, enc=enc, code=torch.cat([qcode, tcode]), mask=torch.cat([qmask, tmask]),
                               rows=rows, nq=t.nq, nt=t.nt, y=dev(t.y), w=dev(t.w), P=dev(t.P),
                               qi=dev(np.repeat(np.arange(t.nq, dtype=np.int32), t.nt // t.nq)),
                               ti=torch.arange(t.nq, t.nq + t.nt, dtype=torch.int32, device=DEV),
                               G=torch.empty((t.nq, t.nt), dtype=torch.float32, device=DEV))
    if kind == "ingest":
        db = _db(case["n"], [_query(200, seed)], seed)
        ascii = ops.decompress(db.packed, db.n_syms, 0)
        if not case["sorted"]:
            db2, _ = synth.shuffled_copy(db, seed=int(seed))
            ascii = ops.decompress(db2.packed, db2.n_syms, 0)
        return SimpleNamespace(kind=kind, ascii=ascii)
    rng = np.random.default_rng(seed)
    lens = rng.integers(50, 1001, size=case["queries"])
    lens[0] = 1000  # the longest query sets the width of the alignment rows
    queries = [_query(L, seed, i) for i, L in enumerate(lens)]
    db = _db(case["n"], queries, seed)
    tab = learned.EmbeddingTable(learned.Encoder.load(device=DEV), db, rows=16_000_000)
    ms = MultiSearch(db, queries, top_prefilter=case["top"], top_hits=case["hits"],
                     proposer=learned.Proposer(tab))
    return SimpleNamespace(kind=kind, ms=ms)


# --------------------------------------------------------------- pass --

def run(s):
    if s.kind == "sw":
        return sseqs_amd.sw(s.query, s.targets)
    if s.kind == "align":
        return sw_affine_backtrack(s.query, s.targets, rows=True)
    if s.kind == "ops":
        ascii = ops.decompress(s.packed, s.n_syms, 0)
        corr = torch.empty(s.len.numel(), dtype=torch.float16, device=DEV)
        ops.warp_corr(corr, s.q.qrev, s.q.lut_a, s.q.lut_b, ascii, s.off, s.len, s.q.k, len(s.query), s.maxlen,
                      s.N, s.rfft)
        lin = ops.sw_cuda_blosum62(s.q.codes, s.good, ascii, s.ends, gap_penalty_param=-1)
        aff = ops.sw_cuda_affine(s.q.codes, s.good2, ascii, s.ends, 11, 1)
        return {"ascii": ascii, "corr": corr, "linear": lin, "affine": aff}
    if s.kind == "targets":
        if s.linear:
            return ops.sw_cuda_blosum62(s.q.codes, s.good, s.ascii, s.ends, gap_penalty_param=-4)
        return ops.sw_cuda_affine(s.q.codes, s.good, s.ascii, s.ends, 11, 1)
    if s.kind == "batches":
        hits = batch_search(s.db, s.query, s.q, bs=50_000_000)
        text = np.zeros((len(hits), 500), np.uint8)
        for row, h in zip(text, hits):
            row[: len(h.seq)] = np.frombuffer(h.seq.encode("latin-1"), np.uint8)
        return {"norm": np.array([h.norm for h in hits], np.float32),
                "affine": np.array([h.affine for h in hits], np.int64),
                "linear": np.array([h.linear for h in hits], np.int64),
                "fft": np.array([h.fft for h in hits], np.float32),
                "text": text}
    if s.kind == "search":
        gh = global_search(s.db, s.q, top_prefilter=s.top, top_hits=s.hits)
        al = backtrack_hits(s.db, s.q, gh.ids, s.ws)
        return {"prefilter": gh.prefilter, "ids": gh.ids, "scores": gh.scores, "info": al.info, "q": al.out_q,
                "t": al.out_t}
    if s.kind == "prefilter":
        return prefilter_scores(s.db, s.q)
    if s.kind == "topk":
        return ops.topk_indices(s.x, s.k, sorted=s.sorted)
    if s.kind == "table":
        return learned.EmbeddingTable(s.enc, s.db).table.view(torch.float8_e4m3fn)
    if s.kind == "train":
        enc = s.enc
        e, znorm, buf = enc.forward(s.code, s.mask, s.rows, train=True)
        de = torch.zeros_like(e)
        loss = torch.zeros(1, dtype=torch.float32, device=DEV)
        st = stream_of(e.device)
        call("sseqs_enc_pair_loss", ptr(e), s.nq + s.nt, ptr(s.qi), ptr(s.ti), ptr(s.y), ptr(s.w), s.nt, ptr(de),
             None, ptr(loss), st)
        call("sseqs_enc_infonce", ptr(e), s.nq, s.nt, ptr(s.P), 0.05, 1.0 / s.nq, ptr(s.G), ptr(de), ptr(loss), st)
        enc.g.zero_()
        enc.backward(de, e, znorm, s.code, s.mask, s.rows, buf)
        return {"e": e, "loss": loss, "grad": enc.g}
    if s.kind == "ingest":
        packed = ops.compress(s.ascii)
        db = SeqDB.from_packed(packed, s.ascii.numel())
        return {"packed": packed, "off": db.seq_off, "len": db.seq_len}
    s.ms.run()
    return {"cand": s.ms.cand, "cand_scores": s.ms.cs, "ids": s.ms.hit_ids, "scores": s.ms.hit_sc,
            "info": s.ms.info, "q": s.ms.out_q, "t": s.ms.out_t}


# --------------------------------------------------------------- work --

# Integer operations of one dynamic programming cell: affine (five maxima, three gap subtractions, one score
# addition) and linear gaps (three maxima, one subtraction, one addition).
AFFINE_OPS, LINEAR_OPS = 9, 5
# The encoder's products for one row: three convolutions of width 9.
ENC_FLOPS = 2.0 * 9 * (64 * 128 + 128 * 128 + 128 * 256)


def _prefilter_flops(q_len, cls, k=4):
    """FFT-equivalent operations of the correlations: k real transforms, products and one inverse."""
    N = np.array([_corr_size(q_len, int(L)) for L in cls.length])
    H = N / 2.0
    return float((cls.count * k * (10 * H * np.log2(H) + 20 * H)).sum())


def work(case):
    kind = case["kind"]
    n, q_len = case.get("n", 0), case.get("q_len", 0)
    if kind in ("sw", "align"):
        res = 284.0 * n
        out = 4.0 * n if kind == "sw" else n * (2 * 250 + 24)
        return {"bytes": res + q_len + out, "flops": AFFINE_OPS * q_len * res}
    if kind == "topk":
        return {"bytes": {"f32": 4.0, "i32": 4.0, "f16": 2.0}[case["dtype"]] * n + 8.0 * case["k"], "flops": n}
    if kind == "ops":
        cls = synth.length_classes(n, median=float(case["median"]), sigma=0.02)
        N = _corr_size(q_len, int(cls.length.max()))
        syms = float(cls.n_syms)
        flops = n * 4 * (10 * (N / 2) * math.log2(N / 2) + 20 * (N / 2))
        flops += q_len * case["median"] * (LINEAR_OPS * (n // 200) + AFFINE_OPS * (n // 2000))
        return {"bytes": syms * 5 / 8 + syms + 10.0 * n, "flops": flops}
    if kind == "train":
        rows = 532.0 * case["queries"] + 288.0 * case["queries"] * case["pairs"]
        return {"bytes": rows + 3 * 4.0 * 518784, "flops": 3 * ENC_FLOPS * rows}
    cls = synth.length_classes(n)
    syms, packed = float(cls.n_syms), cls.n_syms * 5 / 8
    if kind == "targets":
        return {"bytes": syms + 12.0 * n, "flops": (LINEAR_OPS if case["linear"] else AFFINE_OPS) * q_len * syms}
    if kind == "table":
        return {"bytes": packed + 12.0 * n + 256.0 * n, "flops": ENC_FLOPS * syms}
    if kind == "ingest":
        return {"bytes": syms + packed + 12.0 * n, "flops": syms}
    if kind == "prefilter":
        return {"bytes": packed + 16.0 * n, "flops": _prefilter_flops(q_len, cls)}
    if kind == "batches":
        cells = q_len * syms
        return {"bytes": packed + 16.0 * n,
                "flops": _prefilter_flops(q_len, cls) + cells * (LINEAR_OPS / 200 + AFFINE_OPS / 2000)}
    if kind == "search":
        sw = AFFINE_OPS * q_len * 284.0 * (min(case["top"], n) + case["hits"])
        return {"bytes": packed + 16.0 * n + case["hits"] * 2.0 * (q_len + 300),
                "flops": _prefilter_flops(q_len, cls) + sw}
    pairs = case["queries"] * 1.0 * (case["top"] + case["hits"])
    return {"bytes": 256.0 * n + pairs * 200, "flops": 2.0 * 256 * n * case["queries"] + AFFINE_OPS * pairs * 525 * 330}


# -------------------------------------------------------------- exact --

AA = "ARNDCQEGHILKMFPSTWYV"


def _letters(packed, off, length, width):
    """ASCII - 64 of sequences at symbol offsets `off`, [n, width], -1 past each length."""
    pos = off[:, None] + torch.arange(width, device=off.device)[None, :]
    keep = torch.arange(width, device=off.device)[None, :] < length[:, None]
    bit = torch.where(keep, pos, off[:, None]) * 5
    byte = bit >> 3
    word = (packed[byte].to(torch.int32) << 8) | packed[byte + 1].to(torch.int32)
    sym = (word >> (11 - (bit & 7)).to(torch.int32)) & 31
    return torch.where(keep, sym, torch.full_like(sym, -1))


def _residue_codes(missing):
    """Code of each letter index 0..31: 0..19 residues, `missing` for the rest."""
    t = torch.full((33,), missing, dtype=torch.int64)
    for i, a in enumerate(AA):
        t[ord(a) - 64] = i
    return t.to(DEV)


def _corr64(packed, off, length, query, size_of):
    """Prefilter scores in 64 bits: half the largest even entry of the circular convolutions' sum."""
    s = prepare_query(query, device="cpu")
    k = s.k
    A = s.lut_a[:k].double().to(DEV)
    B = torch.cat([s.lut_b[:k].double(), torch.zeros(k, 2, dtype=torch.float64)], 1).to(DEV)  # 21 letters + pads
    pad = B.shape[1] - 1
    codes = _residue_codes(20)
    codes[32] = pad
    qrev = s.qrev.long().to(DEV)
    out = torch.empty(off.numel(), dtype=torch.float64, device=DEV)
    N_of = size_of(length.cpu().numpy())
    for N in np.unique(N_of):
        where = torch.from_numpy(np.nonzero(N_of == N)[0]).to(DEV)
        N = int(N)
        a = torch.zeros(k, N, dtype=torch.float64, device=DEV)
        a[:, : min(qrev.numel(), N)] = A[:, qrev][:, :N]
        fa = torch.fft.rfft(a)
        step = max(1, (1 << 26) // N)
        for c in range(0, where.numel(), step):
            w = where[c:c + step]
            sym = _letters(packed, off[w].long(), length[w].long().clamp(max=N), N)
            code = codes[torch.where(sym < 0, torch.full_like(sym, 32), sym).long()]
            f = torch.zeros(w.numel(), N // 2 + 1, dtype=torch.complex128, device=DEV)
            for r in range(k):
                f += torch.fft.rfft(B[r][code]) * fa[r]
            out[w] = 0.5 * torch.fft.irfft(f, n=N)[:, ::2].max(1).values
    return out


def _encoder64(w, code, mask, row0, length):
    """Unit embeddings in 64 bits of sequences laid out in rows (differentiable in the weights)."""
    m = mask[:, None].to(torch.float64)
    x = w["E"][code.long()] * m
    for name in ("1", "2", "3"):
        xp = torch.nn.functional.pad(x, (0, 0, 4, 4))
        y = w["b" + name]
        for t in range(9):
            y = y + xp[t:t + x.shape[0]] @ w["W" + name][t]
        x = torch.nn.functional.gelu(y, approximate="tanh") * m
    ids = torch.repeat_interleave(torch.arange(row0.numel(), device=DEV), length.long())
    first = torch.cumsum(length.long(), 0) - length.long()
    at = row0.long()[ids] + torch.arange(ids.numel(), device=DEV) - first[ids]
    z = torch.zeros(row0.numel(), x.shape[1], dtype=torch.float64, device=DEV).index_add(0, ids, x[at])
    z = z / length[:, None].double()
    return z / z.norm(dim=1, keepdim=True)


def _weights64(grad=False):
    with np.load(learned.WEIGHTS_PATH) as f:
        return {k: torch.from_numpy(f[k]).double().to(DEV).requires_grad_(grad) for k in f.files}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("search", "prefilter"):
        query = _query(case["q_len"], seed)
        db = _db(case["n"], [query], seed)
        sizes = lambda L: np.maximum(  # noqa: E731
            _corr_size(case["q_len"], 1), np.minimum(2048, 1 << np.ceil(np.log2(np.maximum(L, 1))).astype(np.int64)))
        pre = _corr64(db.packed, db.seq_off, db.seq_len, query, sizes)
        if kind == "prefilter":
            return pre
        return {"prefilter": pre, "ids": None, "scores": None, "info": None, "q": None, "t": None}
    if kind == "ops":
        s = _batch(case, seed)
        N = _corr_size(case["q_len"], s.maxlen)
        corr = _corr64(s.packed, s.off, s.len, s.query, lambda L: np.full(L.shape, N, np.int64))
        return {"ascii": None, "corr": corr, "linear": None, "affine": None}
    if kind == "table":
        db = _db(case["n"], [_query(300, seed, i) for i in range(4)], seed)
        w, out = _weights64(), []
        codes = _residue_codes(20)
        codes[32] = 21
        for c in range(0, db.n, 1000):
            off, ln = db.seq_off[c:c + 1000].long(), db.seq_len[c:c + 1000].long()
            width = int(ln.max()) + 4
            sym = _letters(db.packed, off, ln, width)
            code = codes[torch.where(sym < 0, torch.full_like(sym, 32), sym).long()].reshape(-1)
            row0 = torch.arange(off.numel(), device=DEV) * width
            out.append(_encoder64(w, code, (sym >= 0).reshape(-1), row0, ln))
        return 16.0 * torch.cat(out)
    if kind == "train":
        s = prepare(case, seed)
        w = _weights64(grad=True)
        e = _encoder64(w, s.code, s.mask, s.rows.row0, s.rows.length)
        cos = (e[s.qi.long()] * e[s.ti.long()]).sum(1)
        loss = (s.w.double() * (cos - s.y.double()) ** 2).mean()
        logits = torch.log_softmax(e[: s.nq] @ e[s.nq:].T / 0.05, 1)
        loss = loss - (s.P.double() * logits).sum() / s.nq
        loss.backward()
        grad = torch.cat([w[name].grad.reshape(-1) for name, _ in learned.SHAPES])
        return {"e": e.detach(), "loss": loss.detach().reshape(1), "grad": grad}
    return None
