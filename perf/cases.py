"""The calls whose speed users of this library see, over the sizes they come in.

Every case goes through the C ABI of include/tweakalign.h (as tweakseq_amd binds it) with host letters or
resident sequences in and scores, coordinates and CIGAR text out.  `listed()` are the cases measured, `draw`
gives others of the same ranges, `prepare` makes what a program holds before the call, `run` is one call,
`work` what it cannot do without, and `exact` the answer in plain numpy where that is quick.
"""
import ctypes
import math
import time

import numpy as np

import tweakseq_amd as ta
from tweakseq_amd import engine as te

PAIR = np.dtype([("a", "u8"), ("la", "i4"), ("p0", "i4"), ("b", "u8"), ("lb", "i4"), ("p1", "i4")])
SEQ_PAIR = np.dtype([("a", "i8"), ("b", "i8")])
RESULT = np.dtype([("score", "i4"), ("a_begin", "i4"), ("a_end", "i4"), ("b_begin", "i4"), ("b_end", "i4"),
                   ("p0", "i4"), ("cigar_off", "i8"), ("cigar_len", "i4"), ("flags", "i4")])
FIELDS = [n for n in RESULT.names if n != "p0"]

AMINO = "ARNDCQEGHILKMFPSTWYV"
# background frequencies of BLOSUM62 (Henikoff & Henikoff 1992), in the order of AMINO
AMINO_FREQ = [.074, .052, .045, .053, .025, .034, .054, .074, .026, .068,
              .099, .058, .025, .047, .039, .057, .051, .013, .032, .073]
AMINO_DRAW = np.frombuffer(AMINO.encode(), np.uint8)[
    np.minimum(np.searchsorted(np.cumsum(AMINO_FREQ) / np.sum(AMINO_FREQ), np.arange(65536) / 65536, "right"), 19)]


# ---------------------------------------------------------------------------------------------------------
# the cases
def listed():
    return [
        # "Realign selection" of two rows in the editor, from a few residues to a whole domain: one call, one
        # pair, the user waits for it.
        dict(name="pair_short", kind="pair", la=24, lb=28, alphabet="protein", mode="global", related=True),
        dict(name="pair_realign", kind="pair", la=300, lb=320, alphabet="protein", mode="global", related=False),
        dict(name="pair_dna_local", kind="pair", la=400, lb=420, alphabet="dna", mode="local", related=True),
        # ... and two whole genes.
        dict(name="pair_gene", kind="pair", la=1500, lb=1571, alphabet="protein", mode="global", related=True),
        # One request of a service: a handful of pairs of very unequal lengths, letters in, CIGARs out.
        dict(name="request_ragged", kind="batch", pairs=16, lo=50, hi=5000, alphabet="protein", mode="global",
             related=False),
        # A search: many homologous pairs, log-normal protein lengths, held on the device, results fetched.
        dict(name="search_65536", kind="held", pairs=65536, median=350, alphabet="protein", mode="local"),
        # Short reads against their windows, one call, letters in, CIGARs out.
        dict(name="reads_24000", kind="batch", pairs=24000, lo=100, hi=250, alphabet="dna", mode="local",
             related=True),
        # The all-against-all scores behind a guide tree, on sequences added once.
        dict(name="all_vs_all_512", kind="all_vs_all", seqs=512, lo=100, hi=600),
        # Long DNA (contigs against a reference), linear-memory path, CIGARs.
        dict(name="long_dna_48", kind="batch", pairs=48, lo=10000, hi=60000, alphabet="dna", mode="global",
             related=True),
        # A burst of requests on resident sequences through the serving queue, submitted together.
        dict(name="serve_64", kind="serve", requests=64, mean_pairs=8, lo=50, hi=2500),
        # "Align all": a progressive multiple alignment.
        dict(name="msa_512", kind="msa", seqs=512, lo=100, hi=600),
        # The consensus row under an alignment.
        dict(name="consensus_512x2000", kind="consensus", seqs=512, cols=2000),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pair", "pair", "batch", "batch", "held", "all_vs_all", "long", "serve", "msa", "consensus"])
    alphabet, mode = rng.choice(["protein", "dna"]), rng.choice(["global", "local"])
    if kind == "pair":
        la = spread(10, 1600)
        return dict(kind="pair", la=la, lb=max(8, int(la * rng.uniform(0.6, 1.5))), alphabet=alphabet, mode=mode,
                    related=rng.random() < 0.7)
    if kind == "batch":
        hi = spread(60, 5000)
        most = max(2, min(24000, int(5e9 / hi ** 2)))
        return dict(kind="batch", pairs=spread(2, most), lo=max(1, int(hi * rng.uniform(0.01, 0.8))), hi=hi,
                    alphabet=alphabet, mode=mode, related=rng.random() < 0.7)
    if kind == "held":
        median = spread(60, 350)
        return dict(kind="held", pairs=spread(512, 65536), median=median, alphabet=alphabet, mode=mode)
    if kind == "all_vs_all":
        return dict(kind="all_vs_all", seqs=spread(16, 512), lo=rng.randint(20, 100), hi=rng.randint(120, 600))
    if kind == "long":
        hi = spread(12000, 60000)
        return dict(kind="batch", pairs=rng.randint(1, 48), lo=8000, hi=hi, alphabet="dna", mode="global",
                    related=True)
    if kind == "serve":
        return dict(kind="serve", requests=spread(2, 64), mean_pairs=rng.randint(1, 8), lo=rng.randint(20, 100),
                    hi=spread(300, 2500))
    if kind == "msa":
        return dict(kind="msa", seqs=spread(3, 512), lo=rng.randint(30, 100), hi=rng.randint(130, 600))
    return dict(kind="consensus", seqs=spread(2, 2000), cols=spread(50, 8000))


# ---------------------------------------------------------------------------------------------------------
# inputs
def letters(rng, alphabet, n):
    if alphabet == "dna":
        return np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, n)]
    return AMINO_DRAW[rng.integers(0, 65536, n, dtype=np.uint16)]


def starts(lens):
    return np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)


def mutate(rng, alphabet, seq, lens, psub, pindel, mean=3.0):
    """Homologues of the sequences laid end to end in `seq`: substitutions, and indels of geometric length."""
    n = len(seq)
    s = np.where(rng.random(n, np.float32) < psub, letters(rng, alphabet, n), seq)
    at = np.flatnonzero(rng.random(n, np.float32) < pindel)
    run = rng.geometric(1.0 / mean, len(at))
    ins = rng.random(len(at)) < 0.5
    count = np.ones(n, np.int64)
    edge = np.bincount(at[~ins], minlength=n + 1) - np.bincount(np.minimum(at[~ins] + run[~ins], n), minlength=n + 1)
    count[np.cumsum(edge[:n]) > 0] = 0
    count[starts(lens)] = 1  # no sequence vanishes
    count[at[ins]] += run[ins]
    out = np.repeat(s, count)
    first = np.cumsum(count) - count
    fresh = np.ones(len(out), bool)
    fresh[first[count > 0]] = False
    out[fresh] = letters(rng, alphabet, int(fresh.sum()))
    return out, np.add.reduceat(count, starts(lens))


def lengths(case, rng, n):
    if "median" in case:
        return np.clip(np.round(np.exp(np.log(case["median"]) + 0.6 * rng.standard_normal(n))), 30, 2000).astype(int)
    return rng.integers(case["lo"], case["hi"] + 1, n)


def pair_letters(case, rng):
    """Both sides of a case's pairs: (letters, lengths) of the a's and of the b's, laid end to end."""
    alphabet = case["alphabet"]
    la = np.array([case["la"]]) if "la" in case else lengths(case, rng, case["pairs"])
    a = letters(rng, alphabet, int(la.sum()))
    if case.get("related", True):
        psub, pindel = (0.10, 0.02) if alphabet == "dna" else (0.25, 0.04)
        b, lb = mutate(rng, alphabet, a, la, psub, pindel)
        if "lb" in case:  # cut or extended to its length
            b = np.concatenate([b, letters(rng, alphabet, case["lb"])])[:case["lb"]]
            lb = np.array([case["lb"]])
    else:
        lb = np.array([case["lb"]]) if "lb" in case else lengths(case, rng, case["pairs"])
        b = letters(rng, alphabet, int(lb.sum()))
    return (a, la), (b, lb)


def family(case, rng):
    """Sequences of one family: three in ten descend from an earlier one."""
    seqs = []
    for _ in range(case["seqs"]):
        if seqs and rng.random() < 0.3:
            p = seqs[rng.integers(0, len(seqs))]
            seqs.append(mutate(rng, "protein", p, np.array([len(p)]), 0.20, 0.05)[0])
        else:
            seqs.append(letters(rng, "protein", int(rng.integers(case["lo"], case["hi"] + 1))))
    return seqs


def params(case, traceback=1):
    dna = case.get("alphabet") == "dna"
    mode = ta.LOCAL if case.get("mode") == "local" else ta.GLOBAL
    return te.make_params(mode=mode, alphabet=ta.DNA if dna else ta.PROTEIN, gap_open=-5 if dna else -11,
                          gap_extend=-2 if dna else -1, match=2, mismatch=-3, traceback=traceback)


def pair_array(a, la, b, lb):
    p = np.zeros(len(la), PAIR)
    p["a"], p["la"] = a.ctypes.data + starts(la).astype(np.uint64), la
    p["b"], p["lb"] = b.ctypes.data + starts(lb).astype(np.uint64), lb
    return p


ENGINE = None


def engine():
    """The program's context on the GPU."""
    global ENGINE
    if ENGINE is None:
        ENGINE = ta.Engine(0)
    return ENGINE


def text_room(case, n):
    """Bytes of CIGAR text set aside for n pairs: a byte for every residue of both sides, by the case's longest (or,
    where lengths are log-normal, by 1.2 times their median: the mean)."""
    return int(n * (2.4 * case["median"] if "median" in case else 2.5 * case.get("hi", 0) + 2 * case.get("la", 0)
                    + 2 * case.get("lb", 0))) + 64


class Out:
    """The buffers a program hands to the calls: results of n pairs and `cap` bytes of CIGAR text."""

    def __init__(self, n, cap):
        self.res = np.zeros(n, RESULT)
        self.text = np.zeros(max(cap, 1), np.uint8)
        self.used = ctypes.c_int64()
        self.views = {f: self.res[f] for f in FIELDS}
        self.args = (ctypes.cast(self.res.ctypes.data, ctypes.POINTER(te.CResult)),
                     ctypes.cast(self.text.ctypes.data, ctypes.c_char_p), cap, ctypes.byref(self.used))

    def take(self, cigars=True):
        return dict(self.views, cigars=self.text) if cigars else dict(self.views)


def rows_of(arr):
    return (ctypes.c_char_p * len(arr))(*[ctypes.cast(r.ctypes.data, ctypes.c_char_p) for r in arr])


def prepare(case, seed):
    rng = np.random.default_rng([seed, 7])
    kind = case["kind"]
    s = dict(kind=kind, ctx=engine().ctx)
    if kind in ("pair", "batch", "held"):
        (a, la), (b, lb) = pair_letters(case, rng)
        p = pair_array(a, la, b, lb)
        s.update(a=a, b=b, la=int(la[0]), lb=int(lb[0]), pairs=p, n=len(p), params=params(case),
                 arr=ctypes.cast(p.ctypes.data, ctypes.POINTER(te.Pair)), out=Out(len(p), text_room(case, len(p))))
        if kind == "pair":
            s["ptr"] = [ctypes.cast(x.ctypes.data, ctypes.c_char_p) for x in (a, b)]
        if kind == "held":
            view = te._Pairs([])
            view.arr, view.n, view.keep = s["arr"], s["n"], [p, a, b]
            s["batch"] = ta.Batch(engine(), view, s["params"])
    elif kind == "all_vs_all":
        h = np.array([engine().seq_add(x.tobytes()) for x in family(case, rng)], np.int64)
        i, j = np.triu_indices(len(h), 1)
        p = np.zeros(len(i), SEQ_PAIR)
        p["a"], p["b"] = h[i], h[j]
        s.update(pairs=p, n=len(p), params=params(case, traceback=0), out=Out(len(p), 0),
                 arr=ctypes.cast(p.ctypes.data, ctypes.POINTER(te.SeqPair)))
    elif kind == "serve":
        # pairs per request: the quantiles of an exponential of their mean, in random order
        q = (np.arange(case["requests"]) + 0.5) / case["requests"]
        s["requests"] = []
        for count in rng.permutation(np.ceil(-case["mean_pairs"] * np.log(1 - q)).astype(int)):
            lens = rng.integers(case["lo"], case["hi"] + 1, 2 * int(count))
            h = [engine().seq_add(letters(rng, "protein", int(x)).tobytes()) for x in lens]
            p = np.array(list(zip(h[::2], h[1::2])), np.int64).view(SEQ_PAIR).reshape(-1)
            mode = "local" if rng.random() < 0.5 else "global"
            s["requests"].append(dict(pairs=p, n=int(count), params=params(dict(mode=mode)),
                                      arr=ctypes.cast(p.ctypes.data, ctypes.POINTER(te.SeqPair)),
                                      out=Out(int(count), text_room(case, int(count)))))
    elif kind == "msa":
        seqs = [np.ascontiguousarray(x) for x in family(case, rng)]
        lens = np.array([len(x) for x in seqs], np.int32)
        cols = np.zeros(max(int(lens.sum()), int(1.3 * case["hi"] * case["seqs"])), np.int32)
        joins, alen = np.zeros((len(seqs) - 1, 2), np.int32), ctypes.c_int32()
        s.update(seqs=seqs, rows=rows_of(seqs), lens=lens, cols=cols, joins=joins, alen=alen, params=params(case))
    else:
        s.update(seqs=alignment(case, rng), out=np.zeros(case["cols"], np.uint8))
        s["rows"] = rows_of(s["seqs"])
    return s


def alignment(case, rng):
    """Aligned rows with conserved and variable columns and runs of gaps."""
    n, m = case["seqs"], case["cols"]
    rows = np.where(rng.random((n, m)) < rng.random(m) * 0.9, letters(rng, "protein", n * m).reshape(n, m),
                    letters(rng, "protein", m))
    gap = (rng.random((n, (m + 15) // 16)) < 0.15).repeat(16, axis=1)[:, :m]
    return np.ascontiguousarray(np.where(gap, np.uint8(ord("-")), rows))


# ---------------------------------------------------------------------------------------------------------
# the calls
def checked(rc, what):
    if rc < 0:
        raise RuntimeError("%s: %d" % (what, rc))
    return rc


def run(s):
    L, kind, ctx = ta.lib(), s["kind"], s["ctx"]
    if kind == "pair":
        out = s["out"]
        checked(L.ta_align_pair(ctx, ctypes.byref(s["params"]), s["ptr"][0], s["la"], s["ptr"][1], s["lb"],
                                *out.args), "ta_align_pair")
        return out.take()
    if kind == "batch":
        out = s["out"]
        checked(L.ta_align_batch(ctx, ctypes.byref(s["params"]), s["arr"], s["n"], *out.args), "ta_align_batch")
        return out.take()
    if kind == "held":
        out, h = s["out"], s["batch"].h
        checked(L.ta_batch_run(ctx, h), "ta_batch_run")
        checked(L.ta_batch_wait(ctx, h), "ta_batch_wait")
        checked(L.ta_batch_results(ctx, h, *out.args), "ta_batch_results")
        return out.take()
    if kind == "all_vs_all":
        out = s["out"]
        checked(L.ta_align_resident(ctx, ctypes.byref(s["params"]), s["arr"], s["n"], *out.args), "ta_align_resident")
        return out.take(cigars=False)
    if kind == "serve":
        waiting = []
        for r in s["requests"]:
            t = ctypes.c_uint64()
            checked(L.ta_submit_resident(ctx, ctypes.byref(r["params"]), r["arr"], r["n"], ctypes.byref(t)), "submit")
            waiting.append((r, t.value))
        while waiting:
            r, t = waiting[0]
            if checked(L.ta_poll(ctx, t, *r["out"].args), "ta_poll") == te.E_PENDING:
                time.sleep(1e-4)
            else:
                waiting.pop(0)
        return {k: np.concatenate([r["out"].take()[k] for r in sorted(s["requests"], key=lambda r: r["n"])])
                for k in FIELDS + ["cigars"]}
    if kind == "msa":
        checked(L.ta_msa(ctx, ctypes.byref(s["params"]), s["rows"],
                         ctypes.cast(s["lens"].ctypes.data, ctypes.POINTER(ctypes.c_int32)), len(s["lens"]),
                         ctypes.byref(s["alen"]), ctypes.cast(s["cols"].ctypes.data, ctypes.POINTER(ctypes.c_int32)),
                         ctypes.cast(s["joins"].ctypes.data, ctypes.POINTER(ctypes.c_int32))), "ta_msa")
        return {"length": s["alen"].value, "columns": s["cols"], "joins": s["joins"]}
    checked(L.ta_consensus(ctx, s["rows"], len(s["seqs"]), s["seqs"].shape[1], -1.0,
                           ctypes.cast(s["out"].ctypes.data, ctypes.c_char_p)), "ta_consensus")
    return s["out"]


# ---------------------------------------------------------------------------------------------------------
# what a call cannot do without: operations of the recurrence (9 a cell, 10 with the local floor), the letters
# read, the results and CIGAR text written
def work(case):
    kind = case["kind"]
    if kind == "consensus":
        return {"bytes": case["seqs"] * case["cols"] + case["cols"], "flops": 2 * 24 * 24 * case["cols"]}
    mean = sq = None
    if "la" in case:
        n, res, cells = 1, case["la"] + case["lb"], case["la"] * case["lb"]
    else:
        if "median" in case:
            mean, sq = case["median"] * math.exp(0.18), case["median"] ** 2 * math.exp(0.72)
        else:
            lo, hi = case["lo"], case["hi"]
            mean, sq = (lo + hi) / 2, (lo * lo + lo * hi + hi * hi) / 3
        if kind in ("all_vs_all", "msa"):
            n = case["seqs"] * (case["seqs"] - 1) // 2
            res, cells = case["seqs"] * mean, n * mean ** 2
        else:
            n = case["pairs"] if kind != "serve" else case["requests"] * case["mean_pairs"]
            related = case.get("related", kind == "held")
            res, cells = 2 * n * mean, n * (sq if related else mean ** 2)
    ops = cells * (10 if case.get("mode") == "local" else 9)
    if kind == "msa":  # and the joins' profile columns, the shorter of them about one sequence long
        ops += 9 * case["seqs"] * mean ** 2
        return {"bytes": 5 * res + 8 * case["seqs"], "flops": ops}
    return {"bytes": res + RESULT.itemsize * n + (0 if kind == "all_vs_all" else res / 8), "flops": ops}


# ---------------------------------------------------------------------------------------------------------
# exact answers
BLOSUM_ORDER = "ARNDCQEGHILKMFPSTWYVBZX"
BLOSUM62 = """
4
-1 5
-2 0 6
-2 -2 1 6
0 -3 -3 -3 9
-1 1 0 0 -3 5
-1 0 0 2 -4 2 5
0 -2 0 -1 -3 -2 -2 6
-2 0 1 -1 -3 0 0 -2 8
-1 -3 -3 -3 -1 -3 -3 -4 -3 4
-1 -2 -3 -4 -1 -2 -3 -4 -3 2 4
-1 2 0 -1 -3 1 1 -2 -1 -3 -2 5
-1 -1 -2 -3 -1 0 -2 -3 -2 1 2 -1 5
-2 -3 -3 -3 -2 -3 -3 -3 -1 0 0 -3 0 6
-1 -2 -2 -1 -3 -1 -1 -2 -2 -3 -3 -1 -2 -4 7
1 -1 1 0 -1 0 0 0 -1 -2 -2 0 -1 -2 -1 4
0 -1 0 -1 -1 -1 -1 -2 -2 -1 -1 -1 -1 -2 -1 1 5
-3 -3 -4 -4 -2 -2 -3 -2 -2 -3 -2 -3 -1 1 -4 -3 -2 11
-2 -2 -2 -3 -2 -1 -2 -3 2 -1 -1 -2 -1 3 -3 -2 -2 2 7
0 -3 -3 -3 -1 -2 -2 -3 -3 3 1 -2 1 -1 -2 -2 0 -3 -1 4
-2 -1 3 4 -3 0 1 -1 0 -3 -4 0 -3 -3 -2 0 -1 -4 -3 -3 4
-1 0 0 1 -3 3 4 -2 0 -3 -3 1 -1 -3 -1 0 -1 -3 -2 -2 1 4
0 -1 -1 -1 -2 -1 -1 -1 -1 -1 -1 -1 -1 -1 -2 0 0 -2 -1 -1 -1 -1 -1
"""


def blosum():
    m = np.zeros((23, 23), np.int64)
    for r, line in enumerate(BLOSUM62.split("\n")[1:-1]):
        m[r, :r + 1] = m[:r + 1, r] = [int(x) for x in line.split()]
    return m


def exact(case, seed):
    if case["kind"] == "pair":
        (a, _), (b, _) = pair_letters(case, np.random.default_rng([seed, 7]))
        return exact_pair(case, a, b)
    if case["kind"] == "consensus":
        return exact_consensus(alignment(case, np.random.default_rng([seed, 7])))
    return None


def exact_pair(case, a, b):
    """Score and end cell of Gotoh's recurrence, a row at a time (no value here for the CIGAR or the start)."""
    dna, local = case["alphabet"] == "dna", case["mode"] == "local"
    order = "ACGT" if dna else BLOSUM_ORDER
    code = np.zeros(256, np.int64)
    for k, ch in enumerate(order):
        code[ord(ch)] = k
    S = np.where(np.eye(4, dtype=bool), 2, -3) if dna else blosum()
    go, ge = (-5, -2) if dna else (-11, -1)
    m, n = len(a), len(b)
    col = np.arange(n + 1, dtype=np.int64)
    low = np.int64(-1 << 40)
    H = np.zeros(n + 1, np.int64) if local else np.where(col > 0, go + (col - 1) * ge, 0)
    F = np.full(n + 1, low)
    best = (0, -1, -1)
    for i in range(m):
        F = np.maximum(H + go, F + ge)
        base = np.maximum(F, np.concatenate([[low], H[:-1] + S[code[a[i]], code[b]]]))
        base[0] = 0 if local else go + i * ge
        if local:
            base = np.maximum(base, 0)
        E = np.concatenate([[low], (np.maximum.accumulate(base - col * ge) + go - ge)[:-1] + col[1:] * ge])
        H = np.maximum(base, E)
        if local and H.max() > best[0]:
            j = int(np.argmax(H))
            best = (int(H[j]), i, j - 1)
    out = {f: None for f in FIELDS}
    out.update(cigars=None, cigar_off=np.zeros(1, np.int64))
    if local:
        out.update({k: np.array([v], np.int32) for k, v in zip(("score", "a_end", "b_end"), best)})
    else:
        out.update(score=H[-1:].astype(np.int32), a_begin=np.zeros(1, np.int32), b_begin=np.zeros(1, np.int32),
                   a_end=np.array([m - 1], np.int32), b_end=np.array([n - 1], np.int32))
    return out


def exact_consensus(rows):
    """Every residue's summed pairing score per column; the first row of the best score, where half agree."""
    n, m = rows.shape
    cls = np.full(256, 23)
    for k, ch in enumerate(BLOSUM_ORDER):
        cls[ord(ch)] = k
    for ch in "JOU":
        cls[ord(ch)] = 22
    S = np.full((24, 24), -4, np.int64)
    S[:23, :23], S[23, 23] = blosum(), 1
    M = (S > 0).astype(np.int64)
    M[23, :23] = M[:23, 23] = 0
    c = cls[rows]
    count = np.stack([(c == k).sum(0) for k in range(24)])
    score = np.take_along_axis(S @ count - np.diag(S)[:, None], c, 0)
    match = np.take_along_axis(M @ count - np.diag(M)[:, None], c, 0)
    first = np.argmax(score, 0)
    at = np.arange(m)
    return np.where(match[first, at] >= n / 2, rows[first, at], ord("?")).astype(np.uint8)
