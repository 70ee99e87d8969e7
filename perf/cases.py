"""The work a program has this framework do, as cases that can be timed.

Every case goes through the public calls of hbseed with synthetic proteins
(background residue frequencies, log-normal lengths, planted homologs).  The
kinds, and what each stands for:

* search    one new protein query against a resident database: lookup
            tables, scan, results on the host (the drop-in for H_BLAST_pre +
            H_BLAST_get_data), from a short peptide against a small protein
            set to a long protein against a two-million-sequence database;
* translated  a new nucleotide query: six frames, SEG masking, then a search;
* gapped    the preliminary gapped extension of a finished scan, the step
            that consumes its HSPs;
* hits      the same step on HSPs that the caller holds (of a batched or
            served search);
* batch     many queries in one batched search;
* served    a burst of mixed requests to a running server;
* volume    one H-BLAST .hDb volume loaded and searched, as the volume loop
            does;
* packed    packed sequences loaded and searched for the first time.

Outputs are whole numbers (counters, coordinates, scores).  Records come back
in the buffers that the program keeps for them (zero past the records), so a
case's outputs have one size whatever its inputs.
"""
import os
import sys

import numpy as np

_PKG = os.path.abspath("h-blast_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hbseed  # noqa: E402

# Word hits per cell of the query residues x subject residues matrix at
# threshold 11 on background frequencies, and the integer operations a hit
# cannot do without (its diagonal, the distance to the diagonal's last hit,
# the window test, the overlap test, the update).
_HITS_PER_CELL = 0.00207
_OPS_PER_HIT = 5
# Operations of one cell of the gapped extension (three scores' maxima and
# gap updates, the best score, the drop-off test), and the cells of one
# extension at the default drop-off on average (207 rows of 34 columns).
_OPS_PER_GAP_CELL = 8
_CELLS_PER_EXTENSION = 7000

_CONTEXT = None


def _context():
    """The one context a program keeps."""
    global _CONTEXT
    if _CONTEXT is None:
        _CONTEXT = hbseed.Context(0)
    return _CONTEXT


def listed():
    return [
        # a peptide against a small protein set (a plasmid, a phage): launches
        # and the host path are all there is
        {"name": "search_60x1k", "kind": "search", "qlen": 60, "subjects": 1000, "long": False,
         "dense": True},
        # an average protein against one organism's proteins
        {"name": "search_350x20k", "kind": "search", "qlen": 350, "subjects": 20000,
         "long": True, "dense": False},
        # an average protein against a curated database, lengths with a long tail
        {"name": "search_350x200k", "kind": "search", "qlen": 350, "subjects": 200000,
         "long": True, "dense": True},
        # the benchmark's query and database
        {"name": "search_1000x2m", "kind": "search", "qlen": 1000, "subjects": 2000000,
         "long": False, "dense": False},
        # a concatenated query batch as H-BLAST passes it, or a giant protein
        {"name": "search_8001x100k", "kind": "search", "qlen": 8001, "subjects": 100000,
         "long": False, "dense": False},
        # the benchmark's translated query length, SEG masked as BLASTX does by default
        {"name": "translated_1500x500k", "kind": "translated", "nt": 1500, "subjects": 500000,
         "long": False},
        # gapped extension of a scan of a large database
        {"name": "gapped_1000x500k", "kind": "gapped", "qlen": 1000, "subjects": 500000,
         "long": False},
        # gapped extension of caller-held HSPs of one query of a batch
        {"name": "hits_350x50k", "kind": "hits", "qlen": 350, "subjects": 50000, "long": True},
        # a batch of queries (the lengths of the batched benchmark)
        {"name": "batch_48x200k", "kind": "batch", "queries": 48, "subjects": 200000,
         "long": False},
        # a burst of requests to a server, one in five translated
        {"name": "served_20x100k", "kind": "served", "queries": 20, "subjects": 100000,
         "long": False},
        # one volume of an H-BLAST database
        {"name": "volume_500x200k", "kind": "volume", "qlen": 500, "subjects": 200000,
         "long": False},
        # a database from FASTA, first query
        {"name": "packed_350x300k", "kind": "packed", "qlen": 350, "subjects": 300000,
         "long": True},
    ]


def _spread(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "translated", "gapped", "hits", "batch",
                       "served", "volume", "packed"])
    case = {"kind": kind, "long": rng.random() < 0.5}
    if kind == "search":
        case["qlen"] = _spread(rng, 30, 24000)
        # at most the cells of the largest listed search
        case["subjects"] = _spread(rng, 500, min(2000000, 8e8 / case["qlen"]))
        case["dense"] = rng.random() < 0.5
    elif kind == "translated":
        case["nt"] = _spread(rng, 300, 6000)
        case["subjects"] = _spread(rng, 1000, min(500000, 7e8 / (2 * case["nt"])))
    elif kind in ("gapped", "hits"):
        case["qlen"] = _spread(rng, 60, 2000)
        case["subjects"] = _spread(rng, 2000, 500000)
    elif kind == "batch":
        case["queries"] = _spread(rng, 3, 48)
        case["subjects"] = _spread(rng, 5000, 200000)
    elif kind == "served":
        case["queries"] = _spread(rng, 2, 20)
        case["subjects"] = _spread(rng, 5000, 100000)
    else:
        case["qlen"] = _spread(rng, 60, 1000)
        case["subjects"] = _spread(rng, 5000, 300000)
    return case


class _State:
    """What a program holds between its calls; gives device memory back."""

    def __init__(self):
        self.case = None
        self.server = self.scan = self.query = self.db = None

    def __del__(self):
        if self.server is not None:
            self.server.stop()
        for h in (self.scan, self.query, self.db):
            if h is not None:
                h.close()


def _database(seed, case, query):
    """Packed sequences, 5% with a homolog of a query segment planted.  "long":
    a long-tailed length distribution (a few sequences past 10,000)."""
    kw = dict(sigma=0.8, hi=35000) if case["long"] else {}
    return hbseed.make_db(seed * 7919 + 11, case["subjects"], plant_query=query,
                          plant_frac=0.05, **kw)


def _batch_queries(seed, n):
    """The batched workload's lengths: log-normal, median 350, 50-3,000."""
    lens = hbseed.lognormal_lengths(seed * 31 + 7, n, 350.0, 0.7, 50, 3000)
    return [hbseed.random_protein(seed * 100003 + i, int(L)) for i, L in enumerate(lens)]


def _nucleotides(seed, nt_len, source):
    """A nucleotide query with two coding regions like the source protein."""
    rng = np.random.default_rng(seed)
    n = min(100, nt_len // 7)
    at = int(rng.integers(0, max(1, len(source) - n)))
    seg = hbseed.homolog(seed * 7 + 1, source[at:at + n], 0.7, 1)
    return hbseed.blastx_nt(seed * 13 + 1, nt_len, seg, seg[::-1].copy())


def _query_residues(case):
    return {"translated": 2.0 * case.get("nt", 0), "batch": 447.0 * case.get("queries", 0),
            "served": (0.8 * 447.0 + 0.2 * 2 * 1327.0) * case.get("queries", 0)}.get(
                case["kind"], float(case.get("qlen", 0)))


def _residues(case):
    sigma = 0.8 if case["long"] else 0.6
    return case["subjects"] * 300.0 * float(np.exp(sigma * sigma / 2))


def _records(case):
    """Room for the HSPs: several times what chance gives plus the homologs."""
    return 4096 + int(2e-6 * _query_residues(case) * _residues(case) + 0.3 * case["subjects"])


def prepare(case, seed):
    s = _State()
    s.case = case
    ctx = _context()
    kind = case["kind"]
    room = _records(case)
    s.buffers = hbseed.ResultBuffers()
    for name, dtype, n in (("stats", hbseed.STATS_DTYPE, case["subjects"]),
                           ("subj", hbseed.SUBJ_HITS_DTYPE, min(case["subjects"], room)),
                           ("hsps", hbseed.HSP_DTYPE, room),
                           ("gstats", hbseed.GSTATS_DTYPE, case["subjects"]),
                           ("ghsps", hbseed.GHSP_DTYPE, room)):
        s.buffers.get(name, dtype, n)
    n_source = case.get("qlen", 1000)
    source = hbseed.random_protein(seed * 6151 + 3, n_source)
    s.residues, s.offsets = _database(seed, case, source)
    if kind in ("search", "gapped", "hits", "volume", "packed"):
        s.spec = hbseed.blastp_query(source)
    if kind == "volume":
        residues, offsets, _ = hbseed.sort_by_length(s.residues, s.offsets)
        s.n = hbseed.hdb_gpu_seqs(case["subjects"])
        s.volume, s.group_len = hbseed.hdb_pack(residues, offsets, s.n)
        return s
    if kind == "packed":
        return s
    s.db = hbseed.Database(ctx, s.residues, s.offsets)
    s.residues = s.offsets = None
    if kind == "translated":
        s.nt = _nucleotides(seed, case["nt"], source)
    elif kind in ("gapped", "hits"):
        s.query = hbseed.Query(ctx, s.spec)
        s.scan = hbseed.Scan(ctx, s.db, s.query)
        s.scan.wait()
        # the gapped cutoff of an E-value of 10 over query x database, bits from
        # the gapped lambda and K of BLOSUM62 11/1
        space = float(case["qlen"]) * float(s.db.residues)
        s.cutoff = [int(np.ceil(np.log(0.041 * space / 10.0) / 0.267))]
        if kind == "hits":
            s.hsps = s.scan.results()[1]
    elif kind == "batch":
        s.specs = [hbseed.blastp_query(q) for q in _batch_queries(seed, case["queries"])]
    elif kind == "served":
        s.specs = [hbseed.blastp_query(q) for q in _batch_queries(seed, case["queries"])]
        for i in range(0, len(s.specs), 5):
            s.specs[i] = hbseed.blastx_query(_nucleotides(seed + i, 600 + 97 * i, source))
        s.server = hbseed.Server(ctx, s.db)
    return s


def _rows(a):
    """The buffer that holds these records, as rows of whole numbers."""
    a = a.base
    return a.view(np.uint32).reshape(len(a), -1)


def _kept(buffers, name, records, at=0):
    """Records of a call that returns new arrays, put into the kept buffer at
    row `at`; returns the next free row."""
    buffers.get(name, records.dtype, at + len(records))[at:] = records
    return at + len(records)


def _search(ctx, db, spec, buffers, dense):
    query = hbseed.Query(ctx, spec)
    scan = hbseed.Scan(ctx, db, query)
    if dense:
        stats, hsps = scan.results(buffers)
        out = {f: stats.base[f] for f in stats.dtype.names}
        out["hsps"] = _rows(hsps)
    else:
        subjects, hsps, totals = scan.results_compact(buffers)
        out = {"subjects": _rows(subjects), "hsps": _rows(hsps), **totals}
    scan.close()
    query.close()
    return out


def run(s):
    ctx = _context()
    kind = s.case["kind"]
    if kind == "search":
        return _search(ctx, s.db, s.spec, s.buffers, s.case["dense"])
    if kind == "translated":
        spec = hbseed.seg_query(hbseed.blastx_query(s.nt))
        return _search(ctx, s.db, spec, s.buffers, False)
    if kind == "gapped":
        stats, hsps = s.scan.gapped(s.cutoff, out=s.buffers)
        return _rows(stats), _rows(hsps)
    if kind == "hits":
        stats, hsps = hbseed.gapped_search(ctx, s.db, s.spec, s.hsps, s.cutoff)
        _kept(s.buffers, "ghsps", hsps)
        return stats.view(np.uint32), len(hsps), _rows(s.buffers.get("ghsps", hsps.dtype, 0))
    counts, at = [], 0
    if kind == "batch":
        batch = hbseed.Batch(ctx, s.db, group_residues=768)
        ids = [batch.add(spec) for spec in s.specs]
        batch.run()
        for i in ids:
            hsps = batch.results(i)
            counts.append(len(hsps))
            at = _kept(s.buffers, "hsps", hsps, at)
        batch.close()
        return np.array(counts), _rows(s.buffers.get("hsps", hsps.dtype, 0))
    if kind == "served":
        for t in [s.server.submit(spec) for spec in s.specs]:
            s.server.wait(t)
            hsps = s.server.results(t)
            counts.append(len(hsps))
            at = _kept(s.buffers, "hsps", hsps, at)
        return np.array(counts), _rows(s.buffers.get("hsps", hsps.dtype, 0))
    if kind == "volume":
        db = hbseed.Database.from_hdb(ctx, s.volume, 512, 192, s.n, s.group_len)
    else:
        db = hbseed.Database(ctx, s.residues, s.offsets)
    out = _search(ctx, db, s.spec, s.buffers, kind == "volume")
    db.close()
    return out


def work(case):
    n = case["subjects"]
    residues = _residues(case)
    qres = _query_residues(case)
    if case["kind"] in ("gapped", "hits"):
        # about one extension in eight sequences at 1,000 residues; records of
        # 32 bytes in and 40 out, the sequences of those records, 16 bytes of
        # counters per sequence
        ext = 0.12 * n * min(1.0, case["qlen"] / 1000.0)
        return {"bytes": 16.0 * n + ext * (32 + 40 + residues / n),
                "flops": ext * _CELLS_PER_EXTENSION * _OPS_PER_GAP_CELL}
    # the sequences once, 12 bytes of counters each, 30 lookup entries per
    # query residue; loading reads and writes the sequences once more
    nbytes = residues + 12.0 * n + 120.0 * qres
    if case["kind"] in ("volume", "packed"):
        nbytes += 2 * residues
    return {"bytes": nbytes, "flops": _HITS_PER_CELL * _OPS_PER_HIT * qres * residues}
