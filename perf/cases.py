"""The work that users of this framework have it do, as cases to time.

A case is one read set (or one batch of them) and the calls that a program
makes on it.  Read sets are drawn on the GPU with torch from the same
distributions as genomix_amd/sim.py (uniform genome, 5% of it in 2 kb repeat
copies at 1% divergence, substitution errors, paired reads with insert
500/50) and reach the library as readids text in device memory, except where
a program holds host buffers (a small job's text, FASTQ files).  Node records
are gathered in a device buffer of the program (a host buffer for the small
jobs), merged records in pinned host memory, which is where a writer of files
has them.
"""

import ctypes
import math

import numpy as np
import torch

from genomix_amd import gx, sizer

DEV = "cuda"
REPEAT_LEN, REPEAT_FRAC, REPEAT_DIV = 2000, 0.05, 0.01
INSERT_MEAN, INSERT_SD = 500, 50


def _set(name, op, genome, k, read_len=150, paired=True, coverage=50.0, error=0.01, **more):
    return dict(name=name, op=op, genome=genome, k=k, read_len=read_len, paired=paired, coverage=coverage,
                error=error, **more)


def listed():
    return [
        # One gradient of the sizing network at its training batch (sizer.train): tiny kernels, one
        # after the other, so launches and latency are all there is.
        {"name": "sizer_gradient_256", "op": "gradient", "batch": 256},
        # A virus genome from host text to host records, graph and merge: the smallest job, where
        # launches, read-backs and host work count.
        _set("virus_5kbp_k21", "host", 5_386, 21, read_len=100, paired=False, coverage=30.0, error=0.005),
        # The plain CPU workload's read set (50 kbp, 100 bp single end, 30x, k = 21), the same calls.
        _set("plasmid_50kbp_k21", "host", 50_000, 21, read_len=100, paired=False, coverage=30.0, error=0.005),
        # Graph build into the 8 partitions of a Hyracks job with several output files.
        _set("parts8_500kbp_k31", "build", 500_000, 31, coverage=40.0, parts=8),
        # A paired FASTQ library in host memory: conversion, graph build and merge.
        _set("fastq_1mbp_k25", "fastq", 1_000_003, 25, read_len=100, coverage=30.0),
        # The driver's default pipeline on two-word keys: build, coverage cutoff, merge, then the
        # coverage, tip and bubble steps with their merges, statistics and FASTA of the result.
        _set("assemble_1mbp_k55", "assemble", 1_000_000, 55, coverage=40.0),
        # The same pipeline on the plain GPU workload's read set.
        _set("assemble_5mbp_k31", "assemble", 5_000_000, 31),
        # The headline: graph build and merge of the plain GPU workload (5 Mbp, 150 bp PE, 50x, k = 31).
        _set("merge_5mbp_k31", "merge", 5_000_000, 31),
        # Graph build alone of the largest genome of the batched workload.
        _set("build_10mbp_k31", "build", 10_000_000, 31, coverage=40.0, parts=1),
        # A build in key-range passes whose records go to a sink, as the builds larger than HBM do,
        # two-word keys.
        _set("stream_10mbp_k55", "stream", 10_000_000, 55, coverage=30.0, range_occ=64_000_000),
        # Many small and middling read sets of mixed k in one call (the batched workload's shape).
        {"name": "batch_12_sets", "op": "batch", "sets": 12, "smallest": 50_000, "largest": 1_000_000, "mix": 1},
        # What the driver reports of a built graph: the coverage cutoff over its nodes and the
        # statistics of the merge.
        _set("report_2mbp_k31", "report", 2_000_003, 31),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gradient", "host", "build", "build", "fastq", "assemble", "assemble", "merge", "merge",
                     "stream", "batch", "report"])
    if op == "gradient":
        return {"op": op, "batch": _log(rng, 32, 4096)}
    if op == "batch":
        return {"op": op, "sets": rng.randint(4, 12), "smallest": 50_000, "largest": _log(rng, 200_000, 1_000_000),
                "mix": rng.randint(2, 1 << 30)}
    lo, hi = {"host": (5_000, 100_000), "build": (100_000, 10_000_000), "fastq": (100_000, 2_000_000),
              "assemble": (100_000, 5_000_000), "merge": (100_000, 5_000_000), "stream": (2_000_000, 10_000_000),
              "report": (100_000, 3_000_000)}[op]
    k = rng.choice([21, 25, 31] if op == "report" else [21, 25, 31, 31, 33, 41, 55, 63])
    c = {"op": op, "genome": _log(rng, lo, hi), "k": k, "read_len": rng.choice([100, 125, 150]),
         "paired": op == "fastq" or rng.random() < 0.6, "coverage": round(rng.uniform(20, 50 if hi <= 5_000_000 else 40), 1),
         "error": round(rng.uniform(0.005, 0.01), 4)}
    if op == "build":
        c["parts"] = rng.choice([1, 1, 2, 8, 64])
    if op == "stream":
        c["coverage"] = round(rng.uniform(20, 30), 1)
        c["range_occ"] = _log(rng, 20_000_000, 100_000_000)
    return c


# ---------------------------------------------------------------------------
# read sets
# ---------------------------------------------------------------------------

def _genome(G, gen):
    g = torch.randint(0, 4, (G,), generator=gen, device=DEV, dtype=torch.uint8)
    copies = int(REPEAT_FRAC * G / REPEAT_LEN)
    if copies:
        fam = torch.randint(0, 4, (REPEAT_LEN,), generator=gen, device=DEV, dtype=torch.uint8).repeat(copies, 1)
        fam = _errors(fam, REPEAT_DIV, gen)
        slot = torch.randperm(G // REPEAT_LEN, generator=gen, device=DEV)[:copies]
        at = (slot * REPEAT_LEN)[:, None] + torch.arange(REPEAT_LEN, device=DEV)
        g[at.reshape(-1)] = fam.reshape(-1)
    return g


def _errors(m, rate, gen):
    hit = torch.rand(m.shape, generator=gen, device=DEV) < rate
    by = torch.randint(1, 4, m.shape, generator=gen, device=DEV, dtype=torch.uint8)
    return torch.where(hit, (m + by) % 4, m)


def _rc(m):
    return 3 - m.flip(-1)


def _mates(c, seed):
    """Code matrices [reads, read_len] of a read set: (mate 1, mate 2 or None)."""
    gen = torch.Generator(DEV)
    gen.manual_seed(seed * 1000003 + c["genome"])
    G, L = c["genome"], c["read_len"]
    g = _genome(G, gen)
    n = max(1, int(round(c["coverage"] * G / ((2 if c["paired"] else 1) * L))))
    cols = torch.arange(L, device=DEV)
    rev = (torch.rand(n, generator=gen, device=DEV) < 0.5)[:, None]
    where = torch.rand(n, generator=gen, device=DEV, dtype=torch.float64)
    if not c["paired"]:
        m = g[(where * (G - L + 1)).long()[:, None] + cols]
        return _errors(torch.where(rev, _rc(m), m), c["error"], gen), None
    frag = torch.randn(n, generator=gen, device=DEV) * INSERT_SD + INSERT_MEAN
    frag = frag.round().long().clamp(L, G)
    start = (where * (G - frag + 1)).long()
    a = g[start[:, None] + cols]
    b = _rc(g[(start + frag - L)[:, None] + cols])
    return (_errors(torch.where(rev, b, a), c["error"], gen), _errors(torch.where(rev, a, b), c["error"], gen))


def _digits(x):
    """Decimal digits of the positive integers x as a byte matrix, left-padded with zero bytes."""
    width = len(str(int(x[-1])))
    d = torch.zeros((len(x), width), dtype=torch.uint8, device=DEV)
    for col in range(width - 1, -1, -1):
        d[:, col] = torch.where(x > 0, 48 + x % 10, torch.zeros_like(x)).to(torch.uint8)
        x = x // 10
    return d


def _rows(n, *cols):
    """The rows of byte matrices and constant bytes side by side, zero bytes dropped."""
    ascii_ = torch.tensor(list(b"ACGT"), dtype=torch.uint8, device=DEV)
    out = []
    for c in cols:
        if isinstance(c, bytes):
            out.append(torch.tensor(list(c), dtype=torch.uint8, device=DEV).expand(n, -1))
        elif c[0] == "codes":
            out.append(ascii_[c[1].long()])
        else:
            out.append(c[1])
    flat = torch.cat(out, dim=1).reshape(-1)
    return flat[flat != 0]


def _readids(m1, m2):
    n = len(m1)
    ids = ("digits", _digits(4 * torch.arange(n, device=DEV) + 2))
    if m2 is None:
        return _rows(n, ids, b"\t", ("codes", m1), b"\n")
    return _rows(n, ids, b"\t", ("codes", m1), b"\t", ("codes", m2), b"\n")


def _fastq(m):
    n, L = m.shape
    name = ("digits", _digits(torch.arange(1, n + 1, device=DEV)))
    return _rows(n, b"@r", name, b"\n", ("codes", m), b"\n+\n" + b"I" * L + b"\n").cpu().numpy().tobytes()


def _batch_sets(c):
    """The read sets of a batch: genomes log-uniform, 100 / 150 bp, single or paired, 20-80x, k mixed."""
    rng = np.random.default_rng(c["mix"])
    out = []
    for i in range(c["sets"]):
        G = int(np.exp(rng.uniform(np.log(c["smallest"]), np.log(c["largest"]))))
        out.append({"genome": G, "read_len": int(rng.choice([100, 150])), "paired": bool(rng.random() < 0.5),
                    "coverage": float(rng.uniform(20, 80)), "error": float(rng.uniform(0.005, 0.02)),
                    "k": int(rng.choice([21, 31, 55]))})
    return out


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------

def prepare(case, seed):
    op = case["op"]
    if op == "gradient":
        gen = torch.Generator(DEV)
        gen.manual_seed(seed)
        net = sizer.load()
        return {"op": op, "net": net, "x": torch.randn((case["batch"], net.din), generator=gen, device=DEV),
                "t": torch.randn((case["batch"], net.dout), generator=gen, device=DEV),
                "grad": torch.empty(net.n, device=DEV), "loss": torch.empty(1, device=DEV)}
    if op == "batch":
        sets = _batch_sets(case)
        s = {"op": op, "text": [_readids(*_mates(c, seed + i)) for i, c in enumerate(sets)],
             "files": [_files(dict(c, op="merge")) for c in sets]}
        _hand_over()
        s["batch"] = gx.GraphBatch([{"k": c["k"], "input": (t.data_ptr(), t.numel())}
                                    for c, t in zip(sets, s["text"])])
        return s
    m1, m2 = _mates(case, seed)
    s = {"op": op, "parts": case.get("parts", 1), "file": _files(case)}
    if op == "fastq":
        s["text"] = (_fastq(m1), _fastq(m2))
    elif op == "host":
        s["text"] = _readids(m1, m2).cpu().numpy().tobytes()
    else:
        s["text"] = _readids(m1, m2)
    del m1, m2
    _hand_over()
    s["b"] = b = gx.GraphBuilder(case["k"], nparts=s["parts"])
    if op == "stream":
        b.set_stream(case["range_occ"], _sink(s["file"]["nodes"]))
    if op == "report":
        b.add_reads_device(s["text"].data_ptr(), s["text"].numel())
        b.finish()
        b.run_unitigs()
        del s["text"]
    return s


def _hand_over():
    """Inputs finished and torch's freed scratch given back: the library works on streams and memory of its own."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()


class _File:
    """Where a program gathers one kind of output: a buffer that is kept from pass to pass, and the bytes used."""

    def __init__(self, capacity, where):
        self.bytes = torch.zeros(int(capacity), dtype=torch.uint8, device=DEV if where == "device" else "cpu",
                                 pin_memory=where == "pinned")
        self.used = 0

    def take_device(self, address, n):
        """Appends n device bytes that the library takes back when this returns."""
        if n:
            self.bytes[self.used:self.used + n].copy_(_view(address, n))
            torch.cuda.current_stream().synchronize()
        self.used += n

    def out(self):
        return {"bytes": self.bytes, "used": self.used}


class _Bytes:
    def __init__(self, address, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "|u1", "data": (address, False), "version": 3}


def _view(address, n):
    return torch.as_tensor(_Bytes(address, n), device=DEV)


def _files(case):
    """The buffers for a case's outputs, larger than any read set of its sizes needs."""
    op = case["op"]
    f = {}
    if op in ("host", "build", "merge", "fastq", "assemble", "stream"):
        f["nodes"] = _File(1.25 * _record_bytes(case) + (1 << 16), "host" if op == "host" else "device")
    if op in ("host", "merge", "fastq"):
        f["merged"] = _File(1.6 * _merged_bytes(case) + (1 << 16), "host" if op == "host" else "pinned")
    if op == "assemble":
        f["merged"] = _File(1.6 * _merged_bytes(case) + (1 << 16), "pinned")
        f["fasta"] = _File(4 * case["genome"] + (1 << 16), "host")
    if op in ("assemble", "report"):
        f["bins"] = {name: np.zeros((1 << 14, 2), np.int64) for name in gx.STAT_NAMES}
    return f


def _nodes(handle, parts, file):
    """The node records of every partition, one after the other, and the partitions' sizes."""
    file.used = 0
    sizes = []
    for part in range(parts):
        p, n = ctypes.c_void_p(), ctypes.c_uint64()
        handle._check(gx.lib().gx_build_part_device(handle._h, part, ctypes.byref(p), ctypes.byref(n)))
        file.take_device(p.value, n.value)
        sizes.append(n.value)
    return dict(file.out(), parts=np.array(sizes, dtype=np.int64))


def _into(file, call, handle, *args):
    """What an emit call writes into a host buffer."""
    w = ctypes.c_size_t()
    handle._check(call(handle._h, *args, ctypes.cast(file.bytes.data_ptr(), ctypes.c_char_p), file.bytes.numel(),
                       ctypes.byref(w)))
    file.used = w.value
    return file.out()


def _sink(file):
    def take(part, address, nbytes, nrec):
        file.take_device(address, nbytes)
    return take


def _consumer(s, out):
    def take(i, view):
        f = s["files"][i]
        out[i] = {"nodes": _nodes(view, 1, f["nodes"]),
                  "merged": _into(f["merged"], gx.lib().gx_unitig_emit, view)}
    return take


def _statistics(stats, bins):
    """graph_stats() as arrays: totals and maxima by name, each statistic's bins as (value, count) rows."""
    out = {"totals": np.array([stats.get("totals", {}).get(n, 0) for n in gx.TOTAL_NAMES + gx.STAT_NAMES], np.int64),
           "maximum": np.array([stats.get("maximum", {}).get(n, 0) for n in gx.STAT_NAMES], np.int64)}
    for name in gx.STAT_NAMES:
        rows = stats.get(name + "-bins", {})
        bins[name][:len(rows)] = np.array([(int(v), n) for v, n in rows.items()], np.int64).reshape(-1, 2)
        out[name] = bins[name]
    return out


def _build(s):
    b, text = s["b"], s["text"]
    b.reset()
    if s["op"] == "fastq":
        b.add_fastq(*text)
    elif s["op"] == "host":
        b.add_reads(text)
    else:
        b.add_reads_device(text.data_ptr(), text.numel())
    b.finish()
    return b


def run(state):
    s, op, lib = state, state["op"], gx.lib()
    if op == "gradient":
        m = s["net"]
        m._check(lib.gx_mlp_gradient_noalloc(m.handle, s["x"].data_ptr(), s["t"].data_ptr(), len(s["x"]),
                                             s["grad"].data_ptr(), s["loss"].data_ptr(), None))
        return {"grad": s["grad"], "loss": s["loss"]}
    if op == "batch":
        out = {}
        s["batch"].run(unitigs=True, consumer=_consumer(s, out))
        return {"nodes": [out[i]["nodes"]["bytes"] for i in sorted(out)],
                "merged": [out[i]["merged"]["bytes"] for i in sorted(out)],
                "used": np.array([(out[i]["nodes"]["used"], out[i]["merged"]["used"]) for i in sorted(out)])}
    f = s["file"]
    if op == "report":
        cut = s["b"].coverage_cutoff()
        return {"cutoff": np.array([cut[key] for key in gx.MIXTURE_KEYS]),
                "merged": _statistics(s["b"].graph_stats("unitigs"), f["bins"])}
    if op == "stream":
        f["nodes"].used = 0
        _build(s)
        return f["nodes"].out()
    b = _build(s)
    if op == "build":
        return _nodes(b, s["parts"], f["nodes"])
    if op == "host":
        nodes = _into(f["nodes"], lib.gx_build_emit_part, b, 0)
        b.run_unitigs()
        return {"nodes": nodes, "merged": _into(f["merged"], lib.gx_unitig_emit, b)}
    if op in ("merge", "fastq"):
        b.run_unitigs()
        return {"nodes": _nodes(b, 1, f["nodes"]), "merged": _into(f["merged"], lib.gx_unitig_emit, b)}
    cut = b.coverage_cutoff()["cutoff"]
    b.run_unitigs()
    b.clean_bad_coverage(cut if cut > 0 else 3.0, emit=False)
    b.clean_tips(emit=False)
    b.clean_bubbles(emit=False)
    return {"nodes": _nodes(b, 1, f["nodes"]), "merged": _into(f["merged"], lib.gx_unitig_emit, b),
            "stats": _statistics(b.graph_stats("unitigs"), f["bins"]),
            "fasta": _into(f["fasta"], lib.gx_dump_fasta, b, gx.GRAPHS["unitigs"])}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _bases(c):
    return c["coverage"] * c["genome"]


def _text_bytes(c):
    lines = _bases(c) / (c["read_len"] * (2 if c["paired"] else 1))
    per = c["read_len"] * (2 if c["paired"] else 1) + (10 if c["paired"] else 9)
    return lines * per * (2 if c["op"] == "fastq" else 1)


def _distinct(c):
    """Distinct k-mers: the genome's, and those that hold an error."""
    occ = _bases(c) * max(1, c["read_len"] - c["k"] + 1) / c["read_len"]
    return min(occ, 0.95 * c["genome"] + occ * (1 - (1 - c["error"]) ** c["k"]))


def _record_bytes(c):
    """Node records: header, key, coverage, two edges on average."""
    return _distinct(c) * (42 + 2.5 * math.ceil(c["k"] / 4)) + _head_bytes(c)


def _head_bytes(c):
    return 8 * _bases(c) / c["read_len"]


def _merged_bytes(c):
    """Merged records: about 14 nodes to a record, each with its key, letters and edges."""
    return _distinct(c) / 14 * (100 + 4 * math.ceil(c["k"] / 4)) + _head_bytes(c)


def _cleaned_bytes(c):
    """The cleaned graph: the genome's letters and the reads' heads."""
    return c["genome"] / 4 + _head_bytes(c)


def work(case):
    op = case["op"]
    if op == "gradient":
        n = sizer.DIN * sizer.HIDDEN + sizer.HIDDEN * sizer.HIDDEN + sizer.HIDDEN * sizer.DOUT
        p = n + 2 * sizer.HIDDEN + sizer.DOUT
        return {"bytes": 4 * (case["batch"] * (sizer.DIN + sizer.DOUT) + 2 * p), "flops": 6 * n * case["batch"]}
    if op == "batch":
        each = [work(dict(s, op="merge")) for s in _batch_sets(case)]
        return {"bytes": sum(w["bytes"] for w in each), "flops": 0}
    if op == "report":  # the nodes' keys, counts, masks and head counts, read once
        return {"bytes": _distinct(case) * (8 * math.ceil(case["k"] / 31.5) + 12), "flops": 0}
    n = _text_bytes(case) + _record_bytes(case)
    if op in ("merge", "host", "fastq"):
        n += _merged_bytes(case)
    if op == "assemble":
        n += _cleaned_bytes(case)
    return {"bytes": n, "flops": 0}


# ---------------------------------------------------------------------------
# the computed numbers in 64 bits
# ---------------------------------------------------------------------------

def exact(case, seed):
    if case["op"] == "gradient":
        return _exact_gradient(case, seed)
    if case["op"] == "report":
        return {"cutoff": _exact_cutoff(case, seed), "merged": None}
    return None


def _exact_gradient(case, seed):
    gen = torch.Generator(DEV)
    gen.manual_seed(seed)
    x = torch.randn((case["batch"], sizer.DIN), generator=gen, device=DEV).cpu().double()
    t = torch.randn((case["batch"], sizer.DOUT), generator=gen, device=DEV).cpu().double()
    p = torch.from_numpy(np.load(sizer.WEIGHTS, allow_pickle=False)).double().requires_grad_()
    at, y = 0, x
    for layer, (i, o) in enumerate(((sizer.DIN, sizer.HIDDEN), (sizer.HIDDEN, sizer.HIDDEN), (sizer.HIDDEN, sizer.DOUT))):
        w, bias = p[at:at + i * o].view(o, i), p[at + i * o:at + i * o + o]
        at += i * o + o
        y = y @ w.t() + bias
        if layer < 2:
            y = torch.tanh(y)
    loss = (y - t).square().sum() / (2 * len(x))
    loss.backward()
    return {"grad": p.grad, "loss": loss.detach().reshape(1)}


def _coverage_bins(case, seed):
    """Distinct canonical k-mers by their number of occurrences (k <= 31)."""
    k = case["k"]
    found = []
    for m in _mates(case, seed):
        if m is None:
            continue
        for rows in m.split(1 << 19):
            c = rows.long()
            n = c.shape[1] - k + 1
            f = torch.zeros((len(c), n), dtype=torch.int64, device=DEV)
            r = torch.zeros_like(f)
            for i in range(k):
                f |= c[:, i:i + n] << (2 * i)
                r |= (3 - c[:, i:i + n]) << (2 * (k - 1 - i))
            found.append(torch.minimum(f, r).reshape(-1))
    _, times = torch.unique(torch.cat(found), return_counts=True)
    v, w = torch.unique(times, return_counts=True)
    return v.cpu().numpy().astype(np.float64), w.cpu().numpy().astype(np.float64)


def _exact_cutoff(case, seed, rounds=10):
    """The exponential + normal mixture fitted to the coverages by EM, and the
    first coverage at which the normal component wins."""
    x, w = _coverage_bins(case, seed)
    theta = np.array([5.0, 20.0, 5.0])  # exponential mean, normal mean and deviation
    prior = np.array([0.5, 0.5])

    def weighted(at):
        e = np.exp(-at / theta[0]) / theta[0]
        g = np.exp(-0.5 * ((at - theta[1]) / theta[2]) ** 2) / (theta[2] * math.sqrt(2 * math.pi))
        return np.stack([e * prior[0], g * prior[1]])

    def members():
        d = weighted(x)
        d[d == 0] = 1e-9
        d /= d.sum(axis=0)
        return d * w

    m = members()
    prior = m.sum(axis=1) / m.sum()
    for _ in range(rounds):
        mean = (m * x).sum(axis=1) / m.sum(axis=1)
        sd = math.sqrt((m[1] * (x - mean[1]) ** 2).sum() / m[1].sum()) or float(np.float32(1e-9))
        theta = np.array([mean[0], mean[1], sd])
        m = members()
        prior = m.sum(axis=1) / m.sum()
    scan = np.arange(1.0, x.max())
    d = weighted(scan)
    won = np.nonzero(d[0] < d[1])[0]
    return np.array([scan[won[0]] if len(won) else 0.0, theta[0], theta[1], theta[2], prior[0], prior[1]])
