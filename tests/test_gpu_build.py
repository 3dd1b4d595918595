"""Parity of the HIP graph build with the CPU oracle (byte for byte).

These are the parity tests proper: every case runs the GPU through the C ABI
(libgenomix_gx.so) and compares the record stream with the oracle's P = 1
restatement of the Hyracks build (edge lists in JDK-7 HashSet order), or,
in canonical mode, with the oracle after sorting each edge list.
"""

import glob
import os
import re
import struct

import numpy as np
import pytest

from oracle import oracle

from .conftest import GOLDEN

pytestmark = pytest.mark.gpu

FIXTURES = sorted(glob.glob(os.path.join(GOLDEN, "hyracks", "**", "*.expected.txt"), recursive=True))


@pytest.fixture(scope="module")
def gx():
    import genomix_amd.gx as g
    return g


def gpu_records(gx, text, k, edge_order="jdk7", method=None):
    return gx.build_graph(text, k, edge_order=edge_order, method=method)[0]


def ora_records(text, k):
    return oracle.build_graph(text, k)[0]


def _show_diff(a, b):
    ta = oracle.dump_text(a).splitlines()
    tb = oracle.dump_text(b).splitlines()
    for i, (x, y) in enumerate(zip(ta, tb)):
        if x != y:
            return f"first differing record {i}:\n gpu: {x}\n ora: {y}"
    return f"record counts {len(ta)} vs {len(tb)}"


def assert_same(got, want):
    if got != want:
        pytest.fail(_show_diff(got, want))


@pytest.mark.parametrize("expected", FIXTURES, ids=[os.path.basename(f) for f in FIXTURES])
def test_fixtures_byte_exact(gx, expected):
    text = open(expected.replace(".expected.txt", ".test.txt"), "rb").read()
    k = int(re.search(r"_k(\d+)\.", os.path.basename(expected)).group(1))
    assert_same(gpu_records(gx, text, k), ora_records(text, k))


def _sim(seed, G, L, cov, err, paired, n_mut=0):
    from genomix_amd import sim
    spec = sim.ReadSetSpec(genome_len=G, read_len=L, coverage=cov, error_rate=err, paired=paired,
                           insert_mean=3 * L, insert_sd=L // 4, seed=seed)
    return sim.simulate(spec)


@pytest.mark.parametrize("k", [3, 4, 5, 8, 11, 21, 31, 32, 33, 47, 55, 63])
@pytest.mark.parametrize("paired", [False, True], ids=["se", "pe"])
@pytest.mark.parametrize("method", ["sort", "hash"])
def test_random_reads_byte_exact(gx, k, paired, method):
    text = _sim(1000 + k, G=3000, L=max(k + 20, 70), cov=12, err=0.01, paired=paired)
    assert_same(gpu_records(gx, text, k, method=method), ora_records(text, k))


@pytest.mark.parametrize("k,G,cov", [(21, 20000, 100), (33, 8000, 150)])
def test_repeat_rich_long_replays_byte_exact(gx, k, G, cov):
    # repeat families at low divergence: k-mers with thousands of records and
    # branching neighbours (the long-run replay path)
    from genomix_amd import sim
    spec = sim.ReadSetSpec(genome_len=G, read_len=100, coverage=cov, error_rate=0.01, paired=True,
                           insert_mean=300, insert_sd=30, repeat_frac=0.3, repeat_len=(200, 400),
                           repeat_div=0.01, seed=31337 + k)
    text = sim.simulate(spec)
    want = ora_records(text, k)
    for method in ("sort", "hash"):
        assert_same(gpu_records(gx, text, k, method=method), want)


@pytest.mark.parametrize("k", [4, 9, 31, 55])
def test_oversized_buckets_byte_exact(gx, k):
    # thousands of homopolymer and dinucleotide reads put far more than one
    # LDS bucket's worth of records on a few keys (global-sort fallback)
    rng = np.random.default_rng(k)
    lines = []
    for i in range(2500):
        unit = ["A", "C", "AC", "GT"][i % 4]
        s = (unit * 60)[:rng.integers(k + 5, 110)]
        s = "".join(c if rng.random() > 0.01 else rng.choice(list("ACGT")) for c in s)
        lines.append(f"{4 * i + 2}\t{s}\n")
    text = "".join(lines).encode()
    want = ora_records(text, k)
    for method in ("sort", "hash"):
        assert_same(gpu_records(gx, text, k, method=method), want)


def test_low_complexity_byte_exact(gx):
    # homopolymers and tandem repeats: self loops, palindromes (even k), many
    # records per node, lists of 4
    rng = np.random.default_rng(7)
    lines = []
    for i in range(300):
        unit = "".join(rng.choice(list("ACGT"), size=rng.integers(1, 5)))
        s = (unit * 80)[: rng.integers(20, 90)]
        s = "".join(c if rng.random() > 0.05 else rng.choice(list("ACGT")) for c in s)
        lines.append(f"{4 * i + 2}\t{s}\n")
    text = "".join(lines).encode()
    for k in (3, 4, 6, 9, 16):
        assert_same(gpu_records(gx, text, k), ora_records(text, k))


def test_line_format_edge_cases(gx):
    text = (b"1\tACGTACGTAC\r\n"            # CRLF
            b"2\tacgtNNACGT\tggccAATTGG\n"  # lowercase; invalid mate 0 still stored as mate
            b"3\t\tCCCCGGGGAT\n"            # empty mate 0
            b"4\tTTTTGGGGCC\t\t\n"          # trailing empty fields dropped
            b"5\tGATTACAGAT\r"              # lone CR terminator
            b"5\tGATTACAGAT\n"              # duplicate readId: TreeSet keeps one
            b"6\tACGTACGTAC")               # no final newline
    for k in (3, 5, 9):
        assert_same(gpu_records(gx, text, k), ora_records(text, k))


@pytest.mark.parametrize("bad", [b"1\n", b"1\tACGT\tACGT\tACGT\n", b"x\tACGTACGT\n", b"1\tACG\n", b"\n",
                                 b"2\tACGTAC\n536870912\tACGTACGT\n", b"1\tACGTAC\n\n2\tACGT\n"])
def test_errors_match_reference(gx, bad):
    with pytest.raises(oracle.OracleError):
        oracle.build_graph(bad, 3)
    with pytest.raises(gx.GxError) as e:
        gx.build_graph(bad, 3)
    assert e.value.code == gx.GX_EINPUT


def test_invalid_lines_without_valid_mates_pass(gx):
    text = b"-5\tNNNN\n7\tACGTTT\n"
    assert_same(gpu_records(gx, text, 3), ora_records(text, 3))


def _sorted_lists(records):
    out = []
    for line in oracle.dump_text(records).splitlines():
        f = line.split("\t")
        for i in (1, 2, 3, 4):
            name, v = f[i].split(":", 1)
            if v != "null":
                v = "[" + ",".join(sorted(v[1:-1].split(","))) + "]"
            f[i] = name + ":" + v
        out.append("\t".join(f))
    return out


@pytest.mark.parametrize("k", [3, 21, 55])
def test_canonical_edge_order_mode(gx, k):
    text = _sim(77 + k, G=2000, L=k + 40, cov=15, err=0.02, paired=False)
    got = gpu_records(gx, text, k, edge_order="canonical")
    assert _sorted_lists(got) == _sorted_lists(ora_records(text, k))
    # canonical mode: each list ascending by neighbour k-mer
    for line in oracle.dump_text(got).splitlines():
        for fld in line.split("\t")[1:5]:
            v = fld.split(":", 1)[1]
            if v != "null":
                items = v[1:-1].split(",")
                assert items == sorted(items)


def test_plain_cpu_workload_byte_exact(gx):
    """The 50 kbp / 100 bp / 30x / 0.5% error / k=21 workload, full size."""
    from genomix_amd import sim
    text = sim.simulate(sim.PLAIN_CPU_50KBP)
    assert_same(gpu_records(gx, text, 21), ora_records(text, 21))


def _iter_records(rec):
    off = 0
    while off < len(rec):
        n, kl = struct.unpack(">ii", rec[off:off + 8])
        yield rec[off + 8:off + 8 + kl], rec[off + 8 + kl:off + 8 + n]
        off += 8 + n


def test_plain_gpu_workload_invariants(gx):
    """5 Mbp, 150 bp PE, 50x, 1% error, k=31: size-independent properties at
    full size (the oracle is too slow here): sum of coverage = occurrences,
    one read head per valid mate, keys strictly increasing in KmerPointable
    order, deterministic bytes across runs."""
    from genomix_amd import sim
    text = sim.simulate(sim.PLAIN_GPU_5MBP)
    with gx.GraphBuilder(31) as b:
        b.add_reads(text)
        b.finish()
        rec = b.part_bytes(0)
        st = b.stats()
        b.reset()
        b.add_reads(text)
        b.finish()
        assert b.part_bytes(0) == rec
    nlines = text.count(b"\n")
    assert st["heads"] == 2 * nlines
    assert st["occurrences"] == 2 * nlines * (150 - 31 + 1)
    total_cov = 0
    prev = None
    nrec = 0
    for key, val in _iter_records(rec):
        kb = key[4:]
        rk = kb[::-1]
        assert prev is None or rk > prev
        prev = rk
        total_cov += struct.unpack(">f", val[-4:])[0]
        nrec += 1
    assert nrec == st["distinct"]
    assert total_cov == st["occurrences"]


def _digest_cases():
    import json
    path = os.path.join(GOLDEN, "digests", "plain_gpu_params.json")
    return json.load(open(path))["cases"]


@pytest.mark.parametrize("case", _digest_cases(), ids=lambda c: f"{c['genome_len'] // 1000}kbp")
def test_plain_gpu_params_byte_parity(gx, case):
    """The 5 Mbp workload's parameters (5% in 2 kb repeat copies at 1%, 150 bp
    PE, insert 500/50, 50x, 1% errors, k = 31) at 0.5 and 1 Mbp: graph and
    unitig records byte-identical to the oracle's, whose SHA-256 digests
    tests/golden/make_c2_digests.py recorded (the oracle needs minutes here)."""
    import dataclasses
    import hashlib
    from genomix_amd import sim
    spec = dataclasses.replace(sim.PLAIN_GPU_5MBP, genome_len=case["genome_len"], seed=case["seed"])
    text = sim.simulate(spec)
    assert hashlib.sha256(text).hexdigest() == case["text_sha256"], "simulator output changed"
    graph, merged = gx.build_and_merge(text, case["k"])
    assert len(graph) == case["graph_bytes"]
    assert hashlib.sha256(graph).hexdigest() == case["graph_sha256"]
    assert len(merged) == case["unitigs_bytes"]
    assert hashlib.sha256(merged).hexdigest() == case["unitigs_sha256"]


@pytest.mark.parametrize("k", [9, 21, 31, 55])
@pytest.mark.parametrize("n", [60, 65, 300, 513, 600, 2100, 8200, 16500])
def test_record_bucket_sizes(gx, k, n):
    """One key bucket of about n records (distinct k-mers that share their
    first eight letters) beside small neighbours, and the same with a k-mer
    repeated 600 times in it: groups of buckets and single buckets in a wave,
    each size of block, sub-buckets above a wave's, oversized buckets."""
    import random
    rng = random.Random(1000 * k + n)

    def rc(s):
        return s[::-1].translate(str.maketrans("ACGT", "TGCA"))

    for repeats in (0, 600):
        reads = []
        for i in range(n):
            s = "AACAGATA" + "".join(rng.choice("ACGT") for _ in range(k - 8))
            reads.append(s + "A")  # ends in A: read forward
        one = "AACAGATA" + "C" * (k - 8) + "A"
        reads += [one if rng.random() < 0.5 else rc(one) for _ in range(repeats)]
        for _ in range(40):
            reads.append("".join(rng.choice("ACGT") for _ in range(k + 30)))
        rng.shuffle(reads)
        text = "".join(f"{4 * i + 2}\t{s}\n" for i, s in enumerate(reads)).encode()
        assert gx.build_graph(text, k)[0] == oracle.build_graph(text, k)[0], repeats


@pytest.mark.parametrize("k", [21, 55])
@pytest.mark.parametrize("occ", [2, 4, 5, 45])
@pytest.mark.parametrize("n", [4095, 4096, 4097, 12289])
def test_occurrence_tiles(gx, k, occ, n):
    """About n occurrences in reads of occ k-mers each, every ninth read with
    a letter outside ACGT (no occurrences): tiles of 4096 occurrences, full
    and with a remainder, whose reads fit the tile's tables and do not, in
    few letters so that keys repeat across the tile's waves."""
    import random
    rng = random.Random(n * occ + k)
    genome = "".join(rng.choice("ACGT") for _ in range(900 + k))
    left, reads = n, []
    while left > 0:
        i = len(reads)
        length = k - 1 + max(2, min(occ, left))
        at = rng.randrange(len(genome) - length + 1)
        s = genome[at:at + length]
        if rng.random() < 0.5:
            s = s[::-1].translate(str.maketrans("ACGT", "TGCA"))
        if i % 9 == 5:
            s = s[:3] + "N" + s[4:]
        else:
            left -= length - k + 1
        reads.append(s)
    text = "".join(f"{i + 1}\t{s}\n" for i, s in enumerate(reads)).encode()
    assert gx.build_graph(text, k)[0] == oracle.build_graph(text, k)[0]


@pytest.mark.parametrize("seed", range(6))
def test_line_and_mate_lengths(gx, seed):
    """Mates of every length up to 70, around the multiples of 32 and 128,
    and on both sides of the lengths that a whole wave takes, one or two to a
    line, in any alignment, upper and lower case, with other letters at any
    place, readIds of up to 20 digits and a sign, empty second fields,
    trailing tabs and every line end."""
    import random
    rng = random.Random(seed)
    lengths = [n for n in range(14, 71)] + [95, 96, 97, 127, 128, 129, 255, 257, 1000, 1023, 1024, 1025, 2047, 2048,
                                            2049, 2100, 4097, 9000]
    rng.shuffle(lengths)

    def mate(n):
        s = "".join(rng.choice("ACGTacgt") for _ in range(n))
        if rng.random() < 0.2:
            i = rng.choice([0, n - 1, rng.randrange(n)])
            s = s[:i] + rng.choice("NnBS@`-. ") + s[i + 1:]
        return s

    lines = []
    for i, n in enumerate(lengths):
        rid = str(3 * i + 1)
        rid = rng.choice(["", "", "+"]) + "0" * rng.choice([0, 0, 1, 15 - len(rid), 16 - len(rid), 20 - len(rid)]) + rid
        line = rid + "\t" + mate(n)
        if rng.random() < 0.4:
            line += "\t" + mate(rng.choice(lengths))
        line += "\t" * rng.choice([0, 0, 0, 1, 9])
        lines.append(line + rng.choice(["\n", "\n", "\r\n", "\r"]))
    text = "".join(lines).encode()
    assert gx.build_graph(text, 11)[0] == oracle.build_graph(text, 11)[0]


@pytest.mark.parametrize("n", [4060, 4100, 8150])
def test_two_word_bucket_tiers(gx, n):
    """A bucket of about n two-word records (distinct k-mers that share their
    first eight letters), on both sides of the two block sizes' border."""
    import random
    rng = random.Random(n)
    reads = ["AACAGATA" + "".join(rng.choice("ACGT") for _ in range(47)) + "A" for _ in range(n)]
    reads += ["".join(rng.choice("ACGT") for _ in range(85)) for _ in range(40)]
    rng.shuffle(reads)
    text = "".join(f"{4 * i + 2}\t{s}\n" for i, s in enumerate(reads)).encode()
    assert gx.build_graph(text, 55)[0] == oracle.build_graph(text, 55)[0]
