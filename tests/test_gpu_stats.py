"""Graph statistics and FASTA dump on the device (include/genomix_stats.h)
against the oracle's restatement over the same graph's records."""

import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gx():
    import genomix_amd.gx as g
    return g


def _text(seed, G=30000, cov=12, paired=True):
    from genomix_amd import sim
    spec = sim.ReadSetSpec(genome_len=G, read_len=100, coverage=cov, error_rate=0.01, paired=paired,
                           insert_mean=300, insert_sd=25, repeat_frac=0.05, repeat_len=(300, 900), repeat_div=0.01,
                           seed=seed)
    return sim.simulate(spec)


@pytest.mark.parametrize("k,paired", [(21, False), (31, True), (55, True)])
def test_stats_and_fasta_match_oracle(gx, k, paired):
    text = _text(6100 + k, paired=paired)
    with gx.GraphBuilder(k) as b:
        b.add_reads(text)
        b.finish()
        nodes = b.part_bytes(0)
        assert b.graph_stats("nodes") == oracle.graph_stats(nodes, k)
        assert b.fasta("nodes") == oracle.dump_fasta(nodes, k)
        u = b.unitigs()
        assert b.graph_stats("unitigs") == oracle.graph_stats(u, k)
        assert b.fasta("unitigs") == oracle.dump_fasta(u, k)
        cleaned = b.clean_bad_coverage(3.0)
        assert b.graph_stats("unitigs") == oracle.graph_stats(cleaned, k)
        assert b.fasta("unitigs") == oracle.dump_fasta(cleaned, k)


@pytest.mark.parametrize("copies", [1, 1023, 1500])
def test_stats_of_wide_ranges(gx, copies):
    """Coverages, head counts and seed scores inside and beyond a block's
    counting window, and (a long unitig that carries many heads) beyond the
    widest histogram, where the values are sorted."""
    import random
    rng = random.Random(copies)
    k = 21
    one = "".join(rng.choice("ACGT") for _ in range(60))
    genome = "".join(rng.choice("ACGT") for _ in range(6000))
    reads = [one] * copies + [genome[p:p + 100] for p in range(0, 5901, 2)]
    text = "".join(f"{4 * i + 2}\t{s}\n" for i, s in enumerate(reads)).encode()
    with gx.GraphBuilder(k) as b:
        b.add_reads(text)
        b.finish()
        assert b.graph_stats("nodes") == oracle.graph_stats(b.part_bytes(0), k)
        u = b.unitigs()
        got = b.graph_stats("unitigs")
        assert got == oracle.graph_stats(u, k)
        assert got["maximum"]["scaffoldSeedScore"] > 1 << 22


@pytest.mark.parametrize("k,lengths", [(21, (1004, 1005, 1024, 2048, 2049)), (33, (992, 993, 5000))])
def test_fasta_of_long_unitigs(gx, k, lengths):
    """Sequences of one chunk, at its edge and of several chunks."""
    import random
    rng = random.Random(k)
    lines = []
    for G in lengths:
        g = "".join(rng.choice("ACGT") for _ in range(G))
        lines += [g[p:p + 100] for p in range(0, G - 99, 30)] + [g[-100:]]
    text = "".join(f"{4 * i + 2}\t{s}\n" for i, s in enumerate(lines)).encode()
    with gx.GraphBuilder(k) as b:
        b.add_reads(text)
        b.finish()
        assert b.fasta("nodes") == oracle.dump_fasta(b.part_bytes(0), k)
        u = b.unitigs()
        assert b.fasta("unitigs") == oracle.dump_fasta(u, k)


def test_stats_errors(gx):
    with gx.GraphBuilder(21) as b:
        b.add_reads(_text(3, G=5000, paired=False))
        with pytest.raises(gx.GxError) as e:
            b.graph_stats("nodes")
        assert e.value.code == gx.GX_ESTATE
        b.finish()
        with pytest.raises(gx.GxError) as e:
            b.graph_stats("unitigs")
        assert e.value.code == gx.GX_ESTATE
