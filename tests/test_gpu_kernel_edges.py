"""The kernels at the sizes where they can go wrong (edges of tiles, groups and
runs, remainders, the smallest and largest of a range), against the oracle.
Integer work: every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from goetia_amd import libgoetia as lg  # noqa: E402
from goetia_amd import _native as N  # noqa: E402
from goetia_amd.reads import ReadBatch  # noqa: E402

STORES = {1: lg.BitStorage, 2: lg.ByteStorage, 3: lg.SparseppSetStorage}


def _pair(oracle, kind, sizes, K, canonical=True, mode=N.MODE_RAW):
    """(graph, oracle storage) over the same table sizes."""
    sh = lg.CanLemireShifter if canonical else lg.FwdLemireShifter
    store = STORES[kind]() if kind == 3 else STORES[kind](sizes)
    g = lg.dBG[STORES[kind], sh].build(store, K)
    g.mode = mode
    return g, oracle.Storage(kind, sizes if kind != 3 else ())


def _reads(seed, lengths, genome=4000, sub=0.02, n_rate=0.0):
    """Reads of the given lengths from either strand of a random genome."""
    rng = np.random.default_rng(seed)
    acgt = np.frombuffer(b'ACGT', np.uint8)
    comp = np.zeros(256, np.uint8)
    comp[acgt] = acgt[::-1]
    g = acgt[rng.integers(0, 4, max(genome, int(max(lengths)) + 1))]
    out = []
    for L in lengths:
        a = int(rng.integers(0, len(g) - L + 1))
        s = g[a:a + L].copy()
        if rng.random() < 0.5:
            s = comp[s[::-1]]
        hit = rng.random(L) < sub
        s[hit] = acgt[rng.integers(0, 4, int(hit.sum()))]
        s[rng.random(L) < n_rate] = ord('N')
        out.append(s)
    off = np.zeros(len(out) + 1, np.int64)
    off[1:] = np.cumsum(lengths)
    return ReadBatch(np.concatenate(out) if out else np.zeros(0, np.uint8), off)


@pytest.mark.parametrize('kind,n_tables', [(1, 1), (1, 4), (1, 9), (2, 1), (2, 4), (2, 9), (3, 0)])
@pytest.mark.parametrize('min_count', [1, 2, 255])
def test_degrees_stop_at_the_first_absent_table(oracle, kind, n_tables, min_count):
    """Small tables (false positives in every one), counts up to 255, and
    windows left out by `only`."""
    K = 21
    g, o = _pair(oracle, kind, [1009, 1013, 1019, 1021, 1031, 1033, 1039, 1049, 1051][:n_tables], K)
    hot = ReadBatch.from_strings([b'ACGTTGCATGTCGCATGATGCATGAGAGCT'] * 260)
    b = _reads(11, [K - 1, K, 40, 150, 333] * 6, genome=900)
    for batch in (hot, b):
        g.insert_sequences(batch)
        o.insert_reads(batch.seq, batch.offsets, K)
    for batch in (ReadBatch.from_strings([hot.read(0)]), b):
        exp = [o.degrees_sequence(batch.read(r), K, True, min_count=min_count) for r in range(batch.n_reads)
               if len(batch.read(r)) >= K]
        ein, eout = (np.concatenate([e[i] for e in exp]) for i in (0, 1))
        ind, outd = g.degrees(batch, min_count=min_count)
        np.testing.assert_array_equal(ind, ein)
        np.testing.assert_array_equal(outd, eout)
        only = (np.arange(len(ind)) % 3 == 0).astype(np.uint8)
        ind, outd = g.degrees(batch, min_count=min_count, only=only)
        np.testing.assert_array_equal(ind, np.where(only, ein, 255))
        np.testing.assert_array_equal(outd, np.where(only, eout, 255))


@pytest.mark.parametrize('spread', [70, 300])
def test_per_read_sums_and_solid_reads_at_every_length(oracle, monkeypatch, spread):
    """Reads of every window count from none to past one round of the lanes
    that share a read: n_new of the binned insert, and the solid filter's
    decision, whose counts start at every alignment."""
    monkeypatch.setenv('GOETIA_AMD_BINNED', '1')
    K, sizes = 21, [20011, 20021]
    lengths = list(range(K - 2, K + spread)) * 2
    b = _reads(5, lengths, genome=6000)
    g, o = _pair(oracle, 2, sizes, K)
    _, e_new = o.insert_reads(b.seq, b.offsets, K)
    np.testing.assert_array_equal(g.insert_sequences(b), e_new)
    assert g.n_unique() == o.n_unique
    for prop, thr in ((0.75, 2), (0.4, 3)):
        g2, o2 = _pair(oracle, 2, sizes, K)
        passed = lg.StreamingSolidFilter.build(g2, prop, thr).filter_sequences(b)
        for r in range(b.n_reads):
            s = b.read(r)
            if len(s) < K:
                assert not passed[r]
                continue
            c = np.asarray(o2.insert_and_query_sequence(s, K))
            share = float(np.float32(int((c < thr).sum())) / np.float32(len(c)))
            assert passed[r] == (not share >= 1.0 - float(np.float32(prop)))
