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


@pytest.mark.parametrize('kind,n_tables', [(1, 1), (1, 4), (1, 6), (2, 2), (2, 4), (2, 9), (3, 0)])
@pytest.mark.parametrize('K,mode', [(21, N.MODE_RAW), (31, N.MODE_SKIP_N), (255, N.MODE_RAW)])
@pytest.mark.parametrize('binned', ['0', '1'])
def test_small_batches_take_windows_together(oracle, monkeypatch, kind, n_tables, K, mode, binned):
    """Batches around one tile of 1024 starts, hot k-mers (several windows of a
    thread on one bin or slot), reads below K, N bases, and a second batch over
    the first one's keys: n_new, flags, counts, counters, tables; through the
    atomic insert and, where the tables allow it, the binned one."""
    monkeypatch.setenv('GOETIA_AMD_BINNED', binned)
    sizes = [4001, 4003, 4007, 4013, 4019, 4021, 4027, 4049, 4051][:n_tables]
    for lengths in ([K], [K - 1, K + 3], [300, 0, 421, 300, 3], [1024], [1025], [257] * 40, [150] * 300):
        g, o = _pair(oracle, kind, sizes, K, mode=mode)
        for seed in (1, 2):
            b = _reads(seed, lengths, genome=max(500, max(lengths)), n_rate=0.003)
            hot = np.frombuffer(b'A' * (K + 40) + b'ACAC' * 100, np.uint8)
            b = ReadBatch(np.concatenate([b.seq, hot]), np.append(b.offsets, b.n_bases + len(hot)))
            _, e_new, e_flags = o.insert_reads_flags(b.seq, b.offsets, K, True, mode)
            n_new, flags = g.insert_sequences(b, new_flags=True)
            np.testing.assert_array_equal(n_new, e_new)
            np.testing.assert_array_equal(flags, np.asarray(e_flags, bool))
            np.testing.assert_array_equal(g.query_sequences(b), o.query_reads(b.seq, b.offsets, K, True, mode))
            assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied
        if kind == 3:
            np.testing.assert_array_equal(g.S.keys(), np.sort(o.exact_keys()))
        else:
            for x, y in zip(g.get_raw(), o.tables()):
                np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize('n_reads', [1, 1023, 1025, 12288, 12289, 16384, 16385])
@pytest.mark.parametrize('binned', ['0', '1'])
def test_layout_of_small_batches(oracle, monkeypatch, n_reads, binned):
    """Either side of the one-launch layout's limit: packed results of reads of
    0 to 60 bases, and one long read over many tiles."""
    monkeypatch.setenv('GOETIA_AMD_BINNED', binned)
    K = 21
    rng = np.random.default_rng(n_reads)
    lengths = rng.integers(0, 60, n_reads)
    lengths[n_reads // 2] = 9000
    b = _reads(n_reads, list(lengths), genome=9500)
    g, o = _pair(oracle, 2, [50021, 50023], K)
    _, e_new = o.insert_reads(b.seq, b.offsets, K)
    np.testing.assert_array_equal(g.insert_sequences(b), e_new)
    np.testing.assert_array_equal(g.query_sequences(b), o.query_reads(b.seq, b.offsets, K))


def test_exact_set_moves_newness_and_grows(oracle):
    """Keys of earlier batches stay old through a rehash (n_new 0 when they
    come again), the all-ones key's stand-in included, and newness ends at the
    smallest window when many reads hold the same keys."""
    K = 25
    g, o = _pair(oracle, 3, (), K)
    for step, n in enumerate((40, 400, 4000, 40, 4000)):
        b = _reads(100 + (step % 3), [80] * n, genome=300 * (1 + n // 10), sub=0.0)
        for _ in range(2):
            _, e_new = o.insert_reads(b.seq, b.offsets, K)
            np.testing.assert_array_equal(g.insert_sequences(b), e_new)
            assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied
    for v in (0, 2 ** 64 - 1, 2 ** 64 - 1, 5):
        assert g.S.insert(v) == o.insert(v)
    b = _reads(7, [120] * 30000, genome=2_000_000)
    _, e_new = o.insert_reads(b.seq, b.offsets, K)
    np.testing.assert_array_equal(g.insert_sequences(b), e_new)
    assert not g.S.insert(2 ** 64 - 1) and not o.insert(2 ** 64 - 1)
    assert g.n_unique() == o.n_unique


@pytest.mark.parametrize('n_tables,sizes', [(1, [8191]), (2, [8192 * 3 + 1, 20011]), (3, [97, 101, 103]),
                                            (4, [2_100_001, 2_100_011, 2_100_017, 2_100_019])])
@pytest.mark.parametrize('sub', ['', '8192'])
def test_insert_and_query_results_by_event_position(oracle, monkeypatch, n_tables, sizes, sub):
    """Tiles whose first window lies in a short read, in a gap between reads or
    mid-read, N bases, counts past 255, a last partial tile; one sub-batch and
    several."""
    monkeypatch.setenv('GOETIA_AMD_SUB_BATCH', sub)
    K = 31
    for seed, lengths in ((1, [40]), (2, [2048, 30, 2047, 31, 1]), (3, [5, 9000, 12, 0, 0, 3000]), (4, [150] * 700)):
        g, o = _pair(oracle, 2, sizes, K, mode=N.MODE_SKIP_N)
        b = _reads(seed, lengths, genome=max(1500, max(lengths)), n_rate=0.002)
        hot = np.frombuffer(b'AC' * 400, np.uint8)
        b = ReadBatch(np.concatenate([b.seq, hot]), np.append(b.offsets, b.n_bases + len(hot)))
        for _ in range(2):
            exp = o.insert_and_query_reads(b.seq, b.offsets, K, True, N.MODE_SKIP_N)
            np.testing.assert_array_equal(g.insert_and_query_sequences(b), exp)
        for x, y in zip(g.get_raw(), o.tables()):
            np.testing.assert_array_equal(x, y)
        assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied


@pytest.mark.parametrize('K,cutoff,chunk,guesses', [(21, 3, '', ''), (31, 5, '2048', ''), (31, 5, '16384', '3'),
                                                    (17, 20, '', '2')])
def test_diginorm_leaves_out_events_of_dropped_reads(oracle, monkeypatch, K, cutoff, chunk, guesses):
    """High coverage over small tables (several events of a step on one bin),
    reads that fill a bucket's step with their own events (tandem repeats),
    N bases, short reads; chunks cut by the guess cap; two batches."""
    monkeypatch.setenv('GOETIA_AMD_DIGINORM_CHUNK', chunk)
    monkeypatch.setenv('GOETIA_AMD_DIGINORM_GUESSES', guesses)
    g, o = _pair(oracle, 2, [9001, 9011, 9013], K, mode=N.MODE_SKIP_N)
    f = lg.DiginormFilter.build(g, cutoff)
    for seed in (1, 2):
        b = _reads(seed, [90, K - 1, K, 150, 70] * 260, genome=1500, sub=0.01, n_rate=0.001)
        rep = np.frombuffer((b'ACGTT' * 60 + b'A' * 90) * 3, np.uint8)
        off = b.offsets
        for _ in range(6):
            off = np.append(off, off[-1] + len(rep))
        b = ReadBatch(np.concatenate([b.seq] + [rep] * 6), off)
        exp = o.diginorm_reads(b.seq, b.offsets, K, cutoff, True, N.MODE_SKIP_N)
        np.testing.assert_array_equal(f.filter_sequences(b), np.asarray(exp, bool))
        for x, y in zip(g.get_raw(), o.tables()):
            np.testing.assert_array_equal(x, y)
        assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied


@pytest.mark.parametrize('kind,max_table,n_reads', [(k, m, n) for k, m in ((1, 40_009), (2, 2_000_003), (2, 60_000_011))
                                                    for n in (130, 900, 9000)]
                         + [(2, 2_000_003, 14_500), (1, 2_000_003, 28_500), (2, 60_000_011, 57_000)])
def test_binned_insert_in_small_groups(oracle, monkeypatch, kind, max_table, n_reads):
    """Batches whose second pass takes 64 tiles per item (up to 9000 reads on a
    256-CU device), 256, 512 and 1024, one or more of the items per counting
    workgroup, and whose counts are scanned by one workgroup or several."""
    monkeypatch.setenv('GOETIA_AMD_BINNED', '1')
    K, sizes = 31, oracle.primes_near_x(4, max_table)
    g, o = _pair(oracle, kind, sizes, K)
    for seed in (1, 2):
        b = _reads(seed, [150] * n_reads, genome=20_000)
        _, e_new = o.insert_reads(b.seq, b.offsets, K)
        np.testing.assert_array_equal(g.insert_sequences(b), e_new)
        if kind == 2:
            exp = o.insert_and_query_reads(b.seq, b.offsets, K)
            np.testing.assert_array_equal(g.insert_and_query_sequences(b), exp)
    for x, y in zip(g.get_raw(), o.tables()):
        np.testing.assert_array_equal(x, y)
    assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied


@pytest.mark.parametrize('kind,sizes', [(1, [97]), (1, [1 << 21, (1 << 21) + 1]), (2, [8191, 8209, 8219, 8221]),
                                        (2, [(1 << 21) - 1, 1 << 21, (1 << 21) + 1, 5_000_011]),
                                        (2, [1 << 28, 3, 70_000_001]), (1, [(1 << 29) - 3, 1 << 21]),
                                        (1, [(1 << 28) - 2 * i for i in range(4)]),
                                        (2, [(1 << 28) - 2 * i for i in range(4)])])
@pytest.mark.parametrize('K,mode', [(1, N.MODE_RAW), (31, N.MODE_SKIP_N), (64, N.MODE_RAW), (255, N.MODE_SKIP_N)])
def test_routed_query_equals_the_direct_one(oracle, monkeypatch, launches, kind, sizes, K, mode):
    """Slices of one bin to 2^21, 1 to 512 digits in all (64 lanes to a run to
    128 digits, 32 to 256: 163 here, 16 past that: 257 and 512), runs longer
    than two rounds of their lanes, N bases, gaps, sub-batches, hashes; present
    and absent windows."""
    g, o = _pair(oracle, kind, [min(s, 5_000_011) for s in sizes], K, mode=mode)
    if max(sizes) > 5_000_011:                          # too large for the oracle here: the direct query is its stand-in
        g, o = _pair(oracle, kind, sizes, K, mode=mode)[0], None
    fill = _reads(1, [300] * 60, genome=6000)
    if o is not None:
        o.insert_reads(fill.seq, fill.offsets, K, True, mode)
    g.insert_sequences(fill)
    for seed, lengths in ((1, [K]), (1, [300] * 60), (2, [K + 1, 0, 5000, 3, 2048, 2047, 1, 400])):
        b = _reads(seed, lengths, genome=6000, n_rate=0.002)
        hot = np.frombuffer(b'A' * 3000, np.uint8)
        b = ReadBatch(np.concatenate([b.seq, hot]), np.append(b.offsets, b.n_bases + len(hot)))
        for sub in ('', '8192'):
            monkeypatch.setenv('GOETIA_AMD_SUB_BATCH', sub)
            monkeypatch.setenv('GOETIA_AMD_ROUTED', '0')
            N.call('gt_profile_reset')
            direct, dh = g.query_sequences(b, with_hashes=True)
            assert launches('query_route') == 0
            monkeypatch.setenv('GOETIA_AMD_ROUTED', '1')
            routed, rh = g.query_sequences(b, with_hashes=True)
            assert launches('query_route') > 0
            np.testing.assert_array_equal(routed, direct)
            np.testing.assert_array_equal(rh, dh)
            np.testing.assert_array_equal(g.query_sequences(b), direct)
        if o is not None:
            np.testing.assert_array_equal(routed, o.query_reads(b.seq, b.offsets, K, True, mode))


def _launches(name):
    """Times a kernel's timer ran since the last reset."""
    import ctypes as C
    n, ms = C.c_uint64(), C.c_double()
    N.call('gt_profile_get', name.encode(), C.byref(n), C.byref(ms))
    return n.value


@pytest.fixture
def launches():
    N.call('gt_profile_enable', 1)
    N.call('gt_profile_reset')
    yield _launches
    N.call('gt_profile_enable', 0)


@pytest.mark.parametrize('kind', [1, 2])
def test_calls_without_room_for_their_events(oracle, monkeypatch, launches, kind):
    """A device that has no room for the event buffers of the binned insert,
    the routed query and insert_and_query: each goes its other way, with the
    same results, and the calls after it are not told of the refusal."""
    K, sizes = 31, [20011, 20021, 20023, 20029]
    monkeypatch.setenv('GOETIA_AMD_BINNED', '1')
    monkeypatch.setenv('GOETIA_AMD_ROUTED', '1')
    g, o = _pair(oracle, kind, sizes, K)
    b = _reads(3, [150] * 2000, genome=20_000)           # 0.3 MB of reads, 10 MB of events
    c = _reads(4, [150] * 2000, genome=20_000)
    monkeypatch.setenv('GOETIA_AMD_ALLOC_LIMIT', str(2 << 20))
    for batch in (b, c, b):
        _, e_new = o.insert_reads(batch.seq, batch.offsets, K)
        np.testing.assert_array_equal(g.insert_sequences(batch), e_new)
        np.testing.assert_array_equal(g.query_sequences(batch), o.query_reads(batch.seq, batch.offsets, K))
    if kind == 2:
        exp = o.insert_and_query_reads(c.seq, c.offsets, K)
        np.testing.assert_array_equal(g.insert_and_query_sequences(c), exp)
    assert launches('bin_hash') == 0 and launches('query_route') == 0
    monkeypatch.delenv('GOETIA_AMD_ALLOC_LIMIT')
    _, e_new = o.insert_reads(c.seq, c.offsets, K)
    np.testing.assert_array_equal(g.insert_sequences(c), e_new)
    np.testing.assert_array_equal(g.query_sequences(c), o.query_reads(c.seq, c.offsets, K))
    assert launches('bin_hash') > 0 and launches('query_route') > 0
    for x, y in zip(g.get_raw(), o.tables()):
        np.testing.assert_array_equal(x, y)
    assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied


@pytest.mark.parametrize('kind', [1, 2])
def test_claims_without_room_for_a_stamp_per_bin(oracle, monkeypatch, kind):
    """Small tables claim directly, a stamp per bin (8 MB here); without room
    for that the hashed map (1 MB) takes the same batches."""
    monkeypatch.setenv('GOETIA_AMD_BINNED', '0')
    K, sizes = 31, [250_007, 250_013, 250_027, 250_031]
    g, o = _pair(oracle, kind, sizes, K)
    for step, limit in enumerate(('', str(4 << 20), str(4 << 20), '')):
        monkeypatch.setenv('GOETIA_AMD_ALLOC_LIMIT', limit)
        if step == 1:                                     # (a storage that took the direct map keeps it)
            g, o = _pair(oracle, kind, sizes, K)
        b = _reads(step, [150] * 120, genome=9000)
        _, e_new, e_flags = o.insert_reads_flags(b.seq, b.offsets, K, True, N.MODE_RAW)
        n_new, flags = g.insert_sequences(b, new_flags=True)
        np.testing.assert_array_equal(n_new, e_new)
        np.testing.assert_array_equal(flags, np.asarray(e_flags, bool))
        assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied


@pytest.mark.parametrize('n_tables,table,n_bases', [(4, (1 << 30) - 35, (1 << 29) + 12_345),
                                                    (5, 1 << 28, (1 << 28) + 12_345)])
def test_claims_of_a_large_batch_stay_within_the_hashed_maps_memory(n_tables, table, n_bases):
    """Nearly 2^32 bins, and 1.3e9 in five tables, under a batch with more
    starts than a claim map's cap has room for: sub-batches, and 8 GiB of
    claims at most (a stamp for each of those bins is 10 to 32 GiB)."""
    import torch
    K, L = 31, 150
    n = (n_bases + L - 1) // L
    gen = torch.Generator(device='cuda')
    gen.manual_seed(1)
    seq = torch.tensor(list(b'ACGT'), dtype=torch.uint8, device='cuda')
    seq = seq[torch.randint(0, 4, (n_bases,), generator=gen, device='cuda', dtype=torch.uint8).to(torch.int32)]
    off = torch.clamp(torch.arange(n + 1, device='cuda', dtype=torch.int64) * L, max=n_bases)
    from goetia_amd.reads import DeviceReads
    d = DeviceReads(seq, off, n_bases)
    n_new = torch.zeros(n, dtype=torch.int64, device='cuda')
    g = lg.dBG[lg.BitStorage, lg.CanLemireShifter].build(lg.BitStorage([table - 2 * i for i in range(n_tables)]), K)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    g.insert_device(d, n_new=n_new)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 9 << 30
    first = int(n_new.sum())
    windows = (n_bases // L) * (L - K + 1) + max(0, n_bases % L - K + 1)
    assert 0.97 * windows < first <= windows and first == g.n_unique()
    g.insert_device(d, n_new=n_new)
    assert int(n_new.sum()) == 0 and g.n_unique() == first


@pytest.mark.parametrize('kind,n_tables,table', [(1, 4, 1_050_000), (2, 4, 1_050_000), (1, 9, 470_000),
                                                 (2, 9, 470_000), (2, 5, 4_000_000), (1, 5, 3000)])
@pytest.mark.parametrize('n_bases', [40_000, 131_071, 393_215, 393_216, 524_289, (1 << 22) - 1, 1 << 22])
def test_atomic_inserts_at_every_shape_of_launch(oracle, monkeypatch, kind, n_tables, table, n_bases):
    """Either side of the sizes where the atomic insert and the query change
    their shape (one wave to a workgroup, four windows of a thread together,
    window by window), over bins that are claimed by hash (more than 2^22, and
    than the batch's own limit) and directly (3000 each, and past the limit);
    more than four and more than eight tables.  Hot k-mers claim one bin from
    many windows, and the second batch meets slots of the first one's keys."""
    monkeypatch.setenv('GOETIA_AMD_BINNED', '0')
    K, sizes = 31, oracle.primes_near_x(n_tables, table)
    g, o = _pair(oracle, kind, sizes, K)
    hot = np.frombuffer(b'A' * 100 + b'ACAC' * 50, np.uint8)
    for seed in (1, 2):
        n, tail = divmod(n_bases - len(hot), 150)
        b = _reads(seed, [150] * n + [tail], genome=max(3000, n_bases // 12), sub=0.01)
        b = ReadBatch(np.concatenate([b.seq, hot]), np.append(b.offsets, n_bases))
        _, e_new, e_flags = o.insert_reads_flags(b.seq, b.offsets, K, True, N.MODE_RAW)
        n_new, flags = g.insert_sequences(b, new_flags=True)
        np.testing.assert_array_equal(n_new, e_new)
        np.testing.assert_array_equal(flags, np.asarray(e_flags, bool))
        np.testing.assert_array_equal(g.query_sequences(b), o.query_reads(b.seq, b.offsets, K))
    assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied
    for x, y in zip(g.get_raw(), o.tables()):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize('kind,n_tables,table,n_reads,empty,filled', [
    (1, 4, 1_000_000, 100, False, False), (1, 4, 1_000_000, 300, True, True), (2, 4, 1 << 25, 1000, True, True),
    (1, 4, 1 << 26, 1100, False, False), (1, 4, 1 << 26, 1300, True, False), (1, 4, 1 << 26, 7000, True, True),
    (2, 2, 1 << 24, 3000, True, False), (2, 1, 1 << 25, 700, True, False), (2, 1, 1 << 25, 7000, True, True),
    (2, 4, 1 << 28, 6000, False, False), (2, 4, 1 << 28, 9400, True, False), (2, 4, 1 << 28, 27_900, True, False),
    (2, 4, 1 << 28, 28_000, True, True), (2, 1, 1 << 28, 3000, False, False)])
def test_batches_are_binned_where_that_is_the_faster_insert(oracle, launches, kind, n_tables, table, n_reads, empty,
                                                            filled):
    """Which insert a batch takes by itself, on both sides of the lines for an
    empty graph and for one that holds k-mers; a reset or new tables make it
    empty, every other call that writes to it does not."""
    sizes = [table - 2 * i for i in range(n_tables)]
    g = _pair(oracle, kind, sizes, 31)[0]
    b = _reads(1, [150] * n_reads, genome=20_000)

    def binned(batch):
        N.call('gt_profile_reset')
        g.insert_sequences(batch)
        assert launches('bin_hash') + launches('claim') == 1
        return launches('bin_hash') > 0
    assert binned(b) == empty
    assert binned(b) == filled
    g.reset()
    g.S.insert_hashes(np.arange(3, dtype=np.uint64))
    assert binned(b) == filled
    g.reset()
    assert binned(b) == empty
    if kind == 2:
        g.reset()
        g.insert_and_query_sequences(_reads(2, [40], genome=100))
        assert binned(b) == filled
        g.reset()
        lg.DiginormFilter.build(g, 5).filter_sequences(_reads(2, [40], genome=100))
        assert binned(b) == filled
    else:
        h = _pair(oracle, kind, sizes, 31)[0]
        g.reset()
        g.S.update_from(h.S)
        assert binned(b) == filled
    if table <= 1_000_000:
        g.reset()
        g.S.set_raw_table(0, g.S.get_raw_tables()[0])
        assert binned(b) == filled


@pytest.mark.parametrize('lengths', [[9000] * 12, [150] * 4000, [31] * 3000 + [4500] * 3, [40, 31, 2000, 33] * 200])
@pytest.mark.parametrize('K,mode,sub', [(31, N.MODE_RAW, ''), (31, N.MODE_SKIP_N, '8192'), (4, N.MODE_SKIP_N, ''),
                                        (255, N.MODE_RAW, '')])
def test_exact_set_newness_among_overlapping_reads(oracle, monkeypatch, lengths, K, mode, sub):
    """Reads that cover their genome many times, so that a window's newness
    moves between reads, runs of windows to one read and to many: long reads,
    reads of one window, several sub-batches; n_new alone and with flags, on an
    empty set, a filled one and one that holds half of the keys."""
    monkeypatch.setenv('GOETIA_AMD_SUB_BATCH', sub)
    for seed in (1, 2):
        g, o = _pair(oracle, 3, (), K, mode=mode)
        for step in (1, 1, 2):
            b = _reads(10 * seed + step, lengths, genome=12_000 if step == 1 else 20_000, sub=0.004, n_rate=0.001)
            _, e_new, e_flags = o.insert_reads_flags(b.seq, b.offsets, K, True, mode)
            if seed == 1:
                n_new, flags = g.insert_sequences(b, new_flags=True)
                np.testing.assert_array_equal(flags, np.asarray(e_flags, bool))
            else:
                n_new = g.insert_sequences(b)
            np.testing.assert_array_equal(n_new, e_new)
            assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied
        np.testing.assert_array_equal(g.S.keys(), np.sort(o.exact_keys()))


def test_exact_set_looks_its_windows_up_only_before_it_may_grow(oracle, launches):
    """Batches that fit the set whatever they hold are inserted in one pass,
    however often they come; one that may not is looked up first."""
    K = 31
    store = lg.SparseppSetStorage.build(capacity_hint=60_000)       # 131072 slots
    g, o = lg.dBG[lg.SparseppSetStorage, lg.CanLemireShifter].build(store, K), oracle.Storage(3, ())
    b = _reads(1, [150] * 250, genome=15_000, sub=0.0)
    for _ in range(6):
        _, e_new = o.insert_reads(b.seq, b.offsets, K)
        np.testing.assert_array_equal(g.insert_sequences(b), e_new)
    assert launches('exact_insert') == 6 and launches('exact_lookup') == 0
    b = _reads(2, [150] * 400, genome=15_000)
    _, e_new = o.insert_reads(b.seq, b.offsets, K)
    np.testing.assert_array_equal(g.insert_sequences(b), e_new)
    assert launches('exact_lookup') == 1
    assert g.n_unique() == o.n_unique and g.n_occupied() == o.n_occupied


@pytest.mark.parametrize('kind,sizes', [(1, [(1 << 30) - 35, 11]), (2, [1 << 30])])
def test_tables_past_the_routed_query_are_read_directly(monkeypatch, launches, kind, sizes):
    """More than 512 slices, and 2^30 bins: not routed even where asked for."""
    monkeypatch.setenv('GOETIA_AMD_ROUTED', '1')
    g = lg.dBG[STORES[kind], lg.CanLemireShifter].build(STORES[kind](sizes), 31)
    b = _reads(1, [300] * 60, genome=6000)
    g.insert_sequences(b)
    assert (g.query_sequences(b) >= 1).all()
    assert launches('query_route') == 0


@pytest.mark.parametrize('kind,sizes', [(1, [60_013]), (2, [60_013]), (2, [60_013, 60_017]), (3, ())])
@pytest.mark.parametrize('n_bases', [(3 << 19) - 1, 3 << 19, 1 << 22])
@pytest.mark.parametrize('with_hashes', [False, True])
def test_queries_of_few_tables_at_every_shape_of_launch(oracle, kind, sizes, n_bases, with_hashes):
    """Either side of the sizes where a query of an exact set or of one or two
    tables changes its shape, alone and with hashes (whose line is another)."""
    K = 31
    g, o = _pair(oracle, kind, sizes, K, mode=N.MODE_SKIP_N)
    fill = _reads(1, [150] * 300, genome=60_000)
    o.insert_reads(fill.seq, fill.offsets, K, True, N.MODE_SKIP_N)
    g.insert_sequences(fill)
    n, tail = divmod(n_bases, 150)
    b = _reads(1, [150] * n + [tail], genome=60_000, sub=0.004, n_rate=0.001)
    exp = o.query_reads(b.seq, b.offsets, K, True, N.MODE_SKIP_N)
    if with_hashes:
        counts, hashes = g.query_sequences(b, with_hashes=True)
        for r in (0, n // 2, n):
            if len(b.read(r)) >= K:
                k0 = int(b.kmer_offsets(K)[r])
                fw, rc = oracle.hash_read(bytes(b.read(r)), K)
                live = exp[k0:k0 + len(fw)] >= 0
                np.testing.assert_array_equal(hashes[k0:k0 + len(fw)][live], np.minimum(fw, rc)[live])
    else:
        counts = g.query_sequences(b)
    np.testing.assert_array_equal(counts, exp)


@pytest.mark.parametrize('n_tables,L,K,n_reads,routed', [
    (4, 150, 31, 70_000, True), (4, 150, 31, 58_000, False), (4, 75, 63, 200_000, False), (4, 75, 55, 700_000, False),
    (4, 101, 41, 160_000, True), (2, 150, 31, 70_000, True), (2, 75, 31, 400_000, True), (2, 101, 63, 400_000, False),
    (1, 150, 31, 200_000, False)])
def test_queries_are_routed_where_windows_are_many(oracle, launches, n_tables, L, K, n_reads, routed):
    """Which way a query goes by itself: by its bases, less those that start no
    window, and by their share."""
    import torch
    from goetia_amd.reads import DeviceReads
    sizes = [(1 << 25) // n_tables - 2 * i for i in range(n_tables)]
    g = _pair(oracle, 2, sizes, K)[0]
    fill = _reads(1, [L] * 2000, genome=40_000, sub=0.0)
    g.insert_sequences(fill)
    d = DeviceReads(torch.from_numpy(np.tile(fill.seq, n_reads // 2000)).cuda(),
                    torch.arange(n_reads + 1, dtype=torch.int64, device='cuda') * L, n_reads * L)
    counts = torch.empty(n_reads * (L - K + 1), dtype=torch.int16, device='cuda')
    g.query_device(d, counts)
    exp = torch.from_numpy(g.query_sequences(fill)).cuda()
    assert bool((counts.view(n_reads // 2000, -1) == exp).all())
    assert (launches('query_route') > 0) == routed
