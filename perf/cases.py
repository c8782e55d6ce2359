"""The work that programs built on goetia_amd have it do, as cases that can be timed.

A case is one call sequence of the package's public entry points over a batch
of reads: insert with per-read new k-mers, query, the one-pass
insert_and_query, degrees of the new k-mers, the diginorm and solid filters,
and the host-memory calls.  Sizes, rates and storages are those of the
benchmark configurations (goetia_amd/workload.py, bench.py, bench_configs.py),
of goetia's defaults (500,000-k-mer intervals, BitStorage(1e6, 4)) and of the
tests.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  reads on the device, the graph, output buffers
    run(state)           one pass; its outputs
    work(case)           bytes a pass cannot do without
    tolerance(case)      every output is a whole number or a byte: exact

There is no exact(): no output is a rounded number.
"""
import math

import torch

from goetia_amd import _native as N
from goetia_amd import libgoetia as lg
from goetia_amd.reads import DeviceReads, ReadBatch

# Reads of length 0 stand for the uneven mix of the exact-set configuration:
# one lognormal read (median 8 kb, sigma 1, 150 bp to 100 kb) for every ten of
# 150 bp, in random order.
MIXED = 0
MIX_MEDIAN, MIX_MAX, MIX_SHORT = 8000.0, 100_000, 150
MIX_MEAN = (10 * MIX_SHORT + 12_900) / 11          # bases per read of the mix

BASE = dict(storage='count', max_table=2 ** 28, n_tables=4, K=31, canonical=True, skip_n=False, read_len=150,
            sub=0.005, n_rate=0.0, hashes=False, param=0)


def _case(name, op, reads, genome, **more):
    c = dict(BASE, op=op, reads=reads, genome=genome)
    c.update(more)
    if name:
        c['name'] = name
    return c


def listed():
    return [
        # A streaming sample's first reads into goetia's default Bloom filter:
        # launches and host work count.
        _case('bloom_first_reads', 'insert', 500, 50_000, storage='bloom', max_table=1_000_000, K=21, sub=0.01),
        # One goetia interval (500,000 k-mers) queried against a filled
        # full-size count-min graph.
        _case('count_query_interval', 'query', 4_167, 5_000_000),
        # One interval into an exact set with forward hashes, then its counts
        # and hashes: the compactor's graph.
        _case('set_interval', 'insert_query', 4_167, 1_000_000, storage='set', canonical=False, hashes=True),
        # The Bloom configuration: 100k reads, K=21, 5 MB of tables, per-read n_new.
        _case('bloom_100k', 'insert', 100_000, 1_000_000, storage='bloom', max_table=10_000_000, K=21, sub=0.01),
        # A parsed chunk in host memory through the numpy calls.
        _case('count_host_chunk', 'host', 100_003, 5_000_000),
        # The chunk of the plain chunk-at-a-time path: 1M reads, insert + query.
        _case('count_chunk_1m', 'insert_query', 1_000_000, 50_000_000, skip_n=True, n_rate=0.0001),
        # The count-min configuration at full size: insert + query.
        _case('count_20m', 'insert_query', 20_000_000, 50_000_000, skip_n=True, n_rate=0.0001),
        # The one-pass insert_and_query on the same kind of reads.
        _case('count_insert_and_query_4m', 'insert_and_query', 4_000_000, 50_000_000, skip_n=True, n_rate=0.0001),
        # The uneven-read configuration at a tenth: exact set, K=25, 5% substitutions.
        _case('set_mixed', 'insert', 220_000, 5_000_000, storage='set', K=25, read_len=MIXED, sub=0.05),
        # Decision nodes: degrees at count >= 2 of every new k-mer.
        _case('degrees_1m', 'degrees', 1_000_000, 4_000_000, sub=0.01, param=2),
        # Digital normalisation at cutoff 20 of reads at 60x.
        _case('diginorm_2m', 'diginorm', 2_000_000, 5_000_000, skip_n=True, n_rate=0.0001, param=20),
        # The streaming solid filter (threshold 2).
        _case('solid_500k', 'solid', 500_000, 5_000_000, sub=0.01, param=2),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(['insert', 'insert', 'query', 'query', 'insert_query', 'insert_query', 'insert_and_query',
                     'degrees', 'diginorm', 'solid', 'host'])
    storage = {'insert': ['bloom', 'count', 'set'], 'query': ['bloom', 'count', 'count', 'set'],
               'insert_query': ['bloom', 'count', 'count', 'set'], 'degrees': ['count', 'bloom', 'set'],
               'host': ['bloom', 'count', 'set']}.get(op, ['count'])
    storage = rng.choice(storage)
    read_len = rng.choice([MIXED, 75, 101, 150, 150, 250, rng.randint(60, 300)])
    mean = read_len or MIX_MEAN
    most = {'host': 30e6, 'degrees': 250e6}.get(op, 600e6) / mean
    reads = _log_uniform(rng, 400, most)
    genome = max(10_000, min(50_000_000, int(reads * mean / _log_uniform(rng, 2, 80))))
    skip_n = rng.random() < 0.5
    return _case(None, op, reads, genome, storage=storage, max_table=_log_uniform(rng, 1_000_000, 2 ** 28),
                 n_tables=rng.choice([4, 4, 4, 3, 2]), K=rng.choice([17, 21, 25, 31, 31, 41, 55, 63]),
                 canonical=rng.random() < 0.8, skip_n=skip_n, read_len=read_len,
                 sub=rng.choice([0.002, 0.005, 0.01, 0.05]), n_rate=0.0001 if skip_n else 0.0,
                 hashes=op in ('query', 'insert_query') and rng.random() < 0.25,
                 param={'degrees': rng.choice([1, 2, 3]), 'diginorm': rng.choice([5, 20, 40]),
                        'solid': rng.choice([1, 2, 3])}.get(op, 0))


# ---------------------------------------------------------------- inputs

def _genome(gen, n):
    return torch.randint(0, 4, (n,), generator=gen, device='cuda', dtype=torch.uint8)


def _lengths(case):
    """Read lengths: a case's own, so that its outputs have one shape for every seed."""
    n, L = case['reads'], case['read_len']
    gen = torch.Generator(device='cuda')
    gen.manual_seed(n)
    if L:
        return torch.full((n,), L, dtype=torch.int64, device='cuda')
    long = torch.exp(torch.randn(n, generator=gen, device='cuda') + math.log(MIX_MEDIAN)).round()
    long = long.clamp(MIX_SHORT, MIX_MAX).to(torch.int64)
    is_long = torch.rand(n, generator=gen, device='cuda') < 1 / 11
    return torch.where(is_long, long, MIX_SHORT)


def _reads(case, gen, genome, lens):
    """Reads from either strand of the genome, with substitutions and N bases."""
    lens = torch.minimum(lens, torch.tensor(genome.numel(), device='cuda'))
    n = lens.numel()
    off = torch.zeros(n + 1, dtype=torch.int64, device='cuda')
    torch.cumsum(lens, 0, out=off[1:])
    start = (torch.rand(n, generator=gen, device='cuda', dtype=torch.float64)
             * (genome.numel() - lens + 1)).to(torch.int64)
    rev = torch.rand(n, generator=gen, device='cuda') < 0.5
    n_bases = int(off[-1])
    seq = torch.empty(n_bases, dtype=torch.uint8, device='cuda')
    letters = torch.tensor(list(b'ACGT'), dtype=torch.uint8, device='cuda')
    host_off = off.cpu()
    r = 0
    while r < n:                                       # about 64M bases at a time
        r1 = int(torch.searchsorted(host_off, host_off[r] + (1 << 26), right=True)) - 1
        r1 = min(n, max(r + 1, r1))
        a, b = int(host_off[r]), int(host_off[r1])
        own = torch.repeat_interleave(torch.arange(r, r1, device='cuda'), lens[r:r1], output_size=b - a)
        j = torch.arange(a, b, device='cuda') - off[own]
        rv = rev[own]
        code = genome[start[own] + torch.where(rv, lens[own] - 1 - j, j)]
        code = torch.where(rv, 3 - code, code)
        hit = torch.rand(b - a, generator=gen, device='cuda') < case['sub']
        step = torch.randint(1, 4, (b - a,), generator=gen, device='cuda', dtype=torch.uint8)
        code = torch.where(hit, (code + step) & 3, code)
        out = letters[code.to(torch.int64)]
        if case['n_rate']:
            bad = torch.rand(b - a, generator=gen, device='cuda') < case['n_rate']
            out = torch.where(bad, torch.tensor(ord('N'), dtype=torch.uint8, device='cuda'), out)
        seq[a:b] = out
        r = r1
    return DeviceReads(seq, off, n_bases)


def _graph(case, n_bases):
    sh = lg.CanLemireShifter if case['canonical'] else lg.FwdLemireShifter
    if case['storage'] == 'set':
        # as the set configuration does: told about how many k-mers to expect
        store = lg.SparseppSetStorage.build(capacity_hint=n_bases)
        kind = lg.SparseppSetStorage
    else:
        kind = lg.BitStorage if case['storage'] == 'bloom' else lg.ByteStorage
        store = kind.build(case['max_table'], case['n_tables'])
    g = lg.dBG[kind, sh].build(store, case['K'])
    g.mode = N.MODE_SKIP_N if case['skip_n'] else N.MODE_RAW
    return g


def prepare(case, seed):
    gen = torch.Generator(device='cuda')
    gen.manual_seed(seed)
    genome = _genome(gen, case['genome'])
    d = _reads(case, gen, genome, _lengths(case))
    nk = int((d.offsets.diff() - case['K'] + 1).clamp(min=0).sum())
    st = {'case': case, 'reads': d, 'g': _graph(case, d.n_bases)}
    op = case['op']
    if op == 'host':
        st['reads'] = ReadBatch(d.seq.cpu().numpy(), d.offsets.cpu().numpy())
        return st
    if op in ('insert', 'insert_query'):
        st['n_new'] = torch.zeros(d.n_reads, dtype=torch.int64, device='cuda')
    if op in ('query', 'insert_query', 'insert_and_query'):
        st['counts'] = torch.empty(nk, dtype=torch.int16, device='cuda')
        st['hashes'] = torch.empty(nk, dtype=torch.int64, device='cuda') if case['hashes'] else None
    if op == 'query':
        # the graph holds earlier reads of the same genome, 5x to 15x deep
        more = dict(case, reads=max(1000, min(500_000, 15 * case['genome'] // 150)), read_len=150)
        st['g'].insert_device(_reads(more, gen, genome, _lengths(more)))
        torch.cuda.synchronize()
    if op == 'degrees':
        st['flags'] = torch.zeros(nk, dtype=torch.uint8, device='cuda')
        st['ind'] = torch.empty(nk, dtype=torch.uint8, device='cuda')
        st['outd'] = torch.empty(nk, dtype=torch.uint8, device='cuda')
    if op in ('diginorm', 'solid'):
        st['passed'] = torch.zeros(d.n_reads, dtype=torch.uint8, device='cuda')
        st['filter'] = (lg.DiginormFilter.build(st['g'], case['param']) if op == 'diginorm' else
                        lg.StreamingSolidFilter.build(st['g'], 0.75, case['param']))
    return st


# ---------------------------------------------------------------- one pass

def run(state):
    case, g, d = state['case'], state['g'], state['reads']
    op = case['op']
    if op == 'query':
        g.query_device(d, state['counts'], hashes=state['hashes'])
        return {'counts': state['counts'], 'hashes': state['hashes']}
    g.reset()                                          # a new sample into the same graph
    if op == 'host':
        n_new = g.insert_sequences(d)
        return {'n_new': n_new.astype('int64'), 'counts': g.query_sequences(d), 'n_unique': g.n_unique()}
    if op == 'insert':
        g.insert_device(d, n_new=state['n_new'])
        return {'n_new': state['n_new']}
    if op == 'insert_query':
        g.insert_device(d, n_new=state['n_new'])
        g.query_device(d, state['counts'], hashes=state['hashes'])
        return {'n_new': state['n_new'], 'counts': state['counts'], 'hashes': state['hashes']}
    if op == 'insert_and_query':
        g.insert_and_query_device(d, state['counts'])
        return {'counts': state['counts']}
    if op == 'degrees':
        g.insert_device(d, new_flags=state['flags'])
        g.degrees_device(d, state['ind'], state['outd'], min_count=case['param'], only=state['flags'])
        return {'flags': state['flags'], 'in': state['ind'], 'out': state['outd']}
    # the reads that pass, and the graph's counters for the filter's report
    state['filter'].filter_device(d, state['passed'])
    return {'passed': state['passed'], 'n_unique': g.n_unique(), 'n_occupied': g.n_occupied()}


def work(case):
    """The reads and offsets once, each output once, and the table bytes that
    the windows reach, once to read and (when inserting) once to write."""
    op = case['op']
    bases = case['reads'] * (case['read_len'] or MIX_MEAN)
    if case['read_len']:
        nk = case['reads'] * max(0, case['read_len'] - case['K'] + 1)
    else:
        nk = bases - case['reads'] * (case['K'] - 1)
    if case['storage'] == 'set':
        touched = 8 * min(nk, case['genome'] + nk * min(1.0, case['sub'] * case['K']))
    else:
        table = case['max_table'] * case['n_tables'] / (8 if case['storage'] == 'bloom' else 1)
        touched = min(table, nk * case['n_tables'])
    out = {'insert': 8 * case['reads'], 'query': 2 * nk, 'insert_query': 8 * case['reads'] + 2 * nk,
           'host': 8 * case['reads'] + 2 * nk, 'insert_and_query': 2 * nk, 'degrees': 3 * nk,
           'diginorm': case['reads'], 'solid': case['reads']}[op] + (8 * nk if case['hashes'] else 0)
    passes = 1 if op == 'query' else 3 if op in ('insert_query', 'host', 'degrees') else 2
    reads = 2 if op in ('insert_query', 'host', 'degrees') else 1
    return {'bytes': reads * (bases + 8 * case['reads']) + out + passes * touched, 'flops': 0}


def tolerance(case):
    return 'exact'
