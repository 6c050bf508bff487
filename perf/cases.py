"""The workloads whose speed this repository is judged by, through its public entry points.

Kinds of case (the field "kind"):
  adam    ops.gpu_adam: row-sparse Adam in place on rows of an HBM table
  replay  gpu_ops.replay_rows: initial states plus the logged Adam steps of cold rows
  init    gpu_ops.init_rows: counter-hash initial states of new rows
  dedup   dedup.adam_dedup: a batch with repeated ids, one Adam step per unique id
  batch   dedup.unique, dedup.embedding_dense_backward and ops.gpu_adam in a row: a training step's backward as
          torch.unique and ATen's embedding backward are called, on a batch laid out by (sample, field)
  train   step.ElaraStep and step.run: a short ELARA training run from nothing, then full states of touched rows

Sizes: bench.py's configurations C1 to C5 (C4 and C5 with smaller tables), the widths and K of the tests, and small
and odd batches of the same kinds.  Every result here is defined bit by bit (fp32 operations in a fixed order), so
the tolerance is "exact"; exact() gives the same results in 64 bits.
"""
import functools
import gc
import random

import numpy as np
import torch

from elara_amd import dedup, gpu_ops, ops, step

LR, B1, B2, EPS = ADAM = (1e-3, 0.9, 0.999, 1e-8)
SEED = 42                      # of the counter-hash init
MAX_GAP = 50                   # logged steps of a row are 1..MAX_GAP apart
DIMS = (16, 24, 30, 32, 48, 64, 96, 100, 128, 192, 200, 256, 512)


def listed():
    return [
        # the update of a small batch's rows in a narrow table: the cost of one call
        dict(name='adam_small', kind='adam', R=100_000, D=32, n=600, idx='int32', order='random'),
        # C1: 65,536 rows of a 1M x 64 table
        dict(name='adam_c1', kind='adam', R=1 << 20, D=64, n=65_536, idx='int64', order='random'),
        # an odd number of rows, ascending as a dedup leaves them, of a width that is no power of two
        dict(name='adam_odd', kind='adam', R=1_000_000, D=96, n=150_001, idx='int32', order='sorted'),
        # C4's rows and width on a table that leaves room for other states
        dict(name='adam_wide', kind='adam', R=4_000_000, D=256, n=262_144, idx='int64', order='random'),
        # C2: the cold rows of a large batch, one to three logged gradients each
        dict(name='replay_c2', kind='replay', n=262_144, D=128, K=3, cmin=1),
        # a small batch's cold rows, some of them with an empty log, in a narrow table
        dict(name='replay_odd', kind='replay', n=5_003, D=32, K=4, cmin=0),
        # the states of a table's new rows
        dict(name='init_new', kind='init', n=1_000_003, D=64),
        # a serving-sized batch: at most 3,072 ids, which ATen sums window by window
        dict(name='dedup_small', kind='dedup', B=100, F=26, V=4_000, alpha=1.1, D=32),
        # an odd batch of a width that is no power of two
        dict(name='dedup_odd', kind='dedup', B=4_099, F=26, V=50_000, alpha=1.1, D=48),
        # C3: 131,072 samples of 26 fields, 10M x 128 table
        dict(name='dedup_c3', kind='dedup', B=131_072, F=26, V=384_615, alpha=1.05, D=128),
        # C5's batch through the ATen-shaped calls (the drop-in use: no bound given)
        dict(name='batch_c5', kind='batch', B=16_384, F=26, lo=1_000, hi=1_000_000, alpha=1.1, D=128, bound=False),
        # C5's batch, width, K and residency over 24 steps, tables of up to 4M rows
        dict(name='train_c5', kind='train', B=16_384, F=26, lo=1_000, hi=4_000_000, alpha=1.1, D=128, K=3, steps=24),
    ]


def _logu(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(('adam', 'adam', 'replay', 'init', 'dedup', 'dedup', 'batch', 'train'))
    D = rng.choice(DIMS)
    if kind == 'adam':
        n = _logu(rng, 100, min(600_000, 2_000_000_000 // (28 * D)))
        R = _logu(rng, max(2 * n, 10_000), max(2 * n, 10_000, 8_000_000_000 // (12 * D) // 4))
        return dict(kind=kind, R=R, D=D, n=n, idx=rng.choice(('int32', 'int64')), order=rng.choice(('random', 'sorted')))
    if kind == 'replay':
        K = rng.choice((1, 2, 3, 3, 3, 4, 5, 8))
        n = _logu(rng, 100, min(400_000, 1_000_000_000 // ((12 + 4 * K) * D)))
        return dict(kind=kind, n=n, D=D, K=K, cmin=rng.choice((0, 1)))
    if kind == 'init':
        return dict(kind=kind, n=_logu(rng, 100, min(2_000_000, 2_000_000_000 // (12 * D))), D=D)
    alpha = rng.choice((1.05, 1.1, 1.2))
    F = rng.choice((1, 3, 8, 13, 26, 39))
    if kind == 'dedup':
        B = _logu(rng, 40, min(131_072, 1_500_000_000 // (4 * D * F)))
        V = _logu(rng, 100, min(400_000, 6_000_000_000 // (12 * D * F)))
        return dict(kind=kind, B=B, F=F, V=V, alpha=alpha, D=D)
    if kind == 'batch':
        B = _logu(rng, 40, min(32_768, 800_000_000 // (4 * D * F)))
        hi = _logu(rng, 2_000, min(1_000_000, 4_000_000_000 // (12 * D * F)))
        return dict(kind=kind, B=B, F=F, lo=100, hi=hi, alpha=alpha, D=D, bound=rng.choice((False, True)))
    D = rng.choice((32, 64, 96, 128))
    F = rng.choice((4, 8, 13, 26))
    return dict(kind=kind, B=_logu(rng, 100, 8_192), F=F, lo=100, hi=_logu(rng, 2_000, 1_000_000), alpha=alpha, D=D,
                K=rng.choice((2, 3, 3, 4)), steps=rng.choice((11, 16, 21)))


# ---- inputs, from the seed alone -------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator('cuda').manual_seed(int(seed))


def _bound(D):
    return float(np.float32(1.0 / np.sqrt(D)))


def _pool(g, R, D):
    """A trained table [R, 3, D]: weights in the init range, first and second moments of gradients of about 1e-3."""
    p = torch.empty(R, 3, D, device='cuda')
    p[:, 0].uniform_(-_bound(D), _bound(D), generator=g)
    p[:, 1].normal_(0, 3e-4, generator=g)
    p[:, 2].normal_(0, 1e-3, generator=g).square_()
    return p


def _grads(g, n, D):
    return torch.randn(n, D, device='cuda', generator=g) * 1e-3


def _vocab(case):
    """Rows of each field's table: V each, or log-uniform in [lo, hi] (fixed by the case)."""
    if 'V' in case:
        return [case['V']] * case['F']
    rng = random.Random(case['F'])
    return [_logu(rng, case['lo'], case['hi']) for _ in range(case['F'])]


def _offsets(vocab):
    return [sum(vocab[:f]) for f in range(len(vocab))]


def _ids(g, case, vocab):
    """A batch's row ids in (sample, field) order: in each field a bounded Zipf(alpha) popularity (the power law's
    distribution function inverted and floored), its ranks spread over the table by a multiplicative bijection."""
    v = torch.tensor(vocab, dtype=torch.float64, device='cuda')
    vi = torch.tensor(vocab, device='cuda')
    off = torch.tensor(_offsets(vocab), device='cuda')
    a = torch.tensor([next(p for p in (1_000_003, 999_983) if x % p) for x in vocab], device='cuda')
    u = torch.rand(case['B'], case['F'], dtype=torch.float64, device='cuda', generator=g)
    e = 1.0 - case['alpha']
    k = ((1.0 + u * ((v + 1.0) ** e - 1.0)) ** (1.0 / e)).floor().long() - 1
    k = torch.minimum(k.clamp(min=0), vi - 1)
    return ((a * k + 7 * torch.arange(case['F'], device='cuda')) % vi + off).reshape(-1)


@functools.lru_cache(maxsize=64)
def _unique_share(B, vocab, alpha):
    """Expected unique ids of a batch over its occurrences."""
    e, U = 1.0 - alpha, 0.0
    for V in vocab:
        x = np.arange(1, V + 2, dtype=np.float64) ** e
        p = (x[1:] - x[:-1]) / ((V + 1.0) ** e - 1.0)
        U += float((1.0 - np.exp(B * np.log1p(-np.minimum(p, 1 - 1e-12)))).sum())
    return U / (B * len(vocab))


def _inputs(case, seed):
    g, kind, D = _gen(seed), case['kind'], case['D']
    t = 1 + seed % 997
    if kind == 'adam':
        pool = _pool(g, case['R'], D)
        slots = torch.randperm(case['R'], device='cuda', generator=g)[:case['n']]
        if case['order'] == 'sorted':
            slots = slots.sort().values
        return dict(pool=pool, slots=slots.to(getattr(torch, case['idx'])), grad=_grads(g, case['n'], D), t=t)
    if kind in ('replay', 'init'):
        n = case['n']
        rows = torch.randint(0, 1 << 22, (n,), device='cuda', generator=g)
        if kind == 'init':
            return dict(rows=rows)
        K = case['K']
        cnt = torch.randint(case['cmin'], K + 1, (n,), device='cuda', generator=g)
        steps = torch.randint(1, MAX_GAP + 1, (n, K), device='cuda', generator=g).cumsum(1)
        steps *= torch.arange(K, device='cuda')[None, :] < cnt[:, None]
        logs = _grads(g, int(cnt.sum()), D)
        return dict(rows=rows, cnt=cnt.int(), steps=steps.int(), offs=cnt.cumsum(0) - cnt, logs=logs)
    vocab = _vocab(case)
    R = sum(vocab)
    if kind in ('dedup', 'batch'):
        ids = _ids(g, case, vocab)
        return dict(pool=_pool(g, R, D), ids=ids, grad=_grads(g, ids.numel(), D), t=t, R=R)
    batches = [_ids(g, case, vocab) for _ in range(case['steps'])]
    grads = [_grads(g, batches[0].numel(), D) for _ in range(4)]
    # the most frequent rows of a few profiling batches stay resident (the static hot set)
    u, c = torch.unique(torch.cat([_ids(g, case, vocab) for _ in range(4)]), return_counts=True)
    n_static = min(u.numel() // 2, 20 * case['B'])
    static = u[torch.sort(c, descending=True, stable=True).indices[:n_static]].sort().values
    # the states read at the end: as many rows as a batch has ids, spread evenly over the rows the run touches
    rows, n = torch.unique(torch.cat(batches)), batches[0].numel()
    rows = rows[torch.arange(n, device='cuda') * rows.numel() // n]
    return dict(batches=batches, grads=grads, static=static, vocab=vocab, R=R, rows=rows)


def prepare(case, seed):
    s = _inputs(case, seed)
    s['case'] = case
    if case['kind'] == 'replay':
        s['table'] = gpu_ops.ScalarTable(*ADAM, case['K'] * MAX_GAP, 'cuda')
    if case['kind'] == 'train':
        # as step.run does around its loop by default: what exists now is kept out of the collector's passes
        gc.collect()
        gc.freeze()
    return s


def run(s):
    case = s['case']
    kind, D = case['kind'], case['D']
    if kind == 'adam':
        ops.gpu_adam(s['pool'], s['slots'], s['grad'], *ADAM, s['t'])
        return s['pool']
    if kind == 'replay':
        return gpu_ops.replay_rows(s['rows'], s['logs'], s['offs'], s['steps'], s['cnt'], D, case['K'], SEED,
                                   _bound(D), s['table'])
    if kind == 'init':
        return gpu_ops.init_rows(s['rows'], D, SEED, _bound(D))
    if kind == 'dedup':
        dedup.adam_dedup(s['pool'], s['ids'], s['grad'], *ADAM, s['t'])
        return s['pool']
    if kind == 'batch':
        u, inv = dedup.unique(s['ids'], s['R'] if case['bound'] else None)
        g = dedup.embedding_dense_backward(s['grad'], inv, u.numel())
        ops.gpu_adam(s['pool'], u, g, *ADAM, s['t'])
        return dict(inv=inv, pool=s['pool'])
    nb, O = case['steps'], s['batches'][0].numel()
    n0 = s['static'].numel()
    es = step.ElaraStep(_offsets(s['vocab']), s['R'], D, n0 + max(case['B'], 256), static_rows=s['static'],
                        K=case['K'], kthr=case['K'], evl=True, L=8, depth=3, st_mode='T', seed=SEED, bound=_bound(D),
                        hp=ADAM, max_step=nb + 2, log_cap=nb * O + 16, mat_cap=nb * O + 16, device='cuda:0',
                        field_layout=True)
    step.run(es, s['batches'], lambda j: s['grads'][j % 4], freeze_gc=False)
    states, code = es.eval_weights(s['rows'], full=True), es.code
    # a step and its backend refer to each other: a finished run's arenas come back with the collector
    del es
    gc.collect()
    return dict(states=states, code=code)


# ---- work and tolerance ----------------------------------------------------------------------------------------

def work(case):
    """Bytes: every input read and output written once.  Flops: about 20 per element and Adam step, one per summed
    gradient element, 12 per initial weight."""
    kind, D = case['kind'], case['D']
    if kind == 'adam':
        n = case['n']
        return dict(bytes=n * (28 * D + (4 if case['idx'] == 'int32' else 8)), flops=20 * n * D)
    if kind == 'replay':
        n, K = case['n'], case['K']
        c = (case['cmin'] + K) / 2
        return dict(bytes=n * (20 + 4 * K + 12 * D + 4 * D * c), flops=n * D * (12 + 20 * c))
    if kind == 'init':
        return dict(bytes=case['n'] * (8 + 12 * D), flops=12 * case['n'] * D)
    O = case['B'] * case['F']
    U = O * _unique_share(case['B'], tuple(_vocab(case)), case['alpha'])
    if kind == 'dedup':
        return dict(bytes=O * (4 * D + 8) + U * 24 * D, flops=O * D + 20 * U * D)
    if kind == 'batch':   # ids, unique ids and inverse; gradients and their sums (written, read); states
        return dict(bytes=O * (4 * D + 24) + U * (32 * D + 16), flops=O * D + 20 * U * D)
    # per step the occurrences' gradients and, per unique row, a full state read and written for about half of them
    # and a logged gradient or a new state for the others; at the end a batch's worth of rows' states
    return dict(bytes=case['steps'] * (O * (4 * D + 8) + U * 16 * D) + O * 24 * D,
                flops=case['steps'] * (O * D + 20 * U * D))


def tolerance(case):
    """Every output is defined bit by bit: fp32 Adam in the reference's operation order, ATen's summation order of
    duplicate ids, the counter hash, sorted unique ids."""
    return 'exact'


# ---- the same results in 64 bits -------------------------------------------------------------------------------

def _adam64(x, g, t):
    """x [n, 3, D] float64 (w, m, v) after one Adam step with gradients g at step t (a number, or one per row)."""
    t = torch.as_tensor(t, dtype=torch.float64, device=x.device).reshape(-1, 1)
    m = B1 * x[:, 1] + (1 - B1) * g
    v = B2 * x[:, 2] + (1 - B2) * g * g
    w = x[:, 0] - LR * (m / (1 - B1 ** t)) / ((v / (1 - B2 ** t)).sqrt() + EPS)
    return torch.stack([w, m, v], 1)


def _fmix32(x):
    x = x ^ (x >> 16)
    x = (x * 0x85EBCA6B) & 0xFFFFFFFF
    x = x ^ (x >> 13)
    x = (x * 0xC2B2AE35) & 0xFFFFFFFF
    return x ^ (x >> 16)


def _init64(rows, D):
    """Initial states [n, 3, D]: MurmurHash3's finalizer of (row * D + j), the row's high word and the seed."""
    key = _fmix32(((rows >> 32) + SEED) & 0xFFFFFFFF)
    x = (rows[:, None] * D + torch.arange(D, device=rows.device)) & 0xFFFFFFFF
    h = _fmix32(x ^ key[:, None] ^ SEED)
    w = ((h >> 8).double() * 2.0 ** -23 - 1.0) * _bound(D)
    return torch.stack([w, torch.zeros_like(w), torch.zeros_like(w)], 1)


def _sum64(inv, grad, U):
    return torch.zeros(U, grad.shape[1], dtype=torch.float64, device='cuda').index_add_(0, inv, grad.double())


def exact(case, seed):
    s, kind, D = _inputs(case, seed), case['kind'], case['D']
    if kind == 'adam':
        rows = s['slots'].long()
        out = s['pool'].double()
        out[rows] = _adam64(out[rows], s['grad'].double(), s['t'])
        return out
    if kind == 'init':
        return _init64(s['rows'], D)
    if kind == 'replay':
        x = _init64(s['rows'], D)
        for k in range(case['K']):
            i = (s['cnt'] > k).nonzero().flatten()
            x[i] = _adam64(x[i], s['logs'][s['offs'][i] + k].double(), s['steps'][i, k])
        return x
    if kind in ('dedup', 'batch'):
        u, inv = torch.unique(s['ids'], return_inverse=True)
        g = _sum64(inv, s['grad'], u.numel())
        out = s['pool'].double()
        out[u] = _adam64(out[u], g, s['t'])
        return out if kind == 'dedup' else dict(inv=None, pool=out)
    rows = torch.unique(torch.cat(s['batches']))
    x = _init64(rows, D)
    for j, ids in enumerate(s['batches']):
        u, inv = torch.unique(ids, return_inverse=True)
        i = torch.searchsorted(rows, u)
        x[i] = _adam64(x[i], _sum64(inv, s['grads'][j % 4], u.numel()), j + 1)
    return dict(states=x[torch.searchsorted(rows, s['rows'])], code=None)
