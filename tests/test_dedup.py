"""Batch dedup and duplicate-id gradient reduction (srm2/train.py:352 torch.unique, train.py:429
embedding_dense_backward) and the fused duplicate-id Adam of config C3.

The sums follow ATen's embedding_dense_backward on this GPU (third-party code the reference calls): up to 3072
indices, per window of 16 consecutive indices the id's gradients left to right, the window sums added into a zeroed
row; above, per id its occurrences in runs of 10, each run summed from zero, the run sums added from zero.  The CPU
tests pin the oracle against ATen's own output (tests/golden/aten_segsum.npz, made on the GPU by
tests/golden/make_aten_segsum.py) and by properties of the two orders; the GPU tests hold the HIP path to the
oracle and to the live ATen op bitwise.
"""
import importlib.util
from pathlib import Path

import numpy as np
import pytest
import torch

from elara_amd import synth
from oracle import oracle as O

HP = synth.ADAM
GOLDEN = Path(__file__).resolve().parent / 'golden'
ATEN_SMALL = 3072


def golden_module():
    spec = importlib.util.spec_from_file_location('make_aten_segsum', GOLDEN / 'make_aten_segsum.py')
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def lr_sum(rows, start=None):
    """Left-to-right float32 sum of rows, starting from `start` (None: from rows[0])."""
    acc = rows[0].astype(np.float32).copy() if start is None else np.float32(start) + rows[0]
    for r in rows[1:]:
        acc = (acc + r).astype(np.float32)
    return acc


def full_sums(ids, g, U):
    """Oracle sums as a [U, D] table (rows without an id are zero), as embedding_dense_backward returns them."""
    u, s, _ = O.segment_sum(ids, g)
    out = np.zeros((U, g.shape[1]), np.float32)
    out[u] = s
    return out


# ------------------------------------------------------------------------------------------------------------ CPU
def test_oracle_segment_sum_matches_aten_golden():
    """The oracle reproduces ATen's embedding_dense_backward bit for bit on both of its paths (fixture made by
    running the ATen op on the GPU)."""
    mod = golden_module()
    z = np.load(GOLDEN / 'aten_segsum.npz')
    assert np.array_equal(z['cases'], mod.CASES)
    for ci, c in enumerate(mod.CASES):
        ids, g = mod.case_inputs(*c)
        assert np.array_equal(mod.checksum(ids, g), z[f'case{ci}_sum']), ci       # same inputs as ATen saw
        assert np.array_equal(bits(full_sums(ids, g, int(c[1]))), z[f'case{ci}_out']), ci


def test_oracle_sort_path_sums_runs_of_ten_from_zero():
    """Above 3072 indices: an id with 205 occurrences (interleaved with 3000 distinct others) sums runs of 10 from
    zero, then the run sums from zero.  Values are chosen so that the plain left-to-right sum and runs of other
    lengths give different bits, and a column of -0.0 comes out +0.0."""
    rng = np.random.default_rng(1)
    n_hot, n = 205, 205 + 3000
    pos = np.sort(rng.choice(n, n_hot, replace=False))
    ids = np.arange(10, 10 + n, dtype=np.int64)
    ids[pos] = 7
    g = (rng.standard_normal((n, 4)) * 1e4).astype(np.float32)
    hot = np.zeros((n_hot, 4), np.float32)
    hot[:, 0] = rng.standard_normal(n_hot).astype(np.float32) * np.float32(1e-3)
    hot[0, 1], hot[1:, 1] = np.float32(1.0), np.float32(2.0 ** -24)
    hot[:, 2] = (rng.standard_normal(n_hot) * 1e4).astype(np.float32)
    hot[:, 3] = np.float32(-0.0)
    g[pos] = hot
    assert n > ATEN_SMALL
    u, s, _ = O.segment_sum(ids, g)
    got = s[np.searchsorted(u, 7)]
    runs = lambda L: lr_sum(np.stack([lr_sum(hot[c:c + L], 0.0) for c in range(0, n_hot, L)]), 0.0)  # noqa: E731
    assert np.array_equal(bits(got), bits(runs(10)))
    for other in (lr_sum(hot), runs(64), runs(9), runs(11)):
        assert not np.array_equal(bits(got), bits(other))
    assert bits(got)[3] == 0                                                   # -0 sums to +0


def test_oracle_window_path_sums_windows_of_sixteen():
    """Up to 3072 indices: per window of 16 positions the id's gradients left to right, then the window sums added
    to a zero row.  Id 5 sits at positions 3, 9, 15 (window 0), 16, 30 (window 1) and 47 (window 2)."""
    rng = np.random.default_rng(4)
    n = 60
    ids = rng.integers(20, 40, n).astype(np.int64)
    at = [3, 9, 15, 16, 30, 47]
    ids[at] = 5
    g = (rng.standard_normal((n, 6)) * np.exp2(rng.integers(-20, 20, (n, 6)))).astype(np.float32)
    g[at, 0] = np.float32(2.0 ** -24)
    g[3, 0] = np.float32(1.0)          # windows of 16: (1 + e + e) + (e + e) keeps 2e; one group or 32 keeps none
    g[at, 5] = np.float32(-0.0)
    got = full_sums(ids, g, 40)[5]
    win = lambda groups: lr_sum(np.stack([lr_sum(g[q]) for q in groups]), 0.0)  # noqa: E731
    want = win([[3, 9, 15], [16, 30], [47]])
    assert np.array_equal(bits(got), bits(want))
    assert not np.array_equal(bits(got), bits(win([[3, 9, 15, 16, 30], [47]])))     # windows of 32
    assert not np.array_equal(bits(got), bits(lr_sum(g[at], 0.0)))                    # one group
    assert bits(got)[5] == 0


def test_oracle_sort_path_depends_only_on_each_ids_occurrence_order():
    """Above 3072 indices, interleaving other ids differently does not change an id's sum."""
    rng = np.random.default_rng(2)
    a = (rng.standard_normal((2150, 8)) * 1e3).astype(np.float32)
    b = (rng.standard_normal((1090, 8))).astype(np.float32)
    x_ids = np.concatenate([np.full(2150, 3), np.full(1090, 9)]).astype(np.int64)
    x_g = np.concatenate([a, b])
    perm = rng.permutation(3240)
    order = np.concatenate([np.sort(perm[:2150]), np.sort(perm[2150:])])   # each id keeps its own order
    y_ids = np.empty(3240, np.int64)
    y_g = np.empty_like(x_g)
    y_ids[order] = x_ids
    y_g[order] = x_g
    ux, sx, _ = O.segment_sum(x_ids, x_g)
    uy, sy, _ = O.segment_sum(y_ids, y_g)
    assert np.array_equal(ux, uy) and np.array_equal(bits(sx), bits(sy))


def test_oracle_segment_sum_matches_torch_unique_and_totals():
    rng = np.random.default_rng(3)
    z = synth.ZipfFields([5000] * 4, 1.05, seed=3, offsets=[0] * 4)
    ids = z.draw(rng, 3000)
    g = rng.standard_normal((ids.size, 8)).astype(np.float32)
    u, s, inv = O.segment_sum(ids, g)
    tu, tinv = torch.unique(torch.from_numpy(ids), return_inverse=True)
    assert np.array_equal(tu.numpy(), u) and np.array_equal(tinv.numpy(), inv)
    # the per-id sums add up to the column totals (fp64 check; tolerance for the fp32 roundings)
    assert np.allclose(s.astype(np.float64).sum(0), g.astype(np.float64).sum(0), rtol=1e-4, atol=1e-2)


def test_zipf_fields_shape_and_range():
    z = synth.ZipfFields([1000, 50, 7], 1.1, seed=4)
    ids = z.draw(np.random.default_rng(4), 2000).reshape(2000, 3)
    assert ids[:, 0].max() < 1000 and ids[:, 1].min() >= 1000 and ids[:, 1].max() < 1050
    assert ids[:, 2].min() >= 1050 and ids[:, 2].max() < 1057
    # rank 0 (the hottest) is the most frequent row of a field
    r = z.ranks(np.random.default_rng(5), 20000)[:, 0]
    assert np.bincount(r).argmax() == 0


# ------------------------------------------------------------------------------------------------------------ GPU
def zipf_case(seed, n_samples, fields, vocab, alpha, D, scale=1e-3):
    rng = np.random.default_rng(seed)
    z = synth.ZipfFields([vocab] * fields, alpha, seed=seed, offsets=[0] * fields)
    ids = z.draw(rng, n_samples)
    g = (rng.standard_normal((ids.size, D)) * scale).astype(np.float32)
    return ids, g


@pytest.mark.gpu
@pytest.mark.parametrize('case', ['zipf', 'big_ids', 'one_id', 'distinct', 'single'])
def test_gpu_unique_matches_torch(dev, case):
    from elara_amd.dedup import unique
    rng = np.random.default_rng(10)
    ids = {'zipf': lambda: zipf_case(10, 20000, 26, 100000, 1.05, 1)[0],
           'big_ids': lambda: rng.integers(0, 2**40, 50000) // 7 * 7,
           'one_id': lambda: np.full(70000, 123456789, np.int64),
           'distinct': lambda: rng.permutation(300000),
           'single': lambda: np.array([5])}[case]().astype(np.int64)
    print(f'[gpu-test] unique {case} n={ids.size}', flush=True)
    u, inv = unique(torch.from_numpy(ids).to(dev))
    tu, tinv = torch.unique(torch.from_numpy(ids), return_inverse=True)
    assert torch.equal(u.cpu(), tu) and torch.equal(inv.cpu(), tinv)


@pytest.mark.gpu
@pytest.mark.parametrize('key_bits', [1, 8, 9, 12, 17, 20, 24, 27, 30, 32, 33, 40, 63])
@pytest.mark.parametrize('n', [1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 70001, (1 << 18) - 1, (1 << 18) + 3,
                               (1 << 20) - 1, 1 << 20, (1 << 21) + 3])
def test_gpu_unique_every_digit_width(dev, key_bits, n):
    """The sort takes 8-, 9- or 10-bit digits (fewer passes: 27-bit keys in 3 passes of 9 bits, 30-bit keys in 3 of
    10) with 1,024 or 256 threads per tile (either side of 2^20 ids), and up to 8,192 ids one block of 1 to 8 keys per
    thread; for each key width from the caller's bound, each gives torch.unique's rows and inverse.  Ids are spread over the
    whole width, with duplicates and the extreme keys 0 and 2^b - 1."""
    from elara_amd.dedup import unique
    rng = np.random.default_rng(key_bits * 7 + n % 5)
    hi = (1 << key_bits) - 1
    ids = rng.integers(0, hi, n, dtype=np.int64, endpoint=True)
    ids[rng.integers(0, n, n // 3)] = ids[rng.integers(0, n, n // 3)]     # duplicates
    ids[:2], ids[-1] = [0, hi], hi
    print(f'[gpu-test] unique key_bits={key_bits} n={n}', flush=True)
    u, inv = unique(torch.from_numpy(ids).to(dev), bound=hi + 1)
    tu, tinv = torch.unique(torch.from_numpy(ids), return_inverse=True)
    assert torch.equal(u.cpu(), tu) and torch.equal(inv.cpu(), tinv)


@pytest.mark.gpu
@pytest.mark.parametrize('D', [128, 64, 30, 200])
def test_gpu_embedding_backward_matches_oracle(dev, D):
    from elara_amd.dedup import embedding_dense_backward
    print(f'[gpu-test] segment sum D={D}', flush=True)
    ids, g = zipf_case(11, 8000, 26, 50000, 1.05, D, scale=1.0)
    u, s, inv = O.segment_sum(ids, g)
    # the reference's call: indices are the inverse (unique positions), num_weights = U
    out = embedding_dense_backward(torch.from_numpy(g).to(dev), torch.from_numpy(inv).to(dev), u.size)
    torch.cuda.synchronize()
    assert np.array_equal(bits(out.cpu().numpy()), bits(s))
    # raw ids as indices, with rows never indexed left zero
    out2 = embedding_dense_backward(torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev), 50000)
    want = np.zeros((50000, D), np.float32)
    want[u] = s
    assert np.array_equal(bits(out2.cpu().numpy()), bits(want))


ATEN_CASES = [(40, 3, 64), (700, 20, 128), (3072, 9, 256), (3072, 400, 30), (3073, 9, 128), (3073, 7, 512),
              (20000, 600, 200), (120000, 1000, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize('n,U,D', ATEN_CASES)
def test_gpu_embedding_backward_matches_aten(dev, n, U, D):
    """Bitwise equal to torch.ops.aten.embedding_dense_backward run on the same GPU (the call of
    srm2/train.py:429), on ATen's windowed path (n <= 3072) and its sorted path, with a hot id, -0.0 gradients and
    gradients over 2^-20 .. 2^20; also through the dedup plan (segment_sum_plan over the inverse)."""
    from elara_amd.dedup import embedding_dense_backward, segment_sum_plan, unique_plan
    print(f'[gpu-test] aten segment sum n={n} U={U} D={D}', flush=True)
    ids, g = golden_module().case_inputs(n, U, D, n + U, U - 1, 3)
    gd, idd = torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev)
    want = torch.ops.aten.embedding_dense_backward(gd, idd, U, -1, False)
    got = embedding_dense_backward(gd, idd, U)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got.cpu().numpy()), bits(want.cpu().numpy()))
    assert np.array_equal(bits(got.cpu().numpy()), bits(full_sums(ids, g, U)))
    u, plan = unique_plan(idd, D, U)
    out = torch.zeros(U, D, device=dev)
    segment_sum_plan(gd, plan, out, u)
    torch.cuda.synchronize()
    assert np.array_equal(bits(out.cpu().numpy()), bits(want.cpu().numpy()))


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1 << 20, (1 << 20) + 1])
def test_gpu_segment_block_offsets_both_ways(dev, n):
    """The segment launches at a batch that fills its tiles and at one id more (512 and 513 segment tiles, whose offsets
    each block sums; the scan launch that gives them above 2,048 tiles: test_gpu_sort_and_segments_at_their_limits):
    unique equals torch.unique and the sums equal ATen's embedding_dense_backward, with a hot id."""
    from elara_amd.dedup import embedding_dense_backward, unique
    U, D = 300_000, 64
    print(f'[gpu-test] block offsets n={n}', flush=True)
    ids, g = golden_module().case_inputs(n, U, D, 11, U - 1, 2)
    gd, idd = torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev)
    u, inv = unique(idd, bound=U)
    tu, tinv = torch.unique(idd, return_inverse=True)
    assert torch.equal(u, tu) and torch.equal(inv, tinv)
    want = torch.ops.aten.embedding_dense_backward(gd, idd, U, -1, False)
    got = embedding_dense_backward(gd, idd, U)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got.cpu().numpy()), bits(want.cpu().numpy()))


@pytest.mark.gpu
@pytest.mark.parametrize('D', [128, 64, 256, 512, 96])
def test_gpu_segment_lengths_at_every_boundary(dev, D):
    """Ids whose occurrence counts sit on each boundary of the kernels' work split -- runs of 10, the first chunk
    of 60 folded by the id's own wave, partial chunks of 60, hot ids (more than 240 occurrences, folded by a whole
    block) -- among 4,000 single-occurrence ids: sums bitwise equal to ATen's and the oracle's, and the fused
    duplicate-id Adam equal to the oracle's sum followed by cpu_adam."""
    from elara_amd.dedup import adam_dedup, embedding_dense_backward
    print(f'[gpu-test] segment boundaries D={D}', flush=True)
    lens = [1, 2, 9, 10, 11, 19, 20, 21, 59, 60, 61, 119, 120, 121, 239, 240, 241, 242, 299, 300, 301, 601, 2999]
    rng = np.random.default_rng(31)
    ids = np.concatenate([np.full(L, 10 + 7 * k) for k, L in enumerate(lens)] + [np.arange(1000, 5000)])
    ids = ids[rng.permutation(ids.size)].astype(np.int64)
    U = 5000
    g = (rng.standard_normal((ids.size, D)) * np.exp2(rng.integers(-12, 12, (ids.size, 1)))).astype(np.float32)
    gd, idd = torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev)
    want = full_sums(ids, g, U)
    got = embedding_dense_backward(gd, idd, U)
    aten = torch.ops.aten.embedding_dense_backward(gd, idd, U, -1, False)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got.cpu().numpy()), bits(want))
    assert np.array_equal(bits(aten.cpu().numpy()), bits(want))
    state = np.zeros((U, 3, D), np.float32)
    state[:, 0] = (rng.standard_normal((U, D)) * 0.05).astype(np.float32)
    gpu = torch.from_numpy(state).to(dev)
    u, s, _ = O.segment_sum(ids, g)
    O.cpu_adam(state, u, s, O.adam_scalars(*HP, 3), 8)
    adam_dedup(gpu, idd, gd, *HP, 3)
    torch.cuda.synchronize()
    assert np.array_equal(bits(gpu.cpu().numpy()), bits(state))


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1, 17, 3072, 3073, 20_000])
@pytest.mark.parametrize('D', [4, 12, 16, 24, 48, 100, 192, 320])
def test_gpu_segment_lengths_in_chunk_layout(dev, D, n):
    """Widths whose rows move in 16-byte chunks (a multiple of 4 other than 64, 128, 256, 512; each number of lanes per
    row and two chunks per lane), both summation orders, with ids on each boundary of the work split: runs of 10,
    the lanes' 4 to 64 occurrence indices, windows of 16, the hot limits (64 windowed, 240 sorted), a hot id that fills
    the staging area several times.  Sums bitwise ATen's on this GPU and the oracle's, the fused Adam the oracle's."""
    from elara_amd.dedup import adam_dedup, embedding_dense_backward
    print(f'[gpu-test] chunk layout D={D} n={n}', flush=True)
    rng = np.random.default_rng(n + D)
    lens = [1, 2, 3, 4, 5, 8, 9, 10, 11, 15, 16, 17, 20, 21, 32, 33, 60, 61, 64, 65, 66, 240, 241, 600]
    lens = lens + [1100] if n > 3072 else lens
    ids = np.concatenate([np.full(L, 10 + 7 * k) for k, L in enumerate(lens)])[:n]
    ids = np.concatenate([ids, 1000 + np.arange(n - ids.size)])
    ids = ids[rng.permutation(n)].astype(np.int64)
    U = 1000 + n
    g = (rng.standard_normal((n, D)) * np.exp2(rng.integers(-12, 12, (n, 1)))).astype(np.float32)
    gd, idd = torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev)
    want = full_sums(ids, g, U)
    got = embedding_dense_backward(gd, idd, U)
    aten = torch.ops.aten.embedding_dense_backward(gd, idd, U, -1, False)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got.cpu().numpy()), bits(want))
    assert np.array_equal(bits(aten.cpu().numpy()), bits(want))
    state = np.zeros((U, 3, D), np.float32)
    state[:, 0] = (rng.standard_normal((U, D)) * 0.05).astype(np.float32)
    gpu = torch.from_numpy(state).to(dev)
    u, s, _ = O.segment_sum(ids, g)
    O.cpu_adam(state, u, s, O.adam_scalars(*HP, 3), 8)
    adam_dedup(gpu, idd, gd, *HP, 3)
    torch.cuda.synchronize()
    assert np.array_equal(bits(gpu.cpu().numpy()), bits(state))


@pytest.mark.gpu
@pytest.mark.parametrize('D', [4, 48, 64, 128, 256, 320, 512])
@pytest.mark.parametrize('n,hot', [(66, 65), (3072, 3072), (3000, 1500), (20_000, 20_000), (20_000, 9_999)])
def test_gpu_hot_ids_fill_the_staging_area_many_times(dev, D, n, hot):
    """One id that holds all or half of a batch (8 to 1,024 rows per staging area by width, the last one partly filled, rows
    added 8 or 4 at a time), both summation orders: sums bitwise ATen's on this GPU and the oracle's."""
    from elara_amd.dedup import embedding_dense_backward
    print(f'[gpu-test] hot id D={D} n={n} hot={hot}', flush=True)
    rng = np.random.default_rng(n + D + hot)
    ids = np.full(n, 3, np.int64)
    ids[rng.choice(n, n - hot, replace=False)] = 100 + np.arange(n - hot)
    g = (rng.standard_normal((n, D)) * np.exp2(rng.integers(-12, 12, (n, 1)))).astype(np.float32)
    g[ids == 3, 0] = np.float32(-0.0)
    U = 101 + n - hot
    gd, idd = torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev)
    got = embedding_dense_backward(gd, idd, U)
    aten = torch.ops.aten.embedding_dense_backward(gd, idd, U, -1, False)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got.cpu().numpy()), bits(full_sums(ids, g, U)))
    assert np.array_equal(bits(got.cpu().numpy()), bits(aten.cpu().numpy()))


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1 << 22, (1 << 22) + 1, 9_000, 530_000])
def test_gpu_sort_and_segments_at_their_limits(dev, n):
    """The sort with its digit counts added up in the scatter (up to 128 tiles of 4,096) and from a scan launch, the
    segment offsets from the blocks and (above 2,048 tiles) from a scan launch, an id that spans many tiles and ids
    whose segment ends in a later tile: unique equals torch.unique and the sums equal ATen's."""
    from elara_amd.dedup import embedding_dense_backward, unique
    print(f'[gpu-test] sort and segments n={n}', flush=True)
    U, D = n // 3 + 2, 8
    gen = torch.Generator(dev).manual_seed(n)
    ids = torch.randint(0, U, (n,), device=dev, generator=gen)
    ids[torch.rand(n, device=dev, generator=gen) < 0.3] = U // 2
    ids[torch.rand(n, device=dev, generator=gen) < 0.01] = U - 1
    g = torch.randn(n, D, device=dev, generator=gen)
    u, inv = unique(ids, bound=U)
    tu, tinv = torch.unique(ids, return_inverse=True)
    assert torch.equal(u, tu) and torch.equal(inv, tinv)
    want = torch.ops.aten.embedding_dense_backward(g, ids, U, -1, False)
    got = embedding_dense_backward(g, ids, U)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.gpu
def test_gpu_aten_golden_cases(dev):
    """The HIP sum reproduces the committed ATen vectors (both paths, -0.0 ids, hot ids)."""
    from elara_amd.dedup import embedding_dense_backward
    mod = golden_module()
    z = np.load(GOLDEN / 'aten_segsum.npz')
    for ci, c in enumerate(mod.CASES):
        print(f'[gpu-test] aten golden case {ci}', flush=True)
        ids, g = mod.case_inputs(*c)
        got = embedding_dense_backward(torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev), int(c[1]))
        torch.cuda.synchronize()
        assert np.array_equal(bits(got.cpu().numpy()), z[f'case{ci}_out']), ci


@pytest.mark.gpu
@pytest.mark.parametrize('D,case', [(128, 'zipf'), (64, 'long'), (30, 'zipf'), (128, 'big_ids'), (128, 'bits27'),
                                    (64, 'bits17')])
def test_gpu_dedup_plan_matches_unique_and_backward(dev, D, case):
    """unique_plan + segment_sum_plan (one sort reused by the sum) give torch.unique's rows and the oracle's sums,
    into rows u or perm[u] (a permutation, and a scatter into a larger output)."""
    from elara_amd.dedup import segment_sum_plan, unique_plan
    print(f'[gpu-test] dedup plan D={D} {case}', flush=True)
    rng = np.random.default_rng(13)
    if case == 'zipf':
        ids, g = zipf_case(14, 9000, 26, 60000, 1.05, D, scale=1.0)
        bound = None
    elif case == 'long':
        ids = np.concatenate([np.full(5000, 77), rng.integers(0, 3000, 30000)])[rng.permutation(35000)].astype(np.int64)
        g = rng.standard_normal((ids.size, D)).astype(np.float32)
        bound = 3000
    elif case in ('bits27', 'bits17'):       # sorts of 3 passes of 9 bits, 2 passes of 9 bits
        bound = 1 << int(case[4:])
        ids = rng.integers(0, bound, 60000).astype(np.int64)
        ids[rng.integers(0, ids.size, 20000)] = ids[rng.integers(0, ids.size, 20000)]
        g = rng.standard_normal((ids.size, D)).astype(np.float32)
    else:
        ids = (rng.integers(0, 2**40, 40000) // 5 * 5).astype(np.int64)
        g = rng.standard_normal((ids.size, D)).astype(np.float32)
        bound = 2**40
    u_ref, s_ref, _ = O.segment_sum(ids, g)
    u, plan = unique_plan(torch.from_numpy(ids).to(dev), D, bound)
    assert torch.equal(u.cpu(), torch.from_numpy(u_ref))
    gd = torch.from_numpy(g).to(dev)
    out = segment_sum_plan(gd, plan)
    torch.cuda.synchronize()
    assert np.array_equal(bits(out.cpu().numpy()), bits(s_ref))
    perm = torch.from_numpy(rng.permutation(u_ref.size).astype(np.int64))
    big = torch.zeros(u_ref.size + 5, D, device=dev)
    segment_sum_plan(gd, plan, big, (perm + 3).to(dev))
    want = np.zeros((u_ref.size + 5, D), np.float32)
    want[perm.numpy() + 3] = s_ref
    torch.cuda.synchronize()
    assert np.array_equal(bits(big.cpu().numpy()), bits(want))


def field_case(case, rng):
    """(ids [nrows * nfields] in (sample, field) order, field bounds) of a batch laid out by field."""
    if case == 'c5':
        tabs = synth.C5Tables(T=26, lo=1e3, hi=4e7, alpha=1.1, seed=3)
        return tabs.batch(rng, 16384), np.append(tabs.toff, tabs.R)
    vocab = {'ragged': [1, 3, 511, 512, 513, 2**17, 70000],       # 5,000 rows: one hot id per tiny field
             'one_field': [2**20],                                  # 16,384 rows, one block
             'wide': [50] * 100,                                    # 100 rows x 100 fields
             'two_keys': [400, 90000, 17],                          # 1,500 rows: 2 keys per thread
             'four_keys': [400, 90000, 17],                         # 3,000 rows: 4 keys per thread
             'big_span': [2**31 - 2, 5, 40000],                     # keys of 31 bits: 4 passes
             'fallback_rows': [3000, 90000, 17],                    # 20,000 rows: the general sort
             'fallback_small': [100] * 26}[case]                    # 2,600 ids: ATen's windowed order
    nrows = {'ragged': 5000, 'one_field': 16384, 'wide': 100, 'two_keys': 1500, 'four_keys': 3000, 'big_span': 12000, 'fallback_rows': 20000,
             'fallback_small': 100}[case]
    z = synth.ZipfFields(vocab, 1.1, seed=int(rng.integers(1 << 30)))
    return z.draw(rng, nrows), np.append(z.offsets, z.offsets[-1] + z.vocab[-1])


@pytest.mark.gpu
@pytest.mark.parametrize('case', ['c5', 'ragged', 'one_field', 'wide', 'two_keys', 'four_keys', 'big_span', 'fallback_rows',
                                  'fallback_small'])
def test_gpu_dedup_plan_fields_matches_general(dev, case):
    """A batch laid out by field, sorted per field (elr_dedup_plan_fields): the unique ids, the inverse and the
    segment sums over its plan are bitwise those of the general sort's plan and the oracle's; the unique count is
    the same.  Covers both result buffers of the plan (27- and 18-bit bounds), fields of one row (a hot segment of
    every occurrence), digit widths at 2^9 +- 1, 31-bit keys, a hundred fields of 100 rows, each number of keys per
    thread (1, 2, 4, 8, 16), and the shapes that go to the general sort."""
    import ctypes
    from elara_amd import _lib
    from elara_amd.dedup import field_bounds, plan_bytes, segment_sum_plan, unique_plan_async
    print(f'[gpu-test] dedup plan by field {case}', flush=True)
    rng = np.random.default_rng(29)
    ids, lo = field_case(case, rng)
    D = 64 if case == 'wide' else 128
    n, nf, bound = ids.size, lo.size - 1, int(lo[-1])
    t = torch.from_numpy(ids).to(dev)
    u1, p1, nu1 = unique_plan_async(t, D, bound)
    u2, p2, nu2 = unique_plan_async(t, D, bound, fields=field_bounds(lo))
    U = int(nu1)
    assert int(nu2) == U
    assert torch.equal(u1[:U], u2[:U])
    g = rng.standard_normal((n, D)).astype(np.float32)
    u_ref, s_ref, _ = O.segment_sum(ids, g)
    assert np.array_equal(u2[:U].cpu().numpy(), u_ref)
    p1.U = p2.U = U
    gd = torch.from_numpy(g).to(dev)
    s1, s2 = segment_sum_plan(gd, p1), segment_sum_plan(gd, p2)
    torch.cuda.synchronize()
    assert np.array_equal(bits(s2.cpu().numpy()), bits(s_ref))
    assert np.array_equal(bits(s1.cpu().numpy()), bits(s2.cpu().numpy()))
    # the inverse (not asked for by the step)
    inv = torch.full((n,), -5, dtype=torch.int64, device=dev)
    uu, nu = torch.empty(n, dtype=torch.int64, device=dev), torch.empty(1, dtype=torch.int64, device=dev)
    buf = torch.empty(plan_bytes(n, D), dtype=torch.uint8, device=dev)
    fb = field_bounds(lo)
    rc = _lib.lib().elr_dedup_plan_fields(_lib.ptr(t), n // nf, nf, fb.ctypes.data, p2.key_bits, _lib.ptr(uu),
                                          _lib.ptr(inv), _lib.ptr(nu), _lib.ptr(buf), buf.numel(), D,
                                          ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    assert int(nu) == U
    assert np.array_equal(u_ref[inv.cpu().numpy()], ids)


@pytest.mark.gpu
def test_gpu_dedup_plan_fields_flags_ids_outside_their_field(dev):
    """An id that is a valid row of another field breaks the layout's contract: the per-field plan reports it as -1
    (a row out of range for the caller) and keeps every other id and segment sum as the general plan gives them."""
    from elara_amd.dedup import field_bounds, segment_sum_plan, unique_plan_async
    print('[gpu-test] dedup plan by field, id outside its field', flush=True)
    rng = np.random.default_rng(31)
    ids, lo = field_case('ragged', rng)
    nf = lo.size - 1
    bad = 7 * nf + 2                                 # sample 7, field 2 ([4, 515)), given a row of field 5
    ids[bad] = lo[5] + 11
    t = torch.from_numpy(ids).to(dev)
    u, plan, nu = unique_plan_async(t, 128, int(lo[-1]), fields=field_bounds(lo))
    U = int(nu)
    got = u[:U].cpu().numpy()
    assert (got == -1).sum() == 1
    good = np.delete(ids, bad)
    keep = got >= 0
    assert np.array_equal(got[keep], np.unique(good))
    plan.U = U
    g = rng.standard_normal((ids.size, 128)).astype(np.float32)
    s = segment_sum_plan(torch.from_numpy(g).to(dev), plan).cpu().numpy()
    # the sort path groups each id's occurrences from its own first one, so the batch without the flagged occurrence
    # sums every other id the same way
    u_ref, s_ref, _ = O.segment_sum(good, np.delete(g, bad, axis=0))
    assert np.array_equal(got[keep], u_ref)
    assert np.array_equal(bits(s[keep]), bits(s_ref))
    assert np.array_equal(bits(s[~keep][0]), bits(g[bad]))


@pytest.mark.gpu
def test_gpu_segment_sum_very_long_segment(dev):
    """One id with 100,000 occurrences (1,563 chunks) next to short ones."""
    from elara_amd.dedup import embedding_dense_backward
    print('[gpu-test] segment sum long', flush=True)
    rng = np.random.default_rng(12)
    ids = np.concatenate([np.full(100000, 3), rng.integers(0, 1000, 20000)])[rng.permutation(120000)].astype(np.int64)
    g = rng.standard_normal((ids.size, 128)).astype(np.float32)
    u, s, _ = O.segment_sum(ids, g)
    out = embedding_dense_backward(torch.from_numpy(g).to(dev), torch.from_numpy(ids).to(dev), 1000)
    torch.cuda.synchronize()
    want = np.zeros((1000, 128), np.float32)
    want[u] = s
    assert np.array_equal(bits(out.cpu().numpy()), bits(want))


@pytest.mark.gpu
@pytest.mark.parametrize('D,idx', [(128, torch.int64), (64, torch.int32), (96, torch.int64)])
def test_gpu_adam_dedup_matches_oracle(dev, D, idx):
    from elara_amd.dedup import adam_dedup
    print(f'[gpu-test] adam_dedup D={D}', flush=True)
    R = 200000
    rng = np.random.default_rng(13)
    state = np.zeros((R, 3, D), np.float32)
    state[:, 0] = (rng.standard_normal((R, D)) * 0.05).astype(np.float32)
    gpu = torch.from_numpy(state).to(dev)
    for t in range(1, 4):
        ids, g = zipf_case(100 + t, 4000, 26, R, 1.05, D)
        u, s, _ = O.segment_sum(ids, g)
        O.cpu_adam(state, u, s, O.adam_scalars(*HP, t), 8)
        adam_dedup(gpu, torch.from_numpy(ids).to(dev, idx), torch.from_numpy(g).to(dev), *HP, t)
    torch.cuda.synchronize()
    assert np.array_equal(bits(gpu.cpu().numpy()), bits(state))


@pytest.mark.gpu
@pytest.mark.parametrize('D,n_field', [(128, 4000), (96, 4000), (64, 4000), (128, 100)])
def test_gpu_adam_dedup_plan_matches_adam_dedup(dev, D, n_field):
    """elr_adam_dedup_plan over a plan sorted ahead on a second stream equals elr_adam_dedup bitwise (n_field 100:
    2,600 ids, ATen's windowed path)."""
    from elara_amd.dedup import adam_dedup, adam_dedup_plan, unique_plan_async
    print(f'[gpu-test] adam_dedup_plan D={D} n={n_field * 26}', flush=True)
    R = 200000
    rng = np.random.default_rng(17)
    state = torch.from_numpy((rng.standard_normal((R, 3, D)) * 0.05).astype(np.float32)).to(dev)
    a, b = state.clone(), state.clone()
    side = torch.cuda.Stream(device=dev)
    main = torch.cuda.current_stream(dev)
    for t in range(1, 4):
        ids_np, g_np = zipf_case(200 + t, n_field, 26, R, 1.05, D)
        ids, g = torch.from_numpy(ids_np).to(dev), torch.from_numpy(g_np).to(dev)
        side.wait_stream(main)
        with torch.cuda.stream(side):
            u, plan, _ = unique_plan_async(ids, D, R)
            ev = torch.cuda.Event()
            ev.record()
        main.wait_event(ev)
        adam_dedup_plan(b, u, g, plan, *HP, t)
        adam_dedup(a, ids, g, *HP, t)
    torch.cuda.synchronize()
    assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.gpu
def test_gpu_dedup_edge_cases(dev):
    from elara_amd.dedup import adam_dedup, embedding_dense_backward, unique
    z = torch.empty(0, dtype=torch.int64, device=dev)
    u, inv = unique(z)
    assert u.numel() == 0 and inv.numel() == 0
    assert embedding_dense_backward(torch.empty(0, 8, device=dev), z, 5).abs().sum().item() == 0
    pool = torch.randn(10, 3, 8, device=dev)
    ref = pool.clone()
    adam_dedup(pool, z, torch.empty(0, 8, device=dev), *HP, 1)
    torch.cuda.synchronize()
    assert torch.equal(pool, ref)
    # ids out of range are skipped by the kernel's check (undefined in the reference)
    adam_dedup(pool, torch.tensor([3, 3, 10, 1 << 20], device=dev), torch.ones(4, 8, device=dev), *HP, 1)
    torch.cuda.synchronize()
    changed = (pool != ref).any(dim=2).any(dim=1).nonzero().flatten().tolist()
    assert changed == [3]
    with pytest.raises(RuntimeError):
        unique(torch.tensor([-1, 2], device=dev))


@pytest.mark.gpu
@pytest.mark.parametrize('n', [300, 3073, 8192, 8193, 30_000])
@pytest.mark.parametrize('C,D', [(10, 8), (200, 64), (4000, 30), (4096, 8), (16_384, 64), (65_536, 8), (300_000, 8),
                                 (1 << 20, 8), (1 << 21, 8)])
def test_gpu_ids_outside_the_table_leave_valid_rows_alone(dev, C, D, n):
    """Ids that are no row, between the occurrences of valid ids whose low bits they share (-1, C, C + row, row + 2^b on
    each side of the digits' widths and of 32 bits, the extremes of int64), in the one-launch plan and the radix passes and
    in both summation orders: every valid row has the oracle's bits, the others are skipped -- adam_dedup, the same over
    a plan, and the sums of embedding_dense_backward."""
    from elara_amd.dedup import adam_dedup, adam_dedup_plan, embedding_dense_backward, unique_plan
    print(f'[gpu-test] ids outside the table C={C} D={D} n={n}', flush=True)
    rng = np.random.default_rng(C + n)
    rows = np.unique(np.concatenate([[0, 5, C - 1, C // 2], rng.integers(0, C, 40)]))
    ids = rng.choice(rows, n).astype(np.int64)
    i64 = np.iinfo(np.int64)
    out = rng.random(n) < 0.4
    b = rng.choice([4, 8, 9, 10, 12, 14, 16, 18, 20, 21, 24, 32, 33, 48], n)
    far = rng.choice(np.array([-1, -2, C, i64.min, i64.max, (1 << 32) - 1]), n)
    alias = np.where(rng.random(n) < 0.5, ids + (np.int64(1) << b), np.where(rng.random(n) < 0.3, C + ids, far))
    ids = np.where(out & ((alias < 0) | (alias >= C)), alias, ids)
    g = (rng.standard_normal((n, D)) * np.exp2(rng.integers(-12, 12, (n, 1)))).astype(np.float32)
    valid = (ids >= 0) & (ids < C)
    assert valid.any() and not valid.all()
    u, s, _ = O.segment_sum(np.where(valid, ids, C), g)     # (the others: one id of their own, dropped here)
    u, s = u[:-1], s[:-1]
    state = (rng.standard_normal((u.size, 3, D)) * 0.05).astype(np.float32)
    state[:, 2] **= 2
    ud, idd, gd = torch.from_numpy(u).to(dev), torch.from_numpy(ids).to(dev), torch.from_numpy(g).to(dev)
    a = torch.full((C, 3, D), 0.5, device=dev)
    a[ud] = torch.from_numpy(state).to(dev)
    b, idle = a.clone(), torch.ones(C, dtype=torch.bool, device=dev)
    idle[ud] = False
    O.cpu_adam(state, np.arange(u.size), s, O.adam_scalars(*HP, 3), 2)
    adam_dedup(a, idd, gd, *HP, 3)
    pu, plan = unique_plan(idd, D, C)
    adam_dedup_plan(b, pu, gd, plan, *HP, 3)
    sums = embedding_dense_backward(gd, idd, C)
    torch.cuda.synchronize()
    assert np.array_equal(bits(a[ud].cpu().numpy()), bits(state)) and bool((a[idle] == 0.5).all())
    assert torch.equal(a, b)
    assert np.array_equal(bits(sums[ud].cpu().numpy()), bits(s)) and not bool(sums[idle].any())
    got = pu.cpu().numpy()
    assert np.array_equal(got[(got >= 0) & (got < C)], u) and (np.diff(got) > 0).all()


class _OraclePipe:
    """The CPU side of a long full-size run: each step's oracle work split into a part that is independent per step
    (`prep`, run by a pool of threads, several steps at once; the oracle's C calls release the GIL) and the part
    that carries state from step to step (`apply`, run here, in step order).  drain() applies every submitted
    step; at most `depth` steps are in flight (each holds its gradients in host memory)."""

    def __init__(self, prep, apply, workers=6, depth=6):
        from concurrent.futures import ThreadPoolExecutor
        self.prep, self.apply, self.depth = prep, apply, depth
        self.pool = ThreadPoolExecutor(workers)
        self.q = []

    def submit(self, t, *args):
        self.q.append((t, self.pool.submit(self.prep, t, *args)))
        while len(self.q) > self.depth:
            self._pop()

    def _pop(self):
        t, f = self.q.pop(0)
        self.apply(t, f.result())

    def drain(self):
        while self.q:
            self._pop()

    def close(self):
        self.drain()
        self.pool.shutdown()


def _draw_all(fn, steps, workers=8):
    """fn(t) for t = 1 .. steps, computed by a pool of threads (each step draws from its own generator)."""
    from concurrent.futures import ThreadPoolExecutor
    with ThreadPoolExecutor(workers) as ex:
        return list(ex.map(fn, range(1, steps + 1)))


@pytest.mark.gpu
def test_gpu_c3_full_size_all_steps(dev):
    """Config C3 at full size and length: 10,000,000 x 128 table, 131,072 x 26 Zipf(1.05) ids per step, all 100
    steps, so the hot rows' m and v accumulate over the whole run.  The touched rows are compared bitwise with the
    oracle (segment sum in ATen's order, then cpu_adam on a compact copy of the touched rows) after steps 10 and 50
    and at the end.  Odd steps take the one-call form (elr_adam_dedup), even steps the plan form bench.py times
    (elr_dedup_plan made beforehand, then elr_adam_dedup_plan)."""
    from elara_amd.dedup import adam_dedup, adam_dedup_plan, unique_plan_async
    from elara_amd.gpu_ops import init_rows
    R, D, B, F, steps = 10_000_000, 128, 131_072, 26, 100
    print(f'[gpu-test] C3 full size, {steps} steps', flush=True)
    z = synth.ZipfFields([R] * F, 1.05, seed=0, offsets=[0] * F)
    ids_all = _draw_all(lambda t: z.draw(np.random.default_rng([0, t]), B), steps)
    seen = np.zeros(R, bool)
    for ids in ids_all:
        seen[ids] = True
    touched = np.flatnonzero(seen).astype(np.int64)
    del seen
    table = init_rows(torch.arange(R, device=dev), D, 0, synth.bound_for(D))
    tt = torch.from_numpy(touched).to(dev)
    compact = table[tt].cpu().numpy()

    def prep(t, ids, g):
        u, s, _ = O.segment_sum(ids, g)
        return np.searchsorted(touched, u).astype(np.int64), s

    def apply(t, us):
        O.cpu_adam(compact, us[0], us[1], O.adam_scalars(*HP, t), 16)

    pipe = _OraclePipe(prep, apply)
    try:
        for t, ids in enumerate(ids_all, start=1):
            g = torch.randn(ids.size, D, device=dev, generator=torch.Generator(dev).manual_seed(t)) * 1e-3
            if t % 2:
                adam_dedup(table, torch.from_numpy(ids).to(dev), g, *HP, t)
            else:
                u, plan, _ = unique_plan_async(torch.from_numpy(ids).to(dev), D, R)
                adam_dedup_plan(table, u, g, plan, *HP, t)
            pipe.submit(t, ids, g.cpu().numpy())
            if t in (10, 50, steps):
                pipe.drain()
                torch.cuda.synchronize()
                assert np.array_equal(bits(table[tt].cpu().numpy()), bits(compact)), f'C3 differs after step {t}'
                print(f'[gpu-test] C3 step {t}: {touched.size} touched rows equal', flush=True)
    finally:
        pipe.close()


@pytest.mark.gpu
def test_gpu_c4_large_row_stress_all_steps(dev):
    """Config C4 at full size and length: 50,000,000 x 256 table (weight + m + v = 153.6 GB in HBM), 262,144 unique
    Zipf(1.1) ids per step, all 50 steps; the touched rows compared bitwise with the oracle's cpu_adam on a
    compact copy (the table exceeds host memory budgets for a full CPU copy) after steps 10 and 25 and at the
    end."""
    from elara_amd.gpu_ops import init_rows
    from elara_amd.ops import gpu_adam
    R, D, n, steps = 50_000_000, 256, 262_144, 50
    print(f'[gpu-test] C4 large rows, {steps} steps', flush=True)
    z = synth.ZipfFields([R], 1.1, seed=4, offsets=[0])
    table = torch.empty(R, 3, D, device=dev)
    for a in range(0, R, 1 << 23):   # init in slices: rows a .. a+8M
        rows = torch.arange(a, min(R, a + (1 << 23)), device=dev)
        init_rows(rows, D, 0, synth.bound_for(D), out=table[a:a + rows.numel()])
    ids_all = _draw_all(lambda t: synth.unique_zipf(np.random.default_rng([4, t]), z, n), steps)
    touched = np.unique(np.concatenate(ids_all))
    tt = torch.from_numpy(touched).to(dev)
    compact = table[tt].cpu().numpy()

    def prep(t, ids):
        g = (np.random.default_rng([40, t]).standard_normal((n, D)) * 1e-3).astype(np.float32)
        return np.searchsorted(touched, ids).astype(np.int64), g

    def apply(t, rg):
        O.cpu_adam(compact, rg[0], rg[1], O.adam_scalars(*HP, t), 16)
        gpu_adam(table, torch.from_numpy(ids_all[t - 1]).to(dev), torch.from_numpy(rg[1]).to(dev), *HP, t)

    pipe = _OraclePipe(prep, apply)
    try:
        for t, ids in enumerate(ids_all, start=1):
            pipe.submit(t, ids)
            if t in (10, 25, steps):
                pipe.drain()
                torch.cuda.synchronize()
                assert np.array_equal(bits(table[tt].cpu().numpy()), bits(compact)), f'C4 differs after step {t}'
                print(f'[gpu-test] C4 step {t}: {touched.size} touched rows equal', flush=True)
    finally:
        pipe.close()
    # the untouched neighbours of a touched row are still their initial state
    probe = np.setdiff1d(np.clip(touched[:1000] + 1, 0, R - 1), touched)[:200]
    assert np.array_equal(bits(table[torch.from_numpy(probe).to(dev)].cpu().numpy()),
                          bits(O.init_rows(probe, D, 0, synth.bound_for(D))))
