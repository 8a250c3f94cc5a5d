"""The kernels' splits of the work at the sizes where they can go wrong (one
unit, a partly filled last unit, many units), against NumPy in 64 bits."""
import sys

import numpy as np
import pytest

import cutc_amd as ct

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    return ct.Context(0)


def coo(dims, nnz, seed):
    rng = np.random.default_rng(seed)
    flat = rng.choice(int(np.prod(dims)), size=nnz, replace=False)
    ind = [a.astype(np.uint32) for a in np.unravel_index(flat, dims)]
    vals = rng.uniform(1.0, 5.0, nnz)
    return ct.Coo.from_arrays(ind, vals, dims), ind, vals


def predict(ind, F):
    h = np.ones((len(ind[0]), F[0].shape[1]))
    for i, f in zip(ind, F):
        h *= f.astype(np.float64)[i]
    return h.sum(1)


@pytest.mark.parametrize("dims", [(60, 50, 40), (20, 15, 12, 10)], ids=["3way", "4way"])
def test_batch_rmse_of_segments(ctx, dims):
    """Per-problem RMSE with problems of one nonzero, about a workgroup's
    walkers and many times a segment's blocks, at every rank.  An FP32 prediction
    of R products of at most 1 is off by at most R 2^-24 = 4e-6."""
    sizes, ranks = [1, 7, 31, 129, 4097, 20011], (8, 16, 32, 64)
    probs, tests, rk, want = [], [], [], []
    rng = np.random.default_rng(5)
    for k, (n, R) in enumerate((n, R) for R in ranks for n in sizes):
        say(f"[batch rmse] n={n} R={R} dims={dims}")
        t, ind, vals = coo(dims, n, 100 + k)
        e, eind, evals = coo(dims, max(1, n // 9), 300 + k)
        F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
        probs.append(t), tests.append(e), rk.append(R)
        want.append((F, np.sqrt(np.mean((vals - predict(ind, F)) ** 2)),
                     np.sqrt(np.mean((evals - predict(eind, F)) ** 2))))
    b = ct.Batch(ctx, probs, tests, rk)
    for p, (F, _, _) in enumerate(want):
        for m, f in enumerate(F):
            b.set_factor(p, m, f)
    tr, te = b.rmse()
    np.testing.assert_allclose(tr, [w[1] for w in want], rtol=1e-6, atol=4e-6)
    np.testing.assert_allclose(te, [w[2] for w in want], rtol=1e-6, atol=4e-6)


def ridge(ind, vals, F, mode, lam):
    h = np.ones((len(vals), F[0].shape[1]))
    for m, f in enumerate(F):
        if m != mode:
            h *= f.astype(np.float64)[ind[m]]
    out = np.zeros_like(F[mode], dtype=np.float64)
    for r in np.unique(ind[mode]):
        s = ind[mode] == r
        out[r] = np.linalg.solve(h[s].T @ h[s] + lam * np.eye(h.shape[1]), h[s].T @ vals[s])
    return out


@pytest.mark.parametrize("R,refine", [(8, 0), (16, 0), (32, 0), (16, 1), (64, 0)])
@pytest.mark.parametrize("dims,nnz", [((1, 40, 30), 1000), ((9, 60, 50), 20000), ((300, 7, 30), 20000),
                                      ((40, 3, 20, 15), 9000)], ids=["one_row", "long", "mixed", "4way"])
def test_als_default_spans(ctx, dims, nnz, R, refine):
    """ALS with the default span over rows of 1 to 300 pieces (eight and fewer
    are summed by the solve, more in groups), rows without nonzeros in the
    middle, against the ridge solutions in 64 bits, at the bar of the parity
    tests (1e-5)."""
    say(f"[als default spans] dims={dims} nnz={nnz} R={R} refine={refine}")
    t, ind, vals = coo(dims, nnz - nnz // 10, 3)
    if dims[0] > 2:  # a row without nonzeros
        keep = ind[0] != 1
        ind, vals = [i[keep] for i in ind], vals[keep]
        t = ct.Coo.from_arrays(ind, vals, dims)
    rng = np.random.default_rng(8)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
    m = ct.Model(ctx, t, None, None, rank=R)
    opt = ct.Options(algorithm=ct.ALS, rank=R, lambda_=0.5, refine=refine, als_kernel=ct.ALS_SPANS)
    for mode in range(len(dims)):
        m.set_factors(F)
        m.als_mode_update(mode, opt)
        want = ridge(ind, vals, F, mode, 0.5)
        e = np.linalg.norm(m.factor(mode) - want) / np.linalg.norm(want)
        assert e < 1e-5, (mode, e)


@pytest.mark.parametrize("R", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("dims,nnz", [((1, 40, 30), 1100), ((3, 300, 50), 31), ((3, 300, 50), 33),
                                      ((700, 9, 40), 32 * 131 + 1), ((5, 600, 80), 32 * 1200), ((12, 3, 40, 15), 9000)],
                         ids=["one_row", "short", "one_span", "rows_in_spans", "rows_over_groups", "4way"])
def test_walk_row_sums(ctx, dims, nnz, R):
    """MTTKRP, and the gradient with its two regularisers, of rows inside one
    walker's span, across walkers and across workgroups, rows that end at a
    span's end, and rows without nonzeros, against 64 bits at the parity
    tests' bars (MTTKRP and gradients 1e-5, loss 1e-6)."""
    import torch
    say(f"[walk sums] dims={dims} nnz={nnz} R={R}")
    t, ind, vals = coo(dims, nnz, 11)
    rng = np.random.default_rng(12)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
    F64 = [f.astype(np.float64) for f in F]
    m = ct.Model(ctx, t, None, None, rank=R)
    m.set_factors(F)
    e = vals - predict(ind, F)
    hs = []
    for mode in range(len(dims)):
        h = np.ones((nnz, R))
        for k, f in enumerate(F64):
            if k != mode:
                h *= f[ind[k]]
        hs.append(h)
        want = np.zeros((dims[mode], R))
        np.add.at(want, ind[mode], vals[:, None] * h)
        assert np.linalg.norm(m.mttkrp(mode) - want) < 1e-5 * np.linalg.norm(want), mode
    dev = [torch.from_numpy(f).cuda() for f in F]
    for per_occ in (False, True):
        G = [torch.full_like(f, 7.0) for f in dev]
        torch.cuda.synchronize()
        loss = m.grad_device([f.data_ptr() for f in dev], [g.data_ptr() for g in G], 0.3, per_occ)
        wl = 0.5 * np.sum(e * e)
        for mode in range(len(dims)):
            c = np.bincount(ind[mode], minlength=dims[mode])[:, None] if per_occ else 1.0
            want = 0.3 * c * F64[mode]
            np.add.at(want, ind[mode], -e[:, None] * hs[mode])
            wl += 0.15 * np.sum(c * F64[mode] ** 2)
            got = G[mode].cpu().numpy()
            assert np.linalg.norm(got - want) < 1e-5 * np.linalg.norm(want), (mode, per_occ)
        assert loss == pytest.approx(wl, rel=1e-6)


@pytest.mark.parametrize("R,mixed", [(8, False), (16, False), (16, True), (32, False), (32, True), (64, True), (128, False)])
@pytest.mark.parametrize("dims,nnz,span,sub", [((1, 40, 30), 1, 2048, 32), ((40, 12, 9), 31, 2048, 32),
                                               ((40, 12, 9), 700, 100, 33), ((9, 30, 6, 7), 3001, 256, 70),
                                               ((3, 500, 400), 140_003, 8, 3), ((4000, 300, 80), 150_001, 64, 32)],
                         ids=["one", "short", "odd_substep", "4way_rounds", "many_walkers", "short_rows"])
def test_sgd_walk_rounds(ctx, dims, nnz, span, sub, R, mixed):
    """The SGD walk with sub-steps of less than a round of nonzeros, of one
    round and of several, with the walkers of part of a wave and of more waves than
    two per SIMD (both lane shapes), runs that go on across rounds, and mode-0
    rows in place and over walkers, against the oracle's schedule in 64 bits at the
    parity tests' bars (1e-5; mixed 2e-4: a delta near a BF16 tie may round
    the other way)."""
    import oracle as O
    say(f"[sgd walk] dims={dims} nnz={nnz} span={span} sub={sub} R={R} mixed={mixed}")
    t, ind, vals = coo(dims, nnz, 21)
    rng = np.random.default_rng(22)
    F = [(0.5 * rng.uniform(-1, 1, (d, R))).astype(np.float32) for d in dims]
    F64 = [f.astype(np.float64) for f in F]
    oc = O.Coo(ind, vals, dims)
    O.sgd_sync_epoch(oc, F64, 1e-3, 0.05, span, sub, 400, order=O.mode_order(oc, 0)[0], nthreads=4, mixed=mixed)
    m = ct.Model(ctx, t, None, None, rank=R)
    m.set_factors(F)
    m.sgd_epoch(ct.Options(algorithm=ct.SGD, rank=R, lambda_=0.05, sgd_scale=1.0, tile_len=span, sgd_substep=sub,
                           sgd_hot_rows=400, precision=ct.PREC_MIXED if mixed else ct.PREC_FP32), lr=1e-3)
    for k, f in enumerate(F64):
        assert np.linalg.norm(m.factor(k) - f) < (2e-4 if mixed else 1e-5) * np.linalg.norm(f), k


@pytest.mark.parametrize("R", [32, 64, 128])
@pytest.mark.parametrize("mixed", [False, True], ids=["fp32", "mixed"])
@pytest.mark.parametrize("rest", [(47, 39), (23, 19, 17)], ids=["3way", "4way"])
def test_als_row_lengths(ctx, rest, mixed, R):
    """The row-fused ALS update of rows of 1 to 67 nonzeros, one of each length and
    one of several Gram steps, and rows without nonzeros, each row against the
    ridge solution in 64 bits (mixed: the oracle's BF16-operand update) at the
    parity tests' bars, row by row (1e-5, 1e-4)."""
    import oracle as O
    say(f"[als row lengths] rest={rest} R={R} mixed={mixed}")
    rng = np.random.default_rng(31)
    lens = [*range(1, 68), 0, 301, 0]
    rng.shuffle(lens)
    rows = np.repeat(np.arange(len(lens)), lens)
    flat = np.concatenate([rng.choice(int(np.prod(rest)), size=n, replace=False) for n in lens])
    ind = [rows.astype(np.uint32), *(a.astype(np.uint32) for a in np.unravel_index(flat, rest))]
    vals = rng.uniform(1.0, 5.0, len(rows))
    dims = (len(lens), *rest)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
    m = ct.Model(ctx, ct.Coo.from_arrays(ind, vals, dims), None, None, rank=R)
    m.set_factors(F)
    m.als_mode_update(0, ct.Options(algorithm=ct.ALS, rank=R, lambda_=0.5, als_kernel=ct.ALS_ROWS,
                                    precision=ct.PREC_MIXED if mixed else ct.PREC_FP32))
    if mixed:
        want = [f.copy() for f in F]
        assert O.als_mode_bf16(O.Coo(ind, vals, dims), 0, want, 0.5) == 0
        want = want[0].astype(np.float64)
    else:
        want = ridge(ind, vals, F, 0, 0.5)
    got = m.factor(0).astype(np.float64)
    for r, n in enumerate(lens):
        assert np.linalg.norm(got[r] - want[r]) <= (1e-4 if mixed else 1e-5) * np.linalg.norm(want[r]), (r, n)


@pytest.mark.parametrize("rest", [(47, 39), (23, 19, 17)], ids=["3way", "4way"])
@pytest.mark.parametrize("longer", [(), (17, 40, 700)], ids=["all_short", "short_and_long"])
def test_als_short_rows_of_rank_32(ctx, rest, longer):
    """The default rank-32 ALS update of 5000 rows, of 1 to 16 nonzeros (their dual
    form; runs of them over tiles and spans) and longer ones between them, eagerly
    and in a batch's captured graph, against the span kernels alone: both solve
    in 64 bits, so row by row they agree to a few FP32 roundings (1e-6), and to the
    ridge solution at the parity tests' bar (1e-5).  Without lambda such rows stay refused."""
    say(f"[als short rows] rest={rest} longer={longer}")
    rng = np.random.default_rng(41)
    lens = rng.integers(1, 17, 5000)
    for k, n in enumerate(longer):
        lens[rng.choice(5000, 40, replace=False)] = n
    lens[[7, 4999]] = 0
    flat = np.concatenate([rng.choice(int(np.prod(rest)), size=n, replace=False) for n in lens])
    ind = [np.repeat(np.arange(5000), lens).astype(np.uint32),
           *(a.astype(np.uint32) for a in np.unravel_index(flat, rest))]
    vals = rng.uniform(1.0, 5.0, len(flat))
    dims = (5000, *rest)
    F = [rng.uniform(-1, 1, (d, 32)).astype(np.float32) for d in dims]
    t = ct.Coo.from_arrays(ind, vals, dims)
    m = ct.Model(ctx, t, None, None, rank=32)
    got = {}
    for kernel in (ct.ALS_AUTO, ct.ALS_SPANS):
        m.set_factors(F)
        m.als_mode_update(0, ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.5, als_kernel=kernel))
        got[kernel] = m.factor(0).astype(np.float64)
    want = ridge(ind, vals, F, 0, 0.5)
    size = np.linalg.norm(want, axis=1)
    assert np.all(np.linalg.norm(got[ct.ALS_AUTO] - got[ct.ALS_SPANS], axis=1) <= 1e-6 * size)
    assert np.all(np.linalg.norm(got[ct.ALS_AUTO] - want, axis=1) <= 1e-5 * size)
    b = ct.Batch(ctx, [t], [None], [32])
    for k, f in enumerate(F):
        b.set_factor(0, k, f)
    b.als(ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.5), iters=1, graph=True)
    m.set_factors(F)
    for k in range(len(dims)):
        m.als_mode_update(k, ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.5))
    for k in range(len(dims)):
        np.testing.assert_array_equal(b.factor(0, k), m.factor(k))
    with pytest.raises(ct.CtcError) as e:
        m.als_mode_update(0, ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.0))
    assert e.value.status == 7


def test_als_rank_32_kernel_by_size(ctx):
    """The default rank-32 ALS update on both sides of the size from which it runs
    the row-fused kernels, against the span kernels: both sum and solve in 64 bits, so
    the factors agree to a few FP32 roundings (1e-6)."""
    for nnz in (3_990_000, 4_010_000):
        say(f"[als rank 32 by size] nnz={nnz}")
        t, _ = ct.synth((3000, 400, 300), nnz, zipf=(1.0, 0.5, 0.0), test_fraction=0.0, seed=9)
        rng = np.random.default_rng(51)
        F = [rng.uniform(-1, 1, (d, 32)).astype(np.float32) for d in t.dims]
        m = ct.Model(ctx, t, None, None, rank=32)
        for mode in range(3):
            got = []
            for kernel in (ct.ALS_AUTO, ct.ALS_SPANS):
                m.set_factors(F)
                m.als_mode_update(mode, ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.05, als_kernel=kernel))
                got.append(m.factor(mode).astype(np.float64))
            assert np.linalg.norm(got[0] - got[1]) <= 1e-6 * np.linalg.norm(got[1]), (nnz, mode)


@pytest.mark.parametrize("R,count,longest", [(8, 3, 1024), (8, 3, 1025), (64, 140, 20_000), (8, 5000, 3000)],
                         ids=["one_block", "two_blocks", "shared_by_58", "one_block_each"])
def test_batch_rmse_of_many_problems(ctx, R, count, longest):
    """Per-problem RMSE where the blocks that share a problem are set by the longest
    one and by the number of problems, with and without test entries.  The bound is
    that of test_batch_rmse_of_segments."""
    say(f"[batch rmse many] R={R} count={count} longest={longest}")
    dims, rng = (40, 35, 30), np.random.default_rng(71)
    sizes = rng.integers(1, 20, count)
    sizes[count // 2] = longest
    probs, tests, wt, we = [], [], [], []
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
    for k, n in enumerate(sizes):
        t, ind, vals = coo(dims, n, 1000 + k)
        e, eind, evals = coo(dims, 3, 90_000 + k)
        probs.append(t), tests.append(e if k % 3 else None)
        wt.append(np.sqrt(np.mean((vals - predict(ind, F)) ** 2)))
        we.append(np.sqrt(np.mean((evals - predict(eind, F)) ** 2)) if k % 3 else 0.0)
    b = ct.Batch(ctx, probs, tests, [R] * count)
    for p in range(count):
        for m, f in enumerate(F):
            b.set_factor(p, m, f)
    for _ in range(2):
        tr, te = b.rmse()
        np.testing.assert_allclose(tr, wt, rtol=1e-6, atol=4e-6)
        np.testing.assert_allclose(te, we, rtol=1e-6, atol=4e-6)


@pytest.mark.parametrize("R,modes,above", [(8, 3, False), (8, 3, True), (16, 3, True), (32, 3, False), (32, 3, True), (32, 4, True)])
def test_sgd_walk_lane_shapes(ctx, R, modes, above):
    """The FP32 SGD walk just below and just above the number of walkers from which a
    lane holds four elements of a row, with spans of 4 nonzeros, against the oracle's
    schedule in 64 bits at the parity tests' bar (1e-5)."""
    import oracle as O
    walkers = 2048 * 256 // R + (1 if above else -1)
    nnz = 4 * walkers - 3
    dims = (9001, 120, 70) if modes == 3 else (9001, 60, 40, 9)
    say(f"[sgd lane shapes] R={R} dims={dims} walkers={walkers}")
    t, ind, vals = coo(dims, nnz, 81)
    rng = np.random.default_rng(82)
    F = [(0.5 * rng.uniform(-1, 1, (d, R))).astype(np.float32) for d in dims]
    F64 = [f.astype(np.float64) for f in F]
    oc = O.Coo(ind, vals, dims)
    O.sgd_sync_epoch(oc, F64, 1e-3, 0.05, 4, 2, 60_000, order=O.mode_order(oc, 0)[0], nthreads=4)
    m = ct.Model(ctx, t, None, None, rank=R)
    m.set_factors(F)
    m.sgd_epoch(ct.Options(algorithm=ct.SGD, rank=R, lambda_=0.05, sgd_scale=1.0, tile_len=4, sgd_substep=2,
                           sgd_hot_rows=60_000), lr=1e-3)
    for k, f in enumerate(F64):
        assert np.linalg.norm(m.factor(k) - f) < 1e-5 * np.linalg.norm(f), k


@pytest.mark.parametrize("R,dims,nnz", [(128, (700, 300, 60), 4096 * 2 * 64 + 5000), (128, (2, 900, 600), 4096 * 2 * 96 + 77),
                                        (64, (900, 120, 40, 9), 4096 * 4 * 64 + 1), (32, (1500, 300, 60), 4096 * 8 * 96 + 33)],
                         ids=["r128_span64", "r128_span96_long", "r64_4way_span64", "r32_span96"])
def test_walk_spans_of_several_chunks(ctx, R, dims, nnz):
    """MTTKRP, the gradient with both regularisers and the training loss where the
    spans are longer than the 32 nonzeros of a small tensor (64 and 96: several chunks
    even at R = 128, where a chunk is 32), with rows inside a span, over its chunks,
    over walkers and over workgroups, against 64 bits at the parity tests' bars
    (1e-5, loss 1e-6)."""
    import torch
    say(f"[walk chunks] R={R} dims={dims} nnz={nnz}")
    t, ind, vals = coo(dims, nnz, 91)
    rng = np.random.default_rng(92)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
    m = ct.Model(ctx, t, None, None, rank=R)
    m.set_factors(F)
    di, dv = [torch.from_numpy(i.astype(np.int64)).cuda() for i in ind], torch.from_numpy(vals.astype(np.float32)).cuda().double()
    D = [torch.from_numpy(f).cuda() for f in F]
    D64 = [f.double() for f in D]

    def others(mode):
        h = torch.ones(nnz, R, dtype=torch.float64, device="cuda")
        for k, f in enumerate(D64):
            if k != mode:
                h *= f[di[k]]
        return h

    e = dv - (others(0) * D64[0][di[0]]).sum(1)
    sq = float((e * e).sum())
    assert m.evaluate(0.0)["loss"] == pytest.approx(sq, rel=1e-6)
    grads = {}
    for per_occ in (False, True):
        G = [torch.full_like(f, 7.0) for f in D]
        torch.cuda.synchronize()
        loss = m.grad_device([f.data_ptr() for f in D], [g.data_ptr() for g in G], 0.3, per_occ)
        cnt = [torch.bincount(i, minlength=f.shape[0]).double()[:, None] if per_occ else 1.0 for i, f in zip(di, D64)]
        want = 0.5 * sq + sum(0.15 * float((c * f * f).sum()) for c, f in zip(cnt, D64))
        assert loss == pytest.approx(want, rel=1e-6)
        grads[per_occ] = [(g.double(), 0.3 * c * f) for g, c, f in zip(G, cnt, D64)]
    for mode in range(len(dims)):
        h = others(mode)
        order = torch.argsort(di[mode], stable=True)
        lens = torch.bincount(di[mode], minlength=dims[mode])

        def row_sums(w):
            return torch.segment_reduce((h * w[:, None])[order], "sum", lengths=lens, unsafe=True)

        want = row_sums(dv)
        got = torch.from_numpy(m.mttkrp(mode)).cuda().double()
        assert float((got - want).norm()) < 1e-5 * float(want.norm()), mode
        adjoint = row_sums(e)
        for per_occ, g in grads.items():
            got, want = g[mode][0], g[mode][1] - adjoint
            assert float((got - want).norm()) < 1e-5 * float(want.norm()), (mode, per_occ)
