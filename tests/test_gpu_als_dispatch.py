"""Which kernels a call runs, read from the context's kernel statistics."""
import sys

import numpy as np
import pytest

import cutc_amd as ct

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def launches(ctx, *names):
    return {n: ctx.kernel_stats(n)[0] for n in names}


def test_autotune_times_the_default_als_kernels():
    """Autotuning rank-32 ALS from the size on from which the row-fused kernels are
    the default times them as well as the spans, and the shape it returns runs."""
    say("[autotune default als]")
    ctx = ct.Context(0)
    t, _ = ct.synth((3000, 400, 300), 4_010_000, zipf=(1.0, 0.5, 0.0), test_fraction=0.0, seed=9)
    m = ct.Model(ctx, t, None, None, rank=32)
    rng = np.random.default_rng(61)
    m.set_factors([rng.uniform(-1, 1, (d, 32)).astype(np.float32) for d in t.dims])
    ctx.set_profiling(True)
    ctx.reset_stats()
    r = m.autotune(ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.05))
    n = launches(ctx, "als_gram", "als_rows_items", "als_rows_chunks")
    say(f"  {r} {n}")
    assert n["als_gram"] > 0 and n["als_rows_items"] + n["als_rows_chunks"] > 0
    ctx.reset_stats()
    m.als_mode_update(0, ct.Options(algorithm=ct.ALS, rank=32, lambda_=0.05, tile_len=r["tile_len"], block=r["block"]))
    n = launches(ctx, "als_gram", "als_rows_items", "als_rows_chunks")
    rows = n["als_rows_items"] + n["als_rows_chunks"] > 0
    assert rows == (r["tile_len"] == 0) and rows != (n["als_gram"] > 0)


def test_als_and_ccd_keep_their_piece_tables():
    """ALS and CCD++ run in turn on one model, whose default spans differ, build
    their tables once each; a third span length replaces one of the two, and every
    update gives what a model of its own gives."""
    say("[piece tables]")
    ctx = ct.Context(0)
    dims, R = (4000, 300, 60), 16
    t, _ = ct.synth(dims, 200_000, zipf=(1.0, 0.5, 0.0), test_fraction=0.0, seed=4)
    rng = np.random.default_rng(62)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in t.dims]
    als, ccd = (ct.Options(algorithm=a, rank=R, lambda_=0.05) for a in (ct.ALS, ct.CCD))
    wide = ct.Options(algorithm=ct.ALS, rank=R, lambda_=0.05, tile_len=512)

    def step(m, opt):
        m.set_factors(F)
        if opt is ccd:
            m.ccd_epoch(opt)
        else:
            for k in range(3):
                m.als_mode_update(k, opt)
        return m.factors()

    alone = {}
    for opt in (als, ccd, wide):
        alone[id(opt)] = step(ct.Model(ctx, t, None, None, rank=R), opt)
    m = ct.Model(ctx, t, None, None, rank=R)
    ctx.set_profiling(True)
    built = []
    for opt in (als, ccd, als, ccd, wide, ccd, wide, als, ccd, als):
        ctx.reset_stats()
        for a, b in zip(step(m, opt), alone[id(opt)]):
            np.testing.assert_array_equal(a, b)
        built.append(ctx.kernel_stats("piece_tables")[0])
    say(f"  built {built}")
    assert built == [3, 3, 0, 0, 3, 0, 0, 3, 3, 0]


def test_fp32_and_mixed_keep_their_row_items():
    """FP32 and mixed row-fused updates run in turn on one model, whose chunks of long
    rows differ, list their rows once each; a third chunk length replaces one of the
    two, and every update gives what a model of its own gives."""
    say("[row items]")
    ctx = ct.Context(0)
    R = 64
    t, _ = ct.synth((3000, 20, 600), 150_000, zipf=(1.0, 0.5, 0.0), test_fraction=0.0, seed=4)
    rng = np.random.default_rng(63)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in t.dims]
    full, mixed, short = (ct.Options(algorithm=ct.ALS, rank=R, lambda_=0.05, **k)
                          for k in ({}, {"precision": ct.PREC_MIXED}, {"tile_len": 96}))

    def step(m, opt):
        m.set_factors(F)
        for k in range(3):
            m.als_mode_update(k, opt)
        return m.factors()

    alone = {id(opt): step(ct.Model(ctx, t, None, None, rank=R), opt) for opt in (full, mixed, short)}
    m = ct.Model(ctx, t, None, None, rank=R)
    ctx.set_profiling(True)
    built = []
    for opt in (full, mixed, full, mixed, short, mixed, short, full, mixed, full):
        ctx.reset_stats()
        for a, b in zip(step(m, opt), alone[id(opt)]):
            np.testing.assert_array_equal(a, b)
        built.append(ctx.kernel_stats("row_items")[0])
    say(f"  built {built}")
    assert built == [3, 3, 0, 0, 3, 0, 0, 3, 3, 0]


@pytest.mark.parametrize("first,then", [(1e7, 4e7), (1e-13, 0.0)], ids=["large", "tiny_then_none"])
def test_batch_graph_of_another_lambda(first, then):
    """A batch's captured run is not replayed for another ridge weight, however large or
    small the two are; without one, short rows stay refused."""
    say(f"[batch graph lambda] {first} then {then}")
    ctx = ct.Context(0)
    R = 32
    t, _ = ct.synth((6000, 300, 200), 40_000, test_fraction=0.0, seed=5)
    rng = np.random.default_rng(64)
    F = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in t.dims]
    b = ct.Batch(ctx, [t], [None], [R])

    def run(lam, graph):
        for k, f in enumerate(F):
            b.set_factor(0, k, f)
        try:
            b.als(ct.Options(algorithm=ct.ALS, rank=R, lambda_=lam), iters=1, graph=graph)
        except ct.CtcError as e:
            return e.status
        return [b.factor(0, k) for k in range(3)]

    run(first, True)
    got, want = run(then, True), run(then, False)
    if then == 0.0:
        assert got == want == 7
    else:
        for a, e in zip(got, want):
            np.testing.assert_array_equal(a, e)


@pytest.mark.parametrize("nnz,kw,rows", [(3_990_000, {}, False), (4_010_000, {}, True), (4_010_000, {"refine": 1}, False),
                                         (4_010_000, {"tile_len": 1024}, False), (4_010_000, {"lambda_": 0.0}, False),
                                         (30_000, {"als_kernel": ct.ALS_ROWS}, True),
                                         (4_010_000, {"als_kernel": ct.ALS_SPANS}, False)],
                         ids=["below", "above", "refined", "tile_len", "no_lambda", "rows_asked", "spans_asked"])
def test_als_rank_32_family(nnz, kw, rows):
    """Which kernels the rank-32 ALS update runs on either side of the size rule and
    where an option decides."""
    say(f"[als rank 32 family] nnz={nnz} {kw}")
    ctx = ct.Context(0)
    t, _ = ct.synth((300, 250, 200), nnz, test_fraction=0.0, seed=9)
    m = ct.Model(ctx, t, None, None, rank=32)
    rng = np.random.default_rng(65)
    m.set_factors([rng.uniform(-1, 1, (d, 32)).astype(np.float32) for d in t.dims])
    ctx.set_profiling(True)
    ctx.reset_stats()
    m.als_mode_update(0, ct.Options(**{**dict(algorithm=ct.ALS, rank=32, lambda_=0.05), **kw}))
    n = launches(ctx, "als_gram", "als_rows_items", "als_rows_chunks")
    say(f"  {n}")
    assert (n["als_rows_items"] + n["als_rows_chunks"] > 0) == rows and (n["als_gram"] == 0) == rows
