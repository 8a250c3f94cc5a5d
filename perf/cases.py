"""What users of cutc_amd run, as measurable cases.

Every case is one call sequence of a completion program on one GPU: an ALS
sweep or mode update, an SGD or CCD++ epoch, a whole solve with its per-epoch
evaluation, a batch of small problems, the differentiable loss with its
backward pass, MTTKRP.  Tensors are synthetic ratings of the benchmark's kind:
distinct coordinates, Zipf or uniform per mode, values from a low-rank CP model
plus noise (rounded to 1..5 where the program rates).  `exact` restates each
call in 64 bits with torch alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

DEV = "cuda"
LAM = 0.05      # ridge weight of the benchmark configurations
SGD_LR = 1e-3   # learning rate of the benchmark's SGD epochs

# shape of the default SGD schedule (walker span, sub-step, hot-row threshold)
SPAN, SUB, HOT = 2048, 32, 65536


def _case(name, kind, dims, nnz, rank, zipf=(0.0, 0.0, 0.0, 0.0), **kw):
    c = {"kind": kind, "modes": len(dims), "nnz": int(nnz), "rank": int(rank)}
    for m, d in enumerate(dims):
        c[f"d{m}"] = int(d)
        c[f"z{m}"] = float(zipf[m])
    c.update(kw)
    return dict(c, name=name) if name else c


# the benchmark tensor's shape: users x items x days
RATINGS, RATINGS_ZIPF = (480189, 17770, 2182), (1.0, 1.0, 0.0)
# the 4-way tensor behind the autograd loss
CONTEXT4, CONTEXT4_ZIPF = (1_000_000, 500_000, 1000, 24), (1.0, 1.0, 0.0, 0.0)


def listed():
    return [
        # a first try on a few thousand ratings: launches and synchronisation are what it pays for
        _case("als sweep 20k r16", "als", (300, 200, 60), 20_000, 16, (1.0, 0.7, 0.0)),
        # the small benchmark configuration as a program runs it: ten ALS epochs, RMSE after each
        _case("als solve 1M r16", "solve", (2000, 1500, 300), 1_000_000, 16, epochs=10),
        # one FP32 ALS sweep over ratings with skewed users and items
        _case("als sweep 20M r32", "als", RATINGS, 20_000_000, 32, RATINGS_ZIPF),
        # mixed precision at rank 128 on a long tensor of mostly short rows: one mode's update
        _case("als mixed update 12M r128", "als_mode", (500_011, 500_011, 1000), 12_000_000, 128, (1.1, 1.1, 0.0),
              mode=0),
        # many small problems of ranks 8 to 64 solved together, ten iterations
        _case("batch 24 problems", "batch", (20000, 20000, 20000), 300_000, 64, problems=24, iters=10),
        # one GPU's share of the ratings tensor over two and over eight: an SGD epoch, default schedule
        _case("sgd epoch 50M r32", "sgd", RATINGS, 50_000_000, 32, RATINGS_ZIPF, mixed=False),
        _case("sgd epoch 12.5M r32", "sgd", RATINGS, 12_500_000, 32, RATINGS_ZIPF, mixed=False),
        # an SGD epoch in mixed precision, rank 64, odd sizes
        _case("sgd mixed epoch 5M r64", "sgd", (120_011, 9001, 777), 5_000_003, 64, (1.0, 0.5, 0.0), mixed=True),
        # the smallest SGD epoch: the schedule's launches are all it is
        _case("sgd epoch 20k r16", "sgd", (300, 200, 60), 20_000, 16, (1.0, 0.7, 0.0), mixed=False),
        # a CCD++ epoch on skewed ratings
        _case("ccd epoch 20M r32", "ccd", RATINGS, 20_000_000, 32, RATINGS_ZIPF),
        # a training step's loss and gradients of a 4-way model through torch.autograd
        _case("grad 4-way 20M r32", "grad", CONTEXT4, 20_000_000, 32, CONTEXT4_ZIPF, per_occurrence=False),
        # MTTKRP of every mode into host arrays
        _case("mttkrp 8M r32", "mttkrp", (50021, 17770, 2182), 8_000_000, 32, RATINGS_ZIPF),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["als", "als", "als_mode", "sgd", "sgd", "ccd", "grad", "mttkrp", "solve", "batch"])
    if kind == "batch":
        return _case(None, kind, (20000, 20000, 20000), _log(rng, 20_000, 250_000), 64, problems=rng.randint(4, 24),
                     iters=rng.randint(3, 10))
    four = rng.random() < (0.6 if kind == "grad" else 0.2)
    top = {"als": 8_000_000, "als_mode": 6_000_000, "sgd": 12_500_000, "ccd": 8_000_000, "grad": 8_000_000,
           "mttkrp": 8_000_000, "solve": 1_000_000}[kind]
    nnz = _log(rng, 120_000 if kind == "grad" else 20_000, top)
    dims = [_log(rng, 150, 400_000), _log(rng, 100, 40_000), _log(rng, 50, 3000)]
    zipf = [rng.choice([0.0, 0.6, 1.0]), rng.choice([0.0, 0.5, 1.0]), 0.0, 0.0]
    if four:
        dims.append(rng.randint(7, 60))
    nnz = max(1000, min(nnz, math.prod(dims) // 8))
    if kind == "als_mode":
        rank = rng.choice([32, 64, 128, 128])
        return _case(None, kind, dims, nnz, rank, zipf, mode=rng.randrange(2))
    if kind == "als":
        rank = rng.choice([8, 16, 32, 32, 64])
        if rank == 64:
            nnz = min(nnz, 3_000_000)
        return _case(None, kind, dims, nnz, rank, zipf)
    if kind == "sgd":
        return _case(None, kind, dims, nnz, rng.choice([8, 16, 32, 32, 64]), zipf, mixed=rng.random() < 0.3)
    if kind == "solve":
        return _case(None, kind, dims[:3], nnz, rng.choice([8, 16, 32]), zipf, epochs=rng.randint(3, 10))
    if kind == "grad":
        return _case(None, kind, dims, nnz, rng.choice([16, 32, 32, 64]), zipf, per_occurrence=rng.random() < 0.3)
    return _case(None, kind, dims, nnz, rng.choice([8, 16, 32, 32]), zipf)


# ------------------------------------------------------------------ inputs --
def _dims(case):
    return [case[f"d{m}"] for m in range(case["modes"])]


def _coords(dims, zipf, nnz, gen):
    """nnz distinct coordinates (or somewhat fewer where a skewed tensor's head is full), mode-0 order."""
    cdf = []
    for d, z in zip(dims, zipf):
        w = np.cumsum(np.arange(1, d + 1, dtype=np.float64) ** -z) if z else None
        cdf.append(None if w is None else torch.from_numpy(w / w[-1]).to(DEV))
    lin = torch.empty(0, dtype=torch.int64, device=DEV)
    for _ in range(8):
        need = nnz - lin.numel()
        if need <= 0:
            break
        n = int(need * 1.3) + 1024
        key = torch.zeros(n, dtype=torch.int64, device=DEV)
        for d, c in zip(dims, cdf):
            u = torch.rand(n, dtype=torch.float64, device=DEV, generator=gen)
            i = (u * d).long() if c is None else torch.searchsorted(c, u)
            key = key * d + i.clamp_(max=d - 1)
        lin = torch.unique(torch.cat([lin, key]))
    if lin.numel() > nnz:
        lin = lin[torch.randperm(lin.numel(), device=DEV, generator=gen)[:nnz]].sort().values
    ind = []
    for d in reversed(dims):
        ind.insert(0, lin % d)
        lin = lin // d
    return ind


def _values(ind, dims, gen, rated):
    truth = [torch.rand(d, 8, dtype=torch.float64, device=DEV, generator=gen) for d in dims]
    n = ind[0].numel()
    v = torch.ones(n, 8, dtype=torch.float64, device=DEV)
    for i, t in zip(ind, truth):
        v *= t[i]
    v = v.sum(1)
    noise = torch.randn(n, dtype=torch.float64, device=DEV, generator=gen)
    if rated:
        v = 3.0 + (v - v.mean()) / v.std() + 0.3 * noise
        return v.round().clamp_(1, 5)
    return (v + 0.1 * noise).float().double()  # what a float32 tensor file holds


def _tensor(case, seed):
    """(indices, values, generator) of the case's tensor for this seed."""
    gen = torch.Generator(device=DEV).manual_seed(0x5EED + 7919 * int(seed))
    dims = _dims(case)
    ind = _coords(dims, [case[f"z{m}"] for m in range(len(dims))], case["nnz"], gen)
    return ind, _values(ind, dims, gen, rated=case["kind"] not in ("grad",)), gen


def _init(dims, rank, gen, positive=False):
    """U(-1, 1) factors; U(0, 0.6) for gradient descent, which a zero-mean start leaves at the saddle at 0."""
    return [torch.rand(d, rank, device=DEV, generator=gen) * 0.6 if positive
            else torch.rand(d, rank, device=DEV, generator=gen) * 2 - 1 for d in dims]


def _split(ind, vals, gen, part):
    test = torch.rand(vals.numel(), device=DEV, generator=gen) < part
    return ([i[~test] for i in ind], vals[~test]), ([i[test] for i in ind], vals[test])


def _problems(case, seed):
    """(dims, rank, (train indices, values), (test ...), factors) of each problem of a batch: log-uniform
    dims, log-normal sizes around the case's, ranks 8, 16, 32 and 64 in turn."""
    gen = torch.Generator(device=DEV).manual_seed(0xBA7C4 + 7919 * int(seed))
    shape = np.random.default_rng(0xBA7C4)  # the problems' sizes are the case's, whatever the seed
    out = []
    for p in range(case["problems"]):
        dims = [int(round(math.exp(shape.uniform(math.log(200), math.log(case[f"d{m}"]))))) for m in range(3)]
        nnz = int(np.clip(math.exp(shape.normal(math.log(case["nnz"]), 0.7)), 5_000, 4 * case["nnz"]))
        nnz = int(min(nnz, 0.25 * math.prod(dims)))
        rank = (8, 16, 32, 64)[p % 4]
        ind = _coords(dims, (0.0, 0.0, 0.0), nnz, gen)
        train, test = _split(ind, _values(ind, dims, gen, rated=False), gen, 0.1)
        out.append((dims, rank, train, test, _init(dims, rank, gen)))
    return out


def _coo(ct, ind, vals, dims):
    return ct.Coo.from_arrays([i.int().cpu().numpy() for i in ind], vals.cpu().numpy(), dims)


class _Device:
    """A model's factor as a torch tensor over the model's own memory."""

    def __init__(self, model, mode):
        self.model = model
        self.__cuda_array_interface__ = {"shape": (model.dims[mode], model.rank), "typestr": "<f4", "version": 3,
                                         "data": (model.factor_device_ptr(mode), False)}


def _views(model):
    return [torch.as_tensor(_Device(model, m), device=DEV) for m in range(model.nmodes)]


_context = None


def _ctx(ct):
    """The program's one device context."""
    global _context
    if _context is None:
        _context = ct.Context(0)
    return _context


def _options(ct, case):
    kind, rank = case["kind"], case["rank"]
    if kind == "sgd":
        return ct.Options(algorithm=ct.SGD, rank=rank, lambda_=LAM, learning_rate=SGD_LR, sgd_scale=1.0,
                          precision=ct.PREC_MIXED if case["mixed"] else ct.PREC_FP32)
    if kind == "ccd":
        return ct.Options(algorithm=ct.CCD, rank=rank, lambda_=LAM)
    if kind == "als_mode":
        return ct.Options(algorithm=ct.ALS, rank=rank, lambda_=LAM, precision=ct.PREC_MIXED, refine=1)
    if kind == "solve":  # tolerance 0 and no early stop: every epoch runs
        return ct.Options(algorithm=ct.ALS, rank=rank, lambda_=LAM, max_epochs=case["epochs"], tolerance=0.0,
                          max_bad_epochs=1000)
    return ct.Options(algorithm=ct.ALS, rank=rank, lambda_=LAM)


# ----------------------------------------------------------------- the call --
def prepare(case, seed):
    import cutc_amd as ct

    kind, opt = case["kind"], _options(ct, case)
    if kind == "batch":
        ps = _problems(case, seed)
        trains = [_coo(ct, *train, dims) for dims, _, train, _, _ in ps]
        tests = [_coo(ct, *test, dims) for dims, _, _, test, _ in ps]
        batch = ct.Batch(_ctx(ct), trains, tests, [p[1] for p in ps])
        return {"kind": kind, "batch": batch, "opt": opt, "iters": case["iters"],
                "F": [[f.cpu().numpy() for f in p[4]] for p in ps]}
    ind, vals, gen = _tensor(case, seed)
    dims = _dims(case)
    test = None
    if kind == "solve":
        (ind, vals), (ti, tv) = _split(ind, vals, gen, 0.1)
        test = _coo(ct, ti, tv, dims)
    F = _init(dims, case["rank"], gen, positive=kind == "grad")
    model = ct.Model(_ctx(ct), _coo(ct, ind, vals, dims), None, test, rank=case["rank"])
    state = {"kind": kind, "model": model, "opt": opt, "modes": case["modes"]}
    if kind == "grad":
        model.prepare(opt)  # every mode's CISS
        state.update(F=[f.requires_grad_() for f in F], per_occurrence=case["per_occurrence"])
        return state
    host = [f.cpu().numpy() for f in F]
    model.set_factors(host)
    model.prepare(opt)
    if kind == "sgd":
        model.sgd_epoch(opt, lr=0.0)  # builds the schedule's tables; at rate 0 the factors stay
    state.update(host=host, views=_views(model), mode=case.get("mode"))
    return state


def run(state):
    kind, opt = state["kind"], state["opt"]
    if kind == "batch":
        batch, n = state["batch"], state["batch"].nproblems
        for p in range(n):
            for m in range(3):
                batch.set_factor(p, m, state["F"][p][m])
        batch.als(opt, iters=state["iters"], graph=True)
        rmse = batch.rmse()
        return {"rmse_tr": rmse[0].astype(np.float32), "rmse_te": rmse[1].astype(np.float32),
                "factors": [np.concatenate([batch.factor(p, m).ravel() for m in range(3)]) for p in range(n)]}
    model = state["model"]
    if kind == "grad":
        from cutc_amd.autograd import completion_loss

        for f in state["F"]:
            f.grad = None
        loss = completion_loss(model, state["F"], LAM, state["per_occurrence"])
        loss.backward()
        return {"loss": loss.detach(), "grads": [f.grad for f in state["F"]]}
    if kind == "mttkrp":
        return [model.mttkrp(m) for m in range(state["modes"])]
    if kind == "solve":
        model.set_factors(state["host"])
        r = model.solve(opt)
        return {"rmse_tr": np.array([h["rmse_tr"] for h in r.history], np.float32),
                "rmse_te": np.array([h["rmse_te"] for h in r.history], np.float32),
                "factors": [model.factor(m) for m in range(state["modes"])]}
    if kind == "als":
        for m in range(state["modes"]):
            model.als_mode_update(m, opt)
    elif kind == "als_mode":
        model.als_mode_update(state["mode"], opt)
        return state["views"][state["mode"]]
    elif kind == "sgd":
        model.sgd_epoch(opt, lr=SGD_LR)
    else:
        model.ccd_epoch(opt)
    return state["views"]


# --------------------------------------------------------- the work it takes --
def work(case):
    """Each nonzero's indices and value once per sweep over the tensor, each factor row once in and (where it
    is updated) once out; the flops of the update rule."""
    n, R, N, nnz, kind = _dims(case), case["rank"], case["modes"], case["nnz"], case["kind"]
    stream, rows = nnz * 4.0 * (N + 1), 4.0 * R * sum(n)
    als = nnz * (R * (R + 1.0) + (N + 1) * R)  # the lower Gram, the products and the right-hand side of one mode
    chol = R ** 3 / 3.0 + 2.0 * R * R
    live = [min(d, nnz) for d in n]
    if kind == "als":
        return {"bytes": N * (stream + rows), "flops": N * als + chol * sum(live)}
    if kind == "als_mode":
        return {"bytes": stream + rows, "flops": als + chol * live[case["mode"]]}
    if kind == "solve":
        e = case["epochs"]
        return {"bytes": e * (N + 1) * (stream + rows), "flops": e * (N * als + 2.0 * N * R * nnz + chol * sum(live))}
    if kind == "sgd":
        return {"bytes": stream + 2 * rows, "flops": nnz * R * (N + N * (N + 3.0))}
    if kind == "ccd":  # per column and mode the residual is read and written beside the indices
        return {"bytes": R * N * nnz * (4.0 * (N - 1) + 8.0) + 2 * rows, "flops": R * N * nnz * (3.0 * N + 4.0)}
    if kind == "grad":
        return {"bytes": N * stream + 2 * rows, "flops": N * nnz * R * (2.0 * N + 2.0)}
    if kind == "mttkrp":
        return {"bytes": N * (stream + rows), "flops": N * nnz * R * (N + 1.0)}
    k, its = case["problems"], case["iters"]
    per = [nnz * (r * (r + 1.0) + 4.0 * r) * 3 for r in (8, 16, 32, 64)]
    return {"bytes": its * k * 3 * stream, "flops": its * k * sum(per) / 4.0}


# ------------------------------------------------------------ in 64 bits --
def _solve_spd(A, b):
    """x of A x = b for a stack of positive definite A (Gauss-Jordan; A and b are overwritten)."""
    for k in range(A.shape[1]):
        inv = 1.0 / A[:, k, k]
        p, q = A[:, k, :] * inv[:, None], b[:, k] * inv
        f = A[:, :, k].clone()
        f[:, k] = 0
        A.baddbmm_(f[:, :, None], p[:, None, :], alpha=-1.0)
        b.sub_(f * q[:, None])
        A[:, k, :], b[:, k] = p, q
    return b


def _als_exact(ind, vals, F, mode, lam):
    """The ridge solution of every row of `mode`; rows without nonzeros become 0."""
    dims, R, P = [f.shape[0] for f in F], F[0].shape[1], 32
    order = torch.argsort(ind[mode], stable=True)
    row = ind[mode][order]
    rows, cnt = torch.unique_consecutive(row, return_counts=True)
    start = torch.cumsum(cnt, 0) - cnt
    pieces = (cnt + P - 1) // P  # a row's nonzeros in pieces of P, so that its Gram is a sum of small products
    first = torch.cumsum(pieces, 0) - pieces
    slot = torch.repeat_interleave(torch.arange(rows.numel(), device=DEV), cnt)
    pos = torch.arange(row.numel(), device=DEV) - start[slot]
    piece, at = first[slot] + pos // P, pos % P
    owner = torch.repeat_interleave(torch.arange(rows.numel(), device=DEV), pieces)
    out = torch.zeros(dims[mode], R, dtype=torch.float64, device=DEV)
    most = max(1, int(1.5e9 / (R * R * 8)))
    ends = torch.cumsum(pieces, 0).cpu()
    nnz_of = torch.cumsum(torch.bincount(piece, minlength=owner.numel()), 0).cpu()
    r0 = 0
    while r0 < rows.numel():
        r1 = min(rows.numel(), r0 + most)
        G = torch.zeros(r1 - r0, R, R, dtype=torch.float64, device=DEV)
        m = torch.zeros(r1 - r0, R, dtype=torch.float64, device=DEV)
        p0, p_end = (int(ends[r0 - 1]) if r0 else 0), int(ends[r1 - 1])
        step = max(1, int(1e9 / (P * R * 8 + R * R * 8)))
        while p0 < p_end:
            p1 = min(p_end, p0 + step)
            a, b = (int(nnz_of[p0 - 1]) if p0 else 0), int(nnz_of[p1 - 1])
            sel = order[a:b]
            h = torch.ones(b - a, R, dtype=torch.float64, device=DEV)
            for s in range(len(F)):
                if s != mode:
                    h *= F[s][ind[s][sel]]
            H = torch.zeros(p1 - p0, P, R, dtype=torch.float64, device=DEV)
            X = torch.zeros(p1 - p0, P, dtype=torch.float64, device=DEV)
            H[piece[a:b] - p0, at[a:b]] = h
            X[piece[a:b] - p0, at[a:b]] = vals[sel]
            to = owner[p0:p1] - r0
            G.index_add_(0, to, torch.bmm(H.transpose(1, 2).contiguous(), H))
            m.index_add_(0, to, (H * X[:, :, None]).sum(1))
            p0 = p1
        G.diagonal(dim1=1, dim2=2).add_(lam)
        out[rows[r0:r1]] = _solve_spd(G, m)
        r0 = r1
    return out


def _row_sum(i, x, rows):
    """Row sums of x (nonzeros x R) by row index i: first in pieces of 256 nonzeros, then the pieces."""
    order = torch.argsort(i, stable=True)
    cnt = torch.bincount(i, minlength=rows)
    pieces = (cnt + 255) // 256
    owner = torch.repeat_interleave(torch.arange(rows, device=DEV), pieces)
    at = torch.arange(owner.numel(), device=DEV) - (torch.cumsum(pieces, 0) - pieces)[owner]
    part = torch.segment_reduce(x[order], "sum", lengths=(cnt[owner] - 256 * at).clamp(max=256), unsafe=True)
    return torch.segment_reduce(part, "sum", lengths=pieces, unsafe=True)


def _predict(ind, F):
    v = F[0][ind[0]].clone()
    for i, f in zip(ind[1:], F[1:]):
        v *= f[i]
    return v.sum(1)


def _rmse(ind, vals, F):
    sq, n, step = 0.0, vals.numel(), 4_000_000
    for a in range(0, n, step):
        sq += float((vals[a:a + step] - _predict([i[a:a + step] for i in ind], F)).square().sum())
    return math.sqrt(sq / n) if n else 0.0


def _sgd_exact(ind, vals, F, lr, lam):
    """One epoch of the default schedule: walkers of SPAN nonzeros step through sub-steps of SUB from the factors
    as the sub-step began; along a run of equal indices a walker keeps its copy of the row; a row adds the sum of
    its runs' changes, or their mean where it is hot."""
    n, N = vals.numel(), len(F)
    F = [f.clone() for f in F]
    W = (n + SPAN - 1) // SPAN
    hot = []
    for i, f in zip(ind, F):
        c = torch.bincount(i, minlength=f.shape[0])
        hot.append((c > HOT) & (c.double() > 4.0 * n / f.shape[0]))
    base = torch.arange(W, device=DEV) * SPAN
    for s in range(0, SPAN, SUB):
        live = torch.zeros(W, dtype=torch.bool, device=DEV)
        total = [torch.zeros_like(f) for f in F]
        runs = [torch.zeros(f.shape[0], dtype=torch.float64, device=DEV) for f in F]
        cur = [torch.zeros(W, dtype=torch.int64, device=DEV) for _ in F]
        v = [torch.zeros(W, F[0].shape[1], dtype=torch.float64, device=DEV) for _ in F]
        v0 = [x.clone() for x in v]

        def hand_in(k, which):
            r = cur[k][which]
            total[k].index_add_(0, r, (v[k] - v0[k])[which])
            runs[k].index_add_(0, r, torch.ones_like(r, dtype=torch.float64))

        for q in range(min(SUB, SPAN - s)):
            e = base + s + q
            ok = e < n
            if not bool(ok.any()):
                break
            e = e.clamp(max=n - 1)
            for k in range(N):
                new = ok & (~live | (ind[k][e] != cur[k]))
                hand_in(k, new & live)
                row = F[k][ind[k][e]]
                cur[k] = torch.where(new, ind[k][e], cur[k])
                v[k] = torch.where(new[:, None], row, v[k])
                v0[k] = torch.where(new[:, None], row, v0[k])
            live = live | ok
            full = v[0].clone()
            for k in range(1, N):
                full *= v[k]
            err = (vals[e] - full.sum(1))[:, None]
            step = []
            for k in range(N):
                o = torch.ones_like(full)
                for j in range(N):
                    if j != k:
                        o = o * v[j]
                step.append(lr * (err * o - lam * v[k]))
            for k in range(N):
                v[k] = torch.where(ok[:, None], v[k] + step[k], v[k])
        for k in range(N):
            hand_in(k, live)
            scale = torch.where(hot[k] & (runs[k] > 0), 1.0 / runs[k].clamp(min=1), torch.ones_like(runs[k]))
            F[k] += total[k] * scale[:, None]
    return F


def _ccd_exact(ind, vals, F, lam):
    """One CCD++ epoch: per column, every mode's column in turn from the residual without that component."""
    F = [f.clone() for f in F]
    e = vals - _predict(ind, F)
    order, count = [torch.argsort(i, stable=True) for i in ind], []
    for i, f in zip(ind, F):
        count.append(torch.bincount(i, minlength=f.shape[0]))

    def row_sums(m, x):
        return torch.segment_reduce(x[order[m]], "sum", lengths=count[m], unsafe=True)

    for f in range(F[0].shape[1]):
        col = [x[:, f].clone() for x in F]
        old = torch.ones_like(e)
        for c, i in zip(col, ind):
            old *= c[i]
        e += old
        for m in range(len(F)):
            h = torch.ones_like(e)
            for k in range(len(F)):
                if k != m:
                    h *= col[k][ind[k]]
            num, den = row_sums(m, e * h), row_sums(m, h * h)
            col[m] = torch.where(count[m] > 0, num / (lam + den), torch.zeros_like(num))
        new = torch.ones_like(e)
        for c, i in zip(col, ind):
            new *= c[i]
        e -= new
        for x, c in zip(F, col):
            x[:, f] = c
    return F


def _grad_exact(ind, vals, F, lam, per_occurrence):
    e = vals - _predict(ind, F)
    loss, grads = 0.5 * e.square().sum(), []
    for m, f in enumerate(F):
        h = torch.ones(vals.numel(), f.shape[1], dtype=torch.float64, device=DEV)
        for k in range(len(F)):
            if k != m:
                h *= F[k][ind[k]]
        c = torch.bincount(ind[m], minlength=f.shape[0]).double()[:, None] if per_occurrence else 1.0
        grads.append(lam * c * f - _row_sum(ind[m], h.mul_(e[:, None]), f.shape[0]))
        loss = loss + 0.5 * lam * (c * f.square()).sum()
    return {"loss": loss, "grads": grads}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        tr_rmse, te_rmse, factors = [], [], []
        for _, _, (ind, vals), (ti, tv), F in _problems(case, seed):
            F = [f.double() for f in F]
            for _ in range(case["iters"]):
                for m in range(3):
                    F[m] = _als_exact(ind, vals, F, m, LAM)
            tr_rmse.append(_rmse(ind, vals, F))
            te_rmse.append(_rmse(ti, tv, F))
            factors.append(torch.cat([f.reshape(-1) for f in F]))
        return {"rmse_tr": np.array(tr_rmse), "rmse_te": np.array(te_rmse), "factors": factors}
    ind, vals, gen = _tensor(case, seed)
    test = None
    if kind == "solve":
        (ind, vals), test = _split(ind, vals, gen, 0.1)
    F = [f.double() for f in _init(_dims(case), case["rank"], gen, positive=kind == "grad")]
    if kind == "grad":
        return _grad_exact(ind, vals, F, LAM, case["per_occurrence"])
    if kind == "mttkrp":
        out = []
        for m, f in enumerate(F):
            h = vals[:, None].expand(-1, f.shape[1]).clone()
            for k in range(len(F)):
                if k != m:
                    h *= F[k][ind[k]]
            out.append(_row_sum(ind[m], h, f.shape[0]))
        return out
    if kind == "als_mode":
        return _als_exact(ind, vals, F, case["mode"], LAM)
    if kind == "sgd":
        return _sgd_exact(ind, vals, F, SGD_LR, LAM)
    if kind == "ccd":
        return _ccd_exact(ind, vals, F, LAM)
    if kind == "als":
        for m in range(len(F)):
            F[m] = _als_exact(ind, vals, F, m, LAM)
        return F
    tr, te = [_rmse(ind, vals, F)], [_rmse(*test, F)]
    for _ in range(case["epochs"]):
        for m in range(len(F)):
            F[m] = _als_exact(ind, vals, F, m, LAM)
        tr.append(_rmse(ind, vals, F))
        te.append(_rmse(*test, F))
    return {"rmse_tr": np.array(tr), "rmse_te": np.array(te), "factors": F}
