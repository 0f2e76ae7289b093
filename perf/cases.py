"""The calls this framework is measured on: ALTO construction, MTTKRP, CP-ALS
(one model, several in lockstep, a server's jobs) and CP-APR, each through
the package's public entry points.

listed() holds the fixed cases, draw() gives more of the same ranges.  A case
is a dict of plain values:

  kind   mttkrp | build | cpals | lockstep | serve | cpapr
  dims   mode sizes, "AxBxC" (lockstep / serve: unused, each job has its own)
  nnz    nonzeros (lockstep / serve: the largest job's; the others are
         spread below it)
  rank   CP rank
  prec   f64 | f32 | bf16 (factor storage; values and sums as the library
         defines them for that precision)
  zipf   exponent of the index distribution (0: uniform)
  iters  CP-ALS iterations / CP-APR outer iterations
  jobs   tensors of a lockstep or serve case
  bits   ALTO key width asked for (0: the library's choice)
"""
import math

import numpy as np
import torch

import alto_amd as A
from alto_amd import serve as S

PREC = {"f64": A.PREC_F64, "f32": A.PREC_F32, "bf16": A.PREC_BF16}
FACTOR = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
INNER = 10  # CP-APR inner iterations (the reference's default)


def _case(name, kind, dims, nnz, rank, prec="f64", zipf=1.1, iters=0, jobs=0, bits=0):
    c = dict(kind=kind, dims=dims, nnz=nnz, rank=rank, prec=prec, zipf=zipf, iters=iters, jobs=jobs, bits=bits)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: all modes of a 10K-nonzero tensor, one of the
        # serving stream's smallest jobs; a pass is launches and latency
        _case("mttkrp tiny", "mttkrp", "183x97x1210", 10_000, 8),
        # the CPU configuration of the benchmark: 1000^3, 1M nonzeros
        _case("mttkrp 1000cube", "mttkrp", "1000x1000x1000", 1_000_000, 16, zipf=0.0),
        # the headline tensor, every mode, in the default precision
        _case("mttkrp headline", "mttkrp", "12092x9184x28818", 76_900_000, 32),
        # the 5-mode shape of the precision study, at half its nonzeros, in
        # the storage meant for it (rank 64, bf16 factors, 128-bit keys)
        _case("mttkrp 5mode bf16", "mttkrp", "50000x50000x10000x2000x512", 100_000_000, 64, prec="bf16", zipf=1.2,
              bits=128),
        # a rank and mode sizes that no vector width divides
        _case("mttkrp odd rank", "mttkrp", "4099x20011x613x77", 6_000_000, 25),
        # a middle-sized job in single precision, below the size from which
        # the streams are ordered by fibers
        _case("mttkrp mid f32", "mttkrp", "30000x5000x2500x300", 3_000_000, 32, prec="f32"),
        # a new tensor: ALTO format, mode streams, first MTTKRP of each mode
        _case("build 20M", "build", "60000x25000x9000", 20_000_000, 16),
        # whole decompositions: upload, 20 iterations, download.  In double
        # precision: 20 solves amplify the rounding of 32-bit sums until two
        # equally good orders of them differ visibly
        _case("cpals 1000cube", "cpals", "1000x1000x1000", 1_000_000, 16, zipf=0.0, iters=20),
        _case("cpals 4mode", "cpals", "20000x6000x900x150", 2_000_000, 64, iters=20),
        # 16 small models of one rank stepped together
        _case("lockstep 16 jobs", "lockstep", "", 200_000, 16, jobs=16, iters=20),
        # jobs submitted at once to the continuous-batching server
        _case("serve 12 jobs", "serve", "", 1_500_000, 16, jobs=12, iters=20),
        # CP-APR of a count tensor, ten inner iterations per mode
        _case("cpapr counts", "cpapr", "262144x65536x16384x1024", 20_000_000, 10, zipf=0.0, iters=2, bits=128),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def dims_for(nmode, nnz, lo=64, hi=1 << 16):
        d = [logint(lo, hi) for _ in range(nmode)]
        while math.prod(d) < 3000 * nnz:  # sparse, as the listed tensors are
            d[d.index(min(d))] *= 3
        return "x".join(str(x | 1 if rng.random() < 0.5 else x) for x in d)

    kind = rng.choice(["mttkrp"] * 5 + ["build", "cpals", "cpals", "lockstep", "serve", "cpapr"])
    rank = rng.choice([8, 16, 32, 64, rng.randint(5, 64), rng.randint(5, 64)])
    if kind == "mttkrp":
        nnz = logint(10_000, 40_000_000)
        return _case("", kind, dims_for(rng.randint(3, 5), nnz), nnz, rank, prec=rng.choice(["f64", "f64", "f32", "bf16"]),
                     zipf=rng.choice([0.0, 1.1, 1.1, 1.2]))
    if kind == "build":
        nnz = logint(50_000, 20_000_000)
        return _case("", kind, dims_for(rng.randint(3, 4), nnz), nnz, min(rank, 32))
    if kind == "cpals":
        nnz = logint(20_000, 3_000_000)
        return _case("", kind, dims_for(rng.randint(3, 4), nnz, hi=20_000), nnz, rank, zipf=rng.choice([0.0, 1.1]),
                     iters=rng.randint(8, 20))
    if kind in ("lockstep", "serve"):
        return _case("", kind, "", logint(100_000, 400_000 if kind == "lockstep" else 1_500_000), min(rank, 32),
                     jobs=rng.randint(6, 16), iters=rng.randint(8, 20))
    nnz = logint(100_000, 10_000_000)
    return _case("", kind, dims_for(rng.randint(3, 4), nnz, lo=1000, hi=1 << 17), nnz, rng.randint(5, 24), zipf=0.0, iters=2)


# ------------------------------------------------------------------ inputs
def _dims(case):
    return [int(x) for x in case["dims"].split("x")]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _first_of_each(cols, dims, n):
    """Positions of the first n distinct coordinates in draw order, and how
    often each was drawn (fewer than n when there are not as many)."""
    key = torch.zeros_like(cols[0])
    for c, d in zip(cols, dims):  # 64-bit wrap-around only merges a few cells
        key = key * d + c
    key, order = torch.sort(key, stable=True)
    head = torch.ones_like(key, dtype=torch.bool)
    head[1:] = key[1:] != key[:-1]
    at = torch.nonzero(head).squeeze(1)
    count = torch.diff(at, append=torch.tensor([key.numel()], device=key.device))
    first, by = torch.sort(order[at])
    return first[:n], count[by][:n]


def _sparse(dims, nnz, zipf, g):
    """nnz distinct coordinates, uniform or Zipf over a random permutation of
    each mode, with lognormal values."""
    table = []
    for d in dims:
        w = torch.arange(1, d + 1, dtype=torch.float64, device="cuda").pow(-zipf).cumsum(0)
        table.append((w / w[-1], torch.randperm(d, generator=g, device="cuda")))

    def drawn(m):
        out = []
        for d, (w, p) in zip(dims, table):
            if zipf == 0:
                out.append(torch.randint(0, d, (m,), generator=g, device="cuda"))
            else:
                u = torch.rand(m, dtype=torch.float64, generator=g, device="cuda")
                out.append(p[torch.searchsorted(w, u).clamp_(max=d - 1)])
        return out

    cols, first = drawn(nnz + nnz // 4 + 64), None
    for _ in range(30):
        first, _ = _first_of_each(cols, dims, nnz)
        if first.numel() == nnz:
            break
        cols = [torch.cat([a, b]) for a, b in zip(cols, drawn(max(nnz // 2, 2 * (nnz - first.numel()))))]
    if first.numel() < nnz:
        raise ValueError(f"{dims} is too small a space for {nnz} distinct coordinates")
    cols = [c[first].contiguous() for c in cols]
    vals = torch.randn(nnz, dtype=torch.float64, generator=g, device="cuda").exp_()
    return cols, vals


def _counts(dims, nnz, rank, g):
    """Count tensor: draws from a rank-`rank` model with Gamma(0.5) factors."""
    cdf = [torch._standard_gamma(torch.full((rank, d), 0.5, dtype=torch.float64, device="cuda"), generator=g).cumsum(1)
           for d in dims]
    cols = [[] for _ in dims]
    for share in (1.3, 1.0, 2.0, 4.0, 8.0):
        per = int(nnz * share / rank) + 16
        for r in range(rank):
            for n, d in enumerate(dims):
                u = torch.rand(per, dtype=torch.float64, generator=g, device="cuda") * cdf[n][r, -1]
                cols[n].append(torch.searchsorted(cdf[n][r], u).clamp_(max=d - 1))
        flat = [torch.cat(c) for c in cols]
        # mix the components before the first nnz cells are taken
        mix = torch.randperm(flat[0].numel(), generator=g, device="cuda")
        flat = [c[mix] for c in flat]
        first, count = _first_of_each(flat, dims, nnz)
        if first.numel() == nnz:
            return [c[first].contiguous() for c in flat], count.to(torch.float64)
    raise ValueError(f"{dims} is too small a space for {nnz} distinct coordinates")


def _host_factors(dims, rank, seed):
    rng = np.random.default_rng(seed)
    return [rng.random((d, rank)) for d in dims]


def _factors(case, g):
    """Dense factors of the case's storage type, entries in (0, 1)."""
    return [torch.rand((d, case["rank"]), dtype=torch.float64, generator=g, device="cuda").to(FACTOR[case["prec"]])
            for d in _dims(case)]


def _jobs(case, seed):
    """The small tensors of a lockstep or serve case: 3-5 modes, nonzeros
    spread over a factor of 20 below case["nnz"]; their sizes are the case's,
    their entries the seed's."""
    rng = np.random.default_rng(case["nnz"])
    out = []
    for k in range(case["jobs"]):
        nnz = int(case["nnz"] * 20 ** (-k / max(case["jobs"] - 1, 1)))
        dims = [int(np.exp(rng.uniform(np.log(100), np.log(4000)))) for _ in range(3 + k % 3)]
        while math.prod(dims) < 3000 * nnz:
            dims[dims.index(min(dims))] *= 3
        out.append((dims, *_sparse(dims, nnz, case["zipf"], _gen(seed * 1000 + k))))
    return out


def _inputs(case, seed):
    g = _gen(seed)
    if case["kind"] == "cpapr":
        return _counts(_dims(case), case["nnz"], case["rank"], g), g
    return _sparse(_dims(case), case["nnz"], case["zipf"], g), g


class _Dev:
    """A torch tensor as the package's device calls take one (ptr, shape)."""

    def __init__(self, t):
        self.t, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)


def _tensor(dims, cols, vals, bits=0, nprtn=16):
    return A.AltoTensor.from_device(dims, [c.data_ptr() for c in cols], vals.data_ptr(), int(vals.numel()), nprtn=nprtn,
                                    lit_bits=bits)


def prepare(case, seed):
    kind, rank = case["kind"], case["rank"]
    if kind in ("lockstep", "serve"):
        jobs = _jobs(case, seed)
        torch.cuda.synchronize()
        if kind == "serve":  # a running server and the jobs' coordinates on the GPU
            return dict(case=case, seed=seed, jobs=jobs, server=S.Server(slots=8, lockstep_nnz=200_000))
        return dict(case=case, ts=[_tensor(d, c, v) for d, c, v in jobs],
                    U=[_host_factors(d, rank, seed * 1000 + k) for k, (d, _, _) in enumerate(jobs)])
    dims = _dims(case)
    (cols, vals), g = _inputs(case, seed)
    torch.cuda.synchronize()  # the library reads the coordinates on its own
    if kind == "build":  # the coordinate lists, and factors for the first MTTKRPs
        return dict(case=case, dims=dims, cols=cols, vals=vals, U=[_Dev(u) for u in _factors(case, g)])
    s = dict(case=case, dims=dims, t=_tensor(dims, cols, vals, case["bits"]))
    if kind == "mttkrp":
        s["U"] = [_Dev(u) for u in _factors(case, g)]
        s["out"] = [_Dev(torch.empty((d, rank), dtype=torch.float64, device="cuda")) for d in dims]
    else:
        s["U"] = _host_factors(dims, rank, seed)
    return s


# ------------------------------------------------------------------ the pass
def run(s):
    case = s["case"]
    kind, rank, prec = case["kind"], case["rank"], PREC[case["prec"]]
    if kind == "mttkrp":
        for m, out in enumerate(s["out"]):
            s["t"].mttkrp_device(m, s["U"], out, prec)
        # sums of 32-bit products: a program with 32-bit (or shorter)
        # factors takes them up as such
        return [o.t if case["prec"] == "f64" else o.t.float() for o in s["out"]]
    if kind == "build":
        t = _tensor(s["dims"], s["cols"], s["vals"], case["bits"])
        outs = [_Dev(torch.empty((d, rank), dtype=torch.float64, device="cuda")) for d in s["dims"]]
        for m, out in enumerate(outs):
            t.mttkrp_device(m, s["U"], out, prec)
        return [o.t for o in outs]
    if kind == "cpals":
        U, lam = [u.copy() for u in s["U"]], np.ones(rank)
        _, fits, _ = s["t"].cpd_als(U, lam, case["iters"], 0.0, prec)
        return dict(U=U, lam=lam, fits=fits)
    if kind == "lockstep":
        models = [A.CpdSession(t, U, prec) for t, U in zip(s["ts"], s["U"])]
        A.cpd_sessions_iterate(models, case["iters"], 0.0)
        out = []
        for m in models:
            U, lam, fit, _ = m.get()
            out.append(dict(U=np.concatenate([u.ravel() for u in U]), lam=lam, fit=fit))
        return out
    if kind == "serve":
        sv, out = s["server"], []
        ids = [sv.submit(d, [c.data_ptr() for c in cols], vals.data_ptr(), rank, case["iters"], 0.0, s["seed"] + k, prec,
                         device=True, nnz=int(vals.numel()), want_factors=True)
               for k, (d, cols, vals) in enumerate(s["jobs"])]
        for j, (d, _, _) in zip(ids, s["jobs"]):
            r, U, lam = sv.result(j, dims=d, rank=rank)
            sv.release(j)
            out.append(dict(U=np.concatenate([u.ravel() for u in U]), lam=lam, fit=r.fit))
            if r.status != 2:
                raise RuntimeError(f"job {j} ended with status {r.status}")
        return out
    U, lam = [u.copy() for u in s["U"]], np.ones(rank)
    r = s["t"].cp_apr(U, lam, case["iters"], INNER)
    return dict(U=U, lam=lam, loglik=r["loglik"], fit=r["ls_fit"], kkt=r["kkt"], inner=r["total_inner"])


def work(case):
    """Per MTTKRP or Phi: coordinates and value of each nonzero once, each
    factor once, the output once; per iteration also the dense step's passes
    over the mode's rows.  Set-up counts its input lists once."""
    kind, R = case["kind"], case["rank"]
    if kind in ("lockstep", "serve"):
        b = f = 0
        for k in range(case["jobs"]):
            n, N = int(case["nnz"] * 20 ** (-k / max(case["jobs"] - 1, 1))), 3 + k % 3
            b += n * 16 * N * case["iters"]
            f += n * R * N * N * case["iters"]
        return {"bytes": float(b), "flops": float(f)}
    dims, nnz = _dims(case), case["nnz"]
    N, rows = len(dims), sum(dims)
    el = {"f64": 8, "f32": 4, "bf16": 2}[case["prec"]]
    word = 16 if sum((d - 1).bit_length() for d in dims) > 64 else 8
    val = 8 if case["prec"] == "f64" else 4
    call_b = N * nnz * (word + val) + (N - 1) * rows * R * el + rows * R * 8
    call_f = N * nnz * R * N
    if kind == "mttkrp":
        return {"bytes": float(call_b), "flops": float(call_f)}
    if kind == "build":
        return {"bytes": float(nnz * 8 * (N + 1) + call_b), "flops": float(call_f)}
    if kind == "cpals":
        it = call_b + rows * R * (8 + 2 * el)
        return {"bytes": float(case["iters"] * it), "flops": float(case["iters"] * (call_f + 4 * rows * R * R))}
    n = case["iters"] * INNER
    return {"bytes": float(n * (call_b + 3 * rows * R * 8)), "flops": float(n * (call_f + 2 * N * nnz * R))}


# ------------------------------------------------------------------ 64-bit values
def _add_rows(out, rows, p):
    """out[rows[i]] += p[i], rows sorted: runs of at most 256 equal rows are
    summed first, so that a heavy row is not one long chain of additions."""
    head = torch.ones_like(rows, dtype=torch.bool)
    head[1:] = rows[1:] != rows[:-1]
    head[::256] = True
    at = torch.nonzero(head).squeeze(1)
    runs = torch.diff(at, append=torch.tensor([rows.numel()], device=rows.device))
    return out.index_add_(0, rows[at], torch.segment_reduce(p, "sum", lengths=runs, axis=0, unsafe=True))


def _mttkrp64(dims, cols, vals, U, mode, chunk=1 << 21):
    out = torch.zeros((dims[mode], U[0].shape[1]), dtype=torch.float64, device="cuda")
    for a in range(0, vals.numel(), chunk):
        rows, by = torch.sort(cols[mode][a:a + chunk])
        p = vals[a:a + chunk][by][:, None]
        for m in range(len(dims)):
            if m != mode:
                p = p * U[m][cols[m][a:a + chunk][by]]
        _add_rows(out, rows, p)
    return out


def _cpals64(dims, cols, vals, U, iters):
    R, normx = U[0].shape[1], float((vals * vals).sum())
    G = [u.T @ u for u in U]
    fits, lam = [], torch.ones(R, dtype=torch.float64, device="cuda")
    for it in range(iters):
        for n in range(len(dims)):
            M = _mttkrp64(dims, cols, vals, U, n)
            V = torch.ones((R, R), dtype=torch.float64, device="cuda")
            for m in range(len(dims)):
                if m != n:
                    V = V * G[m]
            X = torch.cholesky_solve(M.T.contiguous(), torch.linalg.cholesky(V)).T.contiguous()
            lam = X.norm(dim=0) if it == 0 else X.amax(0).clamp(min=1.0)
            U[n] = X / lam
            G[n] = U[n].T @ U[n]
        H = lam[:, None] * lam[None, :]
        for m in range(len(dims)):
            H = H * G[m]
        res = normx + abs(float(H.sum())) - 2 * float(((U[-1] * M).sum(0) * lam).sum())
        fits.append(1 - (math.sqrt(res) if res > 0 else res) / math.sqrt(normx))
    return U, lam, fits


def _cpapr64(dims, cols, vals, U, iters, epsilon=1e-5, tiny=1e-10, kappa=1e-2):
    R, N = U[0].shape[1], len(dims)
    lam = torch.ones(R, dtype=torch.float64, device="cuda")
    phi, kkt, last, total = [None] * N, [0.0] * N, [], 0

    def products(n):
        p = None
        for m in range(N):
            if m != n:
                p = U[m][cols[m]] if p is None else p * U[m][cols[m]]
        return p

    def normalise(n):
        s = U[n].abs().sum(0)
        U[n] = U[n] / s
        return lam * s

    for n in range(N):
        lam = normalise(n)
    it = 0
    for it in range(iters):
        for n in range(N):
            if it > 0:
                U[n] = torch.where((U[n] < tiny) & (phi[n] > 1), U[n] + kappa, U[n])
            U[n], lam = U[n] * lam, torch.ones_like(lam)
            rows, by = torch.sort(cols[n])
            pi, x = products(n)[by], vals[by]
            for _ in range(INNER):
                total += 1
                w = x / (U[n][rows] * pi).sum(1).clamp(min=tiny)
                phi[n] = _add_rows(torch.zeros_like(U[n]), rows, pi * w[:, None])
                kkt[n] = float(torch.minimum(U[n], 1 - phi[n]).abs().max())
                if kkt[n] < epsilon:
                    break
                U[n] = U[n] * phi[n]
            lam = normalise(n)
        last.append(max(kkt))
        if it > 0 and abs(last[-1] - last[-2]) <= epsilon * epsilon:
            break
    else:
        it = iters
    U[0], lam = U[0] * lam, torch.ones_like(lam)
    loglik = float((vals * (products(0) * U[0][cols[0]]).sum(1).clamp(min=tiny).log()).sum() - U[0].sum())
    lam = normalise(0)
    normx, M = float((vals * vals).sum()), _mttkrp64(dims, cols, vals, U, N - 1)
    H = lam[:, None] * lam[None, :]
    for u in U:
        H = H * (u.T @ u)
    res = normx + abs(float(H.sum())) - 2 * float(((U[-1] * M).sum(0) * lam).sum())
    fit = 1 - (math.sqrt(res) if res > 0 else res) / math.sqrt(normx)
    return U, lam, loglik, fit, last[it - 1], total


def _server_factors(dims, rank, seed):
    """The server's starting model: SplitMix64 of (seed, mode, index), in (0, 1]."""
    out = []
    for m, d in enumerate(dims):
        with np.errstate(over="ignore"):
            z = np.arange(1, d * rank + 1, dtype=np.uint64) + np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15)
            z = z + (np.uint64(m) << np.uint64(56))
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z = z ^ (z >> np.uint64(31))
        out.append(((z >> np.uint64(11)).astype(np.float64) + 1.0).reshape(d, rank) * 2.0 ** -53)
    return out


def exact(case, seed):
    def model(dims, cols, vals, U):
        U, lam, fits = _cpals64(dims, cols, vals, [torch.from_numpy(u).cuda() for u in U], case["iters"])
        return [u.cpu().numpy() for u in U], lam.cpu().numpy(), fits

    kind, rank = case["kind"], case["rank"]
    if kind in ("lockstep", "serve"):
        out = []
        for k, (d, cols, vals) in enumerate(_jobs(case, seed)):
            U0 = _host_factors(d, rank, seed * 1000 + k) if kind == "lockstep" else _server_factors(d, rank, seed + k)
            U, lam, fits = model(d, cols, vals, U0)
            out.append(dict(U=np.concatenate([u.ravel() for u in U]), lam=lam, fit=fits[-1]))
        return out
    dims = _dims(case)
    (cols, vals), g = _inputs(case, seed)
    if kind in ("mttkrp", "build"):
        U = [u.double() for u in _factors(case, g)]
        return [_mttkrp64(dims, cols, vals, U, m) for m in range(len(dims))]
    U = _host_factors(dims, rank, seed)
    if kind == "cpals":
        U, lam, fits = model(dims, cols, vals, U)
        return dict(U=U, lam=lam, fits=np.array(fits))
    U, lam, loglik, fit, kkt, inner = _cpapr64(dims, cols, vals, [torch.from_numpy(u).cuda() for u in U], case["iters"])
    return dict(U=[u.cpu().numpy() for u in U], lam=lam.cpu().numpy(), loglik=loglik, fit=fit, kkt=kkt, inner=inner)
