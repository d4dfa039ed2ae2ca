"""Performance cases of the sparse MTTKRP / CP library, through its Python binding.

Every case is a call (or the two or three calls that belong together) that a
program working with a sparse tensor makes: the MTTKRP of each format, all
modes or the root mode, the tensor-times-matrix product, a CP-ALS fit, a
completion training step, and the path from a tensor on the device to the
first all-mode result.  Tensors are made on the GPU from the seed: distinct
coordinates, uniform or Zipf per mode (hot rows at low indices) in arbitrary
order, the shapes and laws of the benchmark and the tests, or generic ones.

A case is a dict of plain values:
  kind    "allmode" | "root" | "ttm" | "cpd" | "complete" | "build"
  dims    mode lengths, "500000x200000x50000"
  skew    Zipf exponent per mode, 0 = uniform, "1.2,1.2,0"
  nnz     nonzeros asked for
  type    format type (the driver's -t value: 3 COO, 8 B-CSF, 9 / 13 / 14 one
          tree for every mode, 10 HB-CSF, 12 MM-CSF)
  mode    root mode of the single-root types
  R       rank
  dtype   factor storage, "f32" | "bf16"
  fbr     fiber split threshold (-f)
  iters   CP-ALS iterations
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mm-csf_amd"))
import mmcsf  # noqa: E402

NO_SPLIT = 99999999  # the library's default -f


def _case(name, kind, dims, skew, nnz, type, R, dtype="f32", mode=0, fbr=128, iters=0):
    c = {"kind": kind, "dims": dims, "skew": skew, "nnz": nnz, "type": type, "mode": mode, "R": R,
         "dtype": dtype, "fbr": fbr, "iters": iters}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small tensor, all modes: an interactive session, a unit of a batch
        # of small problems; launches and latency count
        _case("allmode_tiny", "allmode", "300x200x100", "0,0,0", 20_000, 12, 32),
        # the plain COO type on a uniform tensor of the benchmark
        _case("coo_uniform", "root", "2000x2000x2000", "0,0,0", 1_000_000, 3, 32),
        # HB-CSF of an odd-sized skewed tensor at a rank that no vector width
        # divides (CP ranks of 5, 10, 25 are common), rooted at a middle mode
        _case("hbcsf_rank10", "root", "123457x70001x9973", "1.1,0,1.1", 3_300_001, 10, 10, mode=1),
        # the benchmark's headline tensor, all modes from MM-CSF, both factor
        # storages: the inner product of every CP iteration
        _case("allmode_skewed", "allmode", "500000x200000x50000", "1.2,1.2,0", 100_000_000, 12, 32),
        _case("allmode_skewed_bf16", "allmode", "500000x200000x50000", "1.2,1.2,0", 100_000_000, 12, 32, "bf16"),
        # four modes at a wide rank
        _case("allmode_4d", "allmode", "100000x50000x20000x1000", "1.1,0,1.1,0", 50_000_000, 12, 64),
        # one tree serving every mode: the layout for tensors whose structure
        # should be held once; the other modes scatter
        _case("onetree_allmode", "allmode", "500000x200000x50000", "1.2,1.2,0", 20_000_000, 14, 32),
        # tensor-times-matrix on the leaf mode (the step of a Tucker sweep)
        _case("ttm_leaf", "ttm", "500000x200000x50000", "1.2,1.2,0", 20_000_000, 8, 32, fbr=NO_SPLIT),
        # a CP-ALS fit of the library's default iteration count
        _case("cpd_als", "cpd", "200000x100000x20000", "1.2,0,0", 20_000_000, 12, 32, iters=10),
        # completion training steps: loss and the gradient of every factor
        _case("complete_r16", "complete", "1000000x500000x100000", "1.1,1.1,0", 50_000_000, 12, 16),
        _case("complete_r64_bf16", "complete", "1000000x500000x100000", "1.1,1.1,0", 20_000_000, 12, 64, "bf16"),
        # a new tensor: format build and the first all-mode MTTKRP on it
        _case("build_allmode", "build", "500000x200000x50000", "1.2,1.2,0", 20_000_000, 12, 32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["allmode", "allmode", "root", "root", "ttm", "cpd", "complete", "build"])
    nd = 4 if kind != "cpd" and rng.random() < 0.3 else 3
    lo, hi = {"allmode": (20_000, 50_000_000), "root": (50_000, 30_000_000), "ttm": (100_000, 20_000_000),
              "cpd": (200_000, 20_000_000), "complete": (1_000_000, 20_000_000),
              "build": (100_000, 20_000_000)}[kind]
    nnz = _log_int(rng, lo, hi)
    type = {"allmode": rng.choice([12, 12, 12, 9, 13, 14]), "root": rng.choice([3, 8, 10]),
            "ttm": 8}.get(kind, 12)
    if type in (9, 13, 14):
        nnz = min(nnz, 20_000_000)
    # mode lengths: spread, with room for distinct coordinates in skewed modes
    while True:
        dims = [_log_int(rng, 300, 500_000) for _ in range(nd)]
        if kind == "ttm" and math.prod(sorted(dims)[:-1]) < 100 * nnz:
            continue
        if 3000 * nnz <= math.prod(dims) < 1 << 62 and len(set(dims)) == nd:
            break
    skew = [rng.choice(["0", "0", "1.1", "1.2"]) for _ in range(nd)]
    skew[max(range(nd), key=lambda m: dims[m])] = "0"
    bf16 = kind != "build" and rng.random() < 0.35
    if kind in ("ttm", "complete") or bf16:
        R = rng.choice([8, 12, 16, 20, 24, 32, 40, 48, 64])
    else:
        R = rng.choice([5, 8, 10, 12, 16, 20, 25, 32, 40, 50, 64])
    if kind == "cpd":
        R = rng.choice([8, 10, 16, 24, 32, 40])
        bf16 = bf16 and R % 4 == 0
    return _case(None, kind, "x".join(map(str, dims)), ",".join(skew), nnz, type, R, "bf16" if bf16 else "f32",
                 mode=rng.randrange(nd), fbr=NO_SPLIT if kind == "ttm" else rng.choice([128, NO_SPLIT]),
                 iters=rng.choice([3, 5, 10]) if kind == "cpd" else 0)


# ---- inputs --------------------------------------------------------------------

def _dims(case):
    return [int(x) for x in case["dims"].split("x")]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _draw_mode(d, alpha, n, g):
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    if not alpha:
        return (u * d).long().clamp_(max=d - 1)
    # summed on the host: a parallel prefix sum may round differently from run to run
    cdf = torch.from_numpy(np.cumsum(np.arange(1, d + 1, dtype=np.float64) ** -alpha)).cuda()
    return torch.searchsorted(cdf, u.mul_(float(cdf[-1]))).clamp_(max=d - 1)


def _distinct(dims, skew, nnz, g):
    """nnz distinct coordinates as linear indices, in random order (fewer where
    the skewed modes run out of free places)."""
    keys = None
    for _ in range(12):
        have = 0 if keys is None else keys.numel()
        if have >= nnz:
            break
        n = int((nnz - have) * (1.3 if have == 0 else 2.5)) + 4096
        k = torch.zeros(n, dtype=torch.int64, device="cuda")
        for d, a in zip(dims, skew):
            k.mul_(d).add_(_draw_mode(d, a, n, g))
        keys = (k if keys is None else torch.cat([keys, k])).sort().values
        first = torch.ones(keys.numel(), dtype=torch.bool, device="cuda")
        torch.ne(keys[1:], keys[:-1], out=first[1:])
        keys = keys[first]
        del k, first
    return keys[torch.randperm(keys.numel(), generator=g, device="cuda")[:nnz]]


def _distinct_fibers(dims, skew, nnz, g):
    """The same with exactly nnz // 2 fibers along the last of dims (the output
    of a tensor-times-matrix product has a row per fiber): every fiber holds
    one nonzero, the others fall on fibers of Zipf and of uniform use."""
    d = dims[-1]
    fib = _distinct(dims[:-1], skew[:-1], nnz // 2, g)
    nf = fib.numel()
    n = 2 * nnz
    at = torch.cat([_draw_mode(nf, 0.9, n // 2, g), _draw_mode(nf, 0.0, n - n // 2, g),
                    torch.arange(nf, device="cuda")])
    keys = fib[at].mul_(d).add_(_draw_mode(d, skew[-1], at.numel(), g)).unique()
    base = torch.ones(keys.numel(), dtype=torch.bool, device="cuda")
    own = keys.div(d, rounding_mode="floor")
    torch.ne(own[1:], own[:-1], out=base[1:])
    more = keys[~base]
    keys = torch.cat([keys[base], more[torch.randperm(more.numel(), generator=g, device="cuda")[:nnz - nf]]])
    return keys[torch.randperm(keys.numel(), generator=g, device="cuda")]


def _coords(case, g):
    """int32 coordinates per mode of distinct nonzeros, in random order."""
    dims = _dims(case)
    skew = [float(x) for x in case["skew"].split(",")]
    order = _order(dims, case["mode"]) if case["kind"] == "ttm" else list(range(len(dims)))
    dims, skew = [dims[m] for m in order], [skew[m] for m in order]
    make = _distinct_fibers if case["kind"] == "ttm" else _distinct
    keys = make(dims, skew, case["nnz"], g)
    inds = [None] * len(dims)
    for m, d in zip(reversed(order), reversed(dims)):
        inds[m] = (keys % d).int()
        keys = keys.div_(d, rounding_mode="floor")
    return inds


def _planted(inds, A, noise, g, chunk=8_000_000):
    """Values of a CP model with factors A, plus noise, at the coordinates."""
    vals = torch.empty(inds[0].numel(), device="cuda")
    for s in range(0, vals.numel(), chunk):
        p = A[0][inds[0][s:s + chunk].long()]
        for a, i in zip(A[1:], inds[1:]):
            p.mul_(a[i[s:s + chunk].long()])
        v = p.sum(1)
        vals[s:s + chunk] = v.add_(torch.randn(v.numel(), generator=g, device="cuda"), alpha=noise)
    return vals


def _inputs(case, seed):
    """(dims, inds, vals, factors) of a case, from the seed alone."""
    g = _gen(seed)
    dims, R = _dims(case), case["R"]
    inds = _coords(case, g)
    if case["kind"] == "cpd":
        # a nonnegative model and a uniform initial guess
        A = [torch.randn((d, R), generator=g, device="cuda").abs_() for d in dims]
        vals = _planted(inds, A, 0.01, g)
        U = [torch.rand((d, R), generator=g, device="cuda") for d in dims]
    elif case["kind"] == "complete":
        # ratings-like values of a rank-16 model and a small random guess
        A = [torch.randn((d, 16), generator=g, device="cuda") * 0.25 for d in dims]
        vals = _planted(inds, A, 0.01, g)
        U = [torch.randn((d, R), generator=g, device="cuda") * 0.3 for d in dims]
    else:
        vals = torch.rand(inds[0].numel(), generator=g, device="cuda")
        U = [torch.rand((d, R), generator=g, device="cuda") for d in dims]
    if case["dtype"] == "bf16" and case["kind"] != "cpd":
        U = [mmcsf.to_bf16(u) for u in U]
    return dims, inds, vals, U


def prepare(case, seed):
    dims, inds, vals, U = _inputs(case, seed)
    X = mmcsf.Tensor.from_torch(dims, inds, vals)
    del inds, vals
    s = {"case": case, "U": U}
    if case["kind"] == "build":
        s["X"] = X
        return s
    s["fmt"] = mmcsf.Format(X, case["type"], mode=case["mode"], fbr_threshold=case["fbr"])
    X.free()
    if case["kind"] == "ttm":
        s["leaf"] = U[s["fmt"].info()["modeOrder"][-1]]
    if case["kind"] == "complete":
        for u in U:
            u.requires_grad_(True)
    return s


def run(state):
    case, U = state["case"], state["U"]
    kind = case["kind"]
    if kind == "allmode":
        outs, _ = mmcsf.mttkrp_allmode(state["fmt"], U)
        return outs
    if kind == "root":
        return mmcsf.mttkrp(state["fmt"], case["mode"], U)
    if kind == "ttm":
        return mmcsf.ttm(state["fmt"], state["leaf"])
    if kind == "cpd":
        F = [u.clone() for u in U]
        lam, st = mmcsf.cpd_als(state["fmt"], F, iters=case["iters"], tol=0.0, mttkrp_bf16=case["dtype"] == "bf16")
        # the model as a program stores it: float32 weights beside float32 factors
        return {"factors": F, "lambda": lam.astype(np.float32),
                "fit": np.array(st["fit_history"], dtype=np.float32)}
    if kind == "complete":
        loss = mmcsf.cp_completion_loss(state["fmt"], U)
        return {"loss": loss.detach(), "grads": torch.autograd.grad(loss, U)}
    fmt = mmcsf.Format(state["X"], case["type"], mode=case["mode"], fbr_threshold=case["fbr"])
    outs, _ = mmcsf.mttkrp_allmode(fmt, U)
    return outs


# ---- what a pass cannot do without ------------------------------------------------

def work(case):
    """Bytes: each stored nonzero's leaf index and value once per output mode
    (a build reads every coordinate and value once instead), each factor row
    that can be used once, each output element once.  Flops: products and
    sums per nonzero and column."""
    dims, n, R, kind = _dims(case), case["nnz"], case["R"], case["kind"]
    N = len(dims)
    es = 2 if case["dtype"] == "bf16" else 4
    fac = sum(min(d, n) * R * es for d in dims)
    outs = sum(d * R * 4 for d in dims)
    if kind == "allmode":
        return {"bytes": N * 8 * n + fac + outs, "flops": N * N * n * R}
    if kind == "build":
        return {"bytes": 4 * (N + 1) * n + N * 8 * n + fac + outs, "flops": N * N * n * R}
    if kind == "root":
        key = 4 * (N - 1) if case["type"] == 3 else 0
        m = case["mode"]
        return {"bytes": (8 + key) * n + fac - min(dims[m], n) * R * es + dims[m] * R * 4, "flops": N * n * R}
    if kind == "ttm":
        leaf = dims[_order(dims, case["mode"])[-1]]
        return {"bytes": 8 * n + min(leaf, n) * R * es + n // 2 * R * 4, "flops": 2 * n * R}
    if kind == "cpd":
        it = case["iters"]
        return {"bytes": it * (N * 8 * n + 2 * fac), "flops": it * (N * N * n * R + sum(4 * d * R * R for d in dims))}
    return {"bytes": N * 8 * n + fac + sum(d * R * es for d in dims), "flops": N * 2 * N * n * R}


# ---- the same results in 64 bits, in plain torch -------------------------------------

def _order(dims, mode):
    """Root mode first, the others by ascending length."""
    return [mode] + sorted((m for m in range(len(dims)) if m != mode), key=lambda m: dims[m])


def _segment_rows(out, seg, perm, contribution, chunk):
    """out[seg[x]] += contribution(x) for x in perm (seg[perm] ascending): per
    chunk a prefix sum along the nonzeros, differenced at the segment ends."""
    n = perm.numel()
    for s in range(0, n, chunk):
        sel = perm[s:s + chunk]
        rows = seg[sel].long()
        c = contribution(sel).t().contiguous().cumsum_(1)          # R x chunk
        last = torch.ones(rows.numel(), dtype=torch.bool, device=rows.device)
        torch.ne(rows[1:], rows[:-1], out=last[:-1])
        at = last.nonzero().squeeze(1)
        tot = c[:, at]
        tot[:, 1:] -= c[:, at[:-1]]
        out.index_add_(0, rows[at], tot.t().contiguous())
    return out


def _mttkrp64(inds, w, U, mode, chunk=None):
    R = U[0].shape[1]
    chunk = chunk or max(1 << 18, (1 << 27) // R)

    def part(sel):
        p = w[sel].double()[:, None]
        for m, u in enumerate(U):
            if m != mode:
                p = p * u[inds[m][sel].long()]
        return p

    out = torch.zeros((U[mode].shape[0], R), dtype=torch.float64, device="cuda")
    return _segment_rows(out, inds[mode], torch.argsort(inds[mode]), part, chunk)


def _ttm64(inds, vals, leaf, order):
    key = torch.zeros(vals.numel(), dtype=torch.int64, device="cuda")
    for m in order[:-1]:
        key.mul_(int(inds[m].max()) + 1).add_(inds[m])
    key, perm = key.sort()
    seg = torch.zeros_like(key)
    seg[1:] = (key[1:] != key[:-1]).long().cumsum(0)
    fibers = int(seg[-1]) + 1
    back = torch.empty_like(seg)
    back[perm] = seg
    i = inds[order[-1]]
    out = torch.zeros((fibers, leaf.shape[1]), dtype=torch.float64, device="cuda")
    return _segment_rows(out, back, perm, lambda sel: vals[sel].double()[:, None] * leaf[i[sel].long()],
                         max(1 << 18, (1 << 27) // leaf.shape[1]))


def _als64(inds, vals, U, iters):
    N, R = len(U), U[0].shape[1]
    U = [u.clone() for u in U]
    G = [u.t() @ u for u in U]
    xx = float(vals.double().square().sum())
    fits = []
    for it in range(iters):
        for m in range(N):
            M = _mttkrp64(inds, vals, U, m)
            H = torch.ones((R, R), dtype=torch.float64, device="cuda")
            for n in range(N):
                if n != m:
                    H = H * G[n]
            U[m] = torch.linalg.solve(H, M.t()).t()
            lam = U[m].norm(dim=0) if it == 0 else U[m].max(dim=0).values.clamp(min=1.0)
            U[m] = U[m] / lam
            G[m] = U[m].t() @ U[m]
        H = torch.ones((R, R), dtype=torch.float64, device="cuda")
        for n in range(N):
            H = H * G[n]
        res = xx + abs(float(lam @ H @ lam)) - 2 * float(((U[-1] * M) @ lam).sum())
        fits.append(1 - (res ** 0.5 if res > 0 else res) / xx ** 0.5)
    for m in range(N):
        nrm = U[m].norm(dim=0)
        lam = lam * nrm
        U[m] = U[m] / torch.where(nrm == 0, torch.ones_like(nrm), nrm)
    return {"factors": U, "lambda": lam, "fit": torch.tensor(fits, dtype=torch.float64)}


def _complete64(inds, vals, U):
    n, R = vals.numel(), U[0].shape[1]
    chunk = max(1 << 18, (1 << 27) // R)
    e = torch.empty(n, dtype=torch.float64, device="cuda")
    for s in range(0, n, chunk):
        p = U[0][inds[0][s:s + chunk].long()]
        for u, i in zip(U[1:], inds[1:]):
            p = p * u[i[s:s + chunk].long()]
        e[s:s + chunk] = p.sum(1) - vals[s:s + chunk].double()
    return {"loss": 0.5 * e.square().sum(), "grads": [_mttkrp64(inds, e, U, m) for m in range(len(U))]}


def exact(case, seed):
    dims, inds, vals, U = _inputs(case, seed)
    U = [u.double() for u in U]
    kind = case["kind"]
    if kind in ("allmode", "build"):
        return [_mttkrp64(inds, vals, U, m) for m in range(len(dims))]
    if kind == "root":
        return _mttkrp64(inds, vals, U, case["mode"])
    if kind == "ttm":
        order = _order(dims, case["mode"])
        return _ttm64(inds, vals, U[order[-1]], order)
    if kind == "cpd":
        return _als64(inds, vals, U, case["iters"])
    return _complete64(inds, vals, U)
