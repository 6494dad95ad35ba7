"""Timed cases of the CP / Tucker path: what a program that uses this package
has it do, through the package's public functions, over the range of sizes.

Each kind of work below is one family of cases:

* ``mttkrp``   -- ``unfolding_dot_khatri_rao`` of every mode of one tensor, the
  call that a program's own alternating loop makes;
* ``cp_grad``  -- ``cp_lstsq_grad``, the gradient with respect to every factor:
  the backward direction, one step of a gradient-based CP fit;
* ``project``  -- ``multi_mode_dot`` to the Tucker core and ``tucker_to_tensor``
  back to the full size: encode and decode with fixed factors;
* ``tucker``   -- a whole ``tucker`` call (HOOI from the SVD init);
* ``parafac``  -- a whole ``parafac`` call, from the default SVD init or from
  factors that the caller has;
* ``hals``     -- a whole ``non_negative_parafac_hals`` call;
* ``batched``  -- ``BatchedCP.run`` on many small problems;
* ``coo``      -- ``unfolding_dot_khatri_rao_coo`` of every mode of a sparse
  tensor, the call that a loop over coordinate data makes.

Tensors are CP or Tucker models with noise, made on the GPU from the seed.
"""
import math

import numpy as np
import torch

import tensorly_amd as tla
from tensorly_amd.batched import BatchedCP
from tensorly_amd.tenalg import unfolding_dot_khatri_rao_coo

DEV = "cuda"


def listed():
    return [
        # a slice of a real fluorescence experiment, order 4, in a program's own loop: the smallest calls,
        # where launches and host work count (the shape of the repository's real-data fixture)
        {"name": "mttkrp_small_order4", "kind": "mttkrp", "shape": "32x12x10x30", "rank": 3, "dtype": "float32",
         "precision": "fp32"},
        # measured data of no particular size: odd modes, a middling rank
        {"name": "mttkrp_odd_f32", "kind": "mttkrp", "shape": "257x301x203", "rank": 20, "dtype": "float32",
         "precision": "fp32"},
        # the same in double precision, the default type of numpy data
        {"name": "mttkrp_odd_f64", "kind": "mttkrp", "shape": "201x179x160", "rank": 16, "dtype": "float64",
         "precision": "fp32"},
        # the largest: a 1 GiB order-4 tensor at the largest rank, split-bf16 arithmetic
        {"name": "mttkrp_order4_bf16x3", "kind": "mttkrp", "shape": "128x128x128x128", "rank": 64,
         "dtype": "float32", "precision": "bf16x3"},
        # one gradient step on the 512 MiB benchmark tensor
        {"name": "cp_grad_512", "kind": "cp_grad", "shape": "512x512x512", "rank": 32, "dtype": "float32"},
        # compress and rebuild a tensor of odd sizes with Tucker factors that the program keeps
        {"name": "project_odd_f32", "kind": "project", "shape": "250x331x190", "rank": "25x30x20",
         "dtype": "float32"},
        # the Tucker benchmark: 256^3 to a 32^3 core
        {"name": "tucker_256", "kind": "tucker", "shape": "256x256x256", "rank": "32x32x32", "dtype": "float32",
         "sweeps": 5},
        # an ordinary first fit of measured data: SVD init (the default), plain ALS
        {"name": "parafac_svd_init", "kind": "parafac", "shape": "149x120x90", "rank": 10, "dtype": "float32",
         "precision": "fp32", "dimtree": False, "init": "svd", "sweeps": 20},
        # the CP benchmark: 512^3, rank 32, the fast sweep, refitting from factors in hand
        {"name": "parafac_512_bf16x3", "kind": "parafac", "shape": "512x512x512", "rank": 32, "dtype": "float32",
         "precision": "bf16x3", "dimtree": True, "init": "given", "sweeps": 5},
        # a non-negative fit of a spectroscopy-sized tensor, going on from factors in hand
        {"name": "hals_256", "kind": "hals", "shape": "256x200x150", "rank": 16, "dtype": "float32", "sweeps": 3},
        # many small problems at once, sizes 8 to 64, ranks 2 to 16
        {"name": "batched_1024", "kind": "batched", "problems": 1024, "sweeps": 5},
        # sparse counts with one short mode, 2 million nonzeros
        {"name": "coo_2m", "kind": "coo", "shape": "1000x1000x1000x10", "nnz": 2000000, "rank": 16,
         "dtype": "float32"},
    ]


# --------------------------------------------------------------------------
def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _shape(rng, nd, lo, hi, smallest, largest):
    """nd mode sizes in [smallest, largest] whose product is spread over the logarithm of [lo, hi]; every second
    draw has sizes that are multiples of 8 or 16 (16 or 32 for the last), the others come as they fall."""
    while True:
        side = _log(rng, lo, hi) ** (1.0 / nd)
        s = [int(round(side * _log(rng, 0.4, 2.5))) for _ in range(nd)]
        if rng.random() < 0.5:
            q = 8 if side < 48 else 16
            s = [max(q, (v + q // 2) // q * q) for v in s[:-1]] + [max(2 * q, (s[-1] + q) // (2 * q) * (2 * q))]
        n = math.prod(s)
        if min(s) >= smallest and max(s) <= largest and lo <= n <= hi:
            return s


def _text(s):
    return "x".join(str(int(v)) for v in s)


def draw(rng):
    kind = rng.choice(["mttkrp", "mttkrp", "mttkrp", "cp_grad", "project", "tucker", "parafac", "hals", "batched",
                       "coo"])
    if kind == "mttkrp":
        nd = rng.choice([3, 3, 4])
        dtype = rng.choice(["float32", "float32", "float32", "float64"])
        s = _shape(rng, nd, 2 ** 13, 2 ** 27 if dtype == "float32" else 2 ** 25, 6, 4096)
        return {"kind": kind, "shape": _text(s), "rank": int(_log(rng, 2, 64.99)), "dtype": dtype,
                "precision": rng.choice(["fp32", "fp32", "bf16x3"]) if dtype == "float32" else "fp32"}
    if kind == "cp_grad":
        s = _shape(rng, 3, 2 ** 15, 2 ** 27, 12, 2048)
        return {"kind": kind, "shape": _text(s), "rank": int(_log(rng, 2, 48.99)), "dtype": "float32"}
    if kind == "project":
        dtype = rng.choice(["float32", "float32", "float64"])
        s = _shape(rng, 3, 2 ** 14, 2 ** 25, 12, 1024)
        return {"kind": kind, "shape": _text(s), "rank": _text(min(v, int(_log(rng, 4, 64.99))) for v in s),
                "dtype": dtype}
    if kind == "tucker":
        s = _shape(rng, 3, 2 ** 15, 2 ** 24, 24, 512)
        return {"kind": kind, "shape": _text(s), "rank": _text(min(v // 3, int(_log(rng, 3, 32.99))) for v in s),
                "dtype": "float32", "sweeps": rng.randint(2, 6)}
    if kind == "parafac":
        init = rng.choice(["svd", "given"])
        s = _shape(rng, 3, 2 ** 15, 2 ** 22 if init == "svd" else 2 ** 26, 24, 512 if init == "svd" else 1024)
        return {"kind": kind, "shape": _text(s), "rank": int(_log(rng, 2, 16.99 if init == "svd" else 32.99)),
                "dtype": "float32", "precision": rng.choice(["fp32", "bf16x3"]) if init == "given" else "fp32",
                "dimtree": rng.random() < 0.5, "init": init, "sweeps": rng.randint(3, 12)}
    if kind == "hals":
        s = _shape(rng, 3, 2 ** 15, 2 ** 25, 24, 512)
        return {"kind": kind, "shape": _text(s), "rank": int(_log(rng, 3, 24.99)), "dtype": "float32",
                "sweeps": rng.randint(2, 4)}
    if kind == "batched":
        return {"kind": kind, "problems": int(_log(rng, 32, 1024.99)), "sweeps": rng.randint(3, 8)}
    nd = rng.choice([3, 4])
    s = [int(_log(rng, 10, 2000)) for _ in range(nd)]
    nnz = int(min(_log(rng, 1e4, 2e6), 0.2 * math.prod(s)))
    return {"kind": "coo", "shape": _text(s), "nnz": nnz, "rank": int(_log(rng, 2, 32.99)), "dtype": "float32"}


# --------------------------------------------------------------------------
def _sizes(case, key="shape"):
    return [int(v) for v in case[key].split("x")]


def _dtype(case):
    return getattr(torch, case["dtype"])


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *s, dtype=torch.float32):
    return torch.randn(s, generator=g, device=DEV, dtype=dtype)


def _rand(g, *s, dtype=torch.float32):
    return torch.rand(s, generator=g, device=DEV, dtype=dtype)


def _kr(factors):
    """Rows of the Khatri-Rao product, the first factor varying slowest."""
    out = factors[0]
    for f in factors[1:]:
        out = (out[:, None, :] * f[None, :, :]).reshape(-1, out.shape[1])
    return out


def _noisy(model, g, level):
    """model + noise of `level` times its norm."""
    e = torch.randn(model.shape, generator=g, device=DEV, dtype=model.dtype)
    e *= level * torch.linalg.vector_norm(model) / math.sqrt(model.numel())
    return model.add_(e)


def _cp_data(case, seed):
    """(tensor, factors near the model's): a CP model with noise that leaves a fit of about 0.7."""
    g, dt, s, r = _gen(seed), _dtype(case), _sizes(case), int(case["rank"])
    if case["kind"] == "hals":  # spectra and concentrations: not negative, small in most places
        f = [_rand(g, n, r, dtype=dt) ** 4 for n in s]
        near = [a + 0.1 * _rand(g, *a.shape, dtype=dt) for a in f]
    else:
        f = [_randn(g, n, r, dtype=dt) for n in s]
        near = [a + 0.3 * _randn(g, *a.shape, dtype=dt) for a in f]
    return _noisy((f[0] @ _kr(f[1:]).T).reshape(s), g, 0.3), near


def _orthonormal(g, n, k, dt):
    return torch.linalg.qr(_randn(g, n, k, dtype=torch.float64).cpu())[0].to(device=DEV, dtype=dt).contiguous()


def _tucker_data(case, seed):
    """(tensor, factors): a Tucker model whose core falls off along each mode, as the spectra of data do."""
    g, dt, s, r = _gen(seed), _dtype(case), _sizes(case), _sizes(case, "rank")
    core = _randn(g, *r, dtype=dt)
    f = []
    for m, (n, k) in enumerate(zip(s, r)):
        fall = (0.1 ** (torch.arange(k, device=DEV, dtype=dt) / k)).reshape([-1 if i == m else 1 for i in range(len(s))])
        core = core * fall
        f.append(_orthonormal(g, n, k, dt))
    x = core
    for m, a in enumerate(f):
        x = _times(x, a, m)
    return _noisy(x.contiguous(), g, 0.3), f


def _batched_data(case, seed):
    """[(tensor on the host, rank)]: factor columns with pairwise cosines near 0.8, 10 % noise."""
    sizes, rs = np.random.RandomState(int(case["problems"])), np.random.RandomState(seed)
    out = []
    for _ in range(int(case["problems"])):
        s, r = sizes.randint(8, 65, 3), int(sizes.randint(2, 17))
        f = []
        for n in s:
            a = 2.0 * rs.standard_normal((n, 1)) + rs.standard_normal((n, r))
            f.append((a / np.linalg.norm(a, axis=0)).astype(np.float32))
        x = f[0] @ (f[1][:, None, :] * f[2][None, :, :]).reshape(-1, r).T
        e = rs.standard_normal(x.shape).astype(np.float32) if x.size < 4096 else rs.rand(*x.shape).astype(np.float32) - 0.5
        x += np.float32(0.1 * np.linalg.norm(x) / np.linalg.norm(e)) * e
        out.append((x.reshape(s), r))
    return out


def _coo_data(case, seed):
    """(coords, values, factors): distinct random coordinates, heavier towards the low indices of each mode."""
    g, dt, s, nnz = _gen(seed), _dtype(case), _sizes(case), int(case["nnz"])
    coords = torch.stack([(n * _rand(g, nnz) ** 2).long().clamp_(max=n - 1) for n in s])
    values = 1.0 + _rand(g, nnz, dtype=dt)
    return coords, values, [_randn(g, n, int(case["rank"]), dtype=dt) for n in s]


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": dict(case), "kind": kind}
    if kind in ("mttkrp", "cp_grad", "parafac", "hals"):
        x, near = _cp_data(case, seed)
        state.update(x=x, factors=near)
    elif kind in ("project", "tucker"):
        x, f = _tucker_data(case, seed)
        state.update(x=x, factors=f)
    elif kind == "batched":
        problems = _batched_data(case, seed)
        b = BatchedCP([p[0] for p in problems], [p[1] for p in problems])
        state.update(batch=b, f0=b.random_init(seed % 100000))
    else:
        coords, values, f = _coo_data(case, seed)
        state.update(coords=coords, values=values, factors=f)
    return state


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "mttkrp":
        with tla.precision(case["precision"]):
            return [tla.unfolding_dot_khatri_rao(state["x"], (None, state["factors"]), m)
                    for m in range(state["x"].dim())]
    if kind == "cp_grad":
        return tla.cp_lstsq_grad((None, state["factors"]), state["x"])[1]
    if kind == "project":
        core = tla.multi_mode_dot(state["x"], state["factors"], transpose=True)
        return core, tla.tucker_to_tensor((core, state["factors"]))
    if kind == "tucker":
        (core, factors), errors = tla.tucker(state["x"], _sizes(case, "rank"), n_iter_max=case["sweeps"], tol=0,
                                             return_errors=True)
        return core, factors, errors
    if kind == "parafac":
        init = "svd" if case["init"] == "svd" else (None, state["factors"])
        (weights, factors), errors = tla.parafac(state["x"], case["rank"], n_iter_max=case["sweeps"], init=init,
                                                 tol=0, return_errors=True, precision=case["precision"],
                                                 dimtree=case["dimtree"])
        return weights, factors, errors
    if kind == "hals":
        (weights, factors), errors = tla.non_negative_parafac_hals(state["x"], case["rank"],
                                                                   init=(None, state["factors"]),
                                                                   n_iter_max=case["sweeps"], tol=1e-12,
                                                                   return_errors=True)
        return weights, factors, errors
    if kind == "batched":
        f, out = state["batch"].run(state["f0"], policy="plain", max_sweeps=case["sweeps"], tol=0.0)
        return f, out["error"], out["sweeps"], out["status"]
    s = _sizes(case)
    return [unfolding_dot_khatri_rao_coo(state["coords"], state["values"], s, (None, state["factors"]), m)
            for m in range(len(s))]


def work(case):
    """Bytes and operations of the calls of one pass, each call's inputs and outputs once."""
    kind = case["kind"]
    if kind == "batched":
        n = int(case["problems"])
        # sizes U{8..64}^3 and ranks U{2..16} in the mean; a sweep needs the tensor for each of the three modes
        cells, rank = 36.0 ** 3, 9.0
        return {"bytes": n * (4 * cells + 2 * 4 * 3 * 36 * rank), "flops": n * case["sweeps"] * 6 * cells * rank}
    s = _sizes(case)
    size = 8 if case["dtype"] == "float64" else 4
    cells = float(math.prod(s))
    if kind == "coo":
        r, nd, nnz = case["rank"], len(s), float(case["nnz"])
        return {"bytes": nd * (nnz * (8 * nd + size) + size * r * sum(s)), "flops": nd * nnz * r * (nd + 1)}
    if kind in ("project", "tucker"):
        r = _sizes(case, "rank")
        flops, left = 0.0, cells
        for n, k in zip(s, r):  # the chain to the core
            flops += 2 * left * k
            left = left / n * k
        if kind == "project":
            return {"bytes": size * (2 * cells + 2 * left), "flops": 2 * flops}
        return {"bytes": size * (cells + left + sum(a * b for a, b in zip(s, r))), "flops": flops * case["sweeps"]}
    r = case["rank"]
    small = size * r * sum(s)
    one = 2 * cells * r
    if kind == "mttkrp":
        return {"bytes": len(s) * (size * cells + small), "flops": len(s) * one}
    if kind == "cp_grad":
        return {"bytes": size * cells + 2 * small, "flops": len(s) * one}
    return {"bytes": size * cells + 2 * small, "flops": case["sweeps"] * len(s) * one}


# --------------------------------------------------------------------------
# The same results in 64 bits from plain torch and numpy.
def _unfold(x, m):
    return torch.movedim(x, m, 0).reshape(x.shape[m], -1)


def _times(x, a, m):
    """a applied to mode m of x."""
    y = a @ _unfold(x, m)
    rest = [n for i, n in enumerate(x.shape) if i != m]
    return torch.movedim(y.reshape([a.shape[0]] + rest), 0, m)


def _mttkrp(x, f, m):
    return _unfold(x, m) @ _kr([a for i, a in enumerate(f) if i != m])


def _hadamard(f, m):
    v = torch.ones((f[0].shape[1],) * 2, dtype=torch.float64, device=f[0].device)
    for i, a in enumerate(f):
        if i != m:
            v = v * (a.T @ a)
    return v


def _error(x, f, last):
    nx = torch.sum(x * x)
    return float(torch.sqrt(torch.abs(nx + torch.sum(_hadamard(f, -1)) - 2 * torch.sum(last * f[-1])) / nx))


def _left(x, m, k):
    """Leading left singular vectors and values of unfolding m, the largest entry of each vector positive."""
    u = _unfold(x, m)
    val, vec = np.linalg.eigh((u @ u.T).cpu().numpy())
    vec, val = vec[:, ::-1][:, :k], np.sqrt(np.maximum(val[::-1][:k], 0))
    sign = np.sign(vec[np.argmax(np.abs(vec), axis=0), np.arange(vec.shape[1])])
    return torch.tensor(vec * sign, device=DEV), torch.tensor(val.copy(), device=DEV)


def _als(x, f, sweeps):
    f, errors = list(f), []
    for _ in range(sweeps):
        for m in range(len(f)):
            last = _mttkrp(x, f, m)
            f[m] = torch.linalg.solve(_hadamard(f, m).cpu(), last.T.cpu()).T.contiguous().to(DEV)
        errors.append(_error(x, f, last))
    return f, errors


def _hals(x, f, sweeps):
    f, errors = [a.cpu() for a in f], []
    for _ in range(sweeps):
        for m in range(len(f)):
            last = _mttkrp(x, [a.to(DEV) for a in f], m).cpu()
            b, a, v = last.numpy().T, _hadamard(f, m).numpy(), f[m].numpy().T.copy()
            first = None
            for _ in range(100):
                moved = 0.0
                for k in range(a.shape[0]):
                    new = np.maximum((b[k] - a[k] @ v + a[k, k] * v[k]) / a[k, k], 0.0)
                    moved += float(np.sum((v - new) ** 2))
                    v[k] = new
                first = moved if first is None else first
                if moved < 1e-8 * first:
                    break
            f[m] = torch.tensor(v.T.copy())
        errors.append(_error(x, [a.to(DEV) for a in f], last.to(DEV)))
    return f, errors


def _als_small(x, f, sweeps):
    x, f = x.astype(np.float64), list(f)
    s, r = x.shape, f[0].shape[1]
    for _ in range(sweeps):
        for m in range(3):
            a, b = [f[i] for i in range(3) if i != m]
            last = np.moveaxis(x, m, 0).reshape(s[m], -1) @ (a[:, None, :] * b[None, :, :]).reshape(-1, r)
            f[m] = np.linalg.solve((a.T @ a) * (b.T @ b), last.T).T
    nx = np.sum(x * x)
    nm = np.sum((f[0].T @ f[0]) * (f[1].T @ f[1]) * (f[2].T @ f[2]))
    return f, math.sqrt(abs(nx + nm - 2 * np.sum(last * f[2])) / nx)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mttkrp", "cp_grad", "parafac", "hals"):
        x, near = _cp_data(case, seed)
        x, f = x.double(), [a.double() for a in near]
        if kind == "mttkrp":
            return [_mttkrp(x, f, m) for m in range(len(f))]
        if kind == "cp_grad":
            return [f[m] @ _hadamard(f, m) - _mttkrp(x, f, m) for m in range(len(f))]
        r = int(case["rank"])
        ones = torch.ones(r, dtype=torch.float64)
        if kind == "hals":
            return (ones,) + tuple(_hals(x, f, case["sweeps"]))
        if case["init"] == "svd":
            f = []
            for m in range(x.dim()):
                u, s = _left(x, m, r)
                f.append(u * s if m == 0 else u)
        return (ones,) + tuple(_als(x, f, case["sweeps"]))
    if kind in ("project", "tucker"):
        x, f = _tucker_data(case, seed)
        x, f = x.double(), [a.double() for a in f]
        errors = []
        if kind == "tucker":
            ranks, nx = _sizes(case, "rank"), float(torch.sum(x * x))
            f = [_left(x, m, k)[0] for m, k in enumerate(ranks)]
            for _ in range(case["sweeps"]):
                for m, k in enumerate(ranks):
                    y = x
                    for i, a in enumerate(f):
                        y = _times(y, a.T, i) if i != m else y
                    f[m] = _left(y, m, k)[0]
                errors.append(math.sqrt(abs(nx - float(torch.sum(_times(y, f[-1].T, x.dim() - 1) ** 2))) / nx))
        core = x
        for i, a in enumerate(f):
            core = _times(core, a.T, i)
        if kind == "tucker":
            return core.contiguous(), f, errors
        y = core
        for i, a in enumerate(f):
            y = _times(y, a, i)
        return core.contiguous(), y.contiguous()
    if kind == "batched":
        every, errors = [], []
        for p, (x, r) in enumerate(_batched_data(case, seed)):
            rs = np.random.RandomState(seed % 100000 + p)
            f0 = [rs.random_sample((n, r)).astype(np.float32).astype(np.float64) for n in x.shape]
            f, e = _als_small(x, f0, case["sweeps"])
            every += [a.reshape(-1) for a in f]
            errors.append(e)
        return np.concatenate(every), np.array(errors), None, None
    coords, values, f = _coo_data(case, seed)
    out = []
    for m, n in enumerate(_sizes(case)):
        t = values.double()[:, None]
        for i, a in enumerate(f):
            t = t * a.double()[coords[i]] if i != m else t
        out.append(torch.zeros((n, t.shape[1]), dtype=torch.float64, device=DEV).index_add_(0, coords[m], t))
    return out
