"""Performance cases: the work a user of this library has it do, through its public entry points.

``listed()`` names the cases, ``draw()`` gives further ones of the same ranges, ``prepare()`` makes what a program
holds before the call, ``run()`` is one pass, ``work()`` the bytes and operations that a pass cannot do without and
``exact()`` the FP64 answer from plain torch.

Matrices follow the benchmark's own distributions.  Unpivoted paths: U[-0.5, 0.5) off the diagonal and a dominant
diagonal (+ n, or d times the row sum).  Pivoted path: U[-0.5, 0.5) everywhere.  The matrix solved is the transpose of
the row-major buffer, as in the reference's LINPACK.
"""
import math
import random

import numpy as np
import torch

from hpcc_fpga_amd import Batch, Context, Server
from hpcc_fpga_amd.linpack import HplError, load_library


def listed():
    return [
        # The substitution alone on a caller's device memory and stream, allocating nothing: a serving loop's or a
        # captured graph's step, the smallest call there is.
        {"name": "noalloc_1024", "path": "noalloc", "n": 1024},
        # The benchmark executable's call on host buffers, at its documented size (-m 8 -b 7): upload, factorise,
        # factor back into the caller's matrix, then upload and solve.
        {"name": "host_fp32_1024", "path": "host", "n": 1024, "block": 128},
        # Repetitions on a resident system, as the benchmark's timed loop (the answer is x; the factor stays on the
        # device for further solves): an ordinary size with the default block ...
        {"name": "fp32_2048", "path": "fp32", "n": 2048, "block": 128},
        # ... an order that only a narrow block divides (-m 117 -b 6) ...
        {"name": "fp32_7488_b64", "path": "fp32", "n": 7488, "block": 64},
        # ... and the large plain FP32 run of bench.py.
        {"name": "fp32_32768", "path": "fp32", "n": 32768, "block": 256},
        # Mixed precision with FP64 refinement, bench.py's headline size.
        {"name": "bf16_ir_65536", "path": "refined", "n": 65536, "block": 256, "prec": "bf16", "method": "ir"},
        # The 8-bit update with GMRES refinement at a mid size.
        {"name": "fp8_gmres_6144", "path": "refined", "n": 6144, "block": 128, "prec": "fp8", "method": "gmres"},
        # Further right-hand sides with a factor that is already there, refined to FP64 accuracy.
        {"name": "rhs16_4096", "path": "rhs", "n": 4096, "block": 256, "prec": "bf16", "nrhs": 16},
        # Partial pivoting (--uniform), refined to FP64 accuracy.
        {"name": "pivoted_6144", "path": "pivoted", "n": 6144, "block": 128},
        # The benchmark built with DATA_TYPE=double.
        {"name": "fp64_8192", "path": "fp64", "n": 8192},
        # Thousands of small systems of uneven order in one solve (bench.py's batch), all solutions fetched.
        {"name": "batch_4096", "path": "batch", "count": 4096, "lo": 32, "hi": 1024, "mix": 7, "prec": "fp16"},
        # A burst of uneven requests to the serving engine with its defaults: new systems from host memory, a fifth of
        # the requests on factors that are kept resident.
        {"name": "serve_20", "path": "serve", "count": 20, "lo": 64, "hi": 4096, "mix": 11, "prec": "fp8"},
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def order(lo, hi, block):
        return max(1, round(log(lo, hi) / block)) * block

    path = rng.choice(["noalloc", "host", "fp32", "fp32", "refined", "refined", "rhs", "pivoted", "fp64", "batch",
                       "serve"])
    if path == "noalloc":
        return {"path": path, "n": order(128, 8192, 32)}
    if path == "host":
        block = rng.choice([32, 64, 128])
        return {"path": path, "n": order(256, 3072, block), "block": block}
    if path == "fp32":
        block = rng.choice([64, 128, 128, 256, 256, 512])
        return {"path": path, "n": order(max(512, block), 24576 if block >= 256 else 8192, block), "block": block}
    if path == "refined":
        block = rng.choice([64, 128, 256, 256])
        method = rng.choice(["ir", "ir", "gmres"])
        return {"path": path, "n": order(1024, 24576 if block >= 256 else 8192, block), "block": block,
                "prec": rng.choice(["bf16", "bf16", "fp16", "fp8"]), "method": method}
    if path == "rhs":
        block = rng.choice([64, 128, 256])
        return {"path": path, "n": order(512, 12288, block), "block": block,
                "prec": rng.choice(["fp32", "bf16", "fp8"]), "nrhs": rng.randint(1, 16)}
    if path == "pivoted":
        block = rng.choice([64, 128, 256])
        return {"path": path, "n": order(512, 6144, block), "block": block}
    if path == "fp64":
        return {"path": path, "n": order(512, 10240, 64)}
    if path == "batch":
        lo = rng.choice([16, 32, 100])
        return {"path": path, "count": round(log(16, 3000)), "lo": lo, "hi": rng.choice([200, 500, 1024]),
                "mix": rng.randrange(10 ** 6), "prec": rng.choice(["fp16", "fp16", "fp32"])}
    return {"path": path, "count": rng.randint(4, 24), "lo": 64, "hi": rng.choice([1024, 2048, 4096]),
            "mix": rng.randrange(10 ** 6), "prec": rng.choice(["fp8", "fp8", "bf16", "fp32"])}


# ---- inputs ------------------------------------------------------------------------------------------------------

def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(n, seed, dominant, dtype=torch.float32):
    """An n x n matrix on the GPU: U[-0.5, 0.5), with n added on the diagonal where `dominant`."""
    a = torch.rand(n, n, generator=_rng(seed), device="cuda", dtype=dtype) - 0.5
    if dominant:
        a.diagonal().add_(float(n))
    return a


def _vectors(n, count, seed):
    """`count` right-hand sides of order n, U[-1, 1) in FP64 (n x count)."""
    return np.random.default_rng([seed, 1]).uniform(-1.0, 1.0, (n, count))


def _factor(n, seed):
    """A factor in the library's encoding with the magnitudes of a diagonally dominant matrix's: multipliers
    and u entries of the size they have for U[-0.5, 0.5) + n on the diagonal."""
    m = torch.rand(n, n, generator=_rng(seed), device="cuda") - 0.5  # M(i, j) at [j, i]
    cols = torch.arange(n, device="cuda")
    low = cols[None, :] > cols[:, None]  # row index i of M above its column j
    m = torch.where(low, m / n, m)
    diag = n * (1.0 + 0.1 * (torch.rand(n, generator=_rng(seed + 1), device="cuda") - 0.5))
    m.diagonal().copy_(-1.0 / diag)
    return m.contiguous()


def _orders(case):
    r = random.Random(case["mix"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return [int(round(math.exp(r.uniform(lo, hi)))) for _ in range(case["count"])]


def _requests(case):
    """(order, right-hand sides, resident factor or None) of each request of a burst."""
    r = random.Random(case["mix"] + 1)
    kept = _orders({**case, "count": 4, "mix": case["mix"] + 2})
    out = []
    for n in _orders(case):
        k = r.randrange(len(kept)) if r.random() < 0.2 else None
        out.append((n if k is None else kept[k], r.randint(1, 16), k))
    return kept, out


def _serve_inputs(case, seed):
    kept, requests = _requests(case)
    ka = [_uniform(n, 1000 * seed + 500 + i, True).cpu().numpy() for i, n in enumerate(kept)]
    a = [None if k is not None else _uniform(n, 1000 * seed + i, True).cpu().numpy()
         for i, (n, _, k) in enumerate(requests)]
    b = [_vectors(n, nrhs, 1000 * seed + i) for i, (n, nrhs, _) in enumerate(requests)]
    return kept, requests, ka, a, b


class _State:
    """A prepared state: the case and what a program holds for it."""

    def __init__(self, case, **held):
        self.case = case
        self.__dict__.update(held)


def prepare(case, seed):
    path = case["path"]
    if path == "noalloc":
        n = case["n"]
        b = torch.from_numpy(_vectors(n, 1, seed)[:, 0].astype(np.float32)).cuda()
        return _State(case, lib=load_library(), lu=_factor(n, seed), b=b, x=torch.empty_like(b))
    if path == "serve":
        kept, requests, ka, a, b = _serve_inputs(case, seed)
        srv = Server(hbm_budget=24 * 10 ** 9, prec=case["prec"], max_n=case["hi"])
        handles = []
        for n, m in zip(kept, ka):
            t = srv.submit(np.ones(n), a=m, keep=True)
            handles.append(srv.wait(t)[1]["factor"])
        return _State(case, srv=srv, handles=handles, requests=requests, a=a, b=b)
    ctx = Context(0)
    if path == "batch":
        bt = Batch(ctx, _orders(case))
        bt.generate(seed)
        bt.autotune(case["prec"])
        return _State(case, ctx=ctx, batch=bt)
    n = case["n"]
    if path == "host":
        return _State(case, ctx=ctx, a=_uniform(n, seed, True).cpu().numpy(),
                        b=_vectors(n, 1, seed)[:, 0].astype(np.float32))
    if path == "fp64":
        a = _uniform(n, seed, True, torch.float64).cpu().numpy()
        ctx.upload_f64(a, _vectors(n, 1, seed)[:, 0].copy())
        return _State(case, ctx=ctx)
    ctx.keep_original(True)
    if path == "fp32":
        ctx.generate(n, mode=0, seed=seed)
    elif path == "refined":
        ctx.generate(n, mode=1, seed=seed, d=1.01)
    elif path == "rhs":
        ctx.upload(_uniform(n, seed, True).cpu().numpy())
        ctx.gefa_dev(case["block"], case["prec"])
        return _State(case, ctx=ctx, b=_vectors(n, case["nrhs"], seed))
    elif path == "pivoted":
        ctx.set_pivoting(True)
        ctx.upload(_uniform(n, seed, False).cpu().numpy())
        ctx.upload_rhs64(_vectors(n, 1, seed)[:, 0])
    else:
        raise HplError(1, f"unknown path {path}")
    return _State(case, ctx=ctx)


# ---- one pass ----------------------------------------------------------------------------------------------------

def run(s):
    case = s.case
    path = case["path"]
    if path == "noalloc":
        s.x.copy_(s.b)
        st = s.lib.hpl_gesl_noalloc(s.lu.data_ptr(), case["n"], case["n"], s.x.data_ptr(),
                                    torch.cuda.current_stream().cuda_stream)
        if st:
            raise HplError(st, "hpl_gesl_noalloc")
        return s.x
    if path == "serve":
        tickets = [s.srv.submit(b, a=a) if k is None else s.srv.submit(b, factor=s.handles[k])
                   for (_, _, k), a, b in zip(s.requests, s.a, s.b)]
        return [s.srv.wait(t)[0] for t in tickets]
    if path == "batch":
        s.batch.solve(case["prec"])
        return np.concatenate([s.batch.get(i)[0] for i in range(case["count"])])
    if path == "host":
        lu, x = s.a.copy(), s.b.copy()
        s.ctx.gefa(lu, case["block"])
        s.ctx.gesl(lu, x)
        return lu, x
    if path == "fp32":
        s.ctx.restore()
        s.ctx.gefa_dev(case["block"])
        s.ctx.gesl_dev()
        return s.ctx.download(matrix=False)[1]
    if path == "fp64":
        s.ctx.restore_f64()
        s.ctx.gefa_dev_f64()
        s.ctx.gesl_dev_f64()
        return s.ctx.download_f64(matrix=False)[1]
    if path == "refined":
        if case["method"] == "ir":
            s.ctx.solve_ir(case["block"], case["prec"])
        else:
            s.ctx.solve_gmres(case["block"], case["prec"])
        return s.ctx.download_solution64()
    if path == "rhs":
        return s.ctx.solve_rhs64(s.b)[0]
    # pivoted: to the accuracy of FP64, which the default tolerance does not ask for
    s.ctx.solve_ir(case["block"], "fp32", tol=1e-15)
    return s.ctx.download_solution64()


# ---- what a pass cannot do without -------------------------------------------------------------------------------

def _solve_work(n, nrhs=1, size=4, factor=True):
    flops = 2.0 * n * n * nrhs + (2.0 / 3.0 * n ** 3 if factor else 0.0)
    # the matrix read (and its factor written), right-hand sides and solutions
    return (2 if factor else 1) * size * float(n) * n + 16.0 * n * nrhs, flops


def work(case):
    path = case["path"]
    if path == "noalloc":
        parts = [_solve_work(case["n"], factor=False)]
    elif path == "rhs":  # the factor, and the original matrix for the residual
        n, nrhs = case["n"], case["nrhs"]
        parts = [(8.0 * n * n + 16.0 * n * nrhs, 4.0 * n * n * nrhs)]
    elif path == "fp64":
        parts = [_solve_work(case["n"], size=8)]
    elif path == "batch":
        parts = [_solve_work(n) for n in _orders(case)]
    elif path == "serve":
        parts = [_solve_work(n, nrhs, factor=k is None) for n, nrhs, k in _requests(case)[1]]
    else:
        parts = [_solve_work(case["n"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ---- the answers in 64 bits --------------------------------------------------------------------------------------

_MASK = (1 << 64) - 1


def _mix(z):
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
    return z ^ (z >> 31)


def _signed(v):
    return v - (1 << 64) if v >> 63 else v


def _counter_uniform(seed, stream, first, count):
    """The generator's U[0, 1) values first .. first + count - 1 (splitmix64's finaliser on a counter), FP64."""
    def shift(z, s):
        return (z >> s) & ((1 << (64 - s)) - 1)

    k = torch.arange(first + 1, first + count + 1, dtype=torch.int64, device="cuda")
    z = k * _signed(0x9E3779B97F4A7C15) + _signed(_mix(seed ^ (stream << 56)))
    z = (z ^ shift(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ shift(z, 27)) * _signed(0x94D049BB133111EB)
    z = z ^ shift(z, 31)
    return shift(z, 40).double() / 16777216.0


def _transposed_product(a, x):
    """a^T x in FP64, the rows of a taken in pieces."""
    out = torch.zeros(a.shape[1], x.shape[1], dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // a.shape[1])
    for r in range(0, a.shape[0], step):
        out += a[r:r + step].double().T.contiguous() @ x[r:r + step]
    return out


def _dominant_solve(a, b):
    """x with a^T x = b for a strongly dominant diagonal, by Jacobi's iteration in FP64 (it gains at least a factor
    of four a step here)."""
    b = b.cuda().double().reshape(a.shape[0], -1)
    d = a.diagonal().double()[:, None]
    x = b / d
    for _ in range(80):
        dx = (b - _transposed_product(a, x)) / d
        x += dx
        if float(dx.abs().max()) <= 1e-17 * float(x.abs().max()):
            break
    return x


def _eliminated(a):
    """LU without pivoting of a^T in the library's encoding, in FP64 on the host."""
    m = a.astype(np.float64)
    n = len(m)
    for k in range(n - 1):  # row k of the buffer is column k of the matrix
        m[k, k] = -1.0 / m[k, k]
        m[k, k + 1:] *= m[k, k]
        m[k + 1:, k + 1:] += m[k + 1:, k:k + 1] * m[k:k + 1, k + 1:]
    m[n - 1, n - 1] = -1.0 / m[n - 1, n - 1]
    return m


def _solved(case, seed):
    path = case["path"]
    n = case.get("n")
    if path == "noalloc":
        m = _factor(n, seed).double().T
        b = torch.from_numpy(_vectors(n, 1, seed)[:, 0].astype(np.float32)).cuda().double()[:, None]
        low = torch.eye(n, dtype=torch.float64, device="cuda") - torch.tril(m, -1)
        up = torch.triu(m, 1) + torch.diag(-1.0 / m.diagonal())
        y = torch.linalg.solve_triangular(low.contiguous(), b, upper=False)
        return torch.linalg.solve_triangular(up.contiguous(), y, upper=True)[:, 0]
    if path == "host":
        a = _uniform(n, seed, True)
        b = _vectors(n, 1, seed)[:, 0].astype(np.float32)
        lu = _eliminated(a.cpu().numpy()) if n <= 1536 else None
        return lu, _dominant_solve(a, torch.from_numpy(b))[:, 0]
    if path == "fp32":
        a = torch.empty(n, n, device="cuda")
        step = max(1, (1 << 26) // n)
        for r in range(0, n, step):
            m = min(step, n - r)
            a[r:r + m] = (_counter_uniform(seed, 0, r * n, m * n) - 0.5).reshape(m, n)
        a.diagonal().add_(float(n))
        ones = torch.ones(n, 1, dtype=torch.float64, device="cuda")
        return _dominant_solve(a, _transposed_product(a, ones).float())[:, 0]
    if path == "refined":  # b = M x_true in FP64
        return 2.0 * _counter_uniform(seed, 1, 0, n) - 1.0
    if path == "rhs":
        return _dominant_solve(_uniform(n, seed, True), torch.from_numpy(_vectors(n, case["nrhs"], seed)))
    if path == "pivoted":
        a = _uniform(n, seed, False).double().T.contiguous()
        b = torch.from_numpy(_vectors(n, 1, seed)).cuda()
        x = torch.linalg.solve(a, b)
        return (x + torch.linalg.solve(a, b - a @ x))[:, 0]
    if path == "fp64":
        a = _uniform(n, seed, True, torch.float64)
        return _dominant_solve(a, torch.from_numpy(_vectors(n, 1, seed)))[:, 0]
    if path == "batch":  # b = M 1 in FP64
        return np.ones(sum(_orders(case)))
    kept, requests, ka, a, b = _serve_inputs(case, seed)
    out = []
    for (_, nrhs, k), m, v in zip(requests, a, b):
        x = _dominant_solve(torch.from_numpy(ka[k] if k is not None else m).cuda(), torch.from_numpy(v))
        out.append(x[:, 0] if nrhs == 1 else x)
    return out


def exact(case, seed):
    return _solved(case, seed)
