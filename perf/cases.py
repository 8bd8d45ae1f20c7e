"""The calls whose speed on the device is tracked, with their inputs, least work and tolerances.

Each case is one pass through the public entry points of rnp2_amd: QR::Factor, MultQ and
GenerateQ on device matrices, the least-squares drivers, the batched form, the request
server and LU.  Everything is seeded; matrices are column-major on the device except for
the server, which takes host arrays.  A factorization works in place, so a pass starts
from the program's own matrix with a device copy into the buffer that is factored.
"""
import ctypes
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import rnp2_amd as R

DT = {"d": torch.float64, "z": torch.complex128}

# What a program keeps for its whole life: one handle (or one server), whatever it solves.
_kept = {}


def _handle():
    if "handle" not in _kept:
        _kept["handle"] = R.Handle()
        _kept["stream"] = torch.cuda.ExternalStream(_kept["handle"].stream)
    return _kept["handle"], _kept["stream"]


def _server():
    if "server" not in _kept:
        _kept["server"] = R.Server(hbm_budget=64 << 30, workers=4, mode=1, max_iter=30, tol=1e-13)
    return _kept["server"]


def listed():
    return [
        # The smallest call of an application: factor a 512 x 256 block and form its Q.
        # The matrix is small enough that launches and dependent latency are all of it.
        {"name": "factor_q_512x256", "op": "factor_q", "dtype": "d", "m": 512, "n": 256},
        # An ordinary, ragged design matrix: neither size a multiple of any tile.
        {"name": "factor_1931x1207", "op": "factor", "dtype": "d", "m": 1931, "n": 1207},
        # The headline: a large square factorization.
        {"name": "factor_8192", "op": "factor", "dtype": "d", "m": 8192, "n": 8192},
        # A tall factorization: many rows per panel.
        {"name": "factor_32768x4096", "op": "factor", "dtype": "d", "m": 32768, "n": 4096},
        # The complex headline.
        {"name": "factor_z4096", "op": "factor", "dtype": "z", "m": 4096, "n": 4096},
        # Applying a stored Q^H to a block of vectors; odd sizes.
        {"name": "multq_6001x1500", "op": "multq", "dtype": "d", "m": 6001, "n": 1999, "k": 1500,
         "side": "L", "trans": "C"},
        # Forming the thin Q of a tall factorization (an orthonormal basis).
        {"name": "generateq_8192x2048", "op": "generateq", "dtype": "d", "m": 8192, "n": 2048, "k": 2048},
        # One right-hand side of an ill-conditioned least-squares problem, FP64 and refined mixed precision.
        {"name": "ls_16384x2048", "op": "ls", "dtype": "d", "m": 16384, "n": 2048, "nrhs": 1, "cond": 1e6},
        {"name": "mixed_ls_16384x2048", "op": "mixed", "dtype": "d", "m": 16384, "n": 2048, "nrhs": 1, "cond": 1e6},
        # Thousands of small uneven least-squares problems in one replayed plan.
        {"name": "batched_10k", "op": "batched", "dtype": "d", "count": 10000, "most": 256, "mix": 0, "plan": True},
        # A burst of least-squares requests of very different sizes through the server.
        {"name": "serve_24", "op": "serve", "dtype": "d", "count": 24, "most": 8192, "mix": 5, "cond": 1e6},
        # A square solver: LU with partial pivoting and a solve with 16 right-hand sides.
        {"name": "lu_solve_8192", "op": "lu", "dtype": "d", "n": 8192, "nrhs": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: every operation, both types, sizes from small to the listed largest."""
    while True:
        op = rng.choice(["factor", "factor", "factor", "factor_q", "multq", "generateq", "ls", "mixed", "batched",
                         "serve", "lu"])
        dt = rng.choice("ddz") if op not in ("mixed", "serve") else "d"
        c = {"op": op, "dtype": dt}
        if op in ("factor", "factor_q", "multq", "generateq"):
            c["m"], c["n"] = _log(rng, 64, 32768), _log(rng, 32, 8192)
            if op in ("factor_q", "generateq") and c["n"] > c["m"]:
                c["m"], c["n"] = c["n"], c["m"]
            if op == "generateq":
                c["k"] = rng.randint(max(1, c["n"] // 2), c["n"])
            if op == "multq":
                c["side"], c["trans"] = rng.choice("LR"), rng.choice("NC")
                q = c["m"] if c["side"] == "L" else c["n"]
                c["k"] = rng.randint(max(1, q // 8), max(1, q // 2))
            if c["m"] * c["n"] > 2 ** 27:
                continue
        elif op in ("ls", "mixed"):
            c["m"] = _log(rng, 128, 16384)
            c["n"] = rng.randint(max(16, c["m"] // 8), c["m"] // 2)
            c["nrhs"], c["cond"] = rng.randint(1, 16), 10.0 ** rng.uniform(2, 6)
        elif op == "batched":
            c.update(count=_log(rng, 100, 10000), most=_log(rng, 48, 256), mix=rng.randint(1, 10 ** 6),
                     plan=rng.random() < 0.5)
            if dt == "z":
                c["count"] = max(100, c["count"] // 2)
        elif op == "serve":
            c.update(count=rng.randint(4, 40), most=_log(rng, 512, 4096), mix=rng.randint(1, 10 ** 6),
                     cond=10.0 ** rng.uniform(3, 6))
        else:
            c["n"], c["nrhs"] = _log(rng, 96, 8192 if dt == "d" else 4096), rng.randint(1, 16)
        # no more than the largest listed factorization; LU's panels are slower, and its largest is listed
        if work(c)["flops"] <= 1.05e12 / (2.5 if dt == "z" else 1) / (2 if op in ("ls", "mixed") else 1):
            return c


# -- inputs ------------------------------------------------------------------------------

def _gen(seed, salt=0):
    return torch.Generator("cuda").manual_seed(int(seed) * 1000003 + salt)


def _gauss(m, n, dt, g):
    """Column-major m x n, entries (or real and imaginary parts) N(0,1)."""
    a = R.colmajor_empty(m, n, DT[dt])
    a.t().copy_(torch.randn((n, m), dtype=DT[dt], device="cuda", generator=g))
    if dt == "z":
        a.mul_(math.sqrt(2.0))
    return a


def _conditioned(m, n, dt, cond, g):
    """G diag(s) V with G Gaussian / sqrt(m), s log-spaced from 1 to 1/cond and V orthogonal (a signed
    Hartley matrix), so the condition number is about cond and no column is aligned with a singular vector."""
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    ang = (i[:, None] * i[None, :]).remainder_(n).mul_(2 * math.pi / n)
    v = ang.cos().add_(ang.sin()).div_(math.sqrt(n))
    v *= torch.randint(0, 2, (n,), device="cuda", generator=g) * 2.0 - 1.0
    s = torch.logspace(0, -math.log10(cond), n, dtype=torch.float64, device="cuda") / math.sqrt(m)
    a = R.colmajor_empty(m, n, DT[dt])
    a.copy_((_gauss(m, n, dt, g) * s) @ v.to(DT[dt]))
    return a


def _ls_input(m, n, nrhs, dt, cond, g):
    a = _conditioned(m, n, dt, cond, g)
    b = R.colmajor_empty(m, nrhs, DT[dt])
    b.copy_(a @ _gauss(n, nrhs, dt, g) + 1e-8 * _gauss(m, nrhs, dt, g))
    return a, b


def _reflectors(q, k, dt, g):
    """A stored factorization of order q with k reflectors: V below the diagonal with columns of norm just
    below one (as in the factorization of a Gaussian matrix), junk (R) above, tau = 2 / (v^H v)."""
    a = _gauss(q, k, dt, g)
    low = a.tril(-1)
    nrm = low.abs().square().sum(0).sqrt()
    want = torch.where(nrm > 0, 0.98, 0.0)
    low *= (want / nrm.clamp_min(1e-30))
    tau = (2.0 / (1.0 + want.square())).to(DT[dt])
    a.copy_(low + a.triu())
    return a, tau


def _shapes(count, most, mix):
    """m log-uniform in [16, most], n uniform in [8, m]."""
    rng = np.random.default_rng(mix)
    m = np.rint(np.exp(rng.uniform(math.log(16), math.log(most), count))).astype(int)
    n = np.array([rng.integers(8, mm + 1) for mm in m])
    return list(zip(m.tolist(), n.tolist()))


def _requests(case):
    """m log-uniform in [64, most], n uniform in [m/8, m/2], 1 to 16 right-hand sides, condition number
    log-uniform in [1e2, cond]."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["count"]):
        m = int(np.rint(np.exp(rng.uniform(math.log(64), math.log(case["most"])))))
        n = int(rng.integers(max(1, m // 8), max(2, m // 2) + 1))
        out.append((m, n, int(rng.integers(1, 17)),
                    float(np.exp(rng.uniform(math.log(1e2), math.log(case["cond"]))))))
    return out


def _inputs(case, seed):
    """What the program starts from, on the device."""
    op, dt, g = case["op"], case["dtype"], _gen(seed)
    if op in ("factor", "factor_q"):
        return {"a": _gauss(case["m"], case["n"], dt, g)}
    if op == "multq":
        q = case["m"] if case["side"] == "L" else case["n"]
        a, tau = _reflectors(q, case["k"], dt, g)
        return {"a": a, "tau": tau, "c": _gauss(case["m"], case["n"], dt, g)}
    if op == "generateq":
        a, tau = _reflectors(case["m"], case["k"], dt, g)
        full = _gauss(case["m"], case["n"], dt, g)
        full[:, :case["k"]].copy_(a)
        return {"a": full, "tau": tau}
    if op in ("ls", "mixed"):
        a, b = _ls_input(case["m"], case["n"], case["nrhs"], dt, case["cond"], g)
        return {"a": a, "b": b}
    if op == "batched":
        desc, na, nt, nb = R.make_batch(_shapes(case["count"], case["most"], case["mix"]), nrhs=1)
        mk = lambda k: torch.randn(k, dtype=DT[dt], device="cuda", generator=g)
        return {"desc": desc, "nt": nt, "a": mk(na), "b": mk(nb)}
    if op == "serve":
        return {"reqs": [_ls_input(m, n, q, dt, cond, _gen(seed, 1 + i))
                         for i, (m, n, q, cond) in enumerate(_requests(case))]}
    if op == "lu":
        return {"a": _gauss(case["n"], case["n"], dt, g), "b": _gauss(case["n"], case["nrhs"], dt, g)}
    raise ValueError(op)


def _host(t):
    """A device matrix as a column-major host array."""
    return t.t().contiguous().cpu().numpy().T


def prepare(case, seed):
    op = case["op"]
    s = dict(_inputs(case, seed), op=op, case=dict(case))
    if op == "serve":
        s["srv"] = _server()
        s["reqs"] = [(_host(a), _host(b)) for a, b in s["reqs"]]
        return s
    s["h"], s["stream"] = _handle()
    dt = DT[case["dtype"]]
    like = lambda t: R.colmajor_empty(*t.shape, t.dtype) if t.dim() == 2 else torch.empty_like(t)
    if op in ("factor", "factor_q"):
        s["wa"] = like(s["a"])
        s["wtau"] = torch.empty(min(s["a"].shape), dtype=dt, device="cuda")
        if op == "factor_q":
            s["wq"] = like(s["a"])
    elif op == "multq":
        s["wc"] = like(s["c"])
    elif op == "generateq":
        s["wa"] = like(s["a"])
    elif op in ("ls", "mixed"):
        if op == "ls":
            s["wa"], s["wb"] = like(s["a"]), like(s["b"])
            s["wtau"] = torch.empty(case["n"], dtype=dt, device="cuda")
        else:
            s["wx"] = R.colmajor_empty(case["n"], case["nrhs"], dt)
    elif op == "batched":
        s["wa"], s["wb"] = like(s["a"]), like(s["b"])
        s["wtau"] = torch.empty(s["nt"], dtype=dt, device="cuda")
        if case["plan"]:
            s["plan"] = s["h"].batched_plan(s["desc"], s["wa"], s["wtau"], s["wb"])
    elif op == "lu":
        s["wa"], s["wb"] = like(s["a"]), like(s["b"])
        s["piv"] = np.zeros(case["n"], dtype=np.uint64)
    torch.cuda.synchronize()
    return s


# -- one pass ----------------------------------------------------------------------------

def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def run(s):
    op = s["op"]
    if op == "serve":
        ids = [s["srv"].submit(a, b)[1] for a, b in s["reqs"]]
        xs = []
        for rid in ids:
            xs.append(s["srv"].poll(rid)[0])
            s["srv"].release(rid)
        return xs
    h, stream = s["h"], s["stream"]
    if op == "factor":
        with torch.cuda.stream(stream):
            s["wa"].copy_(s["a"])
        h.geqrf(s["wa"], s["wtau"])
        return [s["wa"], s["wtau"]]
    if op == "factor_q":
        with torch.cuda.stream(stream):
            s["wa"].copy_(s["a"])
            h.geqrf(s["wa"], s["wtau"])
            s["wq"].copy_(s["wa"])
        h.orgqr(s["wq"], s["wtau"])
        return [s["wa"], s["wtau"], s["wq"]]
    if op == "multq":
        with torch.cuda.stream(stream):
            s["wc"].copy_(s["c"])
        h.ormqr(s["case"]["side"], s["case"]["trans"], s["a"], s["tau"], s["wc"])
        return [s["wc"]]
    if op == "generateq":
        with torch.cuda.stream(stream):
            s["wa"].copy_(s["a"])
        h.orgqr(s["wa"], s["tau"])
        return [s["wa"]]
    if op == "ls":
        with torch.cuda.stream(stream):
            s["wa"].copy_(s["a"])
            s["wb"].copy_(s["b"])
        h.gels(s["wa"], s["wtau"], s["wb"])
        return [s["wa"], s["wtau"], s["wb"]]
    if op == "mixed":
        h.gels_mixed(s["a"], s["b"], s["wx"], max_iter=30, tol=1e-13)
        return [s["wx"]]
    if op == "batched":
        with torch.cuda.stream(stream):
            s["wa"].copy_(s["a"])
            s["wb"].copy_(s["b"])
        if "plan" in s:
            s["plan"].run()
        else:
            h.geqrf_batched(s["desc"], s["wa"], s["wtau"], s["wb"])
        return [s["wa"], s["wtau"], s["wb"]]
    # LU goes through the drop-in C entry points with device matrices and host pivots; they order
    # nothing against torch's stream, so the copies are waited for.
    n, L, pre = s["case"]["n"], R.lib(), s["case"]["dtype"]
    s["wa"].copy_(s["a"])
    s["wb"].copy_(s["b"])
    torch.cuda.current_stream().synchronize()
    piv = s["piv"].ctypes.data_as(ctypes.c_void_p)
    info = getattr(L, f"rnpx_{pre}getrf")(n, n, _p(s["wa"]), n, piv)
    st = getattr(L, f"rnpx_{pre}getrs")(b"N", n, s["case"]["nrhs"], _p(s["wa"]), n, piv, _p(s["wb"]), n)
    if info < 0 or st != 0:
        raise RuntimeError(f"LU failed: {info}, {st}")
    return [s["wa"], s["piv"].view(np.int64), s["wb"]]


# -- least work --------------------------------------------------------------------------

def _qr_flops(m, n):
    k = min(m, n)
    return 4.0 * m * n * k - 2.0 * (m + n) * k * k + 4.0 * k ** 3 / 3.0


def _ls_work(m, n, q):
    """Factor, Q^H b, the triangular solve; A and b in, x out."""
    return _qr_flops(m, n) + q * (4.0 * m * n - n * n), 8.0 * (m * n + m * q + n * q)


def work(case):
    """Elements read once and written once (the factors are an output), and the operations of the
    algorithm; a complex element is 16 bytes and a complex operation four real ones."""
    op, z = case["op"], case["dtype"] == "z"
    if op in ("factor", "factor_q"):
        m, n = case["m"], case["n"]
        by, fl = 8.0 * 2 * m * n, _qr_flops(m, n)
        if op == "factor_q":
            by, fl = by + 8.0 * m * n, 2 * fl
    elif op == "multq":
        m, n, k = case["m"], case["n"], case["k"]
        q, r = (m, n) if case["side"] == "L" else (n, m)
        by, fl = 8.0 * (q * k + 2 * m * n), 2.0 * r * k * (2 * q - k)
    elif op == "generateq":
        m, n, k = case["m"], case["n"], case["k"]
        by, fl = 8.0 * (m * k + m * n), 4.0 * m * n * k - 2.0 * (m + n) * k * k + 4.0 * k ** 3 / 3.0
    elif op in ("ls", "mixed"):
        fl, by = _ls_work(case["m"], case["n"], case["nrhs"])
        if op == "ls":
            by += 8.0 * case["m"] * case["n"]  # the factors are handed back
    elif op == "batched":
        by = fl = 0.0
        for m, n in _shapes(case["count"], case["most"], case["mix"]):
            f, b = _ls_work(m, n, 1)
            fl, by = fl + f, by + b + 8.0 * m * n
    elif op == "serve":
        by = fl = 0.0
        for m, n, q, _ in _requests(case):
            f, b = _ls_work(m, n, q)
            fl, by = fl + f, by + b
    else:
        n, q = case["n"], case["nrhs"]
        by, fl = 8.0 * (2 * n * n + 2 * n * q), 2.0 * n ** 3 / 3.0 + 2.0 * n * n * q
    return {"bytes": by * (2 if z else 1), "flops": fl * (4 if z else 1)}


def tolerance(case):
    """About four times what another order of the FP64 sums shows; solutions carry the condition number."""
    op = case["op"]
    if op in ("ls", "mixed", "serve"):
        r = 1e-15 * max(case["cond"], 1e3)
        return {"rel": r, "max": min(0.5, 20 * r)}
    if op == "batched":
        # nearly square random problems: the worst of thousands of condition numbers decides
        return {"rel": 1e-10, "max": 1e-9}
    if op == "lu":
        return {"rel": 1e-10, "max": 1e-9, "differ": 0.0}
    return {"rel": 4e-14, "max": 2e-11}


# -- the same in plain torch -------------------------------------------------------------

def _cpu_qr(a):
    """LAPACK's factorization.  The last row of a complex matrix with m <= n has a reflector of length one
    (it makes R's diagonal real); MKL leaves it out of its blocked loop, so it is applied here if need be."""
    fac, tau = torch.geqrf(a)
    i = a.shape[0] - 1
    if a.is_complex() and a.shape[0] <= a.shape[1] and tau[i] == 0 and fac[i, i].imag != 0:
        beta = -torch.sign(fac[i, i].real) * fac[i, i].abs()
        tau[i] = (beta - fac[i, i]) / beta
        fac[i, i + 1:] *= 1 - tau[i].conj()
        fac[i, i] = beta
    return fac, tau


def _cpu_ls(a, b):
    fac, tau = _cpu_qr(a)
    n = a.shape[1]
    y = torch.ormqr(fac, tau, b, True, True)
    x = torch.linalg.solve_triangular(fac[:n].triu(), y[:n], upper=True)
    y[:n] = x
    return fac, tau, y


def exact(case, seed):
    op = case["op"]
    if work(case)["flops"] > 8e11:
        return None
    i = _inputs(case, seed)
    c = lambda t: t.cpu()
    if op in ("factor", "factor_q"):
        fac, tau = _cpu_qr(c(i["a"]))
        return [fac, tau] + ([torch.linalg.householder_product(fac, tau)] if op == "factor_q" else [])
    if op == "multq":
        return [torch.ormqr(c(i["a"]), c(i["tau"]), c(i["c"]), case["side"] == "L", case["trans"] == "C")]
    if op == "generateq":
        return [torch.linalg.householder_product(c(i["a"]), c(i["tau"]))]
    if op == "ls":
        return list(_cpu_ls(c(i["a"]), c(i["b"])))
    if op == "mixed":
        return [_cpu_ls(c(i["a"]), c(i["b"]))[2][:case["n"]]]
    if op == "serve":
        return [_cpu_ls(c(a), c(b))[2][:a.shape[1]] for a, b in i["reqs"]]
    if op == "batched":
        a, b = c(i["a"]), c(i["b"])
        oa, ot, ob = torch.empty_like(a), torch.empty(i["nt"], dtype=a.dtype), torch.empty_like(b)
        threads = torch.get_num_threads()

        def one(d):
            m, n, ao, to, bo = (int(d[f]) for f in ("m", "n", "a_off", "tau_off", "b_off"))
            fac, tau, y = _cpu_ls(a[ao:ao + m * n].view(n, m).t(), b[bo:bo + m].view(1, m).t())
            oa[ao:ao + m * n].view(n, m).t().copy_(fac)
            ot[to:to + n] = tau
            ob[bo:bo + m] = y[:, 0]

        torch.set_num_threads(1)
        try:
            with ThreadPoolExecutor(8) as pool:
                list(pool.map(one, i["desc"]))
        finally:
            torch.set_num_threads(threads)
        return [oa, ot, ob]
    a, b = c(i["a"]), c(i["b"])
    lu, piv = torch.linalg.lu_factor(a)
    return [lu, (piv.to(torch.int64) - 1), torch.linalg.lu_solve(lu, piv, b)]
