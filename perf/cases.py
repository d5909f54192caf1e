"""The work that users of this framework have it do, as cases to time.

Every case goes through a public entry point: the Python module `diffrg_amd` (threshold_batch,
ft_batch, SEBatch, FlowServer, QuadratureProvider), or, for the drop-in C++ templates, the test
library that instantiates them with a user KERNEL (tests/native/libdfrg_kat.so, as bench.py does).
Sizes are those of the repository's workloads (diffrg_amd/workloads.py) and tests, and generic ones
around them: ensembles of fields, ragged Matsubara rules, single integrals.

A case is a dict of plain values; `listed()` names the measured ones, `draw(rng)` gives one more of
the same ranges, `prepare(case, seed)` is what a program holds before the call, `run(state)` is one
pass, `exact(case, seed)` is the same result from plain numpy or torch in 64 bits.
"""
import ctypes
import math
import os

import numpy as np
import torch

import diffrg_amd as D

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(D.__file__)))
MODES = {"fp64": D.FP64, "mixed": D.MIXED}
X_EXTENT, K = 20.0, 1.0
COORD = (1e-3, 40.0, 6.0)  # start, stop, bias of the dressing tables' logarithmic coordinates
TEMPS = (0.01, 0.05, 0.1, 0.2, 0.3)
FLOW = {"rho_max": 4.0, "N": 4.0, "m2_0": 0.2, "lam": 1.0}
FLOW_STEPS = 2000  # the server's default: RK4 from k = 1 to 1e-3


# ---------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # one field grid of an LPA potential: 256 threshold integrals, one call per flow step; the
        # smallest call, where the launch counts
        {"name": "threshold-grid-fp64", "kind": "threshold", "n": 256, "nx": 64, "d": 4, "mode": "fp64"},
        # the same integral over an ensemble of parameter sets times a field grid, odd size
        {"name": "threshold-ensemble-mixed", "kind": "threshold", "n": 131071, "nx": 64, "d": 3, "mode": "mixed"},
        # 512 external momenta of a finite-temperature two-propagator diagram, |n| <= 64 summed
        {"name": "finite-T-512-mixed", "kind": "finite_T", "n": 512, "nx": 48, "nm": 64, "ragged": False,
         "radial_mode": 1, "d": 4, "mode": "mixed"},
        # a full (p0, |p|) grid at several temperatures, each with a Matsubara rule of its own length
        {"name": "finite-T-grid-fp64", "kind": "finite_T", "n": 8191, "nx": 48, "nm": 96, "ragged": True,
         "radial_mode": 0, "d": 4, "mode": "fp64"},
        # one self-energy integral, asked for alone
        {"name": "selfenergy-1-fp64", "kind": "selfenergy", "n": 1, "nq": 64, "na": 32, "n_tab": 128, "mode": "fp64"},
        # a self-energy on a 64-point momentum grid (the headline workload), in both precisions
        {"name": "selfenergy-64-mixed", "kind": "selfenergy", "n": 64, "nq": 64, "na": 32, "n_tab": 128,
         "mode": "mixed"},
        {"name": "selfenergy-64-fp64", "kind": "selfenergy", "n": 64, "nq": 64, "na": 32, "n_tab": 128,
         "mode": "fp64"},
        # thousands of diagrams of uneven orders, each with a table of its own (the largest batch)
        {"name": "uneven-4096-mixed", "kind": "uneven", "n": 4096, "mode": "mixed"},
        # the same kind of batch at full precision, fewer diagrams
        {"name": "uneven-1023-fp64", "kind": "uneven", "n": 1023, "mode": "fp64"},
        # RG flows of O(4) potentials with grids of different sizes, submitted together and served
        # until the last has finished
        {"name": "flows-24", "kind": "flows", "n": 24, "min_grid": 64, "max_grid": 1024},
        # the quadrature rules of a run that begins, or whose temperature or RG scale has changed:
        # Gauss-Legendre orders and Matsubara rules at new (T, E)
        {"name": "rules", "kind": "rules", "n_gl": 3, "max_order": 128, "n_mats": 3},
        # the drop-in C++ template with a user KERNEL: table, integrator and one request per momentum
        {"name": "template-64", "kind": "template", "n": 64, "nq": 64, "na": 32, "n_tab": 128, "call": "request"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["threshold", "threshold", "finite_T", "finite_T", "selfenergy", "selfenergy", "uneven",
                       "flows", "rules", "template"])
    mode = rng.choice(["fp64", "mixed"])
    if kind == "threshold":
        return {"kind": kind, "n": _log(rng, 16, 131071), "nx": rng.randint(12, 128), "d": rng.choice([2, 3, 4, 5]),
                "mode": mode}
    if kind == "finite_T":
        return {"kind": kind, "n": _log(rng, 16, 8191), "nx": rng.randint(12, 96), "nm": rng.randint(8, 128),
                "ragged": rng.random() < 0.5, "radial_mode": rng.choice([0, 1]), "d": rng.choice([3, 4]), "mode": mode}
    if kind == "selfenergy":
        return {"kind": kind, "n": _log(rng, 1, 256), "nq": rng.randint(12, 128), "na": rng.choice([8, 16, 32, 64]),
                "n_tab": rng.randint(32, 256), "mode": mode}
    if kind == "uneven":
        return {"kind": kind, "n": _log(rng, 64, 1023), "mode": mode}
    if kind == "flows":
        lo = _log(rng, 16, 512)
        return {"kind": kind, "n": rng.randint(1, 16), "min_grid": lo, "max_grid": rng.randint(lo, 1024)}
    if kind == "rules":
        return {"kind": kind, "n_gl": rng.randint(1, 4), "max_order": _log(rng, 32, 512), "n_mats": rng.randint(1, 4)}
    return {"kind": kind, "n": _log(rng, 1, 128), "nq": rng.randint(12, 96), "na": rng.randint(6, 40),
            "n_tab": rng.randint(32, 256), "call": rng.choice(["request", "request", "get"])}


# -------------------------------------------------------------------------------------- their inputs

def _dressing(r, n):
    """A smooth dressing function Z in (0.5, 1.5): a random sum of four waves through tanh."""
    i = np.arange(n)
    xi = sum((2.0 * r.random() - 1.0) / m * np.sin(m * math.pi * i / (n - 1) + 2.0 * math.pi * r.random())
             for m in range(1, 5))
    return 1.0 + 0.5 * np.tanh(xi)


def _spread(first, last, n):
    """n whole numbers from first to last, a little off an even spacing so that they are not round."""
    v = np.linspace(first, last, n)
    off = 0.2 * abs(last - first) / max(1, n - 1)
    return np.clip(np.round(v - off * np.sin(1.0 + np.arange(n))), min(first, last), max(first, last)).astype(int)


def _momenta(r, n):
    """External momenta, log-uniform over the tables' range."""
    return np.exp(np.log(COORD[0]) + r.random(n) * math.log(COORD[1] / COORD[0]))


def _inputs(case, seed):
    """The case's input values on the host, from the seed alone."""
    r = np.random.default_rng([int(seed), 17])
    kind = case["kind"]
    if kind == "threshold":
        return {"m2": -0.8 + 4.8 * r.random(case["n"])}
    if kind == "finite_T":
        n = case["n"]
        t = r.integers(0, len(TEMPS), n)
        T = np.array(TEMPS)[t]
        nm = np.full(len(TEMPS), case["nm"])
        if case["ragged"]:  # fewer frequencies at higher temperature
            nm = np.maximum(4, (case["nm"] * np.minimum(1.0, 0.08 / np.array(TEMPS) + 0.1 * r.random(5))).astype(int))
        off = np.concatenate([[0], np.cumsum(nm)[:-1]])
        return {"T": T, "p0": 2.0 * math.pi * T * r.integers(0, 8, n), "pabs": 2.0 * r.random(n),
                "m1": -0.5 + 3.5 * r.random(n), "m2": -0.5 + 3.5 * r.random(n),
                "mx": np.concatenate([2.0 * math.pi * TEMPS[i] * np.arange(1, nm[i] + 1) for i in range(5)]),
                "mw": np.concatenate([np.full(nm[i], TEMPS[i]) for i in range(5)]),
                "m_off": off[t].astype(np.int32), "m_n": nm[t].astype(np.int32)}
    if kind in ("selfenergy", "template"):
        return {"p": np.sort(_momenta(r, case["n"])), "Z": _dressing(r, case["n_tab"])}
    if kind == "uneven":
        n = case["n"]
        sizes = r.integers(32, 257, n)
        return {"p": _momenta(r, n), "nq": np.array([16, 32, 64, 128])[r.integers(0, 4, n)],
                "na": np.array([8, 16, 32, 64])[r.integers(0, 4, n)], "tables": [_dressing(r, s) for s in sizes]}
    if kind == "flows":
        return {"flows": [{"n_grid": int(g), "T": float(T), "mu": float(m), **FLOW} for g, T, m in
                          zip(_spread(case["min_grid"], case["max_grid"], case["n"]),
                              0.01 + 0.29 * r.random(case["n"]), 0.4 * r.random(case["n"]))]}
    if kind == "rules":
        # E follows the RG scale; E/T sets a rule's length, up to the longest before it becomes the vacuum rule
        E = np.exp(r.uniform(math.log(0.05), math.log(2.0), case["n_mats"]))
        x = np.exp(np.linspace(math.log(90.0), math.log(0.5), case["n_mats"]))
        return {"orders": [int(o) for o in _spread(case["max_order"], case["max_order"] // 4, case["n_gl"])],
                "mats": [(float(e / t), float(e)) for e, t in zip(E, x)]}
    raise ValueError(kind)


_qp = None


def _provider():
    """The quadrature provider a program makes once."""
    global _qp
    if _qp is None:
        D.init(0)
        _qp = D.QuadratureProvider()
    return _qp


class Buffer(D.DeviceArray):
    """A torch tensor's memory as an argument of the library's calls."""

    def __init__(self, t):
        self.tensor, self.ptr, self.n = t, t.data_ptr(), t.numel()
        self.dtype, self.nbytes = np.dtype(str(t.dtype).split(".")[1]), t.numel() * t.element_size()

    def free(self):
        self.ptr = None


def _buf(a):
    return Buffer(torch.from_numpy(np.ascontiguousarray(a)).cuda())


def _out(n):
    return Buffer(torch.zeros(n, dtype=torch.float64, device="cuda"))


# ------------------------------------------------------------------------------ prepare and one pass

def prepare(case, seed):
    D.init(0)
    h, kind = _inputs(case, seed), case["kind"]
    qp = _provider()
    s = {"case": case, "qp": qp}
    if kind == "threshold":
        s.update(m2=_buf(h["m2"]), x=_buf(qp.get_points(case["nx"])), w=_buf(qp.get_weights(case["nx"])),
                 out=_out(case["n"]))
    elif kind == "finite_T":
        s["dev"] = {k: _buf(v) for k, v in h.items()}
        s["dev"].update(x=_buf(qp.get_points(case["nx"])), w=_buf(qp.get_weights(case["nx"])))
        s["out"] = _out(case["n"])
    elif kind == "selfenergy":
        s["batch"] = D.SEBatch(qp, h["p"], case["nq"], case["na"], [h["Z"]] * case["n"], *COORD, X_EXTENT, K)
        s["out"] = _out(case["n"])
    elif kind == "uneven":
        s["batch"] = D.SEBatch(qp, h["p"], h["nq"], h["na"], h["tables"], *COORD, X_EXTENT, K)
        s["out"] = _out(case["n"])
    elif kind == "flows":
        s["flows"] = h["flows"]
        s["server"] = D.FlowServer(qp, hbm_budget=1 << 24, max_resident=64, steps_per_launch=25)
    elif kind == "rules":
        s.update(h)
    else:
        s["kat"] = kat = ctypes.CDLL(os.path.join(ROOT, "tests", "native", "libdfrg_kat.so"))
        kat.kat_last_error.restype = ctypes.c_char_p
        s.update(h, out=np.zeros(case["n"]))
    torch.cuda.synchronize()
    return s


def _dp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "threshold":
        D.threshold_batch(s["m2"], s["x"], s["w"], s["out"], X_EXTENT, K, MODES[case["mode"]], case["d"])
        return s["out"].tensor
    if kind == "finite_T":
        D.ft_batch(s["dev"], s["out"], 6.0 if case["radial_mode"] else X_EXTENT, K, MODES[case["mode"]], case["d"],
                   case["radial_mode"])
        return s["out"].tensor
    if kind in ("selfenergy", "uneven"):
        s["batch"].run(s["out"], MODES[case["mode"]])
        return s["out"].tensor
    if kind == "flows":
        server = s["server"]
        ids = [server.submit(**f) for f in s["flows"]]
        while True:
            resident, queued, _ = server.progress()
            if resident == 0 and queued == 0:
                break
        return [server.result(i)[0] for i in ids]
    if kind == "rules":
        qp = D.QuadratureProvider()
        got = [(qp.get_points(o), qp.get_weights(o)) for o in s["orders"]]
        got += [(qp.get_matsubara_points(T, E), qp.get_matsubara_weights(T, E)) for T, E in s["mats"]]
        qp.close()
        return got
    f = s["kat"].kat_selfenergy if case["call"] == "request" else s["kat"].kat_selfenergy_get
    rc = f(case["nq"], case["na"], ctypes.c_double(X_EXTENT), ctypes.c_double(K), _dp(s["p"]), case["n"], _dp(s["Z"]),
           case["n_tab"], *[ctypes.c_double(c) for c in COORD], _dp(s["out"]))
    if rc:
        raise RuntimeError(s["kat"].kat_last_error())
    return s["out"]


# ------------------------------------------------------------------------------ work and tolerance

def work(case):
    """Inputs read once, outputs written once, and the arithmetic of the integrands with one division,
    exponential, logarithm or root as 10 operations."""
    h, kind, n = _inputs(case, 1), case["kind"], case["n"] if "n" in case else 1
    if kind == "threshold":  # per node: sum, reciprocal, square, product and sum
        return {"bytes": 16.0 * n + 16 * case["nx"], "flops": 15.0 * n * case["nx"] + 40 * case["nx"]}
    if kind == "finite_T":  # per frequency pair: three denominators, their reciprocal, the sum
        pairs = float(h["m_n"].sum()) * case["nx"]
        return {"bytes": 56.0 * n + 16 * (len(h["mx"]) + case["nx"]), "flops": 26.0 * pairs + 60.0 * n * case["nx"]}
    if kind in ("selfenergy", "template"):  # per node: |p - q|, table index, exponential, reciprocal
        return {"bytes": 16.0 * n + 8 * case["n_tab"] + 16 * (case["nq"] + case["na"]),
                "flops": 54.0 * n * case["nq"] * case["na"] ** 2}
    if kind == "uneven":
        evals = float((h["nq"].astype(float) * h["na"].astype(float) ** 2).sum())
        return {"bytes": 24.0 * n + 8.0 * sum(len(t) for t in h["tables"]), "flops": 54.0 * evals}
    if kind == "flows":  # per grid point, step and stage: 64 nodes of two threshold integrals
        points = float(sum(f["n_grid"] for f in h["flows"]))
        return {"bytes": 8.0 * points, "flops": points * FLOW_STEPS * 4 * (64 * 2 * 45.0 + 40)}
    # rules: a root or eigenvalue to full precision takes the recurrence of its order a few times
    sizes = [float(o) for o in h["orders"]] + [_mats_size(T, E) for T, E in h["mats"]]
    return {"bytes": 16.0 * sum(sizes), "flops": sum(60.0 * m * m for m in sizes)}


def tolerance(case):
    kind = case["kind"]
    if kind == "flows":  # rounding carried through thousands of steps
        return {"rel": 1e-11, "max": 1e-10}
    if kind == "rules":  # relative error of the smallest nodes and weights
        return {"rel": 1e-13, "max": 1e-12}
    if case.get("mode") == "mixed" and kind in ("selfenergy", "uneven"):  # single-precision seeds, stated as 1e-8
        return {"rel": 4e-9, "max": 1e-8}
    return {"rel": 1e-13, "max": 1e-12}  # sums in 64 bits


# ------------------------------------------------------------------- the same results in plain 64 bits

def _gl(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1.0), 0.5 * w


def _selfenergy(p, nq, na, Z):
    (x, wx), (c, wc) = _gl(nq), _gl(na)
    start, stop, bias = COORD
    b = (stop - start) / math.expm1(bias)

    def G(y):
        idx = np.clip(np.log1p((y - start) / b) * (len(Z) - 1) / bias, 0, len(Z) - 1)
        i = np.minimum(idx.astype(int), len(Z) - 2)
        z = Z[i] * (1.0 - (idx - i)) + Z[i + 1] * (idx - i)
        return 1.0 / (z * y * y + K * K * np.exp(-y * y / (K * K)))

    q = K * np.sqrt(x * X_EXTENT)
    xr = q * q / (K * K)
    c1 = 2.0 * c - 1.0
    el = 2 * math.pi / (2 * math.pi) ** 4 * (q * q / 2 * K * K) * wx * X_EXTENT
    fq = el * 2.0 * np.exp(-xr) * K * K * (1.0 + xr) * G(q) ** 2
    pq = np.sqrt(np.maximum(p * p + q[:, None] ** 2 - 2.0 * p * q[:, None] * c1, 0.0))
    return float((fq[:, None] * (2.0 * wc * np.sqrt(1.0 - c1 * c1)) * G(pq)).sum() * (2.0 * wc).sum())


def _threshold_nodes(nx, d):
    x, w = _gl(nx)
    q = K * np.sqrt(x * X_EXTENT)
    S = 2.0 * math.pi ** (d / 2.0) / math.gamma(d / 2.0)
    e = np.exp(-q * q / K ** 2)
    el = S / (2 * math.pi) ** d * q ** (d - 2) / 2 * K * K * w * X_EXTENT
    return el * 2.0 * e * K * K * (1.0 + q * q / K ** 2), q * q + K * K * e


def _finite_T(case, h):
    x, w = _gl(case["nx"])
    d = case["d"]
    S = 2.0 * math.pi ** ((d - 1) / 2.0) / math.gamma((d - 1) / 2.0) / (2 * math.pi) ** (d - 1)
    if case["radial_mode"]:
        q, el = 6.0 * x, S * (6.0 * x) ** (d - 2) * 6.0 * w
    else:
        q = K * np.sqrt(x * X_EXTENT)
        el = S * q ** (d - 3) / 2 * K * K * w * X_EXTENT
    q2 = q * q
    e = np.exp(-q2 / K ** 2)
    f = torch.from_numpy(el * 2.0 * e * K * K * (1.0 + q2 / K ** 2)).cuda()
    a1, q2 = torch.from_numpy(q2 + K * K * e).cuda(), torch.from_numpy(q2).cuda()
    out = np.zeros(case["n"])
    for off in np.unique(h["m_off"]):
        at = np.nonzero(h["m_off"] == off)[0]
        nm = int(h["m_n"][at[0]])
        W = torch.from_numpy(np.concatenate([[0.0], h["mx"][off:off + nm]])).cuda()
        for part in np.array_split(at, max(1, len(at) // 256)):
            T, p0, pa, m1, m2 = (torch.from_numpy(h[k][part]).cuda()[:, None, None]
                                 for k in ("T", "p0", "pabs", "m1", "m2"))
            wt = torch.from_numpy(np.concatenate([[0.0], h["mw"][off:off + nm]])).cuda()[None, None, :].clone()
            s = q2[None, :, None] + pa * pa
            d1, a2 = W ** 2 + a1[None, :, None] + m1, s + K * K * torch.exp(-s / K ** 2) + m2
            both = 1.0 / ((W + p0) ** 2 + a2) + 1.0 / ((p0 - W) ** 2 + a2)
            g = f[None, :, None] / d1 ** 2 * both
            tot = (g * wt).sum((1, 2)) + 0.5 * T[:, 0, 0] * g[:, :, 0].sum(1)
            out[part] = tot.cpu().numpy()
    return out


def _flows(case, h):
    """All flows at once: RK4 on the concatenated grids, stencils by index."""
    x, w = _gl(64)
    xr = torch.from_numpy(x * X_EXTENT).cuda()
    e = torch.exp(-xr)
    A, Dj = xr + e, torch.sqrt(xr) * torch.from_numpy(w).cuda() * X_EXTENT * e * (1.0 + xr) / (2 * math.pi ** 2)
    n = [f["n_grid"] for f in h["flows"]]
    col = lambda f: torch.from_numpy(np.concatenate([np.full(m, f(d)) for m, d in zip(n, h["flows"])])).cuda()
    hh, T = col(lambda d: d["rho_max"] / (d["n_grid"] - 1)), col(lambda d: d["T"])
    i = torch.from_numpy(np.concatenate([np.arange(m) for m in n])).cuda()
    first, last = i == 0, i == torch.from_numpy(np.concatenate([np.full(m, m - 1) for m in n])).cuda()
    rho, Tc, here = i * hh, T[:, None], torch.arange(len(i), device="cuda")
    at = lambda k: (here + k).clamp(0, len(i) - 1)
    idx = {k: at(k) for k in (-2, -1, 1, 2)}

    def S2(E2):
        E = torch.sqrt(E2)
        a = torch.exp(-E / Tc)
        return ((1 + a) / -torch.expm1(-E / Tc)) / (4 * E ** 3) + 4 * a / torch.expm1(-E / Tc) ** 2 / (8 * Tc * E2)

    def rhs(u, k):
        m1, m2, p1, p2 = u[idx[-1]], u[idx[-2]], u[idx[1]], u[idx[2]]
        up = torch.where(first, -3 * u + 4 * p1 - p2, torch.where(last, 3 * u - 4 * m1 + m2, p1 - m1)) / (2 * hh)
        upp = torch.where(first, u - 2 * p1 + p2, torch.where(last, u - 2 * m1 + m2, p1 - 2 * u + m1)) / (hh * hh)
        I = lambda m: k ** 5 * (S2(k * k * A + m[:, None]) @ Dj)
        return 0.5 * ((FLOW["N"] - 1) * up * I(u) + (3 * up + 2 * rho * upp) * I(u + 2 * rho * up))

    u, dt = FLOW["m2_0"] + FLOW["lam"] / 2 * rho, math.log(1e3) / FLOW_STEPS
    for st in range(FLOW_STEPS):
        ka, kb, kc = math.exp(-st * dt), math.exp(-(st + 0.5) * dt), math.exp(-(st + 1) * dt)
        k1 = rhs(u, ka)
        k2 = rhs(u + 0.5 * dt * k1, kb)
        k3 = rhs(u + 0.5 * dt * k2, kb)
        k4 = rhs(u + dt * k3, kc)
        u = u + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
    return [v.clone() for v in torch.split(u, n)]


def _mats_size(T, E):
    m = 5 + int(math.sqrt(4.0 * 100 * E / (math.pi ** 2 * T)))
    return max(32, min(128, 2 * math.ceil(m / 2)))


def _matsubara(T, E):
    """The Gaussian rule of the Matsubara sum: nodes and weights from the eigenproblem of its recurrence."""
    n = _mats_size(T, E)
    j = np.arange(n)
    a = 2.0 * math.pi ** 2 / (4 * j + 1) / (4 * j + 5)
    a[0] = math.pi ** 2 / 15
    b = math.pi ** 4 / ((4.0 * j[1:] - 1) * (4 * j[1:] + 3)) / (4.0 * j[1:] + 1) ** 2
    lam, v = np.linalg.eigh(np.diag(a) + np.diag(np.sqrt(b), 1) + np.diag(np.sqrt(b), -1))
    return 2 * math.pi * T / np.sqrt(lam), T * math.pi ** 2 / 6 * v[0] ** 2 / lam


def exact(case, seed):
    h, kind = _inputs(case, seed), case["kind"]
    if kind == "threshold":
        f, a = (torch.from_numpy(v).cuda() for v in _threshold_nodes(case["nx"], case["d"]))
        return torch.cat([(1.0 / (a + m[:, None]) ** 2) @ f for m in torch.from_numpy(h["m2"]).cuda().split(65536)])
    if kind == "finite_T":
        return torch.from_numpy(_finite_T(case, h))
    if kind in ("selfenergy", "template"):
        return np.array([_selfenergy(p, case["nq"], case["na"], h["Z"]) for p in h["p"]])
    if kind == "uneven":
        return np.array([_selfenergy(*a) for a in zip(h["p"], h["nq"], h["na"], h["tables"])])
    if kind == "flows":
        return _flows(case, h)
    return [_gl(o) for o in h["orders"]] + [_matsubara(T, E) for T, E in h["mats"]]
