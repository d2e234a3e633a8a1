"""The work a user of this library has it do, as measurable cases.

One case is a dict of plain values; prepare() makes what the user's program
holds before the call (the caps objects, the frequencies and m of the blocks,
or matrices on the device), run() is one pass through the public entry
points, exact() the same results in plain numpy/torch at 64 bits.

Kinds of work:
  block    one (ξ, m) block: caps_logdetD, the call of the reference's CLI
  batch    all m = 0 .. n_m - 1 at the first n_xi frequencies of one geometry
           (one Matsubara frequency, or the blocks of an energy)
  mixed    n perfect-reflector blocks, each of its own geometry, one batch
  matrix   the round-trip matrix of one block on the host (caps_M_init)
  energy   a whole free energy: Matsubara sum (T > 0), ξ integral (T = 0)
  lu       log|det| of n general matrices already on the device, the
           allocation-free entry for callers inside a captured stream

Sizes: the geometries of the tests, the benchmark and the manual (R/L = 20,
60, 100, 200, 2000 with ldim 120 .. 12000) and the ranges between.
"""
import ctypes
import math
import os

import numpy as np
import torch

L0 = 1e-6                      # plate-sphere distance (m)
C, KB, HBAR, HBAR_EV = 299792458.0, 1.38064852e-23, 1.0545718e-34, 6.582119514e-16
DRUDE_EV = (9.0, 0.035)        # gold-like Drude metal: ωp, γ in eV
GOLD = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tests", "golden", "gold.csv")


def listed():
    return [
        # one small block: the latency of a single call
        {"name": "block_small", "kind": "block", "rbyl": 20.0, "ldim": 120, "xi": 1.0, "m": 1, "material": "pr"},
        # one block with a dense determinant algorithm (its own shortcut rules)
        {"name": "block_dense", "kind": "block", "rbyl": 50.0, "ldim": 251, "xi": 3.0, "m": 2, "material": "drude",
         "detalg": "LU"},
        # one block of the R/L = 200 configuration, as the plain driver computes them one by one
        {"name": "block_drude", "kind": "block", "rbyl": 200.0, "ldim": 1200, "xi": 165.0, "m": 5,
         "material": "drude"},
        # one block at the largest aspect ratio, N = 24000
        {"name": "block_large", "kind": "block", "rbyl": 2000.0, "ldim": 12000, "xi": 2.0, "m": 10,
         "material": "pr"},
        # the matrix elements themselves, for a caller with its own use of M
        {"name": "matrix", "kind": "matrix", "rbyl": 60.0, "ldim": 361, "xi": 2.0, "m": 2, "material": "drude"},
        # all m of one frequency at a small aspect ratio: many small matrices
        {"name": "batch_small", "kind": "batch", "rbyl": 20.0, "ldim": 120, "xi": 1.0, "n_xi": 1, "n_m": 121,
         "material": "pr"},
        # one Matsubara frequency of tabulated gold, as a resumed or distributed run asks for
        {"name": "batch_gold", "kind": "batch", "rbyl": 100.0, "ldim": 701, "xi": 41.5, "n_xi": 1, "n_m": 77,
         "material": "gold"},
        # the blocks of the first two Matsubara frequencies of the R/L = 200 energy
        {"name": "batch_drude", "kind": "batch", "rbyl": 200.0, "ldim": 1200, "xi": 165.0, "n_xi": 2, "n_m": 111,
         "material": "drude"},
        # a sweep over geometries, dimensions 600 .. 6000 in one batch
        {"name": "mixed", "kind": "mixed", "n": 64, "rbyl": 50.0, "rbyl_to": 500.0, "xi": 0.1, "xi_to": 300.0},
        # a whole energy at room temperature, planned by the surrogate and replayed as graphs
        {"name": "energy_T300", "kind": "energy", "rbyl": 100.0, "ldim": 701, "T": 300.0, "mode": "surrogate",
         "material": "drude", "epsrel": 1e-6, "graph": True},
        # a whole zero-temperature energy: many small batches, one per refinement level
        {"name": "energy_T0", "kind": "energy", "rbyl": 20.0, "ldim": 120, "T": 0.0, "mode": "batched",
         "material": "pr", "epsrel": 1e-6, "graph": False},
        # general matrices (no structure assumed) in a serving loop
        {"name": "lu", "kind": "lu", "dim": 1200, "n": 4},
    ]


def draw(rng):
    def log(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))

    kind = rng.choice(["block", "block", "batch", "batch", "mixed", "matrix", "energy", "lu"])
    if kind == "lu":
        dim = int(log(30, 2000))
        return {"kind": kind, "dim": dim, "n": max(1, min(int(log(1, 64)), 6000 // dim))}
    if kind == "mixed":
        a = log(12, 300)
        return {"kind": kind, "n": int(log(2, 80)), "rbyl": a, "rbyl_to": a * rng.uniform(1.2, 4), "xi": 0.1,
                "xi_to": log(10, 300)}
    top = {"block": 1500, "batch": 200, "matrix": 120, "energy": 120}[kind]
    rbyl = log(10, top)
    ldim = max(20, int(rbyl * rng.uniform(5, 7)))
    material = rng.choice(["pr", "drude", "gold"])
    if kind == "energy":
        return {"kind": kind, "rbyl": rbyl, "ldim": ldim, "T": 300.0, "mode": "batched", "material": material,
                "epsrel": log(1e-8, 1e-5), "graph": rng.random() < 0.5}
    case = {"kind": kind, "rbyl": rbyl, "ldim": ldim, "xi": log(0.1, 2 * rbyl), "material": material}
    if kind == "batch":
        n_xi = rng.choice([1, 1, 2, 5])
        return dict(case, n_xi=n_xi, n_m=max(1, int(log(2, min(120, 4 * math.sqrt(ldim) + 2)) / n_xi)))
    case["m"] = int(log(1, 4 * math.sqrt(ldim))) - 1
    if kind == "block" and rbyl < 200:
        case["detalg"] = rng.choice(["HODLR", "HODLR", "LU", "QR"])
    return case


# ---- inputs -----------------------------------------------------------------

def _inputs(case, seed):
    """What the seed decides: the geometry and the frequencies, within a few
    per cent of the case's; the geometries of a mixed batch."""
    rng = np.random.default_rng(seed)
    if case["kind"] == "lu":
        return {"gen": int(rng.integers(1 << 40))}
    if case["kind"] == "mixed":
        out = []
        for _ in range(case["n"]):
            r = math.exp(rng.uniform(math.log(case["rbyl"]), math.log(case["rbyl_to"])))
            ldim = max(20, math.ceil(6 * r))
            out.append((r, ldim, float(rng.uniform(case["xi"], case["xi_to"])), int(rng.integers(0, ldim // 4 + 1))))
        return {"blocks": out}
    rbyl = case["rbyl"] * (1 + 0.02 * rng.uniform(-1, 1))
    if case["kind"] == "energy":
        return {"rbyl": rbyl}
    xi = case["xi"] * (1 + 0.02 * rng.uniform(-1, 1))
    if case["kind"] != "batch":
        return {"rbyl": rbyl, "xi": xi}
    return {"rbyl": rbyl, "blocks": [(j * xi, m) for j in range(1, case["n_xi"] + 1) for m in range(case["n_m"])]}


def _object(case, rbyl, ldim):
    import caps_amd
    c = caps_amd.Caps(rbyl * L0, L0, ldim=ldim, detalg=case.get("detalg"))
    if case.get("material") == "drude":
        c.set_drude(*DRUDE_EV)
    elif case.get("material") == "gold":
        c.set_material(GOLD)
    return c


def _lu_matrices(case, seed):
    """Column-major matrices with eigenvalues of order one; every third needs row interchanges."""
    dim, n = case["dim"], case["n"]
    gen = torch.Generator(device="cuda").manual_seed(_inputs(case, seed)["gen"])
    A = torch.randn((n, dim, dim), generator=gen, dtype=torch.float64, device="cuda")
    plain = torch.arange(n, device="cuda") % 3 != 0
    A[plain] *= 0.3 / math.sqrt(dim)
    A[plain] += torch.eye(dim, dtype=torch.float64, device="cuda")
    return A


def prepare(case, seed):
    import caps_amd
    i = _inputs(case, seed)
    kind = case["kind"]
    if kind == "lu":
        fn = caps_amd.lib().capsx_lu_logdet_batch_noalloc
        fn.restype = ctypes.c_int
        fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
        A = _lu_matrices(case, seed)
        return {"case": case, "fn": fn, "A": A, "work": torch.empty_like(A),
                "out": torch.empty(case["n"], dtype=torch.float64, device="cuda")}
    if kind == "mixed":
        objs = [_object(case, r, ldim) for r, ldim, _, _ in i["blocks"]]
        return {"case": case, "objs": objs, "xis": np.array([b[2] for b in i["blocks"]]),
                "ms": np.array([b[3] for b in i["blocks"]], dtype=np.int32)}
    c = _object(case, i["rbyl"], case["ldim"])
    s = {"case": case, "caps": c}
    if kind == "batch":
        s["xis"] = np.array([x for x, _ in i["blocks"]])
        s["ms"] = np.array([m for _, m in i["blocks"]], dtype=np.int32)
    elif kind == "energy":
        c.set_graph(case["graph"])
        if case["mode"] == "surrogate":
            from caps_amd import surrogate
            s["mlp"] = surrogate.MLP.load()
            s["mlp"].attach(c, *DRUDE_EV)
    else:
        s["xi"] = i["xi"]
    return s


def run(state):
    import caps_amd
    case = state["case"]
    kind = case["kind"]
    if kind == "block":
        return np.float64(state["caps"].logdetD(state["xi"], case["m"]))
    if kind == "batch":
        return state["caps"].logdetD_batch(state["xis"], state["ms"])
    if kind == "mixed":
        return caps_amd.logdetD_multi(state["objs"], state["xis"], state["ms"])
    if kind == "matrix":
        return state["caps"].matrix(state["xi"], case["m"])[:2]
    if kind == "energy":
        F, _, used = state["caps"].free_energy(case["T"], cutoff=1e-9, epsrel=case["epsrel"], mode=case["mode"],
                                               drude_xi0=True)
        return np.float64(F), used
    state["work"].copy_(state["A"])
    n, dim = case["n"], case["dim"]
    if state["fn"](state["work"].data_ptr(), dim, dim, n, state["out"].data_ptr(),
                   torch.cuda.current_stream().cuda_stream) != 0:
        raise RuntimeError("capsx_lu_logdet_batch_noalloc refused its input")
    return state["out"]


# ---- what a pass cannot do without --------------------------------------------

def _block_work(ldim, m):
    """Flops of one determinant: 1 - M is 1 - F^T F with a row of F per wave
    number and polarization; some 2.2 sqrt(2 lmax) + 30 wave numbers resolve
    the integrands up to l = lmax, so the smaller of the two Gram matrices
    has D = min(twice that, 2 ldim) rows: a symmetric product of the other
    extent's depth and a Cholesky factorization."""
    rows = 2 * (2.2 * math.sqrt(2 * (ldim + m)) + 30)
    D, K = min(rows, 2 * ldim), max(rows, 2 * ldim)
    return D * D * K + D ** 3 / 3


def work(case):
    kind = case["kind"]
    if kind == "lu":
        n, dim = case["n"], case["dim"]
        return {"bytes": 8.0 * n * dim * dim, "flops": 2 / 3 * n * dim ** 3}
    if kind == "mixed":
        blocks = _inputs(case, 1)["blocks"]
        return {"bytes": 8.0 * len(blocks), "flops": sum(_block_work(b[1], b[3]) for b in blocks)}
    ldim = case["ldim"]
    if kind == "matrix":
        rows = 2 * (2.2 * math.sqrt(2 * (ldim + case["m"])) + 30)
        return {"bytes": 8.0 * (2 * ldim) ** 2, "flops": rows * (2 * ldim) ** 2}
    if kind == "block":
        return {"bytes": 8.0, "flops": _block_work(ldim, case["m"])}
    if kind == "batch":
        n = case["n_xi"] * case["n_m"]
        return {"bytes": 8.0 * n, "flops": sum(_block_work(ldim, m) for m in range(case["n_m"])) * case["n_xi"]}
    # energies: the m-sums of the frequencies that count end near m = 7.5 sqrt(R/L) each
    n = 7.5 * math.sqrt(case["rbyl"]) * (9 if case["T"] > 0 else 20)
    return {"bytes": 8.0, "flops": n * _block_work(ldim, 30)}


# ---- the results in plain numpy ------------------------------------------------
# Each element of M is an integral over the wave number x = cosh θ in [1, ∞) of
# products p_l p_l', p_l t_l', t_l t_l' with p_l = m P_l^m/√(x²-1) and
# t_l = √(x²-1) dP_l^m/dx, the Fresnel coefficients and e^{-2ξx}; on a
# quadrature grid M = F^T F with one row of F per node and polarization.

def _ratios(x, L):
    """I_{l-1/2}(x)/I_{l+1/2}(x), l = 0..L (backward recurrence; entry 0 unused)."""
    top = L + 100 + int(2 * x) if x < 200 else L + 300 + int(8 * math.sqrt(x * 20))
    r = (top + 0.5 + math.hypot(top + 0.5, x)) / x
    out = np.zeros(L + 1)
    for l in range(top - 1, 0, -1):
        r = (2 * l + 1) / x + 1 / r
        if l <= L:
            out[l] = r
    return out


def _mie(chi, eps, L):
    """√|a_l|, √|b_l| for l = 1..L as mantissas and powers of two (chi: ξ R/c, eps: ε - 1 of the sphere)."""
    r = _ratios(chi, L + 1)
    kap = np.zeros(L + 2)
    kap[1] = 1 / (1 + 1 / chi)                       # K_{l-1/2}/K_{l+1/2}
    for l in range(1, L + 1):
        kap[l + 1] = 1 / ((2 * l + 1) / chi + kap[l])
    # √(π/2 I_{l+1/2}/K_{l+1/2})
    lead = 0.5 * (math.log1p(-math.exp(-2 * chi)) - math.log(2) + 2 * chi)
    e = math.floor(lead / math.log(2))
    s = math.exp(lead - e * math.log(2))
    sm, se = np.zeros(L), np.zeros(L, dtype=np.int64)
    for l in range(1, L + 1):
        s, de = math.frexp(s * math.sqrt(kap[l] / r[l]))
        e += de
        sm[l - 1], se[l - 1] = s, e
    l = np.arange(1, L + 1)
    k, rn1 = kap[1:L + 1], r[2:L + 2]
    if math.isinf(eps):
        fa, fb = (l + 1 + chi / rn1) / (l + chi * k), np.ones(L)
    else:
        n = math.sqrt(1 + eps)
        q = _ratios(n * chi, L + 1)
        gd = chi * (k + n * q[1:L + 1])
        fa = (eps * (l + 1) + n * n * chi / rn1 - n * chi / q[2:L + 2]) / (eps * (chi * k + l) + gd)
        fb = chi * (n / q[2:L + 2] - 1 / rn1) / gd
    return sm * np.sqrt(fa), sm * np.sqrt(fb), se


def _grid(xi, lmax, h=0.5):
    """x - 1 and the weights of the trapezoidal rule in v, x = 1 + A² softplus(v)²."""
    alpha, nu = 2 * xi, 2 * lmax + 2.5
    xp = math.hypot(1, nu / alpha)
    g = lambda x: nu * math.acosh(x) - alpha * x  # noqa: E731
    x = xp
    while g(x) > g(xp) - 80:
        x = 1 + (x - 1) * 1.02 + 0.5 / alpha
    A = 0.5 / math.sqrt(alpha)
    s = math.sqrt(max(x - 1, 90 / alpha)) / A
    v = np.arange(-19.0, s + h, h)
    sp = np.logaddexp(0, v)
    return A * A * sp * sp, 2 * A * A * sp / (1 + np.exp(-v)) * h


def _rows(rbyl, ldim, xi, ms, eps):
    """F of the blocks m in ms (ascending) at one frequency: yields (rows, 2 ldim) arrays, columns a_l then b_l."""
    lmin = [1 if m == 0 else max(m, math.floor(m / math.sqrt(2 / rbyl) + 0.5) - ldim // 2) for m in ms]
    mm = np.array([max(m, 1) for m in ms])
    lmax = max(lmin) + ldim - 1
    am, bm, me = _mie(xi / (1 + 1 / rbyl), eps, lmax)
    xm1, w = _grid(xi, lmax)
    x = 1 + xm1
    x2 = xm1 * (x + 1)
    sx = np.sqrt(x2)
    if math.isinf(eps):
        rte = rtm = np.ones_like(x)
    else:
        y = eps / (x * x)
        bb = y / (np.sqrt(1 + y) + 1)
        rte, rtm = bb / (2 + bb), (eps - bb) / (eps + 2 + bb)
    # √((l-m)!/(l+m)!) P_l^m e^{-ξx} √w at l = m, as p 2^E; then the recurrence in l
    base = np.array([[math.lgamma(2 * q + 1) / 2 - q * math.log(2) - math.lgamma(q + 1)] for q in mm]) \
        + 0.5 * mm[:, None] * np.log(x2) - xi * x + 0.5 * np.log(w)
    E = np.floor(base / math.log(2))
    p, prev, E = np.exp(base - E * math.log(2)), np.zeros_like(base), E.astype(np.int32)
    lo = np.array(lmin) - mm
    J = int(lo.max()) + ldim
    P, T, EE = (np.zeros((J,) + base.shape) for _ in range(3))
    M1 = mm[:, None].astype(float)
    zero = np.array([[m == 0] for m in ms])
    for j in range(J):
        l = M1 + j
        r0 = np.sqrt((l - M1) * (l + M1))
        g = np.sqrt((2 * l + 1) / (l * (l + 1)))
        P[j] = np.where(zero, 0.0, g * M1 * p / sx)
        T[j] = np.where(zero, g * p * np.sqrt(l * (l + 1)), g * (l * x * p - r0 * prev) / sx)
        EE[j] = E
        nxt = ((2 * l + 1) * x * p - r0 * prev) / np.sqrt((l + 1 - M1) * (l + 1 + M1))
        prev, p = p, nxt
        big = p > 1e150
        if big.any():
            s = np.where(big, 2.0 ** -400, 1.0)
            p, prev, E = p * s, prev * s, E + 400 * big
    for b in range(len(ms)):
        j, l = slice(int(lo[b]), int(lo[b]) + ldim), slice(lmin[b] - 1, lmin[b] - 1 + ldim)
        e = EE[j, b].T.astype(np.int32) + me[l].astype(np.int32)[None]
        Pb, Tb = P[j, b].T, T[j, b].T
        stm, ste = np.sqrt(rtm)[:, None], np.sqrt(rte)[:, None]
        yield np.vstack([np.hstack([np.ldexp(stm * Tb * am[l], e), np.ldexp(stm * Pb * bm[l], e)]),
                         np.hstack([np.ldexp(ste * Pb * am[l], e), np.ldexp(ste * Tb * bm[l], e)])])


def _logdet(F, dense=False):
    """log det(1 - F^T F) with the library's rules for small traces."""
    keep = np.abs(F).max(axis=1) > 1e-30 * np.abs(F).max()
    F = F[keep]
    tr = float(np.sum(F * F))
    if tr < 1e-8:
        return -tr
    G = F @ F.T if F.shape[0] < F.shape[1] else F.T @ F
    tr2 = float(np.sum(G * G))
    if dense:
        nrm = math.sqrt(tr2)
        if nrm < 1 and abs((nrm * nrm / 2 + nrm + math.log1p(-nrm)) / (-tr - tr2 / 2)) < 1e-8:
            return -tr - tr2 / 2
    if tr < 0.02:
        s, P, k = -tr - tr2 / 2, G @ G, 3
        while tr ** k > 1e-17 * tr:
            s -= float(np.sum(P * G)) / k
            P, k = P @ G, k + 1
        return s
    return 2 * float(np.sum(np.log(np.diag(np.linalg.cholesky(np.eye(len(G)) - G)))))


def _eps(case, rbyl, xi):
    """ε(iξ) - 1 of the case's material at ξ(L+R)/c = xi."""
    w = xi * C / ((rbyl + 1) * L0)
    if case.get("material", "pr") == "pr":
        return math.inf
    if case["material"] == "drude":
        wp, ga = DRUDE_EV[0] / HBAR_EV, DRUDE_EV[1] / HBAR_EV
        return wp * wp / (w * (w + ga))
    tab = np.loadtxt(GOLD)
    assert tab[0, 0] <= w <= tab[-1, 0]
    return float(np.interp(w, tab[:, 0], tab[:, 1] - 1))


def _msum(case, rbyl, xi, cutoff=1e-9):
    """Σ'_m logdetD(ξ, m) up to and with the first m below the cutoff, and the number of terms."""
    eps, v = _eps(case, rbyl, xi), []
    for m0 in range(0, 100000, 16):
        for F in _rows(rbyl, case["ldim"], xi, range(m0, m0 + 16), eps):
            v.append(_logdet(F))
            if v[-1] == 0 or v[-1] / v[0] < cutoff:
                return math.fsum(v) - v[0] / 2, len(v)


def _energy(case, rbyl):
    x = 1 / rbyl
    if case["T"] > 0:
        # the ξ = 0 Drude term in closed form, then the Matsubara sum
        Z = (1 + x) * (1 - math.sqrt((x * x + 2 * x) / (x * x + 2 * x + 1)))
        s1 = s2 = 0.0
        for l in range(1, 100000):
            a = Z ** (2 * l)
            v1, v2 = (2 * l + 1) * math.log1p(-a * Z), a * Z * (1 - a) / (1 - a * Z)
            s1, s2 = s1 + v1, s2 + v2
            if abs(v1 / s1) < 1e-16 and abs(v2 / s2) < 1e-16:
                break
        v0 = 0.5 * (s1 + math.log1p(-(1 - Z * Z) * s2))
        step = 2 * math.pi * KB * (rbyl + 1) * L0 * case["T"] / (HBAR * C)
        total, used = v0 / 2, 0
        for n in range(1, 100000):
            v, k = _msum(case, rbyl, n * step)
            total, used = total + v, used + k
            if abs(v / v0) < case["epsrel"]:
                return step / math.pi * total, used
    # ∫ F_ξ dξ by the Fourier-Chebyshev rule on [0, ∞), levels doubled until two agree
    alpha = 2 * x / (1 + x)
    cut = -(1 + 1 / x) * math.log(2 * x * 1e-100) / 2 if x < 0.1 else math.inf
    known, used, last, M = {}, 0, None, 5
    while True:
        total = 0.0
        for i in range(1, M):
            t = math.pi * i / M
            xi = 1 / math.tan(t / 2) ** 2 / alpha
            key = i / M
            if key not in known:
                known[key], k = (0.0, 0) if xi > cut else _msum(case, rbyl, xi)
                used += k
            w = 8 * math.sin(t) / (1 - math.cos(t)) ** 2 / M * math.fsum(math.sin(j * t) / j for j in range(1, M, 2))
            total += w * known[key]
        if last is not None and abs(1 - last / total) < case["epsrel"]:
            return total / alpha / math.pi, used
        last, M = total, 2 * M


def exact(case, seed):
    i = _inputs(case, seed)
    kind = case["kind"]
    if kind == "lu":
        return torch.linalg.slogdet(_lu_matrices(case, seed))[1]
    if kind == "mixed":
        if sum(b[1] for b in i["blocks"]) > 200000:
            return None
        return np.array([_logdet(next(_rows(r, ldim, xi, [m], math.inf))) for r, ldim, xi, m in i["blocks"]])
    dense = case.get("detalg", "HODLR") != "HODLR"
    if kind == "energy":
        # (F, blocks in the sums); the number is a whole number, compared as it is
        return (np.float64(_energy(case, i["rbyl"])[0]), None) if case["rbyl"] * case["ldim"] < 80000 else None
    if kind == "batch":
        out = []
        for j in range(case["n_xi"]):
            xi = i["blocks"][j * case["n_m"]][0]
            for m0 in range(0, case["n_m"], 24):
                ms = range(m0, min(m0 + 24, case["n_m"]))
                out += [_logdet(F, dense) for F in _rows(i["rbyl"], case["ldim"], xi, ms, _eps(case, i["rbyl"], xi))]
        return np.array(out)
    F = next(_rows(i["rbyl"], case["ldim"], i["xi"], [case["m"]], _eps(case, i["rbyl"], i["xi"])))
    if kind == "block":
        return np.float64(_logdet(F, dense))
    M = F.T @ F
    N = 2 * case["ldim"]
    order = np.arange(N).reshape(2, N // 2).T.ravel()    # a_l, b_l columns interleaved
    return M[np.ix_(order, order)], None
