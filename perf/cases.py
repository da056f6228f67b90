"""Performance cases of the Chebyshev path: what users of this package run.

Every case goes through the public entry points of ``tbtk_amd.engine.Engine``
and the host helpers of ``tbtk_amd.kpm``, in the way the C++ property extractor
and ``bench.py`` use them: moments of one start vector, of blocks of sites, of
random vectors and of batches of models, and the energy contraction in its
three forms. Models are the lattices of ``tbtk_amd.lattice``.

listed() are the fixed cases, draw() gives more of the same ranges, prepare()
builds what a program holds before the call (handle, model on the device,
lookup table, coefficient arrays), run() is one pass, work() what a pass cannot
do without, exact() the same outputs in plain 64-bit torch.
"""
import math

import numpy as np
import torch

from tbtk_amd import engine as X
from tbtk_amd import kpm
from tbtk_amd import lattice as L

BROADENING = 1e-6   # the solver's default Lorentz broadening

# Model families: scale factors above the Gershgorin bound of the amplitudes
# and disorder used here, states per cell, stored entries per row.
SCALE = {"square_spin": 6.0, "nambu": 7.0, "honeycomb": 9.2, "square": 5.0, "cubic": 7.5,
         "flux": 5.0}
ORBITALS = {"square_spin": 2, "nambu": 4, "honeycomb": 4, "square": 1, "cubic": 1, "flux": 1}
ROW = {"square_spin": 5, "nambu": 6, "honeycomb": 4, "square": 5, "cubic": 7, "flux": 5}
REAL_H = {"square_spin": True, "nambu": True, "honeycomb": True, "square": True, "cubic": True,
          "flux": False}


def listed():
    return [
        # One site's local density of states on a 30x30 lattice with spin: the
        # smallest call, the size of the reference's templates and tests.
        dict(name="ldos_small", kind="ldos", model="square_spin", lx=30, ly=30, M=1000, E=1000,
             sites=2),
        # The same on a medium disordered sample with odd extents.
        dict(name="ldos_mid", kind="ldos", model="square_spin", lx=173, ly=211, M=1500, E=1201,
             sites=1),
        # The bench's headline model: 2,097,152 states, 4000 moments.
        dict(name="ldos_large", kind="ldos", model="square_spin", lx=1024, ly=1024, M=4000,
             E=2000, sites=1),
        # Off-diagonal retarded Green's functions in a magnetic field (complex H
        # whose bond values vary along x), from one site to its surroundings.
        dict(name="green_flux", kind="green", model="flux", lx=257, ly=301, M=1000, E=1000, to=9),
        # LDOS along a line cut of a superconductor (Nambu, 1,048,576 states):
        # 256 sites in FP32 blocks with moment doubling, Jackson damping.
        dict(name="block_nambu", kind="block", model="nambu", lx=512, ly=512, M=1000, E=1000,
             sites=256, doubling=True),
        # A few sites of a honeycomb ribbon, plain (undoubled) block moments.
        dict(name="block_ribbon", kind="block", model="honeycomb", lx=40, ly=997, M=777, E=801,
             sites=37, doubling=False),
        # Density of states of a cubic sample from random-phase vectors.
        dict(name="trace_cubic", kind="trace", model="cubic", lx=96, ly=100, lz=90, M=512, E=1000,
             vectors=32),
        # A sweep over samples: uneven models advanced together.
        dict(name="uneven_batch", kind="uneven", models=16, layout=4, states=100000, M=1500),
        # Map of on-site and neighbour Green's functions over many sites in FP64,
        # the pattern form of the property extractor.
        dict(name="map_multi", kind="multi", model="square_spin", lx=47, ly=53, M=600, E=500,
             sites=700, to=3),
        # A new energy window for many known moment vectors: table and FP64
        # contraction.
        dict(name="contract_table", kind="contract", vectors=1001, M=2000, E=1500, gtype=1),
        # Many vectors through the matrix-core contraction.
        dict(name="contract_mfma", kind="mfma", vectors=4096, M=2048, E=2001, gtype=1),
        # The extractor's default: few vectors, no table.
        dict(name="contract_direct", kind="direct", vectors=4, M=1000, E=1000, gtype=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, model, lo, hi):
    """Extents of a model of between lo and hi states, not always square."""
    n = _log_int(rng, lo, hi)
    per = ORBITALS[model]
    if model == "cubic":
        e = max(3, int((n / per) ** (1 / 3)))
        lx = max(3, int(e * rng.uniform(0.8, 1.2)))
        ly = max(3, int(e * rng.uniform(0.8, 1.2)))
        return dict(lx=lx, ly=ly, lz=max(3, n // (per * lx * ly)))
    e = max(3, int((n / per) ** 0.5))
    lx = max(3, int(e * rng.uniform(0.6, 1.5)))
    return dict(lx=lx, ly=max(3, n // (per * lx)))


def draw(rng):
    kind = rng.choice(["ldos", "ldos", "ldos", "green", "block", "block", "trace", "uneven",
                       "multi", "contract", "mfma", "direct"])
    if kind == "ldos":
        model = rng.choice(["square_spin", "nambu", "honeycomb", "square", "cubic", "flux"])
        hi = 1_000_000 if model == "flux" else 2_000_000
        return dict(kind=kind, model=model, **_extents(rng, model, 500, hi),
                    M=_log_int(rng, 200, 4000), E=_log_int(rng, 200, 2000),
                    sites=rng.randint(1, 2))
    if kind == "green":
        model = rng.choice(["flux", "square_spin", "honeycomb", "nambu"])
        return dict(kind=kind, model=model, **_extents(rng, model, 500, 500_000),
                    M=_log_int(rng, 200, 2000), E=_log_int(rng, 200, 1500), to=rng.randint(2, 40))
    if kind == "block":
        model = rng.choice(["nambu", "honeycomb", "square", "square_spin", "flux"])
        sites = _log_int(rng, 3, 256)
        return dict(kind=kind, model=model, **_extents(rng, model, 3000, 500_000),
                    M=_log_int(rng, 100, 1000), E=_log_int(rng, 200, 1000), sites=sites,
                    doubling=rng.random() < 0.6)
    if kind == "trace":
        model = rng.choice(["cubic", "square", "honeycomb"])
        return dict(kind=kind, model=model, **_extents(rng, model, 3000, 800_000),
                    M=_log_int(rng, 100, 512), E=_log_int(rng, 200, 1000),
                    vectors=_log_int(rng, 2, 64))
    if kind == "uneven":
        return dict(kind=kind, models=rng.randint(3, 24), layout=rng.randint(1, 1 << 20),
                    states=_log_int(rng, 5000, 100_000), M=_log_int(rng, 300, 1500))
    if kind == "multi":
        model = rng.choice(["square_spin", "honeycomb", "nambu", "flux"])
        return dict(kind=kind, model=model, **_extents(rng, model, 1000, 8000),
                    M=_log_int(rng, 100, 600), E=_log_int(rng, 100, 500),
                    sites=_log_int(rng, 20, 700), to=rng.randint(1, 4))
    if kind == "contract":
        return dict(kind=kind, vectors=_log_int(rng, 1, 1000), M=_log_int(rng, 100, 2000),
                    E=_log_int(rng, 100, 1500), gtype=rng.randint(0, 3))
    if kind == "mfma":
        return dict(kind=kind, vectors=_log_int(rng, 30, 4000), M=_log_int(rng, 100, 2048),
                    E=_log_int(rng, 100, 2000), gtype=rng.randint(0, 3))
    return dict(kind=kind, vectors=_log_int(rng, 1, 30), M=_log_int(rng, 100, 2000),
                E=_log_int(rng, 100, 1500), gtype=rng.randint(0, 3))


# ------------------------------------------------------------------ inputs --

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _states(case):
    return case["lx"] * case["ly"] * case.get("lz", 1) * ORBITALS[case["model"]]


def _builder(case, seed, spec):
    """The lattice as a device spec, or as the host model of the same CSR."""
    lx, ly, m = case["lx"], case["ly"], case["model"]
    if m == "square_spin":
        f, a, kw = (L.square_spin_spec if spec else L.square_spin), (lx, ly), dict(disorder=1.0)
    elif m == "nambu":
        f, a, kw = (L.nambu_swave_spec if spec else L.nambu_swave), (lx, ly), dict(disorder=0.5)
    elif m == "honeycomb":
        f, a = (L.honeycomb_ribbon_spec if spec else L.honeycomb_ribbon), (lx, ly)
        kw = dict(disorder=0.5)
    elif m == "cubic":
        f, a, kw = (L.cubic_spec if spec else L.cubic), (lx, ly, case["lz"]), dict(disorder=1.0)
    elif m == "square":
        f, a, kw = (L.square_spec if spec else L.square), (lx, ly), dict(disorder=0.5)
    else:
        f, a, kw = L.square, (lx, ly), dict(disorder=0.5, flux=0.01)
    return f(*a, seed=seed, **kw)


def _set_model(eng, case, seed):
    if case["model"] == "flux":
        eng.set_csr(_builder(case, seed, False).csr(), SCALE["flux"])
    else:
        eng.set_lattice(_builder(case, seed, True), SCALE[case["model"]])


def _window(scale):
    return -0.98 * scale, 0.98 * scale


def _centre(case):
    """The basis index of the middle cell's first state."""
    lz = case.get("lz", 1)
    return (((case["lx"] // 2) * case["ly"] + case["ly"] // 2) * lz + lz // 2) * \
        ORBITALS[case["model"]]


def _picked(case, seed):
    """The start and target states of a case."""
    rng = np.random.default_rng(seed + 77)
    n, kind = _states(case), case["kind"]
    if kind == "ldos":
        c = _centre(case)
        return [min(n - 1, c + k) for k in range(case["sites"])]
    if kind == "green":
        c = _centre(case)
        step = case["ly"] * ORBITALS[case["model"]]
        near = [c + a * step + b * ORBITALS[case["model"]] for a in range(-3, 4)
                for b in range(-3, 4)]
        near = sorted({x for x in near if 0 <= x < n})
        k = min(case["to"], len(near))
        return c, [int(x) for x in rng.choice(near, k, replace=False)]
    if kind == "block":
        if case["model"] == "nambu":     # a line cut along y through the middle
            cut = case["lx"] // 2 * case["ly"]
            cell = cut + np.arange(case["sites"]) % case["ly"]
            return np.sort(cell * 4 + np.arange(case["sites"]) // case["ly"] % 4)
        return np.sort(rng.choice(n, min(n, case["sites"]), replace=False))
    froms = np.sort(rng.choice(n, min(n, case["sites"]), replace=False))
    tos = [[int((f + d) % n) for d in (0, 1, case["ly"], 2)[:case["to"]]] for f in froms]
    return froms, tos


def _uneven(case, seed):
    """Specs, scales, sites and moment counts; sizes come from the case alone."""
    rng = np.random.default_rng(case["layout"])
    specs, scales, sites, moments = [], [], [], []
    for i in range(case["models"]):
        honey = bool(rng.integers(2))
        width, length = int(rng.integers(20, 201)), int(rng.integers(50, 2001))
        per = 4 if honey else 1
        length = max(2, min(length, case["states"] // (per * width)))
        f = L.honeycomb_ribbon_spec if honey else L.square_spec
        sp = f(width, length, disorder=0.5, seed=seed + i)
        specs.append(sp)
        scales.append(SCALE["honeycomb" if honey else "square"])
        moments.append(int(rng.integers(case["M"] // 3, case["M"] + 1)))
        b = int(rng.integers(1, 65))
        sites.append(np.sort(rng.choice(sp.basis_size, b, replace=False)))
    return specs, scales, sites, moments


def _coefficients(case, seed):
    """Moment-like vectors: bounded cosines of a few levels each, decaying in n."""
    rng = np.random.default_rng(seed + 5)
    K, M = case["vectors"], case["M"]
    n = torch.arange(M, dtype=torch.float64, device=_dev())
    c = torch.zeros((K, M), dtype=torch.complex128, device=_dev())
    for _ in range(4):
        th = rng.uniform(0.05, math.pi - 0.05, size=(K, 1))
        w = rng.uniform(0.1, 0.4, size=(K, 1)) * np.exp(1j * rng.uniform(0, 6.28, size=(K, 1)))
        c += torch.from_numpy(w).to(c.device) * torch.cos(torch.from_numpy(th).to(c.device) * n)
    return (c * torch.from_numpy(_jackson(M)).to(c.device)).cpu().numpy()


def _jackson(M):
    q, n = math.pi / (M + 1), np.arange(M)
    return ((M - n + 1) * np.cos(q * n) + np.sin(q * n) / math.tan(q)) / (M + 1)


def prepare(case, seed):
    kind = case["kind"]
    eng = X.Engine(0)
    st = dict(kind=kind, eng=eng, case=case)
    if kind in ("ldos", "green", "block", "trace", "multi"):
        s = SCALE[case["model"]]
        _set_model(eng, case, seed)
        lo, hi = _window(s)
        eng.lut_generate(case["M"], case["E"], lo, hi, s)
        if kind in ("block", "trace"):
            eng.set_damping(X.DAMP_JACKSON)
        st["pick"] = None if kind == "trace" else _picked(case, seed)
        st["seed"] = seed
    elif kind == "uneven":
        specs, scales, st["sites"], st["moments"] = _uneven(case, seed)
        eng.multi_set_lattices(specs, scales)
    else:
        st["c"] = _coefficients(case, seed)
        if kind == "mfma":
            eng.lut_generate(case["M"], case["E"], *_window(6.0), 6.0)
    return st


def run(st):
    eng, case, kind = st["eng"], st["case"], st["kind"]
    if kind == "ldos":
        out = {}
        for i, f in enumerate(st["pick"]):
            c = eng.moments(f, [f], case["M"])
            G = eng.contract(kpm.lorentz(c, BROADENING), X.NONPRINCIPAL)
            out["c%d" % i], out["G%d" % i], out["ldos%d" % i] = c, G, kpm.ldos_from_gf(G)
        return out
    if kind == "green":
        frm, to = st["pick"]
        c = eng.moments(frm, to, case["M"])
        return {"c": c, "G": eng.contract(kpm.lorentz(c, BROADENING), X.RETARDED)}
    if kind == "block":
        c = eng.moments_block(st["pick"], case["M"], X.DOUBLING if case["doubling"] else 0)
        return {"c": c, "G": eng.contract(c, X.NONPRINCIPAL)}
    if kind == "trace":
        c = eng.moments_trace(case["vectors"], st["seed"], case["M"], X.DOUBLING)
        return {"c": c, "G": eng.contract(c, X.NONPRINCIPAL)}
    if kind == "uneven":
        return eng.multi_moments(st["sites"], st["moments"], X.DOUBLING)
    if kind == "multi":
        froms, tos = st["pick"]
        c = np.concatenate(eng.moments_multi(froms, tos, case["M"]))
        return {"c": c, "G": eng.contract(kpm.lorentz(c, BROADENING), X.NONPRINCIPAL)}
    if kind == "contract":
        eng.lut_generate(case["M"], case["E"], *_window(6.0), 6.0)
        return eng.contract(st["c"], case["gtype"])
    if kind == "mfma":
        eng.coeffs_upload(st["c"])
        return eng.contract_mfma(case["gtype"])
    lo, hi = _window(6.0)
    return eng.contract_direct(st["c"], case["gtype"], case["E"], lo, (hi - lo) / (case["E"] - 1),
                               6.0)


# -------------------------------------------------------------------- work --

def work(case):
    """Inputs read once, outputs written once; multiply-adds of the recurrence
    (two per entry and component for a real H, four for a complex one) and of
    the contraction."""
    kind = case["kind"]
    if kind == "uneven":
        specs, _, sites, moments = _uneven(case, 0)
        b = f = 0.0
        for sp, s, m in zip(specs, sites, moments):
            row = sp.max_row_entries()
            b += sp.basis_size * 12.0 * row + 16.0 * len(s) * m
            f += 2.0 * sp.basis_size * row * len(s) * (m / 2)
        return {"bytes": b, "flops": f}
    M, E = case["M"], case["E"]
    if kind in ("contract", "mfma", "direct"):
        K = case["vectors"]
        return {"bytes": 16.0 * K * (M + E), "flops": (8.0 if case["gtype"] < 2 else 4.0) * K * M * E}
    N, row = _states(case), ROW[case["model"]]
    vecs = case["vectors"] if kind == "trace" else case["sites"] if kind != "green" else 1
    outs = {"green": case.get("to", 1), "multi": vecs * case.get("to", 1), "trace": 1}.get(kind, vecs)
    steps = M / 2 if kind == "trace" or case.get("doubling") else M
    per = 2.0 if REAL_H[case["model"]] and kind != "trace" else 8.0 if kind != "trace" else 4.0
    return {"bytes": N * (12.0 if REAL_H[case["model"]] else 20.0) * row + 16.0 * outs * (M + E),
            "flops": per * N * row * vecs * steps + 4.0 * outs * M * E}


# ------------------------------------------------------------------- exact --

def _ell(model, scale):
    """Columns and 2 H / s of every row, padded with the row itself and zero."""
    rp, col, val = model.csr()
    n = rp.size - 1
    rp = rp.astype(np.int64)
    length = np.diff(rp)
    W = int(length.max())
    cols = np.repeat(np.arange(n, dtype=np.int64)[:, None], W, axis=1)
    vals = np.zeros((n, W), dtype=np.complex128)
    row = np.repeat(np.arange(n), length)
    slot = np.arange(col.size) - np.repeat(rp[:-1], length)
    cols[row, slot] = col
    vals[row, slot] = val * (2 / scale)
    if not np.any(vals.imag):
        vals = np.ascontiguousarray(vals.real)
    d = _dev()
    return [torch.from_numpy(np.ascontiguousarray(cols[:, s])).to(d) for s in range(W)], \
        [torch.from_numpy(np.ascontiguousarray(vals[:, s])).to(d) for s in range(W)]


def _apply(ell, x):
    out = torch.zeros_like(x)
    for c, v in zip(*ell):
        y = x.index_select(0, c)
        out.addcmul_(y, v if x.dim() == 1 else v[:, None])
    return out


def _start(n, dtype, froms):
    x = torch.zeros((n, len(froms)), dtype=dtype, device=_dev())
    x[torch.as_tensor(np.asarray(froms)).to(x.device), torch.arange(len(froms), device=x.device)] = 1
    return x


def _gathered(ell, n, froms, rows, cols, M):
    """moments[l, m] = T_m(H/s)[rows[l], start cols[l]], by the recurrence."""
    x = _start(n, ell[1][0].dtype, froms)
    r, c = torch.as_tensor(np.asarray(rows)).to(x.device), torch.as_tensor(np.asarray(cols)).to(x.device)
    out = torch.zeros((M, len(rows)), dtype=x.dtype, device=x.device)
    out[0] = x[r, c]
    y = _apply(ell, x) * 0.5 if M > 1 else x
    for m in range(1, M):
        out[m] = y[r, c]
        if m + 1 < M:
            x, y = y, _apply(ell, y).sub_(x)
    return out.t().to(torch.complex128).cpu().numpy().copy()


def _doubled(ell, x, M):
    """moments[b, m] = <x_b|T_m|x_b> from half the recurrence."""
    def dot(a, b):
        return (a.conj() * b).sum(0)
    out = torch.zeros((M + 2, x.shape[1]), dtype=torch.complex128, device=x.device)
    y = _apply(ell, x) * 0.5
    mu0, mu1 = dot(x, x), dot(y, x)
    for n in range((M + 1) // 2):
        out[2 * n] = mu0 if n == 0 else 2 * dot(x, x) - mu0
        out[2 * n + 1] = mu1 if n == 0 else 2 * dot(y, x) - mu1
        x, y = y, _apply(ell, y).sub_(x)
    return out[:M].t().cpu().numpy().copy()


def _phases(n, R, seed):
    """exp(2 pi i u), u the 53-bit splitmix64 uniform of (seed, r n + i)."""
    with np.errstate(over="ignore"):
        c = np.arange(n * R, dtype=np.uint64)
        z = np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15) + c * np.uint64(0xD1B54A32D192ED03) + \
            np.uint64(0x632BE59BD9B4E019)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = (z >> np.uint64(11)).astype(np.float64) / 9007199254740992.0
    t = torch.from_numpy(u).to(_dev()).reshape(R, n).t().contiguous() * (2 * math.pi)
    return torch.complex(torch.cos(t), torch.sin(t))


def _contracted(c, gtype, E, scale, window):
    """G(E) of the moment vectors c, from the closed form of the expansion."""
    c = torch.from_numpy(np.ascontiguousarray(c)).to(_dev())
    M = c.shape[1]
    lo, hi = window
    x = (lo + torch.arange(E, dtype=torch.float64, device=c.device) * ((hi - lo) / (E - 1))) / scale
    th = torch.arange(M, dtype=torch.float64, device=c.device)[:, None] * torch.acos(x)[None, :]
    half = torch.ones(M, dtype=torch.float64, device=c.device)
    half[0] = 0.5
    pre = (2 / scale) / torch.sqrt(1 - x * x)
    cs = (c * half).contiguous()
    cos, sin = torch.cos(th).to(torch.complex128), torch.sin(th).to(torch.complex128)
    if gtype == X.PRINCIPAL:
        g = (cs @ sin) * pre
    elif gtype == X.NONPRINCIPAL:
        g = (cs @ cos) * (1j * pre)
    elif gtype == X.RETARDED:
        g = (cs @ (cos - 1j * sin)) * (-1j * pre)
    else:
        g = (cs @ (cos + 1j * sin)) * (1j * pre)
    return g.cpu().numpy()


def _lorentz(c):
    M = c.shape[1]
    lam = BROADENING * M
    return c * (np.sinh(lam * (1 - np.arange(M) / M)) / math.sinh(lam))[None, :]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("contract", "mfma", "direct"):
        return _contracted(_coefficients(case, seed), case["gtype"], case["E"], 6.0, _window(6.0))
    if kind == "uneven":
        specs, scales, sites, moments = _uneven(case, seed)
        out = []
        for i, (sp, sc, st, m) in enumerate(zip(specs, scales, sites, moments)):
            f = L.honeycomb_ribbon if sp.orbitals == 4 else L.square
            p = sp.params
            ell = _ell(f(p["lx"], p["ly"], disorder=0.5, seed=seed + i), sc)
            out.append(_doubled(ell, _start(sp.basis_size, ell[1][0].dtype, st), m))
        return out
    M, E, s = case["M"], case["E"], SCALE[case["model"]]
    ell = _ell(_builder(case, seed, False), s)
    n = _states(case)
    if kind == "ldos":
        out = {}
        for i, f in enumerate(_picked(case, seed)):
            c = _gathered(ell, n, [f], [f], [0], M)
            G = _contracted(_lorentz(c), X.NONPRINCIPAL, E, s, _window(s))
            out["c%d" % i], out["G%d" % i], out["ldos%d" % i] = c, G, G.imag.sum(0) / math.pi
        return out
    if kind == "green":
        f, to = _picked(case, seed)
        c = _gathered(ell, n, [f], to, [0] * len(to), M)
        return {"c": c, "G": _contracted(_lorentz(c), X.RETARDED, E, s, _window(s))}
    if kind == "multi":
        froms, tos = _picked(case, seed)
        c = _gathered(ell, n, froms, [t for ts in tos for t in ts],
                      [j for j, ts in enumerate(tos) for _ in ts], M)
        return {"c": c, "G": _contracted(_lorentz(c), X.NONPRINCIPAL, E, s, _window(s))}
    if kind == "block":
        c = _doubled(ell, _start(n, ell[1][0].dtype, _picked(case, seed)), M)
    else:
        ell = (ell[0], [v.to(torch.complex128) for v in ell[1]])
        c = _doubled(ell, _phases(n, case["vectors"], seed), M).sum(0)
    G = _contracted(np.atleast_2d(c) * _jackson(M)[None, :], X.NONPRINCIPAL, E, s, _window(s))
    return {"c": c, "G": G}
