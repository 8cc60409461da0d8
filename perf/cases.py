"""Timed cases of the framework's main paths, through its public entry points.

Kinds (the key "kind" of a case):

  mie      one sphere through the pymiecoated drop-in (Mie): efficiencies and
           S1, S2 at two angles, scalars in and out;
  coated   a device-resident batch of coated spheres through gm_mie_batch,
           with or without the stored a_n, b_n;
  chain    one step of the runoptics chain (RunopticsChain): Mie, S1/S2, size
           integration, P normalisation and optionally the GSF moments, at
           FP64 or a reduced S1/S2 precision, eager or replayed as a graph;
  lut      bulk rows of a batch of LUT slabs (LutSweep.run), with the sweep's
           40 shared size distributions or each slab's own;
  predict  surrogate rows and gate flags of n queries (Surrogate.predict);
  train    one training step of the surrogate network (gradient and Adam);
  table    a whole runoptics table from a particle description (build_table).

Grids and ranges are those of bench.py, the tests and the LUT sweep.
"""
import math
import os

import numpy as np
import torch

ANG_TABLE = 371     # angles of a runoptics table
N_R = 3000          # dry radii of the LUT sweep
CORE = 1.95 + 0.79j  # black-carbon core of the coated batches
DIMS = (6, 256, 256, 256, 256, 35)


def listed():
    return [
        # one particle at a time, as an interactive user or a per-particle loop calls it
        {"name": "mie_one_sphere", "kind": "mie", "x": 23.7, "coated": False},
        # a small device batch: latency and launches count
        {"name": "coated_1266_points", "kind": "coated", "n_r": 211, "n_lam": 3, "n_ratio": 2,
         "n_shell": 1, "coeffs": False},
        # the framework's headline batch: efficiencies of 8.4M coated spheres
        {"name": "coated_8.4m_points", "kind": "coated", "n_r": 5000, "n_lam": 20, "n_ratio": 7,
         "n_shell": 12, "coeffs": False},
        # the same particles for a caller that goes on to S1/S2: a_n, b_n stored
        {"name": "coated_1.05m_coefficients", "kind": "coated", "n_r": 1250, "n_lam": 20,
         "n_ratio": 7, "n_shell": 6, "coeffs": True},
        # one runoptics size grid, 10 wavelengths, replayed in a serving loop
        {"name": "chain_20k_181_fp64_graph", "kind": "chain", "n_r": 2000, "n_lam": 10,
         "r_lo": 0.005, "r_hi": 20.0, "lam_lo": 0.3, "lam_hi": 2.5, "n_ang": 181, "prec": 0,
         "ng": 0, "mixed": False, "graph": True},
        # large spheres (dust, cloud) at a fine angle grid, with GSF moments
        {"name": "chain_40k_1801_fp64", "kind": "chain", "n_r": 5000, "n_lam": 8, "r_lo": 0.1,
         "r_hi": 100.0, "lam_lo": 0.3, "lam_hi": 1.0, "n_ang": 1801, "prec": 0, "ng": 300,
         "mixed": True, "graph": False},
        # the same spheres at the fastest S1/S2 precision
        {"name": "chain_40k_1801_bf16x3", "kind": "chain", "n_r": 5000, "n_lam": 8, "r_lo": 0.1,
         "r_hi": 100.0, "lam_lo": 0.3, "lam_hi": 1.0, "n_ang": 1801, "prec": 2, "ng": 0,
         "mixed": True, "graph": False},
        # one batch of the LUT sweep: shared size distributions, FP64
        {"name": "lut_400_slabs_fp64", "kind": "lut", "n_slab": 400, "n_psd": 0, "prec": "fp64"},
        # the surrogate's plain re-solve: one size distribution per slab, FP32 S1/S2
        {"name": "lut_512_queries_fp32", "kind": "lut", "n_slab": 512, "n_psd": 1, "prec": "fp32"},
        # serving a million surrogate queries
        {"name": "predict_1m", "kind": "predict", "n": 1000000},
        # a training step of the surrogate at its default batch
        {"name": "train_16384", "kind": "train", "n": 16384},
        # a whole organic-carbon-like table with its GSF moments
        {"name": "table_oc_61x36", "kind": "table", "n_lam": 61, "n_rh": 36, "per_decade": 800,
         "n_mom": 129},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["mie", "coated", "chain", "chain", "lut", "lut", "predict", "train",
                       "table"])
    if kind == "mie":
        return {"kind": kind, "x": round(math.exp(rng.uniform(math.log(0.05), math.log(900.0))), 4),
                "coated": rng.random() < 0.5}
    if kind == "coated":
        return {"kind": kind, "n_r": log_int(1, 2500), "n_lam": rng.randint(1, 20),
                "n_ratio": rng.randint(1, 7), "n_shell": rng.randint(1, 6),
                "coeffs": rng.random() < 0.5}
    if kind == "chain":
        prec = rng.choice([0, 0, 1, 2])
        return {"kind": kind, "n_r": log_int(60, 5000), "n_lam": rng.randint(1, 8),
                "r_lo": 0.005, "r_hi": round(math.exp(rng.uniform(0.0, math.log(100.0))), 3),
                "lam_lo": 0.3, "lam_hi": rng.choice([1.0, 2.5]),
                "n_ang": rng.choice([19, 91, 181, 361, log_int(50, 1801), 1801]), "prec": prec,
                "ng": 0 if prec else rng.choice([0, 129, 300]), "mixed": rng.random() < 0.5,
                "graph": rng.random() < 0.3}
    if kind == "lut":
        return {"kind": kind, "n_slab": log_int(1, 400), "n_psd": rng.choice([0, 0, 1, 3]),
                "prec": rng.choice(["fp64", "fp32"])}
    if kind == "predict":
        return {"kind": kind, "n": log_int(1, 1000000)}
    if kind == "train":
        return {"kind": kind, "n": log_int(100, 16384)}
    return {"kind": kind, "n_lam": rng.randint(3, 40), "n_rh": rng.randint(2, 36),
            "per_decade": log_int(60, 800), "n_mom": rng.choice([0, 129])}


# ---- inputs ---------------------------------------------------------------


def _mie_args(case, seed):
    """(x, m, y, m2) of one sphere; y, m2 None when it has no shell."""
    rng = np.random.default_rng([1, seed])
    size = case["x"] * rng.uniform(0.99, 1.01)
    if not case["coated"]:
        return size, complex(rng.uniform(1.33, 1.6), 10 ** rng.uniform(-6, -1)), None, None
    return size * rng.uniform(0.3, 0.9), CORE, size, complex(rng.uniform(1.33, 1.45))


def _coated_axes(case, seed):
    """The product grid's axes: radii and wavelengths (um; the same for every
    seed, so that stored coefficients keep their length), core/shell ratios,
    real shell indices mixed with water by the growth factor."""
    rng = np.random.default_rng([2, seed])
    r = np.logspace(-2, 1, case["n_r"]) if case["n_r"] > 1 else np.array([1.0])
    lam = np.linspace(0.3, 3.0, case["n_lam"])
    ratio = np.linspace(0.3, 0.9, case["n_ratio"]) + rng.uniform(-0.02, 0.02, case["n_ratio"])
    gf = np.linspace(1.0, 2.5, case["n_shell"])
    shell = 1.33 + (1.45 + rng.uniform(-0.01, 0.01) - 1.33) / gf ** 3
    core = CORE + complex(rng.uniform(-0.02, 0.02), rng.uniform(-0.02, 0.02))
    return r, lam, ratio, shell, core


def _coated_points(case, seed):
    """x, y [n] and the shell index m2 [n] (device), points ordered
    [shell][ratio][wavelength][radius], and the core index."""
    r, lam, ratio, shell, core = _coated_axes(case, seed)
    f = {"dtype": torch.float64, "device": "cuda"}
    yy = (2 * np.pi * torch.tensor(r, **f)[None, :] / torch.tensor(lam, **f)[:, None]).reshape(-1)
    shape = (shell.size, ratio.size, yy.numel())
    y = yy.expand(shape).reshape(-1).contiguous()
    x = (torch.tensor(ratio, **f)[:, None] * yy[None, :]).expand(shape).reshape(-1).contiguous()
    m2 = torch.tensor(shell, **f)[:, None, None].expand(shape).reshape(-1).contiguous()
    return x, y, m2, core


def _chain_args(case, seed):
    """x [n], m (scalar or [n]), angles, number weights [rows][n], wavelengths."""
    rng = np.random.default_rng([3, seed])
    n_r, n_lam = case["n_r"], case["n_lam"]
    r = np.logspace(math.log10(case["r_lo"]), math.log10(case["r_hi"]), n_r) * rng.uniform(0.99, 1)
    lam = np.linspace(case["lam_lo"], case["lam_hi"], n_lam)
    x = (2 * np.pi * r[None, :] / lam[:, None]).ravel()
    if case["mixed"]:
        m = rng.uniform(1.33, 1.60, x.size) + 1j * 10 ** rng.uniform(-6, -2, x.size)
    else:
        m = complex(1.53 + rng.uniform(-0.02, 0.02), 0.005 * rng.uniform(0.8, 1.2))
    mode = math.sqrt(case["r_lo"] * case["r_hi"]) * rng.uniform(1.4, 1.6)
    p = np.exp(-np.log(r / mode) ** 2 / (2 * math.log(2.0) ** 2)) / r * np.gradient(r)
    w = np.zeros((n_lam, x.size))
    for i in range(n_lam):
        w[i, i * n_r:(i + 1) * n_r] = p / p.sum()
    return x, m, np.linspace(0.0, 180.0, case["n_ang"]), w, lam


def _lut_args(case, seed):
    """lam, m_dry, gf of the slabs: wavelengths spread over 0.2-40 um in
    shuffled strata, the other axes uniform in the sweep's ranges."""
    from geosmie_amd.lut_sweep import SU_GF
    rng = np.random.default_rng([4, seed])
    n = case["n_slab"]
    u = (np.arange(n) + rng.uniform(0.3, 0.7, n)) / n
    lam = 0.2 * (40.0 / 0.2) ** rng.permutation(u)
    m = rng.uniform(1.30, 1.80, n) + 1j * 10 ** rng.uniform(-8, 0, n)
    return lam, m, SU_GF[rng.permutation(n) % SU_GF.size]


def _queries(n, seed):
    """Surrogate queries uniform in the sweep's ranges, float32 [n, 6]."""
    from geosmie_amd.surrogate import make_queries
    rng = np.random.default_rng([5, seed])
    gf = (1 - rng.uniform(0, 1 - 2.16 ** -3.0, n)) ** (-1.0 / 3.0)
    return make_queries(np.exp(rng.uniform(math.log(0.01), math.log(5.0), n)),
                        rng.uniform(1.4, 2.6, n), rng.uniform(1.30, 1.80, n),
                        np.exp(rng.uniform(math.log(1e-8), 0.0, n)),
                        np.exp(rng.uniform(math.log(0.2), math.log(40.0), n)), gf)


def _model_file():
    import geosmie_amd
    return os.path.join(os.path.dirname(geosmie_amd.__file__), "data", "surrogate_lut.npz")


def _table_args(case, seed):
    """An organic-carbon-like particle (one lognormal bin) and a water table."""
    rng = np.random.default_rng([6, seed])
    lam = np.geomspace(0.25e-6, 40.0e-6, case["n_lam"])
    mr = 1.53 + rng.uniform(-0.02, 0.02) - 0.05 * np.log(lam / 1e-6) / np.log(40.0)
    mi = -(0.005 * rng.uniform(0.8, 1.2) + 0.05 * (lam / 40e-6))
    rh = np.linspace(0.0, 0.99, case["n_rh"])
    par = {"rhop0": 1800.0, "rh": list(rh),
           "rhDep": {"type": "simple", "params": {"gf": list(1.0 + 1.52 * rh ** 4)}},
           "psd": {"type": "lognorm", "params": {
               "r0": [[0.0212e-6]], "rmax0": [[0.3e-6]], "rmin0": [[1e-10]], "sigma": [[2.20]],
               "numperdec": [case["per_decade"]], "fracs": [[1.0]]}},
           "mList": [np.array([lam, mr, mi])]}
    wl = np.linspace(0.2e-6, 45e-6, 60)
    return par, np.array([wl, 1.33 + 0.0 * wl, 1e-8 + 0.3 * (wl / 45e-6)])


# ---- prepare and run ------------------------------------------------------


def prepare(case, seed):
    from geosmie_amd import _lib
    st = {"case": case}
    kind = case["kind"]
    if kind == "mie":
        x, m, y, m2 = _mie_args(case, seed)
        st["args"] = {"m": m, "x": x} if y is None else {"m": m, "x": x, "m2": m2, "y": y}
    elif kind == "coated":
        x, y, m2, core = _coated_points(case, seed)
        n = x.numel()
        eps = torch.empty((n, 2), dtype=torch.float64, device="cuda")
        eps[:, 0], eps[:, 1] = (core * core).real, (core * core).imag
        eps2 = torch.zeros((n, 2), dtype=torch.float64, device="cuda")
        eps2[:, 0] = m2 * m2
        st.update(n=n, x=x, y=y, eps=eps, eps2=eps2, size_max=float(y.max()),
                  ctx=_lib.private_ctx(),
                  props=torch.empty((6, n), dtype=torch.float64, device="cuda"))
        if case["coeffs"]:
            total = int(_nmax(y).sum())
            st["off"] = torch.empty(n + 1, dtype=torch.int64, device="cuda")
            st["an"] = torch.empty((total, 2), dtype=torch.float64, device="cuda")
            st["bn"] = torch.empty((total, 2), dtype=torch.float64, device="cuda")
    elif kind == "chain":
        from geosmie_amd.pipeline import RunopticsChain
        x, m, ang, w, lam = _chain_args(case, seed)
        n_r = case["n_r"]
        st["chain"] = RunopticsChain(x, m, ang, w, lam,
                                     [(i * n_r, n_r) for i in range(case["n_lam"])],
                                     precision=case["prec"], gsf_ng=case["ng"])
        if case["graph"]:
            st["chain"].capture()
    elif kind == "lut":
        from geosmie_amd.lut_sweep import LutSweep, full_grid
        g = full_grid()
        st["lam"], st["m"], st["gf"] = _lut_args(case, seed)
        st["w"] = None
        if case["n_psd"]:
            st["sweep"] = LutSweep(g["r"], rmode=[1.0], sigma=[2.0], precision=case["prec"])
            rng = np.random.default_rng([7, seed])
            k = case["n_slab"] * case["n_psd"]
            st["w"] = st["sweep"].weights_dev(np.exp(rng.uniform(np.log(0.01), np.log(5.0), k)),
                                              rng.uniform(1.4, 2.6, k))
        else:
            st["sweep"] = LutSweep(g["r"], g["rmode"], g["sigma"], precision=case["prec"])
    elif kind == "predict":
        from geosmie_amd.surrogate import Surrogate
        st["sur"] = Surrogate.load(_model_file())
        st["q"] = torch.from_numpy(_queries(case["n"], seed)).cuda()
    elif kind == "train":
        st["X"], st["Y"], st["cw"], st["mlp"] = _train_args(case, seed)
    elif kind == "table":
        st["params"], st["water"] = _table_args(case, seed)
    return st


def _train_args(case, seed):
    """Standardised features and targets of one minibatch (the committed
    network's rows with 1% noise stand for the sweep's), the loss weights and
    a network at the start of its training."""
    from geosmie_amd.surrogate import MLP, N_OUT, Surrogate, training_arrays
    sur = Surrogate.load(_model_file())
    q = _queries(case["n"], seed)
    rows, _ = sur.predict(q)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rows *= 1 + 0.01 * torch.randn(rows.shape, generator=gen, device="cuda")
    X, Y = training_arrays(sur, q, rows)
    cw = np.ones(N_OUT, np.float32)
    cw[:3] = 1000.0
    cw[3] = 0.0
    mlp = MLP(DIMS, params=_train_params(seed), weight_terms=2)
    return X, Y, torch.from_numpy(cw / cw.sum() * N_OUT).cuda(), mlp


def _train_params(seed):
    """Initial parameters: uniform weights of variance 2 / fan_in (1 / fan_in
    in the last layer), zero biases."""
    rng = np.random.default_rng([8, seed])
    out = []
    for i, o in zip(DIMS, DIMS[1:]):
        a = math.sqrt((6.0 if o != DIMS[-1] else 3.0) / i)
        out += [rng.uniform(-a, a, i * o), np.zeros(o)]
    return np.concatenate(out).astype(np.float32)


def run(st):
    from geosmie_amd import _lib
    kind = st["case"]["kind"]
    if kind == "mie":
        from geosmie_amd import Mie
        p = Mie(**st["args"])
        q = [p.qext(), p.qsca(), p.qabs(), p.qb(), p.asy(), p.qratio()]
        return np.array(q), np.array([p.S12(1.0), p.S12(-0.5)])
    if kind == "coated":
        lib, P, s = _lib.lib(), _lib.ptr, _lib.stream()
        off, an, bn = st.get("off"), st.get("an"), st.get("bn")
        if off is not None:
            _lib.check(lib.gm_coef_offsets(st["ctx"], st["n"], P(st["y"]), P(off), s),
                       "gm_coef_offsets")
        _lib.check(lib.gm_mie_batch(st["ctx"], st["n"], P(st["x"]), P(st["y"]), P(st["eps"]), None,
                                    P(st["eps2"]), st["size_max"], P(off), P(an), P(bn),
                                    P(st["props"]), None, _lib.GM_MIE_SORT, s), "gm_mie_batch")
        return {"props": st["props"]} if off is None else {"props": st["props"], "an": an, "bn": bn}
    if kind == "chain":
        c = st["chain"]
        if c.graph is not None:
            c.replay()
        else:
            c.step()
        out = {"pmat": c.d_pm, "pback": c.d_back, "scalars": c.d_sc, "props": c.d_props}
        if c.gsf_ng:
            out["pmom"] = c.d_pmom
        return out
    if kind == "lut":
        return st["sweep"].run(st["lam"], st["m"], st["gf"], w=st["w"])
    if kind == "predict":
        rows, flags = st["sur"].predict(st["q"])
        return {"rows": rows, "flags": flags}
    if kind == "train":
        mlp = st["mlp"]
        mlp.grad(st["X"], st["Y"], st["cw"])
        mlp.adam(4e-6)      # the first step of the warmup to 2e-3
        return {"loss": mlp.loss, "grads": mlp.g, "params": mlp.p}
    from geosmie_amd.runoptics import build_table
    return build_table(st["params"], water=st["water"], n_mom=st["case"]["n_mom"]).data


# ---- work -----------------------------------------------------------------


def _nmax(s):
    """n_max = round(2 + s + 4 s^(1/3)) of sizes s (numpy or torch)."""
    v = 2 + s + 4 * s ** (1.0 / 3.0)
    return (torch.round(v) if isinstance(v, torch.Tensor) else np.rint(v))


def work(case):
    """Bytes: inputs once and outputs once.  Flops: per point 10 per D_n step
    (three chains when coated) and 70 per series term; 8 per series term and
    angle (real U P and V M products); 2 per multiply-add of the size
    integration, the GSF products and the network."""
    kind = case["kind"]
    if kind == "mie":
        n = float(_nmax(case["x"]))
        return {"bytes": 48.0 + 64.0 + 80.0, "flops": 100 * n + 16 * n}
    if kind == "coated":
        r, lam, ratio, shell, core = _coated_axes(case, 0)
        y = (2 * np.pi * r[None, :] / lam[:, None]).ravel()
        reps = ratio.size * shell.size
        nm = _nmax(y)
        nmx = np.rint(np.maximum(nm, abs(core) * y) + 16)
        return {"bytes": float(reps) * (96.0 * y.size + (32 * float(nm.sum()) if case["coeffs"] else 0)),
                "flops": float(reps * (30 * nmx + 70 * nm).sum())}
    if kind == "chain":
        x, m, ang, w, lam = _chain_args(case, 0)
        nm = _nmax(x)
        nmx = np.rint(np.maximum(nm, np.abs(m) * x) + 16)
        rows, na, ng = lam.size, ang.size, case["ng"]
        return {"bytes": 8.0 * (3 * x.size + x.size + 2 * float(nm.max()) * na + 6 * x.size
                                + rows * (4 * na + 22 + 6 * ng)),
                "flops": float((10 * nmx + 70 * nm).sum() + 8 * nm.sum() * na
                               + 8 * x.size * na + rows * 12.0 * na * ng)}
    if kind == "lut":
        lam, m, gf = _lut_args(case, 0)
        r = np.logspace(math.log10(0.005), math.log10(50.0), N_R)
        nm = sum(float(_nmax(2 * np.pi * g * r / L).sum()) for L, g in zip(lam, gf))
        n_psd = case["n_psd"] or 40
        w = 8.0 * N_R * n_psd * (case["n_slab"] if case["n_psd"] else 1)
        return {"bytes": w + case["n_slab"] * (32.0 + 140 * n_psd),
                "flops": 80 * nm + 8 * nm * ANG_TABLE
                + 2.0 * case["n_slab"] * n_psd * N_R * (ANG_TABLE + 4)}
    macs = float(sum(a * b for a, b in zip(DIMS, DIMS[1:])))
    if kind == "predict":
        return {"bytes": case["n"] * (24.0 + 140 + 4) + 4 * macs, "flops": 2 * macs * case["n"]}
    if kind == "train":
        return {"bytes": case["n"] * (24.0 + 140) + 4 * macs * 8, "flops": 6 * macs * case["n"]}
    n_x = 3.9 * case["per_decade"]              # grid points over about four decades
    x = np.geomspace(2e-5, 19.0, max(2, int(n_x)))
    nm = float(_nmax(x).sum())
    ent = case["n_lam"] * case["n_rh"]
    return {"bytes": ent * 8.0 * (6 * ANG_TABLE + 30 + 6 * case["n_mom"]),
            "flops": ent * (nm * (80 + 8 * ANG_TABLE) + 8 * n_x * ANG_TABLE
                            + 12.0 * ANG_TABLE * case["n_mom"])}


# ---- the same outputs in plain 64-bit torch --------------------------------


def _riccati(x, N):
    """psi, chi [N + 2][len(x)] of orders -1..N at real x: both upward, psi above
    n = x by the downward ratio psi_n / psi_{n-1}."""
    psi = torch.empty((N + 2,) + x.shape, dtype=x.dtype, device=x.device)
    chi = torch.empty_like(psi)
    psi[0], psi[1], chi[0], chi[1] = torch.cos(x), torch.sin(x), -torch.sin(x), torch.cos(x)
    top = max(N, int(x.max())) + 24 + int(8 * float(x.max()) ** (1.0 / 3.0))
    r = torch.zeros_like(x)
    for n in range(top, 0, -1):
        r = 1.0 / ((2 * n + 1) / x - r)
        if n <= N:
            psi[n + 1] = r
    for n in range(1, N + 1):
        up = (2 * n - 1) / x * psi[n] - psi[n - 1]
        psi[n + 1] = torch.where(x >= n, up, psi[n + 1] * psi[n])
        chi[n + 1] = (2 * n - 1) / x * chi[n] - chi[n - 1]
    return psi, chi


def _log_derivative(z, nmx, N):
    """D_n(z), n = 1..N, downward from D_nmx = 0 ([N + 1][len(z)])."""
    out = torch.zeros((N + 1,) + z.shape, dtype=z.dtype, device=z.device)
    d = torch.zeros_like(z)
    for n in range(int(nmx.max()), 1, -1):
        q = n / z
        d = torch.where(n <= nmx, q - 1.0 / (d + q), d)
        if n - 1 <= N:
            out[n - 1] = d
    return out


def _coefficients(x, m, y=None, m2=None):
    """a_n, b_n [N][points] (zero above each point's n_max) and n_max: spheres of
    index m and size x, or with a real shell m2 out to y (Bohren and Huffman,
    Absorption and Scattering of Light by Small Particles, eqs. 4.88, 8.2)."""
    size = x if y is None else y
    nm = _nmax(size)
    N = int(nm.max())
    big = torch.abs(m) * size if y is None else torch.maximum(torch.abs(m), m2) * size
    nmx = torch.round(torch.maximum(nm, big) + 16)
    D = _log_derivative(m * x, nmx, N)
    psi, chi = _riccati(size, N)
    if y is not None:
        pv, cv = _riccati(m2 * x, N)
        pw, cw = _riccati(m2 * y, N)
    an = torch.zeros((N,) + x.shape, dtype=torch.complex128, device=x.device)
    bn = torch.zeros_like(an)
    for n in range(1, N + 1):
        p1, p, c1, c = psi[n], psi[n + 1], chi[n], chi[n + 1]
        xi, xi1 = torch.complex(p, -c), torch.complex(p1, -c1)
        if y is None:
            da, db = D[n] / m + n / x, D[n] * m + n / x
        else:
            v, w = m2 * x, m2 * y
            dpv, dcv = pv[n] - n / v * pv[n + 1], cv[n] - n / v * cv[n + 1]
            dpw, dcw = pw[n] - n / w * pw[n + 1], cw[n] - n / w * cw[n + 1]
            A = (m2 * D[n] * pv[n + 1] - m * dpv) / (m2 * D[n] * cv[n + 1] - m * dcv)
            B = (m * D[n] * pv[n + 1] - m2 * dpv) / (m * D[n] * cv[n + 1] - m2 * dcv)
            da = (dpw - A * dcw) / (pw[n + 1] - A * cw[n + 1]) / m2 + n / y
            db = (dpw - B * dcw) / (pw[n + 1] - B * cw[n + 1]) * m2 + n / y
        live = n <= nm
        an[n - 1] = torch.where(live, (da * p - p1) / (da * xi - xi1), 0)
        bn[n - 1] = torch.where(live, (db * p - p1) / (db * xi - xi1), 0)
    return an, bn, nm


def _efficiencies(an, bn, size):
    """qext, qsca, qabs, qb, asy, qratio [6][points]."""
    n = torch.arange(1, an.shape[0] + 1, dtype=torch.float64, device=an.device)[:, None]
    c = 2 * n + 1
    s2 = size ** 2
    qext = 2 * (c * (an.real + bn.real)).sum(0) / s2
    qsca = 2 * (c * (an.abs() ** 2 + bn.abs() ** 2)).sum(0) / s2
    q = (c * (1 - 2 * (n % 2)) * (an - bn)).sum(0)
    qb = q.abs() ** 2 / s2
    pair = (an[:-1] * an[1:].conj() + bn[:-1] * bn[1:].conj()).real
    asy = (n * (n + 2) / (n + 1))[:-1] * pair
    asy = asy.sum(0) + (c / (n * (n + 1)) * (an * bn.conj()).real).sum(0)
    return torch.stack([qext, qsca, qext - qsca, qb, 4 / s2 * asy / qsca, qb / qsca])


def _angle_rows(mu, N):
    """pi_n, tau_n times (2n + 1) / (n (n + 1)), [N][angles]."""
    p = torch.zeros((N + 1, mu.numel()), dtype=torch.float64, device=mu.device)
    t = torch.zeros_like(p)
    p[1] = 1.0
    for n in range(1, N + 1):
        if n > 1:
            p[n] = ((2 * n - 1) * mu * p[n - 1] - n * p[n - 2]) / (n - 1)
        t[n] = n * mu * p[n] - (n + 1) * p[n - 1]
    k = torch.arange(1, N + 1, dtype=torch.float64, device=mu.device)[:, None]
    f = (2 * k + 1) / (k * (k + 1))
    return p[1:] * f, t[1:] * f


def _amplitudes(an, bn, P, T):
    """S1, S2 [angles][points]."""
    P, T = P[:an.shape[0]].t().contiguous(), T[:an.shape[0]].t().contiguous()

    def mul(R, c):
        return torch.complex(R @ c.real.contiguous(), R @ c.imag.contiguous())
    return mul(P, an) + mul(T, bn), mul(T, an) + mul(P, bn)


def _chunks(size, most=1 << 62, terms=1.5e7):
    """Index tensors of at most `most` points with similar series lengths, of
    bounded work."""
    order = torch.argsort(size, descending=True)
    nm = _nmax(size)
    a = 0
    while a < order.numel():
        k = min(most, max(1, int(terms / float(nm[order[a]]))))
        yield order[a:a + k]
        a += k


def exact(case, seed):
    kind = case["kind"]
    f = {"dtype": torch.float64, "device": "cuda"}
    if kind == "mie":
        x, m, y, m2 = _mie_args(case, seed)
        tx, tm = torch.tensor([x], **f), torch.tensor([m], dtype=torch.complex128, device="cuda")
        if y is None:
            an, bn, _ = _coefficients(tx, tm)
        else:
            an, bn, _ = _coefficients(tx, tm, torch.tensor([y], **f),
                                      torch.tensor([m2.real], **f))
        q = _efficiencies(an, bn, tx if y is None else torch.tensor([y], **f))
        P, T = _angle_rows(torch.tensor([1.0, -0.5], **f), an.shape[0])
        s1, s2 = _amplitudes(an, bn, P, T)
        return q[:, 0].cpu().numpy(), torch.stack([s1[:, 0], s2[:, 0]], 1).cpu().numpy()
    if kind == "coated":
        x, y, m2, core = _coated_points(case, seed)
        out = {"props": torch.empty((6, x.numel()), **f)}
        m = torch.tensor(core, dtype=torch.complex128, device="cuda")
        if case["coeffs"]:
            off = torch.cumsum(_nmax(y), 0) - _nmax(y)
            total = int(_nmax(y).sum())
            out["an"], out["bn"] = torch.empty((total, 2), **f), torch.empty((total, 2), **f)
        for i in _chunks(y):
            an, bn, nm = _coefficients(x[i], m.expand(i.numel()), y[i], m2[i])
            out["props"][:, i] = _efficiencies(an, bn, y[i])
            if case["coeffs"]:
                n = torch.arange(an.shape[0], device="cuda")[:, None]
                live = n < nm
                at = (off[i] + n)[live].long()
                out["an"][at] = torch.view_as_real(an[live])
                out["bn"][at] = torch.view_as_real(bn[live])
        return out
    if kind == "chain":
        return _exact_chain(case, seed)
    if kind == "predict":
        return {"rows": _exact_rows(case, seed), "flags": None}
    if kind == "train":
        return _exact_train(case, seed)
    # lut, table: whole sweeps and tables take longer than this is worth; their layers
    # (Mie, S1/S2, the size integration) are the chain's
    return None


def _exact_chain(case, seed):
    f = {"dtype": torch.float64, "device": "cuda"}
    x, m, ang, w, lam = _chain_args(case, seed)
    tx = torch.tensor(x, **f)
    tm = torch.tensor(np.broadcast_to(m, x.shape).copy(), dtype=torch.complex128, device="cuda")
    tw = torch.tensor(w, **f)
    rows, na, n_r = lam.size, ang.size, case["n_r"]
    props = torch.empty((6, x.size), **f)
    pm = torch.zeros((rows, 4, na), **f)
    P, T = _angle_rows(torch.tensor(np.cos(np.radians(ang)), **f), int(_nmax(tx).max()))
    for i in _chunks(tx, most=8000):
        an, bn, _ = _coefficients(tx[i], tm[i])
        props[:, i] = _efficiencies(an, bn, tx[i])
        s1, s2 = _amplitudes(an, bn, P, T)
        a1, a2, c = s1.abs() ** 2, s2.abs() ** 2, s1 * s2.conj()
        for e, v in enumerate(((a1 + a2) / 2, (a2 - a1) / 2, c.real, c.imag)):
            pm[:, e] += tw[:, i] @ v.t().contiguous()
    th = torch.tensor(np.radians(ang), **f)
    g = pm[:, 0] * torch.sin(th)
    pm *= 2 / (0.5 * (g[:, 1:] + g[:, :-1]) * (th[1:] - th[:-1])).sum(1)[:, None, None]
    back = pm[:, [0, 1, 2, 3, 0, 2], -1]
    sc = torch.empty((rows, 16), **f)
    rho = 1000.0
    for r in range(rows):
        k = slice(r * n_r, (r + 1) * n_r)
        rr, ww, q = tx[k] * float(lam[r]) / (2 * math.pi), tw[r, k], props[:, k]
        num, S2, S3, S4 = (float((rr ** e * ww).sum()) for e in (0, 2, 3, 4))
        aw = ww * rr ** 2
        qext, qsca, qabs, qb = (float((aw * q[e]).sum()) / S2 for e in range(4))
        sw = aw * q[1]
        g_, cs, ce = (float((sw * v).sum() / sw.sum())
                      for v in (q[4], q[1] * math.pi * rr ** 2, q[0] * math.pi * rr ** 2))
        vol, reff, rm = 4 / 3 * math.pi * S3 / num, S3 / S2, S4 / S3
        rmass = 4 / 3 * math.pi * rho * rm ** 3
        mc = 1 / rho / reff * rmass / rmass      # the mass of the dry particle is the same
        sc[r] = torch.tensor([num, math.pi * S2 / num, vol, vol * rho, reff, rmass, qext, qsca,
                              qabs, qb, g_, cs, ce, 0.75 * qsca * mc, 0.75 * qext * mc,
                              0.75 * qb * mc / (4 * math.pi)], **f)
    out = {"pmat": pm.reshape(-1), "pback": back.reshape(-1), "scalars": sc.reshape(-1),
           "props": props.reshape(-1)}
    if case["ng"]:
        out["pmom"] = None
    return out


def _model():
    return {k: torch.tensor(v, device="cuda").double() for k, v in
            np.load(_model_file()).items() if v.dtype.kind == "f"}


def _network(p, a):
    """The network of parameters p (FP64) at inputs a."""
    at = 0
    for k, (i, o) in enumerate(zip(DIMS, DIMS[1:])):
        W, b = p[at:at + i * o].view(o, i), p[at + i * o:at + i * o + o]
        at += i * o + o
        a = a @ W.t() + b
        if k < len(DIMS) - 2:
            a = a * torch.sigmoid(a)
    return a


def _features(q, z):
    """Standardised network features of queries, and ln B, the saturated bulk
    Rayleigh extinction that scales Qext."""
    dry = 1 - q[:, 5]
    lx = q[:, 0] - torch.log(q[:, 4]) + math.log(2 * math.pi)
    mr, mi = 1.33 + (q[:, 2] - 1.33) * dry, torch.exp(q[:, 3]) * dry
    x = torch.stack([lx, q[:, 1], mr, torch.log(mi), -torch.log(dry) / 3 - torch.log(q[:, 4]),
                     q[:, 5]], 1)
    m = torch.complex(mr, mi)
    K = (m * m - 1) / (m * m + 2)
    Q = (8 / 3 * K.abs() ** 2 * torch.exp(4 * lx + 6 * torch.log(q[:, 1]) ** 2)
         + 4 * K.imag * torch.exp(lx))
    return (x - z["feat_mean"]) / z["feat_std"], torch.log(Q) - torch.log1p(Q / 2)


def _exact_rows(case, seed):
    z = _model()
    q = torch.from_numpy(_queries(case["n"], seed)).cuda().double()
    out = []
    for part in q.split(100000):
        x, lnb = _features(part, z)
        t = _network(z["params"], x) * z["tgt_std"] + z["tgt_mean"]
        l2 = 2 * torch.arange(t.shape[1] - 3, device="cuda") + 1
        out.append(torch.cat([torch.exp(t[:, :1] + lnb[:, None]),
                              torch.exp(t[:, 1:2]).clamp(max=1.0), torch.exp(t[:, 2:3]),
                              t[:, 3:] * l2], 1))
    return torch.cat(out)


def _exact_train(case, seed):
    X, Y, cw, _ = _train_args(case, seed)
    p = torch.from_numpy(_train_params(seed)).cuda().double().requires_grad_(True)
    loss = (((_network(p, X.double()) - Y.double()) ** 2).mean(0) * cw.double()).sum()
    loss.backward()
    return {"loss": loss.detach().reshape(1), "grads": p.grad, "params": None}
