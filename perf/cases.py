"""The work that a program gives this library, as cases that can be timed and checked.

Every analysis entry point is covered over the range that it is used on: the
smallest calls (a Lorenz-96 teaching setup, the tutorial grid), regional and
global analyses of ordinary size, the full global workload, and the passes
around the analysis (forecast, verification, training of the learned
inflation).  Inputs follow the paths' real statistics: correlated Gaussian
background fields, observations drawn from a truth with their own error
variances, device-resident ensembles except where a host program owns small
arrays.

An analysis updates its ensemble in place, so a pass first puts the
background into the ensemble's buffer (the forecast's role in a cycled
program), ordered on the library's stream.
"""
import math

import numpy as np
import torch

import metada_amd as mda
from metada_amd import _lib as L
from metada_amd import learned

DEV = "cuda:0"
EARTH_KM = 6371.0
PREC = {"fp64": L.PREC_FP64, "fp32": L.PREC_FP32, "bf16x3": L.PREC_BF16X3}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the one-step stochastic EnKF on a 40-variable Lorenz-96 ring, host
        # arrays: the smallest call, where launches and copies count
        {"name": "enkf_l96_k20", "kind": "enkf", "nx": 40, "ny": 1, "k": 20, "p": 20,
         "rvar": "constant", "host": True},
        # the tutorial's grid and ensemble with the reference's own LETKF
        # semantics, host arrays
        {"name": "letkf_tutorial_k9", "kind": "letkf", "coord": "grid", "nx": 36, "ny": 18,
         "nlev": 1, "k": 9, "p": 28, "radius": 6.0, "prec": "fp64", "form": "refcompat",
         "host": True},
        # one cycle of the Lorenz-96 twin experiment (N = 4000, k = 40, every
        # second variable): ensemble forecast, then the LETKF
        {"name": "cycle_l96_k40", "kind": "cycle", "N": 4000, "k": 40, "every": 2,
         "support": 16.0, "steps": 1},
        # global analysis of moderate resolution in FP64
        {"name": "letkf_global_k40_fp64", "kind": "letkf", "coord": "geo", "nx": 256, "ny": 128,
         "nlev": 20, "k": 40, "p": 40000, "radius": 1000.0, "prec": "fp64", "form": "standard",
         "host": False},
        # the full global workload, 1024 x 512 x 40, a million observations
        {"name": "letkf_global_k64_bf16x3", "kind": "letkf", "coord": "geo", "nx": 1024,
         "ny": 512, "nlev": 40, "k": 64, "p": 1000000, "radius": 500.0, "prec": "bf16x3",
         "form": "standard", "host": False},
        # a regional domain in grid coordinates with the 50 members of an
        # operational-size ensemble
        {"name": "letkf_regional_k50_fp64", "kind": "letkf", "coord": "grid", "nx": 200,
         "ny": 160, "nlev": 30, "k": 50, "p": 30000, "radius": 10.0, "prec": "fp64",
         "form": "standard", "host": False},
        # independent analyses of mixed ensemble sizes over clustered
        # observations, as one batch
        {"name": "letkf_batch_k32_64_128", "kind": "batch", "nx": 192, "ny": 96, "nlev": 10,
         "k0": 32, "k1": 64, "k2": 128, "p": 60000, "radius": 500.0, "prec": "bf16x3"},
        # global ETKF: all observations, one transform for the whole state
        {"name": "etkf_k64", "kind": "etkf", "nx": 2048, "ny": 1024, "k": 64, "p": 100000,
         "rvar": "mixed"},
        # stochastic EnKF with its gain and conditioning diagnostics, each
        # observation with its own error
        {"name": "enkf_k80", "kind": "enkf", "nx": 512, "ny": 512, "k": 80, "p": 1500,
         "rvar": "mixed", "host": False},
        # local weighted EnKF on a 2048 x 2048 state
        {"name": "lwenkf_k64", "kind": "lwenkf", "nx": 2048, "ny": 2048, "k": 64, "p": 512,
         "radius": 0.05, "taper": "gaussian", "weights": "adaptive"},
        # learned inflation: prediction for every column, then a training
        # step (loss, gradient, Adam) on one batch
        {"name": "mlp_train_32768", "kind": "mlp", "m": 32768, "ncol": 131072},
        # verification of an ensemble: scores against a truth, mean and
        # scaled perturbations
        {"name": "verify_k40", "kind": "verify", "nx": 1024, "ny": 1024, "k": 40},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["enkf", "enkf", "letkf", "letkf", "letkf", "letkf", "cycle", "batch",
                       "etkf", "lwenkf", "mlp", "verify"])
    ks = [9, 10, 16, 20, 24, 25, 30, 32, 36, 40, 48, 50, 51, 60, 64, 80, 96, 100, 128]
    k = rng.choice(ks)
    if kind == "enkf":
        p = _log(rng, 12, 2000)
        n = _log(rng, 40, min(400000, int(3.2e10 / (p * k))))
        return {"kind": kind, "nx": n, "ny": 1, "k": k, "p": p,
                "rvar": rng.choice(["constant", "mixed"]), "host": n * k < 60000}
    if kind == "letkf":
        coord = rng.choice(["geo", "grid"])
        # columns up to what k leaves of a bounded k^3 total
        ncol = _log(rng, 300, int(min(40000, 2.5e9 / k ** 3)))
        nx = max(8, int(round(math.sqrt(ncol * rng.uniform(1.2, 2.2)))))
        ny = max(4, ncol // nx)
        p = _log(rng, 40, 40000)
        form = "refcompat" if nx * ny < 3000 and rng.random() < 0.3 else "standard"
        radius = rng.uniform(300.0, 1500.0) if coord == "geo" else rng.uniform(3.0, 14.0)
        prec = "fp64" if form == "refcompat" else rng.choice(["fp64", "fp64", "fp32", "bf16x3"])
        return {"kind": kind, "coord": coord, "nx": nx, "ny": ny, "nlev": _log(rng, 1, 32),
                "k": k, "p": p, "radius": round(radius, 2), "prec": prec, "form": form,
                "host": nx * ny * k < 30000}
    if kind == "cycle":
        return {"kind": kind, "N": _log(rng, 40, 6000), "k": rng.choice([10, 20, 24, 30, 40, 50]),
                "every": rng.choice([1, 2, 3]), "support": round(rng.uniform(6.0, 24.0), 1),
                "steps": rng.choice([1, 1, 2, 4])}
    if kind == "batch":
        nx = _log(rng, 40, 128)
        return {"kind": kind, "nx": nx, "ny": nx // 2, "nlev": _log(rng, 2, 12),
                "k0": rng.choice([16, 20, 32]), "k1": rng.choice([40, 48, 64]),
                "k2": rng.choice([64, 100, 128]), "p": _log(rng, 4000, 40000),
                "radius": round(rng.uniform(400.0, 1000.0), 1),
                "prec": rng.choice(["fp64", "fp32", "bf16x3"])}
    if kind == "etkf":
        return {"kind": kind, "nx": _log(rng, 2000, 2000000), "ny": 1, "k": k,
                "p": _log(rng, 50, 100000), "rvar": rng.choice(["constant", "mixed"])}
    if kind == "lwenkf":
        p = _log(rng, 24, 700)
        return {"kind": kind, "nx": _log(rng, 600, int(4e10 / (p * k))), "ny": 1, "k": k, "p": p,
                "radius": round(rng.uniform(0.03, 0.5), 3),
                "taper": rng.choice(["gaussian", "exponential", "gaspari_cohn"]),
                "weights": rng.choice(["uniform", "adaptive", "inverse_var"])}
    if kind == "mlp":
        return {"kind": kind, "m": _log(rng, 1000, 100000), "ncol": _log(rng, 1000, 200000)}
    return {"kind": "verify", "nx": _log(rng, 1000, int(4e7 / k)), "ny": 1, "k": k}


# ---------------------------------------------------------------------------
# inputs, made on the GPU from the seed alone
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * (int(seed) % 2000003) + 17)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _fields(g, m, nlev, ny, nx, cells):
    """m unit-variance Gaussian random fields [m][nlev * ny * nx], correlated
    over about `cells` grid cells in the horizontal and 3 levels, cut from a
    periodic grid of power-of-two sides."""
    nxp = 1 << max(2, (nx - 1).bit_length())
    nyp = 1 << max(2, (ny - 1).bit_length()) if ny > 1 else 1
    fx = torch.fft.rfftfreq(nxp, device=DEV, dtype=torch.float64)
    fy = torch.fft.fftfreq(nyp, device=DEV, dtype=torch.float64)
    a = -2.0 * (math.pi * cells / 2.0) ** 2
    h = torch.exp(a * (fy[:, None] ** 2 + fx[None, :] ** 2))
    w = torch.full_like(fx, 2.0)
    w[0] = w[-1] = 1.0
    scale = 1.0 / math.sqrt(float((w[None, :] * h ** 2).sum()) / (nxp * nyp))
    lev = torch.arange(nlev, device=DEV, dtype=torch.float64)
    mix = torch.exp(-0.5 * ((lev[:, None] - lev[None, :]) / 1.5) ** 2)
    mix = mix / mix.square().sum(1, keepdim=True).sqrt()
    out = torch.empty(m, nlev * ny * nx, device=DEV, dtype=torch.float64)
    for j in range(m):
        z = _randn(g, nlev, nyp, nxp)
        if nyp > 1:
            z = torch.fft.irfft2(torch.fft.rfft2(z) * h, s=(nyp, nxp))
        else:
            z = torch.fft.irfft(torch.fft.rfft(z) * h, n=nxp)
        z = z[:, :ny, :nx].reshape(nlev, -1) * scale
        out[j] = torch.matmul(mix, z).reshape(-1)
    return out


def _stencil(x, y, z, nx, ny, nlev, periodic):
    """Trilinear stencil (8 taps; 4 on one level) at grid positions: index and
    weight tensors [p][taps]."""
    p = x.numel()
    i0 = torch.floor(x).long()
    tx = x - i0
    j0 = torch.clamp(torch.floor(y).long(), 0, max(ny - 2, 0))
    ty = torch.clamp(y - j0, 0.0, 1.0)
    if periodic:
        i0, i1 = i0 % nx, (i0 + 1) % nx
    else:
        i0 = torch.clamp(i0, 0, max(nx - 2, 0))
        tx = torch.clamp(x - i0, 0.0, 1.0)
        i1 = torch.clamp(i0 + 1, max=nx - 1)
    j1 = torch.clamp(j0 + 1, max=ny - 1)
    levels = [(torch.zeros_like(i0), torch.ones_like(x))]
    if nlev > 1:
        k0 = torch.clamp(torch.floor(z).long(), 0, nlev - 2)
        tz = z - k0
        levels = [(k0, 1.0 - tz), (k0 + 1, tz)]
    cols, ws = [], []
    for kk, wz in levels:
        for jj, wy in ((j0, 1.0 - ty), (j1, ty)):
            for ii, wx in ((i0, 1.0 - tx), (i1, tx)):
                cols.append((kk * ny + jj) * nx + ii)
                ws.append(wz * wy * wx)
    return torch.stack(cols, 1).reshape(p, -1), torch.stack(ws, 1).reshape(p, -1)


def _variances(g, p, kind):
    """R diagonal: one instrument, or instruments and reports of differing error."""
    if kind == "constant":
        return torch.full((p,), 0.25, device=DEV, dtype=torch.float64)
    return (0.3 + 0.9 * _rand(g, p)) ** 2


def _positions(g, case, p):
    """Observation positions: (loc_a, loc_b, grid x, grid y) of the case's
    coordinate system."""
    nx, ny = case["nx"], case["ny"]
    if case.get("coord") == "geo":
        u, v = _rand(g, p), _rand(g, p)
        lat, lon = torch.rad2deg(torch.asin(2.0 * u - 1.0)), 360.0 * v
        if case["kind"] == "batch":  # 50 blobs of 300 km over a uniform tenth
            nb = max(1, p // 10)
            c_lat = torch.rad2deg(torch.asin(2.0 * _rand(g, 50) - 1.0))
            c_lon = 360.0 * _rand(g, 50)
            which = torch.randint(0, 50, (p - nb,), generator=g, device=DEV)
            dn, de = 300.0 * _randn(g, p - nb), 300.0 * _randn(g, p - nb)
            bl = (c_lat[which] + torch.rad2deg(dn / EARTH_KM)).clamp(-89.999, 89.999)
            lat[nb:] = bl
            lon[nb:] = c_lon[which] + torch.rad2deg(de / (EARTH_KM * torch.cos(torch.deg2rad(bl))))
            lon = torch.remainder(lon, 360.0)
        return lat, lon, lon / (360.0 / nx) - 0.5, (lat + 90.0) / (180.0 / ny) - 0.5
    x, y = _rand(g, p) * (nx - 1), _rand(g, p) * (ny - 1)
    return x, y, x, y


def _problem(case, g, k, p):
    """Background, observations and H of one analysis, all device tensors."""
    nx, ny, nlev = case["nx"], case["ny"], case.get("nlev", 1)
    geo = case.get("coord") == "geo"
    cells = max(2.0, 200.0 / (2.0 * math.pi * EARTH_KM / nx)) if geo else max(2.0, nx / 40.0)
    F = _fields(g, k + 1, nlev, ny, nx, cells)
    truth, Xb = F[k].clone(), F[:k]
    a, b, gx, gy = _positions(g, case, p)
    z = _rand(g, p) * (nlev - 1)
    col, w = _stencil(gx, gy, z, nx, ny, nlev, geo)
    var = _variances(g, p, case.get("rvar", "mixed" if case.get("prec") == "fp64" else "constant"))
    yo = (truth[col] * w).sum(1) + var.sqrt() * _randn(g, p)
    return {"Xb": Xb, "truth": truth, "a": a, "b": b, "col": col, "w": w, "var": var, "yo": yo}


def _columns(case):
    nx, ny = case["nx"], case["ny"]
    if case.get("coord") != "geo":
        return None, None
    lon = (torch.arange(nx, device=DEV, dtype=torch.float64) + 0.5) * 360.0 / nx
    lat = -90.0 + (torch.arange(ny, device=DEV, dtype=torch.float64) + 0.5) * 180.0 / ny
    return (lat[:, None].expand(ny, nx).reshape(-1).contiguous(),
            lon[None, :].expand(ny, nx).reshape(-1).contiguous())


def _objects(case, P, host=False):
    """The library's observation, operator and geometry objects for a problem."""
    p, taps = P["col"].shape
    rp = torch.arange(0, taps * p + 1, taps, device=DEV)
    out = (lambda t: t.cpu().numpy()) if host else (lambda t: t.contiguous())
    coord = L.COORD_GEOGRAPHIC if case.get("coord") == "geo" else L.COORD_GRID
    obs = mda.Observation(out(P["yo"]), out(P["var"]), out(P["a"]), out(P["b"]), coord=coord)
    H = mda.ObsOperator(out(rp), out(P["col"].reshape(-1)), out(P["w"].reshape(-1)))
    ca, cb = _columns(case)
    geom = mda.ColumnGeometry(coord, None if ca is None else out(ca),
                              None if cb is None else out(cb))
    return obs, H, geom


def _ctx():
    return mda.default_context()


def _stream(ctx):
    return torch.cuda.ExternalStream(ctx.stream, device=torch.device(DEV))


def _analysis_config(case):
    return mda.Config({"analysis": {"inflation": 1.05, "inflation_method": "multiplicative",
                                    "localization_radius": case.get("radius", 1.0),
                                    "localization_function": case.get("taper", "gaussian"),
                                    "weighting_scheme": case.get("weights", "uniform")}})


def _ensemble(case, Xb, host):
    X = Xb.cpu().numpy().copy() if host else torch.empty_like(Xb)
    return X, mda.Ensemble(X, case["nx"], case["ny"], case.get("nlev", 1))


def _mlp_inputs(case, g):
    """Features, targets and a network part-way through its training."""
    m, ncol = case["m"], case["ncol"]
    x = _randn(g, m, 8).float()
    target = (1.0 + 0.3 * torch.nn.functional.softplus(x[:, 0] + 0.5 * x[:, 3])).float()
    feat = _randn(g, ncol, 8).float()
    par = torch.cat([_randn(g, 512) * 0.35, _randn(g, 64) * 0.1, _randn(g, 4096) * 0.12,
                     _randn(g, 64) * 0.1, _randn(g, 64) * 0.2,
                     torch.full((1,), -1.0, device=DEV, dtype=torch.float64)]).float()
    m1 = (1e-3 * _randn(g, par.numel())).float()
    m2 = (1e-5 * (0.5 + _rand(g, par.numel()))).float()
    return x, target, feat, par, m1, m2


def _cycle_inputs(case, g):
    N, k = case["N"], case["k"]
    x = 8.0 + 2.0 * _randn(g, N)
    for _ in range(60):
        x = _l96_rk4(x, 0.05)
    Xb = x[None, :] + _randn(g, k, N)
    idx = torch.arange(0, N, case["every"], device=DEV)
    yo = x[idx] + _randn(g, idx.numel())
    return x, Xb.contiguous(), idx, yo


def prepare(case, seed):
    g, ctx, kind = _gen(seed), _ctx(), case["kind"]
    s = {"case": case, "ctx": ctx, "host": bool(case.get("host")), "stream": _stream(ctx)}
    if kind == "mlp":
        x, target, feat, par, m1, m2 = _mlp_inputs(case, g)
        net = learned.Inflator(ctx, device=DEV)
        net.params, net.m1, net.m2, net.step = par.contiguous(), m1, m2, 200
        s.update(net=net, x=x.contiguous(), target=target.contiguous(), feat=feat.contiguous())
        return s
    if kind == "cycle":
        N = case["N"]
        _, Xb, idx, yo = _cycle_inputs(case, g)
        lon = np.arange(N) * 360.0 / N
        oi = idx.cpu().numpy()
        p = len(oi)
        X = torch.empty_like(Xb)
        s.update(Xb=Xb, X=X, ens=mda.Ensemble(X, N, 1, 1),
                 model=mda.Lorenz96Model(mda.Config({"forcing": 8.0, "dt": 0.05, "scheme": "rk4",
                                                     "num_steps": case["steps"]}), ctx=ctx),
                 geom=mda.ColumnGeometry(L.COORD_GEOGRAPHIC, np.zeros(N), lon),
                 H=mda.ObsOperator(np.arange(p + 1, dtype=np.int64), oi, np.ones(p)),
                 obs=mda.Observation(yo.cpu().numpy(), np.ones(p), np.zeros(p), lon[oi],
                                     coord=L.COORD_GEOGRAPHIC),
                 cfg=mda.Config({"inflation": 1.05, "localization_radius":
                                 case["support"] * 2.0 * math.pi * EARTH_KM / N}))
        return s
    if kind == "batch":
        parts = []
        for i in range(3):
            c = dict(case, coord="geo")
            P = _problem(c, g, case["k%d" % i], case["p"])
            obs, H, geom = _objects(c, P)
            X, ens = _ensemble(c, P["Xb"], False)
            f = mda.LETKF(ens, obs, H, mda.Config({"inflation": 1.05,
                                                   "localization_radius": case["radius"]}),
                          geometry=geom, ctx=ctx, precision=PREC[case["prec"]])
            parts.append({"X": X, "Xb": P["Xb"], "filter": f})
        s["parts"] = parts
        return s
    if kind == "verify":
        F = _fields(g, case["k"] + 1, 1, case["ny"], case["nx"], max(2.0, case["nx"] / 40.0))
        s["truth"] = F[case["k"]].clone()
        s["ens"] = mda.Ensemble(F[:case["k"]], case["nx"], case["ny"], 1)
        return s
    P = _problem(case, g, case["k"], case["p"])
    obs, H, geom = _objects(case, P, s["host"])
    X, ens = _ensemble(case, P["Xb"], s["host"])
    s.update(X=X, ens=ens, obs=obs, H=H, geom=geom,
             Xb=P["Xb"].cpu().numpy() if s["host"] else P["Xb"])
    if kind in ("enkf", "lwenkf"):
        Z = _randn(g, case["p"], case["k"])
        s["Z"] = Z.cpu().numpy() if s["host"] else Z
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _background(s):
    if s["host"]:
        np.copyto(s["X"], s["Xb"])
    else:
        with torch.cuda.stream(s["stream"]):
            s["X"].copy_(s["Xb"])


_RESULTS = ("innovation_norm", "background_spread", "analysis_spread", "max_kalman_gain",
            "min_kalman_gain", "condition_number")


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    if kind == "mlp":
        net = s["net"]
        with torch.cuda.stream(s["stream"]):
            rho = net.predict(s["feat"])
            loss, grad = net.loss_grad(s["x"], s["target"])
            net.step += 1
            ctx.check(ctx.lib.mda_mlp_adam_step(ctx.h, net.params.data_ptr(), net.m1.data_ptr(),
                                                net.m2.data_ptr(), grad.data_ptr(), net.step,
                                                1e-4, 0.9, 0.999, 1e-8, 1))
        return {"rho": rho, "loss": loss, "grad": grad, "params": net.params, "m1": net.m1,
                "m2": net.m2}
    if kind == "verify":
        scores = mda.metrics(s["ens"], s["truth"], ctx=ctx)
        mean = s["ens"].RecomputeMean(ctx)
        pert = s["ens"].Perturbations(1.05, ctx)
        return {"scores": scores, "mean": mean, "pert": pert}
    if kind == "batch":
        with torch.cuda.stream(s["stream"]):
            for q in s["parts"]:
                q["X"].copy_(q["Xb"])
        mda.letkf_batch([q["filter"] for q in s["parts"]])
        return [q["X"] for q in s["parts"]]
    _background(s)
    if kind == "cycle":
        s["model"].runEnsemble(s["ens"])
        mda.LETKF(s["ens"], s["obs"], s["H"], s["cfg"], geometry=s["geom"], ctx=ctx).Analyse()
        return s["X"]
    if kind == "letkf":
        f = mda.LETKF(s["ens"], s["obs"], s["H"],
                      mda.Config({"inflation": 1.05, "localization_radius": case["radius"]}),
                      geometry=s["geom"], ctx=ctx, form=case["form"],
                      precision=PREC[case["prec"]])
        diag = f.Analyse()
        return {"X": s["X"], "local_obs": diag["total_local_obs"],
                "most_local_obs": diag["max_local_obs"]}
    if kind == "etkf":
        mda.ETKF(s["ens"], s["obs"], s["H"], mda.Config({"inflation": 1.05}), ctx=ctx).Analyse()
        return s["X"]
    if kind == "enkf":
        f = mda.EnKF(s["ens"], s["obs"], s["H"], _analysis_config(case), ctx=ctx)
    else:  # "gaspari_cohn" evaluates Gaspari & Cohn (1999)
        f = mda.LWEnKF(s["ens"], s["obs"], s["H"], _analysis_config(case), ctx=ctx,
                       gc_form="standard")
    f.Analyse(Z=s["Z"])
    r = f.getAnalysisResults()
    out = {"X": s["X"], "results": [r[name] for name in _RESULTS]}
    if kind == "lwenkf":
        out["weights"] = f.weights
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _local_mean(case):
    """Mean number of observations within the radius of a column."""
    if case.get("coord") == "geo" or case["kind"] == "batch":
        return case["p"] * (1.0 - math.cos(case["radius"] / EARTH_KM)) / 2.0
    area = math.pi * case["radius"] ** 2
    return case["p"] * min(1.0, area / (case["nx"] * case["ny"]))


def _letkf_work(case, k):
    ncol = case["nx"] * case["ny"]
    nlev, p = case.get("nlev", 1), case["p"]
    taps = 8 if nlev > 1 else 4
    pl = _local_mean(case)
    flops = ncol * (2.0 * pl * k * k + 2.0 * pl * k + 9.0 * k ** 3 + 2.0 * nlev * k * k)
    return (2.0 * ncol * nlev * k * 8 + p * (taps * 16 + 40.0), flops)


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        m, c = case["m"], case["ncol"]
        per = 2.0 * (8 * 64 + 64 * 64 + 64)
        return {"bytes": 36.0 * m + 36.0 * c + 7 * 4801 * 4, "flops": 3.0 * per * m + per * c}
    if kind == "cycle":
        c = {"kind": "letkf", "coord": "grid", "nx": case["N"], "ny": 1, "nlev": 1,
             "p": case["N"] // case["every"], "radius": case["support"]}
        k, pl = case["k"], 2.0 * case["support"] / case["every"]
        return {"bytes": 4.0 * c["nx"] * k * 8 + c["p"] * 104.0,
                "flops": c["nx"] * (2.0 * pl * k * k + 9.0 * k ** 3) +
                40.0 * case["steps"] * c["nx"] * k}
    if kind == "batch":
        w = [_letkf_work(case, case["k%d" % i]) for i in range(3)]
        return {"bytes": sum(v[0] for v in w), "flops": sum(v[1] for v in w)}
    k, n = case["k"], float(case["nx"]) * case["ny"]
    if kind == "verify":
        return {"bytes": 8.0 * n * (2 * k + 2), "flops": n * k * (6.0 + 4.0 * math.log2(k))}
    if kind == "letkf":
        b, f = _letkf_work(case, k)
        return {"bytes": b, "flops": f}
    p = case["p"]
    b = 2.0 * n * k * 8 + p * 104.0
    if kind == "etkf":
        return {"bytes": b, "flops": 2.0 * n * k * k + 2.0 * p * k * k}
    b += p * k * 8.0
    if kind == "lwenkf":
        return {"bytes": b, "flops": 4.0 * n * p * k + 2.0 * p * p * k + p ** 3 / 3.0}
    return {"bytes": b, "flops": 2.0 * n * p * k + 2.0 * n * k * k + 4.0 * p * k * k}


# ---------------------------------------------------------------------------
# the same results in 64 bits with plain torch
# ---------------------------------------------------------------------------
RHO = float(np.float32(1.05))  # config reals are float-narrowed


def _l96_rk4(x, dt):
    def f(v):
        return (torch.roll(v, -1, -1) - torch.roll(v, 2, -1)) * torch.roll(v, 1, -1) - v + 8.0
    k1 = f(x)
    k2 = f(x + 0.5 * dt * k1)
    k3 = f(x + 0.5 * dt * k2)
    k4 = f(x + dt * k3)
    return x + dt / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + k4)


def _obs_space(P):
    hx = torch.stack([(x[P["col"]] * P["w"]).sum(1) for x in P["Xb"]], 1)  # [p][k]
    ybar = hx.mean(1)
    return ybar, hx - ybar[:, None], P["yo"] - ybar


def _taper_gc(z):
    near = (((-0.25 * z + 0.5) * z + 0.625) * z - 5.0 / 3.0) * z * z + 1.0
    zz = z.clamp_min(1e-3)
    far = ((((zz / 12.0 - 0.5) * zz + 0.625) * zz + 5.0 / 3.0) * zz - 5.0) * zz + 4.0 - \
        2.0 / (3.0 * zz)
    return torch.where(z <= 1.0, near, torch.where(z < 2.0, far, torch.zeros_like(z)))


def _unit(lat, lon):
    la, lo = torch.deg2rad(lat), torch.deg2rad(lon)
    return torch.stack([la.cos() * lo.cos(), la.cos() * lo.sin(), la.sin()], 1)


def _inv_sqrt(A):
    """A^-1/2 of a batch of SPD matrices: coupled Newton iteration."""
    c = A.abs().sum(2).max(1).values[:, None, None]
    eye = torch.eye(A.shape[1], device=A.device, dtype=A.dtype)
    Y, Z = A / c, eye.expand_as(A).contiguous()
    for _ in range(60):
        R = 1.5 * eye - 0.5 * torch.bmm(Z, Y)
        Y, Z = torch.bmm(Y, R), torch.bmm(R, Z)
        if float((R - eye).abs().max()) < 1e-14:
            break
    return 0.5 * (Z + Z.transpose(1, 2)) / c.sqrt()


def _exact_letkf(case, P, k, radius, geo_cols, form):
    """(analysis, sum and maximum of the local observation counts)."""
    nx, ny, nlev, dev = case["nx"], case["ny"], case.get("nlev", 1), P["Xb"].device
    ncol = nx * ny
    p = P["yo"].numel()
    _, Y, d = _obs_space(P)
    iu = torch.triu_indices(k, k, device=dev)
    YY = Y[:, iu[0]] * Y[:, iu[1]]
    R = torch.cat([YY, Y * d[:, None]], 1)
    del YY
    X = P["Xb"].reshape(k, nlev, ncol)
    out = torch.empty_like(X)
    total, most = 0, 0
    if geo_cols is not None:
        uo, uc = _unit(P["a"], P["b"]), _unit(*geo_cols)
    g = torch.arange(ncol, device=dev, dtype=torch.float64)
    step = max(1, min(4096, int(1.2e8 / p), int(4e8 / (k * k))))
    for c0 in range(0, ncol, step):
        c1 = min(ncol, c0 + step)
        if geo_cols is not None:
            ch2 = sum((uc[c0:c1, i:i + 1] - uo[None, :, i]) ** 2 for i in range(3))
            dist = 2.0 * EARTH_KM * torch.asin((0.5 * ch2.sqrt()).clamp(max=1.0))
        else:
            gx, gy = torch.remainder(g[c0:c1], nx), torch.floor(g[c0:c1] / nx)
            dist = ((gx[:, None] - P["a"][None, :]) ** 2 +
                    (gy[:, None] - P["b"][None, :]) ** 2).sqrt()
        inside = dist <= radius
        count = inside.sum(1)
        total, most = total + int(count.sum()), max(most, int(count.max()))
        if form == "standard":
            W = torch.where(inside, _taper_gc(dist / (radius / 2.0)), torch.zeros_like(dist))
            W = W / P["var"][None, :]
        else:
            W = inside.double()
        M = W @ R
        del W, dist, inside
        C = torch.zeros(c1 - c0, k, k, device=dev, dtype=torch.float64)
        C[:, iu[0], iu[1]] = M[:, :iu.shape[1]]
        C[:, iu[1], iu[0]] = M[:, :iu.shape[1]]
        b = M[:, iu.shape[1]:]
        eye = torch.eye(k, device=dev, dtype=torch.float64)
        if form == "standard":
            S = _inv_sqrt(C + (k - 1) / RHO * eye)
            T = torch.bmm(S, torch.bmm(S, b[:, :, None])) + math.sqrt(k - 1) * S
        else:
            A = (C + (k - 1) * eye).cpu().numpy()
            Pa = RHO * np.linalg.inv(A)
            Pa = 0.5 * (Pa + Pa.transpose(0, 2, 1))
            wa = np.einsum("gij,gj->gi", Pa, b.cpu().numpy())
            Wa = math.sqrt(k - 1) * np.linalg.cholesky(Pa)
            T = torch.diag_embed(torch.from_numpy(wa + Wa.sum(2)).to(dev))
        T = torch.where((count == 0)[:, None, None], math.sqrt(RHO) * eye, T)
        x = X[:, :, c0:c1].permute(2, 1, 0)  # [col][lev][member]
        xm = x.mean(2, keepdim=True)
        xa = xm + torch.bmm((x - xm).contiguous(), T.contiguous())
        out[:, :, c0:c1] = xa.permute(2, 1, 0)
    return out.reshape(k, -1), total, most


def _norms(P, scale, d, Xa, k, n):
    xp = (P["Xb"] - P["Xb"].mean(0)) * scale
    xa = Xa - Xa.mean(0)
    return (float(d.norm()), math.sqrt(float(xp.square().sum()) / (n * k)),
            math.sqrt(float(xa.square().sum()) / (n * k)))


def _exact_enkf(case, P, Z):
    k, p = case["k"], case["p"]
    n = P["Xb"].shape[1]
    scale = math.sqrt(RHO)
    _, Y, d = _obs_space(P)
    S = (Y @ Y.T) / (k - 1) + torch.diag(P["var"])
    Sh = S.cpu()
    ev = torch.linalg.eigvalsh(Sh)
    G = torch.linalg.solve(Sh, Y.cpu()).to(Y.device) / (k - 1)  # [p][k]
    D = d[:, None] + P["var"].sqrt()[:, None] * Z - Y
    xm = P["Xb"].mean(0)
    xp = (P["Xb"] - xm) * scale
    T = torch.eye(k, device=Y.device, dtype=torch.float64) + G.T @ D
    Xa = xm + T.T @ xp
    hi, lo = -math.inf, math.inf
    step = max(1, int(2e8 / p))
    for i in range(0, n, step):
        K = G @ xp[:, i:i + step]
        hi, lo = max(hi, float(K.max())), min(lo, float(K.min()))
    dn, sb, sa = _norms(P, scale, d, Xa, k, n)
    return {"X": Xa, "results": [dn, sb, sa, hi, lo, float(ev[-1] / ev[0])]}


def _lw_taper(dist, case):
    nd = dist / float(np.float32(case["radius"]))
    if case["taper"] == "gaussian":
        return torch.exp(-0.5 * nd * nd)
    if case["taper"] == "exponential":
        return torch.exp(-nd)
    return _taper_gc(nd)


def _exact_lwenkf(case, P, Z):
    k, p = case["k"], case["p"]
    n, dev = P["Xb"].shape[1], P["Xb"].device
    scale = math.sqrt(RHO)
    ybar, Y, d = _obs_space(P)
    xm = P["Xb"].mean(0)
    if case["weights"] == "uniform":
        w = torch.full((k,), 1.0 / k, device=dev, dtype=torch.float64)
    else:
        ss = torch.stack([(x - xm).square().sum() for x in P["Xb"]])
        w = 1.0 / ((ss.sqrt() if case["weights"] == "adaptive" else ss) + 1e-8)
    w = w / w.sum()
    i = torch.arange(p, device=dev, dtype=torch.float64)
    S = ((Y * w) @ Y.T) * _lw_taper((i[:, None] - i[None, :]).abs() / p, case) + \
        torch.diag(P["var"])
    Sh = S.cpu()
    ev = torch.linalg.eigvalsh(Sh).abs()
    G = torch.linalg.solve(Sh.T, Y.cpu()).to(dev) / (k - 1)
    D = P["yo"][:, None] + P["var"].sqrt()[:, None] * Z - (ybar[:, None] + Y)
    Xa = torch.empty_like(P["Xb"])
    hi, lo = -math.inf, math.inf
    step = max(1, int(5e7 / p))
    for s0 in range(0, n, step):
        xp = (P["Xb"][:, s0:s0 + step] - xm[s0:s0 + step]) * scale
        t = torch.arange(s0, s0 + xp.shape[1], device=dev, dtype=torch.float64)
        K = (xp.T @ G.T) * _lw_taper((t[:, None] - i[None, :]).abs() / max(n, p), case)
        hi, lo = max(hi, float(K.max())), min(lo, float(K.min()))
        Xa[:, s0:s0 + step] = xm[s0:s0 + step] + (xp + (K @ D).T)
    dn, sb, sa = _norms(P, scale, d, Xa, k, n)
    return {"X": Xa, "results": [dn, sb, sa, hi, lo, float(ev.max() / ev.min())],
            "weights": w}


def _exact_mlp(case, g):
    x, target, feat, par, m1, m2 = _mlp_inputs(case, g)
    q = par.double().requires_grad_(True)

    def net(v):
        W1, b1 = q[:512].view(64, 8), q[512:576]
        W2, b2, W3, b3 = q[576:4672].view(64, 64), q[4672:4736], q[4736:4800], q[4800]
        h = torch.tanh(torch.tanh(v.double() @ W1.T + b1) @ W2.T + b2)
        return 1.0 + torch.nn.functional.softplus(h @ W3 + b3)
    rho = net(feat).detach()
    loss = (net(x) - target.double()).square().mean()
    loss.backward()
    gr = q.grad
    a = 0.9 * m1.double() + 0.1 * gr
    v = 0.999 * m2.double() + 0.001 * gr * gr
    new = par.double() - 1e-4 * (a / (1 - 0.9 ** 201)) / ((v / (1 - 0.999 ** 201)).sqrt() + 1e-8)
    return {"rho": rho, "loss": float(loss), "grad": gr, "params": new, "m1": a, "m2": v}


def _exact_verify(case, g):
    k = case["k"]
    F = _fields(g, k + 1, 1, case["ny"], case["nx"], max(2.0, case["nx"] / 40.0))
    X, t = F[:k], F[k]
    mean = X.mean(0)
    df = mean - t
    spread = (X - mean).square().sum(0).div(k - 1).sqrt().mean()
    st = torch.zeros_like(t)
    for x in X:
        st += (x - t).abs()
    # sum over all pairs of |x_a - x_b| from the sorted members
    sd = torch.zeros_like(t)
    step = 1 << 18
    rank = (2.0 * torch.arange(k, device=DEV, dtype=torch.float64) - (k - 1))[:, None]
    for i in range(0, t.numel(), step):
        sd[i:i + step] = 2.0 * (X[:, i:i + step].sort(0).values * rank).sum(0)
    crps = (st / k - sd / (2.0 * k * k)).mean()
    mc, tc = mean - mean.mean(), t - t.mean()
    corr = (mc * tc).sum() / (mc.square().sum() * tc.square().sum()).sqrt()
    scores = {"rmse": float(df.square().mean().sqrt()), "bias": float(df.mean()),
              "correlation": float(corr), "crps": float(crps), "avg_spread": float(spread)}
    return {"scores": scores, "mean": mean, "pert": (X - mean) * 1.05}


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "mlp":
        return _exact_mlp(case, g)
    if kind == "verify":
        return _exact_verify(case, g)
    if kind == "cycle":
        N = case["N"]
        _, Xb, idx, yo = _cycle_inputs(case, g)
        for _ in range(case["steps"]):
            Xb = _l96_rk4(Xb, float(np.float32(0.05)))
        lon = torch.arange(N, device=DEV, dtype=torch.float64) * 360.0 / N
        P = {"Xb": Xb, "col": idx[:, None], "w": torch.ones_like(yo)[:, None], "yo": yo,
             "var": torch.ones_like(yo), "a": torch.zeros_like(yo), "b": lon[idx]}
        radius = float(np.float32(case["support"] * 2.0 * math.pi * EARTH_KM / N))
        c = {"nx": N, "ny": 1, "nlev": 1}
        return _exact_letkf(c, P, case["k"], radius, (torch.zeros_like(lon), lon), "standard")[0]
    if kind == "batch":
        out = []
        for i in range(3):
            c = dict(case, coord="geo")
            P = _problem(c, g, case["k%d" % i], case["p"])
            out.append(_exact_letkf(c, P, case["k%d" % i], float(np.float32(case["radius"])),
                                    _columns(c), "standard")[0])
        return out
    if kind == "letkf" and float(case["nx"]) * case["ny"] * case["p"] > 2e10:
        return None  # the brute-force local sets of the full workload take minutes
    P = _problem(case, g, case["k"], case["p"])
    if kind == "letkf":
        cols = _columns(case)
        X, total, most = _exact_letkf(case, P, case["k"], float(np.float32(case["radius"])),
                                      cols if cols[0] is not None else None, case["form"])
        return {"X": X, "local_obs": total, "most_local_obs": most}
    if kind == "etkf":
        k = case["k"]
        _, Y, d = _obs_space(P)
        Yr = Y / P["var"][:, None]
        Pa = np.linalg.inv((Yr.T @ Y).cpu().numpy() + (k - 1) * np.eye(k))
        Wa = math.sqrt(k - 1) * np.linalg.cholesky(0.5 * (Pa + Pa.T))
        T = torch.from_numpy((Pa @ (Yr.T @ d).cpu().numpy())[:, None] + Wa).to(DEV)
        xm = P["Xb"].mean(0)
        return xm + T.T @ ((P["Xb"] - xm) * RHO)
    Z = _randn(g, case["p"], case["k"])
    return _exact_enkf(case, P, Z) if kind == "enkf" else _exact_lwenkf(case, P, Z)
