"""Analyses at the sizes where a kernel's tiles, its search or the rule that
chooses it can go wrong, against the oracle."""
import math

import numpy as np
import pytest

from cases import latlon_case, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.fixture(scope="module")
def mda():
    import metada_amd
    return metada_amd


@pytest.fixture(scope="module")
def ctx(mda):
    c = mda.Context(0)
    yield c
    c.close()


# ---- bucket start table: long gaps, crowded buckets, search boundaries ---------------------
@pytest.mark.parametrize("p", [1, 2, 63, 64, 65, 4096, 4097, 6000])
@pytest.mark.parametrize("where", ["parallel", "point", "poles"])
def test_bucket_ranges_match_oracle(mda, ctx, orc, p, where):
    """Observations on one parallel, nearly at one point (one bucket holds
    them all) or at both poles (the gap spans the grid): local counts and the
    analysis equal the oracle's."""
    rng = np.random.default_rng(p + len(where))
    nlon, nlat, k = 36, 18, 8
    lonc, latc = (np.arange(nlon) + 0.5) * 10.0, -90 + (np.arange(nlat) + 0.5) * 10.0
    col_lon, col_lat = (v.ravel().copy() for v in np.meshgrid(lonc, latc))
    if where == "parallel":
        lat, lon = np.full(p, 5.0), rng.uniform(0, 360, p)
    elif where == "point":
        lat, lon = 15.0 + rng.uniform(0, 1e-3, p), 44.9 + rng.uniform(0, 1e-3, p)
    else:
        lat = np.where(rng.random(p) < 0.5, -86.0, 86.0) + rng.uniform(-1, 1, p)
        lon = rng.uniform(0, 360, p)
    X = rng.standard_normal((k, nlon * nlat))
    Yb, yo, var = rng.standard_normal((k, p)), rng.standard_normal(p), rng.uniform(1, 2, p)
    ens = mda.Ensemble(X.copy(), nlon, nlat, 1)
    f = mda.LETKF(ens, mda.Observation(yo, var, lat, lon, coord=mda._lib.COORD_GEOGRAPHIC),
                  mda.ObsOperator(hx=Yb), mda.Config({"inflation": 1.05,
                                                      "localization_radius": 700.0}),
                  geometry=mda.ColumnGeometry(mda._lib.COORD_GEOGRAPHIC, col_lat, col_lon),
                  ctx=ctx)
    f.Analyse()
    prob = orc.Problem(k, nlon, nlat, 1, orc.COORD_GEOGRAPHIC, col_lat, col_lon, lat, lon, yo,
                       var, f.inflation, f.localization_radius)
    Xo, _, nloc = orc.letkf_standard(prob, X, Yb)
    np.testing.assert_array_equal(f.local_counts(), nloc)
    assert nloc.max() > 0
    assert rel_err(ens.data, Xo) < TOL


# ---- ensemble sizes between the eigensolver's block sizes -----------------------------------
def _latlon(mda, ctx, case, X, radius, **kw):
    ens = mda.Ensemble(X.copy(), case["nlon"], case["nlat"], case["nlev"])
    f = mda.LETKF(ens, mda.Observation(case["yo"], case["var"], case["lat"], case["lon"],
                                       coord=mda._lib.COORD_GEOGRAPHIC), case["H"],
                  mda.Config({"inflation": 1.05, "localization_radius": radius}),
                  geometry=mda.ColumnGeometry(mda._lib.COORD_GEOGRAPHIC, case["col_lat"],
                                              case["col_lon"]), ctx=ctx, **kw)
    f.Analyse()
    return f, ens.data


@pytest.mark.parametrize("k", [2, 3, 7, 9, 15, 17, 19, 21, 31, 33, 39, 41, 47, 49, 50, 63, 65,
                               76, 77, 100, 127])
def test_letkf_every_k_matches_oracle(mda, ctx, orc, k):
    """k runs in the next larger block (8, 16, 20, 32, 40, 48, 64, 128): the
    transforms and the analysis (T kept, and applied by the eigenvector
    kernel) equal the oracle's."""
    case = latlon_case(nlon=18, nlat=9, nlev=2, k=k, p=700, seed=300 + k, nmodes=96)
    prob = orc.Problem(k, 18, 9, 2, orc.COORD_GEOGRAPHIC, case["col_lat"], case["col_lon"],
                       case["lat"], case["lon"], case["yo"], case["var"],
                       float(np.float32(1.05)), 3000.0)
    Xo, To, _ = orc.letkf_standard(prob, case["X"], case["H"].apply_host(case["X"]), want_T=True)
    f, Xk = _latlon(mda, ctx, case, case["X"], 3000.0, keep_transforms=True)
    cols = np.array([0, 40, 161])
    assert rel_err(f.transforms(cols), To[cols]) < TOL
    assert rel_err(Xk, Xo) < TOL
    assert f.diag["max_jacobi_sweeps"] == 0
    assert rel_err(_latlon(mda, ctx, case, case["X"], 3000.0)[1], Xo) < TOL


@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("k,ks", [(7, 8), (16, 16), (19, 20), (32, 32), (40, 40), (47, 48),
                                  (64, 64)])
def test_letkf_eigenvalue_kernels_match_jacobi(mda, ctx, k, ks, over):
    """Bisection up to 128 columns per row of the block, QL beyond."""
    nlon, nlat = 2 * ks, 64 + over
    case = latlon_case(nlon=nlon, nlat=nlat, nlev=1, k=k, p=500, seed=700 + k, nmodes=96)
    L = mda._lib
    f, X = _latlon(mda, ctx, case, case["X"], 4000.0)
    _, Xj = _latlon(mda, ctx, case, case["X"], 4000.0, eig_method=L.EIG_JACOBI)
    # near-degenerate columns may fail the eigenvector checks: a few in ten thousand
    assert f.diag["n_fallback_columns"] <= nlon * nlat // 100
    assert rel_err(X, Xj) < TOL


@pytest.mark.parametrize("prec", ["FP32", "BF16X3"])
@pytest.mark.parametrize("k,radius", [(10, 500.0), (25, 3000.0), (50, 1500.0), (50, 6000.0),
                                      (100, 1500.0), (100, 9000.0)])
def test_letkf_reduced_precision_blocks_match_jacobi(mda, ctx, k, radius, prec):
    """The same reduced-precision Gram through the padded block and through
    Jacobi, with columns of fewer and of more than k observations: equal to
    the eigensolvers' FP64 rounding."""
    case = latlon_case(nlon=18, nlat=9, nlev=2, k=k, p=700, seed=400 + k, nmodes=96)
    L = mda._lib
    kw = dict(precision=getattr(L, "PREC_" + prec))
    fa, Xa = _latlon(mda, ctx, case, case["X"], radius, **kw)
    fj, Xj = _latlon(mda, ctx, case, case["X"], radius, eig_method=L.EIG_JACOBI, **kw)
    few = int(((fa.local_counts() > 0) & (fa.local_counts() < k)).sum())
    if prec == "FP32":  # BF16x3 stays with Jacobi at these sizes
        assert fa.diag["n_fallback_columns"] >= few
    assert rel_err(Xa, Xj) < TOL


# ---- EnKF gain and spread diagnostics: tiles of 16 observations, 32 points, 16 members ------
@pytest.mark.parametrize("k,n,p", [(2, 1, 1), (16, 31, 15), (17, 33, 16), (33, 128, 17),
                                   (50, 129, 33), (64, 1000, 40), (80, 257, 100),
                                   (100, 64, 31), (112, 300, 48), (113, 65, 20),
                                   (128, 4100, 60)])
def test_enkf_diagnostics_match_oracle(mda, ctx, orc, k, n, p):
    rng = np.random.default_rng(1000 * k + p)
    X = 3.0 + rng.standard_normal((k, n))
    Yb, yo = rng.standard_normal((k, p)), rng.standard_normal(p)
    var, Z = rng.uniform(0.5, 2.0, p), rng.standard_normal((p, k))
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    f = mda.EnKF(ens, mda.Observation(yo, var, np.zeros(p), np.zeros(p)),
                 mda.ObsOperator(hx=Yb), mda.Config({"analysis": {"inflation": 1.1}}), ctx=ctx)
    f.Analyse(Z=Z)
    Xo, d = orc.enkf_analyse(X, Yb, yo, var, Z, f.inflation_factor)
    assert rel_err(ens.data, Xo) < TOL
    r = f.getAnalysisResults()
    for key in ("max_kalman_gain", "min_kalman_gain", "background_spread", "analysis_spread",
                "innovation_norm", "condition_number"):
        # the gain's rounding scales with its largest entry
        scale = max(abs(d["max_kalman_gain"]), abs(d["min_kalman_gain"])) \
            if "gain" in key else abs(d[key])
        assert abs(r[key] - d[key]) <= 1e-10 * scale, (key, r[key], d[key])


# ---- cond(S) of the EnKF: dense in LDS (p <= 128), from E (one variance), by inertia --------
@pytest.mark.parametrize("k,p,var", [
    (2, 2, "mixed"), (5, 3, "mixed"), (40, 63, "mixed"), (20, 127, "constant"),
    (64, 128, "mixed"), (2, 129, "mixed"), (17, 129, "constant"), (17, 130, "mixed"),
    (64, 300, "mixed"), (64, 700, "constant"), (113, 500, "mixed"), (128, 257, "mixed"),
    (128, 1000, "few"), (30, 400, "few"), (30, 200, "pair"), (40, 131, "spread")])
def test_enkf_condition_number(mda, ctx, k, p, var):
    """cond(S) against a dense eigenvalue solve: all variances distinct, one,
    three (multiplicities above k), one pair of smallest ones, or spread over
    four decades."""
    rng = np.random.default_rng(7 * k + p)
    Yb = rng.standard_normal((k, p)) @ (np.eye(p) + 0.3 * np.eye(p, k=1))
    R = {"mixed": rng.uniform(0.1, 1.5, p), "constant": np.full(p, 0.25),
         "few": rng.choice([0.1, 0.4, 2.0], p), "spread": 10.0 ** rng.uniform(-3, 1, p),
         "pair": np.r_[0.05, 0.05, rng.uniform(0.2, 1.0, p - 2)]}[var]
    ens = mda.Ensemble(rng.standard_normal((k, 24)), 24, 1, 1)
    f = mda.EnKF(ens, mda.Observation(rng.standard_normal(p), R, np.zeros(p), np.zeros(p)),
                 mda.ObsOperator(hx=Yb), mda.Config({"analysis": {"inflation": 1.0}}), ctx=ctx)
    f.Analyse()
    Y = Yb - Yb.mean(0)
    lam = np.linalg.eigvalsh(Y.T @ Y / (k - 1) + np.diag(R))
    want = lam[-1] / lam[0]
    # both sides carry the rounding of the smallest eigenvalue: cond * eps
    assert abs(f.getAnalysisResults()["condition_number"] - want) <= \
        want * max(1e-11, 64 * want * 2.2e-16)


# ---- global transform: 32 points a wavefront, 256 a block, members in steps of 16 -----------
@pytest.mark.parametrize("k,n", [(2, 1), (3, 15), (16, 17), (17, 31), (32, 33), (48, 255),
                                 (49, 256), (64, 257), (65, 511), (96, 1000), (113, 70),
                                 (128, 300)])
def test_etkf_transform_matches_oracle(mda, ctx, orc, k, n):
    rng = np.random.default_rng(50 * k + n)
    p = 37
    X, Yb = 5.0 + rng.standard_normal((k, n)), rng.standard_normal((k, p))
    yo, var = rng.standard_normal(p), rng.uniform(0.5, 2.0, p)
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    f = mda.ETKF(ens, mda.Observation(yo, var, np.zeros(p), np.zeros(p)),
                 mda.ObsOperator(hx=Yb), mda.Config({"inflation": 1.1}), ctx=ctx)
    f.Analyse()
    assert rel_err(ens.data, orc.etkf_analyse(X, Yb, yo, var, f.inflation)) < TOL


# ---- global Gram: steps of 4 observations, one or many partial blocks, two row groups -------
@pytest.mark.parametrize("k", [2, 16, 33, 64, 65, 80, 113, 128])
@pytest.mark.parametrize("p", [1, 3, 65, 129, 1030, 33000])
def test_global_filters_every_p_match_oracle(mda, ctx, orc, k, p):
    """ETKF and EnKF over observation counts around the Gram's block sizes,
    one observation invalid; the EnKF's noalloc twin is bit-equal elsewhere."""
    rng = np.random.default_rng(k * 7919 + p)
    n = 20
    X, Yb = rng.standard_normal((k, n)), rng.standard_normal((k, p))
    yo, var = rng.standard_normal(p), rng.uniform(0.5, 2.0, p) * max(1.0, p / 50.0)
    if p > 1:
        var[p // 2] = np.inf
    obs = mda.Observation(yo, var, np.zeros(p), np.zeros(p))
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    f = mda.ETKF(ens, obs, mda.ObsOperator(hx=Yb), mda.Config({"inflation": 1.1}), ctx=ctx)
    f.Analyse()
    ok = np.isfinite(var)  # an invalid observation has weight 0
    assert rel_err(ens.data, orc.etkf_analyse(X, Yb[:, ok], yo[ok], var[ok], f.inflation)) < TOL
    if p > 1030:
        return
    Z = rng.standard_normal((p, k))
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    g = mda.EnKF(ens, obs, mda.ObsOperator(hx=Yb),
                 mda.Config({"analysis": {"inflation": 1.1}}), ctx=ctx)
    g.Analyse(Z=Z)
    Y, d = Yb - Yb.mean(0), yo - Yb.mean(0)
    Y, d, Zk, R = Y[:, ok], d[ok], Z[ok], var[ok]
    K = np.linalg.solve(Y.T @ Y / (k - 1) + np.diag(R), Y.T) / (k - 1)
    D = d[:, None] + np.sqrt(R)[:, None] * Zk - Y.T
    Xp = (X - X.mean(0)) * np.sqrt(g.inflation_factor)
    assert rel_err(ens.data, X.mean(0) + (np.eye(k) + K.T @ D).T @ Xp) < TOL


# ---- LWEnKF update: 32 points a wavefront, tiles of 16 observations, members in steps of 16 --
@pytest.mark.parametrize("k,n,p,fn", [
    (2, 5, 3, "gaussian"), (16, 31, 16, "cutoff"), (17, 32, 17, "exponential"),
    (33, 129, 33, "gaussian"), (48, 20, 150, "gaspari_cohn"), (64, 100, 15, "gaussian"),
    (65, 40, 100, "exponential"), (100, 257, 47, "gaussian"), (128, 33, 65, "gaspari_cohn")])
def test_lwenkf_update_matches_oracle(mda, ctx, orc, k, n, p, fn):
    rng = np.random.default_rng(31 * k + n)
    X, Yb = 2.0 + rng.standard_normal((k, n)), rng.standard_normal((k, p))
    yo, var = rng.standard_normal(p), rng.uniform(0.5, 2.0, p)
    Z = rng.standard_normal((p, k))
    cfg = mda.Config({"analysis": {"inflation": 1.1, "localization_radius": 0.3,
                                   "localization_function": fn, "weighting_scheme": "adaptive"}})
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    f = mda.LWEnKF(ens, mda.Observation(yo, var, np.zeros(p), np.zeros(p)),
                   mda.ObsOperator(hx=Yb), cfg, ctx=ctx, gc_form="standard")
    f.Analyse(Z=Z)
    Xo, w, d, _ = orc.lwenkf_analyse(X, Yb, yo, var, Z, f.inflation_factor,
                                     f.localization_radius, fn, "adaptive", gc_standard=True)
    assert rel_err(ens.data, Xo) < TOL
    np.testing.assert_allclose(f.weights, w, rtol=1e-12)
    r = f.getAnalysisResults()
    for key in ("background_spread", "analysis_spread", "max_kalman_gain", "min_kalman_gain",
                "innovation_norm", "condition_number"):
        scale = max(abs(d["max_kalman_gain"]), abs(d["min_kalman_gain"])) \
            if "gain" in key else abs(d[key])
        assert abs(r[key] - d[key]) <= 1e-9 * scale, (key, r[key], d[key])


# ---- dense S of the LWEnKF: LDS reduction to p = 128, a launch per column beyond; elimination
# ---- in blocks of 16 columns (8 beyond p = 1024), a thread per row to 1024, two to 2048 -------
@pytest.mark.parametrize("p", [1, 2, 3, 15, 16, 17, 127, 129, 130, 255, 257, 512, 513, 1023, 1025,
                               2047, 2049])
def test_lwenkf_dense_algebra_with_pivoting(mda, ctx, orc, p):
    # observations of very different scale, strongly correlated: the largest entry of a column
    # of S is off the diagonal in some steps of each size above 3
    k, n = 6, 40
    rng = np.random.default_rng(p)
    scale = 10.0 ** rng.uniform(-0.75, 0.75, p)
    X = 2.0 + rng.standard_normal((k, n))
    Yb = scale * (rng.standard_normal((k, 1)) + 0.1 * rng.standard_normal((k, p)))
    yo, var = scale * rng.standard_normal(p), 0.2 * scale ** 2
    Z = rng.standard_normal((p, k))
    cfg = mda.Config({"analysis": {"inflation": 1.1, "localization_radius": 5.0 * p,
                                   "localization_function": "gaussian",
                                   "weighting_scheme": "uniform"}})
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    f = mda.LWEnKF(ens, mda.Observation(yo, var, np.zeros(p), np.zeros(p)),
                   mda.ObsOperator(hx=Yb), cfg, ctx=ctx, gc_form="standard")
    f.Analyse(Z=Z)
    if p <= 257:
        Xo, _, d, _ = orc.lwenkf_analyse(X, Yb, yo, var, Z, f.inflation_factor,
                                         f.localization_radius, "gaussian", "uniform",
                                         gc_standard=True)
        cond = d["condition_number"]
    else:  # the oracle's singular values take minutes there
        def taper(rows, size):
            d = np.abs(np.arange(rows)[:, None] - np.arange(p)) / size
            return np.exp(-0.5 * (d / f.localization_radius) ** 2)
        Y, Xp = Yb - Yb.mean(0), (X - X.mean(0)) * np.sqrt(f.inflation_factor)
        S = taper(p, p) * (Y.T @ Y / k) + np.diag(var)
        K = np.linalg.solve(S, Y.T @ Xp).T / (k - 1) * taper(n, max(n, p))
        Xo = X.mean(0) + Xp + (yo + np.sqrt(var) * Z.T - Yb) @ K.T
        ev = np.linalg.eigvalsh(S)
        cond = ev[-1] / ev[0]
    # cond(S) eps per solve and per singular value, over p-term sums; growth of 100
    tol = 100 * np.finfo(float).eps * cond * max(4.0, np.sqrt(p))
    assert tol < 1e-5
    assert rel_err(ens.data, Xo) < tol
    r = f.getAnalysisResults()
    assert abs(r["condition_number"] / cond - 1.0) < tol


# ---- verification scores: members held in registers, and the general form beyond 128 --------
@pytest.mark.parametrize("k,n", [(2, 1), (7, 300), (8, 255), (9, 257), (40, 1000), (41, 64),
                                 (63, 500), (65, 33), (97, 100), (128, 270), (129, 50)])
def test_metrics_every_k(mda, ctx, k, n):
    rng = np.random.default_rng(k + n)
    X, t = 280.0 + rng.standard_normal((k, n)), 280.0 + rng.standard_normal(n)
    m = mda.metrics(mda.Ensemble(X, n, 1, 1), t, ctx=ctx)
    mean = X.mean(0)
    crps = (np.abs(X - t).mean(0) -
            np.abs(X[:, None] - X[None]).sum((0, 1)) / (2.0 * k * k)).mean()
    # values near 280 with unit spread: 280 eps per difference, k terms
    for key, want in (("crps", crps), ("avg_spread", X.std(0, ddof=1).mean()),
                      ("bias", (mean - t).mean()), ("rmse", np.sqrt(((mean - t) ** 2).mean()))):
        assert abs(m[key] - want) < 1e-12 * max(1.0, k / 8), key


# ---- MLP: 16 samples a wavefront step, 64 a block, up to 256 (gradient) / 1024 blocks -------
@pytest.mark.parametrize("m", [1, 15, 17, 63, 64, 65, 1023, 16385, 70001])
def test_mlp_every_m_matches_oracle(mda, ctx, orc, m):
    import ctypes as C
    rng = np.random.default_rng(m)
    p = np.concatenate([rng.standard_normal(512) * 0.35, rng.standard_normal(64) * 0.1,
                        rng.standard_normal(4096) * 0.12, rng.standard_normal(64) * 0.1,
                        rng.standard_normal(64) * 0.2, [-1.0]]).astype(np.float32)
    feat = rng.standard_normal((m, 8)).astype(np.float32)
    target = (1.0 + rng.random(m)).astype(np.float32)
    rho, grad, loss = np.empty(m, np.float32), np.empty_like(p), C.c_double()
    ctx.check(ctx.lib.mda_mlp_forward(ctx.h, p.ctypes.data, feat.ctypes.data, m,
                                      rho.ctypes.data, 0))
    ctx.check(ctx.lib.mda_mlp_loss_grad(ctx.h, p.ctypes.data, feat.ctypes.data,
                                        target.ctypes.data, m, C.byref(loss), grad.ctypes.data, 0))
    p64, f64 = p.astype(np.float64), feat.astype(np.float64)
    # FP32 sums of 64 terms, twice: 64 eps at most on values of order one
    np.testing.assert_allclose(rho, orc.mlp_forward(p64, f64), rtol=64 * 6e-8)
    lo, go = orc.mlp_loss_grad(p64, f64, target.astype(np.float64))
    assert abs(loss.value - lo) <= 128 * 6e-8 * max(lo, 1e-3)
    assert np.linalg.norm(grad - go) <= 128 * 6e-8 * np.linalg.norm(go)


# ---- observation sorts: one workgroup up to 4096, 1024 or 4096 keys a block beyond ----------
@pytest.mark.parametrize("p", [3, 1023, 1025, 4095, 4096, 4097, 30000, 262143, 262150])
def test_observation_order_matches_oracle(mda, ctx, orc, p):
    """Local sets and the analysis through both sorts (buckets and first
    stencil taps) and a multi-level state."""
    rng = np.random.default_rng(p)
    nlon, nlat, nlev, k = 24, 12, 9, 8
    lonc, latc = (np.arange(nlon) + 0.5) * 15.0, -90 + (np.arange(nlat) + 0.5) * 15.0
    col_lon, col_lat = (v.ravel().copy() for v in np.meshgrid(lonc, latc))
    lat, lon = np.degrees(np.arcsin(rng.uniform(-1, 1, p))), rng.uniform(0, 360, p)
    H = mda.ObsOperator.trilinear_latlon(lat, lon, rng.uniform(0, nlev - 1, p), nlon, nlat, nlev)
    X = rng.standard_normal((k, nlon * nlat * nlev))
    yo, var = rng.standard_normal(p), rng.uniform(1, 2, p) * max(1.0, p / 500.0)
    ens = mda.Ensemble(X.copy(), nlon, nlat, nlev)
    f = mda.LETKF(ens, mda.Observation(yo, var, lat, lon, coord=mda._lib.COORD_GEOGRAPHIC), H,
                  mda.Config({"inflation": 1.05, "localization_radius": 900.0}),
                  geometry=mda.ColumnGeometry(mda._lib.COORD_GEOGRAPHIC, col_lat, col_lon),
                  ctx=ctx)
    f.Analyse()
    prob = orc.Problem(k, nlon, nlat, nlev, orc.COORD_GEOGRAPHIC, col_lat, col_lon, lat, lon, yo,
                       var, f.inflation, f.localization_radius)
    Xo, _, nloc = orc.letkf_standard(prob, X, H.apply_host(X))
    np.testing.assert_array_equal(f.local_counts(), nloc)
    assert rel_err(ens.data, Xo) < TOL


# ---- host arrays: staged together up to 512 KB each and 4 MB in all, copied singly beyond ----
@pytest.mark.parametrize("nx,p", [(64, 10), (8192, 500), (8193, 500), (8192, 65536),
                                  (8000, 65537), (9000, 130000)])
def test_host_arrays_equal_device_arrays(mda, ctx, nx, p):
    """The same analyses from host arrays and from device tensors, to the last
    bit, one call right after the other on one context."""
    import torch
    rng = np.random.default_rng(nx + p)
    k = 8
    X, x = rng.standard_normal((k, nx)), rng.uniform(0, nx - 1, p)
    i = np.minimum(x.astype(np.int64), nx - 2)
    col, w = np.stack([i, i + 1], 1).ravel(), np.stack([i + 1 - x, x - i], 1).ravel()
    rp = np.arange(0, 2 * p + 1, 2)
    yo, var, Z = rng.standard_normal(p), rng.uniform(1, 2, p) * 50, rng.standard_normal((p, k))
    out = {}
    for where in ("host", "device", "host again"):
        t = (lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()) if where == "device" \
            else (lambda a: a.copy())
        obs = mda.Observation(t(yo), t(var), t(x), t(np.zeros(p)))
        H = mda.ObsOperator(t(rp), t(col), t(w))
        a, b = (mda.Ensemble(t(X), nx, 1, 1) for _ in range(2))
        torch.cuda.synchronize()
        mda.LETKF(a, obs, H, mda.Config({"inflation": 1.05, "localization_radius": 12.0}),
                  ctx=ctx).Analyse()
        f = mda.EnKF(b, obs, H, mda.Config({"analysis": {"inflation": 1.1}}), ctx=ctx)
        f.Analyse(Z=t(Z))
        r = f.getAnalysisResults()
        out[where] = (a.to_host(), b.to_host(), [r["max_kalman_gain"], r["analysis_spread"]])
    for where in ("device", "host again"):
        for u, v in zip(out["host"], out[where]):
            np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("k", [2, 3, 9, 17, 65, 81, 97])
def test_metrics_crps_with_an_outlying_first_member(mda, ctx, k):
    """One point, member 0 at the power of two V, the others at zero, V so large
    that its 2 (k - 1) differences add up to at most 1.2e308: whole multiples
    of V, exact.  The score is V / k - (k - 1) V / k^2 = V / k^2, off by the
    rounding of the two quotients (eps / 2 of V / k each) and of their
    difference; a pair sum with more copies of member 0 would overflow."""
    V = 2.0 ** np.floor(np.log2(0.6e308 / (k - 1)))
    X = np.zeros((k, 1))
    X[0] = V
    m = mda.metrics(mda.Ensemble(X, 1, 1, 1), np.zeros(1), ctx=ctx)
    assert abs(m["crps"] / (V / k / k) - 1.0) <= (k + 3) * np.finfo(float).eps


# ---- FP64 ensembles between the block sizes: as close to 64 bits as Jacobi ------------------
S = 120  # binary places of the whole numbers below


def _fixed(v):
    """A float64 array as whole numbers of 2^-S, without rounding above 2^-S."""
    return np.array([int(np.ldexp(x, 60)) << (S - 60) if abs(x) > 1e-2 else int(np.ldexp(x, S))
                     for x in np.ravel(v)], object).reshape(np.shape(v))


def _float(v, places):
    return np.array([float(x) for x in np.ravel(v)]).reshape(np.shape(v)) * 2.0 ** -places


def _exact_transform(A, b, k, factor):
    """A^-1 b 1^T + factor sqrt(k-1) A^-1/2 in whole numbers of 2^-S, for
    whole-number A and b: float64 steps on residuals without rounding."""
    lam, V = np.linalg.eigh(A.astype(float))
    root = np.sqrt(lam)
    Z, w = _fixed((V / root) @ V.T), _fixed(np.zeros(k))
    eye = np.array([[(1 << 2 * S) * int(i == j) for j in range(k)] for i in range(k)], object)
    for _ in range(3):
        R = _float(eye - Z.dot(A.dot(Z)), 2 * S)
        Z = Z + _fixed(V @ ((V.T @ R @ V) / (root[:, None] + root)) @ V.T)
        w = w + _fixed(V @ ((V.T @ _float((b << S) - A.dot(w), S)) / lam))
    assert np.abs(R).max() < 1e-9  # of the last but one; the last step squares it
    return w[:, None] + (factor * math.isqrt((k - 1) << 2 * S) * Z >> S)


@pytest.mark.parametrize("var", [16.0, 1.0, 2.0 ** -6])
@pytest.mark.parametrize("p", [5, 300])
@pytest.mark.parametrize("k", [2, 7, 9, 15, 17, 21, 31, 33, 39, 41, 47, 50, 63, 65, 100, 127])
def test_letkf_between_blocks_is_as_accurate_as_jacobi(mda, ctx, k, p, var):
    """Whole-number H(x) of mean zero, a cutoff of weight one and a power of two
    as variance make Gram and right-hand side exact, so T = wbar 1^T + W can be
    held against its exact value: no further off than Jacobi's, or at rounding
    level."""
    L = mda._lib
    rng = np.random.default_rng(k * 1000 + p)
    Yb = rng.integers(-8, 9, (k, p)).astype(float)
    Yb[:, 1:] += 2 * Yb[:, :1]  # correlated: eigenvalues far apart
    Yb[-1] -= Yb.sum(0)
    yo = rng.integers(-20, 21, p).astype(float)
    out = {}
    for method in ("AUTO", "JACOBI"):
        ens = mda.Ensemble(rng.standard_normal((k, 12)), 4, 3, 1)
        f = mda.LETKF(ens, mda.Observation(yo, np.full(p, var), np.ones(p), np.ones(p)),
                      mda.ObsOperator(hx=Yb), mda.Config({"inflation": 1.0,
                                                          "localization_radius": 50.0}),
                      ctx=ctx, eig_method=getattr(L, "EIG_" + method), keep_transforms=True)
        f.params.localization = L.LOC_CUTOFF
        f.Analyse()
        out[method] = f.transforms([0, 11])
    # whole numbers: unit A and unit b, unit = 16 or 1, with the root's factor 4 or 1
    unit = max(var, 1.0)
    A = (Yb @ Yb.T * (unit / var) + unit * (k - 1) * np.eye(k)).astype(np.int64).astype(object)
    b = (Yb @ yo * (unit / var)).astype(np.int64).astype(object)
    T = _exact_transform(A, b, k, math.isqrt(int(unit)))
    size = np.sqrt((_float(T, S) ** 2).sum())
    err = {m: max(np.sqrt((_float(_fixed(t) - T, S) ** 2).sum()) for t in v) / size
           for m, v in out.items()}
    # 8 eps: the rounding of T itself and of wbar's two products
    assert err["AUTO"] <= max(err["JACOBI"], 8 * np.finfo(float).eps), err


@pytest.mark.parametrize("combine", ["MATRIX", "ELEMENTWISE"])
@pytest.mark.parametrize("form", ["PRIOR", "POSTERIOR"])
@pytest.mark.parametrize("k", [5, 13, 18, 25, 36, 44, 50, 90])
def test_letkf_between_blocks_every_form_matches_jacobi(mda, ctx, monkeypatch, k, form, combine):
    """Inflation forms, combinations, an inflation per column, empty columns,
    one pass and passes of 50 columns."""
    L = mda._lib
    case = latlon_case(nlon=18, nlat=9, nlev=3, k=k, p=350, seed=900 + k, cluster=True, nmodes=96)
    rho = np.random.default_rng(k).uniform(1.0, 1.4, 162)
    X = {}
    for method, chunk in (("JACOBI", None), ("AUTO", None), ("AUTO", "50")):
        if chunk:
            monkeypatch.setenv("MDA_LETKF_CHUNK_COLS", chunk)
        ens = mda.Ensemble(case["X"].copy(), 18, 9, 3)
        f = mda.LETKF(ens, mda.Observation(case["yo"], case["var"], case["lat"], case["lon"],
                                           coord=L.COORD_GEOGRAPHIC), case["H"],
                      mda.Config({"inflation": 1.1, "localization_radius": 1800.0}),
                      geometry=mda.ColumnGeometry(L.COORD_GEOGRAPHIC, case["col_lat"],
                                                  case["col_lon"]), ctx=ctx, rho_column=rho,
                      eig_method=getattr(L, "EIG_" + method))
        f.params.inflation_form = getattr(L, "INFLFORM_" + form)
        f.params.combine = getattr(L, "COMBINE_" + combine)
        f.Analyse()
        assert f.diag["n_empty_columns"] > 0
        X[method, chunk] = ens.data.copy()
    np.testing.assert_array_equal(X["AUTO", "50"], X["AUTO", None])
    assert rel_err(X["AUTO", None], X["JACOBI", None]) < TOL


@pytest.mark.parametrize("prec", ["FP32", "BF16X3"])
@pytest.mark.parametrize("k,radius,few_columns", [(10, 500.0, True), (25, 1500.0, True),
                                                  (50, 1500.0, True), (50, 9000.0, False),
                                                  (100, 9000.0, False)])
def test_letkf_reduced_precision_between_blocks_solver(mda, ctx, orc, k, radius, few_columns, prec):
    """Which solver a reduced-precision Gram gets at a size between the blocks:
    BF16x3 Jacobi for every column, FP32 the tridiagonal one, which columns with
    fewer than k observations leave at once (and others by its checks); the
    analysis within the 1e-4 of the FP64 oracle that these contractions are
    stated to keep."""
    L = mda._lib
    case = latlon_case(nlon=18, nlat=9, nlev=2, k=k, p=700, seed=400 + k, nmodes=96)
    f, X = _latlon(mda, ctx, case, case["X"], radius, precision=getattr(L, "PREC_" + prec))
    nloc = f.local_counts()
    few = int(((nloc > 0) & (nloc < k)).sum())
    assert (few > 0) == few_columns
    if prec == "BF16X3":
        assert f.diag["n_fallback_columns"] == 0 and f.diag["max_jacobi_sweeps"] > 0
        assert not f.column_flags().any()
    else:
        assert few <= f.diag["n_fallback_columns"]
        assert (f.column_flags()[(nloc > 0) & (nloc < k)] == 16).all()
    prob = orc.Problem(k, 18, 9, 2, orc.COORD_GEOGRAPHIC, case["col_lat"], case["col_lon"],
                       case["lat"], case["lon"], case["yo"], case["var"],
                       float(np.float32(1.05)), float(np.float32(radius)))
    Xo, _, _ = orc.letkf_standard(prob, case["X"], case["H"].apply_host(case["X"]))
    inc = Xo - case["X"]
    assert np.sqrt(((X - Xo) ** 2).mean()) < 1e-4 * np.sqrt((inc ** 2).mean())
