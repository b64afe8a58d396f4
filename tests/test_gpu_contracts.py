"""What calls promise each other: results that stay readable, calls that are
accepted, errors that leave things as they were."""
import ctypes as C

import numpy as np
import pytest

from cases import latlon_case, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mda():
    import metada_amd
    return metada_amd


@pytest.fixture()
def ctx(mda):
    c = mda.Context(0)
    yield c
    c.close()


def _letkf(mda, ctx, case, radius, **kw):
    L = mda._lib
    ens = mda.Ensemble(case["X"].copy(), case["nlon"], case["nlat"], case["nlev"])
    f = mda.LETKF(ens, mda.Observation(case["yo"], case["var"], case["lat"], case["lon"],
                                       coord=L.COORD_GEOGRAPHIC), case["H"],
                  mda.Config({"inflation": 1.05, "localization_radius": radius}),
                  geometry=mda.ColumnGeometry(L.COORD_GEOGRAPHIC, case["col_lat"],
                                              case["col_lon"]), ctx=ctx, **kw)
    return f, ens


def _flags(ctx, ncol):
    out = np.full(ncol, -1, np.int32)
    ctx.check(ctx.lib.mda_letkf_last_column_flags(ctx.h, out.ctypes.data))
    return out


def _features(ctx, f):
    from metada_amd.analysis import _obs_struct
    es, ek = f.ensemble.struct()
    gs, gk = f.geometry.struct()
    os_, ok = _obs_struct(f.obs)
    hs, hk = f.obs_op.struct()
    out = np.empty((es.nx * es.ny, 8), np.float32)
    ctx.check(ctx.lib.mda_letkf_inflation_features(ctx.h, C.byref(f.params), C.byref(es),
                                                   C.byref(gs), C.byref(os_), C.byref(hs), None,
                                                   out.ctypes.data, 0))
    return out


# ---- inflation features between an analysis and the reading of its results ------------------
@pytest.mark.parametrize("k,prec", [(25, "FP32"), (50, "BF16X3"), (16, "FP64")])
def test_features_leave_the_last_analysis_readable(mda, ctx, k, prec):
    """Column flags (FP32 between the block sizes: columns with fewer than k
    observations are flagged), counts and kept transforms are the analysis's
    own after a features call on the same problem and on a larger one (more
    columns, larger blocks)."""
    case = latlon_case(nlon=18, nlat=9, nlev=2, k=k, p=300, seed=500 + k)
    f, ens = _letkf(mda, ctx, case, 1500.0, precision=getattr(mda._lib, "PREC_" + prec),
                    keep_transforms=True)
    f.Analyse()
    cols = np.array([0, 40, 161])
    flags, counts, T = _flags(ctx, 162), f.local_counts().copy(), f.transforms(cols)
    if prec == "FP32":
        assert (flags != 0).any()
    feat = _features(ctx, f)
    big = latlon_case(nlon=36, nlat=18, nlev=2, k=64, p=900, seed=600 + k)
    _features(ctx, _letkf(mda, ctx, big, 1500.0)[0])
    np.testing.assert_array_equal(_flags(ctx, 162), flags)
    np.testing.assert_array_equal(f.local_counts(), counts)
    np.testing.assert_array_equal(f.transforms(cols), T)
    # and the features are those of a context that has run nothing else
    c2 = mda.Context(0)
    f2, e2 = _letkf(mda, c2, case, 1500.0)
    e2.data[:] = ens.data
    np.testing.assert_array_equal(_features(c2, f2), feat)
    c2.close()


# ---- gain extremes when no entry of the gain is a number ------------------------------------
def test_lwenkf_extremes_of_a_gain_without_numbers(mda, ctx):
    """A background of NaN with finite H(x): the LWEnKF has no gain entry to
    compare and reports the empty maximum and minimum, -inf and +inf."""
    k, n, p = 8, 200, 20
    rng = np.random.default_rng(3)
    ens = mda.Ensemble(np.full((k, n), np.nan), n, 1, 1)
    f = mda.LWEnKF(ens, mda.Observation(rng.standard_normal(p), np.ones(p), np.zeros(p),
                                        np.zeros(p)),
                   mda.ObsOperator(hx=rng.standard_normal((k, p))),
                   mda.Config({"analysis": {"inflation": 1.1, "localization_radius": 0.3,
                                            "localization_function": "gaussian",
                                            "weighting_scheme": "uniform"}}), ctx=ctx)
    f.Analyse(Z=rng.standard_normal((p, k)))
    r = f.getAnalysisResults()
    assert r["max_kalman_gain"] == -np.inf and r["min_kalman_gain"] == np.inf


# ---- transforms without keep_transforms ------------------------------------------------------
@pytest.mark.parametrize("prec", ["FP64", "FP32", "BF16X3"])
@pytest.mark.parametrize("k", [7, 10, 15, 21, 25, 31, 41, 47, 49, 50, 63, 80])
def test_transforms_between_block_sizes_are_readable(mda, ctx, k, prec):
    """Only k in {16, 32, 48, 64} need keep_transforms: elsewhere the default
    stores T, the same one, and the analysis is the same to the bit."""
    case = latlon_case(nlon=18, nlat=9, nlev=3, k=k, p=400, seed=800 + k)
    kw = {"precision": getattr(mda._lib, "PREC_" + prec)}
    cols = np.array([0, 40, 80, 161])
    f, ens = _letkf(mda, ctx, case, 2500.0, **kw)
    f.Analyse()
    T = f.transforms(cols)
    g, ens_kept = _letkf(mda, ctx, case, 2500.0, keep_transforms=True, **kw)
    g.Analyse()
    np.testing.assert_array_equal(T, g.transforms(cols))
    np.testing.assert_array_equal(ens.data, ens_kept.data)


# ---- elimination that meets no finite number -------------------------------------------------
@pytest.mark.parametrize("p,where", [(5, 0), (16, 15), (40, 20), (300, 17), (1030, 1029)])
@pytest.mark.parametrize("size", [1e160, 1e308])
def test_lwenkf_infinite_covariance_is_an_error(mda, ctx, p, where, size):
    """One observation whose spread overflows S (to infinities, or to NaN off
    the diagonal): MDA_E_NUMERIC, and the ensemble as it was."""
    k, n = 6, 50
    rng = np.random.default_rng(p)
    Yb = rng.standard_normal((k, p))
    Yb[:, where] = size * np.array([1, -1, 1, -1, 1, -1])
    X = rng.standard_normal((k, n))
    ens = mda.Ensemble(X.copy(), n, 1, 1)
    f = mda.LWEnKF(ens, mda.Observation(rng.standard_normal(p), np.ones(p), np.zeros(p),
                                        np.zeros(p)),
                   mda.ObsOperator(hx=Yb),
                   mda.Config({"analysis": {"inflation": 1.1, "localization_radius": 0.3,
                                            "localization_function": "gaussian",
                                            "weighting_scheme": "uniform"}}), ctx=ctx)
    with pytest.raises(mda._lib.MdaError) as e:
        f.Analyse(Z=rng.standard_normal((p, k)))
    assert e.value.code == -4
    np.testing.assert_array_equal(ens.data, X)
