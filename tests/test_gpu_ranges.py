"""Analyses at the sizes where a kernel's tiles, its search or the rule that
chooses it can go wrong, against the oracle."""
import numpy as np
import pytest

from cases import rel_err

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
