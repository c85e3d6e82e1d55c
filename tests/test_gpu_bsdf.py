"""GPU hair BSDF (FP32) against the FP64 oracle restating disney_hair.cuh.
Bar: relative error <= 1e-5 on 2^20 seeded queries,
measured where the FP64 value is above 1e-7 x the batch median."""
import numpy as np
import pytest

from tests import oracle_lib as ol
from tests.gen import ALPHA_2DEG, bsdf_queries, uniforms

pytestmark = pytest.mark.gpu

N = 1 << 20


def rel_err(g, o):
    floor = 1e-7 * np.median(np.abs(o[o > 0])) if np.any(o > 0) else 1e-30
    m = np.abs(o) > floor
    return np.abs(g[m] - o[m]) / np.abs(o[m]), m


@pytest.mark.parametrize("params", [(0.3, 0.3, ALPHA_2DEG), (0.6, 0.5, 0.0), (0.15, 0.6, 3 * ALPHA_2DEG)])
def test_eval_matches_fp64(gpu, params):
    q = bsdf_queries(N, seed=1234)
    prm = ol.hair_params(*params)
    f64, p64 = ol.hair_eval(q, prm, 0)
    f32, p32 = gpu.hair_bsdf_eval(q, *params)
    ef, _ = rel_err(f32.astype(np.float64), f64)
    ep, _ = rel_err(p32.astype(np.float64), p64)
    print(f"params={params} f: p99.9={np.quantile(ef, 0.999):.2e} max={ef.max():.2e}; "
          f"pdf: p99.9={np.quantile(ep, 0.999):.2e} max={ep.max():.2e}")
    assert np.quantile(ef, 0.999) <= 1e-5
    assert np.quantile(ep, 0.999) <= 1e-5
    assert ef.max() <= 1e-3 and ep.max() <= 1e-3


def test_eval_edge_inputs(gpu):
    """Grazing directions, h = +-1, sigma_a = 0 and large sigma_a stay finite."""
    q = bsdf_queries(4096, seed=7)
    q[:1024, 6] = np.float32(0.99999)
    q[1024:2048, 6] = np.float32(-0.99999)
    q[2048:3072, 7:10] = 0.0
    q[3072:, 7:10] = 50.0
    prm = ol.hair_params(0.3, 0.3, ALPHA_2DEG)
    f64, p64 = ol.hair_eval(q, prm, 0)
    f32, p32 = gpu.hair_bsdf_eval(q, 0.3, 0.3, ALPHA_2DEG)
    assert np.all(np.isfinite(f32)) and np.all(np.isfinite(p32))
    ef, _ = rel_err(f32.astype(np.float64), f64)
    print(f"edge inputs: p99 {np.quantile(ef, 0.99):.2e} max {ef.max():.2e}")
    # FP32 conditioning at |h| -> 1 and grazing angles: asin/atan2 near their
    # branch limits amplify one-ulp input differences
    assert np.quantile(ef, 0.99) <= 1e-4


def test_sample_matches_fp64(gpu):
    q = bsdf_queries(N // 4, seed=99)
    u = uniforms(q.shape[0], 4, 100)
    prm = ol.hair_params(0.3, 0.3, ALPHA_2DEG)
    wi64, f64, p64, l64 = ol.hair_sample(q, u, prm, 0)
    wi32, f32, p32, l32 = gpu.hair_bsdf_sample(q, u, 0.3, 0.3, ALPHA_2DEG)
    same_lobe = l32 == l64
    print(f"lobe agreement {same_lobe.mean():.6f}")
    assert same_lobe.mean() > 0.9999
    ang = np.linalg.norm(wi32.astype(np.float64) - wi64, axis=1)
    good = same_lobe & (ang < 1e-4)
    print(f"direction agreement {good.mean():.6f}, median angle {np.median(ang):.2e}")
    assert good.mean() > 0.999
    # the pdf returned with a sample equals the pdf of evaluating that direction
    qq = q.copy()
    qq[:, 3:6] = wi32
    fe, pe = gpu.hair_bsdf_eval(qq, 0.3, 0.3, ALPHA_2DEG)
    # same function, different kernels: FMA contraction may differ by an ulp
    np.testing.assert_allclose(pe, p32, rtol=2e-5, atol=1e-30)
    np.testing.assert_allclose(fe, f32, rtol=2e-5, atol=1e-30)
    # and the sampled f, pdf match the FP64 oracle where the direction matched
    e = np.abs(p32[good].astype(np.float64) - p64[good]) / p64[good]
    assert np.quantile(e, 0.999) <= 1e-4


def edge_queries(case, n=257):
    """A ragged count of queries beside the places where the streams change
    formula: the arc sine's halves (|h| = 1/2 and 1), the arc tangent's octants
    (tan(pi / 8), the axes with either sign of zero), the longitudinal lobe's
    Bessel argument of 12, directions along the fibre."""
    q = bsdf_queries(n, seed=11)
    if case == "h":
        q[:, 6] = np.resize(np.float32([0.5, np.nextafter(np.float32(0.5), np.float32(1)), -0.5, 0.0, -0.0, 0.99, -0.99]), n)
    elif case == "azimuth":
        a = np.resize(np.arange(-16, 17) * (np.pi / 16), n) + np.resize([0.0, 1e-7, -1e-7, 1e-3], n)
        r = np.sqrt(1.0 - q[:, 3].astype(np.float64) ** 2)
        q[:, 4], q[:, 5] = r * np.cos(a), r * np.sin(a)
        q[:, 1] = np.resize(np.float32([0.0, -0.0]), n)
        q[:, 2] = np.sqrt(1.0 - q[:, 0].astype(np.float64) ** 2) * np.resize([1.0, 1.0, -1.0], n)
    else:
        assert case == "along"
        q[:, 0] = np.resize(np.float32([1.0, -1.0]), n)
        q[:, 1:3] = np.resize(np.float32([0.0, 0.0, -0.0, 0.0, -0.0, -0.0]), 2 * n).reshape(n, 2)
    return q


@pytest.mark.parametrize("beta", [0.12, 0.3, 0.6])
@pytest.mark.parametrize("case", ["h", "azimuth", "along"])
def test_streams_at_the_edges_of_their_formulas(gpu, case, beta):
    """Against FP64: an azimuth off by a rounding (pi 2^-23) moves N_p by that
    over its scale s, a sine or cosine product off by two roundings moves M_p
    by those over v; three of the first and four of the second may add up. The
    lobe is the FP64 one wherever the draw is not beside an edge."""
    q = edge_queries(case)
    u = uniforms(q.shape[0], 4, 12)
    prm = ol.hair_params(beta, beta, ALPHA_2DEG)
    s = np.sqrt(np.pi / 8) * (0.265 * beta + 1.194 * beta**2 + 5.372 * beta**22)
    v = 0.25 * (0.726 * beta + 0.812 * beta**2 + 3.7 * beta**20) ** 2  # the narrowest lobe's
    tol = 2.0**-23 * (3 * np.pi / s + 4 / v) + 1e-6
    f64, p64 = ol.hair_eval(q, prm, 0)
    f32, p32 = gpu.hair_bsdf_eval(q, beta, beta, ALPHA_2DEG)
    for g, o in ((f32, f64), (p32, p64)):
        e = np.linalg.norm(g - o) / np.linalg.norm(o)
        print(f"{case} {beta}: {e:.2e} of {tol:.2e}")
        assert np.all(np.isfinite(g)) and e <= tol
    wi64, sf64, sp64, l64 = ol.hair_sample(q, u, prm, 0)
    wi32, sf32, sp32, l32 = gpu.hair_bsdf_sample(q, u, beta, beta, ALPHA_2DEG)
    same = l32 == l64
    assert same.sum() >= same.size - 1
    assert np.all(np.isfinite(wi32)) and np.abs(np.linalg.norm(wi32, axis=1) - 1).max() <= 4e-7
    # the direction's azimuth and inclination carry the rounding of a draw
    # next to 0 or 1 (2^-24 of it over the logistic's or the lobe's slope)
    assert np.quantile(np.linalg.norm(wi32 - wi64, axis=1)[same], 0.95) <= 2e-5
    e = np.abs(sp32[same] - sp64[same]) / sp64[same]
    assert np.median(e) <= tol


@pytest.mark.parametrize("beta", [0.3, 0.08])
def test_streams_with_opaque_fibres_and_draws_at_the_ends(gpu, beta):
    """An absorption that is infinite, or overflows over the fibre's length,
    transmits nothing, as in FP64; and draws of exactly 0 and 1 (the cdf at
    beta 0.08 reaches 0 and 1 in FP32) sample the lobes' ends. Directions: the
    azimuth is off by a rounding of pi at most (2^-22), the inclination's
    sine and cosine products by four of 2^-24. Values: as in
    test_streams_at_the_edges_of_their_formulas."""
    q = bsdf_queries(258, seed=5)
    q[:, 7] = np.resize(np.float32([np.inf, 1e38, 3e38, 100.0, 2000.0, 1e20]), 258)
    q[::3, 8] = np.inf
    q[::5, 7:10] = np.inf
    u = uniforms(258, 4, 6)
    u[:, 3] = np.resize(np.float32([0.0, 1.0, 2.0**-24]), 258)
    u[::7, 1] = np.resize(np.float32([0.0, 1.0]), u[::7].shape[0])
    prm = ol.hair_params(beta, beta, ALPHA_2DEG)
    s = np.sqrt(np.pi / 8) * (0.265 * beta + 1.194 * beta**2)
    v = 0.25 * (0.726 * beta + 0.812 * beta**2) ** 2
    tol = 2.0**-23 * (3 * np.pi / s + 4 / v) + 1e-6
    f32, p32 = gpu.hair_bsdf_eval(q, beta, beta, ALPHA_2DEG)
    for g, o in zip((f32, p32), ol.hair_eval(q, prm, 0)):
        assert np.all(np.isfinite(g)) and np.linalg.norm(g - o) <= tol * np.linalg.norm(o)
    wi64, _, _, l64 = ol.hair_sample(q, u, prm, 0)
    wi32, sf32, sp32, l32 = gpu.hair_bsdf_sample(q, u, beta, beta, ALPHA_2DEG)
    assert np.all(np.isfinite(wi32)) and np.all(np.isfinite(sf32)) and np.all(np.isfinite(sp32))
    np.testing.assert_array_equal(l32, l64)
    assert np.abs(wi32 - wi64).max() <= 2.0**-22 * np.pi + 4 * 2.0**-24 + 1e-6
