"""Coordinates and weights that are NaN, infinite or negative, compared bit for bit
with the oracle through every form of the neighbour stages."""
import numpy as np
import pytest

from cluestering_amd import CLUE_Convolutional_Kernels as K

from _support import Case, assert_same

pytestmark = pytest.mark.gpu

# None: the library's choice (teams of waves at these sizes). The others keep one wave
# per item: over candidate blocks, scanning whole tiles, and in the tiles' own order.
TUNINGS = [None, dict(group_queries=True), dict(group_queries=True, nh_plain_scan=True),
           dict(group_queries=False)]

METRICS = [None, K.EuclideanMetric([1.0, 2.0]), K.EuclideanMetric([1.0, 0.0]),
           K.PeriodicEuclideanMetric([0.0, 90.0]), K.PeriodicEuclideanMetric([110.0, 90.0]),
           K.ManhattanMetric(), K.ChebyshevMetric(), K.ChebyshevMetric([1.0, 2.0]),
           K.MahalanobisMetric()]


def _check(case, ctx, oracle, tuning=None):
    print(f"[case] {case.name} n={case.n} ndim={case.ndim} {case.dtype}", flush=True)
    if tuning is not None:
        ctx.set_tuning(xcd_chunk_log2=4, block_waves=1, **tuning)
    try:
        gpu = case.run_gpu(ctx)
    finally:
        ctx.set_tuning()
    assert_same(gpu, case.run_oracle(oracle), case.name)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tuning", TUNINGS)
@pytest.mark.parametrize("metric", METRICS)
@pytest.mark.parametrize("special", [np.nan, np.inf])
def test_special_coordinates(gpu_ctx, oracle_mod, special, metric, tuning, dtype):
    """Some points have NaN or infinite coordinates, in one dimension or both. The
    Chebyshev distances leave a NaN difference out of their maximum, so such a point
    is near others by its other coordinates; under the other metrics it is near none.
    Flat kernel: beyond the radius, the oracle's other kernels make a NaN distance a NaN
    density of every point that looks at the candidate's tile."""
    for n, ppt, every in ((120, 1000, 120), (3000, 0, 97), (3000, 12, 10)):
        rng = np.random.default_rng(n + ppt)
        x = rng.uniform(0, 100 if n == 120 else 60, (2, n))
        odd = np.arange(0, n, every)
        x[rng.integers(0, 2, odd.size), odd] = special
        x[:, odd[::7]] = special
        if np.isinf(special):
            x[:, odd] *= rng.choice([-1.0, 1.0], odd.size)
        sigma = rng.uniform(0.5, 1.5, (2, n)) if metric is not None and metric.tag == "mahalanobis" else None
        _check(Case(x, rng.uniform(0.5, 1.5, n), 5.0 if n == 120 else 2.0, 3.0, 6.0 if n == 120 else 3.0,
                    metric=metric, sigma=sigma, points_per_tile=ppt, dtype=dtype,
                    name=f"{special} {metric} {tuning} ppt={ppt}"), gpu_ctx, oracle_mod, tuning)


@pytest.mark.parametrize("kernel", [K.ExponentialKernel(0.5, 1.0), K.GaussianKernel(0.8, 1.3)])
@pytest.mark.parametrize("tuning", TUNINGS)
def test_nan_coordinates_chebyshev_kernels(gpu_ctx, oracle_mod, tuning, kernel):
    """The Chebyshev distances of NaN coordinates are numbers, also under the kernels
    that compute with them; three dimensions, one of them NaN in whole tiles."""
    rng = np.random.default_rng(11)
    n = 4000
    x = rng.uniform(0, 20, (3, n))
    x[1, rng.random(n) < 0.05] = np.nan
    x[2, x[0] < 3] = np.nan
    for metric in (K.ChebyshevMetric(), K.ChebyshevMetric([1.0, 0.5, 2.0])):
        _check(Case(x, rng.uniform(0.5, 1.5, n), 1.5, 3.0, 2.5, kernel=kernel, metric=metric,
                    points_per_tile=40, name=f"nan {metric} {kernel} {tuning}"), gpu_ctx, oracle_mod, tuning)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tuning", TUNINGS)
def test_negative_metric_weight_out_of_box(gpu_ctx, oracle_mod, tuning, dtype):
    """A negative metric weight makes the sum under the root negative: here between
    the first point and the third, whose tile its search box does not hold, while the
    second point, of the first's tile, looks at it. No pair within a search box
    has a negative sum."""
    x = np.array([[0.0, 2.0, 0.0, 10.0], [0.0, 4.8, 5.6, 10.0]])
    _check(Case(x, [1.0, 2.0, 4.0, 8.0], 0.5, 1.0, 0.5, metric=K.EuclideanMetric([1.0, -0.02]),
                points_per_tile=1, dtype=dtype, name=f"negative weight {tuning}"), gpu_ctx, oracle_mod,
           tuning)


def test_runs_after_an_error(gpu_ctx, oracle_mod):
    """An error left by another call ends a launch early, with its copies and kernels under
    way. The calls that follow wait for them before they write the descriptors again."""
    rng = np.random.default_rng(8)
    cases = []
    for sizes in ([700] * 40, [9000, 3, 2500]):
        n = sum(sizes)
        cases.append(Case(rng.uniform(0, 30, (2, n)), rng.uniform(0.5, 1.5, n), 1.0, 3.0, 1.5, sizes=sizes,
                          name=f"after an error, {len(sizes)} events"))
    refs = [c.run_oracle(oracle_mod) for c in cases]
    points = [c.points(gpu_ctx) for c in cases]
    for k in (0, 1, 0, 1):
        with pytest.raises(Exception):
            gpu_ctx.empty(1 << 50, np.uint8)
        try:
            cases[1 - k].clusterer(gpu_ctx).make_clusters_batched(points[1 - k], cases[1 - k].sizes)
        except Exception:
            pass  # the error that was left
        cases[k].clusterer(gpu_ctx).make_clusters_batched(points[k], cases[k].sizes)
        out = points[k].results()
        out["seeds"] = None
        assert_same(out, refs[k], cases[k].name)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tuning", TUNINGS)
@pytest.mark.parametrize("n", [40, 3000])
def test_flat_sums_with_weights_beyond_numbers(gpu_ctx, n, tuning, dtype):
    """Flat kernel, unit weights but for one infinite, one NaN and two whose sum overflows:
    their neighbours' sums are infinite or NaN, every other point's is exact, though
    the waves that met them take their sums again with selects."""
    from cluestering_amd.device import Clusterer, PointsDevice
    rng = np.random.default_rng(78)
    xy = rng.uniform(0, np.sqrt(n) * 0.7, size=(2, n)).astype(dtype)
    xy[:, :6] = [[-9.0, -8.5, 90.0, 90.5, 200.0, 200.5], np.zeros(6)]
    w = np.ones(n, dtype)
    w[1], w[3] = np.inf, np.nan
    w[4] = w[5] = np.finfo(dtype).max * 0.75
    if tuning is not None:
        gpu_ctx.set_tuning(xcd_chunk_log2=4, block_waves=1, **tuning)
    try:
        p = PointsDevice.from_host(gpu_ctx, xy, w, dtype=dtype)
        Clusterer(gpu_ctx, 1.0, 2.0).make_clusters(p, None, K.FlatKernel(0.5))
    finally:
        gpu_ctx.set_tuning()
    rho = p.rho.to_host()
    x, y = xy
    near = np.sqrt((x[:, None] - x[None]) ** 2 + (y[:, None] - y[None]) ** 2) <= 1
    want = 0.5 * near.sum(1) + 0.5   # the point itself counts 1
    assert rho[0] == np.inf and rho[1] == np.inf and rho[4] == np.inf and rho[5] == np.inf
    assert np.isnan(rho[2]) and np.isnan(rho[3])
    np.testing.assert_array_equal(rho[6:], want[6:].astype(dtype))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tuning", TUNINGS)
@pytest.mark.parametrize("metric", [None, K.ManhattanMetric(), K.ChebyshevMetric()])
def test_flat_sums_at_extreme_radii(gpu_ctx, oracle_mod, metric, tuning, dtype):
    """Radii whose threshold times a power of two cannot stand for the comparison (too
    small, too large, infinite), beside ones where it can."""
    rng = np.random.default_rng(12)
    n = 500
    tiny, huge = (1e-10, 1e19) if dtype == np.float32 else (1e-19, 1e37)
    for dc in (tiny, tiny * 100, huge, huge / 100, np.inf):
        scale = 1.0 if np.isinf(dc) else dc
        x = np.round(rng.uniform(0, 4, (2, n)), 1) * scale
        _check(Case(x, rng.uniform(0.5, 1.5, n), dc, 3.0, dc, metric=metric, points_per_tile=50, dtype=dtype,
                    name=f"radius {dc} {metric} {tuning}"), gpu_ctx, oracle_mod, tuning)
