"""GPU parity: every output of the HIP path (rho, nearest_higher, delta, is_seed,
cluster_index, seeds) is compared bit for bit with the oracle on the same inputs."""
import numpy as np
import pytest

from cluestering_amd import CLUE_Convolutional_Kernels as K
from cluestering_amd import synthetic
from cluestering_amd.device import Plan, debug_math

from _support import Case, assert_same
from conftest import read_points

pytestmark = pytest.mark.gpu


def _workload_case(w, name):
    return Case(w.coords, w.weight, w.dc, w.rhoc, w.dm, kernel=w.kernel, metric=w.metric,
                wrapped=w.wrapped, sizes=w.sizes, name=name)


def _check(case, ctx, oracle):
    print(f"[case] {case.name} n={case.n} ndim={case.ndim}", flush=True)
    gpu = case.run_gpu(ctx)
    ref = case.run_oracle(oracle)
    assert_same(gpu, ref, case.name)
    seeds = np.nonzero(ref.is_seed)[0]
    np.testing.assert_array_equal(gpu["seeds"], seeds)
    return gpu, ref


def test_device_math_bits(gpu_ctx, oracle_mod):
    rng = np.random.default_rng(7)
    a = np.concatenate([
        rng.uniform(0, 10, 20000), rng.uniform(0, 1e-3, 5000), 10.0 ** rng.uniform(-40, 38, 5000),
        np.array([0.0, 1.0, 2.0, 2.25, 4.0, np.inf], np.float64)]).astype(np.float32)
    b = rng.uniform(0.1, 10, a.size).astype(np.float32)
    s, _, q = debug_math(gpu_ctx, a, b)
    np.testing.assert_array_equal(s.view(np.uint32), np.sqrt(a).view(np.uint32))
    np.testing.assert_array_equal(q.view(np.uint32), (a / b).view(np.uint32))
    x = np.concatenate([rng.uniform(-110, 90, 20000), rng.uniform(-2, 0, 5000),
                        np.array([0.0, -0.0, -87.3, 88.7, 89.0, -104.0, -103.9], np.float64)])
    x = x.astype(np.float32)
    _, e, _ = debug_math(gpu_ctx, x, np.ones_like(x))
    np.testing.assert_array_equal(e.view(np.uint32), oracle_mod.expf_array(x).view(np.uint32))


def _bits_range(lo_bits, hi_bits):
    return np.arange(lo_bits, hi_bits, dtype=np.uint32).view(np.float32)


def test_device_sqrt_correctly_rounded(gpu_ctx):
    """The stages' square root (hardware estimate + rounding test) equals the
    correctly rounded IEEE sqrt. Every float in [1, 4) covers both exponent
    parities of every mantissa; every float in [2^-97, 2^-94) and [2^126, +inf]
    covers the ends of the fast range; then specials and a random sample."""
    ranges = [(0x3F800000, 0x40800000),   # [1, 4)
              (0x0F000000, 0x10800000),   # [2^-97, 2^-94): the switch at 2^-96
              (0x7E800000, 0x7F800001)]   # [2^126, +inf]
    for lo, hi in ranges:
        a = _bits_range(lo, hi)
        s, _, _ = debug_math(gpu_ctx, a, np.ones_like(a))
        bad = np.nonzero(s.view(np.uint32) != np.sqrt(a).view(np.uint32))[0]
        assert bad.size == 0, f"range {lo:#x}: first mismatch at {a[bad[0]]!r}"
    rng = np.random.default_rng(8)
    a = np.concatenate([rng.integers(0, 0x7F800000, 1 << 22, dtype=np.uint32).view(np.float32),
                        np.array([0.0, -0.0, 1e-45, 1e-40, 1.17549435e-38, np.inf], np.float32)])
    s, _, _ = debug_math(gpu_ctx, a, np.ones_like(a))
    np.testing.assert_array_equal(s.view(np.uint32), np.sqrt(a).view(np.uint32))
    neg = np.array([-1.0, -1e-30, -np.inf, np.nan], np.float32)
    s, _, _ = debug_math(gpu_ctx, neg, np.ones_like(neg))
    assert np.isnan(s).all()


def test_blobs2d_16k(gpu_ctx, oracle_mod):
    _check(_workload_case(synthetic.blobs2d_16k(), "blobs2d_16k"), gpu_ctx, oracle_mod)


def test_blobs2d_uniform_weights_64k(gpu_ctx, oracle_mod):
    _check(_workload_case(synthetic.blobs2d_1m(n=1 << 16), "blobs2d_64k"), gpu_ctx, oracle_mod)


def test_detector3d_periodic_exp_64k(gpu_ctx, oracle_mod):
    _check(_workload_case(synthetic.detector3d_1m(n=1 << 16), "detector3d_64k"), gpu_ctx,
           oracle_mod)


def test_batched_gaussian(gpu_ctx, oracle_mod):
    w = synthetic.batch2d_4096(n_events=24, lo=256, hi=8192)
    gpu, ref = _check(_workload_case(w, "batch24"), gpu_ctx, oracle_mod)
    assert gpu["n_clusters"] == ref.n_seeds


@pytest.mark.parametrize("tuning", [(0, -1, 4, 0), (1, -1, 4, 0), (1, 0, 4, 0), (1, 4, 4, 0),
                                    (0, 6, 4, 0), (1, 12, 4, 0), (1, 2, 8, 0), (1, 4, 16, 0),
                                    (0, -1, 16, 0), (1, 4, 1, 1), (1, 6, 1, 32), (1, -1, 2, 8),
                                    (0, 12, 4, 16), (0, -1, 1, 1)])
def test_tunings_do_not_change_results(gpu_ctx, oracle_mod, tuning):
    """Every launch tuning (query grouping on/off, XCD chunking, waves per
    workgroup, persistent waves pulling from the work-item queues) gives the same
    bits: a 2-D gaussian batch with dense tiles and a 3-D periodic exponential
    event. (0, -1, 1, 1): one persistent wave per CU, far fewer than the batch's
    work items, beside the nearest-higher plain scan, which has no persistent
    form and keeps one wave per item."""
    from cluestering_amd import _capi
    group, xcd, waves, persistent = tuning
    gpu_ctx.set_tuning(group_queries=bool(group), xcd_chunk_log2=xcd, block_waves=waves,
                       persistent=persistent)
    try:
        for w, name in [(synthetic.batch2d_4096(n_events=12, lo=4096, hi=30000), "batch12"),
                        (synthetic.detector3d_1m(n=1 << 15), "detector3d_32k")]:
            # No values from an earlier run may survive in the workspace.
            _capi.check(_capi.load().clue_debug_poison(gpu_ctx.handle))
            _check(_workload_case(w, f"{name} tuning={tuning}"), gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("kernel", [K.FlatKernel(0.5), K.ExponentialKernel(0.5, 1.0),
                                    K.GaussianKernel(1.0, 1.0), K.FlatKernel(2.0),
                                    K.GaussianKernel(0.7, 1.3), K.ExponentialKernel(1.7, 0.8),
                                    K.GaussianKernel(0.5, 2.0)])
@pytest.mark.parametrize("metric", [None, K.EuclideanMetric(), K.EuclideanMetric([1.0, 2.0]),
                                    K.ManhattanMetric(), K.ChebyshevMetric(),
                                    K.ChebyshevMetric([1.0, 2.0])])
def test_kernels_and_metrics(gpu_ctx, oracle_mod, kernel, metric):
    c, w = read_points("data_4096.csv")
    w = np.random.default_rng(3).uniform(0.5, 1.5, w.size).astype(np.float32)
    _check(Case(c, w, 1.5, 10.0, 1.5, kernel=kernel, metric=metric, name=f"{kernel}-{metric}"),
           gpu_ctx, oracle_mod)


@pytest.mark.parametrize("ndim", list(range(1, 11)))
def test_dimensions(gpu_ctx, oracle_mod, ndim):
    rng = np.random.default_rng(100 + ndim)
    n = 3000
    centres = rng.uniform(0, 20, size=(6, ndim))
    lab = rng.integers(0, 6, n)
    x = (centres[lab] + rng.normal(0, 0.6, size=(n, ndim))).T.astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    _check(Case(x, w, 1.2 + 0.3 * ndim, 3.0, 2.0 + 0.3 * ndim, name=f"dim{ndim}"), gpu_ctx,
           oracle_mod)


def test_options_tags_uncertainty_sigma(gpu_ctx, oracle_mod):
    c, w = read_points("data_4096.csv")
    rng = np.random.default_rng(11)
    n = w.size
    tags = rng.permutation(n).astype(np.uint32)
    u = rng.uniform(0.5, 1.5, n).astype(np.float32)
    sigma = rng.uniform(0.0, 1.0, size=(2, n)).astype(np.float32)
    _check(Case(c, w, 1.5, 10.0, 1.5, tags=tags, name="tags"), gpu_ctx, oracle_mod)
    _check(Case(c, w, 1.5, 10.0, 1.5, u=u, name="uncertainty"), gpu_ctx, oracle_mod)
    _check(Case(c, w, 1.5, 10.0, 1.5, sigma=sigma, name="sigma"), gpu_ctx, oracle_mod)
    _check(Case(c, w, 1.5, 10.0, 1.5, sigma=sigma + 0.5, metric=K.MahalanobisMetric(),
                name="mahalanobis"), gpu_ctx, oracle_mod)
    _check(Case(c, w, 1.5, 10.0, 1.5, seed_dc=3.0, name="seed_dc"), gpu_ctx, oracle_mod)


def test_periodic_opposite_angles(gpu_ctx, oracle_mod):
    c, w = read_points("opposite_angles.csv")
    metric = K.PeriodicEuclideanMetric([0.0, float(2 * np.float32(np.pi))])
    gpu, _ = _check(Case(c, w, 0.2, 5.0, 0.2, metric=metric, wrapped=(0, 1), name="periodic"),
                    gpu_ctx, oracle_mod)
    assert gpu["cluster_index"].max() + 1 == 1  # tests/test_clustering.cpp:237-270


def test_tag_tie_break_known_answer(gpu_ctx, oracle_mod):
    # tests/test_clustering.cpp:517-567
    x = np.zeros((2, 2), np.float32)
    w = np.ones(2, np.float32)
    gpu, _ = _check(Case(x, w, 1.0, 0.0, 1.0, name="tie"), gpu_ctx, oracle_mod)
    assert list(gpu["nearest_higher"]) == [1, -1] and list(gpu["is_seed"]) == [0, 1]
    gpu, _ = _check(Case(x, w, 1.0, 0.0, 1.0, tags=np.array([100, 1], np.uint32), name="tie-tags"),
                    gpu_ctx, oracle_mod)
    assert list(gpu["nearest_higher"]) == [-1, 0] and list(gpu["is_seed"]) == [1, 0]


def test_mahalanobis_known_answer(gpu_ctx, oracle_mod):
    # tests/test_mahalanobis.cpp:10-43
    x = np.array([[2.0, 4.0]], np.float32)
    w = np.ones(2, np.float32)
    gpu, _ = _check(Case(x, w, 1.0, 0.3, name="maha-none"), gpu_ctx, oracle_mod)
    assert gpu["cluster_index"].max() + 1 == 2
    gpu, _ = _check(Case(x, w, 1.0, 0.3, metric=K.MahalanobisMetric(),
                         sigma=np.array([[2.0, 2.0]], np.float32), name="maha-sigma"),
                    gpu_ctx, oracle_mod)
    assert gpu["cluster_index"].max() + 1 == 1


def test_edge_cases(gpu_ctx, oracle_mod):
    _check(Case(np.array([[1.0], [2.0]], np.float32), np.ones(1, np.float32), 1.0, 0.5,
                name="single"), gpu_ctx, oracle_mod)
    x = np.full((2, 500), 3.0, np.float32)  # zero range in every dimension
    _check(Case(x, np.ones(500, np.float32), 1.0, 2.0, name="degenerate"), gpu_ctx, oracle_mod)
    c, w = read_points("data_1024.csv")
    for ppt in (1, 7, 100000):
        _check(Case(c, w, 1.5, 10.0, 1.5, points_per_tile=ppt, name=f"ppt{ppt}"), gpu_ctx,
               oracle_mod)
    _check(Case(c, w, 1.5, 1e9, 1.5, name="no-seeds"), gpu_ctx, oracle_mod)


def test_batched_with_empty_and_tiny_events(gpu_ctx, oracle_mod):
    from cluestering_amd.device import Clusterer, PointsDevice
    c, w = read_points("data_1024.csv")
    sizes = np.array([0, 300, 1, 0, 2, 721], np.uint32)
    _, ref = _check(Case(c, w, 1.3, 10.0, 1.3, sizes=sizes, name="ragged"), gpu_ctx, oracle_mod)
    # getSampleAssociations: the event of every cluster, in the caller's numbering.
    pts = PointsDevice.from_host(gpu_ctx, c, w)
    eoc = gpu_ctx.empty(w.size, np.int32)
    k = Clusterer(gpu_ctx, 1.3, 10.0, 1.3).make_clusters_batched(pts, sizes, event_of_cluster=eoc)
    assert k == ref.n_seeds
    np.testing.assert_array_equal(eoc.to_host()[:k], ref.event_of_cluster)


def test_batched_event_size_boundaries(gpu_ctx, oracle_mod):
    """Events on both sides of the seed stage's LDS limit (at most 32,768 points:
    links and labels resolved in LDS; above: jumping passes in memory and the label
    chase), with the event of every cluster, and lone events on both sides of the
    8,192 points up to which a lone event takes the fused per-event stages."""
    from cluestering_amd.device import Clusterer, PointsDevice
    rng = np.random.default_rng(17)
    sizes = np.array([32768, 32769, 45000, 100, 32767], np.uint32)
    parts = [synthetic._event2d(rng, int(n)) for n in sizes]
    c = np.ascontiguousarray(np.concatenate([p[0] for p in parts], axis=1))
    w = np.ascontiguousarray(np.concatenate([p[1] for p in parts]))
    kern = K.GaussianKernel(1.0, 1.0)
    _, ref = _check(Case(c, w, 1.5, 5.0, 2.0, kernel=kern, sizes=sizes, name="lds-boundary"),
                    gpu_ctx, oracle_mod)
    pts = PointsDevice.from_host(gpu_ctx, c, w)
    eoc = gpu_ctx.empty(w.size, np.int32)
    k = Clusterer(gpu_ctx, 1.5, 5.0, 2.0).make_clusters_batched(pts, sizes, None, kern,
                                                              event_of_cluster=eoc)
    assert k == ref.n_seeds
    np.testing.assert_array_equal(eoc.to_host()[:k], ref.event_of_cluster)
    for n in (8192, 8193):
        cn, wn = synthetic._event2d(rng, n)
        _check(Case(np.ascontiguousarray(cn), np.ascontiguousarray(wn), 1.5, 5.0, 2.0, kernel=kern,
                    name=f"lone-{n}"), gpu_ctx, oracle_mod)


def test_batched_reference_fixture(gpu_ctx, oracle_mod):
    # tests/test_batched_clustering.cpp:8-65: 10 copies of data_1024 give 10x the clusters.
    c, w = read_points("data_1024.csv")
    cb, wb = np.tile(c, (1, 10)), np.tile(w, 10)
    gpu, ref = _check(Case(cb, wb, 1.3, 10.0, 1.3, sizes=[1024] * 10, name="batched-fixture"),
                      gpu_ctx, oracle_mod)
    single = Case(c, w, 1.3, 10.0, 1.3).run_gpu(gpu_ctx)
    assert gpu["n_clusters"] == 10 * (single["cluster_index"].max() + 1)


def test_determinism_and_graph_replay(gpu_ctx, oracle_mod):
    w = synthetic.batch2d_4096(n_events=12, lo=256, hi=4096)
    case = _workload_case(w, "replay")
    ref = case.run_oracle(oracle_mod)
    clus = case.clusterer(gpu_ctx)
    pts = case.points(gpu_ctx)
    plan = Plan(clus, pts, w.sizes, case.metric, case.kernel)
    for rep in range(3):
        pts.cluster_index.fill_bytes(0xFF)
        pts.rho.fill_bytes(0)
        plan.launch()
        gpu_ctx.synchronize()
        out = pts.results()
        assert_same(out, ref, f"replay{rep}")
        # eager work between replays
        clus.make_clusters_batched(pts, w.sizes, case.metric, case.kernel)
        assert_same(pts.results(), ref, f"eager{rep}")
    plan.close()


def _blobs(ndim, n, seed, spread=0.6, n_centres=8):
    rng = np.random.default_rng(seed)
    centres = rng.uniform(0, 20, size=(n_centres, ndim))
    lab = rng.integers(0, n_centres, n)
    x = (centres[lab] + rng.normal(0, spread, size=(n, ndim))).T
    return x, rng.uniform(0.5, 1.5, n)


@pytest.mark.parametrize("metric", [None, K.EuclideanMetric([1.0, 2.5, 0.5]), K.ManhattanMetric(),
                                    K.ChebyshevMetric(), K.ChebyshevMetric([2.0, 1.0, 0.5]),
                                    K.PeriodicEuclideanMetric([0.0, 12.0, 0.0]),
                                    K.PeriodicEuclideanMetric([7.0, 9.0, 25.0]),
                                    K.EuclideanMetric([1.0, 0.0, 2.0])])
def test_nh_block_layout_matches_plain_scan(gpu_ctx, oracle_mod, metric):
    """The nearest-higher stage over Morton-ordered candidate blocks with box and
    key culling gives the plain scan's bits, for every metric with a box bound
    (a zero weight included), including flat-kernel densities full of exact ties
    and a batch of events."""
    from cluestering_amd import _capi
    x, w = _blobs(3, 12000, 41)
    wrapped = ()
    if metric is not None and metric.tag == "periodic_euclidean":
        wrapped = tuple(int(p > 0) for p in metric.params)
        for d, p in enumerate(metric.params):
            if p > 0:
                x[d] = np.mod(x[d], p)
    x = x.astype(np.float32)
    cases = [Case(x, w, 1.1, 6.0, 1.6, kernel=K.GaussianKernel(1.0, 1.0), metric=metric,
                  wrapped=wrapped, name=f"{metric}-gauss"),
             Case(x, np.ones_like(w), 0.9, 4.0, 1.4, kernel=K.FlatKernel(1.0), metric=metric,
                  wrapped=wrapped, name=f"{metric}-flat-ties"),
             Case(x, w, 1.1, 6.0, 2.2, seed_dc=2.8, kernel=K.ExponentialKernel(0.5, 1.0),
                  metric=metric, wrapped=wrapped, sizes=[3000, 64, 1, 8935], name=f"{metric}-batch"),
             # A search box wider than the grid: with wrapping, tiles recur in the walk.
             Case(x[:, :3000], w[:3000], 0.8, 2.0, 4.5, kernel=K.FlatKernel(0.5), metric=metric,
                  wrapped=wrapped, name=f"{metric}-wide-box")]
    try:
        for plain in (False, True):
            gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1,
                               nh_plain_scan=plain)
            for case in cases:
                _capi.check(_capi.load().clue_debug_poison(gpu_ctx.handle))
                case.name = f"{case.name.split(' plain=')[0]} plain={plain}"
                _check(case, gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("ndim", [1, 2, 5, 10])
def test_nh_block_layout_dimensions(gpu_ctx, oracle_mod, ndim):
    from cluestering_amd import _capi
    x, w = _blobs(ndim, 6000, 60 + ndim, spread=0.5)
    gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1)
    try:
        for dtype in (np.float32, np.float64):
            _capi.check(_capi.load().clue_debug_poison(gpu_ctx.handle))
            _check(Case(x, w, 0.9 + 0.3 * ndim, 3.0, 1.2 + 0.3 * ndim, name=f"dim{ndim}-{dtype.__name__}",
                        dtype=dtype), gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("plain", [False, True])
def test_duplicates_zero_and_negative_weights(gpu_ctx, oracle_mod, plain, dtype):
    """Exact duplicate points (zero distances, equal densities broken by tag) and
    weights that are zero or negative (densities <= 0, whose keys carry no tag),
    through both nearest-higher scans, bit for bit against the oracle."""
    from cluestering_amd import _capi
    rng = np.random.default_rng(77)
    base = rng.uniform(0, 12, size=(2, 1500)).astype(np.float32)
    x = np.concatenate([base, base[:, :700], base[:, :300]], axis=1)  # duplicates
    n = x.shape[1]
    w = rng.choice(np.array([1.0, 0.0, -0.5, 2.0], np.float32), size=n, p=[0.55, 0.15, 0.15, 0.15])
    gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1, nh_plain_scan=plain)
    try:
        for kernel in (K.FlatKernel(0.5), K.GaussianKernel(1.0, 1.0)):
            _capi.check(_capi.load().clue_debug_poison(gpu_ctx.handle))
            _check(Case(x, w, 0.9, 0.5, 1.3, kernel=kernel, dtype=dtype,
                        name=f"dups-{kernel} plain={plain} {np.dtype(dtype).name}"),
                   gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("plain", [False, True])
def test_large_tiles(gpu_ctx, oracle_mod, plain):
    """Tiles of thousands of points (points_per_tile = 3000): the block scan reads a
    tile's block boxes in several rounds of 64."""
    from cluestering_amd import _capi
    x, w = _blobs(2, 20000, 88, spread=1.5, n_centres=4)
    gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1, nh_plain_scan=plain)
    try:
        _capi.check(_capi.load().clue_debug_poison(gpu_ctx.handle))
        _check(Case(x, w, 0.7, 4.0, 1.1, kernel=K.GaussianKernel(1.0, 1.0), points_per_tile=3000,
                    name=f"large-tiles plain={plain}"), gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [40, 3000])
def test_flat_sums_with_infinite_and_nan_weights(gpu_ctx, n, dtype):
    """Flat kernel, unit weights but for one infinite and one NaN: their neighbours'
    sums are infinite or NaN, every other point's sum is exact and untouched."""
    from cluestering_amd.device import Clusterer, PointsDevice
    print(f"[case] non-finite weights n={n} {np.dtype(dtype)}", flush=True)
    rng = np.random.default_rng(77)
    xy = rng.uniform(0, np.sqrt(n) * 0.7, size=(2, n)).astype(dtype)
    xy[:, :4] = np.array([[-9.0, -8.5, 90.0, 90.5], [0.0, 0.0, 0.0, 0.0]], dtype)
    w = np.ones(n, dtype)
    w[1], w[3] = np.inf, np.nan
    p = PointsDevice.from_host(gpu_ctx, xy, w, dtype=dtype)
    Clusterer(gpu_ctx, 1.0, 2.0).make_clusters(p, None, K.FlatKernel(0.5))
    rho = p.rho.to_host()
    x, y = xy
    near = np.sqrt((x[:, None] - x[None]) ** 2 + (y[:, None] - y[None]) ** 2) <= 1
    want = 0.5 * near.sum(1) + 0.5   # the point itself counts 1
    assert rho[0] == np.inf and rho[1] == np.inf
    assert np.isnan(rho[2]) and np.isnan(rho[3])
    np.testing.assert_array_equal(rho[4:], want[4:].astype(dtype))


@pytest.mark.parametrize("kernel", [K.FlatKernel(0.5), K.ExponentialKernel(0.7, 1.2),
                                    K.GaussianKernel(1.0, 1.0), K.GaussianKernel(0.8, 1.3)])
@pytest.mark.parametrize("metric", [None, K.EuclideanMetric([1.0, 0.0]), K.ManhattanMetric(),
                                    K.ChebyshevMetric([1.0, 2.0]), K.MahalanobisMetric(),
                                    K.PeriodicEuclideanMetric([0.0, 40.0]),
                                    K.PeriodicEuclideanMetric([50.0, 40.0])])
def test_one_wave_per_item(gpu_ctx, oracle_mod, kernel, metric):
    """A fixed tuning keeps the kernels of large launches (one wave per item) at sizes
    that teams of waves would take."""
    c, w = read_points("data_4096.csv")
    rng = np.random.default_rng(5)
    w = rng.uniform(0.5, 1.5, w.size).astype(np.float32)
    sigma = rng.uniform(0.3, 1.0, size=c.shape).astype(np.float32) \
        if metric is not None and metric.tag == "mahalanobis" else None
    gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1)
    try:
        _check(Case(c, w, 1.5, 10.0, 1.7, kernel=kernel, metric=metric, sigma=sigma,
                    name=f"{kernel}-{metric}"), gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 63, 65, 255, 256, 257, 512, 1024, 1279, 1281, 4097])
def test_team_list_sizes(gpu_ctx, oracle_mod, n, dtype):
    """One tile whose points all reach each other: the teams' lists fill, empty and
    end at every boundary (8, 16, 64, 256 and 1,024 candidates and what is left)."""
    rng = np.random.default_rng(n)
    x = rng.normal(0, 0.4, size=(2, n)).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    for kernel in (K.FlatKernel(0.5), K.GaussianKernel(0.9, 1.0)):
        case = Case(x, w, 1.0, 3.0, 1.5, kernel=kernel, points_per_tile=100000, dtype=dtype,
                    name=f"list {n} {kernel}")
        print(f"[case] {case.name} {np.dtype(dtype)}", flush=True)
        assert_same(case.run_gpu(gpu_ctx), case.run_oracle(oracle_mod), case.name)


@pytest.mark.parametrize("fixed", [False, True])
def test_equal_tags_keep_the_first_candidate(gpu_ctx, oracle_mod, fixed):
    """Equal user tags, coordinates on a coarse grid and unit weights: many candidates
    agree in distance, density and tag, and the first in the reference's order wins."""
    rng = np.random.default_rng(9)
    n = 6000
    x = rng.integers(0, 40, size=(2, n)).astype(np.float32)
    w = np.ones(n, np.float32)
    tags = rng.integers(0, 3, n).astype(np.uint32)
    if fixed:
        gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1)
    try:
        _check(Case(x, w, 2.5, 10.0, 4.5, tags=tags, name=f"equal tags fixed={fixed}"), gpu_ctx,
               oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("sizes", [(0, 0, 300, 0), (0, 8193, 0), (0, 30000)])
def test_lone_event_among_empty_ones(gpu_ctx, oracle_mod, sizes):
    """One event with points in the batch: its descriptor goes as a kernel argument."""
    from cluestering_amd.device import Clusterer, PointsDevice
    rng = np.random.default_rng(4)
    sizes = np.array(sizes, np.uint32)
    c, w = (np.ascontiguousarray(a) for a in synthetic._event2d(rng, int(sizes.sum())))
    kern = K.GaussianKernel(1.0, 1.0)
    _, ref = _check(Case(c, w, 1.5, 5.0, 2.0, kernel=kern, sizes=sizes, name=f"lone {sizes}"),
                    gpu_ctx, oracle_mod)
    pts = PointsDevice.from_host(gpu_ctx, c, w)
    eoc = gpu_ctx.empty(w.size, np.int32)
    k = Clusterer(gpu_ctx, 1.5, 5.0, 2.0).make_clusters_batched(pts, sizes, None, kern,
                                                              event_of_cluster=eoc)
    assert k == ref.n_seeds
    np.testing.assert_array_equal(eoc.to_host()[:k], ref.event_of_cluster)


@pytest.mark.parametrize("points_per_tile", [20000, 79, 70, 20, 19, 1])
def test_tile_key_widths(gpu_ctx, oracle_mod, points_per_tile):
    """1, 256, 289, 1,024, 1,089 and 20,164 tiles: keys of 0 to 15 bits, in one or two
    radix passes of one of the two widths."""
    rng = np.random.default_rng(points_per_tile)
    c = rng.uniform(0, 100, (2, 20000)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, 20000).astype(np.float32)
    _check(Case(c, w, 1.0, 3.0, 1.5, points_per_tile=points_per_tile,
                name=f"points_per_tile={points_per_tile}"), gpu_ctx, oracle_mod)


def test_lone_event_above_a_million_points(gpu_ctx, oracle_mod):
    """More than 512 chunks (each result of the extremes stage covers two) and more
    than 32,768 words of seed bits (counted by a scan, not by one kernel)."""
    rng = np.random.default_rng(21)
    n = (1 << 20) + 1
    c = rng.uniform(0, 1000, (2, n)).astype(np.float32)
    c[:, -1] = 1003.0                     # the last point, alone in its chunk, is the maximum
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    _check(Case(c, w, 1.0, 3.0, 1.5, name="2^20+1"), gpu_ctx, oracle_mod)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("ndim", [1, 3, 5])
@pytest.mark.parametrize("n,points_per_tile", [(1, 0), (1023, 0), (1025, 0), (8191, 8), (8192, 0),
                                               (8192, 7)])
def test_small_lone_events(gpu_ctx, oracle_mod, n, points_per_tile, ndim, dtype):
    """A lone event's own tile and seed kernels (up to 8,192 points and 1,024 tiles):
    whole and partial rounds, with every optional column and without."""
    rng = np.random.default_rng(n + ndim)
    c = rng.uniform(0, 20, (ndim, n)).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    u = rng.uniform(0.5, 1.5, n).astype(dtype)
    sigma = rng.uniform(0.0, 0.3, size=(ndim, n)).astype(dtype)
    tags = rng.permutation(n).astype(np.uint32)
    for more in ({}, {"u": u, "sigma": sigma, "tags": tags}):
        case = Case(c, w, 1.0, 2.0, 1.5, points_per_tile=points_per_tile, dtype=dtype,
                    name=f"lone n={n} ndim={ndim} {np.dtype(dtype)} {sorted(more)}", **more)
        print(f"[case] {case.name}", flush=True)
        assert_same(case.run_gpu(gpu_ctx), case.run_oracle(oracle_mod), case.name)


@pytest.mark.parametrize("ndim,n", [(5, 100000), (3, 200000)])
def test_many_nearly_empty_tiles(gpu_ctx, oracle_mod, ndim, n):
    """Tiles of less than a point on average, whose boxes would exceed their 4 MiB: the
    stages do without (161,051 tiles for teams of waves, 205,379 for one wave per item)."""
    rng = np.random.default_rng(ndim)
    c = rng.uniform(0, 10, (ndim, n)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    _check(Case(c, w, 0.2, 1.5, 0.3, points_per_tile=1, name=f"ndim={ndim} n={n}"), gpu_ctx,
           oracle_mod)


@pytest.mark.parametrize("n", [1, 21845, 21846, 65536, 65537])
def test_host_arrays_of_staged_sizes(gpu_ctx, n):
    """Host calls on both sides of the largest copy that goes through pinned memory
    (262,140 and 262,152 bytes of points; 256 KiB and more per result, which together
    exceed the block), one after the other, against the device-resident call."""
    import ctypes as C

    from cluestering_amd import _capi
    from cluestering_amd.device import Clusterer, PointsDevice
    rng = np.random.default_rng(n)
    lib = _capi.load()
    kern = K.GaussianKernel(1.0, 1.0)
    for _ in range(2):
        c, w = (np.ascontiguousarray(a) for a in synthetic._event2d(rng, n))
        data = np.ascontiguousarray(np.vstack([c, w[None, :]]), dtype=np.float32)
        p = _capi.make_params(2, 1.5, 5.0, 2.0, None, kern.kind, kern.params)
        out = [np.empty(n, t) for t in (np.int32, np.int32, np.float32, np.int32)]
        at = [a.ctypes.data_as(C.c_void_p) for a in out]
        _capi.check(lib.clue_make_clusters_host(gpu_ctx.handle, C.byref(p), n,
                                                data.ctypes.data_as(C.c_void_p), at[0], None, 0,
                                                at[1], at[2], at[3]))
        pts = PointsDevice.from_host(gpu_ctx, c, w)
        Clusterer(gpu_ctx, 1.5, 5.0, 2.0).make_clusters(pts, kernel=kern)
        np.testing.assert_array_equal(out[0], pts.cluster_index.to_host())
        np.testing.assert_array_equal(out[1], pts.is_seed.to_host())
        np.testing.assert_array_equal(out[2].view(np.uint32), pts.rho.to_host().view(np.uint32))
        np.testing.assert_array_equal(out[3], pts.nearest_higher.to_host())


@pytest.mark.parametrize("n", [1, 3, 5000, 32700, 33000])
def test_work_item_scans(gpu_ctx, oracle_mod, n):
    """1 to 33,124 tiles in launches of one wave per item: the items per tile are scanned
    by one workgroup up to 32,768 tiles, by the general scan above."""
    rng = np.random.default_rng(n)
    c = rng.uniform(0, 50, (2, n)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    gpu_ctx.set_tuning(group_queries=True, xcd_chunk_log2=4, block_waves=1)
    try:
        _check(Case(c, w, 0.6, 3.0, 0.9, points_per_tile=1, name=f"items n={n}"), gpu_ctx,
               oracle_mod)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("small,count", [(5, 2), (5, 3), (5, 3000), (300, 40), (2049, 9)])
def test_large_event_among_small_ones(gpu_ctx, oracle_mod, small, count, dtype):
    """An event of 1,521 tiles sends its batch down the radix path, whose sort takes the
    events' chunks as blocks (2 and 9 small events) or, where most would be nearly empty,
    2,048 points whatever their events."""
    from cluestering_amd.device import Clusterer, PointsDevice
    rng = np.random.default_rng(small + count)
    sizes = np.full(count + 1, small, np.uint32)
    sizes[count // 2] = 3000
    n = int(sizes.sum())
    c = rng.uniform(0, 30, (2, n)).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    kern = K.GaussianKernel(1.0, 1.0)
    gpu, ref = _check(Case(c, w, 1.0, 1.5, 1.5, kernel=kern, sizes=sizes, points_per_tile=2, dtype=dtype,
                           name=f"{count} x {small}"), gpu_ctx, oracle_mod)
    assert gpu["n_clusters"] == ref.n_seeds
    pts = PointsDevice.from_host(gpu_ctx, c, w, dtype=dtype)
    algo = Clusterer(gpu_ctx, 1.0, 1.5, 1.5)
    algo.points_per_tile = 2
    eoc = gpu_ctx.empty(n, np.int32)
    k = algo.make_clusters_batched(pts, sizes, None, kern, event_of_cluster=eoc)
    event = np.repeat(np.arange(count + 1), sizes)
    np.testing.assert_array_equal(eoc.to_host()[:k], event[np.nonzero(ref.is_seed)[0]])


@pytest.mark.parametrize("sizes", [[3000], [300, 0, 2000], [131072], [16] * 3000])
def test_fixing_the_chosen_tuning_keeps_it(gpu_ctx, oracle_mod, sizes):
    """get_tuning reports what a run would use, teams of waves among it, and fixing that
    changes nothing."""
    rng = np.random.default_rng(3)
    n = int(sum(sizes))
    case = Case(rng.uniform(0, 40, (2, n)), rng.uniform(0.5, 1.5, n), 1.0, 3.0, 1.5, sizes=sizes,
                name=f"tuning of {len(sizes)} events")
    params = case.clusterer(gpu_ctx).params(2)
    chosen = gpu_ctx.get_tuning(params, sizes)
    assert chosen["team"] == (n <= 49152 and len(sizes) < 3000)
    gpu_ctx.set_tuning(**chosen)
    try:
        assert gpu_ctx.get_tuning(params, sizes) == chosen
        _check(case, gpu_ctx, oracle_mod)
    finally:
        gpu_ctx.set_tuning()
    assert gpu_ctx.get_tuning(params, sizes) == chosen
