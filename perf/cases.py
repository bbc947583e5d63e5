"""The work that users of this package have it do, as cases to be timed.

Every case goes through a public entry point: Clusterer.make_clusters (one event
resident on the device), Clusterer.make_clusters_batched, a Plan (a batch captured
once and launched again and again), CLUE_GPU_HIP.mainRun (host arrays in, labels
out, the call behind CLUEstering.clusterer) and get_clusters (the cluster -> points
map). The point clouds follow cluestering_amd.synthetic, drawn on the GPU:

  blobs     5-50 Gaussian blobs (sigma 1) in [0, 100]^ndim, 20 % uniform noise
  wide      2-D, blobs of sigma 0.5-2 and 15 % noise at a constant density, so the
            box grows with the points (200 blobs in [0, 1000]^2 at 2^20 points)
  detector  3-D showers in (x, y, periodic phi), rescaled to one radius, 20 % noise,
            lognormal weights (2000 showers at 2^20 points)

Events of a batch have sizes spread evenly over the logarithm of their range, in a
fixed shuffled order, so a case's work does not depend on its seed.
"""
import math
import random

import numpy as np
import torch

from cluestering_amd import CLUE_Convolutional_Kernels as K
from cluestering_amd import CLUE_GPU_HIP
from cluestering_amd.device import Clusterer, Context, Plan, PointsDevice, get_clusters

PERIOD = float(np.float32(20.0 * np.pi))  # of the rescaled phi
FULL = ("cluster_index", "is_seed", "rho", "nearest_higher", "delta")


def listed():
    def case(name, call, layout, ndim, n, kernel, **more):
        return dict({"name": name, "call": call, "layout": layout, "ndim": ndim, "n": n, "kernel": kernel,
                     "width": 1.0, "amplitude": 1.0, "metric": "euclidean", "dtype": "float32", "events": 1,
                     "smallest": n, "sigma": False, "uncertainty": False, "tags": False}, **more)
    return [
        # The smallest events of a stream, one call each: latency and launches.
        case("event2d_300", "event", "blobs", 2, 300, "flat"),
        # An ordinary event, at the size below which one workgroup builds its tiles.
        case("event2d_5003", "event", "blobs", 2, 5003, "gauss"),
        # The single-event workload of the benchmark.
        case("event2d_16384", "event", "blobs", 2, 16384, "flat"),
        # One large image-like cloud.
        case("wide2d_1m", "event", "wide", 2, 1 << 20, "flat"),
        # One large detector readout with a wrapped coordinate.
        case("detector3d_1m", "event", "detector", 3, 1 << 20, "exp", metric="periodic"),
        # The same in double precision, with density uncertainties, as C++ users of Clusterer<3, double> run it.
        case("detector3d_40001_f64", "event", "detector", 3, 40001, "exp", metric="periodic", dtype="float64",
             uncertainty=True),
        # Many dimensions (embeddings), a weighted metric and a general gaussian.
        case("blobs6d_20011", "event", "blobs", 6, 20011, "gauss", width=1.3, metric="weighted_euclidean"),
        # Points with resolutions: Mahalanobis distances, per-point sigmas and user tags.
        case("sigmas3d_30000", "event", "blobs", 3, 30000, "flat", metric="mahalanobis", sigma=True, tags=True),
        # The headline workload: a launch over thousands of events, replayed.
        case("plan2d_4096", "plan", "blobs", 2, 65536, "gauss", events=4096, smallest=256),
        # What a server folds into one launch: events of very different sizes, not captured.
        case("batch3d_48", "batch", "detector", 3, 262144, "exp", metric="periodic", events=48, smallest=256),
        # Host data in, labels out: the Python drop-in.
        case("host2d_100003", "host", "blobs", 2, 100003, "flat"),
        # The members of every cluster, after a clustering.
        case("map3d_1m", "map", "detector", 3, 1 << 20, "exp", metric="periodic"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["event"] * 6 + ["plan", "batch", "host", "map"])
    layout = rng.choice(["blobs", "wide", "detector"])
    c = {"call": call, "layout": layout, "ndim": {"wide": 2, "detector": 3}.get(layout, 2), "n": 0,
         "kernel": rng.choice(["flat", "exp", "gauss"]), "width": 1.0, "amplitude": 1.0, "metric": "euclidean",
         "dtype": "float32", "events": 1, "smallest": 0, "sigma": False, "uncertainty": False, "tags": False}
    if c["kernel"] != "flat":
        c["width"] = rng.choice([0.5, 1.0, 1.0, 1.3])
        c["amplitude"] = rng.choice([1.0, 1.0, 2.0])
    if layout == "detector":
        c["metric"] = "periodic"
    if call in ("plan", "batch"):
        c["layout"] = layout = "detector" if layout == "detector" else "blobs"
        c["ndim"] = 3 if layout == "detector" else 2
        c["events"] = _log(rng, 2, 512)
        c["smallest"] = 256
        c["n"] = _log(rng, 1024, 65536 if c["events"] > 64 else 262144)
        return c
    if call in ("host", "map"):
        c["n"] = c["smallest"] = _log(rng, 1000, 1 << 20) if layout != "blobs" else _log(rng, 1000, 131072)
        return c
    top = {"blobs": 65536, "wide": 1 << 20, "detector": 1 << 20}[layout]
    if layout == "blobs":
        c["ndim"] = rng.choice([1, 2, 2, 2, 3, 4, 5, 6, 8])
        c["metric"] = rng.choice(["euclidean"] * 3 + ["weighted_euclidean", "manhattan", "chebyshev", "mahalanobis"])
        top = 65536 if c["ndim"] <= 3 else 30000
        c["sigma"] = c["metric"] == "mahalanobis"
        c["uncertainty"] = rng.random() < 0.2
        c["tags"] = rng.random() < 0.2
    if rng.random() < 0.2:
        c["dtype"], top = "float64", min(top, 65536)
    c["n"] = c["smallest"] = _log(rng, 256, top)
    return c


# ---- parameters ------------------------------------------------------------------

def _radii(c):
    """(dc, rhoc, dm) of the layout."""
    if c["layout"] == "detector":
        return 1.0, 4.0, 1.5
    if c["layout"] == "wide":
        return 1.5, 8.0, 2.5
    if c["ndim"] == 2 or c["metric"] == "mahalanobis":
        return 1.5, 5.0, 2.0
    return 0.75 + 0.4 * c["ndim"], 3.0, 1.25 + 0.4 * c["ndim"]


def _weights(c):
    return [1.0 + 0.25 * (d % 3) for d in range(c["ndim"])]


def _metric(c):
    return {"euclidean": lambda: K.EuclideanMetric(), "weighted_euclidean": lambda: K.EuclideanMetric(_weights(c)),
            "manhattan": lambda: K.ManhattanMetric(), "chebyshev": lambda: K.ChebyshevMetric(),
            "mahalanobis": lambda: K.MetricDescriptor("mahalanobis"),
            "periodic": lambda: K.PeriodicEuclideanMetric([0.0, 0.0, PERIOD])}[c["metric"]]()


def _kernel(c):
    if c["kernel"] == "flat":
        return K.FlatKernel(0.5)
    if c["kernel"] == "exp":
        return K.ExponentialKernel(0.5 * c["width"], c["amplitude"])
    return K.GaussianKernel(c["width"], c["amplitude"])


def _wrapped(c):
    return (0, 0, 1) if c["metric"] == "periodic" else ()


def _sizes(c):
    e = c["events"]
    if e == 1:
        return np.array([c["n"]], np.uint32)
    s = [int(c["smallest"] * (c["n"] / c["smallest"]) ** ((k + 0.5) / e)) for k in range(e)]
    random.Random(e).shuffle(s)
    return np.array(s, np.uint32)


# ---- inputs ----------------------------------------------------------------------

def _inputs(c, seed):
    """(coords [ndim][n], weight [n], more) on the GPU in the case's type."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)
    f64 = dict(device="cuda", dtype=torch.float64)

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(shape, generator=g, **f64)

    def normal(*shape):
        return torch.randn(shape, generator=g, **f64)

    sizes = torch.from_numpy(_sizes(c).astype(np.int64)).cuda()
    events, total, D = len(sizes), int(sizes.sum()), c["ndim"]
    event = torch.repeat_interleave(torch.arange(events, device="cuda"), sizes)
    place = torch.arange(total, device="cuda") - (torch.cumsum(sizes, 0) - sizes)[event]
    if c["layout"] == "blobs":
        share, half = 0.8, None
        groups = torch.randint(5, 51, (events,), generator=g, device="cuda")
    else:
        full, share = (200, 0.85) if c["layout"] == "wide" else (2000, 0.8)
        groups = torch.clamp(torch.round(full * sizes.double() / (1 << 20)), min=1).long()
        half = (1000.0 if c["layout"] == "wide" else 150.0) * torch.sqrt(groups.double() / full)
    per = torch.clamp((share * sizes.double() / groups).long(), min=1)
    group = place // per[event]
    noise = group >= groups[event]
    first = torch.cumsum(groups, 0) - groups
    at = first[event] + torch.minimum(group, groups[event] - 1)
    of = torch.repeat_interleave(torch.arange(events, device="cuda"), groups)  # event of each group
    columns = []
    for d in range(D):
        if c["layout"] == "blobs":
            lo, hi, spread = 0.0, 100.0, 1.0
        elif c["layout"] == "wide":
            if d == 0:
                spreads = uniform(0.5, 2.0, len(of))
            lo, hi, spread = 0.0, half, spreads[at]
        else:
            lo, hi, spread = (-half, half, 1.5) if d < 2 else (-math.pi, math.pi, 0.05)
        def over(v, index):
            return v[index] if isinstance(v, torch.Tensor) else v
        centre = uniform(over(lo, of), over(hi, of), len(of))
        x = torch.where(noise, uniform(over(lo, event), over(hi, event), total), centre[at] + spread * normal(total))
        if c["layout"] == "detector":
            x = x / 2.0 if d < 2 else (torch.remainder(x + math.pi, 2 * math.pi) - math.pi) / 0.1
        columns.append(x)
    dtype = getattr(torch, c["dtype"])
    coords = torch.stack(columns).to(dtype)
    weight = (torch.exp(normal(total)) if c["layout"] == "detector" else uniform(0.5, 1.5, total)).to(dtype)
    more = {}
    if c["sigma"]:
        more["sigma"] = uniform(0.5, 1.5, D, total).to(dtype)
    if c["uncertainty"]:
        more["u"] = uniform(0.5, 1.5, total).to(dtype)
    if c["tags"]:
        more["tags"] = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    return coords, weight, more


def _labels(c, seed):
    """Cluster ids as a clustering of the layout gives them (a blob or shower each,
    its noise in no cluster), the points in no order."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)
    n = c["n"]
    groups = {"blobs": 27, "wide": round(200 * n / (1 << 20)), "detector": round(2000 * n / (1 << 20))}[c["layout"]]
    groups = max(1, groups)
    per = max(1, int((0.85 if c["layout"] == "wide" else 0.8) * n / groups))
    group = torch.arange(n, device="cuda") // per
    labels = torch.where(group < groups, group, torch.full_like(group, -1))
    return labels[torch.randperm(n, generator=g, device="cuda")].to(torch.int32)


class _View:
    """A device array as torch takes it, without a copy."""

    def __init__(self, array, shape=None):
        self.array = array  # kept alive with the tensor
        self.__cuda_array_interface__ = {"shape": shape or array.shape, "typestr": array.dtype.str.replace("u4", "i4"),
                                         "data": (array.ptr, False), "version": 2}


def _tensor(array, shape=None):
    return torch.as_tensor(_View(array, shape), device="cuda")


_contexts = []


def _context():
    if not _contexts:
        _contexts.append(Context(0))
    return _contexts[0]


class State:
    pass


def prepare(case, seed):
    c, s = case, State()
    s.call, s.metric, s.kernel = c["call"], _metric(c), _kernel(c)
    if c["call"] == "map":
        s.points = PointsDevice(_context(), c["n"], c["ndim"])
        _tensor(s.points.cluster_index).copy_(_labels(c, seed))
        s.points.clustered = True
        torch.cuda.synchronize()
        return s
    coords, weight, more = _inputs(c, seed)
    dc, rhoc, dm = _radii(c)
    if c["call"] == "host":
        s.ndim, s.n = c["ndim"], int(coords.shape[1])
        s.data = torch.cat([coords, weight[None]]).cpu().numpy()
        s.labels = np.empty(s.n, np.int32)
        s.parameters = (dc, rhoc, dm, dc, list(_wrapped(c)) or [0] * s.ndim)
        return s
    ctx = _context()
    s.points = p = PointsDevice(ctx, int(coords.shape[1]), c["ndim"], np.dtype(c["dtype"]))
    _tensor(p.coords).copy_(coords)
    _tensor(p.weight).copy_(weight)
    if "sigma" in more:
        p.sigma = ctx.empty((c["ndim"], p.n), p.dtype)
        _tensor(p.sigma).copy_(more["sigma"])
    if "u" in more:
        p.density_uncertainty = ctx.empty(p.n, p.dtype)
        _tensor(p.density_uncertainty).copy_(more["u"])
    if "tags" in more:
        p.tags = ctx.empty(p.n, np.uint32)
        _tensor(p.tags).copy_(more["tags"])
    s.outputs = {k: _tensor(getattr(p, k)) for k in FULL}
    torch.cuda.synchronize()
    s.algorithm = Clusterer(ctx, dc, rhoc, dm)
    s.algorithm.set_wrapped_coordinates(*_wrapped(c))
    s.sizes = _sizes(c)
    if c["call"] == "plan":
        s.plan = Plan(s.algorithm, p, s.sizes, s.metric, s.kernel)
    return s


def run(s):
    if s.call == "event":
        s.algorithm.make_clusters(s.points, s.metric, s.kernel)
        return s.outputs
    if s.call == "plan":
        s.plan.launch()
        return s.outputs
    if s.call == "batch":
        clusters = s.algorithm.make_clusters_batched(s.points, s.sizes, s.metric, s.kernel)
        return dict(s.outputs, clusters=clusters)
    if s.call == "host":
        dc, rhoc, dm, seed_dc, wrapped = s.parameters
        CLUE_GPU_HIP.mainRun(dc, rhoc, dm, seed_dc, wrapped, s.data, s.labels, s.kernel, s.ndim, None, s.n, 0, s.metric)
        return {"labels": s.labels}
    m = get_clusters(s.points)
    return {"offsets": _tensor(m.offsets, (m.n_bins + 1,)), "indexes": _tensor(m.indexes, (m.n_members,))}


# ---- what a pass cannot do without -----------------------------------------------

def _ball(c):
    """(share of a blob's pairs within dc, volume within dc), for the Euclidean ball."""
    dc, D = _radii(c)[0], c["ndim"]
    # P(chi-squared with D degrees <= x) by its series.
    x = dc * dc / 2.0 / 2.0  # a pair of sigma-1 points differs by sigma sqrt(2)
    term = total = math.exp(-x + (D / 2.0) * math.log(x) - math.lgamma(D / 2.0 + 1.0))
    for k in range(1, 200):
        term *= x / (D / 2.0 + k)
        total += term
    return min(1.0, total), math.pi ** (D / 2.0) / math.gamma(D / 2.0 + 1.0) * dc ** D


def work(case):
    """Bytes: every input and output once. Operations: the metric and the kernel of
    the expected pairs within the density radius (blob mates and noise)."""
    c, sizes = case, _sizes(case).astype(np.float64)
    n, D, b = float(sizes.sum()), c["ndim"], 8 if c["dtype"] == "float64" else 4
    if c["call"] == "map":
        return {"bytes": 8.0 * n, "flops": n}
    inputs = n * b * (D + 1 + (D if c["sigma"] else 0) + bool(c["uncertainty"])) + (4 * n if c["tags"] else 0)
    outputs = 4 * n if c["call"] == "host" else n * (12 + 2 * b)
    share, volume = _ball(c)
    if c["layout"] == "detector":  # spread 0.75, 0.75, 0.5 after rescaling; constant density
        share, groups, box = min(1.0, 2.5 * share), np.maximum(1, np.round(2000 * sizes / (1 << 20))), None
        around = n * 0.2 * volume * (1 << 20) / (150.0 * 150.0 * PERIOD)
    elif c["layout"] == "wide":
        groups, around = np.maximum(1, np.round(200 * sizes / (1 << 20))), n * 0.15 * volume * (1 << 20) / 1e6
    else:
        groups, around = np.full(len(sizes), 27.5), float((sizes * sizes).sum()) * 0.2 * min(1.0, volume / 100.0 ** D)
    pairs = float((0.64 * sizes * sizes / groups).sum()) * share + around
    return {"bytes": inputs + outputs, "flops": pairs * (3 * D + (2 if c["kernel"] == "flat" else 20))}


# ---- the densities in 64 bits ------------------------------------------------------

def exact(case, seed):
    """The local densities, straight from their definition: rho_i is the sum over the
    points j of the event within dc of K(d_ij) w_j, with K(i, i) = 1. The other
    outputs are whole numbers and choices among them. Mahalanobis distances are left
    out: there the search box, and so the candidates, follow one point's sigma."""
    c = case
    if c["call"] in ("host", "map") or c["metric"] == "mahalanobis":
        return None
    coords, weight, _ = _inputs(c, seed)
    x, w, D = coords.double(), weight.double(), c["ndim"]
    kind = np.float64 if c["dtype"] == "float64" else np.float32
    dc, width, amplitude = (float(kind(v)) for v in (_radii(c)[0], c["width"], c["amplitude"]))
    if c["kernel"] == "exp":
        width = float(kind(0.5 * c["width"]))
    sizes = torch.from_numpy(_sizes(c).astype(np.int64)).cuda()
    event = torch.repeat_interleave(torch.arange(len(sizes), device="cuda"), sizes)
    gap = 1e6  # between events on the sorting axis, wider than any cloud
    key, order = torch.sort(x[0] + gap * event)
    x, w, event = x[:, order], w[order], event[order]
    reach = dc * 1.001  # in the first dimension (no weight is below 1)
    n, chunk = int(key.numel()), 2048
    starts = torch.arange(0, n, chunk, device="cuda")
    ends = torch.clamp(starts + chunk, max=n)
    lo = torch.searchsorted(key, key[starts] - reach).cpu().tolist()
    hi = torch.searchsorted(key, key[ends - 1] + reach, right=True).cpu().tolist()
    rho = torch.empty(n, device="cuda", dtype=torch.float64)
    weights = _weights(c) if c["metric"] == "weighted_euclidean" else [1.0] * D
    for k, (a, b) in enumerate(zip(lo, hi)):
        q0, q1 = k * chunk, min(n, (k + 1) * chunk)
        if b - a > 65536:  # a dense first dimension: fewer queries at a time
            parts = [(p, min(q1, p + 256)) for p in range(q0, q1, 256)]
        else:
            parts = [(q0, q1)]
        for p0, p1 in parts:
            total = None
            for d in range(D):
                t = (x[d, p0:p1, None] - x[d, None, a:b]).abs_()
                if c["metric"] == "periodic" and d == 2:
                    t = torch.minimum(t, PERIOD - t)
                if c["metric"] in ("manhattan", "chebyshev"):
                    pass
                else:
                    t = t.square_().mul_(weights[d]) if weights[d] != 1.0 else t.square_()
                if total is None:
                    total = t
                elif c["metric"] == "chebyshev":
                    total = torch.maximum(total, t)
                else:
                    total = total.add_(t)
            if c["metric"] in ("manhattan", "chebyshev"):
                near = total <= dc
            else:
                near = total <= dc * dc
            if len(sizes) > 1:
                near &= event[p0:p1, None] == event[None, a:b]
            if c["kernel"] == "flat":
                value = torch.full_like(total, 0.5)
            elif c["kernel"] == "exp":
                value = (total if c["metric"] in ("manhattan", "chebyshev") else total.sqrt_()).mul_(-width).exp_().mul_(amplitude)
            else:
                square = total.square_() if c["metric"] in ("manhattan", "chebyshev") else total
                value = square.mul_(-1.0 / (2.0 * width * width)).exp_().mul_(amplitude)
            value.mul_(near)
            own = torch.arange(p0, p1, device="cuda")
            value[own - p0, own - a] = 1.0
            rho[p0:p1] = value @ w[a:b]
    out = torch.empty_like(rho)
    out[order] = rho
    answer = {k: None for k in FULL}
    answer["rho"] = out
    if c["call"] == "batch":
        answer["clusters"] = None
    return answer
