"""The kernels of large launches (one wave per item) at small sizes, which a fixed tuning
keeps: the parity tests of every dimension, metric, kernel and option in both precisions
again, over candidate blocks and scanning whole tiles in their own order."""
import numpy as np
import pytest

from cluestering_amd import CLUE_Convolutional_Kernels as K

from _support import Case, assert_same
from test_gpu_f64 import (test_f64_batched, test_f64_blobs_flat_and_gaussian,  # noqa: F401
                          test_f64_detector3d_periodic_exp, test_f64_dimensions, test_f64_metrics,
                          test_f64_options_tags_uncertainty_sigma, test_f64_tag_tie_break_known_answer)
from test_gpu_parity import (test_batched_event_size_boundaries, test_batched_gaussian,  # noqa: F401
                             test_batched_with_empty_and_tiny_events, test_dimensions, test_edge_cases,
                             test_kernels_and_metrics, test_mahalanobis_known_answer,
                             test_options_tags_uncertainty_sigma, test_periodic_opposite_angles,
                             test_tag_tie_break_known_answer)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, params=[True, False], ids=["grouped", "ungrouped"])
def one_wave_per_item(gpu_ctx, request):
    gpu_ctx.set_tuning(group_queries=request.param, xcd_chunk_log2=4, block_waves=1)
    yield
    gpu_ctx.set_tuning()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kernel,reach", [(K.ExponentialKernel(1.0, 1.0), 85.0),
                                          (K.ExponentialKernel(1.0, 1.0), 120.0)]
                         + [(K.GaussianKernel(2.0 ** k, 1.0), np.sqrt(85.0 * 2 * 4.0 ** k)) for k in range(-5, 5)])
def test_kernel_values_in_range(gpu_ctx, oracle_mod, kernel, reach, dtype):
    """exp over the range the density stage evaluates without range handling (arguments down
    to -85), and with it (to -120): pairs of points far from each other, the first
    weightless, so that its density is the kernel's value itself, bit for bit. The
    gaussians are those whose 2 sigma^2 is folded into the exp's constants, and one
    beyond them at each end."""
    rng = np.random.default_rng(41)
    n = 1 << 16
    d = np.concatenate([rng.uniform(0, reach, n // 2), reach * 2.0 ** rng.uniform(-30, 0, n // 2)])
    x = np.stack([np.ravel(np.column_stack([np.zeros(n), d])), np.repeat(np.arange(n) * 1024.0, 2)])
    case = Case(x, np.tile([0.0, 1.0], n), reach, 3.0, reach, kernel=kernel, points_per_tile=64, dtype=dtype,
                name=f"{kernel} to {reach:.3g}")
    gpu, ref = case.run_gpu(gpu_ctx), case.run_oracle(oracle_mod)
    assert np.unique(ref.rho).size > n // 2  # the values, not sums that lost them
    assert_same(gpu, ref, case.name)
