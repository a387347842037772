"""A budget that the caller has set defers rays at every size, also on images
where the default one does not: against the oracle, counts included."""
import pytest

from test_gpu_march_bounds import test_rays_past_the_map as rays_past_the_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("budget", [2, 16])
def test_budget_of_the_caller_on_a_large_image(gpu, budget):
    rays_past_the_map(gpu, 721, 1281, 0.005, budget)
