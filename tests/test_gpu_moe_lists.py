"""The lists of routes grouped by expert, where they change form: more routes than the grouping keeps in registers (8192), lists of
places in LDS (up to 128 KiB of them) or written straight to memory."""
import pytest

import test_gpu_moe_grouped as grouped

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("routes,E,skew", [(8192, 5, False), (8193, 5, True), (16127, 8, False), (16129, 8, True), (16700, 3, False), (20001, 40, True)])
def test_lists(ctx, orc, routes, E, skew):
    grouped.test_grouped_gather(ctx, orc, 4, 64, routes, E, 192, 20, skew)
