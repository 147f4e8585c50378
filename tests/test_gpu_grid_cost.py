"""What sizing a grid by the density rule costs beside building it at that size,
for more cells than are counted in LDS: at most a build at each size, whatever
the photons' spread (all in one cell among them). Times are the least of several
calls in turn. And the rule's edge for maps of few cells that several workgroups
count."""
import time

import pytest
from test_gpu_grid_sizing import test_density_edge as density_edge

pytestmark = pytest.mark.gpu

UNIT = (0.0, 0.0, 0.0, 1.0, 1.0, 1.0)


@pytest.mark.parametrize("spread", ["uniform", "one_cell"])
def test_rule_costs_at_most_two_builds(ctx, spread):
    import torch

    n, desired = 2_000_000, 100  # 20000 cells at the reference size
    ph = torch.rand((9, n), generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
    if spread == "one_cell":
        ph[0:3] = 0.5 + 1e-4 * ph[0:3]
    final = ctx.grid_build(ph, UNIT, desired=desired)
    cell = final.info.cell_size
    final.close()
    best = {}
    for _ in range(5):
        for c in (0.0, cell):
            ctx.sync()
            t0 = time.perf_counter()
            g = ctx.grid_build(ph, UNIT, cell_size=c, desired=desired)
            ctx.sync()
            best[c] = min(best.get(c, 1e9), time.perf_counter() - t0)
            g.close()
    assert best[0.0] < 4 * best[cell], best


@pytest.mark.parametrize("where", ["first", "last", "spread"])
@pytest.mark.parametrize("n,desired", [(100_000, 1000), (1_000_000, 2000), (2_000_000, 130)])
def test_density_edge_of_few_cells(ctx, n, desired, where):
    density_edge(ctx, n, desired, where)
