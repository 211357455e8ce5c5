"""RHF on both sides of the size above which the one-launch SCF step gives way
to the general loop (84 functions), held to the equations of its result as
test_gpu_small_scf.py holds the smaller sizes, with its tolerances."""
import pytest

import test_gpu_small_scf as small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [82, 83, 84, 85, 86])
def test_solution_at_the_limit(ctx, n):
    print(f"[small] n = {n}", flush=True)
    small.test_solution_at_tile_edges(ctx, n)
