"""The transforms' limit of 404 functions is refused by name, before any work."""
import numpy as np
import pytest

from myqc_amd import molecules as M
from myqc_amd.hip import MyqcError

pytestmark = pytest.mark.gpu


def test_above_the_limit(ctx):
    Z, x = M.water_cluster(57, seed=1, box=14.0)
    Z, xyz = list(Z) + [2] * 6, np.concatenate([M.to_bohr(Z, x), [[60.0 + 6.0 * k, 0.0, 0.0] for k in range(6)]])
    ctx.set_system(Z, xyz)
    n = ctx.n
    assert n == 405
    C = np.eye(n)
    for call in (lambda: ctx.ao2mo(C, 4, download=False), lambda: ctx.ao2mo_uhf(C, C, 4, 3, download=False),
                 lambda: ctx.ao2mo_cis_uhf(C, C, 4, 3, download=False)):
        with pytest.raises(MyqcError, match="404 functions"):
            call()
