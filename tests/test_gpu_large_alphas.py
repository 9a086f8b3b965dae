"""Steps of the largest grids away from alpha = 2 and without the 2/3 rule: the
y passes with roots and with the ka table, on both rectangles."""
import pytest

from helpers import params_for
from test_gpu_small_grids import _steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,alpv,truncate", [(4096, 1.5, 0), (4096, 1.0, 0), (8192, 1.5, 1),
                                             (8192, 1.0, 0), (8192, 1.5, 0)])
def test_forced_steps_of_the_largest_grids(oracle_mod, n, alpv, truncate):
    """Two forced RK4 steps with the fused boundary between them (1e-12 as for
    the smaller grids)."""
    p = params_for(n, alpv=alpv, truncate=truncate, ring=(63.0, 65.0))
    assert _steps(oracle_mod, p, 2) < 1e-12
