"""The free-boundary V-cycle's small-level kernels (one thread per 2x2 block,
bd_mg.hip) at level sizes on both sides of their tiles of 16 and with odd and
even sides: the preconditioner differs from the one of two sweeps a smoothing
(a launch per colour) only in speed of convergence, so the two projections
agree to the solve's threshold, 1e-20 mean square."""
import numpy as np
import pytest

from stz_amd import bd_bench

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("N", [63, 64, 95, 126, 130, 161])
def test_projection_over_level_sizes(N, form):
    print("case bd levels", N, form, flush=True)
    vel, its = [], []
    for nu in (1, 2):
        g = bd_bench.setup(N)
        g.set_precision(form)
        g.set_solver(nu, nu)
        g.projection_step(0.5)
        info = g.last_solve()
        assert info["status"] == 0 and info["residual"] <= info["tolerance"], info
        vel.append(g.get_vel())
        its.append(info["iterations"])
        g.close()
    err = float(np.linalg.norm(vel[0] - vel[1]) / np.linalg.norm(vel[1]))
    print(N, form, "iterations", its, "difference %.1e" % err)
    assert its[0] <= 4 * its[1] + 20
    assert err < 1e-7  # as test_projection_mixed_preconditioner


# levels on both sides of 65536 rows (253, 261 and 262 nodes a side below the
# top), where the Galerkin products' tiles change, with odd and even sides: a
# wrong coarse row costs iterations, and those of a V-cycle do not depend on
# the grid but for the surface's place in its cells
@pytest.mark.parametrize("N", [520, 522])
def test_coarse_products_on_large_levels(N):
    its = []
    for k in (504, N):
        print("case bd products", k, flush=True)
        g = bd_bench.setup(k)
        g.projection_step(0.5)
        info = g.last_solve()
        assert info["status"] == 0 and info["residual"] <= info["tolerance"], info
        its.append(info["iterations"])
        g.close()
    print(N, "iterations", its)
    assert its[1] <= 1.5 * its[0] + 3
