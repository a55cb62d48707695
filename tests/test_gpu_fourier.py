"""The direct solve of the projection (Fourier modes along x, block recurrences
along y; stz_mg_config.direct_nodes > 0) and what decides between it and
V-cycles.

* Against the dense FP64 system (tests/dense.py) on small grids of every kind
  of width the row transform treats differently (2, 3, 4, 5 and other primes,
  odd and even) and of the smallest heights.
* Against the V-cycle solve (direct_nodes = 0) of the same system to a tight
  threshold at the edges of the mode kernel's row ranges and the row
  transform's lengths; the largest of both by the residual alone.
* A correction after a failed test, the failure of a solve whose threshold
  cannot be met, and NaN in the source.
* Tiled and per-colour V-cycle kernels on a grid that solves directly unless
  asked for V-cycles.

Tolerances: two solutions with residuals r1 and r2 differ by at most (|r1| +
|r2|) / lambda, lambda = (mu + viscosity/dt) (pi / height)^2 the operator's
smallest eigenvalue (the smoothest mode along y).  The residuals are at most
the threshold's, or, at the rounding floor, a few eps times the diagonal
times the solution."""
import math

import numpy as np
import pytest

from dense import top_dense, top_product
from stz_amd import ShearSim, StzError
from stz_amd.problems import simple_shear

pytestmark = pytest.mark.gpu


VISCDT = 0.1


def smallest_eigenvalue(p, viscdt):
    return (p["mu"] + viscdt) * (math.pi / (p["by"] - p["ay"])) ** 2


def diagonal(p, viscdt):
    Kmu = p["K"] + 4 * p["mu"] / 3 + viscdt
    return 2 * Kmu * ((p["m"] / (p["bx"] - p["ax"])) ** 2 + (p["n"] / (p["by"] - p["ay"])) ** 2)


def differ(a, b):
    """2-norm of the difference (a number, so that a failure prints one)"""
    return float(np.linalg.norm(a - b))


def solve(p, form, b, tol, **kw):
    g = ShearSim(p, form)
    g.set_mg_config(tol_mult=tol, nu1=2, nu2=2, **kw)
    g.mg_setup(VISCDT)
    g.mg_set_src(b)
    g.set_vel(np.zeros_like(b))
    info = g.mg_solve()
    z = g.get_vel()
    g.close()
    return z, info


@pytest.mark.parametrize("m,n", [(4, 9), (5, 9), (8, 5), (9, 7), (12, 20), (14, 8), (22, 6), (25, 24), (30, 17),
                                 (15, 30), (26, 12)])
def test_direct_solve_equals_dense_solve(m, n):
    print("case fourier dense", m, n, flush=True)
    p = simple_shear(m, n)
    b = np.random.default_rng(m + 100 * n).normal(size=(n + 1, m, 2))
    z, info = solve(p, "fp64", b, 1e-10)
    assert info["status"] == 0 and info["total_cycles"] == 1 and info["cycles"] == 0, info
    zd = np.linalg.solve(top_dense(p, VISCDT), b.ravel()).reshape(z.shape)
    floor = 16 * 2.2e-16 * diagonal(p, VISCDT) / smallest_eigenvalue(p, VISCDT)
    assert floor < 1e-8
    assert differ(z, zd) <= floor * np.linalg.norm(zd)


# row lengths with prime stages (alone, two of a kind, two kinds, before
# others) and with a stage of eight
@pytest.mark.parametrize("m,n", [(7, 9), (49, 7), (77, 6), (38, 14), (57, 8), (40, 10), (56, 9)])
def test_row_transform_of_any_length(m, n):
    test_direct_solve_equals_dense_solve(m, n)


# rows n - 1 at both sides of 128, 256, 512 (rows per thread, waves), widths
# with each fixed length and with the general transform
@pytest.mark.parametrize("m,n", [(128, 129), (256, 130), (128, 257), (144, 258), (512, 100), (240, 300), (96, 513),
                                 (160, 514), (1024, 64), (64, 1026)])
def test_direct_solve_equals_v_cycles(m, n):
    print("case fourier vs V-cycles", m, n, flush=True)
    p = simple_shear(m, n)
    # square cells, so that V-cycles converge quickly
    p["by"], p["ay"] = n / m, -n / m
    b = np.random.default_rng(m + n).normal(size=(n + 1, m, 2))
    z, info = solve(p, "fp64", b, 1e-12)
    assert info["status"] == 0 and info["total_cycles"] == 1, info
    zv, iv = solve(p, "fp64", b, 1e-12, direct_nodes=0)
    assert iv["status"] == 0 and iv["cycles"] > 1, iv
    r = math.sqrt(m * (n + 1)) * (math.sqrt(info["residual"]) + math.sqrt(iv["residual"]))
    err, bound = differ(z, zv), r / smallest_eigenvalue(p, VISCDT)
    norm = float(np.linalg.norm(zv))
    print(m, n, "difference %.2e, bound %.2e, V-cycles %d" % (err / norm, bound / norm, iv["cycles"]))
    assert bound < 1e-7 * norm and err <= bound


# the largest of everything: rows at both sides of 1024 and 2048 and the most
# there are, each compile-time length on its own and in workgroups of four
# rows (from 1020 interior rows on), the widest general length
@pytest.mark.parametrize("m,n", [(8, 1025), (8, 1026), (8, 2049), (8, 2050), (8, 4097), (2048, 8), (4096, 8),
                                 (2160, 8), (512, 1021), (1024, 1022), (2048, 1023), (4096, 1021)])
def test_residual_of_the_largest_variants(m, n):
    """the host's residual of the solution is at the rounding floor: 9 products
    of the operator a row, and as much again for the solve"""
    print("case fourier largest", m, n, flush=True)
    p = simple_shear(m, n)
    p["by"], p["ay"] = n / m, -n / m
    b = np.random.default_rng(m + n).normal(size=(n + 1, m, 2))
    z, info = solve(p, "fp64", b, 1.0)
    assert info["status"] == 0 and info["total_cycles"] == 1, info
    r = float(np.linalg.norm(b - top_product(p, VISCDT, z)))
    floor = 2 * 9 * 2.2e-16 * diagonal(p, VISCDT) * float(np.linalg.norm(z))
    print(m, n, "residual %.1e of the source, floor %.1e" % (r / np.linalg.norm(b), floor / np.linalg.norm(b)))
    assert floor < 1e-3 * np.linalg.norm(b) and r <= floor


# one more row, and a width whose rows and prime root table no longer fit
@pytest.mark.parametrize("m,n,direct", [(24, 4097, True), (24, 4098, False), (2112, 64, True), (2240, 64, False)])
def test_limits_of_the_direct_launches(m, n, direct):
    print("case fourier limits", m, n, flush=True)
    g = ShearSim(simple_shear(m, n), "fp64")
    g.mg_setup(VISCDT)
    assert g.solves_directly == direct
    g.close()


# a general length, a compile-time one, the same in the mixed form, and four
# rows a workgroup
@pytest.mark.parametrize("m,n,form", [(240, 96, "fp64"), (256, 96, "fp64"), (256, 96, "mixed"), (512, 1021, "fp64")])
def test_corrections_and_failure(m, n, form):
    """a threshold under the rounding floor: corrections until the predictor's
    limit, then the failure V-cycles end in; the state is left uncorrected"""
    print("case fourier failure", m, n, form, flush=True)
    p = simple_shear(m, n)
    rng = np.random.default_rng(2)
    g = ShearSim(p, form)
    planes = np.zeros((10,) + g.plane_shape)
    planes[2:6] = 0.1 * rng.normal(size=(4,) + g.plane_shape)
    planes[6] = 0.03
    g.set_fields(planes)
    g.set_mg_config(tol_mult=1e-40, predict_init=1, predict_max_iters=4)
    g.time = 2.0
    g.advection_step(0.2)
    before = g.get_field("p")
    with pytest.raises(StzError) as e:
        g.projection_step(0.2)
    info = g.last_solve()
    assert e.value.code == 3 and info["cycles"] == 3 and info["total_cycles"] == 4, info
    assert np.array_equal(g.get_field("p"), before)
    # the same state at a threshold that is met: the iterate, corrected three
    # times, and a fresh solve agree
    z = g.get_vel()
    g.set_mg_config(tol_mult=1.0, predict_max_iters=2048)
    g.projection_step(0.2)
    assert g.last_solve()["cycles"] == 0
    floor = 4 * 2.2e-16 * diagonal(p, 0.1) / smallest_eigenvalue(p, 0.1)
    assert floor < 1e-8
    assert differ(g.get_vel(), z) <= floor * np.linalg.norm(z)
    g.close()


def test_general_lengths_of_different_sizes_in_one_process():
    """the general-length kernels take 72 bytes of LDS a column: 2160 is the
    widest that fits, and a narrower grid that also needs a raised limit,
    set up in between, must leave it in place"""
    def new(m):
        print("case fourier widths", m, flush=True)
        g = ShearSim(simple_shear(m, 8), "fp64")
        g.mg_setup(VISCDT)
        g.mg_set_src(np.random.default_rng(m).normal(size=(9, m, 2)))
        return g

    def solve_again(g):
        g.set_vel(np.zeros((9, g.m, 2)))
        info = g.mg_solve()
        assert info["status"] == 0 and info["total_cycles"] == 1, info
        return g.get_vel()

    wide = new(2160)
    first = solve_again(wide)
    narrow = new(960)
    solve_again(narrow)
    assert np.array_equal(solve_again(wide), first)
    wide.close()
    narrow.close()


def test_which_solver_is_taken():
    """the reported solver is the one that runs: V-cycle solves of a mixed form
    evaluate FP64 residuals (refinements), also where they count no cycle"""
    print("case fourier choice", flush=True)
    for m, n, form, kw, direct in [(128, 128, "mixed", {}, False), (256, 128, "mixed", {}, True),
                                   (256, 128, "mixed", {"direct_nodes": 0}, False),
                                   (128, 128, "fp64", {}, True), (64, 64, "fp64", {}, False),
                                   (128, 128, "fp64", {"predict_decay": 7}, False),
                                   (128, 128, "fp64", {"predict_decay": 8}, True),
                                   (44, 30, "fp64", {}, True), (44, 30, "fp64", {"predict_decay": 2}, False),
                                   (256, 160, "fp64", {"predict_decay": 2}, True)]:
        g = ShearSim(simple_shear(m, n), form)
        with pytest.raises(StzError):
            g.solves_directly
        g.set_mg_config(predict_init=0, **kw)
        g.mg_setup(VISCDT)
        assert g.solves_directly == direct, (m, n, form, kw)
        g.mg_set_src(np.zeros((n + 1, m, 2)))
        g.set_vel(np.zeros((n + 1, m, 2)))
        info = g.mg_solve()  # zero source and velocity: the first test passes
        assert info["cycles"] == 0 and info["total_cycles"] == 1, info
        if form == "mixed":
            assert (info["refinements"] == 0) == direct, info
        g.close()


def test_nan_source():
    print("case fourier nan", flush=True)
    p = simple_shear(240, 96)
    b = np.zeros((97, 240, 2))
    b[50, 7, 1] = math.nan
    with pytest.raises(StzError) as e:
        solve(p, "mixed", b, 1.0)
    assert e.value.code in (3, 4)


@pytest.mark.parametrize("form", ["fp64", "mixed"])
def test_tiled_v_cycles_match_per_colour_v_cycles(form):
    print("case tiled V-cycles", form, flush=True)
    p = simple_shear(256)
    b = np.random.default_rng(8).normal(size=(257, 256, 2))
    out = [solve(p, form, b, 1e-2, kernels=k, direct_nodes=0) for k in (0, 1)]
    (za, ia), (zb, ib) = out
    assert ia["cycles"] == ib["cycles"] > 1, (ia, ib)
    # the same iterates: rounding of 20 cycles, far below the stopping error
    assert differ(za, zb) <= 1e-12 * np.linalg.norm(zb)
