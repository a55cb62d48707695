"""The free-boundary V-cycle's small-level kernels (one thread per 2x2 block,
bd_mg.hip) at level sizes on both sides of their tiles of 16 and with odd and
even sides: the preconditioner differs from the one of two sweeps a smoothing
(a launch per colour) only in speed of convergence, so the two projections
agree to the solve's threshold, 1e-20 mean square.

The V-cycle itself (Galerkin products, sweeps, transfers, bottom level) is
compared through the first BiCGStab iteration, which applies it twice: with
max_iter = 1 the solve stops there, and its iterate is the host's, formed with
scipy from the assembled operator."""
import numpy as np
import pytest
import scipy.sparse as sp

from dense import P1
from stz_amd import StzError, bd_bench
from stz_amd.bd import BdSim
from stz_amd.problems import bd_params, plate_hole_phi
from test_gpu_c3 import sparse_operator

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


def plate(m, n):
    """the plate of bd_bench on m x n square cells, chi uniform"""
    h = n / m
    box = (-1.0, 1.0, -h, h)
    g = BdSim(bd_params(m, n, box))
    g.set_level_set(plate_hole_phi(m, n, box, 0.9 * h, 0.4 * min(1.0, h)))
    status, _ = g.status()
    g.set_cell("chi", np.where(status < 4, 600.0 / 21000.0, 0.0))
    X, Y = g.node_coords()
    g.set_node("X", X)
    g.set_node("Y", Y)
    g.set_edge_velocity(-1e-4, 1e-4)
    g.post_process(True)
    return g


def of_stencil(blocks, m, n):
    """the sparse matrix of a level of m x n nodes whose rows all have these
    nine 2x2 blocks (entries off the level left out)"""
    A = sp.csr_matrix((2 * m * n, 2 * m * n))
    for k in range(9):
        x = sp.eye(m, k=k % 3 - 1)
        y = sp.eye(n, k=k // 3 - 1)
        A = A + sp.kron(sp.kron(y, x), blocks[k])
    return A.tocsr()


def stencil_at(A, m, i, j):
    """the nine blocks of row (i, j)"""
    row = 2 * (i + m * j)
    cols = [2 * ((i + k % 3 - 1) + m * (j + k // 3 - 1)) for k in range(9)]
    return [A[row:row + 2, c:c + 2].toarray() for c in cols]


class HostVCycle:
    """the preconditioner on the host: coarse sizes (m + 2) >> 1 while more than
    10 nodes, less two levels; P^T A P, but that a row whose fine rows are all
    interior takes the stencil of a row far from the level's edges; four-colour
    block Gauss-Seidel, 20 sweeps on the bottom level"""

    def __init__(self, d, blocks):
        n, m = d.shape
        dims, (am, an) = [(m, n)], ((m + 2) >> 1, (n + 2) >> 1)
        while am * an > 10:
            dims.append((am, an))
            am, an = (am + 2) >> 1, (an + 2) >> 1
        dims = dims[:-2]
        self.A, self.P, self.sweep_data = [sparse_operator(d, blocks)], [], []
        interior = d.ravel() == -1
        inner = list(blocks.reshape(-1, 9, 2, 2)[np.flatnonzero(interior)[0]])
        for (fm, fn), (cm, cn) in zip(dims, dims[1:]):
            W = sp.kron(sp.csr_matrix(P1(fn, cn, False)), sp.csr_matrix(P1(fm, cm, False))).tocsr()
            P = sp.kron(W, sp.identity(2)).tocsr()
            A = (P.T @ self.A[-1] @ P).tocsr()
            assert min(fm, fn) >= 7
            P15 = sp.kron(sp.kron(sp.csr_matrix(P1(15, 8, False)), sp.csr_matrix(P1(15, 8, False))), sp.identity(2))
            inner = stencil_at((P15.T @ of_stencil(inner, 15, 15) @ P15).tocsr(), 8, 4, 4)
            interior = (abs(W).T @ ~interior) == 0
            keep = sp.diags(np.repeat(~interior, 2).astype(float))
            A = (keep @ A + (sp.identity(2 * cm * cn) - keep) @ of_stencil(inner, cm, cn)).tocsr()
            self.P.append(P)
            self.A.append(A)
        for (lm, ln), B in zip(dims, self.A):
            node = np.arange(lm * ln)
            colour = (node % lm & 1) + 2 * (node // lm & 1)
            per = []
            for c in range(4):
                k = node[colour == c]
                rows = np.stack([2 * k, 2 * k + 1], 1).ravel()
                D = np.stack([[np.asarray(B[2 * k + a, 2 * k + b]).ravel() for b in range(2)] for a in range(2)])
                per.append((rows, B[rows], np.linalg.inv(np.moveaxis(D, 2, 0))))
            self.sweep_data.append(per)

    def sweep(self, l, z, b):
        for rows, B, Dinv in self.sweep_data[l]:
            r = (b[rows] - B @ z).reshape(-1, 2, 1)
            z[rows] += (Dinv @ r).ravel()

    def __call__(self, b, l=0):
        z = np.zeros_like(b)
        if l + 1 == len(self.A):
            for _ in range(20):
                self.sweep(l, z, b)
            return z
        self.sweep(l, z, b)
        z += self.P[l] @ self(self.P[l].T @ (b - self.A[l] @ z), l + 1)
        self.sweep(l, z, b)
        return z


# levels on both sides of the 16 x 16 tiles with odd and even sides; below the
# top 261 (Galerkin tiles of 16, block kernel) and 301 nodes (too many tiles)
@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("m,n", [(N, N) for N in (47, 63, 64, 95, 126, 130, 161, 520, 600)] +
                         [(150, 47), (47, 130), (300, 96)])
def test_first_iteration_equals_the_host_v_cycle(m, n, form):
    print("case bd host V-cycle", m, n, form, flush=True)
    g = plate(m, n)
    g.set_precision(form)
    g.step_forward_quasistatic(0.5, 1)
    g.advection_step(0.5)
    g.post_process(False)
    d, blocks, b = g.operator(0.5)
    x0, b = g.get_vel().ravel().copy(), b.ravel()
    g.set_solver(max_iter=1)
    with pytest.raises(StzError) as e:
        g.projection_step(0.5)
    assert e.value.code == 3 and g.last_solve()["iterations"] == 1
    x = g.get_vel().ravel()
    g.close()
    M = HostVCycle(d, blocks)
    A = M.A[0]
    r = b - A @ x0
    ph = M(r)
    v = A @ ph
    alpha = (r @ r) / (r @ v)
    s = r - alpha * v
    sh = M(s)
    t = A @ sh
    want = alpha * ph + (t @ s) / (t @ t) * sh
    err = float(np.linalg.norm(x - x0 - want) / np.linalg.norm(want))
    print(m, n, form, "levels", len(M.A), "difference %.1e" % err)
    # FP64: some 20 sweeps and 2 a level, a few roundings each (measured up to
    # 1e-12); FP32: the same with its unit, 6e-8, less what the FP64 sums of the
    # iteration average out (measured up to 1.2e-6).  One coarse row off by its
    # prolongation weights shows at 5e-4 or more.
    assert err < (1e-11 if form == "fp64" else 1e-5)
