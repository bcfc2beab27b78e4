"""Operator products from the reference blocks (meshes of translated copies of
one element): solves on blocks, on meshes with elements missing, on skewed
elements, with a mass term, and on a cracked mesh (two nodes at one place, where
the lattice is not unique and the assembled values are used), against a
sparse direct solve of the assembled matrix; the FP32 product against the
assembled FP64 one."""
import dataclasses

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from asend3d_amd import api, problems
from conftest import gpu_case

pytestmark = pytest.mark.gpu


def reduced(p, keep):
    """The problem on the elements of the mask, unused nodes dropped."""
    m = p.mesh
    conn = m.conn[keep]
    used = np.unique(conn)
    new = np.full(m.n_nodes, -1, dtype=np.int64)
    new[used] = np.arange(used.size)
    clamp = new[p.clamp_nodes][new[p.clamp_nodes] >= 0].astype(np.int32)
    xyz = m.xyz[used]
    conn = new[conn].astype(np.int32)
    return build(xyz, conn, p.E[keep], p.nu[keep], clamp, p.etype)


def build(xyz, conn, E, nu, clamp, etype):
    _, di, n_dof = api.reorder_nodes(xyz, conn, 3, [[clamp]] * 3, 48)
    pen = np.concatenate([di[clamp, c] for c in range(3)]).astype(np.int64)
    f = np.random.default_rng(1).standard_normal(n_dof)
    f[pen] = 0.0
    return dict(xyz=xyz, conn=conn, E=E, nu=nu, di=di, n_dof=n_dof, pen=pen, f=f, etype=etype)


def case(name):
    p = problems.heterogeneous(*{"block 7x3x3": (7, 3, 3), "block 8x6x5": (8, 6, 5)}.get(name, (9, 5, 4)), seed=3)
    m = p.mesh
    n = m.n_el
    whole = np.ones(n, bool)
    if name == "brickim":
        return reduced(dataclasses.replace(p, etype=81), whole)
    if name == "holes":  # an L, a hole through the middle and a lone corner contact
        e = np.arange(n)
        i, j, k = e % m.nx, e // m.nx % m.ny, e // (m.nx * m.ny)
        return reduced(p, ~((i > 5) & (j > 2)) & ~((i == 3) & (j == 2)) & ~((i == 1) & (k == 1) & (j == 0)))
    if name == "skew":
        s = reduced(p, whole)
        A = np.array([[1.0, 0.3, 0.1], [0.0, 1.0, 0.2], [0.0, 0.0, 1.0]])
        return {**s, "xyz": np.ascontiguousarray(s["xyz"] @ A.T)}
    if name == "crack":  # the upper elements of one plane get their own nodes over half the section
        xyz, conn = m.xyz.copy(), m.conn.copy()
        e = np.arange(n)
        up = (e // (m.nx * m.ny) == 2) & (e % m.nx >= 4)
        at = np.unique(conn[up][:, :4])
        at = at[m.xyz[at, 0] > m.xyz[:, 0].max() * 0.6]
        dup = np.full(m.n_nodes, -1)
        dup[at] = m.n_nodes + np.arange(at.size)
        c = conn[up][:, :4]
        conn[np.flatnonzero(up)[:, None], np.arange(4)] = np.where(dup[c] >= 0, dup[c], c)
        return build(np.vstack([xyz, xyz[at]]), conn.astype(np.int32), p.E, p.nu, p.clamp_nodes, 8)
    return reduced(p, whole)


# 128 nodes (whole slices), 378 and 300 (a partial one)
@pytest.mark.parametrize("name", ["block 7x3x3", "block 8x6x5", "block 9x5x4", "brickim", "holes", "skew", "crack"])
@pytest.mark.parametrize("mass", [False, True])
def test_solves_match_assembled_matrix(ctx, name, mass):
    gpu_case(f"reference-block solve {name} mass={mass}")
    s = case(name)
    E = np.full_like(s["E"], 7.0e4) if mass else s["E"]
    ctx.upload_mesh(s["etype"], s["xyz"], s["di"], s["n_dof"], s["conn"], E, s["nu"], np.full(E.size, 2.7e-9))
    ctx.set_penalty(s["pen"], 0.0)
    assert ctx.uniform_elements()
    ctx.assemble(c_mass=4.0e13 if mass else 0.0)
    rp, cols, vals = ctx.get_matrix()
    K = sp.csr_matrix((vals, cols, rp), shape=(s["n_dof"], s["n_dof"])).tocsc()
    ref = spla.spsolve(K, s["f"])
    for method, tol, bar in ((api.SOLVE_PCG_FP64, 1e-11, 1e-8), (api.SOLVE_IR_MIXED, 1e-10, 1e-7)):
        u, st = ctx.solve(s["f"], ctx.opts(method, api.PC_JACOBI, tol=tol, max_it=200000, max_outer=60))
        assert st.converged
        # the solves' own residual is that of the assembled matrix
        res = np.linalg.norm(s["f"] - K @ u) / np.linalg.norm(s["f"])
        assert res <= 4 * tol, (res, st.rel_residual)
        assert np.linalg.norm(u - ref) <= bar * np.linalg.norm(ref)


def test_moduli_update_and_other_assemblies(ctx):
    """The products follow every assembly: new moduli, then a tangent (assembled
    values), then the moduli again."""
    gpu_case("reference-block operator across assemblies")
    p = problems.heterogeneous(10, 4, 4, seed=5)
    problems.upload(ctx, p)
    o = ctx.opts(api.SOLVE_PCG_FP64, api.PC_JACOBI, tol=1e-11, max_it=100000)
    E2 = p.E[::-1].copy()

    def check():
        rp, cols, vals = ctx.get_matrix()
        K = sp.csr_matrix((vals, cols, rp), shape=(p.n_dof, p.n_dof)).tocsc()
        u, st = ctx.solve(p.f, o)
        ref = spla.spsolve(K, p.f)
        assert np.linalg.norm(u - ref) <= 1e-8 * np.linalg.norm(ref)
        return u

    ctx.assemble()
    u1 = check()
    ctx.update_moduli(E2)
    ctx.assemble()
    check()
    ctx.nl_assemble(20.0 * u1)
    check()
    ctx.update_moduli(p.E)
    ctx.assemble()
    assert np.array_equal(check(), u1)


@pytest.mark.parametrize("dims", [(7, 3, 3), (13, 6, 5)])
def test_fp32_product(ctx, dims):
    gpu_case(f"reference-block FP32 product {dims}")
    p = problems.heterogeneous(*dims, seed=2)
    problems.upload(ctx, p)
    ctx.set_grid(*dims)
    ctx.assemble()
    x = np.random.default_rng(3).standard_normal(p.n_dof)
    y = ctx.spmv(x, 64)
    # 8 elements x 24 products of FP32 values, each rounded to 2^-24
    free = np.ones(p.n_dof, bool)
    free[p.pen_dofs] = False
    d = ctx.mg_apply(0, x) - y
    assert np.linalg.norm(d[free]) <= 1e-6 * np.linalg.norm(y[free])
    assert np.abs(d[~free] / y[~free]).max() <= 1e-6


# step kernels that add the product's partial sums themselves: more product
# workgroups than they take (assembled values, 8,375 slices by four: folded first)
# and several slices to a workgroup (reference blocks)
@pytest.mark.parametrize("distorted", [True, False])
def test_many_partial_sums(ctx, distorted):
    gpu_case(f"PCG on 536,000 nodes distorted={distorted}")
    p = problems.cantilever(66, 89, 88, 66.0, 89.0, 88.0, E=7.0e4, nu=0.3, traction=(0.0, 0.0, -1.0))
    if distorted:
        p = problems.distorted(p, 3)
    problems.upload(ctx, p)
    ctx.assemble()
    assert ctx.uniform_elements() != distorted
    u, st = ctx.solve(p.f, ctx.opts(api.SOLVE_PCG_FP64, api.PC_JACOBI, tol=1e-6, max_it=5000, check_every=33))
    assert st.converged and st.iterations < 1500
    res = np.linalg.norm(p.f - ctx.spmv(u)) / np.linalg.norm(p.f)
    assert res <= 1.01e-6, res


# constraint sets that touch few slices, more of them, and fewer again
def constraint_sets(p):
    x = p.mesh.xyz
    di = np.asarray(p.dof_index).reshape(-1, 6)[:, :3]
    left, right, floor = (np.isclose(x[:, 0], 0.0), np.isclose(x[:, 0], x[:, 0].max()), np.isclose(x[:, 2], 0.0))
    half = left & (x[:, 1] <= 0.5 * x[:, 1].max())
    return [di[s].reshape(-1).astype(np.int64) for s in (left, left | right | floor, half)]


@pytest.mark.parametrize("precond", [api.PC_MG, api.PC_LEARNED])
def test_new_constraints_between_solves(precond):
    """A context whose captured iterations have run goes on after each new set
    of constraints as a context that never had another one: the same
    iterations and solution, and that of the assembled matrix."""
    gpu_case(f"constraints changed between multigrid solves, preconditioner {precond}")
    dims = (33, 9, 7)
    p = problems.heterogeneous(*dims, seed=6, sigma_ln=0.7)
    f = np.random.default_rng(2).standard_normal(p.n_dof)

    def make():
        c = api.Context(0)
        c.learned_init(1)
        problems.upload(c, p)
        c.set_grid(*dims)
        return c

    def solve(c, pen):
        c.set_penalty(pen, 0.0)
        c.assemble()
        rhs = f.copy()
        rhs[pen] = 0.0
        u, st = c.solve(rhs, c.opts(api.SOLVE_IR_MIXED, precond, tol=1e-9, inner_tol=1e-3, max_it=2000, check_every=3))
        assert st.converged and st.fallback_used == 0
        rp, cols, vals = c.get_matrix()
        ref = spla.spsolve(sp.csr_matrix((vals, cols, rp), shape=(p.n_dof, p.n_dof)).tocsc(), rhs)
        assert np.linalg.norm(u - ref) <= 1e-5 * np.linalg.norm(ref)
        return u, st.iterations

    old = make()
    for k, pen in enumerate(constraint_sets(p)):
        new = make()
        (u, it), (u_new, it_new) = solve(old, pen), solve(new, pen)
        assert it == it_new and np.array_equal(u, u_new), (k, it, it_new)
        new.close()
    old.close()


def test_new_network_between_solves():
    """A network made anew after solves with captured iterations, its arrays in
    other places (some of the old ones taken by another context's)."""
    gpu_case("network made anew between solves")
    dims = (17, 7, 6)
    p = problems.heterogeneous(*dims, seed=6, sigma_ln=0.7)
    o = api.Context.opts(api.SOLVE_IR_MIXED, api.PC_LEARNED, tol=1e-9, inner_tol=1e-3, max_it=2000, check_every=3)

    def make(seed):
        c = api.Context(0)
        c.learned_init(seed)
        problems.upload(c, p)
        c.set_grid(*dims)
        c.assemble()
        c.learned_train(4, seed=3)
        return c

    old = make(1)
    old.solve(p.f, o)
    old.learned_init(2)
    new = make(2)
    old.learned_train(4, seed=3)
    for _ in range(2):
        (u, st), (u_new, st_new) = old.solve(p.f, o), new.solve(p.f, o)
        assert st.converged and st.fallback_used == 0 and st.iterations == st_new.iterations
        assert np.array_equal(u, u_new)
    new.close()
    old.close()


@pytest.mark.parametrize("mode", [api.NM_FP64, api.NM_MIXED])
def test_new_constraints_between_newmark_runs(mode):
    """The same of Newmark steps, whose captured launches also outlive a change
    of the constraints."""
    gpu_case(f"constraints changed between Newmark runs, solver {mode}")
    p = problems.cantilever(20, 5, 4)
    n = 30
    fac = np.sin(np.pi * np.arange(n) / n)
    f = np.random.default_rng(4).standard_normal(p.n_dof)

    def make(pen):
        c = api.Context(0)
        problems.upload(c, p, rho=np.full(p.mesh.n_el, 7850.0))
        c.set_penalty(pen, 0.0)
        c.newmark_set_solver(mode)
        c.newmark_setup(5e-5, 0.25, 0.5)
        return c

    def run(c):
        _, u, v, a, st = c.newmark_run(n, f, fac, tol=1e-10, max_it_step=400)
        assert st.graph_used == 1 and st.unconverged_steps == 0
        return u, v, a, st.total_iterations

    sets = constraint_sets(p)
    old = make(sets[0])
    for k, pen in enumerate(sets):
        if k:
            old.set_penalty(pen, 0.0)
        new = make(pen)
        a, b = run(old), run(new)
        assert a[3] == b[3] and all(np.array_equal(x, y) for x, y in zip(a[:3], b[:3])), (k, a[3], b[3])
        new.close()
    old.close()
