"""Operator sweeps and solves at the edges of the work-group tiles of the diagonal-view
traversals (16, 32 or 64 lanes along k, one, two or four cells per lane, marches of 1 to 16
planes) and of the CSR traversal, against the oracle.

The tile shape follows from the extents: these straddle each lane split, leave partial tiles
along k and j, and reach a march of every length from one plane (small grids) to sixteen."""
import numpy as np
import pytest

import dare_amd as da
import oracle as orc
from conftest import bits_equal

pytestmark = pytest.mark.gpu

SHAPES = [(5, 3, 16), (3, 17, 31), (2, 9, 32), (40, 5, 33), (9, 33, 64), (4, 4, 66), (2, 2, 96), (19, 6, 130),
          (70, 20, 24), (37, 41, 43), (66, 34)]
OPS = ["diff", "conv", "react"]


def system(ctx, rng, shape, op):
    import torch
    ncomp = 2 if op == "react" else 1
    dim = len(shape)
    go = orc.grid(list(shape), size=[0.1 * m for m in shape], ghost=2, ncomp=ncomp)
    cells = int(np.prod(shape))
    pad = int(np.prod([m + 4 for m in shape])) * ncomp
    kw = dict(dt=5e-3, bc_type=[1, 2, 1, 1, 2, 1][:2 * dim], bc_value=[0.3, 0.0, -1.0, 0.5, 0.0, 0.25][:2 * dim])
    arr = {}
    if op == "diff":
        kw["diff"] = 0.4
    elif op == "conv":
        arr["diff_cell"] = rng.uniform(0.1, 0.9, size=pad)
        kw["limiter"] = da.VANLEER
        arr["vel"] = [rng.uniform(-1, 1, size=cells // shape[d] * (shape[d] + 1)) for d in range(dim)]
    else:
        kw["diff_comp"] = [0.2, 0.5]
        k = rng.uniform(0.1, 10, size=(cells, 2))
        arr["react"] = np.stack([-k[:, 0], k[:, 1], k[:, 0], -k[:, 1]], axis=1).ravel()
    phi = rng.uniform(size=pad)
    ref = orc.assemble(go, orc.terms(**kw, **arr), phi)
    g = da.Grid.make(list(shape), size=[0.1 * m for m in shape], ghost=2, ncomp=ncomp)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    darr = {k: [dev(v) for v in a] if isinstance(a, list) else dev(a) for k, a in arr.items()}
    t = da.Terms.make(**kw, **darr)
    A = da.Csr(ctx)
    da.build_structure(ctx, A, g, t)
    b, x = dev(np.zeros(len(ref[3]))), dev(np.zeros(len(ref[3])))
    da.fill_values(ctx, A, g, t, dev(phi), b, x)
    ctx.synchronize()
    return A, b, x, ref, (t, darr)


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("shape", SHAPES)
def test_sweep_and_solves_on_tile_edges(ctx, rng, shape, op):
    import torch
    A, b, x0, (rp, col, val, rhs, ox0), keep = system(ctx, rng, shape, op)
    n = len(rhs)
    xs, ws = rng.normal(size=n), rng.normal(size=n)
    y = torch.zeros_like(b)
    if len(shape) < 3:                      # the CSR values are written on demand
        A.download()
    d = da.spmv_dot(ctx, A, torch.from_numpy(xs).cuda(), y, torch.from_numpy(ws).cuda())
    exp = orc.spmv(rp, col, val, xs)
    assert bits_equal(y.cpu().numpy(), exp)
    assert abs(d - float(exp @ ws)) <= 1e-12 * float(np.abs(exp) @ np.abs(ws))
    tol = 1e-12 * np.linalg.norm(rhs)
    xo, ok, it, *_ = orc.bicgstab2(rp, col, val, rhs, ox0, tol, 300)
    assert ok
    x = x0.clone()
    r = da.bicgstab2(ctx, A, b, x, tol=tol, tol_kind=0, max_it=300)
    assert r["converged"] == 1 and abs(r["iterations"] - it) <= 1
    assert abs(r["bnorm"] - np.linalg.norm(rhs)) <= 1e-13 * np.linalg.norm(rhs)
    assert np.max(np.abs(x.cpu().numpy() - xo)) <= 1e-12 * np.max(np.abs(xo)) + tol
    for precond in (0, 1):
        x = x0.clone()
        r = da.refine_mixed(ctx, A, b, x, tol=1e-10, tol_kind=1, inner_tol=1e-4, precond=precond)
        assert r["converged"] == 1
        assert np.linalg.norm(rhs - orc.spmv(rp, col, val, x.cpu().numpy())) <= 1e-10 * np.linalg.norm(rhs)
    A.close()


@pytest.mark.parametrize("shape,op", [((20, 163, 161), "conv"), ((41, 160, 161), "diff"), ((100, 101, 104), "conv"),
                                      ((112, 98, 96), "diff"), ((134, 135, 66), "conv"), ((71, 150, 150), "diff"),
                                      ((103, 200, 128), "react"), ((60, 2000, 22), "diff")])
def test_sweep_and_solves_on_both_sides_of_the_tile_rules_lines(ctx, rng, shape, op):
    """Half a million to 2.7 M rows: narrow tiles below the line and wide ones above it, marches of 2 to
    16 planes chosen by how evenly they fall on the CUs, with the last tile and the last march cut."""
    test_sweep_and_solves_on_tile_edges(ctx, rng, shape, op)


@pytest.mark.parametrize("shape,op", [((600, 701), "conv"), ((1446, 1450), "conv"), ((1450, 1447), "diff"),
                                      ((1698, 1699), "diff"), ((20000, 4, 4), "conv"), ((101, 102, 103), "diff")])
def test_solves_on_both_sides_of_the_fused_steps_lines(ctx, rng, shape, op):
    """CSR steps whose work-groups loop over their rows, CSR and view solves just below and just above
    the row counts from which the separate kernels take over, and tiles that are mostly idle."""
    test_sweep_and_solves_on_tile_edges(ctx, rng, shape, op)


@pytest.mark.parametrize("n", [1, 257])
def test_breakdown_after_the_first_x_update_keeps_it(ctx, n):
    """A multiple of the identity breaks the method down in its first pass after step 10 (r = 0,
    so the second gamma is 0): x has then moved to the solution, as in the oracle's order of the
    updates -- in the FP64 solve, and in the zero-guess FP32 solve inside the refinement."""
    import torch
    rp, col, val = np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.full(n, 2.0)
    A = da.Csr(ctx)
    da.upload_host_csr(ctx, A, rp, col, val)
    b = np.arange(1, n + 1, dtype=np.float64)
    xo, ok, it, res, _ = orc.bicgstab2(rp, col, val, b, np.zeros(n), 1e-30, 10)
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    r = da.bicgstab2(ctx, A, torch.from_numpy(b).cuda(), x, tol=1e-30, tol_kind=0, max_it=10)
    assert r["status"] == da.DARE_ERR_BREAKDOWN and not ok
    assert bits_equal(x.cpu().numpy(), xo) and np.array_equal(xo, b / 2)
    x.zero_()
    r = da.refine_mixed(ctx, A, torch.from_numpy(b).cuda(), x, tol=0.0, tol_kind=0, max_refine=1)
    assert np.array_equal(x.cpu().numpy(), b / 2)
    A.close()


def test_jacobi_scaled_views_of_half_and_full_fills_agree(ctx, rng):
    """4 M rows, where the FP32 column-scaled view's C slot is taken as 1 and not stored: the view
    scaled from a fill that left E, N, T out and the one scaled from all seven slots give the same
    mixed and FP64 Jacobi solves bit for bit, to a true residual below the tolerance."""
    import torch
    n = [128, 128, 256]
    g = da.Grid.make(n, ghost=2)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    D = torch.rand(g.num_padded, generator=gen, dtype=torch.float64, device="cuda") + 0.1
    phi = torch.rand(g.num_padded, generator=gen, dtype=torch.float64, device="cuda")
    t = da.Terms.make(dt=2e-5, diff_cell=D, bc_type=[1, 2, 1, 1, 2, 1], bc_value=[0.3, 0, -1.0, 0.5, 0, 0.25])
    got = {}
    for half in (True, False):
        A = da.Csr(ctx)
        da.build_structure(ctx, A, g, t)
        da.set_symmetric_traversal(A, half)
        b = torch.zeros(g.num_cells, dtype=torch.float64, device="cuda")
        x = torch.zeros_like(b)
        for mixed in (True, False):
            da.fill_values(ctx, A, g, t, phi, b, x)
            if mixed:
                r = da.refine_mixed(ctx, A, b, x, tol=1e-10, precond=1)
            else:
                r = da.bicgstab2(ctx, A, b, x, tol=1e-10, tol_kind=1, precond=1)
            assert r["converged"] == 1
            y = torch.zeros_like(x)
            assert da.residual(ctx, A, b, x, y, norm=True) <= 1.01e-10 * float(b.norm())
            got[half, mixed] = (x.cpu().numpy().copy(), r["iterations"])
        A.close()
    for mixed in (True, False):
        assert bits_equal(got[True, mixed][0], got[False, mixed][0]) and got[True, mixed][1] == got[False, mixed][1]


def v_cycle(A, shape, r):
    """The multigrid preconditioner as its definition reads: aggregates of 2 x 2 x 2 cells, coarse
    operator P^T E P + P^T L P / 2 (E the row sums, L the rest), W = 0.8 / diag, one damped Jacobi
    sweep before and after, twelve on the first level of at most 1024 rows."""
    import scipy.sparse as sp
    n = A.shape[0]
    W = 0.8 / A.diagonal()
    if v_cycle.depth and n <= 1024:
        z = W * r
        for _ in range(11):
            z = z + W * (r - A @ z)
        return z
    idx = np.indices(shape).reshape(3, -1) // 2
    coarse = [(m + 1) // 2 for m in shape]
    P = sp.csr_matrix((np.ones(n), (np.arange(n), np.ravel_multi_index(tuple(idx), coarse))),
                      shape=(n, int(np.prod(coarse))))
    E = sp.diags(np.asarray(A.sum(axis=1)).ravel())
    Ac = (P.T @ E @ P + 0.5 * (P.T @ (A - E) @ P)).tocsr()
    z = W * r
    v_cycle.depth += 1
    z = z + P @ v_cycle(Ac, coarse, P.T @ (r - A @ z))
    v_cycle.depth -= 1
    return z + W * (r - A @ z)


v_cycle.depth = 0


@pytest.mark.parametrize("op", ["diff", "conv"])
@pytest.mark.parametrize("shape", [(12, 11, 9), (3, 17, 31), (18, 17, 2), (40, 40, 3), (9, 33, 64), (5, 3, 66),
                                   (2, 9, 130), (19, 20, 24), (37, 41, 43)])
def test_multigrid_pass_matches_the_definition(ctx, rng, shape, op):
    """One BiCGStab2 pass with the V-cycle, symmetric (E, N, T slots not read) and not, at odd
    extents and at the edges of the runs of 2 to 64 cells along k. The pass is a handful of
    products and dots whose rounding (1e-16 times the condition of its 2 x 2 least-squares step,
    below 1e4) stays under 1e-11 of the solution; a misplaced coefficient shows from 1e-4 up."""
    import scipy.sparse as sp
    A, b, x, (rp, col, val, rhs, _), keep = system(ctx, rng, shape, op)
    M = sp.csr_matrix((val, col, rp), shape=(len(rhs),) * 2)
    prec = lambda p: v_cycle(M, list(shape), p)
    mul = lambda p: M @ prec(p)
    r = rh = u = rhs
    v = mul(u)
    alpha = (rh @ r) / (rh @ v)
    y, r1 = alpha * u, r - alpha * v
    s = mul(r1)
    beta = alpha * (rh @ s) / (rh @ r)
    v = s - beta * v
    w = mul(v)
    alpha = (rh @ s) / (rh @ w)
    u, r1, s = r1 - beta * u, r1 - alpha * v, s - alpha * w
    t = mul(s)
    om1, mu, nu, tau, om2 = r1 @ s, s @ s, s @ t, t @ t, r1 @ t
    om2 = (om2 - nu * om1 / mu) / (tau - nu * nu / mu)
    om1 = (om1 - nu * om2) / mu
    ref = prec(y + om1 * r1 + om2 * s + alpha * u)
    x.zero_()
    da.bicgstab2(ctx, A, b, x, tol=1e-300, tol_kind=0, max_it=1, precond=da.PRECOND_MG)
    got = x.cpu().numpy()
    assert np.max(np.abs(got - ref)) <= 1e-9 * np.max(np.abs(ref))
    A.close()


@pytest.mark.parametrize("op", ["diff", "var", "conv", "react", "all"])
@pytest.mark.parametrize("shape,per", [([9], [0]), ([2], [1]), ([1, 7], [1, 0]), ([2, 5], [1, 1]), ([3, 40], [0, 1]),
                                       ([17, 16], [0, 0]), ([1, 2, 5], [1, 1, 0]), ([3, 2, 9], [0, 1, 1])])
def test_csr_rows_of_every_instantiation_match_oracle(ctx, rng, shape, per, op):
    """Row pointers, columns and values, bit for bit: each combination of terms with its own fill
    kernel, and periodic axes of one and two cells, whose neighbours share a column and merge (not
    with a reaction, where the oracle keeps one of two equal columns; the device adds them)."""
    import torch
    if op == "react" and any(p and m <= 2 for p, m in zip(per, shape)):
        pytest.skip("the oracle does not merge columns of rows with cross-component entries")
    dim, ncomp = len(shape), 2 if op == "react" else 1
    cells, pad = int(np.prod(shape)), int(np.prod([m + 4 for m in shape])) * ncomp
    edge = lambda e: [0 if per[f // 2] else e[f] for f in range(2 * dim)]
    kw = dict(dt=5e-3, bc_type=edge([1, 2, 1, 1, 2, 1]), bc_value=edge([0.3, 0.0, -1.0, 0.5, 0.0, 0.25]))
    arr = {}
    if op in ("var", "all"):
        arr["diff_cell"] = rng.uniform(0.1, 0.9, size=pad)
        arr["source"] = rng.uniform(-1, 1, size=pad)
    else:
        kw["diff"] = 0.4
    if op in ("conv", "all"):
        kw["limiter"] = da.VANLEER
        arr["vel"] = [rng.uniform(-1, 1, size=cells // shape[d] * (shape[d] + 1)) for d in range(dim)]
    if op == "react":
        arr["react"] = rng.uniform(-5, 5, size=4 * cells)
    if op == "all":
        kw["bc_type"] = edge([3, 2, 1, 1, 2, 1])
    phi = rng.uniform(size=pad)
    go = orc.grid(shape, size=[0.1 * m for m in shape], ghost=2, ncomp=ncomp, periodic=per)
    rp, col, val, rhs, x0 = orc.assemble(go, orc.terms(**kw, **arr), phi)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    darr = {k: [dev(v) for v in a] if isinstance(a, list) else dev(a) for k, a in arr.items()}
    g = da.Grid.make(shape, size=[0.1 * m for m in shape], ghost=2, ncomp=ncomp, periodic=per)
    t = da.Terms.make(**kw, **darr)
    A = da.Csr(ctx)
    da.build_structure(ctx, A, g, t)
    b, x = dev(np.zeros(len(rhs))), dev(np.zeros(len(rhs)))
    da.fill_values(ctx, A, g, t, dev(phi), b, x)
    ctx.synchronize()
    grp, gcol, gval = A.download()
    assert np.array_equal(grp, rp) and np.array_equal(gcol, col)
    assert bits_equal(gval, val) and bits_equal(b.cpu().numpy(), rhs) and bits_equal(x.cpu().numpy(), x0)
    A.close()


@pytest.mark.parametrize("shape", [(5, 7, 9), (21, 18, 33), (24, 23, 30), (161, 163, 163), (162, 163, 162)])
def test_symmetric_sweeps_of_every_extent_give_the_same_bits(ctx, rng, shape):
    """Four slots of a symmetric view instead of seven, one or two cells a lane, cached and (from
    4 M rows) streaming, in FP64 and FP32: the partner coefficients are the same numbers in the same
    order, so products, solutions and passes agree bit for bit."""
    import torch
    got = []
    A, b, x0, *_, keep = system(ctx, rng, shape, "diff")
    t = keep[0]
    g = da.Grid.make(list(shape), size=[0.1 * m for m in shape], ghost=2)
    phi = torch.from_numpy(rng.uniform(size=int(np.prod([m + 4 for m in shape])))).cuda()
    v = torch.from_numpy(rng.normal(size=b.numel())).cuda()
    for on in (True, False):
        da.set_symmetric_traversal(A, on)
        da.fill_values(ctx, A, g, t, phi, b, x0)
        y = torch.zeros_like(v)
        da.spmv_dot(ctx, A, v, y, b)
        xs = [x0.clone() for _ in range(3)]
        r = [da.bicgstab2(ctx, A, b, xs[0], tol=1e-9, tol_kind=1, max_it=40),
             da.refine_mixed(ctx, A, b, xs[1], tol=1e-9, tol_kind=1, inner_tol=1e-3),
             da.bicgstab2(ctx, A, b, xs[2], tol=1e-9, tol_kind=1, max_it=40, precond=da.PRECOND_MG)]
        assert all(q["converged"] == 1 for q in r)
        got.append(([a.cpu().numpy() for a in [y] + xs], [q["iterations"] for q in r]))
    assert all(bits_equal(p, q) for p, q in zip(got[0][0], got[1][0])) and got[0][1] == got[1][1]
    A.close()


@pytest.mark.parametrize("c", [0.0, 2.0])
@pytest.mark.parametrize("shape", [(4, 6), (5, 7, 9), (6, 7, 10), (9, 8, 12), (128, 128, 256), (161, 163, 161),
                                   (161, 163, 163)])
def test_views_that_are_multiples_of_the_identity(ctx, rng, shape, c):
    """Cells of volume 1 without diffusion: the operator is (1 / dt) I with explicit zeros beside its
    diagonal, whose solves break down in their first pass, before step 10 (0 I, x stays) and after it
    (2 I, x has moved to the solution), in the fused steps and in the separate kernels, on four slots
    and on seven. Whole numbers make every sum exact, so x is the oracle's to the bit."""
    import torch
    go = orc.grid(list(shape), size=list(map(float, shape)), ghost=1)
    g = da.Grid.make(list(shape), size=list(map(float, shape)), ghost=1)
    kw = dict(dt=1 / c if c else 0.0, diff=0.0, bc_type=[1] * 6, bc_value=[0.0] * 6)
    rp, col, val, *_ = orc.assemble(go, orc.terms(**kw), np.zeros(int(np.prod([m + 2 for m in shape]))))
    n = len(rp) - 1
    b, x0 = (rng.integers(-8, 9, size=n).astype(np.float64) for _ in range(2))
    xo, ok, it, *_ = orc.bicgstab2(rp, col, val, b, x0, 1e-30, 10)
    assert not ok and it == 1 and np.array_equal(xo, b / 2 if c else x0)
    bd, phi = torch.from_numpy(b).cuda(), torch.zeros(g.num_padded, dtype=torch.float64, device="cuda")
    A = da.Csr(ctx)
    t = da.Terms.make(**kw)
    da.build_structure(ctx, A, g, t)
    x = torch.zeros_like(bd)
    for symmetric in (True, False):
        if len(shape) == 3:
            da.set_symmetric_traversal(A, symmetric)
        da.fill_values(ctx, A, g, t, phi, torch.zeros_like(bd), x)
        for precond in (0, 1) if c else (0,):
            x.copy_(torch.from_numpy(x0))
            r = da.bicgstab2(ctx, A, bd, x, tol=1e-30, tol_kind=0, max_it=10, precond=precond)
            assert r["status"] == da.DARE_ERR_BREAKDOWN and r["converged"] == 0 and r["iterations"] == 1
            assert bits_equal(x.cpu().numpy(), xo)
            x.copy_(torch.from_numpy(x0))
            r = da.refine_mixed(ctx, A, bd, x, tol=1e-30, tol_kind=0, precond=precond)
            assert r["status"] == da.DARE_ERR_BREAKDOWN and r["converged"] == 0 and r["refinements"] == 1
            assert np.array_equal(x.cpu().numpy(), xo)
    A.close()


@pytest.mark.parametrize("copies", [1, 128])
@pytest.mark.parametrize("M,b,loose", [([[-1, 2], [-1, 0]], [1, 0], 0), ([[-2, -2], [2, 1]], [2, 0], 0),
                                       ([[-2, 2, -1], [0, -1, -2], [0, 1, 0]], [0, 1, 0], 0),
                                       ([[-2, 1, 0], [2, 2, 2], [1, 0, -1]], [0, 2, 0], 0),
                                       ([[-2, 1, 0], [2, 2, 2], [1, 0, -1]], [0, 2, 0], 1.5)])
def test_breakdown_at_mu_and_tau(ctx, M, b, loose, copies):
    """Blocks whose first pass ends at mu == 0 (s = 0) or at tau == 0 (t parallel to s) in exact binary
    fractions: x keeps step 10 alone, and at tau == 0 the true residual decides on convergence."""
    import scipy.sparse as sp
    import torch
    S = sp.kron(sp.eye(copies), sp.csr_matrix(np.ones_like(M))).tocsr()
    S.sort_indices()
    rp, col = S.indptr.astype(np.int32), S.indices.astype(np.int32)
    val, b = np.tile(np.asarray(M, np.float64).ravel(), copies), np.tile(np.asarray(b, np.float64), copies)
    tol = loose * np.sqrt(copies) if loose else 1e-30
    xo, ok, it, res, _ = orc.bicgstab2(rp, col, val, b, np.zeros(len(b)), tol, 10)
    assert ok == bool(loose) and it == 1 and np.any(xo)
    A = da.Csr(ctx)
    da.upload_host_csr(ctx, A, rp, col, val)
    x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    r = da.bicgstab2(ctx, A, torch.from_numpy(b).cuda(), x, tol=tol, tol_kind=0, max_it=10)
    assert r["status"] == (0 if ok else da.DARE_ERR_BREAKDOWN)
    assert r["converged"] == ok and r["iterations"] == it and r["residual"] == res
    assert bits_equal(x.cpu().numpy(), xo)
    A.close()


@pytest.mark.parametrize("op", ["diff", "conv"])
def test_solves_of_more_planes_than_a_launch_has_along_z(ctx, rng, op):
    test_sweep_and_solves_on_tile_edges(ctx, rng, (66000, 2, 3), op)
