"""Diagonal views whose rows wrap around an axis, against the oracle.

On a grid with a periodic axis every row's missing neighbour is the cell at the other end of its
axis unless a boundary edit removed the entry, whichever axis it is: periodic axes, axes whose
faces carry no edit beside a periodic one, and axes with an edit at one face only. Products,
solves of every kind and the multigrid pass, four slots against seven."""
import numpy as np
import pytest

import dare_amd as da
import oracle as orc
from conftest import bits_equal
from test_gpu_tiles import v_cycle

pytestmark = pytest.mark.gpu

# (periodic, boundary types)
WRAPS = {"all": ([1, 1, 1], [0, 0, 0, 0, 0, 0]), "axis0": ([1, 0, 0], [0, 0, 1, 2, 2, 1]),
         "axis1": ([0, 1, 0], [1, 2, 0, 0, 2, 1]), "axis2": ([0, 0, 1], [1, 2, 2, 1, 0, 0]),
         "edits_on_a_periodic_axis": ([1, 0, 1], [1, 2, 1, 1, 0, 0]),
         "no_edits_beside": ([0, 0, 1], [0, 0, 1, 2, 0, 0]), "no_edits_beside_k": ([1, 0, 0], [0, 0, 2, 1, 0, 0]),
         "edit_below": ([1, 0, 1], [1, 0, 2, 1, 0, 0]), "edit_above": ([1, 0, 1], [0, 1, 2, 1, 0, 0]),
         "edit_below_k": ([0, 0, 1], [1, 2, 1, 1, 2, 0]), "edit_below_beside_k": ([1, 0, 0], [0, 0, 1, 0, 1, 0])}


def system(ctx, rng, shape, wrap, op):
    import torch
    per, bc = WRAPS[wrap]
    cells, pad = int(np.prod(shape)), int(np.prod([m + 4 for m in shape]))
    size = [0.1 * m for m in shape]
    kw = dict(dt=5e-3, bc_type=bc, bc_value=[0.3, 0.0, -1.0, 0.5, 0.0, 0.25])
    arr = {}
    if op == "diff":
        kw["diff"] = 0.4
    else:
        arr["diff_cell"] = rng.uniform(0.1, 0.9, size=pad)
    if op == "conv":
        kw["limiter"] = da.VANLEER
        arr["vel"] = [rng.uniform(-1, 1, size=cells // shape[d] * (shape[d] + 1)) for d in range(3)]
    phi = rng.uniform(size=pad)
    ref = orc.assemble(orc.grid(list(shape), size=size, ghost=2, periodic=per), orc.terms(**kw, **arr), phi)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    darr = {k: [dev(v) for v in a] if isinstance(a, list) else dev(a) for k, a in arr.items()}
    g = da.Grid.make(list(shape), size=size, ghost=2, periodic=per)
    t = da.Terms.make(**kw, **darr)
    A = da.Csr(ctx)
    da.build_structure(ctx, A, g, t)
    b, x = dev(np.zeros(cells)), dev(np.zeros(cells))
    fill = lambda: da.fill_values(ctx, A, g, t, phi_d, b, x)
    phi_d = dev(phi)
    fill()
    ctx.synchronize()
    return A, b, x, ref, fill, (darr, phi_d)


@pytest.mark.parametrize("op", ["diff", "var", "conv"])
@pytest.mark.parametrize("wrap", list(WRAPS))
@pytest.mark.parametrize("shape", [(6, 5, 8), (5, 7, 9), (2, 3, 4), (3, 2, 2), (4, 9, 66), (9, 33, 64)])
def test_products_and_solves_of_wrapped_views_match_oracle(ctx, rng, shape, wrap, op):
    """Well conditioned systems (below 10): the recurrence's residual stays within 1e-13 ||b|| of the
    true one, and a wrong or misplaced coefficient moves it by 1e-3 and more."""
    import scipy.sparse as sp
    import torch
    A, b, x0, (rp, col, val, rhs, ox0), fill, keep = system(ctx, rng, shape, wrap, op)
    n = len(rhs)
    M = sp.csr_matrix((val, col, rp), shape=(n, n))
    v, w = rng.normal(size=n), rng.normal(size=n)
    vd, wd, y = torch.from_numpy(v).cuda(), torch.from_numpy(w).cuda(), torch.zeros_like(b)
    got = []
    for symmetric in (True, False):
        da.set_symmetric_traversal(A, symmetric)
        fill()
        assert bits_equal(b.cpu().numpy(), rhs) and bits_equal(x0.cpu().numpy(), ox0)
        da.spmv_dot(ctx, A, vd, y, wd)
        # at most eight products a row, in another order than the oracle's at the wraps
        assert np.all(np.abs(y.cpu().numpy() - M @ v) <= 16 * 2.0 ** -53 * (abs(M) @ np.abs(v)))
        out = [y.cpu().numpy().copy()]
        for precond in (0, 1, da.PRECOND_MG):
            for mixed in (False, True):
                x = x0.clone()
                if mixed:
                    r = da.refine_mixed(ctx, A, b, x, tol=1e-10, tol_kind=1, inner_tol=1e-4, precond=precond)
                else:
                    r = da.bicgstab2(ctx, A, b, x, tol=1e-10, tol_kind=1, max_it=60, precond=precond)
                assert r["converged"] == 1, (precond, mixed, r)
                x = x.cpu().numpy()
                assert np.linalg.norm(rhs - M @ x) <= 1.01e-10 * np.linalg.norm(rhs), (precond, mixed)
                out.append(x)
        grp, gcol, gval = A.download()
        assert np.array_equal(grp, rp) and np.array_equal(gcol, col) and bits_equal(gval, val)
        got.append(out)
    assert all(bits_equal(p, q) for p, q in zip(*got))
    A.close()


@pytest.mark.parametrize("shape,wrap,op", [((162, 163, 162), "all", "diff"), ((161, 163, 163), "axis0", "diff"),
                                           ((128, 128, 260), "no_edits_beside", "conv")])
def test_products_and_solves_of_wrapped_views_above_four_million_rows(ctx, rng, shape, wrap, op):
    test_products_and_solves_of_wrapped_views_match_oracle(ctx, rng, shape, wrap, op)


@pytest.mark.parametrize("op", ["diff", "var", "conv"])
@pytest.mark.parametrize("shape", [(1, 6, 8), (6, 1, 4), (5, 4, 1), (1, 1, 6), (1, 5, 64)])
def test_products_and_solves_of_views_with_a_periodic_axis_of_one_cell(ctx, rng, shape, op):
    """A cell coupled to itself through both faces: the check on the device decides on the symmetric
    traversals, and the entries merge on the diagonal of the CSR rows."""
    test_products_and_solves_of_wrapped_views_match_oracle(ctx, rng, shape, "all", op)


@pytest.mark.parametrize("op", ["diff", "conv"])
@pytest.mark.parametrize("wrap", list(WRAPS))
@pytest.mark.parametrize("shape", [(12, 11, 9), (3, 17, 32), (18, 17, 2), (9, 33, 64), (2, 9, 130)])
def test_multigrid_pass_on_wrapped_views_matches_the_definition(ctx, rng, shape, wrap, op):
    """One BiCGStab2 pass with the V-cycle as its definition reads, where aggregates couple around the
    axes, also those of a last layer of one cell and of coarse axes of one and two cells. A handful
    of products and dots, rounding under 1e-11 of the solution (the condition of the pass's 2 x 2
    least-squares step is below 1e4)."""
    import scipy.sparse as sp
    A, b, x, (rp, col, val, rhs, _), fill, keep = system(ctx, rng, shape, wrap, op)
    M = sp.csr_matrix((val, col, rp), shape=(len(rhs),) * 2)
    ref = one_pass(M, shape, rhs)[0]
    x.zero_()
    da.bicgstab2(ctx, A, b, x, tol=1e-300, tol_kind=0, max_it=1, precond=da.PRECOND_MG)
    got = x.cpu().numpy()
    assert np.max(np.abs(got - ref)) <= 1e-9 * np.max(np.abs(ref))
    A.close()


def one_pass(M, shape, rhs):
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
    cond = np.linalg.cond([[mu, nu], [nu, tau]])
    om2 = (om2 - nu * om1 / mu) / (tau - nu * nu / mu)
    om1 = (om1 - nu * om2) / mu
    return prec(y + om1 * r1 + om2 * s + alpha * u), cond
