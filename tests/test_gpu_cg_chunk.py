"""The captured chunk of CG iterations (more rows than are launched one by one)
is replayed only for the SpMV it holds: a matrix whose values change between two
solves into the same vectors may get another packed form in the same memory."""
import numpy as np
import pytest

from conftest import bits_equal

pytestmark = pytest.mark.gpu


def test_solve_after_the_packed_form_changed():
    """The first conductivity needs 16-bit fields; with 4096 more everywhere the
    sum's values vary by a few last places only and 12-bit fields (six words per
    row instead of seven) go into the words that are there.  The second solve's
    x, iterations and norm are those of a matrix that was never solved before."""
    import minife_amd as m
    dims = (230, 100, 64)
    print("case captured chunk, packed form changed", dims, flush=True)
    ctx = m.Context(0)
    ne = dims[0] * dims[1] * dims[2]
    k1 = 1.0 + np.random.default_rng(0).integers(0, 2 ** 13, ne) * 2.0 ** -52
    kappas = [m.Vector.from_numpy(k, ctx) for k in (k1, np.full(ne, 4096.0))]
    mesh = m.simple_mesh_description([0, dims[0], 0, dims[1], 0, dims[2]])

    def matrix():
        A = m.CSRMatrix(ctx)
        assert m.generate_matrix_structure(mesh, A) == 0
        m.make_local_matrix(A)
        return A, m.Vector(A.nrows, ctx)

    def add(A, b, kappa):
        m.assemble_FE_data(mesh, A, b, kappa=kappa)
        for value, rows in ((0.0, mesh.bc_rows_0), (1.0, mesh.bc_rows_1)):
            m.impose_dirichlet(value, A, b, dims[0] + 1, dims[1] + 1, dims[2] + 1, rows)

    def solve(A, b, x):
        x.fill(0.0)
        r = m.cg_solve(A, b, x, max_iter=60, tolerance=0.0)
        return x.to_numpy(), r.num_iters, r.normr

    A, b = matrix()
    x = m.Vector(A.nrows, ctx)
    add(A, b, kappas[0])
    solve(A, b, x)
    form1 = m.spmv_plan(A)["pack"]
    add(A, b, kappas[1])
    got = solve(A, b, x)
    form2 = m.spmv_plan(A)["pack"]
    assert m.pack_row_layout(form2)[0] <= m.pack_row_layout(form1)[0] and form1 != form2
    A2, b2 = matrix()
    for k in kappas:
        add(A2, b2, k)
    want = solve(A2, b2, m.Vector(A2.nrows, ctx))
    assert got[1:] == want[1:]
    assert bits_equal(got[0], want[0])
    ctx.close()
