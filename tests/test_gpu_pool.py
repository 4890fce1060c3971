"""Device memory kept between matrices: a matrix built in memory that earlier
ones gave back, of the same and of other sizes, and from two contexts in two
threads, equals one built first (structure, values, b, and a CG's x)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _build(m, ctx, dims):
    mesh, A, b = m.build_problem(*dims, ctx=ctx)
    x = m.Vector(A.nrows, ctx)
    m.cg_solve(A, b, x, max_iter=30)
    h = A.to_host()
    out = [h["row_offsets"], h["cols"], h["vals"].view(np.uint64), b.to_numpy().view(np.uint64),
           x.to_numpy().view(np.uint64)]
    for o in (A, b, x):
        o.close()
    return out


@pytest.mark.parametrize("sizes", [((9, 8, 7), (9, 8, 7), (9, 8, 8), (9, 8, 7)),
                                   ((40, 33, 29), (1, 1, 1), (40, 33, 30), (40, 33, 29))])
def test_matrices_in_kept_memory(sizes):
    import minife_amd as m
    first = {}
    ctx = m.Context(0)
    for dims in sizes:
        print("case pool", dims, flush=True)
        fresh = m.Context(0)
        want = first.setdefault(dims, _build(m, fresh, dims))
        fresh.close()
        for a, w in zip(_build(m, ctx, dims), want):
            assert np.array_equal(a, w)
    got = {}

    def work(k):
        c = m.Context(0)
        got[k] = [_build(m, c, dims) for dims in sizes]
        c.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        for dims, out in zip(sizes, got[k]):
            for a, w in zip(out, first[dims]):
                assert np.array_equal(a, w)
    ctx.close()
