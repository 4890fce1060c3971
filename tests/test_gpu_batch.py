"""GPU batched boxes: many independent miniFE problems assembled and solved by
FP64 CG in one cooperative persistent launch.

Checks: every problem's assembled operator (structure, values, right-hand
side) is bit-identical to the oracle's single-box assembly; the solutions
reach the requested residual when it is recomputed on the CPU from the
downloaded operator; iteration counts match the oracle's serial CG to within
the rounding of the tree-reduced dots; solved to 1e-13, each box equals the
oracle's serial single-box CG to 1e-13 within 1e-11 normwise; the 64-box
workload (sides uniform on [16, 96], seed 0) converges in every box to 1e-10
(and 1e-13, three boxes checked against the oracle's single solves).
"""
import sys

import numpy as np
import pytest

from conftest import bits_equal

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def mfe():
    import minife_amd
    minife_amd.lib()
    return minife_amd


def check_problem(mfe, oracle_mod, B, p, dims, rel_tol, exact=True):
    got = B.download(p)
    P = oracle_mod.build_problem(*dims)
    A = P["A"]
    assert np.array_equal(got["row_offsets"], A.row_offsets), dims
    assert np.array_equal(got["cols"], A.cols), dims
    if exact:
        assert bits_equal(got["vals"], A.vals), dims
        assert bits_equal(got["b"], P["b"]), dims
    b = P["b"]
    res = b - oracle_mod.matvec(A, got["x"])
    true_rel = float(np.linalg.norm(res) / np.linalg.norm(b))
    assert true_rel <= 4 * rel_tol, (dims, true_rel)
    return P, got, true_rel


def test_small_batch_matches_oracle(mfe, oracle_mod):
    dims = [(1, 1, 1), (2, 3, 4), (17, 3, 5), (10, 10, 10), (3, 4, 5), (5, 1, 2), (1, 9, 1)]
    say(f"batch small {dims}")
    B = mfe.Batch(dims)
    say(f"  info {B.info()}")
    out = B.solve(max_iter=2000, rel_tol=1e-10)
    assert out["status"] == mfe.MFE_OK
    say(f"  iters {out['iters'].tolist()} rel {out['rel_residual'].max():.2e}")
    for p, d in enumerate(dims):
        P, got, true_rel = check_problem(mfe, oracle_mod, B, p, d, 1e-10)
        bn = float(np.sqrt(oracle_mod.dot(P["b"], P["b"])))
        r = oracle_mod.cg_solve(P["A"], P["b"], max_iter=2000, tol=1e-10 * bn)
        assert abs(int(out["iters"][p]) - r["num_iters"]) <= 2, (d, out["iters"][p], r["num_iters"])
        xs = r["x"]
        assert np.max(np.abs(got["x"] - xs)) <= 1e-8 * max(1.0, np.max(np.abs(xs)))
    # a second solve of the same batch gives the same bits (deterministic)
    x0 = B.download(3, matrix=False)["x"]
    B.solve(max_iter=2000, rel_tol=1e-10)
    assert bits_equal(B.download(3, matrix=False)["x"], x0)
    # the 10^3 box verifies against the analytic solution like the driver
    assert oracle_mod.verify_solution(10, 10, 10, x0)[0] == 0
    # every box solved to 1e-13 equals the oracle's single-box solve to 1e-13
    # normwise within 1e-11
    out = B.solve(max_iter=5000, rel_tol=1e-13)
    assert out["status"] == mfe.MFE_OK
    for p, d in enumerate(dims):
        check_against_single_solve(oracle_mod, B, p, d)


def check_against_single_solve(oracle_mod, B, p, dims, rel=1e-13, bound=1e-11):
    """Box p (solved by the batch to `rel`) against the oracle's serial CG of
    the same box to `rel`: ||x_batch - x_ref|| <= bound ||x_ref||."""
    P = oracle_mod.build_problem(*dims)
    bn = float(np.sqrt(oracle_mod.dot(P["b"], P["b"])))
    ref = oracle_mod.cg_solve(P["A"], P["b"], max_iter=20000, tol=rel * bn)["x"]
    x = B.download(p, matrix=False)["x"]
    err = float(np.linalg.norm(x - ref) / np.linalg.norm(ref))
    assert err <= bound, (dims, err)
    return err


def test_batch_max_iter_and_zero_iterations(mfe, oracle_mod):
    say("batch max_iter")
    B = mfe.Batch([(6, 5, 4), (3, 3, 3)])
    out = B.solve(max_iter=3, rel_tol=1e-12)
    assert out["iters"].tolist() == [3, 3]
    out = B.solve(max_iter=0, rel_tol=1e-12)
    assert out["iters"].tolist() == [0, 0]
    assert np.all(B.download(0, matrix=False)["x"] == 0.0)


def test_batch_64_boxes(mfe, oracle_mod):
    from minife_amd.workloads import batch_boxes
    dims = batch_boxes(0)
    say(f"batch 64: sides {dims.min()}..{dims.max()}")
    B = mfe.Batch(dims)
    inf = B.info()
    say(f"  info {inf}")
    first = B.solve(max_iter=5000, rel_tol=1e-10)  # model-balanced
    out = B.solve(max_iter=5000, rel_tol=1e-10)  # balanced by the first solve's iterations
    ps = out["problem_seconds"]
    say(f"  first {first['seconds']:.3f} s (problems {first['problem_seconds'].min():.3f}.."
        f"{first['problem_seconds'].max():.3f}), rebalanced {out['seconds']:.3f} s "
        f"({ps.min():.3f}..{ps.max():.3f}); iters {out['iters'].min()}..{out['iters'].max()}, "
        f"sum {int(out['iters'].sum())}")
    assert out["status"] == mfe.MFE_OK
    assert np.all(out["rel_residual"] <= 1e-10)
    # a new division changes the dots' summation order, hence the rounding; CG
    # near its stopping test can then take a few iterations more or fewer
    d = np.abs(first["iters"].astype(int) - out["iters"].astype(int))
    assert np.all(d <= np.maximum(2, 0.05 * first["iters"])), d
    vol = dims.prod(axis=1)
    picks = {int(np.argmin(vol)), int(np.argmax(vol)), 7}
    for p in sorted(picks):
        _, _, tr = check_problem(mfe, oracle_mod, B, p, tuple(int(v) for v in dims[p]), 1e-10)
        say(f"  problem {p} {tuple(dims[p])}: bit-exact operator, true rel residual {tr:.2e}")
    out = B.solve(max_iter=20000, rel_tol=1e-13)
    assert out["status"] == mfe.MFE_OK and np.all(out["rel_residual"] <= 1e-13)
    for p in sorted(picks):
        err = check_against_single_solve(oracle_mod, B, p, tuple(int(v) for v in dims[p]))
        say(f"  problem {p} at 1e-13: |x - x_oracle|/|x_oracle| = {err:.2e}")


# No interior node, one, a tile's edge (256 rows), slots of 10 bits, cubes (the
# near-zero slots up to 22), analytically zero edge neighbours and 2a^2 = b^2 + c^2
# (20 bits).
@pytest.mark.parametrize("dims", [(1, 1, 40), (2, 2, 2), (7, 7, 3), (24, 20, 31), (33, 33, 33),
                                  (48, 48, 96), (75, 15, 105)])
def test_batch_packed_values_are_exact(mfe, monkeypatch, dims):
    """The CG on packed stencil values gives the bits of the CG on the values
    themselves (the partial sums of both are grouped alike)."""
    say(f"batch packed {dims}")
    same_bits_without_packing(mfe, monkeypatch, [dims, (5, 4, 3)])


def test_batch_packed_values_are_exact_two_rows_per_thread(mfe, monkeypatch):
    """The same where the launches are large enough for two rows per thread."""
    boxes = [(128, 128, 128), (48, 48, 96), (75, 15, 105), (2, 2, 2), (1, 1, 40), (31, 30, 17)]
    say(f"batch packed {boxes}")
    same_bits_without_packing(mfe, monkeypatch, boxes)


def same_bits_without_packing(mfe, monkeypatch, boxes):
    out, xs = [], []
    for pack in ("1", "0"):
        monkeypatch.setenv("MINIFE_BATCH_PACK", pack)
        B = mfe.Batch(boxes)
        out.append(B.solve(max_iter=60, rel_tol=1e-12))
        xs.append([B.download(p, matrix=False)["x"] for p in range(len(boxes))])
    assert out[0]["iters"].tolist() == out[1]["iters"].tolist()
    assert out[0]["iters"][0] > 0
    for a, b in zip(*xs):
        assert bits_equal(a, b)
