"""The CG's SpMV on the packed boundary stream in every form, at sizes below the one
from which the solver reads it (timing variant 13): y equals the oracle's bit for
bit, as it does on the full boundary values (variant 1)."""
import numpy as np
import pytest

from conftest import bits_equal, pack_groups, pack_plan, wpack_groups, wpack_plan

pytestmark = pytest.mark.gpu

# what one (block, plane, lower slot) group is set to, so that the stream needs the
# form: multiples of one quantum spanning `span` quanta (None: the values as they are)
PLANTS = {"all10": None, "all12": (9, 4093), "all16": (9, 4094), "cube10+near22": (12, 2 ** 22 - 3),
          "cube12+near24": (12, 2 ** 24 - 3), "cube16+near32": (10, 2 ** 30)}


def planted(oracle, dims, slot, span, block):
    """The box problem's matrix with the boundary entries of one group, and their
    mirrors, replaced."""
    A = oracle.build_problem(*dims)["A"]
    ro, cols, v = A.row_offsets, A.cols, A.vals.copy()
    gx, gy, gz = (d + 1 for d in dims)
    bx, by, z = block
    dz, dy, dx = slot // 9 - 1, (slot // 3) % 3 - 1, slot % 3 - 1
    pos, mir = [], []
    for iy in range(16 * by, min(16 * by + 16, gy)):
        for ix in range(16 * bx, min(16 * bx + 16, gx)):
            cx, cy, cz = ix + dx, iy + dy, z + dz
            if not (0 <= cx < gx and 0 <= cy < gy and 0 <= cz < gz) or \
                    (cx // 16 == ix // 16 and cy // 16 == iy // 16):
                continue
            r, c = ix + gx * (iy + gy * z), cx + gx * (cy + gy * cz)
            pos.append(ro[r] + int(np.searchsorted(cols[ro[r]:ro[r + 1]], c)))
            mir.append(ro[c] + int(np.searchsorted(cols[ro[c]:ro[c + 1]], r)))
    base = next((a for a in v[pos] if a != 0.0), np.float64(-0.01)).view(np.int64)
    bits = base + np.random.default_rng(span).integers(0, span + 1, len(pos))
    bits[0], bits[-1] = base, base + span
    v[pos] = v[mir] = bits.view(np.float64)
    return oracle.CSR(np.arange(A.nrows, dtype=np.int32), ro, cols, v)


# blocks at the x and y edges that are partial, down to one column or line of nodes;
# few planes and many (several z chunks); values that are dyadic
@pytest.mark.parametrize("dims", [(20, 18, 6), (34, 33, 3), (17, 16, 130), (32, 16, 64)])
@pytest.mark.parametrize("form", sorted(PLANTS))
def test_cg_spmv_on_the_packed_boundary_stream(oracle_mod, form, dims):
    import minife_amd as m
    print("case boundary stream", form, dims, flush=True)
    if PLANTS[form]:
        slot, span = PLANTS[form]
        block = (1, 0, dims[2] // 2) if slot in (9, 12) else (0, 1, dims[2] // 2)
        Ao = planted(oracle_mod, dims, slot, span, block)
    else:
        Ao = oracle_mod.build_problem(*dims)["A"]
    assert wpack_plan(wpack_groups(Ao, dims)) == form
    ctx = m.Context(0)
    n = Ao.nrows
    A = m.CSRMatrix.from_host(Ao.row_offsets, Ao.cols, Ao.vals, ctx=ctx)
    mesh = m.simple_mesh_description([0, dims[0], 0, dims[1], 0, dims[2]])
    # no conductivity: the loop takes the structure for the box's and adds +0.0
    kappa = m.Vector(dims[0] * dims[1] * dims[2], ctx)
    m.perform_element_loop(mesh, mesh.global_box, A, m.Vector(n, ctx), kappa=kappa)
    info = m.spmv_plan(A)
    assert info["pack"] == pack_plan(pack_groups(Ao, dims)) and info["wpack"] == form
    xh = np.random.default_rng(sum(dims)).standard_normal(n)
    want = oracle_mod.matvec(Ao, xh)
    x, y = m.Vector.from_numpy(xh, ctx), m.Vector(n, ctx)
    for variant in (13, 1):
        y.fill(7.0)
        m.time_matvec(A, x, y, variant=variant, reps=1)
        assert bits_equal(y.to_numpy(), want), variant
    ctx.close()
