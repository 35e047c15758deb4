"""power_iterate on narrow-band matrices (k_dia.hip: dia_steps_kernel, several
iterations per launch) takes bitwise the steps of the host-driven loop
(do_spmv, then cpy_vector_from_gpu): diagonal counts 1..8, reaches around the
limits of its range, matrices smaller than a workgroup's range, iteration
counts around the steps of a launch; x ends as a copy of y."""
import numpy as np
import pytest

from clspmv_amd import cocktail as CK
from clspmv_amd import matrix as M

pytestmark = pytest.mark.gpu


def _band(n, offsets, seed):
    rng = np.random.default_rng(seed)
    r, c = [], []
    for o in offsets:
        rows = np.arange(max(0, -o), min(n, n - o))
        r.append(rows)
        c.append(rows + o)
    r, c = np.concatenate(r), np.concatenate(c)
    v = (rng.standard_normal(r.size) * (0.3 / len(offsets))).astype(np.float32)
    order = np.lexsort((c, r))
    return M.CooMatrix.from_arrays(r[order].astype(np.int32), c[order].astype(np.int32), v[order], n, n)


CASES = [
    (1, [0]), (5, [-1, 0, 1]), (1000, [3]), (1023, [-2, 0]), (1025, [-40, 0, 40]), (4097, [-64, -1, 0, 1]),
    (40000, [-200, -1, 0, 1, 200]), (65537, [0, 1, 2, 3, 4, 5]), (70001, [-511, -3, -1, 0, 1, 3, 900]),
    (90001, [-700, -2, -1, 0, 1, 2, 699, 700]), (300000, [-4000, 0, 4000]), (300000, [-5000, 0, 5000]),
    (12000, [-6000, 0, 6000]),
]


@pytest.mark.parametrize("tables", ["mi355x", "reference"])
@pytest.mark.parametrize("n,offsets", CASES, ids=[f"{n}x{len(o)}" for n, o in CASES])
def test_steps_equal_host_loop(ctx, tables, n, offsets):
    coo = _band(n, offsets, n)
    t = CK.BenchTables(CK.MI355X_TABLES if tables == "mi355x" else CK.REFERENCE_TABLES)
    mat = CK.analyze_matrix(coo, t)
    x, y0 = M.gen_vector(n, 41), M.gen_vector(n, 42)
    for k in (1, 2, 3, 13, 40):
        a, b = CK.GpuCocktail(ctx, mat, x, y0), CK.GpuCocktail(ctx, mat, x, y0)
        ya, yb = CK.power_iterate(ctx, a, k), CK.power_iterate_host(ctx, b, k)
        assert np.isfinite(yb).all()
        assert np.array_equal(ya.view(np.uint32), yb.view(np.uint32)), (k, [p["kernel"] for p in a.part_infos()])
        # one more product from x = y on both sides shows x too
        a.do_spmv(1)
        b.do_spmv(1)
        assert np.array_equal(a.result_to_cpu().view(np.uint32), b.result_to_cpu().view(np.uint32)), k
        a.free()
        b.free()
