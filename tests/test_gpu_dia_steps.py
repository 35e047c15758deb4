"""power_iterate on narrow-band matrices (k_dia.hip: dia_steps_kernel, several
iterations per launch) takes bitwise the steps of the host-driven loop
(do_spmv, then cpy_vector_from_gpu): 1 to 8 diagonals, reaches from 0 to the
limits of its range, matrices smaller than a workgroup's range, every number of
row slots, iteration counts around the steps of a launch; x ends as a copy of
y.  Each matrix is one DIA part by itself, of both kernels (one row per lane,
four), and the launches that the call takes are looked at."""
import ctypes as C

import numpy as np
import pytest

from clspmv_amd import _lib as L
from clspmv_amd import cocktail as CK
from clspmv_amd import matrix as M

pytestmark = pytest.mark.gpu


def _dia(n, offsets):
    """The band as a DIA matrix (filled here: the COO converter refuses
    padding as large as some of these)."""
    rng = np.random.default_rng(n)
    length = (n + 31) // 32 * 32
    data = np.zeros((len(offsets), length), np.float32)
    for d, o in enumerate(offsets):
        i = np.arange(max(0, -o), min(n, n - o))
        data[d, i] = rng.standard_normal(i.size) * (0.3 / len(offsets))
    offs = np.array(offsets, np.int32)
    s = L.Dia(L.MatInfo(n, n, int(np.count_nonzero(data))), offs.size, n, length,
              offs.ctypes.data_as(C.POINTER(C.c_int)), data.ctypes.data_as(C.POINTER(C.c_float)))
    return s, (offs, data)


# several iterations per launch; the row slots of a thread in the last column
CASES = [
    (1, [0], 2), (2, [0, 1], 2), (5, [-1, 0, 1], 2), (255, [-3, 0, 2, 254], 2), (1000, [3], 2), (1023, [-2, 0], 2),
    (1025, [-40, 0, 40], 2), (4097, [-64, -1, 0, 1], 2), (40000, [-200, -1, 0, 1, 200], 4),
    (65537, [0, 1, 2, 3, 4, 5], 2), (70001, [-511, -3, -1, 0, 1, 3, 900], 8),
    (90001, [-700, -2, -1, 0, 1, 2, 699, 700], 8), (300000, [0], 2), (300000, [-2000, 0, 2000], 10),
    (700000, [-1000, -3, -1, 0, 1, 2, 5, 999], 10),
]
# one by one: the range does not fit, or costs more than it saves
ONE_BY_ONE = [
    (12000, [-6000, 0, 6000]), (300000, [-4000, 0, 4000]), (300000, [-1500, -2, -1, 0, 1, 2, 3, 1500]),
    (50001, list(range(-4, 5))),
]


def _compare(ctx, n, offsets, method, counts):
    # a partition of one DIA part
    dia, _keep = _dia(n, offsets)
    mat = CK.CocktailMatrix()
    mat.s.ifusedia, mat.s.dia_meth_num, mat.s.dia = 1, method, dia
    mat.s.mat_width, mat.s.mat_height, mat.s.mat_nnz = n, n, dia.matinfo.nnz
    x, y0 = M.gen_vector(n, 41), M.gen_vector(n, 42)
    launches = {}
    try:
        for k in counts:
            a, b = CK.GpuCocktail(ctx, mat, x, y0), CK.GpuCocktail(ctx, mat, x, y0)
            info = a.part_infos()
            assert [p["kernel"] for p in info] == ["dia_row4" if method == 1 else "dia_row"]
            launches[k] = L.lib().clspmv_power_iterate_launches(a.h, k)
            ya, yb = CK.power_iterate(ctx, a, k), CK.power_iterate_host(ctx, b, k)
            assert np.isfinite(yb).all()
            assert np.array_equal(ya.view(np.uint32), yb.view(np.uint32)), k
            # one more product from x = y on both sides shows x too
            a.do_spmv(1)
            b.do_spmv(1)
            assert np.array_equal(a.result_to_cpu().view(np.uint32), b.result_to_cpu().view(np.uint32)), k
            a.free()
            b.free()
    finally:
        mat.s.ifusedia, mat.s.dia = 0, L.Dia()  # the arrays are numpy's
    return launches


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("n,offsets,slots", CASES, ids=[f"{n}x{len(o)}" for n, o, _ in CASES])
def test_steps_equal_host_loop(ctx, method, n, offsets, slots):
    launches = _compare(ctx, n, offsets, method, (1, 2, 3, 13, 40))
    assert launches[1] == 0 and 2 <= launches[40] < 40, launches
    rows = min(n, (n + 255) // 256 + 2 * -(-40 // launches[40]) * max(abs(o) for o in offsets))
    assert next(u for u in (2, 4, 8, 10) if rows <= 1024 * u) == slots


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("n,offsets", ONE_BY_ONE, ids=[f"{n}x{len(o)}" for n, o in ONE_BY_ONE])
def test_one_by_one_where_that_is_faster(ctx, method, n, offsets):
    launches = _compare(ctx, n, offsets, method, (1, 2, 13))
    assert not any(launches.values()), launches
