"""Mixed-precision DIA whose diagonals come in threes of consecutive offsets
(k_mixed.hip: dia_mixed_kernel<CODEC, true>) gives bitwise the sums of the
one-by-one loop: the same matrix with one more, all-zero diagonal takes that
loop.  Sizes around the lane's 4 rows, the wave's 256 and the workgroup's
1024, counts of triples around the 3 in flight, rectangular matrices, x short
of and beyond the band."""
import ctypes as C
from types import SimpleNamespace

import numpy as np
import pytest

from clspmv_amd import _lib as L
from clspmv_amd import matrix as M

pytestmark = pytest.mark.gpu


def _dia(rows, cols, offsets, seed, zero=None):
    """The band as a DIA matrix (filled here: the COO converter refuses
    padding as large as some of these); `zero` adds an all-zero diagonal."""
    offs = sorted(offsets + ([] if zero is None else [zero]))
    length = (rows + 255) // 256 * 256
    data = np.zeros((len(offs), length), np.float32)
    rng = np.random.default_rng(seed)
    for o in offsets:
        i = np.arange(max(0, -o), min(rows, cols - o))
        data[offs.index(o), i] = rng.standard_normal(i.size)
    offs = np.array(offs, np.int32)
    s = L.Dia(L.MatInfo(cols, rows, int(np.count_nonzero(data))), offs.size, rows, length,
              offs.ctypes.data_as(C.POINTER(C.c_int)), data.ctypes.data_as(C.POINTER(C.c_float)))
    return SimpleNamespace(s=s, keep=(offs, data))


def _threes(*starts):
    return [s + j for s in starts for j in range(3)]


CASES = [
    (3, 3, [-1, 0, 1], 2), (5, 9, _threes(0, 3), 7), (255, 255, _threes(-1), 5), (1023, 1025, _threes(-17, -1, 15), 30),
    (1024, 1024, _threes(-33, -1, 31, 40), -40), (1025, 900, _threes(-200, -1, 99), 300),
    (4097, 4097, _threes(-70, -67, -64, -1, 62, 65, 68), 200), (2049, 70000, _threes(0, 500, 60000), 1000),
    (30000, 30000, _threes(-931, -901, -871, -31, -1, 29, 869, 899, 929), 2000),
]


@pytest.mark.parametrize("codec", [L.VAL_FP16_ROW, L.VAL_FP8_SLICE, L.VAL_I16_ROW])
@pytest.mark.parametrize("rows,cols,offsets,zero", CASES, ids=[f"{c[0]}x{c[1]}x{len(c[2])}" for c in CASES])
def test_triples_equal_single_diagonals(ctx, codec, rows, cols, offsets, zero):
    x, y0 = M.gen_vector(cols, 51), M.gen_vector(rows, 52)
    out = []
    for z in (None, zero):
        dia = _dia(rows, cols, offsets, rows + cols, z)
        part = M.MixedPart(ctx, L.FMT_DIA, dia, codec)
        dx, dy = M.DeviceArray.from_numpy(ctx, x), M.DeviceArray.from_numpy(ctx, y0)
        part.spmv(dx, dy, 1)
        out.append(dy.download())
        for p in (dx, dy, part):
            p.free()
    assert np.isfinite(out[1]).all() and not np.array_equal(out[1], y0)
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
