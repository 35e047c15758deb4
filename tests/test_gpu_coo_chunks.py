"""The COO kernel (k_coo.hip) at the edges of its chunks: rows that end on a
512-entry chunk boundary or reach 63, 64 and 65 entries past it, rows over
several chunks, chunks of single-entry rows, a last chunk of one entry, and x
ranges around the ones staged in LDS for both workgroup sizes.  The part and
the allocation-free entry point give the same bits.  Tolerance: the FP32 bar
of oracle.parity_report."""
import numpy as np
import pytest

from clspmv_amd import matrix as M
from oracle import oracle as O
from tests.test_zz_no_alloc import _noalloc, _part

pytestmark = pytest.mark.gpu


def _coo(lens, width, seed, first=0, span=None):
    lens = np.asarray(lens)
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(lens.size), lens).astype(np.int32)
    c = (first + rng.integers(0, width - first if span is None else span, r.size)).astype(np.int32)
    if span is not None:  # both ends of the range in every chunk
        c[::512], c[1::512] = first, first + span - 1
    v = rng.standard_normal(r.size).astype(np.float32)
    return M.CooMatrix.from_arrays(r, c, v, width, int(lens.size))


CASES = {
    "one entry": lambda: _coo([1], 1, 1),
    "rows end on chunk boundaries": lambda: _coo([512, 256, 256, 512, 1], 900, 2),
    "single entry rows, last chunk of one": lambda: _coo(np.ones(1025, int), 700, 3),
    "511 breaks and 512": lambda: _coo(np.r_[2, np.ones(511, int), np.ones(600, int)], 700, 4),
    "63 past": lambda: _coo([475, 100, 400, 7, 300], 900, 5),
    "64 past": lambda: _coo([476, 100, 400, 7, 300], 900, 6),
    "65 past": lambda: _coo([477, 100, 400, 7, 300], 900, 7),
    "64 past, at the end": lambda: _coo([476, 100], 900, 8),
    "65 past, at the end": lambda: _coo([477, 100], 900, 9),
    "one row over chunks": lambda: _coo([300, 2000, 3, 5000], 900, 10),
    "whole chunks of one row, then 64 and 65": lambda: _coo([512 * 3 + 64, 448, 512 * 2 + 65, 10], 900, 11),
    "empty rows": lambda: _coo([0, 0, 5, 0, 700, 0, 0, 9, 0] * 40, 900, 12),
    "x range 3040": lambda: _coo(np.full(1000, 9), 9000, 13, first=4, span=3040),
    "x range 3041": lambda: _coo(np.full(1000, 9), 9000, 14, first=4, span=3041),
    "x range 6080, 512 threads": lambda: _coo(np.full(120000, 9), 9000, 15, first=4, span=6080),
    "x range 6081, 512 threads": lambda: _coo(np.full(120000, 9), 9000, 16, first=4, span=6081),
    "x range to the end of x": lambda: _coo(np.full(500, 11), 2003, 17, first=1003, span=1000),
}


@pytest.mark.parametrize("name", CASES)
def test_chunk_edges(ctx, name):
    coo = CASES[name]()
    x, y0 = M.gen_vector(coo.width, 21), M.gen_vector(coo.height, 22)
    y = _part(ctx, coo, x, y0)
    rep = O.parity_report(y, coo, x, y0)
    assert rep["ok"], (name, rep)
    assert np.array_equal(y.view(np.uint32), _noalloc(ctx, coo, x, y0).view(np.uint32)), name
