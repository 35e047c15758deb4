"""The adaptive CSR part's row groups (k_csr.hip: csr_adaptive_kernel) at the
edges of their layout: row lengths around the 64-entry limit, empty rows,
rows too far apart for 16-bit offsets, x ranges around the staged window and
the 16-bit columns, every number of lanes per row, padding next to an infinite
x entry, and skewed row lengths, whose groups become STREAM blocks.  Tolerance: the FP32 bar of oracle.parity_report."""
import numpy as np
import pytest

from clspmv_amd import _lib as L
from clspmv_amd import matrix as M
from oracle import oracle as O
from tests.helpers import gpu_spmv

pytestmark = pytest.mark.gpu


def _rows(lens, width, seed, first=0, span=None, at=None, height=None):
    """Row i (or at[i]) holds lens[i] distinct sorted columns of
    [first, first + span), the range's two ends in the first row that has two
    entries."""
    rng = np.random.default_rng(seed)
    span = width - first if span is None else span
    r, c = [], []
    ends = False
    for i, n in enumerate(lens):
        cols = rng.choice(span, size=n, replace=False)
        if n >= 2 and not ends:
            cols = np.concatenate([[0, span - 1], rng.choice(np.arange(1, span - 1), size=n - 2, replace=False)])
            ends = True
        r.append(np.full(n, i if at is None else at[i], np.int32))
        c.append((first + np.sort(cols)).astype(np.int32))
    r, c = np.concatenate(r), np.concatenate(c)
    v = rng.standard_normal(r.size).astype(np.float32)
    return M.CooMatrix.from_arrays(r, c, v, width, len(lens) if height is None else height)


def _lens(n, lo, hi, seed):
    return np.random.default_rng(seed).integers(lo, hi + 1, n)


CASES = {
    "one entry": lambda: _rows([1], 1, 1),
    "64 and 65 and empty": lambda: _rows([64, 0, 65, 1, 0, 63, 64, 1024, 1025, 2] * 7, 3000, 2),
    "one group and one row more": lambda: _rows(_lens(513, 1, 3, 3), 4000, 3),
    "far apart rows": lambda: _rows(_lens(40, 1, 9, 4), 5000, 4, at=np.arange(40) * 5000 + np.arange(40) // 20 * 65536,
                                    height=400000),
    "x range 10240": lambda: _rows(_lens(512, 30, 40, 5), 30000, 5, first=4, span=10240),
    "x range 10241": lambda: _rows(_lens(512, 30, 40, 6), 30000, 6, first=4, span=10241),
    "x range 65536": lambda: _rows(_lens(600, 4, 12, 7), 70001, 7, first=8, span=65536),
    "x range 65537": lambda: _rows(_lens(600, 4, 12, 8), 70001, 8, first=8, span=65537),
    "x range not from a multiple of 4, to the end of x": lambda: _rows(_lens(300, 20, 30, 9), 2003, 9, first=1003),
}


@pytest.mark.parametrize("name", CASES)
def test_row_group_edges(ctx, name):
    coo = CASES[name]()
    x, y0 = M.gen_vector(coo.width, 11), M.gen_vector(coo.height, 12)
    y, info = gpu_spmv(ctx, L.FMT_CSR_VECTOR, M.coo2csr(coo), x, y0, 1)
    rep = O.parity_report(y, coo, x, y0)
    assert rep["ok"], (name, info, rep)


@pytest.mark.parametrize("rows,lo,hi", [(140001, 1, 6), (60000, 4, 9), (20001, 10, 17), (9000, 20, 33), (777, 64, 64)])
def test_lanes_per_row(ctx, rows, lo, hi):
    # 1, 2, 4, 8 and 16 lanes per row
    coo = _rows(_lens(rows, lo, hi, rows), 5000, rows)
    x, y0 = M.gen_vector(coo.width, 13), M.gen_vector(coo.height, 14)
    y, info = gpu_spmv(ctx, L.FMT_CSR_VECTOR, M.coo2csr(coo), x, y0, 1)
    rep = O.parity_report(y, coo, x, y0)
    assert rep["ok"], (info, rep)


@pytest.mark.parametrize("span", [3000, 40000, 80000])
def test_padding_keeps_infinities_out(ctx, span):
    # column 0 (what padding points at) is infinite and used by row 0 only
    lens = _lens(700, 1, 7, 21)
    lens[0] = 2
    coo = _rows(lens, span, 21)
    use0 = coo.col_id == 0
    use0[coo.row_id == 0] = False
    coo.col_id[use0] = 1
    x, y0 = M.gen_vector(coo.width, 22), M.gen_vector(coo.height, 23)
    x[0] = np.inf
    y, _ = gpu_spmv(ctx, L.FMT_CSR_VECTOR, M.coo2csr(coo), x, y0, 1)
    assert np.isinf(y[0]) and np.isfinite(y[1:]).all()


def _one_in(n, rows, rest, seed=0):
    lens = np.full(rows, rest)
    lens[seed % n::n] = 64
    return lens


def _power_law(rows, exponent, seed):
    return np.minimum(np.random.default_rng(seed).zipf(exponent, rows), 64)


def _mixed_groups():
    # even and skewed groups in turn; empty and long rows within and between
    # the skewed ones; the last group is partly filled
    lens = np.concatenate([_lens(512, 5, 9, 1), _one_in(256, 512, 1), _lens(512, 1, 3, 2), _one_in(512, 512, 2, 511),
                           _one_in(100, 77, 1)])
    lens[512 + 40:512 + 60] = 0
    lens[[512 + 3, 512 + 200, 1023, 1600, 2000, lens.size - 1]] = [65, 2000, 1024, 1025, 100, 70]
    return lens


SKEWED = {
    "one row of 64 in 512": lambda: _one_in(512, 20000, 1),
    "one row of 64 in 64": lambda: _one_in(64, 20000, 2),
    "64 first in a group of one": lambda: _one_in(600, 500, 1),
    "power law 2.5": lambda: _power_law(20011, 2.5, 1),
    "power law 1.8": lambda: _power_law(20011, 1.8, 2),
    "even and skewed groups": _mixed_groups,
}


@pytest.mark.parametrize("width", [4000, 200000])
@pytest.mark.parametrize("name", SKEWED)
def test_skewed_groups_are_not_padded(ctx, name, width):
    lens = SKEWED[name]()
    coo = _rows(lens, width, 31)
    x, y0 = M.gen_vector(coo.width, 32), M.gen_vector(coo.height, 33)
    y, info = gpu_spmv(ctx, L.FMT_CSR_VECTOR, M.coo2csr(coo), x, y0, 1)
    rep = O.parity_report(y, coo, x, y0)
    assert rep["ok"], (name, info, rep)
    # at most 1.5 times the entries and row pointers of CSR (several lanes per
    # row), and beside them 5 bytes per row and 16 per 8 rows or per block, a
    # group's descriptors and the long rows' lists
    csr = 8 * coo.nnz + 4 * (lens.size + 1)
    assert info["stored_bytes"] <= 1.5 * csr + 8 * lens.size + 1024, (name, info, csr)
