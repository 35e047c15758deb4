"""The regrouped BCSR kernel (k_block.hip: bcsr_group_kernel) at its edges:
every block shape, one to sixteen lanes per block row, ragged and empty block
rows, a width that no block column divides, one group and one row more, and
the parts that keep the plain kernel (a block row far longer than the rest, or
skewed rows that regrouping would pad); padding next to an infinite x entry.  Tolerance: the FP32 bar of
oracle.parity_report."""
import numpy as np
import pytest

from clspmv_amd import _lib as L
from clspmv_amd import matrix as M
from oracle import oracle as O
from tests.helpers import gpu_spmv

pytestmark = pytest.mark.gpu


def _coo(lens, bh, bw, width, seed):
    """Block row i holds lens[i] full bh x bw blocks (columns a multiple of 4
    apart, clipped at the matrix' edge)."""
    rng = np.random.default_rng(seed)
    slots = (width + bw - 1) // bw
    rows, cols = [], []
    for i, n in enumerate(lens):
        for b in rng.choice(slots, size=min(n, slots), replace=False):
            r, c = np.meshgrid(np.arange(bh), np.arange(bw), indexing="ij")
            keep = b * bw + c < width
            rows.append((i * bh + r)[keep])
            cols.append((b * bw + c)[keep])
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((cols, rows))
    vals = rng.standard_normal(rows.size).astype(np.float32)
    return M.CooMatrix.from_arrays(rows[order].astype(np.int32), cols[order].astype(np.int32), vals, width,
                                   len(lens) * bh)


def _check(ctx, coo, bw, bh, kernel):
    x, y0 = M.gen_vector(coo.width, 31), M.gen_vector(coo.height, 32)
    y, info = gpu_spmv(ctx, L.FMT_BCSR, M.coo2b4csr(coo, bw, bh), x, y0)
    rep = O.parity_report(y, coo, x, y0)
    assert rep["ok"], (info, rep)
    assert kernel in info["kernel"], info
    return info


@pytest.mark.parametrize("width", [804, 803])
@pytest.mark.parametrize("bh,bw", [(h, w) for h in (1, 2, 4, 8) for w in (4, 8)])
def test_block_shapes(ctx, bh, bw, width):
    lens = np.random.default_rng(bh * 10 + bw).integers(0, 9, 257)
    _check(ctx, _coo(lens, bh, bw, width, bh + bw), bw, bh, "_G")


@pytest.mark.parametrize("rows,lo,hi,lanes", [(140001, 1, 3, 1), (40000, 4, 6, 2), (5000, 8, 13, 4), (129, 17, 30, 8)])
def test_lanes_per_block_row(ctx, rows, lo, hi, lanes):
    lens = np.random.default_rng(rows).integers(lo, hi + 1, rows)
    _check(ctx, _coo(lens, 1, 4, 1000, rows), 4, 1, f"_G{lanes}")


@pytest.mark.parametrize("width", [804, 803])
@pytest.mark.parametrize("bh,bw", [(8, 8), (8, 4), (4, 8)])
def test_sixteen_lanes_per_block_row(ctx, bh, bw, width):
    # blocks of eight float4 and more only: a block row feeds its lanes one each
    lens = np.random.default_rng(bh * 10 + bw).integers(16, 34, 130)
    _check(ctx, _coo(lens, bh, bw, width, bh + bw), bw, bh, "_G16")


def test_one_long_block_row_keeps_the_plain_kernel(ctx):
    _check(ctx, _coo([3] * 200 + [400] + [2] * 100, 4, 4, 4000, 7), 4, 4, "_L")


@pytest.mark.parametrize("every,rest,kernel", [(256, 1, "_L"), (64, 3, "_L"), (16, 3, "_L"), (3, 40, "_G")])
def test_skewed_block_rows_are_not_padded(ctx, every, rest, kernel):
    lens = np.full(2000, rest)
    lens[5::every] = 64
    info = _check(ctx, _coo(lens, 4, 4, 4000, every), 4, 4, kernel)
    # 64 bytes of values and 4 of column a block, 1.5 times the blocks at most
    # but for the last group's; a few bytes a row beside them
    assert info["stored_bytes"] <= 1.5 * 68 * lens.sum() + 16 * lens.size + 68 * 256 * 64 / 4


def test_padding_keeps_infinities_out(ctx):
    # block column 0 (what padding points at) is infinite, used by row 0 only
    coo = _coo(np.random.default_rng(9).integers(1, 8, 300), 4, 4, 2000, 9)
    use0 = (coo.col_id < 4) & (coo.row_id >= 4)
    keep = ~use0
    coo = M.CooMatrix.from_arrays(np.r_[0, coo.row_id[keep]], np.r_[0, coo.col_id[keep]], np.r_[1.0, coo.data[keep]],
                                  coo.width, coo.height)
    x, y0 = M.gen_vector(coo.width, 31), M.gen_vector(coo.height, 32)
    x[0] = np.inf
    y, _ = gpu_spmv(ctx, L.FMT_BCSR, M.coo2b4csr(coo, 4, 4), x, y0)
    assert not np.isfinite(y[0]) and np.isfinite(y[4:]).all()
