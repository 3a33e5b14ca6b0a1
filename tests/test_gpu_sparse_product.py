"""The two kernels of the handle-level products, C tile by C tile (few tile pairs in each C tile) and by
windows of C: every entry point against the CPU oracle on both sides of the rule between them, at
the edges of runs, waves and words."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def random_tiles(ns, occupied, seed):
    """An ns x ns grid with about that share of occupied tiles: one bit, a few, half of them, all."""
    rng = np.random.default_rng(seed)
    n = max(1, int(round(occupied * ns * ns)))
    pos = np.unique(rng.integers(0, ns * ns, n)) if occupied < 1 else np.arange(ns * ns)
    row, col = (pos // ns).astype(np.uint32), (pos % ns).astype(np.uint32)
    data = np.zeros((len(pos), 64), np.uint64)
    bits = rng.choice([1, 1, 1, 2, 5, 18, 64, 65], len(pos))
    for k in range(18):
        t = np.nonzero((bits > k) & (bits <= 18))[0]
        np.bitwise_or.at(data, (t, rng.integers(0, 64, len(t))), np.uint64(1) << rng.integers(0, 64, len(t)).astype(np.uint64))
    half = bits == 64
    data[half] = rng.integers(0, 1 << 64, (int(half.sum()), 64), dtype=np.uint64)
    data[bits == 65] = ~np.uint64(0)
    off = np.zeros(ns + 1, np.uint32)
    np.add.at(off, row.astype(np.int64) + 1, 1)
    return ns, np.cumsum(off).astype(np.uint32), row, col, data


def want_product(a, bt):
    _, c_row, c_col, tp = O.tile_symbolic(a[0], a[1], a[3], bt[1], bt[3])
    return c_row, c_col, O.tile_numeric(a[0], a[1:], bt[1:], c_row, c_col), tp


# Pairs per C tile from 1 to 13 (12: the last by tiles); 153 K C tiles: runs of several; the widest grid
# with bitmaps and the first without.
@pytest.mark.parametrize("ns,occupied", [(1, 1.0), (2, 1.0), (12, 1.0), (13, 1.0), (17, 0.1), (63, 0.2), (65, 0.45),
                                         (300, 0.02), (4096, 0.0015), (16384, 2e-5), (16385, 2e-5)])
@pytest.mark.parametrize("prepare", [False, True])
def test_both_kernels_match_oracle(ctx, ns, occupied, prepare):
    import matrixgraph_amd as M

    ah, bh = random_tiles(ns, occupied, 1), random_tiles(ns, occupied, 2)
    c_row, c_col, c_data, tp = want_product(ah, bh)
    a, bt = (M.TiledMatrix.upload(ctx, M.HostTiledMatrix(*h)) for h in (ah, bh))
    if prepare:
        a.prepare_operand()
        bt.prepare_operand()
    c, st = M.multiply_symbolic(ctx, a, bt)
    assert st["tile_products"] == tp
    M.multiply_numeric(ctx, a, bt, c)
    got = c.download()
    assert np.array_equal(got.row_idx, c_row) and np.array_equal(got.col_idx, c_col)
    assert np.array_equal(got.data, c_data)
    M.multiply_numeric(ctx, a, bt, c)  # ORs into what is there
    assert np.array_equal(c.download().data, c_data)
    c.close()
    for min_bits in (0, 5, 4097):
        c, _ = M.multiply_symbolic(ctx, a, bt)
        dense = M.multiply_numeric_dense(ctx, a, bt, c, min_bits)
        assert dense == (tp if min_bits == 0 else 0 if min_bits == 4097 else dense)
        assert np.array_equal(c.download().data, c_data), min_bits
        c.close()
    keep = np.any(c_data != 0, axis=1)
    n_num = int(keep.sum())
    for cap in (M.PRUNED_EXACT, M.PRUNED_STRUCTURAL, max(1, n_num // 3), max(1, n_num)):
        c, ps = M.multiply_pruned(ctx, a, bt, cap)
        got = c.download()
        assert np.array_equal(got.row_idx, c_row[keep]) and np.array_equal(got.col_idx, c_col[keep]), cap
        assert np.array_equal(got.data, c_data[keep]), cap
        assert ps["numeric_tiles"] == n_num
        c.close()


@pytest.mark.parametrize("ns,occupied", [(1, 1.0), (12, 1.0), (13, 1.0), (300, 0.02)])
@pytest.mark.parametrize("prepare", [False, True])
def test_same_matrix_on_both_sides(ctx, ns, occupied, prepare):
    """A passed as both operands (C = A * A^T): one pass makes both operands' inputs."""
    import matrixgraph_amd as M

    h = random_tiles(ns, occupied, 3)
    c_row, c_col, c_data, _ = want_product(h, h)
    a = M.TiledMatrix.upload(ctx, M.HostTiledMatrix(*h))
    if prepare:
        a.prepare_operand()
    c, _ = M.multiply(ctx, a, a)
    got = c.download()
    assert np.array_equal(got.row_idx, c_row) and np.array_equal(got.col_idx, c_col)
    assert np.array_equal(got.data, c_data)


def test_result_layout_of_another_product(ctx):
    """A C from a symbolic pass of other operands, and one uploaded by the caller: the tiles it has are
    the product's, whatever the number of pairs that made it."""
    import matrixgraph_amd as M

    ah, bh = random_tiles(40, 0.05, 4), random_tiles(40, 0.05, 5)
    a, bt = (M.TiledMatrix.upload(ctx, M.HostTiledMatrix(*h)) for h in (ah, bh))
    full = M.TiledMatrix.upload(ctx, M.HostTiledMatrix(*random_tiles(40, 1.0, 6)))
    c_row, c_col, c_data, _ = want_product(ah, bh)
    want = np.zeros((1600, 64), np.uint64)
    want[c_row.astype(np.int64) * 40 + c_col] = c_data
    c, _ = M.multiply_symbolic(ctx, full, full)
    M.multiply_numeric(ctx, a, bt, c)
    assert np.array_equal(c.download().data, want)
    rows, cols = np.arange(1600, dtype=np.uint32) // 40, np.arange(1600, dtype=np.uint32) % 40
    c = M.TiledMatrix.upload(ctx, M.HostTiledMatrix(40, np.arange(41, dtype=np.uint32) * 40, rows, cols,
                                                    np.zeros((1600, 64), np.uint64)))
    M.multiply_numeric(ctx, a, bt, c)
    assert np.array_equal(c.download().data, want)
