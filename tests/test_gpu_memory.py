"""Device memory kept between objects: results dropped while work is still queued, threads with
their own contexts, and blocks given back with the last context. Every result is compared with the
oracle's, so a block handed out too early would show."""
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def square(M, ctx, scale, seed):
    el = M.EdgeList.rmat(ctx, scale, 16, 0.57, 0.19, 0.19, seed)
    a, at = el.to_tiled_matrix(False), el.to_tiled_matrix(True)
    el.close()
    return a, at


def oracle_square(scale, seed):
    n = 1 << scale
    s, d = O.rmat_edges(scale, 16, 0.57, 0.19, 0.19, seed)
    ah, ath = O.edges_to_tiles(n, s, d), O.edges_to_tiles(n, s, d, transpose=True)
    _, c_row, c_col, _ = O.tile_symbolic(ah[0], ah[1], ah[3], ath[1], ath[3])
    return O.tile_numeric(ah[0], ah[1:], ath[1:], c_row, c_col)


def test_dropped_results_do_not_reach_later_ones(ctx):
    import matrixgraph_amd as M

    want = {seed: oracle_square(11, seed) for seed in (1, 2)}
    ops = {seed: square(M, ctx, 11, seed) for seed in (1, 2)}
    for i in range(12):
        seed = 1 + i % 2
        c, _ = M.multiply(ctx, *ops[seed])
        c.close()  # the numeric pass may still be running
        c, _ = M.multiply(ctx, *ops[3 - seed])
        assert np.array_equal(c.download().data, want[3 - seed])
        c.close()


def test_threads_with_their_own_contexts():
    import matrixgraph_amd as M

    want = {seed: oracle_square(10, seed) for seed in range(4)}
    bad = []

    def work(seed):
        c = M.Context(0)
        for _ in range(8):
            a, at = square(M, c, 10, seed)
            p, _ = M.multiply(c, a, at)
            if not np.array_equal(p.download().data, want[seed]):
                bad.append(seed)
            for m in (p, a, at):
                m.close()
        c.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("size", [1, 511, 512, 513, 3 << 20, 200 << 20])
def test_buffers_come_back_zeroed(ctx, size):
    import matrixgraph_amd as M

    for _ in range(3):
        b = M.DeviceBuffer(ctx, size)
        assert not b.to_array(np.uint8).any()
        b.close()
        b = M.DeviceBuffer.from_array(ctx, np.full(size, 7, np.uint8))
        assert (b.to_array(np.uint8) == 7).all()
        b.close()


def test_second_free_is_refused(ctx):
    """Freeing a buffer twice is an error, whether its block is kept (1 MiB) or went back to the driver
    (one too large to keep), and the next buffers are memory of their own."""
    import ctypes as C

    import matrixgraph_amd as M

    lib = M.lib()
    for size in (1 << 20, 4 << 30):
        p = C.c_void_p()
        assert lib.mg_buffer_alloc(ctx.h, size, C.byref(p)) == 0
        assert lib.mg_buffer_free(ctx.h, p) == 0
        assert lib.mg_buffer_free(ctx.h, p) != 0
    a, b = (M.DeviceBuffer.from_array(ctx, np.full(1 << 20, v, np.uint8)) for v in (1, 2))
    assert a.ptr != b.ptr
    assert (a.to_array(np.uint8) == 1).all() and (b.to_array(np.uint8) == 2).all()
    a.close()
    b.close()


def pool_bytes(M):
    """Bytes of the device's default pool that are handed out (temporaries and contexts' scratch)."""
    import ctypes as C

    lib, pool, used = M.lib(), C.c_void_p(), C.c_uint64()
    assert lib.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert lib.hipMemPoolGetAttribute(pool, 7, C.byref(used)) == 0  # hipMemPoolAttrUsedMemCurrent
    return used.value


def test_frontier_download_keeps_a_bounded_piece():
    """A frontier of several pieces, in the engine's permuted strip order: what the context keeps after
    the download is one piece of 64 MiB, and the frontier is the oracle's."""
    import matrixgraph_amd as M

    scale, n_src = 18, 4096
    n = 1 << scale
    with M.Context(0) as c:
        el = M.EdgeList.rmat(c, scale, 16, 0.57, 0.19, 0.19, 9)
        at = el.to_tiled_matrix(True)
        el.close()
        w = M.Walk(c, at, n_src, 1)
        sources = O.sample_sources(n, n_src, 3)
        w.run(sources, 1)
        before = pool_bytes(M)
        got = w.frontier(1)
        assert pool_bytes(M) - before <= 64 << 20
        w.close()
        at.close()
    s, d = O.rmat_edges(scale, 16, 0.57, 0.19, 0.19, 9)
    assert np.array_equal(got, O.walk_frontiers(n, s, d, sources, 1, W=64)[1])


def test_scratch_above_the_limit_is_given_back():
    """300 M uploaded edges (all the same) sort in 4.8 GB of scratch, more than the 1/64 of the card that a
    context keeps: none of it stays. A small upload's scratch does."""
    import ctypes as C

    import matrixgraph_amd as M

    free, total = C.c_size_t(), C.c_size_t()
    with M.Context(0) as c:
        assert M.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        n = total.value // 64 // 16 + (1 << 20)
        ids = np.zeros(n, np.uint32)
        before = pool_bytes(M)
        el = M.EdgeList.upload(c, 7, ids, ids)
        assert el.info() == (7, 1)
        el.close()
        assert pool_bytes(M) == before
        el = M.EdgeList.upload(c, 7, ids[:1 << 20], ids[:1 << 20])
        assert el.info() == (7, 1)
        el.close()
        assert (16 << 20) <= pool_bytes(M) - before <= total.value // 64


def test_prepare_without_memory_for_column_words():
    """2.25 M full tiles, whose column words (1.2 GB) do not fit beside what else is on the device: the
    operand is prepared without them, and its products are the same."""
    import ctypes as C

    import matrixgraph_amd as M

    lib, ns = M.lib(), 1500
    free, total = C.c_size_t(), C.c_size_t()
    filled = []
    with M.Context(0) as c:
        bt = M.TiledMatrix.upload(c, M.HostTiledMatrix(
            ns, np.arange(ns + 1, dtype=np.uint32) * ns, np.repeat(np.arange(ns, dtype=np.uint32), ns),
            np.tile(np.arange(ns, dtype=np.uint32), ns), np.full((ns * ns, 64), ~np.uint64(0))))
        off = np.full(ns + 1, 3, np.uint32)
        off[0] = 0
        data = np.zeros((3, 64), np.uint64)
        data[:, 5] = np.uint64(1) << np.uint64(9)
        a = M.TiledMatrix.upload(c, M.HostTiledMatrix(ns, off, np.zeros(3, np.uint32), np.array([0, 7, 1499], np.uint32), data))
        want, _ = M.multiply(c, a, bt)
        M.multiply_numeric(c, a, bt, want)
        try:
            while True:
                assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
                if free.value < 1 << 30:
                    break
                p = C.c_void_p()
                assert lib.hipMalloc(C.byref(p), C.c_size_t(min(free.value - (800 << 20), 64 << 30))) == 0
                filled.append(p)
            bt.prepare_operand()
            assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
            assert free.value > 256 << 20  # the words are not there
        finally:
            for p in filled:
                assert lib.hipFree(p) == 0
        got, _ = M.multiply(c, a, bt)
        got, want = got.download(), want.download()
        assert np.array_equal(got.data, want.data) and len(got.data) == ns
        assert (got.data[:, 5] == ~np.uint64(0)).all() and not np.delete(got.data, 5, axis=1).any()
        dense, _ = M.multiply_symbolic(c, a, bt)
        assert M.multiply_numeric_dense(c, a, bt, dense, 1) == 3 * ns
        assert np.array_equal(dense.download().data, want.data)
        for m in (a, bt, dense):
            m.close()


@pytest.mark.parametrize("size", [(1 << 64) - 1, (1 << 64) - 600, 1 << 50])
def test_impossible_sizes_are_out_of_memory(ctx, size):
    import ctypes as C

    import matrixgraph_amd as M

    p = C.c_void_p(1)
    assert M.lib().mg_buffer_alloc(ctx.h, C.c_size_t(size), C.byref(p)) == 3  # MG_ERR_OOM
    assert not p.value
