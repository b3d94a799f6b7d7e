"""Columns between host and device at the sizes where the copy changes form:
below and from 2 MiB to the host (a ring of pinned slots from there on), fewer
chunks than slots, more, a last chunk that is not full, and from 32 MiB to the
device.  What is put in comes out, byte for byte, from two threads at once too.
"""
import threading

import numpy as np
import pytest

from pvcriemannsolvers_amd import meshgen, spatial

pytestmark = pytest.mark.gpu


# 2560 bytes per cell of degree 3: 1.8, 2.3, 15.7, 17.6, 32.5, 33.9 and 36.9 MB
@pytest.mark.parametrize("size", [(8, 9, 10), (9, 10, 10), (17, 19, 19), (19, 19, 19), (23, 23, 24), (23, 23, 25),
                                  (24, 25, 24)])
def test_round_trip(size):
    g = spatial.FiniteElement(meshgen.box_hex(*size), degree=3, riemann="hllc", bcs=[("inviscid_wall", None)] * 6)
    rng = np.random.default_rng(size[0])
    u = 1 + 1e-2 * rng.random((g.column_size // 5, 5))
    u[:, 4] += 9
    u = u.reshape(-1)
    g.set_solution_column(u)
    r = g.get_residual_column()
    assert np.isfinite(r).all()
    wrong = []

    def read(get, want):
        for _ in range(3):
            if not np.array_equal(get(), want):
                wrong.append(get.__name__)

    threads = [threading.Thread(target=read, args=a) for a in ((g.get_solution_column, u), (g.get_residual_column, r))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    g.close()


def test_batch_columns_of_different_sizes():
    """Cases smaller than the one the ring was made for."""
    walls = [("inviscid_wall", None)] * 6
    batch = spatial.Batch([(meshgen.box_hex(n, 9, 9), 3, walls) for n in (3, 40, 9, 90)])
    columns = []
    for i, (cells, nodes) in enumerate(batch.sizes):
        u = 1 + 1e-2 * np.random.default_rng(i).random(cells * nodes * 5)
        batch.set_solution_column(i, u)
        columns.append(u)
    for i, u in enumerate(columns):
        np.testing.assert_array_equal(batch.get_solution_column(i), u)
    batch.close()


def test_reads_from_two_threads_complete():
    """Solution and residual, which pass through one buffer, read over and over by
    two threads: every read returns, and returns its own column."""
    g = spatial.FiniteElement(meshgen.box_hex(19, 19, 19), degree=3, riemann="hllc", bcs=[("inviscid_wall", None)] * 6)
    rng = np.random.default_rng(7)
    u = 1 + 1e-2 * rng.random((g.column_size // 5, 5))
    u[:, 4] += 9
    g.set_solution_column(u.reshape(-1))
    want = {g.get_solution_column: u.reshape(-1), g.get_residual_column: g.get_residual_column()}
    seen = {get: [] for get in want}

    def read(get):
        for _ in range(8):
            seen[get].append(np.array_equal(get(), want[get]))

    threads = [threading.Thread(target=read, args=(get,)) for get in want]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(seen[get] == [True] * 8 for get in want)
    g.close()
