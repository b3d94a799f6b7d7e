"""FR kernels at the edges of their tiles: cells that do not fill a workgroup
(16, 7, 4, 3, 1 cells for degrees 1..5), single cells, the last cell of a mesh
whose cells go two to a wavefront (degree 3, more than 4096 cells), and
neighbours turned against each other, whose lines are gathered in every
direction.  Tolerances as in tests/test_fr_gpu.py: the same FP64 formulas summed
in another order, 1e-12 relative (Roe, HLLC), 1e-7 for the exact solver's
stopping rule; the mixed form's residual 1e-5 of its max norm.
"""
import numpy as np
import pytest

import oracle_lib as ol
from pvcriemannsolvers_amd import meshgen, spatial
from test_boundary_cpu import rotate_cells
from test_fr_gpu import RIEMANN, TOL, conservative, density_wave, make_pair, rel

pytestmark = pytest.mark.gpu

LEFT, RIGHT = conservative(1.0, (0.1, 0, 0), 1.0), conservative(0.125, (0, 0, 0), 0.1)
BCS = [("smart", LEFT), ("smart", RIGHT)] + [("inviscid_wall", None)] * 4
EDGES = [(1, 1), (1, 15), (1, 16), (1, 17), (2, 6), (2, 7), (2, 8), (3, 1), (3, 3), (3, 5),
         (4, 2), (4, 3), (4, 4), (5, 1), (5, 3)]


@pytest.mark.parametrize("degree,cells", EDGES)
@pytest.mark.parametrize("riemann", ["roe", "hllc", "exact"])
def test_tile_edges_turned_cells(degree, cells, riemann):
    mesh = rotate_cells(meshgen.box_hex(cells, 1, 1, hi=(1.0, 0.1, 0.1), shuffle_seed=cells), degree)
    o, g = make_pair(mesh, degree, riemann, BCS)
    u = density_wave(o.node_coords(), seed=cells)
    g.set_solution_column(u.reshape(-1))
    assert rel(g.get_residual_column(), o.residual(u).reshape(-1)) < TOL[riemann]
    np.testing.assert_array_equal(g.get_solution_column(), u.reshape(-1))
    g.close()


@pytest.mark.parametrize("degree", [1, 2, 3, 4, 5])
def test_mixed_turned_cells(degree):
    mesh = rotate_cells(meshgen.box_hex(5, 3, 3, periodic=(True,) * 3, shuffle_seed=3), 17)
    o = ol.FrOracle(mesh, q=degree + 1, riemann=RIEMANN["roe"])
    g = spatial.FiniteElement(mesh, degree=degree, riemann="roe", precision="mixed")
    u = density_wave(o.node_coords(), seed=7)
    g.set_solution_column(u.reshape(-1))
    assert rel(g.get_residual_column(), o.residual(u).reshape(-1)) < 1e-5
    g.close()


@pytest.mark.parametrize("riemann,jitter", [("roe", 0.0), ("hllc", 0.0), ("roe", 0.2), ("exact", 0.0)])
def test_two_cells_per_wavefront(riemann, jitter):
    """4335 cells: the last wavefront has one; a step and the time step folded into it.
    (Spacing 1/16, so that cell sizes carry no rounding of the coordinates: with
    1/17 that alone moves this residual by 3e-12.)"""
    mesh = rotate_cells(meshgen.box_hex(17, 17, 15, hi=(17 / 16, 17 / 16, 15 / 16), periodic=(True,) * 3,
                                        jitter=jitter, seed=4, shuffle_seed=5), 6)
    o, g = make_pair(mesh, 3, riemann)
    u = density_wave(o.node_coords(), seed=8)
    g.set_solution_column(u.reshape(-1))
    assert rel(g.get_residual_column(), o.residual(u).reshape(-1)) < TOL[riemann]
    dt = g.get_time_step(0.1)
    ref = o.rk3(u.reshape(-1), dt, n_steps=1)
    g.rk3_update(0.0, dt)
    assert rel(g.get_solution_column(), ref) < TOL[riemann]
    expect = o.time_step(ref, 0.1)
    assert abs(g.get_time_step(0.1) - expect) <= (1e-12 if riemann != "exact" else 1e-7) * expect
    g.close()


@pytest.mark.parametrize("degree", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("size", [(1, 1, 1), (7, 5, 3), (17, 16, 16)])
@pytest.mark.parametrize("jitter", [0.0, 0.2])
def test_time_step_of_any_node(degree, size, jitter):
    """The smallest length / (|u| + c), wherever the fastest node lies: read of a
    state and folded into a step's last stage."""
    mesh = meshgen.box_hex(*size, jitter=jitter, seed=9, shuffle_seed=2)
    o, g = make_pair(mesh, degree, "roe", [("smart", LEFT)] * 6)
    u = density_wave(o.node_coords(), seed=3).reshape(len(mesh["cells"]), -1, 5)
    rng = np.random.default_rng(degree)
    places = [(0, 0), (-1, -1)] + [(rng.integers(u.shape[0]), rng.integers(u.shape[1])) for _ in range(4)]
    for cell, node in places:
        v = u.copy()
        v[cell, node, 4] *= 9
        g.set_solution_column(v.reshape(-1))
        expect = o.time_step(v.reshape(-1), 0.1)
        assert abs(g.get_time_step(0.1) - expect) <= 1e-12 * expect
        g.rk3_update(0.0, 0.01 * expect)
        state = g.get_solution_column()
        fused, expect = g.get_time_step(0.1), o.time_step(state, 0.1)
        assert abs(fused - expect) <= 1e-12 * expect
        g.set_solution_column(state)
        assert g.get_time_step(0.1) == fused
    g.close()


@pytest.mark.parametrize("degree,size", [(3, (17, 17, 15)), (3, (6, 5, 4)), (1, (6, 5, 4)), (2, (6, 5, 4)),
                                         (4, (6, 5, 4)), (5, (6, 5, 4))])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_bad_values_reach_face_neighbours_only(degree, size, value):
    """A NaN or an infinity in one cell leaves the cells that share its wavefront
    or workgroup, but no face, as they are."""
    mesh = meshgen.box_hex(*size, periodic=(True,) * 3, shuffle_seed=3)
    g = spatial.FiniteElement(mesh, degree=degree, riemann="roe")
    n = len(mesh["cells"])
    u = density_wave(g.sample_points(), seed=2).reshape(n, -1)
    g.set_solution_column(u.reshape(-1))
    want = g.get_residual_column().reshape(n, -1)
    faces = g.faces()
    for cell in (0, n // 2, n // 2 + 1, n - 1):
        bad = u.copy()
        bad[cell, 0] = value
        g.set_solution_column(bad.reshape(-1))
        got = g.get_residual_column().reshape(n, -1)
        near = {cell}
        for a, b in zip(faces["holder"], faces["sharer"]):
            if a == cell or b == cell:
                near |= {int(a), int(b)}
        far = np.setdiff1d(np.arange(n), sorted(near))
        np.testing.assert_array_equal(got[far], want[far])
    g.close()


@pytest.mark.parametrize("cell", [0, 2166, 4333, 4334])
def test_folded_time_step_of_an_odd_last_cell(cell):
    """4335 cells of degree 3, two to a wavefront, the last one with its
    wavefront to itself: with a cell whose fastest node gains speed in the step, the
    minimum folded into stage 3, which writes over the state it reads, is that of the
    state it wrote."""
    mesh = meshgen.box_hex(17, 17, 15, shuffle_seed=2)
    o, g = make_pair(mesh, 3, "roe", [("smart", LEFT)] * 6)
    u = density_wave(o.node_coords(), seed=3).reshape(len(mesh["cells"]), -1, 5)
    u[cell, :, 4] *= np.random.default_rng(0).uniform(5, 9, 64)
    g.set_solution_column(u.reshape(-1))
    dt = g.get_time_step(0.1)
    g.rk3_update(0.0, dt)
    fused = g.get_time_step(0.1)
    assert fused < 0.99 * dt
    state = g.get_solution_column()
    g.set_solution_column(state)
    assert fused == g.get_time_step(0.1)
    expect = o.time_step(state, 0.1)
    assert abs(fused - expect) <= 1e-12 * expect
    g.close()


@pytest.mark.parametrize("riemann", ["hllc", "exact"])
@pytest.mark.parametrize("degree,size", [(3, (17, 17, 15)), (3, (6, 5, 4)), (2, (6, 5, 4))])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_bad_values_stay_local_with_every_solver(riemann, degree, size, value):
    """As test_bad_values_reach_face_neighbours_only, whose solver is Roe's."""
    mesh = meshgen.box_hex(*size, periodic=(True,) * 3, shuffle_seed=3)
    g = spatial.FiniteElement(mesh, degree=degree, riemann=riemann)
    n = len(mesh["cells"])
    u = density_wave(g.sample_points(), seed=2).reshape(n, -1)
    g.set_solution_column(u.reshape(-1))
    want = g.get_residual_column().reshape(n, -1)
    faces = g.faces()
    cell = n - 1
    u[cell, 0] = value
    g.set_solution_column(u.reshape(-1))
    got = g.get_residual_column().reshape(n, -1)
    near = {cell} | {int(a + b - cell) for a, b in zip(faces["holder"], faces["sharer"]) if cell in (a, b)}
    far = np.setdiff1d(np.arange(n), sorted(near))
    np.testing.assert_array_equal(got[far], want[far])
    assert not np.isfinite(got[cell]).all()
    g.close()
