"""DG stage kernel at the edges of its workgroups (6 tetrahedra; 8 or 3
hexahedra of degree 1 or 2): single cells, one cell short of a workgroup, one
over; every boundary family, all solvers, the step and the time step folded into
it.  Tolerances as in tests/test_dg_gpu.py: the same FP64 formulas summed in
another order, 1e-12 relative; the exact solver's stopping rule 1e-7.
"""
import numpy as np
import pytest

from pvcriemannsolvers_amd import meshgen
from test_dg_gpu import MIXED_BCS, TOL, make_pair, rel, smooth_state

pytestmark = pytest.mark.gpu


def first_tets(n):
    """The first n tetrahedra of a box, their free faces tagged in turn."""
    mesh = meshgen.box_tet(3, 1, 1, hi=(0.75, 0.25, 0.25))
    cells = mesh["cells"][:n]
    faces = np.concatenate([cells[:, [0, 1, 2]], cells[:, [0, 1, 3]], cells[:, [0, 2, 3]], cells[:, [1, 2, 3]]])
    _, first, counts = np.unique(np.sort(faces, axis=1), axis=0, return_index=True, return_counts=True)
    bfaces = faces[np.sort(first[counts == 1])]
    return dict(mesh, cells=np.ascontiguousarray(cells), bface_nodes=np.ascontiguousarray(bfaces),
                bface_tags=(np.arange(len(bfaces)) % 6).astype(np.int32))


@pytest.mark.parametrize("kind,cells", [("tet", 1), ("tet", 5), ("tet", 7), ("tet", 13),
                                        ("hex", 1), ("hex", 2), ("hex", 4), ("hex", 7), ("hex", 9)])
@pytest.mark.parametrize("degree", [1, 2])
@pytest.mark.parametrize("riemann", ["roe", "hllc", "exact"])
def test_workgroup_edges(kind, cells, degree, riemann):
    mesh = first_tets(cells) if kind == "tet" else meshgen.box_hex(cells, 1, 1, hi=(0.25 * cells, 0.25, 0.25))
    o, g = make_pair(mesh, degree, riemann, MIXED_BCS)
    u = o.approximate(smooth_state(o.cells()["xyz"]))
    g.set_solution_column(u)
    assert rel(g.get_residual_column(), o.residual(u)) <= TOL[riemann]
    dt = g.get_time_step(0.05)
    g.rk3_update(0.0, dt)
    ref = o.rk3(u, dt, 1)
    assert rel(g.get_solution_column(), ref) <= TOL[riemann]
    expect = o.time_step(ref, 0.05)
    assert abs(g.get_time_step(0.05) - expect) <= TOL[riemann] * expect
    g.close()


@pytest.mark.parametrize("mesh,degree", [(lambda: meshgen.box_tet(11, 11, 11, jitter=0.1, seed=3), 2),
                                         (lambda: meshgen.box_tet(12, 12, 10, jitter=0.1, seed=4), 2),
                                         (lambda: meshgen.box_tet(12, 12, 10, jitter=0.1, seed=5), 1),
                                         (lambda: meshgen.box_hex(21, 20, 20, shuffle_seed=6), 1)])
def test_exact_solver_on_both_sides_of_the_face_pass(mesh, degree):
    """7986 cells solve their own faces; 8640 and 8400 read a face pass."""
    mesh = mesh()
    o, g = make_pair(mesh, degree, "exact", MIXED_BCS)
    u = o.approximate(smooth_state(o.cells()["xyz"]))
    g.set_solution_column(u)
    assert rel(g.get_residual_column(), o.residual(u)) <= TOL["exact"]
    dt = g.get_time_step(0.05)
    g.rk3_update(0.0, dt)
    assert rel(g.get_solution_column(), o.rk3(u, dt, 1)) <= TOL["exact"]
    g.close()


@pytest.mark.parametrize("kind", ["tet", "hex"])
@pytest.mark.parametrize("degree", [1, 2])
@pytest.mark.parametrize("riemann", ["roe", "hllc", "exact"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_bad_values_reach_face_neighbours_only(kind, degree, riemann, value):
    """A NaN or an infinity in one cell leaves the cells that share its workgroup,
    but no face, as they are."""
    mesh = meshgen.box_tet(3, 3, 3, jitter=0.1, seed=3) if kind == "tet" else meshgen.box_hex(6, 4, 4, shuffle_seed=3)
    o, g = make_pair(mesh, degree, riemann, MIXED_BCS)
    n = len(mesh["cells"])
    u = o.approximate(smooth_state(o.cells()["xyz"])).reshape(n, -1)
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
        assert not np.isfinite(got[cell]).all()
    g.close()
