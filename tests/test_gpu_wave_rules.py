"""The element-matrix kernel over its rules of few and many points: tiles of
2 x 2 node pairs and single pairs, points in registers and spread over the
lanes, stores through LDS and from the lanes.  Each against the oracle (the CPU
path for the rule that it does not hold), and the same bits for every admitted
number of elements per wavefront.  Likewise the Neo-Hookean tangent's stores."""
import pytest
import torch

import tensormesh_amd as tm
from oracle import fem
from tensormesh_amd import _native as nat
from tensormesh_amd.mesh import unit_cube_hex, unit_cube_tet, unit_square_quad, unit_square_tri

pytestmark = pytest.mark.gpu
DEV = "cuda"
#: cell -> (mesh, rules): a rule for each size the instances hold (4, 8, 16 and 32 points) that the cell has
CELLS = {
    "triangle": (lambda: unit_square_tri(5, 0.1, 1), (2, 5, 6)),
    "triangle6": (lambda: unit_square_tri(4, 0.1, 1, order=2), (2, 5, 7)),
    "triangle10": (lambda: unit_square_tri(3, 0.1, 1, order=3), (2, 5, 6)),
    "tetra": (lambda: unit_cube_tet(2, 0.1, 1), (2, 3, 5, 7)),
    "tetra10": (lambda: unit_cube_tet(2, 0.1, 1, order=2), (2, 3, 5, 7)),
    "tetra20": (lambda: unit_cube_tet(1, 0.1, 1, order=3), (2, 3, 5, 7)),
    "quad": (lambda: unit_square_quad(5, 0.1, 1), (2, 3, 5)),
    "quad9": (lambda: unit_square_quad(4, 0.1, 1, order=2), (2, 3, 5)),
    "hexahedron": (lambda: unit_cube_hex(3, 0.1, 1), (1, 2, 3)),
    "hexahedron27": (lambda: unit_cube_hex(2, 0.1, 1, order=2), (1, 2, 3)),
}


@pytest.mark.parametrize("cell,q", [(c, q) for c, (_, rules) in CELLS.items() for q in rules])
@pytest.mark.parametrize("form", ["laplace", "mass", "linear_elasticity"])
def test_rules(cell, q, form):
    print(f"case wave rules {cell} order {q} {form}", flush=True)
    m = CELLS[cell][0]()
    cls = {"laplace": tm.LaplaceElementAssembler, "mass": tm.MassElementAssembler,
           "linear_elasticity": tm.LinearElasticityElementAssembler}[form]
    for n in (1, m.elements().shape[0]):
        m1 = tm.Mesh(m.points, {cell: m.elements()[:n]})
        if cell.startswith("quad") and q == 5:
            want = cls.from_mesh(m1, quadrature_order=q)().values
        else:
            want = fem.assemble_bilinear(m1.points, m1.elements(), cell, q, form, E=1.0, nu=0.3)[0]
        for dtype in (torch.float64, torch.float32):
            md = tm.Mesh(m1.points.to(dtype), m1.cells).to(DEV)
            A = cls.from_mesh(md, quadrature_order=q)
            # float64: the bar of the parity tests.  float32: the points are
            # rounded to 2^-24 of the unit cube where an element is at least
            # 1/5 wide and at most three times as steep at its corners, which
            # the block takes to the fourth power; then the sum of the blocks
            tol = 1e-12 if dtype == torch.float64 else 4 * 3 * 5 * 2.0 ** -23 + 24 * 2.0 ** -24
            for sym in (True, False):
                A.symmetric_slots, got = sym, {}
                for e in (None, 1, 2):
                    A.epw = e
                    try:
                        got[e] = A().values
                    except nat.NativeError:
                        assert e == 2
                assert (got[None].cpu().double().reshape(want.shape) - want).abs().max() <= tol * want.abs().max()
                for e, v in got.items():
                    assert torch.equal(v, got[None]), (dtype, sym, e)


# cells with few blocks per wavefront, and those of one wavefront per workgroup
@pytest.mark.parametrize("cell,q", [("triangle", 2), ("quad", 2), ("tetra", 2), ("tetra", 7), ("tetra20", 2), ("hexahedron27", 2)])
def test_neo_hookean_blocks_from_the_lanes(cell, q):
    m = {"triangle": lambda: unit_square_tri(3, 0.1, 1), "quad": lambda: unit_square_quad(3, 0.1, 1),
         "tetra": lambda: unit_cube_tet(2, 0.1, 1), "tetra20": lambda: unit_cube_tet(1, 0.1, 1, order=3),
         "hexahedron27": lambda: unit_cube_hex(1, 0.1, 1, order=2)}[cell]()
    P, c, D = m.points, m.elements(), m.points.shape[1]
    u = 0.03 * torch.stack([torch.sin(P[:, 1]), P[:, 0] * P[:, -1], 0.5 * P[:, 0] ** 2][:D], 1)
    _, loc = fem.neohookean_element_tangent(P, c, cell, q, u, 1.0, 0.3)
    want = torch.zeros(m.n_points, m.n_points, D, D, dtype=torch.float64)
    want.index_put_((c[:, :, None].expand(-1, -1, c.shape[1]), c[:, None, :].expand(-1, c.shape[1], -1)), loc, accumulate=True)
    want = want.permute(0, 2, 1, 3).reshape(D * m.n_points, -1)
    A = tm.NeoHookeanModel.from_mesh(m.to(DEV), quadrature_order=q, E=1.0, nu=0.3)
    for sym in (True, False):
        A.symmetric_slots, first = sym, None
        for epw in (None, 1, 2):
            A.epw = epw
            if epw == 2 and (cell in ("tetra20", "hexahedron27") or q == 7):
                continue   # a wavefront takes one of these
            _, K = A.residual_and_tangent(u.to(DEV))
            assert (K.to_dense().cpu() - want).abs().max() <= 1e-12 * want.abs().max()
            first = K.values if first is None else first
            assert torch.equal(K.values, first)
