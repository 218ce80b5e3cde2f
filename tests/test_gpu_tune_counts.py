"""epw = "auto" times the kernel's own choice of elements per wavefront beside
the others, and that choice gives the same bits."""
import json

import pytest
import torch

import tensormesh_amd as tm
from tensormesh_amd import tune
from tensormesh_amd.mesh import unit_cube_hex, unit_cube_tet, unit_square_quad, unit_square_tri

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_auto_times_the_default(dtype, tmp_path, monkeypatch):
    print(f"case auto counts {dtype}", flush=True)
    path = tmp_path / "tune.json"
    monkeypatch.setenv("TENSORMESH_AMD_TUNE_CACHE", str(path))
    monkeypatch.setattr(tune, "_TUNER", None)
    at = lambda m: tm.Mesh(m.points.to(dtype), m.cells).to(DEV)
    m10, m4, mh = at(unit_cube_tet(3, 0.1, 2, order=2)), at(unit_cube_tet(4, 0.1, 2)), at(unit_cube_hex(3, 0.1, 2))
    P, u4 = m10.points, 1e-3 * torch.stack([3 * m4.points[:, 0], -m4.points[:, 1], 0.5 * m4.points[:, 2]], 1)
    u10 = 0.03 * torch.stack([torch.sin(P[:, 1]), P[:, 0] * P[:, 2], 0.5 * P[:, 0] ** 2], 1)
    E = dict(E=1.0, nu=0.3)
    cases = [("wave", tm.LinearElasticityElementAssembler.from_mesh(m10, **E), lambda A: A().values),
             ("wave", tm.LaplaceElementAssembler.from_mesh(mh), lambda A: A().values),
             ("neohookean", tm.NeoHookeanModel.from_mesh(m10, **E), lambda A: A.residual_and_tangent(u10)[1].values),
             ("j2", tm.J2Plasticity.from_mesh(m4, E=200.0, nu=0.3, sig0=0.25, H=1.0),
              lambda A: A.residual_and_tangent(u4)[1].values)]
    for kernel, A, run in cases:
        want = run(A)
        before = set(json.loads(path.read_text())) if path.exists() else set()
        A.epw = "auto"
        assert torch.equal(run(A), want), kernel
        new = [k for k in json.loads(path.read_text()) if k not in before]
        assert len(new) == 1 and f"|epw|{kernel}|" in new[0]
        timed = json.loads(path.read_text())[new[0]]["ms"]
        assert "0" in timed and len(timed) >= 3
        for e in timed:
            A.epw = int(e)
            assert torch.equal(run(A), want), (kernel, e)


@pytest.mark.parametrize("cell", ["triangle6", "triangle10", "tetra10", "tetra20", "quad", "quad9", "hexahedron", "hexahedron27"])
def test_two_elements_are_admitted_for_short_rules(cell):
    """One-point rules leave room for two elements of every cell."""
    print(f"case two elements {cell}", flush=True)
    order = 2 if cell[-1] in "69" or cell in ("tetra10", "hexahedron27") else 3 if cell[-2:] in ("10", "20") else 1
    make = {"tri": unit_square_tri, "tet": unit_cube_tet, "qua": unit_square_quad, "hex": unit_cube_hex}[cell[:3]]
    m = make(2, 0.1, 1, order=order).to(DEV)
    assert list(m.cells) == [cell]
    for A in (tm.MassElementAssembler.from_mesh(m, quadrature_order=1),
              tm.LinearElasticityElementAssembler.from_mesh(m, quadrature_order=1, E=1.0, nu=0.3)):
        want = A().values
        for A.epw in (1, 2):
            assert torch.equal(A().values, want)
