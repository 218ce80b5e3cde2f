"""Systems that a whole-solve launch (tm_pcg_run) cannot hold end it without a
result, and the two-launch steps solve them: the same bits as with ``chunk``,
which asks for those steps."""
import numpy as np
import pytest
import torch

import tensormesh_amd as tm
from tensormesh_amd import _native as nat
from tensormesh_amd.mesh import unit_cube_tet, unit_square_tri
from tensormesh_amd.solve import BatchedPCG

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _laplace(mesh):
    m = mesh.to(DEV)
    K = tm.LaplaceElementAssembler.from_mesh(m)()
    return tm.Condenser(m.boundary_mask)(K, torch.ones(m.n_points, dtype=torch.float64, device=DEV))


def _falls_back(s, f, want):
    assert s._run_plan() is not None
    for x, y in zip(s.solve(f), want):
        assert torch.equal(x, y)
    assert s._run is None   # found out by that solve


# 8 entries per thread, rows of up to 15: one workgroup, and several
@pytest.mark.parametrize("n", [8, 17])
def test_rows_longer_than_the_plan(n):
    print(f"case long rows {n}", flush=True)
    K, f = _laplace(unit_cube_tet(n, 0.15, 1))
    assert int((K.row_ptr[1:] - K.row_ptr[:-1]).max()) > 8
    a, b = (BatchedPCG(K.row_ptr, K.col_indices, K.values, [0, K.shape[0]], rtol=1e-10) for _ in range(2))
    want = a.solve(f, chunk=32)
    wgs = -(-np.diff(b._sys_blk) // 4)
    b._run = b._make_plan(1, 8, int(wgs.max()), wgs)
    assert (b._run.n_launch == 0) == (K.shape[0] <= 1024)
    _falls_back(b, f, want)


# two systems of 361 rows (a workgroup each), and of 6,241 (several), of which
# the first has an entry in a column of the second and the other way round
@pytest.mark.parametrize("n", [20, 80])
def test_columns_of_another_system(n):
    print(f"case columns of another system {n}", flush=True)
    K, f = _laplace(unit_square_tri(n, 0.2, 1))
    N = K.shape[0]
    assert N == (n - 1) ** 2
    last = torch.tensor([N - 1], device=DEV)
    row = torch.cat([K.row_indices, K.row_indices + N, last, last + 1])
    col = torch.cat([K.col_indices, K.col_indices + N, last + 1, last])
    val = torch.cat([K.values, K.values, torch.full((2,), -1e-3, dtype=torch.float64, device=DEV)])
    order = torch.argsort(row * 2 * N + col)
    rp = torch.zeros(2 * N + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(torch.bincount(row, minlength=2 * N), 0)
    a, b = (BatchedPCG(rp, col[order], val[order], [0, N, 2 * N], rtol=1e-10) for _ in range(2))
    ff = torch.cat([f, 2 * f])
    want = a.solve(ff, chunk=32)
    assert torch.isfinite(want[0]).all()
    _falls_back(b, ff, want)


class _Lib:
    """The library, with ``tm_pcg_run`` ending in a status of its own."""

    def __init__(self, lib, status):
        self._lib, self._status, self.calls = lib, status, 0

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def tm_pcg_run(self, *args):
        self.calls += 1
        return self._status


@pytest.mark.parametrize("name", ["TM_ERR_HIP", "TM_ERR_UNSUPPORTED"])
def test_a_refused_launch(name, monkeypatch):
    print(f"case refused launch {name}", flush=True)
    K, f = _laplace(unit_square_tri(60, 0.2, 1))
    a, b = (BatchedPCG(K.row_ptr, K.col_indices, K.values, [0, K.shape[0]], rtol=1e-10) for _ in range(2))
    want = a.solve(f, chunk=32)
    lib = _Lib(nat.lib(), getattr(nat, name))
    monkeypatch.setattr(nat, "lib", lambda: lib)
    _falls_back(b, f, want)
    assert lib.calls == 1


@pytest.mark.parametrize("n", [20, 60])   # one workgroup, and several
def test_budgets_beyond_one_launch(n, monkeypatch):
    """A budget past 32 bits is no limit to a solve that converges; one past the
    steps of a launch goes on in chunks."""
    print(f"case budgets {n}", flush=True)
    K, f = _laplace(unit_square_tri(n, 0.2, 1))
    a, b = (BatchedPCG(K.row_ptr, K.col_indices, K.values, [0, K.shape[0]], rtol=1e-10) for _ in range(2))
    want = a.solve(f, chunk=32)
    for max_iter in (2 ** 31, 2 ** 32 + 64, 10 ** 12):
        for x, y in zip(b.solve(f, max_iter=max_iter), want):
            assert torch.equal(x, y)
    assert b._run is not None and int(want[1]) > 32
    monkeypatch.setattr(BatchedPCG, "RUN_MAX_STEPS", 32)
    x0 = torch.linspace(-1, 1, K.shape[0], dtype=torch.float64, device=DEV)
    for kw in ({}, {"max_iter": 32}, {"max_iter": 64}, {"x0": x0}):
        want = a.solve(f, chunk=32, **kw)
        for x, y in zip(b.solve(f, **kw), want):
            assert torch.equal(x, y)
    assert b._run is not None


def test_no_memory_for_the_workspace(monkeypatch):
    print("case no memory for the workspace", flush=True)
    K, f = _laplace(unit_square_tri(60, 0.2, 1))
    a, b = (BatchedPCG(K.row_ptr, K.col_indices, K.values, [0, K.shape[0]], rtol=1e-10) for _ in range(2))
    want = a.solve(f, chunk=32)
    empty = torch.empty

    def full(*args, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no memory")
        return empty(*args, **kw)
    monkeypatch.setattr(torch, "empty", full)
    for x, y in zip(b.solve(f), want):
        assert torch.equal(x, y)
    assert b._run is None


@pytest.mark.parametrize("bad", [0, 2])   # the system whose last row is too long: in the first group, in the last
def test_one_of_several_groups_ends_without_a_result(bad, monkeypatch):
    """Groups launched after one that ended, and before it: all are solved again."""
    print(f"case groups {bad}", flush=True)
    systems = [_laplace(unit_square_tri(n, 0.2, n)) for n in (70, 60, 50)]
    rows, cols, vals, offs = [], [], [], [0]
    for k, (K, _) in enumerate(systems):
        N = K.shape[0]
        r, c, v = K.row_indices, K.col_indices, K.values
        if k == bad:   # nine more entries, zeros, on the last row
            r = torch.cat([r, torch.full((9,), N - 1, device=DEV)])
            c = torch.cat([c, torch.arange(9, device=DEV)])
            v = torch.cat([v, torch.zeros(9, dtype=torch.float64, device=DEV)])
            order = torch.argsort(r * N + c)
            r, c, v = r[order], c[order], v[order]
        rows.append(r + offs[-1]); cols.append(c + offs[-1]); vals.append(v); offs.append(offs[-1] + N)
    rp = torch.zeros(offs[-1] + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(torch.bincount(torch.cat(rows), minlength=offs[-1]), 0)
    a, b = (BatchedPCG(rp, torch.cat(cols), torch.cat(vals), offs, rtol=1e-10) for _ in range(2))
    f = torch.cat([f for _, f in systems])
    want = a.solve(f, chunk=32)
    wgs = -(-np.diff(b._sys_blk) // 4)
    b._run = b._make_plan(1, 8, int(wgs.max()), wgs)
    assert b._run.n_launch == 3
    _falls_back(b, f, want)
