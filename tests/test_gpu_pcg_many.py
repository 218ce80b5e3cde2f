"""Stacks of more systems than the host reads the scalars of
(BatchedPCG.HOST_SYSTEMS): the flags are tested on the device, with the same
iterates, counts and residuals as for a stack read whole."""
import pytest
import torch

from tensormesh_amd.solve import BatchedPCG

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _stack(n_sys, n):
    """n_sys tridiagonal systems of n rows, each with a diagonal of its own."""
    i = torch.arange(n_sys * n, device=DEV)
    at = i % n
    keep = torch.stack([at > 0, at >= 0, at < n - 1], 1)
    rp = torch.zeros(n_sys * n + 1, dtype=torch.int64, device=DEV)
    rp[1:] = torch.cumsum(keep.sum(1), 0)
    off = -torch.ones_like(i, dtype=torch.float64)
    val = torch.stack([off, 2.0 + 1.0 / (1.0 + i // n), off], 1)
    return rp, torch.stack([i - 1, i, i + 1], 1)[keep], val[keep], list(range(0, n_sys * n + 1, n))


@pytest.mark.parametrize("n_sys", [BatchedPCG.HOST_SYSTEMS, BatchedPCG.HOST_SYSTEMS + 1])
@pytest.mark.parametrize("kw", [{}, {"chunk": 8}, {"graph": False}, {"max_iter": 5}])
def test_scalars_on_the_device(n_sys, kw, monkeypatch):
    print(f"case {n_sys} systems {kw}", flush=True)
    rp, ci, val, offs = _stack(n_sys, 24)
    f = torch.linspace(1, 2, offs[-1], dtype=torch.float64, device=DEV)
    s = BatchedPCG(rp, ci, val, offs, rtol=1e-10)
    assert s._state().is_cuda == (n_sys > BatchedPCG.HOST_SYSTEMS)
    got = s.solve(f, **kw)
    last = s._last_iters
    assert last == int(got[1].max()) and (bool((got[2] <= 1e-10).all()) or "max_iter" in kw)
    monkeypatch.setattr(BatchedPCG, "HOST_SYSTEMS", 4096)
    t = BatchedPCG(rp, ci, val, offs, rtol=1e-10)
    for x, y in zip(got, t.solve(f, **kw)):
        assert x.is_cuda and torch.equal(x, y)
    assert t._last_iters == last
