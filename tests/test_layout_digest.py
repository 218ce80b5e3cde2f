"""Layout digests that are computed on demand: what a copy, a file or a moved
Condenser holds, on the CPU (the meta device stands for another one)."""
import copy
import io
import pickle

import pytest
import torch

import tensormesh_amd as tm
from oracle import fem
from tensormesh_amd.mesh import unit_square_tri
from tensormesh_amd.sparse import LazyDigest, SparseMatrix


@pytest.fixture
def digests(monkeypatch):
    """Calls that hashed an index so far."""
    calls, plain = [], SparseMatrix._digest
    monkeypatch.setattr(SparseMatrix, "_digest", staticmethod(lambda r, c: calls.append(r.numel()) or plain(r, c)))
    return calls


def _block_matrix(n=4):
    m = unit_square_tri(n, 0.1, 1)
    A = tm.LinearElasticityElementAssembler.from_mesh(m, E=1.0, nu=0.3)
    return m, A, A()


def _want(K):
    return fem.layout_hash(K.row_indices, K.col_indices)


def _held(obj):
    """Index tensors that an unresolved digest of obj holds."""
    h = obj._layout_hash
    return h._index or () if isinstance(h, LazyDigest) else ()


def test_a_copy_on_another_device_holds_its_own_indices(digests):
    _, _, K = _block_matrix()
    there = K.to("meta")
    assert all(i.device.type == "meta" for i in _held(there)) and len(_held(there)) == 2
    assert K.to(torch.float32)._layout_hash is K._layout_hash and K.cpu()._layout_hash is K._layout_hash
    assert not digests and K.layout_hash == _want(K) and len(digests) == 1
    assert K.to("meta").layout_hash == K.layout_hash and len(digests) == 1   # known: nothing to hash there


def test_files_and_deep_copies(digests):
    m, A, K = _block_matrix()
    Kc = copy.deepcopy(K)
    assert not digests and Kc.row_indices is _held(Kc)[0] and Kc.row_indices is not K.row_indices
    assert Kc.layout_hash == _want(K)
    for load in (pickle.loads(pickle.dumps(K)), _saved(K)):
        assert _held(load) == () and load.layout_hash == _want(K)
    assert copy.deepcopy(A)().layout_hash == _want(K)


def _saved(obj):
    f = io.BytesIO()
    torch.save(obj, f)
    f.seek(0)
    return torch.load(f, weights_only=False)


def test_a_moved_condenser_lets_go_of_its_indices():
    m, _, K = _block_matrix()
    cond = tm.Condenser(m.boundary_mask.repeat_interleave(2))
    Ki, _ = cond(K, torch.ones(K.shape[0], dtype=torch.float64))
    here = [id(i) for i in Ki._layout_hash._index]
    assert here == [id(cond.inner_row), id(cond.inner_col)]
    cond.to("meta")
    assert all(i.device.type == "meta" for i in cond._inner_hash._index)
    assert cond.layout_hash == _want(K) and not isinstance(vars(cond).get("_layout"), LazyDigest)
    assert Ki.layout_hash == _want(Ki)


def test_condensing_the_same_indices_hashes_nothing(digests):
    m, A, K = _block_matrix()
    f = torch.ones(K.shape[0], dtype=torch.float64)
    cond = tm.Condenser(m.boundary_mask.repeat_interleave(2))
    assert cond.layout_hash is None
    cond(K, f)
    cond(A(), f)
    cond(K.detach(), f)
    assert A().has_same_layout(K) and not digests
    same = SparseMatrix(K.values, K.row_indices.clone(), K.col_indices.clone(), K.shape)
    cond(same, f)                                   # other tensors: compared by digest
    assert cond.layout_hash == _want(K) and len(digests) == 2
    other = SparseMatrix(K.values, K.row_indices, K.col_indices.flip(0), K.shape)
    with pytest.raises(AssertionError, match="layout of the matrix is changed"):
        cond(other, f)
    _, _, K5 = _block_matrix(5)
    assert not K5.has_same_layout(K) and not K.has_same_layout(K5) and K.has_same_layout(_want(K))
    with pytest.raises(TypeError):
        K.has_same_layout(None)


def test_condenser_files(digests):
    m, _, K = _block_matrix()
    f = torch.ones(K.shape[0], dtype=torch.float64)
    cond = tm.Condenser(m.boundary_mask.repeat_interleave(2))
    cond(K, f)
    state = cond.__getstate__() if hasattr(cond, "__getstate__") else cond.__dict__
    old = dict(state, layout_hash=_want(K))         # as written before digests were computed on demand
    del old["_layout"]
    older = tm.Condenser.__new__(tm.Condenser)
    older.__setstate__(old)
    for c in (older, _saved(cond), copy.deepcopy(cond)):
        assert c.layout_hash == _want(K)
        c(K, f)
