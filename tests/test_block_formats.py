"""Blocks without DGL are plain tuples; a DGL that turns up later is used from then on."""
import sys
import types

import pytest
import torch


def _stub_dgl(made):
    dgl, het = types.ModuleType("dgl"), types.ModuleType("dgl.heterograph")

    class DGLBlock:
        def __init__(self, *args):
            made.append(args)

    het.DGLBlock = DGLBlock
    index = types.SimpleNamespace(create_unitgraph_from_csr=lambda *a, **k: "csr", create_unitgraph_from_coo=lambda *a, **k: "coo")
    dgl.heterograph_index, dgl.heterograph = index, het
    return dgl, het


def test_blocks_with_and_without_dgl(monkeypatch):
    import shmtensor_amd
    shmtensor_amd.install_aliases()
    from shmtensor_amd.shmtensor import sampling
    monkeypatch.setitem(sys.modules, "dgl", None)            # (an import of it fails)
    monkeypatch.setattr(sampling, "_dgl_missing", False)
    a, b = torch.tensor([0, 2]), torch.tensor([1, 0])
    for _ in range(2):                                       # the failed look-up, and the one that remembers it
        assert isinstance(sampling.create_block_from_csc(a, b, torch.Tensor(), 2, 1), sampling.CSCBlock)
        assert isinstance(sampling.create_block_from_coo(a, b, 2, 1), sampling.COOBlock)
    made = []
    dgl, het = _stub_dgl(made)
    monkeypatch.setitem(sys.modules, "dgl", dgl)             # imported by someone after that
    monkeypatch.setitem(sys.modules, "dgl.heterograph", het)
    assert isinstance(sampling.create_block_from_csc(a, b, torch.Tensor(), 2, 1), het.DGLBlock)
    assert isinstance(sampling.create_block_from_coo(a, b, 2, 1), het.DGLBlock) and len(made) == 2


@pytest.fixture
def importable_dgl(tmp_path, monkeypatch):
    """Writes a dgl module and puts it on the import path; what was imported of it is gone afterwards."""
    before = {name: sys.modules.pop(name) for name in ("dgl", "dgl.heterograph") if name in sys.modules}

    def make(source):
        (tmp_path / "dgl.py").write_text(source)
        monkeypatch.syspath_prepend(str(tmp_path))

    yield make
    for name in ("dgl", "dgl.heterograph"):
        sys.modules.pop(name, None)
    sys.modules.update(before)


def _loader(sampling, monkeypatch):
    """A loader built without a GPU (its tensors stay where they are)."""
    monkeypatch.setattr(sampling.capi, "pin_memory", lambda t: None)
    monkeypatch.setattr(sampling, "_unpin", lambda t: None)
    monkeypatch.setattr(torch.Tensor, "cuda", lambda self: self)
    return sampling.GPUSamplingDataloader(torch.tensor([0, 1, 2]), torch.tensor([1, 0]), torch.arange(2), 1, [1])


def test_a_new_loader_looks_again(monkeypatch, importable_dgl):
    import shmtensor_amd
    shmtensor_amd.install_aliases()
    from shmtensor_amd.shmtensor import sampling
    monkeypatch.setattr(sampling, "_dgl_missing", True)
    importable_dgl("found = True\n")
    assert sampling._dgl() is None
    _loader(sampling, monkeypatch)
    assert sampling._dgl().found


def test_no_stub_is_left_behind():
    assert not hasattr(sys.modules.get("dgl"), "found")
