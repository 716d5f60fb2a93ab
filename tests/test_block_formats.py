"""Blocks without DGL are plain tuples; a DGL that turns up later is used from then on."""
import sys
import types

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


def test_a_new_loader_looks_again(monkeypatch, tmp_path):
    import shmtensor_amd
    shmtensor_amd.install_aliases()
    from shmtensor_amd.shmtensor import sampling
    monkeypatch.delitem(sys.modules, "dgl", raising=False)
    monkeypatch.setattr(sampling, "_dgl_missing", True)
    (tmp_path / "dgl.py").write_text("found = True\n")
    monkeypatch.syspath_prepend(str(tmp_path))
    assert sampling._dgl() is None
    assert sampling._dgl(look_again=True).found
    monkeypatch.delitem(sys.modules, "dgl")
