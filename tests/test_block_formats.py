"""Blocks without DGL are plain tuples; a DGL that turns up later is used from then on."""
import sys
import threading
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
    a, b = torch.tensor([0, 2]), torch.tensor([1, 0])
    for _ in range(2):
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


def _is_csc(sampling):
    block = sampling.create_block_from_csc(torch.tensor([0, 2]), torch.tensor([1, 0]), torch.Tensor(), 2, 1)
    return isinstance(block, sampling.CSCBlock)


STUB = """
import sys, threading, types
if hasattr(sys, "_stub_gate"):
    sys._stub_gate[0].set()
    sys._stub_gate[1].wait(30)
__path__ = []
class DGLBlock:
    def __init__(self, *args): pass
heterograph = types.ModuleType("dgl.heterograph")
heterograph.DGLBlock = DGLBlock
sys.modules["dgl.heterograph"] = heterograph
heterograph_index = types.SimpleNamespace(create_unitgraph_from_csr=lambda *a, **k: "csr")
found = True
"""


def _sampling():
    import shmtensor_amd
    shmtensor_amd.install_aliases()
    from shmtensor_amd.shmtensor import sampling
    return sampling


def test_functions_look_for_a_dgl_every_time(importable_dgl):
    """A dgl that becomes importable after a failed look is used by the next block, without a new loader."""
    sampling = _sampling()
    assert _is_csc(sampling)
    importable_dgl(STUB)
    assert not _is_csc(sampling)


def test_a_loader_looks_once_and_when_the_path_changes(monkeypatch, importable_dgl):
    sampling = _sampling()
    searches = []

    class Finder:
        @staticmethod
        def find_spec(name, *_):
            if name == "dgl":
                searches.append(name)

    monkeypatch.setattr(sys, "meta_path", [Finder] + sys.meta_path)
    hop = (torch.tensor([0, 1]), None, torch.tensor([0, 1]), torch.tensor([1]))
    monkeypatch.setattr(sampling.capi, "sample_blocks", lambda *a, **k: [[hop]])
    loader = _loader(sampling, monkeypatch)
    assert len(searches) == 1
    for _ in range(3):
        assert isinstance(loader._sample_group(0, 1, 0)[0][2][0], sampling.CSCBlock)
    assert len(searches) == 1
    importable_dgl(STUB)
    assert not isinstance(loader._sample_group(0, 1, 0)[0][2][0], sampling.CSCBlock)


def test_a_dgl_that_is_being_imported_is_waited_for(importable_dgl, monkeypatch):
    """A thread that builds blocks while another one is in the middle of importing dgl gets the whole module."""
    sampling = _sampling()
    assert _is_csc(sampling)
    begun, go = threading.Event(), threading.Event()
    monkeypatch.setattr(sys, "_stub_gate", (begun, go), raising=False)
    importable_dgl(STUB)
    results = []

    def build():
        try:
            results.append(_is_csc(sampling))
        except Exception as exc:
            results.append(exc)

    threads = [threading.Thread(target=lambda: __import__("dgl"), daemon=True), threading.Thread(target=build, daemon=True)]
    threads[0].start()
    assert begun.wait(30)
    threads[1].start()
    threads[1].join(0.5)
    assert results == []          # (waits for the import)
    go.set()
    for t in threads:
        t.join(30)
    assert results == [False]


def test_no_stub_is_left_behind():
    assert not hasattr(sys.modules.get("dgl"), "found")
