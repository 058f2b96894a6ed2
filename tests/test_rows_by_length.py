"""The order of rows that a graph keeps for the GAT layer over its inputs (DGLGraph.rows_by_length):
when it is handed out, and what a failed build leaves.  The device is played by a stand-in."""
import ctypes
import types

import pytest
import torch

from graphiler_amd import capi, graph


class _Device:
    """The library and the stream of a build, as a list of what was done in which order."""

    def __init__(self, n_light):
        self.done, self.n_light, self.cuda_stream = [], n_light, 0

    def synchronize(self):
        self.done.append("waited")

    def ga_gat_rows_longest(self, n_edges):
        return 2

    def ga_gat_rows_workspace_bytes(self, n, longest):
        return 256

    def ga_gat_rows_build(self, pointer, n, longest, rows, light, *rest):
        ctypes.c_int32.from_address(light).value = self.n_light
        self.done.append("rows")
        return 0

    def ga_gat_pieces_build(self, *args):
        self.done.append("pieces")
        return 0


def _graph(monkeypatch, n_light):
    dev = _Device(n_light)
    monkeypatch.setattr(capi, "load", lambda: dev)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: dev)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    i = lambda *v: torch.tensor(v, dtype=torch.int32)
    coo = torch.zeros(4, dtype=torch.int64)
    g = graph.DGLGraph(i(0, 3, 4), i(0, 0, 0, 0), i(0, 1, 2, 3), i(0, 4, 4), i(0, 0, 0, 1), i(0, 1, 2, 3),
                       coo, coo.clone())
    return g, dev


@pytest.mark.parametrize("n_light", [1, 2])
def test_pieces_are_there_when_the_order_is_kept(monkeypatch, n_light):
    """A call on another stream takes the kept order without asking: nothing of it may be in flight."""
    g, dev = _graph(monkeypatch, n_light)
    assert g.rows_by_length() is g.rows_by_length()
    assert dev.done == (["rows", "pieces", "waited"] if n_light < 2 else ["rows"])


def test_an_order_that_did_not_fit_is_tried_again(monkeypatch):
    g, dev = _graph(monkeypatch, 2)
    build = dev.ga_gat_rows_workspace_bytes

    def full(*args):
        raise torch.OutOfMemoryError("full")
    dev.ga_gat_rows_workspace_bytes = full
    assert g.rows_by_length() is None
    dev.ga_gat_rows_workspace_bytes = build
    assert g.rows_by_length() is not None
