"""Which kernels a call launches, from the graph that a capture of it makes."""
from __future__ import annotations

import re
import tempfile
import warnings
from pathlib import Path

import pytest
import torch


def kernels(call) -> list[str]:
    """The names of this library's kernels in one call, in launch order."""
    from rwkv7mi.model import graph_capture

    call()  # grows the workspaces
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    g.enable_debug_mode()
    with graph_capture(g):
        call()
    with tempfile.TemporaryDirectory() as d:
        dot = Path(d) / "graph.dot"
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")  # (torch announces the dump)
            g.debug_dump(str(dot))
        if not dot.exists():
            pytest.skip("this runtime does not print graphs")
        text = dot.read_text()
    return [m[2][:int(m[1])] for m in re.finditer(r"_ZN7rwkv7mi(\d+)(\w+)", text)]
