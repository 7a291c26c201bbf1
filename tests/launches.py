"""Which kernels a call launches: what a dispatch rule chose, where two kernels give
the same bits and the test is about the choice."""

from __future__ import annotations

import json

import torch
from torch.profiler import ProfilerActivity, profile


def launches(call, tmp_path) -> list[tuple[str, int]]:
    """(kernel name, workgroups along x) of this package's kernels, in the order of their launch."""
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    path = tmp_path / "trace.json"
    p.export_chrome_trace(str(path))
    events = [e for e in json.loads(path.read_text())["traceEvents"] if e.get("cat") == "kernel" and "fmx::" in e["name"]]
    assert events, "no kernel of this package in the trace"
    return [(e["name"], e["args"]["grid"][0]) for e in sorted(events, key=lambda e: e["ts"])]
