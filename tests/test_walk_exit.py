"""The walk kernels' early exit (CPU, on the kernels' source): the overflow
and pause flags are raised by workgroups of the same launch, so a workgroup
that starts meanwhile takes them from one thread, behind a barrier, and
leaves or stays as a whole. A timing of workgroups that would show the
opposite is not something a test can ask of the device."""

from __future__ import annotations

import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "yggdrax_amd", "csrc", "ygg_walk_flat.hip")


def _functions():
    """name -> body of every device function and kernel, comments removed."""
    text = re.sub(r"/\*.*?\*/", " ", open(SOURCE).read(), flags=re.S)
    text = re.sub(r"//[^\n]*", " ", text)
    out = {}
    for m in re.finditer(r"\b(__global__|__device__)\b[^;{]*?\b(\w+)\s*\(", text):
        brace = text.index("{", m.end())
        depth, i = 0, brace
        while True:
            depth += {"{": 1, "}": -1}.get(text[i], 0)
            i += 1
            if depth == 0:
                break
        name = re.search(r"(\w+)\s*\((?:[^()]|\([^()]*\))*\)\s*$", text[m.start():brace])
        out[name.group(1) if name else m.group(2)] = text[brace:i]
    return out



def test_one_thread_reads_the_flags_for_its_workgroup():
    body = _functions()["walk_stopped"]
    guard = body.index("if (threadIdx.x == 0)")
    barrier = body.index("__syncthreads()")
    loads = [m.start() for m in re.finditer(r"atomic_load_agent\(&a\.flags", body)]
    assert len(loads) == 4
    assert all(guard < at < body.index(";", guard) < barrier for at in loads)
    assert body.index("return s_stop") > barrier


@pytest.mark.parametrize("kernel", ["k_walk_flat", "k_walk_persist"])
def test_kernels_leave_by_the_shared_word(kernel):
    body = _functions()[kernel]
    assert "if (walk_stopped(a, sh.stop)) return;" in body
    assert not re.search(r"atomic_load_agent\(&a\.flags", body)
