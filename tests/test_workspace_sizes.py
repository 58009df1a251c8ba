"""Workspace queries do not shrink as n grows, so that a caller who sizes one
workspace for the largest n can use it for every smaller one; and a sort
just below a change of tile runs in a workspace sized just above it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from yggdrax_amd import _lib

# where the sort changes its kernel or tile (12288 pairs, 3 * 2^16, 3 * 2^19),
# and where the room at those is caught up with again
EDGES = [1, 1024, 4096, 8192, 12288, 16384, 3 << 16, 4 << 16, 3 << 19, 4 << 19, 1 << 24]


def _sizes():
    out = set()
    for e in EDGES:
        out.update(n for n in range(e - 3, e + 4) if n > 0)
        out.update(int(e * f) for f in np.linspace(1.0, 1.4, 41))
    return sorted(out)


QUERIES = {
    "morton_sort": lambda lib, n: lib.ygg_morton_sort_workspace_bytes(n),
    "morton_sort_reorder": lambda lib, n: lib.ygg_morton_sort_reorder_workspace_bytes(n),
    "grouped": lambda lib, n: lib.ygg_grouped_workspace_bytes(n),
    "scan": lambda lib, n: lib.ygg_scan_workspace_bytes(n),
    "octree_meta": lambda lib, n: lib.ygg_octree_meta_workspace_bytes(n),
    "radix_build": lambda lib, n: lib.ygg_radix_build_workspace_bytes(n, 1),
}
for _kb, _bits in ((4, 18), (4, 32), (8, 9), (8, 37), (8, 63), (8, 64)):
    for _d in (0, 8, 9, 10, 11):
        QUERIES[f"sort{8 * _kb}_{_bits}bits_d{_d}"] = (
            lambda lib, n, kb=_kb, b=_bits, d=_d: lib.ygg_sort_workspace_bytes(n, kb, 0, b, d))


@pytest.mark.parametrize("name", list(QUERIES))
def test_workspace_never_shrinks(name):
    lib = _lib.load()
    last = 0
    for n in _sizes():
        need = QUERIES[name](lib, n)
        assert need >= last, (name, n, need, last)
        last = need


@pytest.mark.gpu
@pytest.mark.parametrize("n,sized_for", [(3 << 16, (3 << 16) + 1), (3 << 16, 200000),
                                         (12288, 12289), (12289, 12289),
                                         ((3 << 16) + 1, (3 << 16) + 1),
                                         (3 << 19, (3 << 19) + 1),
                                         ((3 << 19) + 1, (3 << 19) + 1)])
def test_sort_in_a_workspace_of_a_larger_one(n, sized_for):
    lib = _lib.load()
    dev = torch.device("cuda")
    print(f"[workspace] n={n} sized_for={sized_for}", flush=True)
    g = torch.Generator(device=dev).manual_seed(n)
    keys = torch.randint(0, 1 << 62, (n,), generator=g, device=dev, dtype=torch.int64)
    keys[::7] = keys[0]
    out = torch.empty_like(keys)
    order = torch.empty(n, dtype=torch.int32, device=dev)
    ws = torch.empty(lib.ygg_sort_workspace_bytes(sized_for, 8, 0, 63, 9), dtype=torch.uint8,
                     device=dev)
    _lib.check(lib.ygg_sort_pairs_u64(keys.data_ptr(), None, out.data_ptr(), order.data_ptr(), n,
                                      0, 63, 9, ws.data_ptr(), ws.numel(), _lib.stream_ptr(dev)),
               "sort")
    want, at = torch.sort(keys, stable=True)
    assert torch.equal(out, want) and torch.equal(order.long(), at)
