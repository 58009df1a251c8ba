"""The walk's node records (ygg_walk_prepare_nodes): every node has one,
also under a level order that names some node twice and leaves another out
(a caller's own topology), whose rank is then 0."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from yggdrax_amd import _lib
from yggdrax_amd.interactions import NODE_RECORD_BYTES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["none", "permutation", "repeated"])
@pytest.mark.parametrize("L", [2, 700])
def test_every_node_has_a_record(L, order):
    lib = _lib.load()
    dev = torch.device("cuda")
    T, NI = 2 * L - 1, L - 1
    print(f"[node records] T={T} order={order}", flush=True)
    rng = np.random.default_rng(T)
    center = rng.normal(size=(T, 3)).astype(np.float32)
    radius, extent = (rng.uniform(0.1, 1.0, T).astype(np.float32) for _ in range(2))
    left, right = (rng.integers(0, T, NI).astype(np.int32) for _ in range(2))
    leaf_pos = np.concatenate([np.full(NI, -1), rng.permutation(L)]).astype(np.int32)
    nbl = rng.permutation(T).astype(np.int32)
    left_out = int(nbl[1])
    if order == "repeated":
        nbl[1] = nbl[0]
    t = {k: torch.from_numpy(v).to(dev) for k, v in dict(
        center=center, radius=radius, extent=extent, left=left, right=right, leaf_pos=leaf_pos,
        nbl=nbl).items()}
    out = torch.full((T * NODE_RECORD_BYTES,), 0x5A, dtype=torch.uint8, device=dev)
    _lib.check(lib.ygg_walk_prepare_nodes(
        t["center"].data_ptr(), t["radius"].data_ptr(), t["extent"].data_ptr(),
        t["left"].data_ptr(), t["right"].data_ptr(), t["leaf_pos"].data_ptr(),
        None if order == "none" else t["nbl"].data_ptr(), T, 0, 1.0, out.data_ptr(),
        _lib.stream_ptr(dev)), "prepare nodes")
    rec = out.cpu().numpy().reshape(T, NODE_RECORD_BYTES)
    f, i = rec[:, :16].copy().view(np.float32), rec[:, 16:].copy().view(np.int32)
    assert np.array_equal(f[:, :3], center) and np.array_equal(f[:, 3], extent)
    none = np.full(L, -1)
    assert np.array_equal(i[:, 0], np.concatenate([left, none]))
    assert np.array_equal(i[:, 1], np.concatenate([right, none]))
    assert np.array_equal(i[:, 2], leaf_pos)
    if order == "permutation":
        assert np.array_equal(i[nbl, 3], np.arange(T))
    elif order == "none":
        assert not i[:, 3].any()
    else:
        assert i[left_out, 3] == 0 and np.array_equal(i[nbl[2:], 3], np.arange(2, T))
