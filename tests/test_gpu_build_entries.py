"""C-ABI build helpers called directly: the one-launch int32 -> int64
widening and the two-stream Morton sort + reorder, each against the plain
form of the same computation."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from yggdrax_amd import _lib, inputs

pytestmark = pytest.mark.gpu


def test_widen_many_arrays_one_launch():
    lib = _lib.load()
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(5)
    sizes = [0, 1, 255, 256, 257, 70001, 1 << 20, 3]
    srcs = [torch.randint(-(1 << 31), (1 << 31) - 1, (n,), generator=g, device=dev,
                          dtype=torch.int32) for n in sizes]
    dsts = [torch.full((n,), -7, dtype=torch.int64, device=dev) for n in sizes]
    items = (_lib.WidenItem * len(sizes))()
    for k, (s, d) in enumerate(zip(srcs, dsts)):
        items[k].src = s.data_ptr() if s.numel() else None
        items[k].dst = d.data_ptr() if d.numel() else None
        items[k].n = s.numel()
    _lib.check(lib.ygg_widen_i32_to_i64(items, len(sizes), _lib.stream_ptr(dev)), "widen")
    torch.cuda.synchronize()
    for s, d in zip(srcs, dsts):
        assert torch.equal(d, s.to(torch.int64))


def test_widen_rejects_bad_arguments():
    lib = _lib.load()
    st = _lib.stream_ptr(torch.device("cuda"))
    too_many = (_lib.WidenItem * (_lib.WIDEN_MAX_ITEMS + 1))()
    assert lib.ygg_widen_i32_to_i64(too_many, _lib.WIDEN_MAX_ITEMS + 1, st) != 0
    bad = (_lib.WidenItem * 1)()
    bad[0].src, bad[0].dst, bad[0].n = None, None, 5  # non-empty item without buffers
    assert lib.ygg_widen_i32_to_i64(bad, 1, st) != 0
    neg = (_lib.WidenItem * 1)()
    neg[0].n = -1
    assert lib.ygg_widen_i32_to_i64(neg, 1, st) != 0


@pytest.mark.parametrize("n", [1, 4097, 1 << 20])
def test_sort_reorder_async_matches_one_stream(n):
    """The two-stream entry gives the one-stream entry's codes, permutation,
    reordered particles and inverse, bit for bit (clustered points)."""
    lib = _lib.load()
    dev = torch.device("cuda")
    pos_np, mass_np = inputs.clustered(n, 7) if n >= 64 else inputs.uniform_cube(n, 7)
    pos = torch.from_numpy(np.ascontiguousarray(pos_np)).to(dev)
    mass = torch.from_numpy(np.ascontiguousarray(mass_np)).to(dev)
    b6 = torch.empty(6, dtype=torch.float32, device=dev)
    bws = torch.empty(256, dtype=torch.uint8, device=dev)
    st = _lib.stream_ptr(dev)
    _lib.check(lib.ygg_infer_bounds(pos.data_ptr(), n, b6.data_ptr(), bws.data_ptr(), 256, st),
               "bounds")
    nbytes = lib.ygg_morton_sort_reorder_workspace_bytes(n)

    def run(side):
        codes = torch.empty(n, dtype=torch.int64, device=dev)
        perm = torch.empty(n, dtype=torch.int32, device=dev)
        ps = torch.empty_like(pos)
        ms = torch.empty_like(mass)
        inv = torch.empty(n, dtype=torch.int64, device=dev)
        ws = _lib.workspace(nbytes, dev)
        args = (pos.data_ptr(), mass.data_ptr(), n, b6.data_ptr(), codes.data_ptr(),
                perm.data_ptr(), ps.data_ptr(), ms.data_ptr(), inv.data_ptr(), 1,
                ws.data_ptr(), ws.numel(), st)
        if side is None:
            _lib.check(lib.ygg_morton_sort_reorder(*args), "sort reorder")
        else:
            _lib.check(lib.ygg_morton_sort_reorder_async(*args, side.cuda_stream),
                       "sort reorder async")
            torch.cuda.current_stream(dev).wait_stream(side)
        torch.cuda.synchronize()
        return codes, perm, ps, ms, inv

    side = torch.cuda.Stream(device=dev)
    ref = run(None)
    got = run(side)
    for a, b in zip(ref, got):
        assert torch.equal(a, b)
    perm = ref[1].long()
    assert torch.equal(ref[2], pos[perm]) and torch.equal(ref[3], mass[perm])
    assert torch.equal(ref[4][perm], torch.arange(n, device=dev))
    assert lib.ygg_morton_sort_reorder_async(
        pos.data_ptr(), mass.data_ptr(), n, b6.data_ptr(), None, None, None, None, None, 1,
        None, 0, st, None) != 0  # no second stream
    print("async reorder n", n, flush=True)


def test_widen_item_layout():
    assert ctypes.sizeof(_lib.WidenItem) == 24


@pytest.mark.parametrize("n", [1, 1023, 12288, 12289, 16384, 16385, (1 << 17) - 1, 1 << 17])
def test_sort_and_bounds_at_path_edges(n):
    """Bounds of aligned and unaligned positions by one workgroup and by many,
    codes with and without digit histograms, the inverse with the gather and
    apart: against numpy."""
    import yggdrax_amd as ygg
    print(f"[build entries] edges n={n}", flush=True)
    rng = np.random.default_rng(n)
    host = rng.normal(size=(n + 1, 3)).astype(np.float32)
    mass = torch.from_numpy(rng.random(n, dtype=np.float32)).cuda()
    both = torch.from_numpy(host).cuda()
    for pos, h in ((both[:n].clone(), host[:n]), (both[1:], host[1:])):
        lo, hi = ygg.infer_bounds(pos)
        span = h.max(0) - h.min(0)
        pad = np.maximum(span * np.float32(0.05), np.float32(1e-6))
        assert np.array_equal(lo.cpu().numpy(), h.min(0) - pad)
        assert np.array_equal(hi.cpu().numpy(), h.max(0) + pad)
        tree, ps, ms, inv = ygg.build_tree(pos, mass, return_reordered=True, leaf_size=8)
        codes = ygg.morton_encode(pos, (lo, hi)).view(torch.int64).cpu().numpy()
        perm = np.argsort(codes, kind="stable")  # 63-bit codes: no sign
        assert np.array_equal(tree.particle_indices.cpu().numpy(), perm)
        assert np.array_equal(ps.cpu().numpy(), h[perm])
        assert np.array_equal(ms.cpu().numpy(), mass.cpu().numpy()[perm])
        assert np.array_equal(inv.cpu().numpy(), np.argsort(perm))
