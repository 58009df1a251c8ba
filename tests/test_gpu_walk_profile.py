"""Launch shapes of the flat walk from the previous walk's generation
profile (ygg_walk_flat's gen_pairs_hint): a profile only sizes the grids
and the first batch of launches, so the lists stay those of the oracle
with no profile, with the true profile, and with a profile that is far
too small (one launch of few workgroups then runs every generation) or too
short (generations past it go by the bound and the tree's size alone), or
names every third generation a large one (launches between generations that
one launch runs together)."""

from __future__ import annotations

import ctypes

import pytest
import torch

import oracle
from tests import parity
from yggdrax_amd import inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import yggdrax_amd as ygg
    pos, mass = inputs.clustered(1 << 16, 11)
    ref = oracle.build_octree(pos, mass, leaf_size=16)
    rgeom = oracle.compute_tree_geometry(ref, ref["positions_sorted"])
    rint, rnb, _ = oracle.build_interactions_and_neighbors(ref, rgeom, theta=0.5,
                                                            mac_type="dehnen")
    tree, ps, _, _ = ygg.build_octree(torch.from_numpy(pos).cuda(), torch.from_numpy(mass).cuda(),
                                      leaf_size=16, return_reordered=True)
    geom = ygg.compute_tree_geometry(tree, ps)
    return ygg, tree, geom, rint, rnb


@pytest.mark.parametrize("profile", ["none", "true", "tiny", "short", "mixed"])
def test_walk_profile_keeps_the_lists(case, monkeypatch, profile):
    from yggdrax_amd import interactions as I
    ygg, tree, geom, rint, rnb = case
    print(f"[walk profile] {profile}", flush=True)
    monkeypatch.setattr(I, "_GEN_PROFILES", type(I._GEN_PROFILES)())
    kw = dict(theta=0.5, mac_type="dehnen")
    if profile != "none":
        ygg.build_interactions_and_neighbors(tree, geom, **kw)  # records the profile
        torch.cuda.synchronize()
        assert len(I._GEN_PROFILES) == 1
        (key, (prof, arr)), = I._GEN_PROFILES.items()
        assert prof[-1] == 0 and max(prof) > 10_000 and list(arr[:len(prof)]) == prof
        if profile == "tiny":
            for k in range(len(prof)):
                arr[k] = 1
        elif profile == "mixed":
            for k in range(0, len(prof), 3):
                arr[k] = 1 << 24
        elif profile == "short":
            for k in range(len(prof) // 3, len(prof)):
                arr[k] = 0xFFFFFFFF
    inter, nbrs = ygg.build_interactions_and_neighbors(tree, geom, **kw)
    torch.cuda.synchronize()
    parity.assert_interactions_equal(inter, rint)
    parity.assert_neighbors_equal(nbrs, rnb)


@pytest.mark.parametrize("polls", [0, 1, 1 << 20])
def test_a_wait_that_runs_out_is_no_overflow(case, monkeypatch, polls):
    """A workgroup that stops waiting for a generation leaves no result: the
    walk is repeated with one launch per generation, at the same queue."""
    from yggdrax_amd import _lib
    from yggdrax_amd import interactions as I
    ygg, tree, geom, rint, rnb = case
    print(f"[walk wait] polls={polls}", flush=True)
    monkeypatch.setattr(I, "_GEN_PROFILES", type(I._GEN_PROFILES)())
    real, calls = _lib.load(), []

    class Lib:
        def __getattr__(self, name):
            return getattr(real, name)

        def ygg_walk_flat(self, p, host_status, ngen, gen_ms, stream):
            again = ctypes.c_int32(-1)
            rc = real.ygg_walk_flat_polls(p, host_status, ngen, gen_ms, polls,
                                          ctypes.byref(again), stream)
            calls.append(again.value)
            return rc

    monkeypatch.setattr(_lib, "load", lambda: Lib())
    inter, nbrs = ygg.build_interactions_and_neighbors(tree, geom, theta=0.5, mac_type="dehnen")
    torch.cuda.synchronize()
    parity.assert_interactions_equal(inter, rint)
    parity.assert_neighbors_equal(nbrs, rnb)
    assert len(calls) == 1  # one walk: no larger queue was tried
    assert calls[0] == (1 if polls == 0 else 0 if polls > 1 else calls[0])


@pytest.fixture(scope="module")
def wide_case():
    """A small tree whose wavefront grows past 196608 pairs (small theta)."""
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import yggdrax_amd as ygg
    pos, mass = inputs.plummer_sphere(8192, 3)
    ref = oracle.build_tree(pos, mass, leaf_size=4)
    rgeom = oracle.compute_tree_geometry(ref, ref["positions_sorted"])
    rint, rnb, _ = oracle.build_interactions_and_neighbors(ref, rgeom, theta=0.2,
                                                            mac_type="dehnen")
    tree, ps, _, _ = ygg.build_tree(torch.from_numpy(pos).cuda(), torch.from_numpy(mass).cuda(),
                                    leaf_size=4, return_reordered=True)
    return ygg, tree, ygg.compute_tree_geometry(tree, ps), rint, rnb


@pytest.mark.parametrize("profile", ["none", "true", "tiny", "late"])
def test_generations_too_large_for_one_launch(wide_case, monkeypatch, profile):
    """Generations of small trees, or hinted as small, that turn out large
    leave the launch that runs many: where the wavefront grows past the bound
    of 64 workgroups (none) or of 16 (tiny), or at the launch's first
    generation (late)."""
    from yggdrax_amd import interactions as I
    ygg, tree, geom, rint, rnb = wide_case
    print(f"[walk hand-back] {profile}", flush=True)
    monkeypatch.setattr(I, "_GEN_PROFILES", type(I._GEN_PROFILES)())
    kw = dict(theta=0.2, mac_type="dehnen")
    if profile != "none":
        ygg.build_interactions_and_neighbors(tree, geom, **kw)
        (key, (prof, arr)), = I._GEN_PROFILES.items()
        assert max(prof) > 196608 > prof[0]
        big = max(range(len(prof)), key=lambda k: prof[k])
        if profile == "tiny":
            for k in range(len(prof)):
                arr[k] = 1
        elif profile == "late":
            for k in range(len(prof)):
                arr[k] = 1 << 20 if k < big else 1
    inter, nbrs = ygg.build_interactions_and_neighbors(tree, geom, **kw)
    torch.cuda.synchronize()
    parity.assert_interactions_equal(inter, rint)
    parity.assert_neighbors_equal(nbrs, rnb)
