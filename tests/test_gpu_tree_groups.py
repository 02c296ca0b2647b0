"""Colleagues and lists with 32 lanes a box at the edges: trees of one, two and
a few boxes, piles of points that refine next to coarse leaves down to the
deepest levels (lists over many levels), targets far from most sources; array
for array against the host builder."""

import numpy as np
import pytest

import test_gpu_tree
from sumpy_amd.tree import build_tree_and_traversal
from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu

pytestmark = pytest.mark.gpu


def _pile(dim, n, depth, rng):
    """n points at distances 2^-1 ... 2^-depth from an off-centre point."""
    d = rng.standard_normal((dim, n))
    return 0.3 + 0.5*2.0**-rng.uniform(0, depth, n)*d/np.linalg.norm(d, axis=0)


@pytest.mark.parametrize(("dim", "n", "depth", "mpb"), [
    (3, 1, 1, 1), (3, 2, 1, 1), (3, 9, 1, 1), (2, 5, 1, 1), (3, 4000, 9, 8), (3, 4000, 17, 3),
    (2, 3000, 26, 2), (2, 500, 12, 20)])
@pytest.mark.parametrize("targets", [False, True])
def test_group_lists(actx, dim, n, depth, mpb, targets):
    rng = np.random.default_rng(n + depth)
    src = _pile(dim, n, depth, rng)
    tgt = rng.random((dim, n//2 + 1)) if targets else None
    host = build_tree_and_traversal(actx, src, tgt, mpb)
    gpu = build_tree_and_traversal_gpu(actx, src, tgt, mpb)
    both = ("pile", src, tgt, mpb, host, gpu)
    test_gpu_tree.test_tree_arrays_equal_host_builder(both)
    test_gpu_tree.test_traversal_arrays_equal_host_builder(both)


@pytest.mark.parametrize(("dim", "n", "depth", "mpb"), [
    (3, 1, 1, 1), (3, 9, 1, 1), (3, 4000, 9, 8), (2, 500, 12, 20)])
def test_lists_1_and_4_without_the_colleagues(actx, monkeypatch, dim, n, depth, mpb):
    """A caller of the C entry may pass no colleagues for these two lists."""
    from sumpy_amd import _capi
    rng = np.random.default_rng(n + depth)
    src, tgt = _pile(dim, n, depth, rng), rng.random((dim, n//2 + 1))
    host = build_tree_and_traversal(actx, src, tgt, mpb)
    call, without = _capi.call, []

    def no_colleagues(name, *args):
        if name == "sumpytree_gpu_list" and args[0] in (1, 4):
            without.append(args[13])
            args = (*args[:13], None, *args[14:])
        call(name, *args)

    monkeypatch.setattr(_capi, "call", no_colleagues)
    gpu = build_tree_and_traversal_gpu(actx, src, tgt, mpb)
    assert without and all(without)
    test_gpu_tree.test_traversal_arrays_equal_host_builder(("pile", src, tgt, mpb, host, gpu))
