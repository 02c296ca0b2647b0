"""Which multipole arrays and wranglers the folded M2L takes: those whose memory
the kernels may read as rows of all boxes.  The others go to the class matrices,
which accept or refuse them."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from sumpy_amd import _capi, m2l_fold
from sumpy_amd.expansion.local import LinearPDEConformingVolumeTaylorLocalExpansion
from sumpy_amd.expansion.m2l import VolumeTaylorM2LWithDenseClassMatrices
from sumpy_amd.expansion.multipole import LinearPDEConformingVolumeTaylorMultipoleExpansion
from sumpy_amd.kernel import HelmholtzKernel, LaplaceKernel

ORDER, NBOXES = 3, 5


def _wrangler(knl, dtype):
    tr = VolumeTaylorM2LWithDenseClassMatrices("fp64")
    ti = SimpleNamespace(
        m2l_translation=tr, get_base_kernel=lambda: knl,
        multipole_expansion=lambda p: LinearPDEConformingVolumeTaylorMultipoleExpansion(knl, p),
        local_expansion=lambda p: LinearPDEConformingVolumeTaylorLocalExpansion(knl, p))
    starts = np.array([0, NBOXES*(ORDER + 1)**2])
    return SimpleNamespace(tree_indep=ti, dtype=np.dtype(dtype),
                           tree=SimpleNamespace(nboxes=NBOXES),
                           multipole_expansions_level_starts=lambda: starts)


@pytest.mark.parametrize("cplx", [False, True])
def test_folded_m2l_takes_plain_arrays_only(cplx):
    wr = _wrangler(HelmholtzKernel(3) if cplx else LaplaceKernel(3), "c16" if cplx else "f8")
    n = NBOXES*(ORDER + 1)**2
    good = torch.ones(n, dtype=torch.complex128 if cplx else torch.float64)
    assert m2l_fold.takes(wr, good)
    other = good.real.contiguous() if cplx else good.to(torch.complex128)
    for bad in (other, good[1:], torch.cat([good, good]), torch.cat([good, good])[::2],
                good.to(torch.complex64 if cplx else torch.float32), torch._neg_view(good),
                torch.complex(good.real, good.real).conj(), good.reshape(NBOXES, -1)):
        assert not m2l_fold.takes(wr, bad)


def test_folded_m2l_wants_the_kernels_dtype():
    """A complex wrangler of a real kernel has real class data, a real one of a
    complex kernel complex class data."""
    lap, helm = LaplaceKernel(3), HelmholtzKernel(3)
    assert m2l_fold.usable(_wrangler(lap, "f8"), ORDER)
    assert m2l_fold.usable(_wrangler(helm, "c16"), ORDER)
    assert not m2l_fold.usable(_wrangler(lap, "c16"), ORDER)
    assert not m2l_fold.usable(_wrangler(helm, "f8"), ORDER)


def test_fold_entry_points_check_row_sizes():
    """Rows of another order are refused before anything is launched."""
    null = [None]*12
    with pytest.raises(ValueError, match="coefficients"):
        _capi.call("sumpyhip_m2l_fold_apply", 0, 0, ORDER, 1, 1, 0, 1, 25, *null, 0, 1, 1,
                   None, None, None)
    with pytest.raises(ValueError, match="row"):
        _capi.call("sumpyhip_m2l_fold_pack", 0, 0, 1, 0, 24, None, None, None, None)
    with pytest.raises(ValueError, match="row"):
        _capi.call("sumpyhip_m2l_fold_pack", 0, 0, 1, 16, 20, None, None, None, None)


def test_folded_m2l_takes_whole_levels():
    """Levels may be left out; a caller's part of a level's target boxes goes to
    the class matrices (the plan holds all of them)."""
    import test_gpu_m2l_fold as t
    from sumpy_amd.array_context import TorchArrayContext
    from sumpy_amd.tree import build_tree_and_traversal
    actx = TorchArrayContext("cpu")
    tree, trav = build_tree_and_traversal(actx, np.random.default_rng(0).random((3, 3000)),
                                          None, 20)
    wr = t._wrangler(actx, trav, ORDER, "fp64", None)
    lists = (trav.target_or_target_parent_boxes, trav.from_sep_siblings_starts,
             trav.from_sep_siblings_lists)
    own = trav.host["level_start_target_or_target_parent_box_nrs"]
    levels = [lev for _, run in m2l_fold.runs(wr, own, *lists) for lev in run]
    assert len(levels) >= 2
    lev = levels[-1]
    without = np.array(own)
    without[lev + 1:] = own[lev]
    assert [lv for _, run in m2l_fold.runs(wr, without, *lists) for lv in run] == levels[:-1]
    part = np.array(own)
    part[lev + 1:] -= 1
    assert m2l_fold.runs(wr, part, *lists) is None


@pytest.mark.gpu
@pytest.mark.parametrize("cplx", [False, True])
def test_folded_m2l_and_other_arrays(actx, cplx):
    """What the class matrices do with the arrays that the folded form leaves to
    them: a strided complex array is translated like its copy, real multipoles of a
    complex kernel like complex ones; strided real arrays, conjugated views, short
    arrays and other precisions are refused."""
    import test_gpu_m2l_fold as t
    from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu
    rng = np.random.default_rng(5)
    pts = torch.from_numpy(rng.random((3, 3000))).to(actx.device)
    _, trav = build_tree_and_traversal_gpu(actx, pts, None, 30)
    wr = t._wrangler(actx, trav, 6, "fp64", 4.0 if cplx else None)
    m = t._random_mpoles(wr, actx, rng)
    want = t._m2l(actx, wr, m)
    scale = want.abs().max()
    strided = torch.stack([m, m], dim=1)[:, 0]
    with pytest.raises(RuntimeError):
        t._m2l(actx, wr, m[:-1])
    if cplx:
        assert (t._m2l(actx, wr, strided) - want).abs().max() < 1e-12*scale
        re = m.real.contiguous()
        want = t._m2l(actx, wr, re.to(torch.complex128))
        assert (t._m2l(actx, wr, re) - want).abs().max() < 1e-12*scale
        with pytest.raises(RuntimeError, match="conjugat"):
            t._m2l(actx, wr, m.conj())
        with pytest.raises(TypeError):
            t._m2l(actx, wr, m.to(torch.complex64))
    else:
        with pytest.raises(ValueError, match="contiguous"):
            t._m2l(actx, wr, strided)
        with pytest.raises(TypeError):
            t._m2l(actx, wr, m.float())


@pytest.mark.gpu
def test_folded_m2l_after_a_change_of_the_lists(actx, monkeypatch):
    """A pair's source box replaced in the traversal's list, in place or by a new
    array: the plan is made again, the result is the class matrices'."""
    import test_gpu_m2l_fold as t
    from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu
    rng = np.random.default_rng(6)
    pts = torch.from_numpy(rng.random((3, 3000))).to(actx.device)
    tree, trav = build_tree_and_traversal_gpu(actx, pts, None, 30)
    wr = t._wrangler(actx, trav, 5, "fp64", None)
    m = t._random_mpoles(wr, actx, rng)
    first = t._m2l(actx, wr, m)
    last = int(trav.from_sep_siblings_lists[-1])
    assert len(set(tree.host["box_levels"][last - 2:last + 1])) == 1
    for change in (lambda v: v[-1:].fill_(last - 1),
                   lambda v: trav.__dict__["_dev"].__setitem__(
                       "from_sep_siblings_lists", torch.cat([v[:-1], v[-1:] - 1]))):
        change(trav.from_sep_siblings_lists)
        got = t._m2l(actx, wr, m)
        with monkeypatch.context() as mp:
            mp.setattr(m2l_fold, "runs", lambda *a: None)
            want = t._m2l(actx, wr, m)
        scale = want.abs().max()
        assert (want - first).abs().max() > 1e-6*scale
        assert (got - want).abs().max() <= 1e-12*scale
        first = want
    assert len(trav.__dict__["_m2l_fold_plans"]) == 1


@pytest.mark.gpu
def test_folded_m2l_with_wide_class_numbers(actx, monkeypatch):
    """Translation classes handed in as 64-bit integers, as the class matrices
    take them."""
    import test_gpu_m2l_fold as t
    from sumpy_amd.tree import TranslationClassesData
    from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu
    rng = np.random.default_rng(7)
    pts = torch.from_numpy(rng.random((3, 3000))).to(actx.device)
    _, trav = build_tree_and_traversal_gpu(actx, pts, None, 30)
    wr = t._wrangler(actx, trav, 5, "fp64", None)
    own = wr.translation_classes_data
    wr.translation_classes_data = TranslationClassesData(
        own.from_sep_siblings_translation_classes.long(),
        own.from_sep_siblings_translation_class_to_distance_vector,
        own.from_sep_siblings_translation_classes_level_starts)
    m = t._random_mpoles(wr, actx, rng)
    got = t._m2l(actx, wr, m)
    with monkeypatch.context() as mp:
        mp.setattr(m2l_fold, "runs", lambda *a: None)
        want = t._m2l(actx, wr, m)
    assert (got - want).abs().max() <= 1e-12*want.abs().max()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("cplx", [False, True])
def test_workgroups_leave_a_slot_for_each(precision, cplx):
    """A workgroup's share of the cost is more than the most expensive slot, so that
    one begins in it (its partial sums are read); whole rounds past the first."""
    for order in (3, 8, 12):
        for resident in (1, 256, 768, 2048):
            for cost in [*range(0, 400, 7), 10**4, 123_457, 10**6, 10**9]:
                g = m2l_fold.workgroups(precision, cplx, order, cost, resident)
                assert 1 <= g <= 6*resident
                assert g == 1 or cost//g > m2l_fold.MAX_SLOT_COST
                assert g <= resident or g % resident == 0
                if precision == "fp64":
                    assert g == max(1, min(resident, cost//80))
