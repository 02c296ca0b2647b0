"""The M2L folded by reflection symmetry (``csrc/m2l_fold.hip``) against the
class-matrix contraction of the single-level operators, and the plan's
invariants on the CPU."""

from functools import partial

import numpy as np
import pytest
import torch

from sumpy_amd import m2l_fold


@pytest.mark.parametrize("order", range(1, 13))
def test_fold_maps_sort_by_parity(order):
    """Every stored coefficient once among the rows and the columns, parity
    classes in whole row blocks and k pairs; the sizes' order rule."""
    ax, nrb, nkp, rbs, kps = m2l_fold.sizes(order)
    row, k, par = m2l_fold.maps(order)
    n = (order + 1)**2
    assert len(row) == 16*nrb and len(k) == 8*nkp
    for m, blocks, size in ((row, rbs, 16), (k, kps, 8)):
        assert sorted(m[m >= 0]) == list(range(n))
        cls = np.repeat(np.arange(1 << ax), np.array(blocks[:1 << ax])*size)
        assert (par[m[m >= 0]] & ((1 << ax) - 1) == cls[m >= 0]).all()


@pytest.mark.parametrize("ax", range(4))
def test_fold_identity(ax):
    """sum_R A_{Rn} X_R = sum_s A_n[t, s] Xh_{par t ^ par s}[s] over every set
    of present reflections, for a matrix with the kernel's symmetry."""
    rng = np.random.default_rng(ax)
    order = 5
    par = m2l_fold.maps(order)[2]
    n, nr = len(par), 1 << ax
    A = rng.standard_normal((n, n))
    X = rng.standard_normal((nr, n))*(rng.random(nr) < 0.7)[:, None]
    sign = np.array([[(-1)**bin(R & d).count("1") for R in range(nr)] for d in range(8)])
    want = np.zeros(n)
    for R in range(nr):
        S = sign[par, R]
        want += S*(A @ (S*X[R]))
    Xh = sign[:nr] @ X
    d = (par[:, None] ^ par[None, :]) & (nr - 1)
    got = (A*Xh[d, np.arange(n)[None, :]]).sum(axis=1)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-13*np.abs(want).max()*n)


def _points(kind, n, rng):
    if kind == "uniform":
        return rng.random((3, n))
    if kind == "gaussian":
        c = rng.random((3, 8))
        return c[:, rng.integers(0, 8, n)] + 0.02*rng.standard_normal((3, n))
    x = rng.standard_normal((3, n))
    return x/np.linalg.norm(x, axis=0)


def _wrangler(actx, trav, order, precision, k):
    from sumpy_amd.expansion.local import LinearPDEConformingVolumeTaylorLocalExpansion
    from sumpy_amd.expansion.m2l import VolumeTaylorM2LWithDenseClassMatrices
    from sumpy_amd.expansion.multipole import LinearPDEConformingVolumeTaylorMultipoleExpansion
    from sumpy_amd.fmm import SumpyExpansionWrangler, SumpyTreeIndependentDataForWrangler
    from sumpy_amd.kernel import HelmholtzKernel, LaplaceKernel
    knl = LaplaceKernel(3) if k is None else HelmholtzKernel(3)
    ti = SumpyTreeIndependentDataForWrangler(
        actx, partial(LinearPDEConformingVolumeTaylorMultipoleExpansion, knl),
        partial(LinearPDEConformingVolumeTaylorLocalExpansion, knl,
                m2l_translation_override=VolumeTaylorM2LWithDenseClassMatrices(precision)),
        [knl], exclude_self=False)
    orders = order if callable(order) else lambda lev: order
    return SumpyExpansionWrangler(ti, trav, np.float64 if k is None else np.complex128,
                                  lambda kn, a, t, lev: orders(lev),
                                  kernel_extra_kwargs=None if k is None else {"k": k})


def _m2l(actx, wr, mpoles):
    trav = wr.traversal
    return wr.multipole_to_local(
        actx, trav.host["level_start_target_or_target_parent_box_nrs"],
        trav.target_or_target_parent_boxes, trav.from_sep_siblings_starts,
        trav.from_sep_siblings_lists, mpoles)


def _random_mpoles(wr, actx, rng):
    """Coefficients of size 1 in every degree."""
    n = int(wr.multipole_expansions_level_starts()[-1])
    m = rng.standard_normal(n)
    if wr.dtype.kind == "c":
        m = m + 1j*rng.standard_normal(n)
    return actx.from_numpy(m)


CASES = [("uniform", 3000, 30), ("uniform", 40_000, 40), ("gaussian", 6000, 20),
         ("sphere", 9000, 25), ("uniform", 70, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["laplace", "helmholtz"])
@pytest.mark.parametrize("order", range(1, 13))
def test_folded_m2l_equals_class_matrices(actx, monkeypatch, order, kind, precision):
    """The same locals as the class-matrix contraction, box by box.  Both sum
    the same products, about 189 (order + 1)^2 of them, in the compute
    precision, the folded form after up to three additions per source: the
    difference stays within a few eps sqrt(189 (order + 1)^2) of the box's
    largest term, taken as 64 eps (order + 1) of the largest local of its degree
    anywhere (random coefficients: no systematic cancellation)."""
    from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu
    rng = np.random.default_rng(order)
    for points, n, mpb in CASES:
        pts = torch.from_numpy(_points(points, n, rng)).to(actx.device)
        tree, trav = build_tree_and_traversal_gpu(actx, pts, None, mpb)
        wr = _wrangler(actx, trav, order, precision, 4.0 if kind == "helmholtz" else None)
        mpoles = _random_mpoles(wr, actx, rng)
        got = _m2l(actx, wr, mpoles)
        assert trav.__dict__.get("_m2l_fold_plans")
        with monkeypatch.context() as m:
            m.setattr(m2l_fold, "runs", lambda *a: None)
            want = _m2l(actx, wr, mpoles)
        again = _m2l(actx, wr, mpoles)
        assert torch.equal(torch.view_as_real(got) if got.is_complex() else got,
                           torch.view_as_real(again) if got.is_complex() else again)
        for lev in range(tree.nlevels):
            _, a = wr.local_expansions_view(got, lev)
            _, b = wr.local_expansions_view(want, lev)
            eps = 2.0**-52 if precision == "fp64" else 2.0**-23
            scale = b.abs().amax(0)
            assert ((a - b).abs() <= 64*eps*(order + 1)*scale).all(), (points, n, lev)


@pytest.mark.gpu
def test_folded_m2l_orders_by_level_and_other_lists(actx, monkeypatch):
    """Orders that differ by level, and lists that are not the traversal's own
    (the general contraction serves those)."""
    from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu
    rng = np.random.default_rng(3)
    pts = torch.from_numpy(_points("uniform", 20_000, rng)).to(actx.device)
    _, trav = build_tree_and_traversal_gpu(actx, pts, None, 20)
    wr = _wrangler(actx, trav, lambda lev: 6 + lev % 2, "fp64", None)
    mpoles = _random_mpoles(wr, actx, rng)
    got = _m2l(actx, wr, mpoles)
    assert trav.__dict__.get("_m2l_fold_plans")
    copied = wr.multipole_to_local(
        actx, trav.host["level_start_target_or_target_parent_box_nrs"],
        trav.target_or_target_parent_boxes.clone(), trav.from_sep_siblings_starts.clone(),
        trav.from_sep_siblings_lists.clone(), mpoles)
    scale = copied.abs().max()
    assert (got - copied).abs().max() <= 1e-12*scale


@pytest.mark.gpu
@pytest.mark.parametrize(("kind", "points", "n", "order"), [
    ("laplace", "uniform", 700_000, 3), ("laplace", "uniform", 700_000, 10),
    ("laplace", "gaussian", 200_000, 7), ("helmholtz", "sphere", 60_000, 8)])
def test_folded_fp32_error_is_the_class_matrices(actx, monkeypatch, kind, points, n, order):
    """In FP32 the folded form is no further from FP64 than the class matrices, on
    the locals of the points' own multipoles, level by level: the rms over boxes
    and coefficients relative to the coefficient's rms, whose own scatter between
    point sets is some percent."""
    from sumpy_amd.tree_gpu import build_tree_and_traversal_gpu
    rng = np.random.default_rng(order)
    pts = torch.from_numpy(_points(points, n, rng)).to(actx.device)
    tree, trav = build_tree_and_traversal_gpu(actx, pts, None, 64)
    k = 4.0 if kind == "helmholtz" else None
    wr64, wr32 = (_wrangler(actx, trav, order, p, k) for p in ("fp64", "fp32"))
    q = rng.standard_normal(n)
    q = actx.from_numpy(q + 1j*rng.standard_normal(n) if k else q)
    h = trav.host
    m = wr64.form_multipoles(actx, h["level_start_source_box_nrs"], trav.source_boxes, [q])
    m = wr64.coarsen_multipoles(actx, h["level_start_source_parent_box_nrs"],
                                trav.source_parent_boxes, m)
    ref, folded = _m2l(actx, wr64, m), _m2l(actx, wr32, m)
    monkeypatch.setattr(m2l_fold, "runs", lambda *a: None)
    matrices = _m2l(actx, wr32, m)
    for lev in range(2, tree.nlevels):
        want = wr64.local_expansions_view(ref, lev)[1]
        size = want.abs().pow(2).mean(0).sqrt()
        if (size == 0).any():
            continue
        err = [float(((wr64.local_expansions_view(x, lev)[1] - want).abs()/size).pow(2)
                     .mean().sqrt()) for x in (folded, matrices)]
        assert err[0] <= 1.05*err[1], (lev, err)
