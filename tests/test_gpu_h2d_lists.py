"""The 2D Bessel kernels with several waves a box: list lengths and box sizes at
the edges of the waves against the same work one list entry at a time, and the
near field over the ranges of its series against scipy."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LISTS = [0, 1, 3, 4, 5, 9]
SIZES = [1, 3, 63, 64, 65, 130]


def _operators(kind):
    from sumpy_amd.expansion.local import H2DLocalExpansion, Y2DLocalExpansion
    from sumpy_amd.expansion.multipole import H2DMultipoleExpansion, Y2DMultipoleExpansion
    from sumpy_amd.kernel import HelmholtzKernel, YukawaKernel
    if kind == "yukawa":
        return YukawaKernel(2), Y2DMultipoleExpansion, Y2DLocalExpansion, {"lam": 3.0}
    return HelmholtzKernel(2), H2DMultipoleExpansion, H2DLocalExpansion, {"k": 3.0}


@pytest.mark.parametrize("der", [False, True])
@pytest.mark.parametrize(("kind", "order"), [("helmholtz", 0), ("helmholtz", 20),
                                             ("helmholtz", 31), ("yukawa", 7)])
def test_h2d_lists_over_waves(actx, kind, order, der):
    """The same terms in another order of the list: within (list + 8) eps of the
    sum of the single entries' sizes (P2L: of their own sums over a wave, 64 eps)."""
    from sumpy_amd import E2PFromCSR, P2EFromCSR
    from sumpy_amd.kernel import AxisSourceDerivative, AxisTargetDerivative
    knl, mcls, lcls, kw = _operators(kind)
    rng = np.random.default_rng(order)
    nb = len(LISTS) + 10
    counts = np.array(SIZES + list(rng.integers(0, 90, 10)), np.int32)
    starts = (np.cumsum(counts) - counts).astype(np.int32)
    centers = np.concatenate([rng.uniform(-.1, .1, (2, len(LISTS))),
                              2 + rng.uniform(0, 2, (2, 10))], axis=1)
    pts = np.repeat(centers, counts, axis=1) + rng.uniform(-.3, .3, (2, counts.sum()))
    lists = [len(LISTS) + rng.permutation(10)[:n] for n in LISTS]
    def dev(a, dtype=None):
        return actx.from_numpy(np.ascontiguousarray(a if dtype is None else np.asarray(a, dtype)))
    n = counts.sum()
    M = dev(rng.standard_normal((nb, 2*order + 1)) + 1j*rng.standard_normal((nb, 2*order + 1)))
    q = dev(rng.standard_normal(n) + 1j*rng.standard_normal(n))
    tkn = [knl, AxisTargetDerivative(0, knl)] if der else [knl]
    skn = [knl, AxisSourceDerivative(1, knl)] if der else [knl]
    box = dict(centers=dev(centers), rscale=0.7, **kw)

    def m2p(boxes, ls):
        return [actx.to_numpy(r) for r in E2PFromCSR(mcls(knl, order), tkn)(
            actx, src_expansions=M, src_base_ibox=0, targets=dev(pts),
            target_boxes=dev(boxes, np.int32), box_target_starts=dev(starts),
            box_target_counts_nonchild=dev(counts), source_box_lists=dev(np.concatenate(
                ls), np.int32), source_box_starts=dev(np.cumsum([0] + [len(x) for x in ls]),
                                                      np.int32),
            result=[torch.zeros(n, dtype=torch.complex128, device=actx.device) for _ in tkn],
            **box)]

    def p2l(boxes, ls):
        L = torch.zeros((nb, 2*order + 1), dtype=torch.complex128, device=actx.device)
        P2EFromCSR(lcls(knl, order), kernels=skn, strength_usage=[0]*len(skn))(
            actx, sources=dev(pts), strengths=[q], tgt_expansions=L, tgt_base_ibox=0,
            target_boxes=dev(boxes, np.int32), box_source_starts=dev(starts),
            box_source_counts_nonchild=dev(counts), source_box_lists=dev(np.concatenate(
                ls), np.int32), source_box_starts=dev(np.cumsum([0] + [len(x) for x in ls]),
                                                      np.int32), **box)
        return [actx.to_numpy(L)]

    eps = 2.0**-52
    for op, factor in ((m2p, 8), (p2l, 64)):
        got = op(np.arange(len(LISTS)), lists)
        want, size = [np.zeros_like(g) for g in got], [np.zeros(g.shape) for g in got]
        for i in range(max(LISTS)):
            boxes = [b for b, x in enumerate(lists) if len(x) > i]
            for w, z, r in zip(want, size, op(boxes, [lists[b][i:i + 1] for b in boxes])):
                w += r
                z += np.abs(r)
        for g, w, z in zip(got, want, size):
            assert (np.abs(g - w) <= (max(LISTS) + factor)*eps*z.max()).all()


def test_h2d_near_field_series(actx):
    """(i/4) H0(k r) at k r about the ends of its series, far below and above:
    the values are within a few eps of |H0| + |J0 log| (scipy's own error
    included: 16 eps), above 4 within the Neumann route's 1e-13."""
    from scipy.special import hankel1
    from sumpy_amd import P2P
    from sumpy_amd.kernel import HelmholtzKernel
    k = 7.0
    x = np.concatenate([np.logspace(-12, 0, 40), 1 + np.linspace(-1e-3, 1e-3, 9),
                        np.linspace(1, 4, 41), 4 + np.linspace(-1e-3, 1e-3, 9),
                        np.linspace(4, 40, 50)])
    tgt = np.stack([x/k, 0*x])
    got, = P2P([HelmholtzKernel(2)], exclude_self=False)(
        actx, actx.from_numpy(tgt), actx.from_numpy(np.zeros((2, 1))),
        [actx.from_numpy(np.ones(1, np.complex128))], k=k)
    want = 0.25j*hankel1(0, k*tgt[0])
    tol = np.where(x <= 4, 16*2.0**-52*(1 + np.abs(np.log(x))), 1e-13)
    assert (np.abs(actx.to_numpy(got) - want) <= tol*(0.25 + np.abs(want))).all()
