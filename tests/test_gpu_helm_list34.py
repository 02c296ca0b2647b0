"""Polynomial M2P and moment P2L of the Helmholtz kernel (potentials, charges)
against the general kernels, which the gradient and dipole forms take: box
sizes at the edges of a wave and its halves, list lengths at the edges of the
waves of a block and of the 64 boxes whose sources are numbered at a time."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LISTS = [0, 1, 3, 4, 5, 8, 9, 70]
SIZES = [0, 1, 31, 32, 33, 64, 65, 97]


def _boxes(rng, nsmall):
    """Boxes 0..7 with SIZES points about the origin, then nsmall boxes of 0 to
    5 points at distances of 2 to 4 (rscale 1): (centers, starts, counts, points)."""
    counts = np.concatenate([SIZES, rng.integers(0, 6, nsmall)]).astype(np.int32)
    dirs = rng.standard_normal((3, nsmall))
    centers = np.concatenate([rng.uniform(-.1, .1, (3, 8)), dirs/np.linalg.norm(dirs, axis=0)
                              * rng.uniform(2, 4, nsmall)], axis=1)
    starts = (np.cumsum(counts) - counts).astype(np.int32)
    pts = np.repeat(centers, counts, axis=1) + rng.uniform(-.5, .5, (3, counts.sum()))
    return centers, starts, counts, pts


def _term_sizes(mis, d, k):
    """The sum of the sizes of the terms h(b,j) h(c,l) x^a y^(2j-b) z^(2l-c)
    g_(a+j+l) of D^(a,b,c) G at the vectors d (3, n): (len(mis), n)."""
    from math import factorial as f
    def h(n, i):
        return f(n)/(f(2*i - n)*f(n - i)*2**(n - i))
    r = np.sqrt((d*d).sum(axis=0))
    g = [np.exp(1j*k*r)/r, np.exp(1j*k*r)*(1j*k*r - 1)/r**3]
    while len(g) <= max(sum(m) for m in mis):
        g.append((-(2*len(g) - 1)*g[-1] - k*k*g[-2])/r**2)
    g, x, y, z = np.abs(g), *np.abs(d)
    return np.array([x**a*sum(h(b, j)*h(c, i)*y**(2*j - b)*z**(2*i - c)*g[a + j + i]
                              for j in range((b + 1)//2, b + 1) for i in range((c + 1)//2, c + 1))
                     for a, b, c in mis])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("order", [1, 2, 3, 7, 8, 11, 12])
def test_helmholtz_list34_forms(actx, order, precision):
    """A term passes at most 4 p + 40 roundings (its powers and coefficient,
    Horner's rule or the sum of 32 sources) before the sums in FP64: within as
    many u of the sum of the terms' sizes.  FP64: every addend counts too, and
    those of the general kernel's sum."""
    from sumpy_amd import E2PFromCSR, P2EFromCSR
    from sumpy_amd.expansion.local import LinearPDEConformingVolumeTaylorLocalExpansion
    from sumpy_amd.expansion.multipole import LinearPDEConformingVolumeTaylorMultipoleExpansion
    from sumpy_amd.kernel import AxisSourceDerivative, AxisTargetDerivative, HelmholtzKernel
    rng = np.random.default_rng(order)
    knl = HelmholtzKernel(3)
    centers, starts, counts, pts = _boxes(rng, 100)
    def dev(a):
        return actx.from_numpy(np.ascontiguousarray(a))
    tol = 4*(200 + 8*order)*2.0**-53 if precision == "fp64" else (40 + 4*order)*2.0**-24
    tb = np.arange(8, dtype=np.int32)
    lstarts = np.concatenate([[0], np.cumsum(LISTS)]).astype(np.int32)
    lists = (8 + np.concatenate([rng.permutation(100)[:n] for n in LISTS])).astype(np.int32)
    common = dict(target_boxes=dev(tb), source_box_starts=dev(lstarts),
                  source_box_lists=dev(lists), centers=dev(centers), rscale=1.0, k=1.5)

    mp = LinearPDEConformingVolumeTaylorMultipoleExpansion(knl, order)
    mis = mp.get_coefficient_identifiers()
    # terms of all degrees alike: derivatives of degree d grow like d!
    size = 1/np.array([np.prod(np.arange(1, sum(m) + 1), dtype=float) for m in mis])
    M = (rng.standard_normal((108, len(mp))) + 1j*rng.standard_normal((108, len(mp))))*size
    res = {}
    for name, kernels in (("fast", [knl]),
                          ("general", [knl] + [AxisTargetDerivative(i, knl) for i in range(3)])):
        res[name] = E2PFromCSR(mp, kernels)(
            actx, src_expansions=dev(M), src_base_ibox=0, targets=dev(pts),
            result=[torch.ones(pts.shape[1], dtype=torch.complex128, device=actx.device)
                    for _ in kernels],
            box_target_starts=dev(starts), box_target_counts_nonchild=dev(counts),
            list34_precision=precision if name == "fast" else "fp64", **common)[0]
    got, want = (actx.to_numpy(res[n]) for n in ("fast", "general"))
    for b in range(8):
        own = slice(starts[b], starts[b] + counts[b])
        sizes = sum((np.abs(M[i]) @ _term_sizes(mis, pts[:, own] - centers[:, i:i + 1], 1.5)
                     for i in lists[lstarts[b]:lstarts[b + 1]]), np.zeros(counts[b]))
        assert (np.abs(got - want)[own] <= tol*(1 + sizes)).all()

    lc = LinearPDEConformingVolumeTaylorLocalExpansion(knl, order)
    q_host = rng.standard_normal(pts.shape[1]) + 1j*rng.standard_normal(pts.shape[1])
    q = dev(q_host)
    out = {}
    for name, skn in (("fast", [knl]), ("general", [knl, AxisSourceDerivative(0, knl)])):
        L = torch.ones((108, len(lc)), dtype=torch.complex128, device=actx.device)
        P2EFromCSR(lc, kernels=skn, strength_usage=list(range(len(skn))))(
            actx, sources=dev(pts), strengths=[q, 0*q][:len(skn)], tgt_expansions=L,
            tgt_base_ibox=0, box_source_starts=dev(starts),
            box_source_counts_nonchild=dev(counts),
            list34_precision=precision if name == "fast" else "fp64", **common)
        out[name] = actx.to_numpy(L)
    assert (out["fast"][8:] == 1).all()
    for b in range(8):
        ids = np.concatenate([np.arange(0)] + [starts[i] + np.arange(counts[i])
                                               for i in lists[lstarts[b]:lstarts[b + 1]]]).astype(int)
        sizes = _term_sizes(mis, centers[:, b:b + 1] - pts[:, ids], 1.5) @ np.abs(q_host[ids])
        assert (np.abs(out["fast"] - out["general"])[b] <= tol*sizes).all()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("order", [6, 11, 12])
def test_helmholtz_m2p_far_targets(actx, order, precision):
    """Targets at up to 6000 scales from a small source box (a deep box beside a
    coarse leaf), where the 12th power of the distance, or its product with the
    moments of large strengths, leaves the range of FP32 while the terms that it
    belongs to vanish; a box without multipoles stays zero.  Tolerance as above."""
    from sumpy_amd import E2PFromCSR
    from sumpy_amd.expansion.multipole import LinearPDEConformingVolumeTaylorMultipoleExpansion
    from sumpy_amd.kernel import AxisTargetDerivative, HelmholtzKernel
    rng = np.random.default_rng(order)
    knl, k = HelmholtzKernel(3), 1e-3
    r = np.array([30., 300, 1500, 1700, 3000, 6000])
    d = rng.standard_normal((3, 4))
    d[:, 0] = [0, 0, -1]
    d[:, 1] = [0, 0, 1]
    pts = (d/np.linalg.norm(d, axis=0))[:, :, None]*r
    pts = pts.reshape(3, -1)
    def dev(a):
        return actx.from_numpy(np.ascontiguousarray(a))
    mp = LinearPDEConformingVolumeTaylorMultipoleExpansion(knl, order)
    mis = mp.get_coefficient_identifiers()
    size = 1/np.array([np.prod(np.arange(1, sum(m) + 1), dtype=float) for m in mis])
    M = (rng.standard_normal((3, len(mp))) + 1j*rng.standard_normal((3, len(mp))))*size
    M[0] *= 1e8
    M[2] = 0
    one = dev(np.array([0, 0, 0], np.int32))
    npts = pts.shape[1]
    for source in range(3):
        res = []
        for kernels, prec in (([knl], precision),
                              ([knl] + [AxisTargetDerivative(i, knl) for i in range(3)], "fp64")):
            res.append(actx.to_numpy(E2PFromCSR(mp, kernels)(
                actx, src_expansions=dev(M), src_base_ibox=0, targets=dev(pts),
                result=[torch.zeros(npts, dtype=torch.complex128, device=actx.device)
                        for _ in kernels],
                target_boxes=one[:1], source_box_starts=dev(np.array([0, 1], np.int32)),
                source_box_lists=dev(np.array([source], np.int32)),
                box_target_starts=one, centers=dev(np.zeros((3, 3))), rscale=1.0, k=k,
                box_target_counts_nonchild=dev(np.array([npts, 0, 0], np.int32)),
                list34_precision=prec)[0]))
        sizes = np.abs(M[source]) @ _term_sizes(mis, pts, k)
        u = 2.0**-53 if precision == "fp64" else 2.0**-24
        assert (np.abs(res[0] - res[1]) <= 4*(200 + 8*order)*u*sizes).all()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("order", [6, 11, 12])
def test_helmholtz_p2l_far_sources(actx, order, precision):
    """The transpose: sources at up to 6000 scales from a small target box, whose
    powers leave the range of FP32.  Tolerance as above; in FP32 relative to the
    largest coefficient, since g_n loses digits below 1e-38."""
    from sumpy_amd import P2EFromCSR
    from sumpy_amd.expansion.local import LinearPDEConformingVolumeTaylorLocalExpansion
    from sumpy_amd.kernel import AxisSourceDerivative, HelmholtzKernel
    rng = np.random.default_rng(order)
    knl, k = HelmholtzKernel(3), 1e-3
    d = rng.standard_normal((3, 4))
    d[:, 0] = [0, 0, -1]
    d[:, 1] = [0, 1, 1]
    def dev(a):
        return actx.from_numpy(np.ascontiguousarray(a))
    lc = LinearPDEConformingVolumeTaylorLocalExpansion(knl, order)
    mis = lc.get_coefficient_identifiers()
    zero = dev(np.array([0, 0], np.int32))
    for r in (30., 300, 1500, 1700, 3000, 6000):
        pts = d/np.linalg.norm(d, axis=0)*r
        q_host = rng.standard_normal(4) + 1j*rng.standard_normal(4)
        q = dev(q_host)
        out = []
        for skn, prec in (([knl], precision), ([knl, AxisSourceDerivative(0, knl)], "fp64")):
            L = torch.zeros((2, len(lc)), dtype=torch.complex128, device=actx.device)
            P2EFromCSR(lc, kernels=skn, strength_usage=list(range(len(skn))))(
                actx, sources=dev(pts), strengths=[q, 0*q][:len(skn)], tgt_expansions=L,
                tgt_base_ibox=0, box_source_starts=zero,
                box_source_counts_nonchild=dev(np.array([4, 4], np.int32)),
                list34_precision=prec, target_boxes=zero[:1],
                source_box_starts=dev(np.array([0, 1], np.int32)),
                source_box_lists=dev(np.array([1], np.int32)),
                centers=dev(np.zeros((3, 2))), rscale=1.0, k=k)
            out.append(actx.to_numpy(L)[0])
        sizes = _term_sizes(mis, -pts, k) @ np.abs(q_host)
        u = 2.0**-53 if precision == "fp64" else 2.0**-24
        if precision == "fp32":
            sizes = sizes.max()
        assert (np.abs(out[0] - out[1]) <= 4*(200 + 8*order)*u*sizes).all(), r
