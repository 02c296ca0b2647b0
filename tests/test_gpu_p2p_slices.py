"""The dense direct sum with several lanes per target (few targets): sizes
where the number of lanes changes and ragged source tiles, against plain
torch in float64."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["lap3", "lap2", "helm3"])
@pytest.mark.parametrize(("nt", "ns"), [(1, 1), (3, 255), (64, 257), (4097, 300), (8200, 70),
                                        (131_073, 5)])
def test_dense_sum_slices(actx, nt, ns, kind, precision):
    """Sums of ns terms of the pair precision in any order: within
    (ns + 8) eps sum |q G| (FP32: coordinates relative to a target keep their
    float32 rounding, 64 eps more per term of these unit-square distances)."""
    from sumpy_amd import P2P
    from sumpy_amd.kernel import HelmholtzKernel, LaplaceKernel
    gen = torch.Generator(device="cuda").manual_seed(nt + ns)
    dim = 2 if kind == "lap2" else 3
    kw = dict(device="cuda", dtype=torch.float64, generator=gen)
    tgt = torch.rand(dim, nt, **kw)
    src = torch.rand(dim, ns, **kw) + 1.5   # apart: no near-singular pairs
    q = torch.randn(ns, **kw)
    args = {}
    if kind == "helm3":
        q = torch.complex(q, torch.randn(ns, **kw))
        args = {"k": 4.0}
    knl = HelmholtzKernel(3) if kind == "helm3" else LaplaceKernel(dim)
    got, = P2P([knl], exclude_self=False, precision=precision)(actx, tgt, src, [q], **args)
    r = sum((tgt[a][:, None] - src[a])**2 for a in range(dim)).sqrt()
    if kind == "lap2":
        G = torch.log(r)/(-2*np.pi)
    else:
        G = 1/(4*np.pi*r)
        if kind == "helm3":
            G = torch.polar(G, 4.0*r)
    want = G.to(q.dtype) @ q
    eps = 2.0**-52 if precision == "fp64" else 2.0**-23
    bound = (ns + (8 if precision == "fp64" else 72))*eps*(G.abs() @ q.abs())
    # log r passes zero: the rounding of r counts against 1, not against log r
    if kind == "lap2":
        bound = bound + (ns + 72)*eps*q.abs().sum()/(2*np.pi)
    assert ((got - want).abs() <= bound + 1e-300).all()
