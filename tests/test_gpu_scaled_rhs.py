"""Jacobi-scaled solves with a general right-hand side: the transposed solves
of the adjoint, forward solves with a caller's b, and the FP32 inner solves of
mixed precision reach the unscaled iteration's solution, whose residual is
checked with the oracle's operator."""
import numpy as np
import pytest

import heomq
from oracle import heom_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nk,ntop,lscale", [(1, 1, False), (2, 3, False), (3, 2, True)])
@pytest.mark.parametrize("transpose", [False, True])
def test_scaled_solve_with_rhs(nk, ntop, lscale, transpose):
    import torch
    m = heomq.Model(heomq.siam(nk=nk, ntop=ntop, V=0.3, lscale=lscale, T=0.2))
    ctx = heomq.Context(m)
    p = O.siam_params(nk=nk, ntop=ntop, V=0.3, T=0.2)
    p.lscale = lscale
    o = O.Model(p)
    # the operator's range: b = Pi A x of a seeded physical state, the trace row on tier 0
    x = torch.from_numpy(O.to_fortran(O.physical_projection(o, O.seeded_ado_vector(o, 3)))).to("cuda:0")
    b = ctx.apply_packed(x, trace=heomq.TRACE_RDO, transpose=transpose)
    got = {}
    for mode in (-1, 0):
        ctx.set_precond(mode)
        y, st = ctx.solve_steady(x=ctx.zeros(), b=b, tol=1e-12, transpose=transpose)
        assert st["precond"] == (1 if mode < 0 else 0)
        r = ctx.apply_packed(y, trace=heomq.TRACE_RDO, transpose=transpose) - b
        assert float(r.norm() / b.norm()) <= 1.01e-12
        got[mode] = y
    assert float((got[-1] - got[0]).norm() / got[0].norm()) <= 1e-8
    if not transpose:
        yo = O.apply(o, O.from_fortran(got[-1].cpu().numpy()), trace_row="rdo")
        ref = O.from_fortran(b.cpu().numpy())
        # rows Pi leaves alone: every tier above 0
        assert np.linalg.norm((yo - ref)[1:]) <= 2e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("nk,ntop", [(1, 2), (3, 3)])
def test_mixed_scaled_inner_solves(nk, ntop):
    m = heomq.Model(heomq.siam(nk=nk, ntop=ntop, V=0.3, lscale=True))
    ctx = heomq.Context(m)
    x64, _ = ctx.solve_steady(tol=1e-12)
    x, st = ctx.solve_steady_mixed(tol=1e-12)
    assert st["relres"] <= 1e-12
    assert float((x - x64).norm() / x64.norm()) <= 1e-9
