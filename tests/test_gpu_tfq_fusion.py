"""Plain and Jacobi-scaled TFQMR iterations with their vector work in the
operator launches (k_apply_packed_tfq): forward and transposed, over the apply
forms and both models, against the five-kernel iteration and the oracle's
operator."""
import numpy as np
import pytest

import heomq
from oracle import heom_oracle as O

pytestmark = pytest.mark.gpu

MODELS = {
    "siam": (lambda: heomq.siam(nk=2, ntop=3, V=0.3, lscale=True, T=0.2), "siam_params",
             dict(nk=2, ntop=3, V=0.3, T=0.2)),
    "dqd": (lambda: heomq.two_impurity(nk=1, ntop=2, V=0.3, lscale=True), "dqd_params", dict(nk=1, ntop=2, V=0.3)),
}
_cache = {}


def setup(name):
    if name not in _cache:
        make, of, kw = MODELS[name]
        p = getattr(O, of)(**kw)
        p.lscale = True
        _cache[name] = (heomq.Model(make()), O.Model(p))
    return _cache[name]


@pytest.mark.parametrize("name", list(MODELS))
@pytest.mark.parametrize("precond", [0, 1])
@pytest.mark.parametrize("transpose", [False, True])
def test_fused_iteration_on_every_form(name, precond, transpose):
    import torch
    m, o = setup(name)
    ctx = heomq.Context(m)
    ctx.set_precond(precond)
    xo = O.physical_projection(o, O.seeded_ado_vector(o, 3))
    b = ctx.apply_packed(torch.from_numpy(O.to_fortran(xo)).to("cuda:0"), trace=heomq.TRACE_RDO, transpose=transpose)
    bo = O.from_fortran(b.cpu().numpy())
    f = O.apply_transpose if transpose else O.apply
    ctx.set_precond_fusion(False)
    y5, st5 = ctx.solve_steady(x=ctx.zeros(), b=b, tol=1e-11, transpose=transpose)
    assert st5["precond"] == precond and not st5["fused_iteration"]
    ctx.set_precond_fusion(True)
    for form in (0, 2, 3, 6, 7):
        used = ctx.set_apply_form(form)
        print(name, precond, transpose, "form", form, "->", used, flush=True)
        y, st = ctx.solve_steady(x=ctx.zeros(), b=b, tol=1e-11, transpose=transpose)
        assert st["precond"] == precond and st["fused_iteration"]
        assert float((y - y5).norm() / y5.norm()) <= 1e-7
        r = bo - O.physical_projection(o, f(o, O.from_fortran(y.cpu().numpy()), trace_row="rdo"))
        assert np.linalg.norm(r) <= 2e-11 * np.linalg.norm(bo)
