"""The dense apply's heavy / light split at its edges: the shallowest
hierarchies, ADO counts that leave the last light group ragged, and a top tier
whose couplings exceed what one light group stages (more than 8 per ADO at
d = 4: nine tiers, and twelve, which only the reference's own arrays hold), against the oracle's dense apply and
transpose."""
import numpy as np
import pytest

import heomq
from oracle import heom_oracle as O
from ref_arrays import reference_arrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,nk,ntop", [("siam", 1, 1), ("siam", 2, 2), ("siam", 1, 9), ("siam", 1, 12), ("siam", 3, 3),
                                           ("dqd", 1, 1), ("dqd", 1, 2)])
def test_dense_apply_split(model, nk, ntop):
    import torch
    make, omake = (heomq.siam, O.siam_params) if model == "siam" else (heomq.two_impurity, O.dqd_params)
    o = O.Model(omake(nk=nk, ntop=ntop, V=0.3))
    if ntop <= 8:
        m = heomq.Model(make(nk=nk, ntop=ntop, V=0.3))
    else:
        m = heomq.Model.from_reference(**reference_arrays(o))
    ctx = heomq.Context(m)
    rng = np.random.default_rng(nk + 10 * ntop)
    x = rng.standard_normal((o.N, o.d, o.d)) + 1j * rng.standard_normal((o.N, o.d, o.d))
    xd = torch.from_numpy(O.to_fortran(x)).to("cuda:0")
    for trace, row in ((heomq.TRACE_LAST, "last"), (heomq.TRACE_NONE, None)):
        y = O.from_fortran(ctx.apply(xd, trace=trace).cpu().numpy())
        ref = O.apply(o, x, trace_row=row)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
        z = O.from_fortran(ctx.apply_transpose(xd, trace=trace).cpu().numpy())
        ref = O.apply_transpose(o, x, trace_row=row)
        assert np.abs(z - ref).max() <= 1e-12 * np.abs(ref).max()
    y = O.from_fortran(ctx.apply_f32(xd.to(torch.complex64), trace=heomq.TRACE_NONE).cpu().numpy())
    ref = O.apply(o, x, trace_row=None)
    assert np.abs(y - ref).max() <= 2e-6 * np.abs(ref).max()
