"""The packed apply's gathers: 32-bit byte offsets (vectors up to 2^26
elements) against the 64-bit ones of larger vectors, forced on the same
layout, over models with one to many lanes per ADO, every form, both
directions, both precisions and the Chebyshev and preconditioned epilogues;
the grouped rows' run splitting (one, two and four parts) and the top-tier
records of small sectors, in LDS and beyond its room, against the oracle."""
import numpy as np
import pytest

import heomq
from oracle import heom_oracle as O

pytestmark = pytest.mark.gpu

MODELS = {"siam_L1": lambda: heomq.siam(nk=1, ntop=1), "siam_L4": lambda: heomq.siam(nk=2, ntop=4, lscale=True),
          "dqd_L1": lambda: heomq.two_impurity(nk=1, ntop=1), "dqd_L3": lambda: heomq.two_impurity(nk=1, ntop=3, lscale=True)}


@pytest.mark.parametrize("name", list(MODELS))
def test_wide_gathers_give_the_same_values(name, monkeypatch):
    import torch
    m = heomq.Model(MODELS[name]())
    narrow = heomq.Context(m)
    monkeypatch.setenv("HEOMQ_WIDE", "1")
    wide = heomq.Context(m)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.view_as_complex(torch.randn(narrow._ptotal, 2, dtype=torch.float64, device="cuda", generator=g))
    for form in range(8):
        used = narrow.set_apply_form(form)
        assert wide.set_apply_form(form) == used
        for dtype in (torch.complex128, torch.complex64):
            for transpose in (False, True):
                ys = [c.apply_packed_raw(x.to(dtype), c.packed_zeros(dtype), transpose=transpose) for c in (narrow, wide)]
                # the same terms in the same order; the two kernels may contract multiply-adds differently
                tol = 1e-15 if dtype == torch.complex128 else 1e-6
                assert float((ys[0] - ys[1]).abs().max()) <= tol * 16 * float(ys[0].abs().max())
        a, b = (c.chebyshev_packed(x.clone(), 0.02, 1)[0] for c in (narrow, wide))
        assert float((a - b).abs().max()) <= 1e-13 * float(a.abs().max())
    if name.startswith("dqd"):
        for form in (2, 3):
            narrow.set_apply_form(form), wide.set_apply_form(form)
            a, b = (c.apply_packed_precond(x, form=4) for c in (narrow, wide))
            two = narrow.apply_packed_precond(x, form=1)
            assert float((a - b).abs().max()) <= 1e-13 * float(a.abs().max())
            assert float((a - two).abs().max()) <= 1e-13 * float(a.abs().max())


@pytest.mark.parametrize("model,nk,ntop", [("siam", 1, 2), ("siam", 4, 3), ("dqd", 1, 1), ("dqd", 2, 2)])
def test_grouped_rows_match_oracle(model, nk, ntop):
    import torch
    make, omake = (heomq.siam, O.siam_params) if model == "siam" else (heomq.two_impurity, O.dqd_params)
    ctx = heomq.Context(heomq.Model(make(nk=nk, ntop=ntop, V=0.3)))
    o = O.Model(omake(nk=nk, ntop=ntop, V=0.3))
    ctx.set_apply_form(3)
    x = O.physical_projection(o, O.seeded_ado_vector(o, 9))
    xd = torch.from_numpy(O.to_fortran(x)).to("cuda:0")
    for transpose, f in ((False, O.apply), (True, O.apply_transpose)):
        y = O.from_fortran(ctx.apply_packed(xd, trace=heomq.TRACE_RDO, transpose=transpose).cpu().numpy())
        ref = O.physical_projection(o, f(o, x, trace_row="rdo"))
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("nk", [8, 9])
def test_small_sector_records_match_oracle(nk):
    # one wave per heavy ADO: a top-tier block stages the records it may use
    # while they are at most 224 (forward M of them, transposed 3 M: 216 at M =
    # 72, 240 at M = 80, which load theirs from memory)
    import torch
    ctx = heomq.Context(heomq.Model(heomq.siam(nk=nk, ntop=2, V=0.3)))
    o = O.Model(O.siam_params(nk=nk, ntop=2, V=0.3))
    assert ctx.apply_form() == (6, 6)
    x = O.physical_projection(o, O.seeded_ado_vector(o, 10))
    xp = ctx.pack(torch.from_numpy(O.to_fortran(x)).to("cuda:0"))
    for transpose, f in ((False, O.apply), (True, O.apply_transpose)):
        ref = O.physical_projection(o, f(o, x, trace_row="rdo"))
        for dtype, tol in ((torch.complex128, 1e-12), (torch.complex64, 2e-6)):
            yp = ctx.apply_packed_raw(xp.to(dtype), ctx.packed_zeros(dtype), transpose=transpose)
            y = O.from_fortran(ctx.unpack(yp.to(torch.complex128)).cpu().numpy())
            assert np.abs(y - ref).max() <= tol * np.abs(ref).max()
