"""The fused block-Jacobi-preconditioned apply: one launch in which every
apply workgroup (a heavy ADO, or a sector-batched run of top-tier ADOs)
applies the inverse (shift - S_K)^-1 to its own outputs before writing them.
It must give the same bits as the apply followed by the one-kernel inverse:
on small models (and against the oracle's dense per-ADO solve), at the
two-impurity workload's full size, and through a whole preconditioned
steady solve.  With the fusion on, the solver also carries TFQMR's vector
work in those launches; its states are checked against the five-kernel
iteration and the oracle's steady state.
"""
import numpy as np
import pytest

import heomq
from oracle import heom_oracle as O

pytestmark = pytest.mark.gpu

CASES = {
    "siam_nk2_L3": (lambda: heomq.siam(nk=2, ntop=3, V=0.3, U=1.5), lambda: O.siam_params(nk=2, ntop=3, V=0.3, U=1.5)),
    "dqd_nk2_L2": (lambda: heomq.two_impurity(nk=2, ntop=2), lambda: O.dqd_params(nk=2, ntop=2)),
    "dqd_nk2_L3": (lambda: heomq.two_impurity(nk=2, ntop=3), lambda: O.dqd_params(nk=2, ntop=3)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_fused_precond_apply_is_the_two_kernel_result(name):
    import torch
    pf, of = CASES[name]
    ctx = heomq.Context(heomq.Model(pf()))
    o = O.Model(of())
    print(f"case {name}", flush=True)
    shift = 0.05 * O.jacobi_ejac(o)[0]
    ctx.set_precond(-1, shift)
    prev = ctx.apply_form()
    ctx.set_apply_form(2, prev[1])   # sector-batched top tier, sliced heavy rows: the fusable form
    x = O.physical_projection(o, O.seeded_ado_vector(o, 47))
    xp = ctx.pack(torch.from_numpy(O.to_fortran(x)).to("cuda:0"))
    y1 = ctx.apply_packed_precond(xp, form=1)
    y4 = ctx.apply_packed_precond(xp, form=4)
    torch.cuda.synchronize()
    assert torch.equal(y1, y4)
    y = O.from_fortran(ctx.unpack(y4).cpu().numpy())
    yo = O.block_jacobi_precondition(o, O.physical_projection(o, O.apply(o, x, trace_row="rdo")), shift)
    assert np.abs(y - yo).max() <= 1e-12 * np.abs(yo).max()
    # a form the fused kernel does not take is refused, not approximated
    ctx.set_apply_form(0, prev[1])
    with pytest.raises(heomq.HeomqError):
        ctx.apply_packed_precond(xp, form=4)
    ctx.set_apply_form(*prev)
    ctx.close()


def test_fused_precond_two_impurity_workload():
    # d = 16, Nk = 6, L = 3, lscale: the fused apply against the two kernels
    # on a random packed vector, then the block-Jacobi-preconditioned steady
    # solve with the fusion on and off
    import torch
    ctx = heomq.Context(heomq.Model(heomq.two_impurity(lscale=True)))
    prev = ctx.apply_form()
    ctx.set_apply_form(2, prev[1])
    g = torch.Generator(device="cuda:0").manual_seed(5)
    n = ctx.packed_zeros().numel()
    xp = torch.complex(torch.randn(n, generator=g, device="cuda:0", dtype=torch.float64),
                       torch.randn(n, generator=g, device="cuda:0", dtype=torch.float64))
    y1 = ctx.apply_packed_precond(xp, form=1)
    y4 = ctx.apply_packed_precond(xp, form=4)
    torch.cuda.synchronize()
    assert torch.equal(y1, y4)
    ctx.set_precond_fusion(True)
    x_on, st_on = ctx.solve_steady(tol=1e-10)
    ctx.set_precond_fusion(False)
    x_off, st_off = ctx.solve_steady(tol=1e-10)
    ctx.set_precond_fusion(True)
    print("fused", st_on, "two kernels", st_off, flush=True)
    assert st_on["status"] == 0 and st_off["status"] == 0
    assert st_on["fused_iteration"] and not st_off["fused_iteration"]
    # the fused iteration has the five-kernel iteration's iterates in exact
    # arithmetic; its reductions are summed in another order (per operator
    # workgroup) and sigma is one recurrence step from a directly summed rt.v,
    # so the iteration counts of the two finite-precision runs differ a little
    # (152 and 162 on this system)
    assert abs(st_on["iters"] - st_off["iters"]) <= 0.15 * st_off["iters"]
    rel = ((x_on - x_off).abs().max() / x_off.abs().max()).item()
    print("relative difference of the two states", rel, flush=True)
    assert rel <= 1e-7
    ctx.set_apply_form(*prev)
    ctx.close()


@pytest.mark.parametrize("name", ["siam_nk2_L3", "dqd_nk2_L2", "dqd_nk2_L3"])
def test_fused_iteration_steady_state_against_the_oracle(name):
    # block Jacobi on the fusable form: the iteration's vector work rides in
    # the two preconditioned launches.  The state's residual through the
    # oracle's operator (one apply: the oracle's own steady solve takes
    # minutes at L = 3), and the state against the five-kernel iteration's.
    import torch
    pf, of = CASES[name]
    ctx = heomq.Context(heomq.Model(pf()))
    o = O.Model(of())
    print(f"case {name}", flush=True)
    ctx.set_precond(2)
    ctx.set_apply_form(2, ctx.apply_form()[1])
    ctx.set_precond_fusion(True)
    x, st = ctx.solve_steady(tol=1e-12)
    print(st, flush=True)
    assert st["status"] == 0 and st["precond"] == 2 and st["fused_iteration"]
    xs = O.from_fortran(x.cpu().numpy())
    e = np.zeros_like(xs)
    e[0, o.d - 1, o.d - 1] = 1.0
    r = e - O.physical_projection(o, O.apply(o, xs, trace_row="rdo"))
    assert np.abs(r).max() <= 1e-10
    ctx.set_precond_fusion(False)
    x5, st5 = ctx.solve_steady(tol=1e-12)
    assert st5["status"] == 0 and not st5["fused_iteration"]
    assert ((x - x5).abs().max() / x5.abs().max()).item() <= 1e-9
    # a second fused solve from the state (after the start's smoothing sweeps)
    ctx.set_precond_fusion(True)
    x2, st2 = ctx.solve_steady(x=x.clone(), tol=1e-12)
    assert st2["status"] == 0
    assert ((x2 - x).abs().max() / x.abs().max()).item() <= 1e-9
    ctx.close()


def test_stalled_unfused_preconditioner_goes_on_fused():
    # block Jacobi without the sector-batched top tier runs unfused; a
    # tolerance below the residual's floor stalls it, and the solve goes on
    # with the plain operator's fused iteration, whose sums need more room
    # than the sparse solve before it (a pattern without the top tier) left
    def model(ntop):
        return heomq.Model(heomq.siam(nk=4, ntop=ntop, V=0.3, T=0.2, lscale=True))
    m = model(3)
    ref, _ = heomq.Context(m).solve_steady(tol=1e-12)
    ctx = heomq.Context(m)
    nnz, ind, irow, icol = (a.copy() for a in m.spa_pattern())
    nnz[model(2).N:] = 0
    ind[model(2).N:] = 0
    ctx.set_spa_pattern(nnz, ind, irow[:nnz.sum()], icol[:nnz.sum()])
    _, st = ctx.solve_steady_spa(tol=1e-10)
    assert st["status"] == 0
    ctx.set_apply_form(0, 0)
    ctx.set_precond(2)
    x, st = ctx.solve_steady(tol=1e-19, maxiter=20000, raise_on_fail=False)
    print(st, flush=True)
    assert st["status"] == heomq._lib.NOT_CONVERGED and st["fused_iteration"]
    assert ((x - ref).abs().max() / ref.abs().max()).item() <= 1e-9


@pytest.mark.parametrize("name,rows", [("dqd_nk2_L2", 3), ("dqd_nk2_L3", 2)])
def test_fused_launch_takes_its_own_heavy_rows(name, rows):
    # by default the plain apply takes the grouped heavy rows (form 3); the
    # fused launch takes them while the heavy ADOs are few (25 here at L = 2)
    # and the sliced ones above (589 at L = 3), bit for bit those forms' own
    # fused launch; a chosen form holds for both
    import torch
    ctx = heomq.Context(heomq.Model(CASES[name][0]()))
    assert ctx.apply_form()[0] == 3
    g = torch.Generator(device="cuda:0").manual_seed(7)
    xp = torch.view_as_complex(torch.randn(ctx.packed_zeros().numel(), 2, generator=g, device="cuda:0",
                                           dtype=torch.float64))
    ctx.set_precond(2, 0.5)
    y = ctx.apply_packed_precond(xp, form=4)
    got = {}
    for form in (2, 3):
        ctx.set_apply_form(form, 2)
        got[form] = ctx.apply_packed_precond(xp, form=4)
        two = ctx.apply_packed_precond(xp, form=1)
        assert ((got[form] - two).abs().max() / two.abs().max()).item() <= 1e-13
    assert torch.equal(y, got[rows]) and not torch.equal(got[2], got[3])


@pytest.mark.parametrize("name", ["dqd_nk2_L2", "dqd_nk2_L3"])
@pytest.mark.parametrize("form", [None, 3])
def test_fused_block_jacobi_iteration_on_grouped_rows(name, form):
    pf, of = CASES[name]
    ctx = heomq.Context(heomq.Model(pf()))
    o = O.Model(of())
    if form is not None:
        ctx.set_apply_form(form, 2)
    x, st = ctx.solve_steady(tol=1e-12)
    assert st["precond"] == 2 and st["fused_iteration"]
    xs = O.from_fortran(x.cpu().numpy())
    e = np.zeros_like(xs)
    e[0, o.d - 1, o.d - 1] = 1.0
    r = e - O.physical_projection(o, O.apply(o, xs, trace_row="rdo"))
    assert np.abs(r).max() <= 1e-10
    ctx.set_precond_fusion(False)
    x5, st5 = ctx.solve_steady(tol=1e-12)
    assert not st5["fused_iteration"]
    assert ((x - x5).abs().max() / x5.abs().max()).item() <= 1e-9


@pytest.mark.parametrize("nk,ntop", [(2, 3), (4, 4)])
def test_small_sectors_keep_the_fused_block_jacobi_iteration(nk, ntop):
    # every sector of the single impurity is small, so the plain apply takes
    # one wave per heavy ADO; block Jacobi still has its fused launch, which
    # the solver takes while the heavy ADOs are few (157 against 5401 here)
    import torch
    ctx = heomq.Context(heomq.Model(heomq.siam(nk=nk, ntop=ntop, V=0.3, U=1.5, lscale=True)))
    ctx.set_precond(2)
    x, st = ctx.solve_steady(tol=1e-11)
    assert st["precond"] == 2 and st["fused_iteration"] == (ntop == 3)
    ctx.set_precond_fusion(False)
    x5, st5 = ctx.solve_steady(tol=1e-11)
    assert not st5["fused_iteration"]
    assert ((x - x5).abs().max() / x5.abs().max()).item() <= 1e-8
    ctx.set_precond_fusion(True)
    g = torch.Generator(device="cuda:0").manual_seed(8)
    xp = torch.view_as_complex(torch.randn(ctx.packed_zeros().numel(), 2, generator=g, device="cuda:0",
                                           dtype=torch.float64))
    for form in (None, 2, 7):
        if form is not None:
            ctx.set_apply_form(form, form)
        y1, y4 = (ctx.apply_packed_precond(xp, form=f) for f in (1, 4))
        assert ((y1 - y4).abs().max() / y1.abs().max()).item() <= 1e-13
