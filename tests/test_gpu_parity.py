"""GPU parity of the HIP hot path against the CPU oracle, through the C-ABI.

Bar (FP64): right-hand sides, constraints and RK states agree with the oracle
to <= 1e-12 in the per-variable norm-relative sense
max|gpu - oracle| / max|oracle| (differences come only from operation order
and the last bit of libm pow/cbrt); pure data movement is bit-exact.
Reference: src/z4c/calculate_z4c_rhs.cpp, src/z4c/adm_z4c.cpp,
src/z4c/z4c.cpp, src/z4c/boundary_conditions.cpp,
src/task_list/task_list_integrators_butcher.cpp.
"""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from z4c_amd import Params, Z4cError  # noqa: E402
from z4c_amd._capi import Z4C_NCON  # noqa: E402
from z4c_amd.initial_data import (brill_lindquist_adm, gauge_wave_adm,  # noqa: E402
                                  octree_blocks, perturbed_flat)
from z4c_amd.z4c import MeshBlockGeom, Z4c  # noqa: E402

TOL = 1e-12
MP_GAUGE = dict(lapse_oplog=2.0, lapse_harmonicf=1.0, lapse_harmonic=0.0, lapse_advect=1.0,
                shift_Gamma=1.0, shift_advect=1.0, shift_eta=2.0, diss=0.02,
                damp_kappa1=0.02, damp_kappa2=0.0, chi_div_floor=1e-5)


def rel(a, b):
    """per-variable max|a-b| / max|b| over the last three axes."""
    a = np.asarray(a); b = np.asarray(b)
    num = np.abs(a - b).reshape(a.shape[0], -1).max(axis=1)
    den = np.abs(b).reshape(b.shape[0], -1).max(axis=1)
    return np.where(den > 0, num / np.where(den > 0, den, 1), num)


def ogeom(g: MeshBlockGeom):
    return orc.Geom.block(g.nx, g.dx, g.xmin)


def oparams(p: Params):
    return orc.Params(**p.as_dict())


def interior(g):
    n = 4
    return (slice(None), slice(n, n + g.nx[2] + 1), slice(n, n + g.nx[1] + 1),
            slice(n, n + g.nx[0] + 1))


def constrained_state(g, p, seed):
    """perturbed flat state with the oracle's AlgConstr applied (host)."""
    u = perturbed_flat(g, seed=seed)
    return orc.algconstr(oparams(p), ogeom(g), np.ascontiguousarray(u))


def run_rhs(z, u_host, mat_host=None):
    u = z.upload(u_host)
    mat = z.upload(mat_host) if mat_host is not None else None
    rhs = z.zeros()
    z.PrepareZ4cDerivatives(u)
    z.Z4cRHS(u, mat, rhs)
    torch.cuda.synchronize()
    return z.download(rhs, 22)


# ---------------------------------------------------------------------------
def test_rhs_single_block_32():
    """One 32^3-cell block (33^3 vertices + 4 ghosts), perturbed flat space."""
    g = MeshBlockGeom.cube(32, 1.0 / 32, 0.0)
    p = Params(**MP_GAUGE)
    u = constrained_state(g, p, seed=1)
    z = Z4c([g], p)
    got = run_rhs(z, [u])[0]
    exp = orc.rhs(oparams(p), ogeom(g), u)
    r = rel(got[interior(g)], exp[interior(g)])
    print("max rel diff per var:", r.max())
    assert np.all(r <= TOL), r
    # ghosts are not written
    gh = got.copy()
    gh[interior(g)] = 0.0
    assert np.all(gh == 0.0)


def _matter(g, seed, amp=1e-2):
    """Random matter fields (rho, S_a, S_ab: src/z4c/z4c.hpp:163-184)."""
    return np.ascontiguousarray(amp * np.random.default_rng(seed).standard_normal((10,) + g.shape))


def test_rhs_with_matter_sources():
    """Z4cRHS with the matter terms (calculate_z4c_rhs.cpp:466-476 and the
    rho / S_a / S_ab terms of K^, Theta, Gam~, A~) against the oracle on two
    uneven blocks, and bit-identical over repeated calls."""
    gs = [MeshBlockGeom.cube(8, 0.1, (0.1, -0.2, 0.3)), MeshBlockGeom.cube(12, 0.07, (1.0, 0.0, 0.0))]
    p = Params(**MP_GAUGE)
    us = [constrained_state(g, p, seed=60 + b) for b, g in enumerate(gs)]
    ms = [_matter(g, 70 + b) for b, g in enumerate(gs)]
    z = Z4c(gs, p)
    u, m = z.upload(us), z.upload(ms, 10)
    outs = []
    for _ in range(3):
        r = z.zeros()
        z.Z4cRHS(u, m, r)
        outs.append(r)
    torch.cuda.synchronize()
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    got = z.download(outs[0], 22)
    for b, g in enumerate(gs):
        exp = orc.rhs(oparams(p), ogeom(g), us[b], ms[b])
        vac = orc.rhs(oparams(p), ogeom(g), us[b])
        assert np.all(rel(got[b][interior(g)], exp[interior(g)]) <= TOL), b
        assert np.abs(exp - vac)[interior(g)].max() > 1e-3  # the sources matter


@pytest.mark.parametrize("faces", [True, False])
def test_fused_step_with_matter_equals_stage_sequence(faces):
    """The fused step with matter sources against the stage sequence, and the
    graph-replayed step refuses matter."""
    gs = _uneven_batch(faces)
    p = Params(**MP_GAUGE)
    host = [constrained_state(g, p, seed=80 + b) for b, g in enumerate(gs)]
    z = Z4c(gs, p)
    m = z.upload([_matter(g, 90 + b) for b, g in enumerate(gs)], 10)
    dt = 0.25 * min(min(g.dx) for g in gs)
    ua, ub = z.upload(host), z.upload(host)
    un, k = z.make_rk_registers()
    work = z.make_step_work()
    z.rk4_step(dt, ua, un, k, mat=m)
    z.rk4_step_fused(dt, ub, work, mat=m)
    torch.cuda.synchronize()
    A, Bf = z.download(ua, 22), z.download(ub, 22)
    for b in range(len(gs)):
        assert np.all(rel(Bf[b], A[b]) <= 1e-14), b
    with pytest.raises(Z4cError):
        z.rk4_step_fused(dt, ub, work, mat=m, graph=True)


def test_fused_step_with_matter_against_oracle():
    g = MeshBlockGeom.cube(12, 1.0 / 12, 0.0)
    p = Params(**MP_GAUGE)
    u0 = constrained_state(g, p, seed=5)
    m0 = _matter(g, 6)
    dt = 0.25 / 12
    exp, _ = orc.rk4_step(oparams(p), ogeom(g), u0.copy(), dt, mat=m0)
    z = Z4c([g], p)
    u = z.upload([u0])
    z.rk4_step_fused(dt, u, z.make_step_work(), mat=z.upload([m0], 10))
    torch.cuda.synchronize()
    assert np.all(rel(z.download(u, 22)[0], exp) <= TOL)


def test_rhs_all_terms_general_power():
    """Strong perturbations, chi = psi^-2, every gauge term (vacuum)."""
    g = MeshBlockGeom.cube(8, 0.05, (0.1, -0.2, 0.3))
    rng = np.random.default_rng(4)
    u = perturbed_flat(g, seed=4, amp=(0.01, 0.05))
    u[19:22] += 0.05 * rng.standard_normal((3,) + g.shape)  # shift of both signs
    mat = None
    for pw in (-4.0, -2.0):
        p = Params(chi_psi_power=pw, lapse_harmonic=0.3, lapse_K=0.5, shift_alpha2Gamma=0.4,
                   shift_H=0.3, damp_kappa1=0.05, damp_kappa2=0.1, diss=0.1,
                   chi_div_floor=1e-5)
        uc = orc.algconstr(oparams(p), ogeom(g), np.ascontiguousarray(u))
        z = Z4c([g], p)
        got = run_rhs(z, [uc])[0]
        exp = orc.rhs(oparams(p), ogeom(g), uc)
        r = rel(got[interior(g)], exp[interior(g)])
        assert np.all(r <= TOL), (pw, r)


def test_rhs_chi_floor_and_cowling():
    g = MeshBlockGeom.cube(6, 0.1, 0.0)
    p = Params(chi_div_floor=0.9995, **{k: v for k, v in MP_GAUGE.items() if k != "chi_div_floor"})
    u = constrained_state(g, p, seed=9)
    z = Z4c([g], p)
    got = run_rhs(z, [u])[0]
    exp = orc.rhs(oparams(p), ogeom(g), u)
    assert np.all(rel(got[interior(g)], exp[interior(g)]) <= TOL)
    p2 = Params(cowling=1)
    z2 = Z4c([g], p2)
    assert np.all(run_rhs(z2, [u])[0] == 0.0)


def test_sommerfeld_faces():
    g = MeshBlockGeom.cube(8, 0.25, (1.0, -3.0, 2.0), faces=63)
    p = Params(**MP_GAUGE)
    u = constrained_state(g, p, seed=2)
    z = Z4c([g], p)
    ud = z.upload([u])
    rhs = z.zeros()
    z.PrepareZ4cDerivatives(ud)
    z.Z4cRHS(ud, None, rhs)
    z.Z4cBoundaryRHS(ud, None, rhs)
    torch.cuda.synchronize()
    got = z.download(rhs, 22)[0]
    og = ogeom(g)
    exp = orc.rhs(oparams(p), og, u)
    orc.boundary_rhs(oparams(p), og, u, [1] * 6, exp)
    assert np.all(rel(got[interior(g)], exp[interior(g)]) <= TOL)


def test_batched_uneven_blocks():
    """Blocks of different sizes and spacings in one launch == oracle per block."""
    geoms = [MeshBlockGeom.cube(n, h, x0, level=l) for n, h, x0, l in
             [(4, 0.5, (0, 0, 0), 0), (6, 0.25, (2, 0, 0), 1), (8, 0.125, (3, 1, 0), 2),
              (5, 0.2, (-1, -1, -1), 1), (3, 0.3, (4, 4, 4), 0)]]
    geoms.append(MeshBlockGeom((4, 6, 5), (0.1, 0.2, 0.15), (0.0, 1.0, 2.0)))
    p = Params(**MP_GAUGE)
    us = [constrained_state(g, p, seed=10 + b) for b, g in enumerate(geoms)]
    z = Z4c(geoms, p)
    got = run_rhs(z, us)
    for b, g in enumerate(geoms):
        exp = orc.rhs(oparams(p), ogeom(g), us[b])
        r = rel(got[b][interior(g)], exp[interior(g)])
        assert np.all(r <= TOL), (b, r)


@pytest.mark.parametrize("pw", [-4.0, -2.0])
def test_prepare_derivatives_aux_output(pw):
    """PrepareZ4cDerivatives' storage.aux (adm_z4c.cpp:1044-1119): the 30
    physical ADM derivatives d alpha, d beta, d gamma by the chain rule from
    the prepared conformal derivatives, both chi_psi_power branches (p = -4
    :1046-1080, general p after it), interior vertices, on two uneven
    blocks; vertices outside the interior are not written."""
    gs = [MeshBlockGeom.cube(8, 0.1, (0.1, -0.2, 0.3)),
          MeshBlockGeom.cube((12, 10, 6), (0.07, 0.05, 0.09), (1.0, 0.0, 0.0))]
    p = Params(**dict(MP_GAUGE, chi_psi_power=pw))
    us = [constrained_state(g, p, seed=80 + b) for b, g in enumerate(gs)]
    z = Z4c(gs, p)
    aux = torch.full((30 * z.total_points,), 7.0, dtype=torch.float64, device=z.device)
    z.PrepareZ4cDerivatives(z.upload(us), aux)
    torch.cuda.synchronize()
    got = z.download(aux, 30)
    for b, g in enumerate(gs):
        _, _, exp = orc.prep_derivs(oparams(p), ogeom(g), us[b], want_aux=True)
        s = interior(g)
        r = rel(got[b][s], exp[s])
        print(f"block {b}, p = {pw}: aux max rel diff {r.max():.3e}")
        assert np.all(r <= TOL), r
        outside = got[b].copy()
        outside[s] = 7.0
        assert np.all(outside == 7.0)


def test_algconstr_parity():
    g = MeshBlockGeom.cube(8, 0.1, 0.0)
    p = Params()
    u = perturbed_flat(g, seed=3, amp=(1e-4, 1e-2))
    u[1:7] *= 1.01  # det > 1: projected branch
    z = Z4c([g], p)
    ud = z.upload([u])
    z.AlgConstr(ud)
    torch.cuda.synchronize()
    got = z.download(ud, 22)[0]
    exp = orc.algconstr(oparams(p), ogeom(g), np.ascontiguousarray(u))
    # pow(det, -1/3): device libm vs glibc may differ in the last bit
    np.testing.assert_allclose(got, exp, rtol=2e-15, atol=1e-18)
    # ranged form with skip_physical touches ghosts only
    ud2 = z.upload([u])
    z.AlgConstr(ud2, rng=(0, g.nn[0] - 1, 0, g.nn[1] - 1, 0, g.nn[2] - 1), skip_physical=True)
    torch.cuda.synchronize()
    got2 = z.download(ud2, 22)[0]
    exp2 = orc.algconstr_range(oparams(p), ogeom(g), np.ascontiguousarray(u), 0, g.nn[0] - 1,
                               0, g.nn[1] - 1, 0, g.nn[2] - 1, True)
    np.testing.assert_allclose(got2, exp2, rtol=2e-15, atol=1e-18)
    assert np.array_equal(got2[interior(g)], u[interior(g)])


def random_adm(g, seed):
    """Smooth, non-conformally-flat ADM data (Gamma~ is O(1), not roundoff)."""
    u = perturbed_flat(g, seed=seed, amp=(1e-3, 5e-2))
    adm = np.zeros((17,) + g.shape)
    adm[0] = u[18]
    adm[1:4] = u[19:22]
    adm[4:10] = u[1:7] * 1.1
    adm[10:16] = u[8:14]
    adm[16] = 1.0
    return adm


def test_adm_to_z4c_parity():
    g = MeshBlockGeom.cube(8, 0.1, (0.0, 0.2, -0.3))
    p = Params(chi_div_floor=1e-5)
    adm = random_adm(g, 21)
    z = Z4c([g], p)
    u, ax = z.zeros(), z.zeros(7)
    z.ADMToZ4c(z.upload([adm]), u, ax)
    torch.cuda.synchronize()
    op, og = oparams(p), ogeom(g)
    exp_u, exp_ax = orc.adm_to_z4c(op, og, np.ascontiguousarray(adm), want_aux_ext=True)
    # cbrt / pow may differ in the last bit between device libm and glibc
    assert np.all(rel(z.download(u, 22)[0], exp_u) <= TOL)
    assert np.all(rel(z.download(ax, 7)[0], exp_ax) <= TOL)


def test_adm_conversions_and_constraints():
    g = MeshBlockGeom.cube(8, 0.5, (1.0, 0.5, -2.0))
    p = Params(chi_div_floor=1e-5, r_max_con=1e300)
    adm = brill_lindquist_adm(g)
    z = Z4c([g], p)
    ad = z.upload([adm])
    u = z.zeros()
    ax = z.zeros(7)
    z.ADMToZ4c(ad, u, ax)
    torch.cuda.synchronize()
    got_u = z.download(u, 22)[0]
    op, og = oparams(p), ogeom(g)
    exp_u, exp_ax = orc.adm_to_z4c(op, og, np.ascontiguousarray(adm), want_aux_ext=True)
    # Brill-Lindquist is conformally flat: g~ = delta up to rounding, so
    # Gamma~ = -d_j g~^ij is rounding noise; bound it absolutely instead.
    novec = [n for n in range(22) if n not in (14, 15, 16)]
    assert np.all(rel(got_u[novec], exp_u[novec]) <= TOL)
    assert np.max(np.abs(got_u[14:17])) < 1e-12 / min(g.dx)
    assert np.all(rel(z.download(ax, 7)[0], exp_ax) <= TOL)
    # Z4cToADM + ADMConstraints on the same (oracle) state
    u2 = z.upload([exp_u])
    adm2 = z.zeros(17)
    z.Z4cToADM(u2, adm2)
    z.PrepareZ4cDerivatives(u2)
    con = z.zeros(7)
    z.ADMConstraints(con, adm2, None, u2)
    torch.cuda.synchronize()
    exp_adm = orc.z4c_to_adm(op, og, exp_u)
    assert np.array_equal(z.download(adm2, 17)[0], exp_adm)
    exp_con = orc.adm_constraints(op, og, exp_u, exp_adm)
    got_con = z.download(con, 7)[0]
    assert np.all(rel(got_con, exp_con) <= TOL), rel(got_con, exp_con)


def test_constraints_perturbed_with_matter_and_cut():
    g = MeshBlockGeom.cube(8, 0.1, (-0.4, -0.4, -0.4))
    p = Params(r_max_con=0.45, chi_div_floor=1e-5)
    u = constrained_state(g, p, seed=6)
    rng = np.random.default_rng(6)
    mat = 0.01 * rng.standard_normal((10,) + g.shape)
    op, og = oparams(p), ogeom(g)
    adm = orc.z4c_to_adm(op, og, u)
    z = Z4c([g], p)
    ud, ad, md = z.upload([u]), z.upload([adm]), z.upload([mat])
    z.PrepareZ4cDerivatives(ud)
    con = z.zeros(7)
    z.ADMConstraints(con, ad, md, ud)
    torch.cuda.synchronize()
    got = z.download(con, 7)[0]
    exp = orc.adm_constraints(op, og, u, adm, np.ascontiguousarray(mat))
    assert np.all(rel(got, exp) <= TOL)
    assert np.array_equal(got == 0.0, exp == 0.0)


def test_rk4_step_frozen_ghosts():
    """One bt_rk4 step in the GR_Z4c stage order (ghosts frozen at u_n)."""
    g = MeshBlockGeom.cube(12, 1.0 / 12, 0.0)
    p = Params(**MP_GAUGE)
    u0 = constrained_state(g, p, seed=5)
    dt = 0.25 / 12
    exp, ks = orc.rk4_step(oparams(p), ogeom(g), u0.copy(), dt)
    z = Z4c([g], p)
    u = z.upload([u0])
    un, k = z.make_rk_registers()
    z.PrepareZ4cDerivatives(u)
    z.rk4_step(dt, u, un, k)
    torch.cuda.synchronize()
    got = z.download(u, 22)[0]
    r = rel(got, exp)
    assert np.all(r <= TOL), r
    for s in range(4):
        rk = rel(z.download(k[s], 22)[0][interior(g)], ks[s][interior(g)])
        assert np.all(rk <= 1e-11), (s, rk)


def _uneven_batch(faces=True):
    """three uneven blocks (sizes, spacings, Sommerfeld faces differ)."""
    # no vertex at the origin: the radiative condition divides by r
    f = (lambda m: m) if faces else (lambda m: 0)
    gs = [MeshBlockGeom.cube(8, 0.125, (-1.1, -0.95, -1.05), faces=f(1 | 8 | 32)),
          MeshBlockGeom.cube(12, 1.0 / 12, (0.0, 0.0, 0.0)),
          MeshBlockGeom.cube(6, 0.25, (0.5, -1.5, 0.25), faces=f(63))]
    return gs


@pytest.mark.parametrize("cowling,faces", [(0, True), (1, True), (0, False), (1, False)])
def test_fused_step_equals_stage_sequence(cowling, faces):
    """z4c_rk4_step (RHS assembly + SumBT + AlgConstr fused per stage, ghosts
    at u_n) against four z4c_rk4_stage calls, over two steps, on a batch of
    uneven blocks: the same sums in the same order.  The stage sequence forms
    its right-hand sides in two passes, the fused step in one kernel."""
    gs = _uneven_batch(faces)
    p = Params(**MP_GAUGE, cowling=cowling)
    host = [constrained_state(g, p, seed=20 + b) for b, g in enumerate(gs)]
    z = Z4c(gs, p)
    dt = 0.25 * min(min(g.dx) for g in gs)
    ua = z.upload(host)
    un, k = z.make_rk_registers()
    ub = z.upload(host)
    work = z.make_step_work()
    z.PrepareZ4cDerivatives(ua)
    for _ in range(2):
        z.set_rhs_form("two passes")
        z.rk4_step(dt, ua, un, k)
        z.set_rhs_form("one kernel")
        z.rk4_step_fused(dt, ub, work)
    torch.cuda.synchronize()
    A, Bf = z.download(ua, 22), z.download(ub, 22)
    for b in range(len(gs)):
        r = rel(Bf[b], A[b])
        print(b, "max rel diff", r.max(), "bit-exact", np.array_equal(Bf[b], A[b]))
        assert np.all(r <= 1e-14), (b, r)
    # ADMConstraints prepares the derivatives of the state it is given: the
    # same constraints after the fused step as after the stage sequence
    adm_a, adm_b = z.zeros(17), z.zeros(17)
    z.Z4cToADM(ua, adm_a)
    z.Z4cToADM(ub, adm_b)
    ca, cb = z.zeros(Z4C_NCON), z.zeros(Z4C_NCON)
    z.ADMConstraints(ca, adm_a, None, ua)
    z.ADMConstraints(cb, adm_b, None, ub)
    torch.cuda.synchronize()
    assert torch.allclose(ca, cb, rtol=1e-10, atol=1e-14)


def test_fused_step_against_oracle():
    """z4c_rk4_step on one block against the oracle's bt_rk4 step."""
    g = MeshBlockGeom.cube(12, 1.0 / 12, 0.0)
    p = Params(**MP_GAUGE)
    u0 = constrained_state(g, p, seed=5)
    dt = 0.25 / 12
    exp, _ = orc.rk4_step(oparams(p), ogeom(g), u0.copy(), dt)
    z = Z4c([g], p)
    u = z.upload([u0])
    z.rk4_step_fused(dt, u, z.make_step_work())
    torch.cuda.synchronize()
    r = rel(z.download(u, 22)[0], exp)
    assert np.all(r <= TOL), r


def test_linear_combinations_exact():
    g = MeshBlockGeom.cube(5, 0.1, 0.0)
    rng = np.random.default_rng(8)
    a, b, c = (rng.standard_normal((22,) + g.shape) for _ in range(3))
    z = Z4c([g], Params())
    og = ogeom(g)
    A, Bd, Cd = z.upload([a]), z.upload([b]), z.upload([c])
    out = z.zeros()
    z.bt_sum(out, A, [Bd, Cd], [1. / 6., 1. / 3.], 0.37)
    torch.cuda.synchronize()
    exp = orc.bt_sum(og, a, [b, c], [1. / 6., 1. / 3.], 0.37)
    assert np.array_equal(z.download(out, 22)[0], exp)
    for w in ([1.0, 0.3, 0.0], [0.0, 0.7, 0.2], [0.5, 0.25, 0.25], [0.0, 1.0, 0.0]):
        o = z.upload([a])
        z.WeightedAve(o, Bd, Cd, w)
        torch.cuda.synchronize()
        exp = orc.weighted_ave(og, a.copy(), b, c, w)
        assert np.array_equal(z.download(o, 22)[0], exp), w
    o = z.upload([a])
    z.AddZ4cRHS(Bd, 0.125, o)
    torch.cuda.synchronize()
    assert np.array_equal(z.download(o, 22)[0], orc.add_rhs(og, b, 0.125, a.copy()))
    assert z.NewBlockTimeStep(0.25) == orc.new_dt(og, 0.25)


def test_periodic_fill_exact():
    g = MeshBlockGeom.cube(6, 1.0 / 6, -0.5)
    rng = np.random.default_rng(12)
    a = rng.standard_normal((22,) + g.shape)
    z = Z4c([g], Params())
    d = z.upload([a])
    z.periodic_fill(d)
    torch.cuda.synchronize()
    exp = orc.periodic_fill(ogeom(g), a.copy())
    assert np.array_equal(z.download(d, 22)[0], exp)


def test_gauge_wave_adm_to_z4c_and_rhs():
    g = MeshBlockGeom((16, 4, 4), (1 / 16,) * 3, (-0.5, -0.125, -0.125))
    p = Params(lapse_oplog=0.0, lapse_harmonic=1.0, shift_Gamma=0.0, shift_eta=0.0,
               shift_advect=0.0, diss=0.02, damp_kappa1=0.02, chi_div_floor=1e-5)
    adm = gauge_wave_adm(g)
    z = Z4c([g], p)
    u = z.zeros()
    z.ADMToZ4c(z.upload([adm]), u)
    torch.cuda.synchronize()
    op, og = oparams(p), ogeom(g)
    exp_u = orc.adm_to_z4c(op, og, np.ascontiguousarray(adm))
    gu = z.download(u, 22)[0]
    assert np.all(rel(gu, exp_u) <= TOL)
    got = run_rhs(z, [exp_u])[0]
    exp = orc.rhs(op, og, exp_u)
    assert np.all(rel(got[interior(g)], exp[interior(g)]) <= TOL)


def test_octree_blocklist_sample():
    """A slice of the uneven-block workload: first 12 blocks of the seeded
    octree with Brill-Lindquist data, RHS parity per block."""
    geoms = octree_blocks(nblocks=128, seed=0)[:12]
    assert len({g.nx for g in geoms}) >= 2
    p = Params(**MP_GAUGE)
    us = []
    for g in geoms:
        adm = brill_lindquist_adm(g)
        us.append(orc.adm_to_z4c(oparams(p), ogeom(g), np.ascontiguousarray(adm)))
    z = Z4c(geoms, p)
    got = run_rhs(z, us)
    for b, g in enumerate(geoms):
        exp = orc.rhs(oparams(p), ogeom(g), us[b])
        assert np.all(rel(got[b][interior(g)], exp[interior(g)]) <= TOL), b


def test_invalid_blocks_rejected():
    bad = MeshBlockGeom.cube(1, 0.1, 0.0)  # < 3 interior vertices
    with pytest.raises(Z4cError):
        Z4c([bad], Params())
    with pytest.raises(Z4cError):
        Z4c([MeshBlockGeom.cube(4, -0.1, 0.0)], Params())
