"""The one-kernel right-hand side against the two-pass form (stencil pass and
algebra pass), which it equals bit for bit: bricks of 17 x 5 x 3 vertices cut
from blocks at, below and above their edges."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from z4c_amd import Params  # noqa: E402
from z4c_amd.initial_data import perturbed_flat  # noqa: E402
from z4c_amd.z4c import MeshBlockGeom, Z4c  # noqa: E402

# cells per axis: vertices are one more
SIZES = [(16, 4, 2), (17, 5, 3), (15, 3, 14), (2, 2, 2), (33, 9, 5), (34, 10, 6), (50, 2, 3),
         (3, 31, 2), (2, 3, 29), (20, 13, 11)]


def _batch(faces=0):
    gs = []
    for b, n in enumerate(SIZES):
        dx = tuple(0.05 + 0.01 * ((b + d) % 3) for d in range(3))
        gs.append(MeshBlockGeom(n, dx, (0.3 + b, -1.0, 0.7), sommerfeld_faces=faces))
    return gs


@pytest.mark.parametrize("params", [
    dict(diss=0.02, damp_kappa1=0.02),
    dict(diss=0.1, damp_kappa1=0.3, damp_kappa2=0.2, chi_psi_power=-2.5, lapse_harmonic=0.7,
         lapse_K=0.3, shift_alpha2Gamma=0.4, shift_H=0.2, lapse_advect=0.5, shift_advect=0.25),
    # chi below its floor on most vertices, harmonic slicing, no shift driver
    dict(diss=0.5, damp_kappa1=0.05, chi_div_floor=1.001, lapse_oplog=0.0, lapse_harmonic=1.0,
         lapse_advect=0.0, shift_Gamma=0.0, shift_eta=0.0, shift_advect=0.0)])
@pytest.mark.parametrize("matter", [False, True])
def test_one_kernel_equals_two_passes(params, matter):
    gs = _batch()
    z = Z4c(gs, Params(**params))
    u = z.upload([perturbed_flat(g, seed=b, amp=(1e-3, 1e-1)) for b, g in enumerate(gs)])
    z.AlgConstr(u)
    mat = None
    if matter:
        gen = torch.Generator(device="cuda").manual_seed(5)
        mat = 1e-2 * torch.randn(10 * z.total_points, dtype=torch.float64, device="cuda",
                                 generator=gen)
    one = torch.full_like(u, 7.0)
    two = torch.full_like(u, 7.0)
    z.set_rhs_form("one kernel")
    z.Z4cRHS(u, mat, one)
    z.set_rhs_form("two passes")
    z.Z4cRHS(u, mat, two)
    assert torch.equal(one, two)
    # written over its own input
    v = u.clone()
    z.set_rhs_form("one kernel")
    z.Z4cRHS(v, mat, v)
    for b in range(len(gs)):
        a, w = z.block_view(one, b, 22), z.block_view(v, b, 22)
        assert torch.equal(a[:, 4:-4, 4:-4, 4:-4], w[:, 4:-4, 4:-4, 4:-4])
    z.close()


def test_two_passes_captured_by_a_new_context():
    """A graph captured around the first right-hand side that needs the
    derivative slots: written over its own input."""
    gs = _batch()
    z = Z4c(gs, Params(diss=0.02))
    u = z.upload([perturbed_flat(g, seed=b) for b, g in enumerate(gs)])
    want = u.clone()
    z.Z4cRHS(u, None, want)
    v = u.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z.Z4cRHS(v, None, v)
    for _ in range(3):
        v.copy_(u)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(v, want)
    z.close()


def test_stencil_threads_do_not_choose_the_form():
    """Fixing or tuning the stencil pass's workgroups leaves the form of the
    right-hand sides, and what it is measured on, as they were."""
    z = Z4c([MeshBlockGeom.cube(32, 0.1, 0.3)], Params(diss=0.02))
    u = z.upload([perturbed_flat(z.blocks[0], seed=1)])
    assert z.rhs_form()[0] == "one kernel"
    z.set_stencil_threads(256)
    assert z.rhs_form()[0] == "one kernel"
    z.set_rhs_form("two passes")
    z.autotune(u, reps=1)
    z.set_stencil_threads(192, block=0)
    assert z.rhs_form()[0] == "two passes"
    z.set_rhs_form("auto")
    assert z.rhs_form()[0] == "one kernel"
    z.close()


def test_small_batch_rule_does_not_change_results():
    """Few small blocks take the two passes, the same blocks among many the
    one kernel."""
    g = [MeshBlockGeom.cube(8, 0.1, 0.2)]
    many = g + [MeshBlockGeom.cube(16, 0.1, 2.0 * b + 3.0) for b in range(8)]
    p = Params(diss=0.02)
    out = []
    for gs, form in ((g, "two passes"), (many, "one kernel")):
        z = Z4c(gs, p)
        assert z.rhs_form()[0] == form
        u = z.upload([perturbed_flat(x, seed=b) for b, x in enumerate(gs)])
        r = z.zeros()
        z.Z4cRHS(u, None, r)
        out.append(z.block_view(r, 0, 22).clone())
        z.close()
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("faces", [0, 63])
@pytest.mark.parametrize("ghosts", [dict(), dict(physical=True)])
def test_step_equals_stages(faces, ghosts):
    """The fused step in one kernel (state registers alternating) against the
    task list's stage sequence with its right-hand sides in two passes, on the
    same ragged blocks."""
    if ghosts and not faces:
        pytest.skip("no face to fill")
    gs = _batch(faces)
    p = Params(diss=0.02, damp_kappa1=0.02)
    z = Z4c(gs, p)
    host = [perturbed_flat(g, seed=20 + b) for b, g in enumerate(gs)]
    a, b = z.upload(host), z.upload(host)
    z.AlgConstr(a)
    z.AlgConstr(b)
    un, k = z.make_rk_registers()
    z.set_rhs_form("two passes")
    z.rk4_step(0.004, a, un, k, **ghosts)
    z.set_rhs_form("one kernel")
    z.rk4_step_fused(0.004, b, z.make_step_work(), **ghosts)
    for q in range(len(gs)):
        x, y = z.block_view(a, q, 22), z.block_view(b, q, 22)
        d = (x - y).abs().amax((1, 2, 3))
        s = x.abs().amax((1, 2, 3))
        # interior sums in another order at the last stage only: a few ulp; the
        # outermost ghosts of a filled face amplify them (weights summing to 31)
        assert bool((d <= (1e-9 if ghosts else 1e-14) * s + 1e-300).all()), (q, (d / s).max())
    z.close()


@pytest.mark.parametrize("n, nblocks, form", [
    ((2, 2, 2), 1, "two passes"), ((4, 4, 4), 16, "two passes"), ((4, 64, 4), 64, "two passes"),
    ((17, 5, 3), 500, "two passes"), ((16, 16, 16), 1, "one kernel"),
    ((32, 32, 32), 1, "one kernel"), ((2, 2, 2), 1024, "one kernel"), ((8, 8, 64), 1, "one kernel")])
def test_form_rule(n, nblocks, form):
    """Batches at which one form is faster by a quarter and more take it, for
    z4c_rhs and for the steps."""
    z = Z4c([MeshBlockGeom(n, (0.1, 0.1, 0.1), (0.3, 0.2, 0.1))] * nblocks, Params())
    assert z.rhs_form() == (form, form)
    z.close()


@pytest.mark.parametrize("faces", [0, 45])
@pytest.mark.parametrize("ghosts", [dict(), dict(periodic=True), dict(physical=True)])
@pytest.mark.parametrize("kw", [dict(), dict(cowling=1), dict(matter=True)])
def test_steps_in_both_forms(faces, ghosts, kw):
    """rk4_step_fused and ls_step in one kernel and in two passes (in place
    without faces) on ragged blocks: the same bits, ghosts included."""
    gs = _batch(faces)
    matter = kw.get("matter")
    z = Z4c(gs, Params(diss=0.02, damp_kappa1=0.02, cowling=kw.get("cowling", 0)))
    host = [perturbed_flat(g, seed=30 + b) for b, g in enumerate(gs)]
    mat = None
    if matter:
        gen = torch.Generator(device="cuda").manual_seed(6)
        mat = 1e-2 * torch.randn(10 * z.total_points, dtype=torch.float64, device="cuda",
                                 generator=gen)
    calls = [lambda u: z.rk4_step_fused(0.004, u, z.make_step_work().fill_(7.0), mat, **ghosts)]
    for name in ("rk1", "rk2", "rk3", "rk4"):
        calls.append(lambda u, t=name: z.ls_step(t, 0.004, u, z.make_ls_work().fill_(7.0), mat,
                                                 **ghosts))
    for call in calls:
        out = []
        for form in ("one kernel", "two passes"):
            z.set_rhs_form(form)
            u = z.upload(host)
            z.AlgConstr(u)
            call(u)
            out.append(u)
        assert torch.equal(out[0], out[1])
    z.close()


def test_zero_right_hand_side_runs_no_stencils():
    """cowling: a stage is a copy with weights; neither stencils nor bricks."""
    z = Z4c([MeshBlockGeom.cube(32, 0.1, 0.3)], Params(cowling=1))
    u = z.upload([perturbed_flat(z.blocks[0], seed=2)])
    z.set_timing(True)
    z.rk4_step_fused(0.01, u, z.make_step_work())
    z.ls_step("rk3", 0.01, u, z.make_ls_work())
    t = z.get_timing()
    assert t["stencil"][1] == 0 and t["assembly"][1] == 7
    z.close()
