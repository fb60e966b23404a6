"""The interior layer's targets on the device where they are not a hole's at
rest: an interior on a background that changes with time (the gauge wave), in
the right-hand side verb, every form of the stepper, a batch, the
vector-Jacobian product and the adjoint, against the oracle, which evaluates
each target at the time of the call."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib
import tgh_desc as TD
from test_gpu_stage import bound, torch_cuda

pytestmark = pytest.mark.gpu


def wave_with_a_layer(tgh, N, roots, q, a=0.05):
    case = tgh.with_interior(tgh.gauge_wave_case(A=a, eps_ko=0.5, gamma0=1.0, gamma2=-0.5),
                             tgh.Interior(center=(0.5, 0.5, 0.5), r_0=0.1, r_1=0.4, rho_max=4.0))
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=q)
    return p, oracle_lib.OracleProblem(TD.TghDesc.from_buffer_copy(bytes(p.desc))), 1.0 / (N * roots)


@pytest.mark.parametrize("N,roots,q", [(8, 4, 2), (14, 2, 4)])
def test_a_layer_on_a_time_dependent_background_follows_it(tgh, N, roots, q):
    torch = torch_cuda()
    p, orc, h = wave_with_a_layer(tgh, N, roots, q)
    t = 0.1
    u0 = orc.fill_exact(t)
    orc.add_noise(u0, 0x1A7E5, 1e-4)
    dt = h / 8
    rhs_tol, step_tol = bound(u0, h, dt)
    du = torch.empty(len(u0), dtype=torch.float64, device="cuda")
    for s in (t, 0.0, 3 * t):  # the verb's target is the call's, whatever came before
        tgh.gh_rhs(du, torch.from_numpy(u0).cuda(), p, s)
        err = float(np.max(np.abs(du.cpu().numpy() - orc.gh_rhs(u0, s, 8))))
        print(f"rhs at t = {s}: {err:.2e} (bound {rhs_tol:.2e})")
        assert err <= rhs_tol
    ref = u0.copy()
    for n in range(2):
        orc.rk4_step(ref, t + n * dt, dt, 8)
    B, S, F, G = tgh.TGH_RK4_BLOCKS, tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_FUSED, tgh.TGH_RK4_GRAPH
    for flags in (0, G, S, F, B, B | G, B | F):
        v = torch.from_numpy(u0).cuda()
        tgh._check(tgh._load().tgh_rk4(p.ptr, C.c_void_p(v.data_ptr()), t, dt, 2, flags))
        err = float(np.max(np.abs(v.cpu().numpy() - ref)))
        print(f"flags {flags}: {err:.2e} (bound {2 * step_tol:.2e})")
        assert err <= 2 * step_tol
    # the transposed right-hand side: 1e-12 of the terms' magnitudes, as in test_gpu_adjoint.py
    rng = np.random.default_rng(10)
    lam, dirn, pd = rng.standard_normal(u0.shape), rng.standard_normal(u0.shape), rng.standard_normal(5)
    _, dF = oracle_lib.gh_rhs_jvp(orc, u0, dirn, t, pd)
    ub, thb = tgh.vjp_rhs(p, torch.from_numpy(u0).cuda(), t, torch.from_numpy(lam).cuda())
    lhs, rhs = float(np.dot(lam, dF)), float(np.dot(ub.cpu().numpy(), dirn) + np.dot(thb, pd))
    scale = float(np.abs(lam * dF).sum())
    print(f"vjp: |diff| / scale = {abs(lhs - rhs) / scale:.2e}")
    assert abs(lhs - rhs) <= 1e-12 * scale
    # rho_max's and rho_ramp's share alone, sums of lambda (u - u_exact): u and
    # u_exact (a sine, a few roundings of 1) cancel to the noise of 1e-4, so
    # each term is good to some 10 eps / 1e-4 = 2e-11 of itself
    pd[:3] = 0.0
    _, dF = oracle_lib.gh_rhs_jvp(orc, u0, np.zeros_like(u0), t, pd)
    err, scale = abs(float(np.dot(lam, dF)) - float(np.dot(thb, pd))), float(np.abs(lam * dF).sum())
    print(f"vjp, the layer's parameters: |diff| / scale = {err / scale:.2e}")
    assert err <= 2e-11 * scale


def test_the_adjoint_reads_each_stages_own_target(tgh):
    """Three steps, a checkpoint every two: dJ/d(gamma2, rho_max, rho_ramp)
    against the oracle's tangent linear model, as in test_gpu_adjoint.py."""
    torch = torch_cuda()
    p, orc, h = wave_with_a_layer(tgh, 8, 4, 2)
    t0, dt, nsteps = 0.1, h / 8, 3
    u0 = orc.fill_exact(t0)
    orc.add_noise(u0, 0x1A7E6, 1e-4)
    ud = torch.from_numpy(u0.copy()).cuda()
    J, grad, _ = tgh.adjoint(p, ud, t0, dt, nsteps, every=2)
    want = np.zeros(5)
    for k in range(2, 5):
        pd = np.zeros(5)
        pd[k] = 1.0
        u, udot = u0.copy(), np.zeros_like(u0)
        for n in range(nsteps):
            oracle_lib.rk4_step_jvp(orc, u, udot, t0 + n * dt, dt, pd)
        want[k] = oracle_lib.error_tangent(orc, u, udot, t0 + nsteps * dt)
    l2, _ = orc.error_norms(u, t0 + nsteps * dt)
    print(f"J {J:.15e} {l2:.15e}; gradient {list(grad[2:])} {list(want[2:])}")
    assert abs(J - l2) <= 1e-12 * l2
    for k in range(2, 5):
        assert abs(grad[k] - want[k]) <= 1e-9 * max(abs(want[k]), 1e-3 * np.max(np.abs(want)))


@pytest.mark.parametrize("graph", [False, True])
def test_a_batch_of_layers_on_waves_steps_each_as_alone(tgh, graph):
    from test_gpu_batch import check_batch_equals_alone
    probs = [wave_with_a_layer(tgh, 8, r, 2, a)[0] for r, a in ((4, 0.05), (5, 0.03))]
    check_batch_equals_alone(tgh, probs, 2, graph)


def moving_hole(tgh, chart, variant, a, roots, v, N=14):
    half = roots * N / 32  # h = 1/16
    args = dict(M=1.0, a=a, v=v, x0=0.1, axis=2, halfwidth=half, r_0=0.35, r_1=0.9, interior=variant)
    case = (tgh.harmonic_kerr_case(**args) if chart == "harmonic"
            else tgh.kerr_schild_case(gauge_source="algebraic", **args))
    return tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=4)


@pytest.mark.parametrize("chart", ["kerr_schild", "harmonic"])
def test_a_moving_frozen_hole_matches_the_oracle_in_every_form(tgh, chart):
    """A :frozen layer has no target and a :frozen core no rate."""
    torch = torch_cuda()
    p = moving_hole(tgh, chart, "frozen", 0.3, 4, 0.3)
    orc = oracle_lib.OracleProblem(TD.TghDesc.from_buffer_copy(bytes(p.desc)))
    h, t = 1.0 / 16, 0.1
    u0 = orc.fill_exact(t)
    orc.add_noise(u0, 0x1A7E7, 1e-6)
    dt = h / 16
    _, step_tol = bound(u0, h, dt)
    ref = u0.copy()
    for n in range(2):
        orc.rk4_step(ref, t + n * dt, dt, 8)
    B, S, F, G = tgh.TGH_RK4_BLOCKS, tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_FUSED, tgh.TGH_RK4_GRAPH
    for flags in (0, G, S, F, B, B | F):
        u = torch.from_numpy(u0).cuda()
        tgh._check(tgh._load().tgh_rk4(p.ptr, C.c_void_p(u.data_ptr()), t, dt, 2, flags))
        err = float(np.max(np.abs(u.cpu().numpy() - ref)))
        print(f"flags {flags}: {err:.2e} (bound {2 * step_tol:.2e})")
        assert err <= 2 * step_tol


@pytest.mark.parametrize("chart", ["kerr_schild", "harmonic"])
@pytest.mark.parametrize("variants", [("frozen", "frozen"), ("frozen", "damped")])
def test_a_batch_takes_moving_frozen_holes(tgh, chart, variants):
    """To an ulp of the state, as test_gpu_batch.py's moving holes."""
    from test_gpu_batch import check_batch_equals_alone
    probs = [moving_hole(tgh, chart, w, a, roots, v)
             for w, a, roots, v in zip(variants, (0.0, 0.3), (3, 4), (0.3, -0.2))]
    check_batch_equals_alone(tgh, probs, 2, True, roundoff=True)


def against_the_oracle(tgh, p, orc, h, t, seed, forms):
    torch = torch_cuda()
    u0 = orc.fill_exact(t)
    orc.add_noise(u0, seed, 1e-6)
    dt = h / 16
    rhs_tol, step_tol = bound(u0, h, dt)
    du = torch.empty(len(u0), dtype=torch.float64, device="cuda")
    tgh.gh_rhs(du, torch.from_numpy(u0).cuda(), p, t)
    err = float(np.max(np.abs(du.cpu().numpy() - orc.gh_rhs(u0, t, 8))))
    print(f"rhs: {err:.2e} (bound {rhs_tol:.2e})")
    assert err <= rhs_tol
    ref = u0.copy()
    orc.rk4_step(ref, t, dt, 8)
    for flags in forms:
        u = torch.from_numpy(u0).cuda()
        tgh._check(tgh._load().tgh_rk4(p.ptr, C.c_void_p(u.data_ptr()), t, dt, 1, flags))
        err = float(np.max(np.abs(u.cpu().numpy() - ref)))
        print(f"flags {flags}: {err:.2e} (bound {step_tol:.2e})")
        assert err <= step_tol
    return u0


def test_a_mesh_inside_a_huge_layer_steps_batches_and_differentiates(tgh):
    """The layer's targets take no more room than the mesh: a cube about r_1 =
    4000 M at h = M/16 would hold 2e15 points."""
    torch = torch_cuda()

    def problem(lo):
        case = tgh.GHCase(None, tgh.KerrSchild(1.0, 0.5), box=[(lo, lo + 1.0)] * 3, periodic=(False,) * 3, eps_ko=0.5,
                          gamma0=1.0, gamma2=0.1, interior=tgh.Interior(r_0=0.8, r_1=4000.0, rho_max=4.0),
                          gauge_source="algebraic")
        return tgh.GHProblem(tgh.gh_forest(None, case, N=8, roots=2), case, q=2)

    p, q = problem(1.0), problem(2.0)
    orc = oracle_lib.OracleProblem(TD.TghDesc.from_buffer_copy(bytes(p.desc)))
    B, S, F = tgh.TGH_RK4_BLOCKS, tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_FUSED
    u0 = against_the_oracle(tgh, p, orc, 1.0 / 16, 0.0, 0x1A7E8, (0, S, F, B))
    us = []
    for x in (p, q):
        us.append(x.statevector())
        tgh.initial_state(us[-1], x, 0.0)
    alone, dt = [u.clone() for u in us], 1.0 / 256
    tgh.gh_solve_batch(tgh.GHBatch([p, q]), us, (0.0, 2 * dt), dt=dt, graph=True)
    for x, u, v in zip((p, q), us, alone):
        tgh.gh_solve(x, v, (0.0, 2 * dt), dt=dt)
        assert torch.isfinite(u).all() and torch.equal(u, v)
    rng = np.random.default_rng(11)
    lam, dirn, pd = rng.standard_normal(u0.shape), rng.standard_normal(u0.shape), rng.standard_normal(5)
    _, dF = oracle_lib.gh_rhs_jvp(orc, u0, dirn, 0.0, pd)
    ub, thb = tgh.vjp_rhs(p, torch.from_numpy(u0).cuda(), 0.0, torch.from_numpy(lam).cuda())
    lhs, rhs = float(np.dot(lam, dF)), float(np.dot(ub.cpu().numpy(), dirn) + np.dot(thb, pd))
    assert abs(lhs - rhs) <= 1e-12 * float(np.abs(lam * dF).sum())


@pytest.mark.parametrize("axis,x0", [(1, 0.3), (3, -0.3)])
def test_a_moving_layer_that_leaves_the_mesh(tgh, axis, x0):
    """25 points an axis, a layer 33 across that reaches over the mesh's face."""
    case = tgh.harmonic_kerr_case(M=1.0, a=0.3, v=0.3, x0=x0, axis=axis, halfwidth=0.75, r_0=0.35, r_1=0.9)
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=12, roots=2), case, q=2)
    orc = oracle_lib.OracleProblem(TD.TghDesc.from_buffer_copy(bytes(p.desc)))
    against_the_oracle(tgh, p, orc, 1.0 / 16, 0.1, 0x1A7E9, (0, tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_BLOCKS))


@pytest.mark.parametrize("center", [(2.5, 2.5, 2.5), (0.9, 0.0, 0.0)])
def test_levels_away_from_the_layer_and_across_it(tgh, center):
    """The box is on the finest level that meets the layer: the mesh's own
    spacing where the finer levels lie elsewhere, theirs where a part of the
    layer is refined and a part is not."""
    case = tgh.kerr_schild_case(M=1.0, a=0.5, halfwidth=4.0, r_0=0.7, r_1=1.5, gauge_source="algebraic")
    f = tgh.hole_forest(None, case, N=8, roots=8, center=center, radii=[0.9, 0.45])
    p = tgh.GHProblem(f, case, q=2, ops=tgh.Operators(prolongation=4))
    assert max(int(lf[0]) for lf in f.leaves) == 2
    orc = oracle_lib.OracleProblem(TD.TghDesc.from_buffer_copy(bytes(p.desc)), leaves=[tuple(lf) for lf in f.leaves],
                                   prolongation=4)
    against_the_oracle(tgh, p, orc, 1.0 / 32, 0.0, 0x1A7EA, (0, tgh.TGH_RK4_FUSED, tgh.TGH_RK4_GRAPH))


PARAMETERS = {
    "harmonic_q4": lambda tgh: (tgh.harmonic_kerr_case(M=1.0, a=0.3, halfwidth=1.5, r_0=0.4, r_1=0.95, gamma2=0.1,
                                                       rho_max=4.0), 12, 4, 4),
    "kerr_schild_sampled_q6": lambda tgh: (tgh.kerr_schild_case(M=1.0, a=0.5, halfwidth=1.6875, r_0=0.71, r_1=1.4,
                                                                gamma2=0.1, rho_max=4.0), 9, 6, 6),
    "kerr_schild_closed_form_q8": lambda tgh: (tgh.kerr_schild_case(M=1.0, a=0.5, halfwidth=1.75, r_0=0.71, r_1=1.5,
                                                                    gamma2=0.1, rho_max=4.0,
                                                                    gauge_source="algebraic"), 14, 4, 8),
}


@pytest.mark.parametrize("name", list(PARAMETERS))
def test_the_parameters_cotangent_alone(tgh, name):
    """theta_bar against the oracle's derivative along a parameter direction with
    the state held: beside the state's own terms, a million times larger, an
    error in it would not show. The layer's terms are sums of u - u_exact and
    the damping's of the constraint, differences of values of size 1 to 1/h that
    cancel to the noise of 1e-4: some 1e3 roundings over that, 2e-9 of each."""
    torch = torch_cuda()
    case, N, roots, q = PARAMETERS[name](tgh)
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=q)
    orc = oracle_lib.OracleProblem(TD.TghDesc.from_buffer_copy(bytes(p.desc)))
    u = orc.fill_exact(0.05)
    orc.add_noise(u, 0x1A7EB, 1e-4)
    rng = np.random.default_rng(12)
    lam, v = rng.standard_normal(u.shape), rng.standard_normal(u.shape)
    ub, thb = tgh.vjp_rhs(p, torch.from_numpy(u).cuda(), 0.05, torch.from_numpy(lam).cuda())
    for k in range(5):
        pd = np.zeros(5)
        pd[k] = 1.0
        _, dF = oracle_lib.gh_rhs_jvp(orc, u, np.zeros_like(u), 0.05, pd)
        want, scale = float(np.dot(lam, dF)), float(np.abs(lam * dF).sum())
        print(f"{tgh.ADJOINT_PARAMS[k]}: {thb[k]:.12e} oracle {want:.12e}, |diff| / scale = "
              f"{abs(thb[k] - want) / scale:.2e}")
        assert abs(thb[k] - want) <= 2e-9 * scale
    _, dF = oracle_lib.gh_rhs_jvp(orc, u, v, 0.05, np.zeros(5))
    assert abs(float(np.dot(lam, dF)) - float(np.dot(ub.cpu().numpy(), v))) <= 1e-12 * float(np.abs(lam * dF).sum())
