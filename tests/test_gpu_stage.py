"""The stepper's one-kernel stage (k_brick_stage, k_block_stage) at the sizes
where its tiles end: meshes that 16 x 4 x 4 and 17 x 5 x 3 tiles do not divide,
a single block, the smallest block of each order, against the oracle's RK4 and
right-hand side."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -52


def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible GPU")
    return torch


def wave(tgh, tgh_desc, N, roots, q):
    case = tgh.gauge_wave_case(eps_ko=0.5, gamma0=1.0, gamma2=-0.5)
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=q)
    return p, tgh_desc.gauge_wave_case(N=N, roots=roots, q=q, eps_ko=0.5, gamma0=1.0, gamma2=-0.5), 1.0 / (N * roots)


def hole(tgh, tgh_desc, N, roots, q):
    h = 1.0 / 16
    r1 = 0.71 + 2 * (q // 2 + 2) * h * (1 + 1e-9)
    half = N * roots * h / 2
    case = tgh.kerr_schild_case(M=1.0, a=0.7, halfwidth=half, r_0=0.71, r_1=r1, gauge_source="algebraic")
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=q)
    return p, tgh_desc.TghDesc.from_buffer_copy(bytes(p.desc)), h


def bound(u, h, dt):
    """A right-hand side sums terms up to |u| / h^2 with a few hundred roundings;
    a step multiplies it by dt, and rounds u a few times itself."""
    m = float(np.max(np.abs(u)))
    return 400 * EPS * m / h ** 2, 400 * EPS * m * dt / h ** 2 + 16 * EPS * m


# (q, N, roots): one 16-point row and a point over it, rows shorter than a
# tile, y and z remainders of 1, 2 and 3, the smallest block of each order;
# meshes of 1 to 243 tiles, whose Pi components 5, 2 and 1 workgroups share
WAVES = [(2, 4, 1), (2, 9, 2), (4, 6, 1), (4, 6, 3), (4, 17, 1), (4, 10, 2), (6, 8, 2), (6, 11, 2), (8, 10, 2), (8, 13, 1),
         (4, 12, 3)]
HOLES = [(2, 13, 4), (4, 13, 4), (4, 11, 5), (6, 18, 3), (8, 27, 2)]


@pytest.mark.parametrize("make,q,N,roots", [(wave, *w) for w in WAVES] + [(hole, *w) for w in HOLES])
def test_stage_matches_the_oracle_at_the_edges_of_its_tiles(tgh, make, q, N, roots):
    torch = torch_cuda()
    import oracle_lib
    import tgh_desc
    p, desc, h = make(tgh, tgh_desc, N, roots, q)
    orc = oracle_lib.OracleProblem(desc)
    u0 = orc.fill_exact(0.1)
    orc.add_noise(u0, 0x57A6E, 1e-6)
    dt = h / 8
    rhs_tol, step_tol = bound(u0, h, dt)
    # the verb: k stored in the state's layout
    u, du = torch.from_numpy(u0).cuda(), torch.empty(len(u0), dtype=torch.float64, device="cuda")
    tgh.gh_rhs(du, u, p, 0.1)
    err = float(np.max(np.abs(du.cpu().numpy() - orc.gh_rhs(u0, 0.1, 8))))
    print(f"rhs: {err:.2e} (bound {rhs_tol:.2e})")
    assert err <= rhs_tol
    # two steps in the stage-value form, on bricks, replayed, and in the block layout's tiles
    ref = u0.copy()
    for n in range(2):
        orc.rk4_step(ref, 0.1 + n * dt, dt, 8)
    for flags in (0, tgh.TGH_RK4_GRAPH, tgh.TGH_RK4_BLOCKS | tgh.TGH_RK4_SPLIT):
        v = torch.from_numpy(u0).cuda()
        tgh._check(tgh._load().tgh_rk4(p.ptr, C.c_void_p(v.data_ptr()), 0.1, dt, 2, flags))
        err = float(np.max(np.abs(v.cpu().numpy() - ref)))
        print(f"flags {flags}: {err:.2e} (bound {2 * step_tol:.2e})")
        assert err <= 2 * step_tol


# (chart, axis, q, N, roots): frames and layer boxes that quads of lanes do not
# fill, at a velocity along each axis
MOVES = [("kerr_schild", 1, 2, 13, 4), ("kerr_schild", 3, 4, 11, 5), ("harmonic", 2, 4, 13, 4), ("harmonic", 1, 2, 9, 6)]


@pytest.mark.parametrize("chart,axis,q,N,roots", MOVES)
def test_a_moving_holes_frame_and_layer_match_the_oracle(tgh, chart, axis, q, N, roots):
    torch = torch_cuda()
    import oracle_lib
    import tgh_desc
    h = 1.0 / 16
    half = N * roots * h / 2
    args = dict(M=1.0, a=0.3, v=0.3, x0=0.1, axis=axis, halfwidth=half, r_0=0.35,
                r_1=0.35 + max(0.55, 2 * (q // 2 + 2) * h * (1 + 1e-9)))
    case = (tgh.harmonic_kerr_case(**args) if chart == "harmonic"
            else tgh.kerr_schild_case(gauge_source="algebraic", **args))
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=q)
    orc = oracle_lib.OracleProblem(tgh_desc.TghDesc.from_buffer_copy(bytes(p.desc)))
    u0 = orc.fill_exact(0.1)
    orc.add_noise(u0, 0x57A6F, 1e-6)
    dt = h / 16
    _, step_tol = bound(u0, h, dt)
    ref = u0.copy()
    for n in range(2):
        orc.rk4_step(ref, 0.1 + n * dt, dt, 8)
    # the stage-value form, the head and Pi components apart, and blocks
    for flags in (0, tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_BLOCKS | tgh.TGH_RK4_SPLIT):
        v = torch.from_numpy(u0).cuda()
        tgh._check(tgh._load().tgh_rk4(p.ptr, C.c_void_p(v.data_ptr()), 0.1, dt, 2, flags))
        err = float(np.max(np.abs(v.cpu().numpy() - ref)))
        print(f"flags {flags}: {err:.2e} (bound {2 * step_tol:.2e})")
        assert err <= 2 * step_tol


# (gauge, v, q, halfwidth, N, roots, r_0, r_1): spacings that are no power of two,
# spheres through grid points whose radius a fused multiply-add in their
# position moves across r_0 (12 to 57 of them) or r_1
EDGES = [("algebraic", 0.0, 2, 1.6, 10, 4, 0.8, 1.44), (None, 0.0, 4, 1.6, 10, 4, 0.8, 1.52),
         ("algebraic", 0.0, 4, 1.4, 14, 4, 0.75, 1.25), ("harmonic", 0.0, 2, 1.4, 14, 4, 0.75, 1.25),
         ("algebraic", 0.3, 4, 1.4, 14, 4, 0.75, 1.25)]


@pytest.mark.parametrize("gauge,v,q,half,N,roots,r0,r1", EDGES)
def test_points_on_the_layers_spheres_are_sorted_as_the_oracle_sorts_them(tgh, gauge, v, q, half, N, roots, r0, r1):
    """A point of the sphere r_0 is the layer's (relaxed at rho_max) or the
    core's (frozen): every form decides as the oracle does, and the layer's
    targets are there for the points that it calls the layer's."""
    torch = torch_cuda()
    import oracle_lib
    import tgh_desc
    args = dict(M=1.0, a=0.5, v=v, halfwidth=half, r_0=r0, r_1=r1, rho_max=4.0)
    case = (tgh.harmonic_kerr_case(**args) if gauge == "harmonic" else tgh.kerr_schild_case(gauge_source=gauge, **args))
    p = tgh.GHProblem(tgh.gh_forest(None, case, N=N, roots=roots), case, q=q)
    orc = oracle_lib.OracleProblem(tgh_desc.TghDesc.from_buffer_copy(bytes(p.desc)))
    h = 2 * half / (N * roots)
    u0 = orc.fill_exact(0.0)
    orc.add_noise(u0, 0x57A70, 1e-4)
    dt = h / 16
    rhs_tol, step_tol = bound(u0, h, dt)
    u, du = torch.from_numpy(u0).cuda(), torch.empty(len(u0), dtype=torch.float64, device="cuda")
    tgh.gh_rhs(du, u, p, 0.0)
    err = float(np.max(np.abs(du.cpu().numpy() - orc.gh_rhs(u0, 0.0, 8))))
    print(f"rhs: {err:.2e} (bound {rhs_tol:.2e})")
    assert err <= rhs_tol
    ref = u0.copy()
    orc.rk4_step(ref, 0.0, dt, 8)
    for flags in (0, tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_BLOCKS | tgh.TGH_RK4_SPLIT, tgh.TGH_RK4_BLOCKS | tgh.TGH_RK4_FUSED):
        w = torch.from_numpy(u0).cuda()
        tgh._check(tgh._load().tgh_rk4(p.ptr, C.c_void_p(w.data_ptr()), 0.0, dt, 1, flags))
        err = float(np.max(np.abs(w.cpu().numpy() - ref)))
        print(f"flags {flags}: {err:.2e} (bound {step_tol:.2e})")
        assert err <= step_tol
    if v == 0.0:
        rng = np.random.default_rng(9)
        lam, du_dir, pd = rng.standard_normal(u0.shape), rng.standard_normal(u0.shape), rng.standard_normal(5)
        _, dF = oracle_lib.gh_rhs_jvp(orc, u0, du_dir, 0.0, pd)
        ub, thb = tgh.vjp_rhs(p, torch.from_numpy(u0).cuda(), 0.0, torch.from_numpy(lam).cuda())
        lhs, rhs = float(np.dot(lam, dF)), float(np.dot(ub.cpu().numpy(), du_dir) + np.dot(thb, pd))
        scale = float(np.abs(lam * dF).sum())
        print(f"vjp: |diff| / scale = {abs(lhs - rhs) / scale:.2e}")
        assert abs(lhs - rhs) <= 1e-12 * scale
