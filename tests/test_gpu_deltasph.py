"""delta-SPH on the GPU against the oracle: one right-hand side and
multi-step RK4 trajectories bit for bit, the float64 error of the float32
path, and Taylor-Green properties at 512^2 (the differentiable-rollout
size)."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from diffsph_amd import _lib, sampling
from diffsph_amd.deltasph import (DeltaSPHConfig, DeltaSPHSolver, analytic_tgv_energy_ratio, compute_timestep,
                                  taylor_green_state)
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _state(ns, seed, jit=0.3, noise=0.1):
    pos, dx = sampling.sample_regular(ns)
    pos = sampling.jitter(pos, dx, jit, seed)
    rng = np.random.default_rng(seed)
    vel = (sampling.taylor_green(pos) + noise * rng.standard_normal(pos.shape)).astype(np.float32)
    n = pos.shape[0]
    rho = (1.0 + 0.01 * rng.standard_normal(n)).astype(np.float32)
    mass = np.full(n, dx * dx, np.float32)
    h = sampling.volume_to_support(dx * dx, 50.0)
    return pos, vel, rho, mass, dx, h


def _oprm(cfg: DeltaSPHConfig):
    return orc.DeltaParams(rho0=cfg.rho0, cs=cfg.cs, delta=cfg.delta, kernel_scale=cfg.kernel_scale,
                           viscosity={"deltaSPH_viscid": 1, "deltaSPH_inviscid": 0, None: -1}[cfg.viscosity],
                           visc_coeff=cfg.nu if cfg.viscosity == "deltaSPH_viscid" else cfg.alpha, eps=cfg.eps,
                           kappa=cfg.kappa, gravity=cfg.gravity or (0.0, 0.0), pi_switch=cfg.pi_switch,
                           eos=0 if cfg.eos == "isoThermal" else 1, diffusion=cfg.diffusion)


def _eq(gpu, ref, what):
    g = gpu.detach().cpu().numpy().reshape(np.shape(ref))
    bad = np.flatnonzero(g.view(np.int32) != np.asarray(ref, np.float32).view(np.int32))
    assert bad.size == 0, f"{what}: {bad.size} values differ, first at {bad[:5]}: {g.ravel()[bad[:3]]} vs " \
                          f"{np.asarray(ref).ravel()[bad[:3]]}"


@pytest.mark.parametrize("ns,seed,visc", [(64, 0, "deltaSPH_viscid"), (48, 1, "deltaSPH_inviscid")])
def test_rhs_matches_oracle_bitexact(ns, seed, visc):
    print(f"case ns={ns} seed={seed} {visc}", flush=True)
    pos, vel, rho, mass, dx, h = _state(ns, seed)
    dev = torch.device("cuda:0")
    T = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    cfg = DeltaSPHConfig(support=h, dx=dx, viscosity=visc, gravity=(0.0, -1.0))
    s = DeltaSPHSolver(T(pos), T(vel), T(mass), T(rho), cfg)
    n = pos.shape[0]
    dudt, drhodt = torch.empty(n, 2, device=dev), torch.empty(n, device=dev)
    terms, L, ev = torch.empty(n, 8, device=dev), torch.empty(n, 4, device=dev), torch.empty(n, 2, device=dev)
    s.rhs(s.pos, s.vel, s.rho, dudt, drhodt, terms, L, ev)
    dom = orc.make_domain((-1, -1), (1, 1), (True, True))
    du, dr, ex = orc.deltaplus_rhs(dom, pos, vel, rho, mass, h, _oprm(cfg))
    _eq(L, ex["L"], "L")
    _eq(ev, ex["ev"], "eigvals")
    _eq(s._grad, ex["grad_rho"], "grad rho")
    _eq(terms, ex["terms"], "terms")
    _eq(dudt, du, "dudt")
    _eq(drhodt, dr, "drhodt")


def _run_pair(ns, steps, seed=0, jit=0.1):
    pos, vel, rho, mass, dx, h = _state(ns, seed, jit=jit, noise=0.0)
    rho[:] = 1.0
    dev = torch.device("cuda:0")
    T = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    cfg = DeltaSPHConfig(support=h, dx=dx)
    s = DeltaSPHSolver(T(pos), T(vel), T(mass), T(rho), cfg)
    dts = []
    for _ in range(steps):
        dts.append(s.step())
    return s, cfg, (pos, vel, rho, mass, h), dts


def test_rk4_trajectory_matches_oracle_bitexact():
    """Taylor-Green 64^2 (jitter 0.1 dx), 6 RK4 steps with the adaptive
    time step: positions, velocities and densities bit for bit; the
    oracle's own time step (global |dudt| norm) agrees with the GPU's."""
    steps = 6
    s, cfg, (pos, vel, rho, mass, h), dts = _run_pair(64, steps)
    dom = orc.make_domain((-1, -1), (1, 1), (True, True))
    st = orc.DeltaState(pos, vel, rho, mass, np.arange(pos.shape[0], dtype=np.int32))
    tp = orc.TimestepParams(support=h, kernel_scale=cfg.kernel_scale, cs=cfg.cs, nu=cfg.nu)
    dt = orc.compute_timestep(tp, cfg.max_dt)
    assert dt == dts[0]
    for k in range(steps):
        st, du = orc.rk4_step(st, dom, h, _oprm(cfg), dts[k])
        dt = orc.compute_timestep(tp, dt, float(np.sqrt((du.astype(np.float64) ** 2).sum())))
        if k + 1 < steps:
            assert dt == pytest.approx(dts[k + 1], rel=1e-6)
    assert np.array_equal(s.uid.cpu().numpy(), st.uid)
    _eq(s.pos, st.pos, "positions")
    _eq(s.vel, st.vel, "velocities")
    _eq(s.rho, st.rho, "densities")
    print(f"dt sequence {dts}", flush=True)


def test_rk4_float64_error_reported():
    """Error of the float32 GPU trajectory against a float64 run of the
    same scheme (same neighbor lists, same time steps), 64^2, 4 steps."""
    steps = 4
    s, cfg, (pos, vel, rho, mass, h), dts = _run_pair(64, steps)
    dom = orc.make_domain((-1, -1), (1, 1), (True, True))
    st = orc.DeltaState(pos.astype(np.float64), vel.astype(np.float64), rho.astype(np.float64),
                        mass.astype(np.float64), np.arange(pos.shape[0], dtype=np.int32))
    for k in range(steps):
        st, _ = orc.rk4_step(st, dom, h, _oprm(cfg), dts[k], dtype=np.float64)
    order = np.argsort(st.uid)
    p, v, r = (t.cpu().numpy().astype(np.float64) for t in s.state_by_uid())
    ep = np.abs(p - st.pos[order]).max() / dts[0]
    ev = np.abs(v - st.vel[order]).max() / np.abs(st.vel).max()
    er = np.abs(r - st.rho[order]).max() / np.abs(st.rho).max()
    print(f"float32 vs float64 after {steps} steps: position/dt {ep:.2e}, velocity {ev:.2e}, density {er:.2e}",
          flush=True)
    assert ev < 1e-5 and er < 1e-5 and ep < 1e-4


def test_taylor_green_512_properties():
    """512^2 = 262k particles (the differentiable-rollout workload): 20
    steps; kinetic energy decays like exp(-4 nu pi^2 t) to within the
    scheme's numerical dissipation, momentum stays zero, density stays
    within Ma^2 = 1e-2 of rho0 (the vortex's own pressure field
    p = -rho0 U^2 (cos 2 pi x + cos 2 pi y)/4 needs |rho - rho0| ~ 5e-3 at
    c_s = 10 U)."""
    dev = torch.device("cuda:0")
    pos, vel, mass, rho, cfg = taylor_green_state(512, dev)
    s = DeltaSPHSolver(pos, vel, mass, rho, cfg)
    e0 = s.kinetic_energy()
    for _ in range(20):
        s.step()
    ratio = s.kinetic_energy() / e0
    ana = analytic_tgv_energy_ratio(s.time, cfg.nu)
    mom = (s.mass[:, None].double() * s.vel.double()).sum(0).abs().max().item()
    drho = (s.rho - cfg.rho0).abs().max().item()
    print(f"t={s.time:.4f} dt={s.dt:.3e} E/E0 {ratio:.6f} analytic {ana:.6f} momentum {mom:.2e} max|rho-rho0| "
          f"{drho:.2e} pairs {s.last_pairs}", flush=True)
    assert abs(ratio - ana) < 0.02 * (1 - ana) + 2e-3
    assert mom < 1e-6 * (s.mass.double().sum().item())
    assert drho < 1e-2


def _dam(res, seed=3, perturb=True):
    from diffsph_amd.deltasph import dam_break_state
    dev = torch.device("cuda:0")
    pos, vel, mass, rho, cfg, walls = dam_break_state(res, dev)
    if perturb:
        rng = np.random.default_rng(seed)
        n = pos.shape[0]
        vel = torch.from_numpy((0.1 * rng.standard_normal((n, 2))).astype(np.float32)).to(dev)
        rho = torch.from_numpy((1.0 + 0.002 * rng.standard_normal(n)).astype(np.float32)).to(dev)
    return pos, vel, mass, rho, cfg, walls


def _owalls(cfg, walls, dom):
    from diffsph_amd.deltasph import MDBC
    return orc.make_walls(dom, walls["pos"].cpu().numpy(), walls["dist"].cpu().numpy(),
                          walls["normal"].cpu().numpy(), float(walls["area"]), cfg.rho0, cfg.support,
                          viscosity=0, visc_coeff=cfg.boundary_alpha, eps=cfg.boundary_eps,
                          mdbc_variant=MDBC[cfg.mdbc])


def _odom(cfg):
    return orc.make_domain(cfg.domain_min, cfg.domain_max, cfg.periodic)


# 2 res^2 rows: 16, 4 (18432) and 1 (233928) lanes per row
@pytest.mark.parametrize("mdbc,res", [("mDBCDensity", 32), ("mDBC_op", 32), ("mDBC_op", 96), ("mDBC_op", 342)])
def test_rhs_with_walls_matches_oracle_bitexact(mdbc, res):
    """Dam break at dx = 1/res with perturbed velocity and density: mDBC wall
    densities (both variants), normalization, density gradient and every
    right-hand side term with the wall pairs, bit for bit."""
    from dataclasses import replace
    print(f"case {mdbc} {res}", flush=True)
    pos, vel, mass, rho, cfg, walls = _dam(res)
    cfg = replace(cfg, mdbc=mdbc)
    s = DeltaSPHSolver(pos, vel, mass, rho, cfg, walls=walls)
    n = s.n
    dev = pos.device
    dudt, drhodt = torch.empty(n, 2, device=dev), torch.empty(n, device=dev)
    terms, L = torch.empty(n, 8, device=dev), torch.empty(n, 4, device=dev)
    s.rhs(s.pos, s.vel, s.rho, dudt, drhodt, terms, L)
    dom = _odom(cfg)
    ow = _owalls(cfg, walls, dom)
    np.testing.assert_array_equal(s.walls.pos.cpu().numpy(), ow.pos)
    _eq(s.walls.ghost, ow.ghost, "ghosts")
    du, dr, ex = orc.deltaplus_rhs(dom, pos.cpu().numpy(), vel.cpu().numpy(), rho.cpu().numpy(),
                                   mass.cpu().numpy(), cfg.support, _oprm(cfg), walls=ow)
    _eq(s.walls.rho, ex["wall_rho"], "mDBC wall density")
    _eq(s.walls.shepard, ex["shepard"], "Shepard density")
    _eq(L, ex["L"], "L")
    _eq(s._grad, ex["grad_rho"], "grad rho")
    _eq(terms, ex["terms"], "terms")
    _eq(dudt, du, "dudt")
    _eq(drhodt, dr, "drhodt")


def test_dam_break_rk4_matches_oracle_bitexact():
    """Dam break at dx = 1/32 from rest, 4 RK4 steps with the adaptive time
    step: fluid positions, velocities and densities bit for bit."""
    pos, vel, mass, rho, cfg, walls = _dam(32, perturb=False)
    s = DeltaSPHSolver(pos, vel, mass, rho, cfg, walls=walls)
    dts = [s.step() for _ in range(4)]
    dom = _odom(cfg)
    ow = _owalls(cfg, walls, dom)
    st = orc.DeltaState(pos.cpu().numpy(), vel.cpu().numpy(), rho.cpu().numpy(), mass.cpu().numpy(),
                        np.arange(pos.shape[0], dtype=np.int32))
    for dt in dts:
        st, _ = orc.rk4_step(st, dom, cfg.support, _oprm(cfg), dt, walls=ow)
    assert np.array_equal(s.uid.cpu().numpy(), st.uid)
    _eq(s.pos, st.pos, "positions")
    _eq(s.vel, st.vel, "velocities")
    _eq(s.rho, st.rho, "densities")
    print(f"dt {dts}", flush=True)


def test_neighbor_list_layouts_identical():
    """Dam break at dx = 1/32, perturbed, with shifting, 3 RK4 steps: the
    one-pass lists (default width), the two-pass lists, and a width that
    every list kind outgrows at first (then widened) give the same
    trajectory bit for bit."""
    from dataclasses import replace
    runs = []
    for w in (67, 0, 4):
        pos, vel, mass, rho, cfg, walls = _dam(32)
        cfg = replace(cfg, neighbor_width=w, shifting=True)
        s = DeltaSPHSolver(pos, vel, mass, rho, cfg, walls=walls)
        dts = [s.step() for _ in range(3)]
        runs.append((s, dts))
    s0, d0 = runs[0]
    assert s0._widths == {}
    assert {"fluid", "ghost"} <= set(runs[2][0]._widths)
    for s, d in runs[1:]:
        assert d == d0 and s.last_pairs == s0.last_pairs
        for a in ("pos", "vel", "rho", "uid"):
            assert torch.equal(getattr(s, a), getattr(s0, a)), a


def test_dam_break_config_properties():
    """The dam-break benchmark (131072 fluid + 9252 wall particles), all
    2000 RK4 steps: the state stays finite, the fluid stays inside the box,
    the column collapses (the front moves right, not faster than the
    shallow-water surge 2 sqrt(g H)), wall densities stay at or above rho0
    (C++ mDBC op) and those of the bottom wall under the column within 1 %
    of rho0 (hydrostatic column: 1 + g H / c_s^2 < 1.003)."""
    from diffsph_amd.deltasph import dam_break_state
    pos, vel, mass, rho, cfg, walls = dam_break_state(256, torch.device("cuda:0"))
    s = DeltaSPHSolver(pos, vel, mass, rho, cfg, walls=walls)
    x0max = float(s.pos[:, 0].max())
    for k in range(2000):
        s.step()
        if (k + 1) % 500 == 0:
            print(f"step {k + 1}: t {s.time:.4f} dt {s.dt:.2e} |u|max {float(s.vel.norm(dim=1).max()):.3f}",
                  flush=True)
    p = s.pos
    assert torch.isfinite(p).all() and torch.isfinite(s.vel).all() and torch.isfinite(s.rho).all()
    assert float(p[:, 0].min()) > 0 and float(p[:, 0].max()) < 4 and float(p[:, 1].min()) > 0
    front = float(p[:, 0].max())
    wr = s.walls.rho
    print(f"t={s.time:.4f} dt={s.dt:.2e} front {x0max:.4f} -> {front:.4f} top {float(p[:, 1].max()):.4f} "
          f"rho [{float(s.rho.min()):.4f}, {float(s.rho.max()):.4f}] wall rho [{float(wr.min()):.4f}, "
          f"{float(wr.max()):.4f}]", flush=True)
    assert front > x0max + 0.05
    assert front < 1.0 + 2 * math.sqrt(9.81 * 2.0) * s.time + 0.05
    assert float(wr.min()) >= cfg.rho0
    wp = s.walls.pos
    under = (wp[:, 0] > 0.1) & (wp[:, 0] < 0.5) & (wp[:, 1] < 0)
    assert int(under.sum()) > 200
    assert float((wr[under] - cfg.rho0).abs().max()) < 0.01 * cfg.rho0


def test_sort_takes_arrays_the_one_pass_permute_does_not():
    """A state array put in place by the caller at an odd 4-byte offset, and
    particle ids of 8 or 16 bits, are permuted as any other."""
    pos, vel, mass, rho, cfg = taylor_green_state(24, torch.device("cuda:0"))
    a, b = DeltaSPHSolver(pos, vel, mass, rho, cfg), DeltaSPHSolver(pos, vel, mass, rho, cfg)
    n = a.n
    buf = torch.zeros(2 * n + 1, device=pos.device)
    buf[1:] = b.vel.flatten()
    b.vel = buf[1:].view(n, 2)
    b.uid = b.uid.to(torch.int16)
    for _ in range(2):
        a.step()
        b.step()
    assert b.uid.dtype == torch.int16 and torch.equal(a.uid, b.uid.to(torch.int32))
    for name in ("pos", "vel", "mass", "rho"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
    b.uid = (b.uid % 100).to(torch.uint8)
    b.step()
    assert b.uid.dtype == torch.uint8


# 16, 4 (up to 2^19) and 1 lanes per ghost, each with a last workgroup that is not full
@pytest.mark.parametrize("ghosts", [5, 16384, 16390, 524291])
def test_mdbc_op_ghost_counts_match_oracle_bitexact(ghosts):
    from diffsph_amd.neighborhood import CellGrid, search
    print(f"case {ghosts}", flush=True)
    rng = np.random.default_rng(ghosts)
    nf, h, per = 1500, 0.13, (True, False)
    f32 = lambda *sh: rng.uniform(-1.0, 1.0, sh).astype(np.float32)  # noqa: E731
    fluid, gpos, wall = f32(nf, 2), f32(ghosts, 2), f32(ghosts, 2)
    fluid[:, 1] *= 0.7  # ghosts without fluid and with up to five neighbors among them
    mass, rho = (4.0 / nf * (1.0 + 0.1 * f32(nf))).astype(np.float32), (1.0 + 0.05 * f32(nf)).astype(np.float32)
    dom_o, dom = orc.make_domain((-1, -1), (1, 1), per), _lib.make_domain((-1, -1), (1, 1), per)
    T = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    g = CellGrid.build(T(fluid), None, dom, h, h_uniform=h)
    si = g.sort_index.long()
    nl = search(g, T(gpos), None, "scatter", layout="sell")
    pr = nl.pairs()
    m, r, x = T(mass)[si].contiguous(), T(rho)[si].contiguous(), T(wall)
    out, shep = torch.empty(ghosts, device="cuda"), torch.empty(ghosts, device="cuda")
    P = _lib.ptr
    _lib.check(_lib.lib().dsph_mdbc(C.byref(pr), P(m), P(r), P(x), C.c_float(1.0), C.c_float(h), 1, P(out), P(shep),
                                    _lib.stream_handle(out.device)), "mdbc")
    off = np.concatenate([[0], np.cumsum(nl.counts.cpu().numpy())]).astype(np.int32)
    ref, rshep = orc.mdbc(dom_o, off, nl.csr_nbr().cpu().numpy(), nl.qpos.cpu().numpy(), g.sorted_pos.cpu().numpy(),
                          h, m.cpu().numpy(), r.cpu().numpy(), wall, 1.0, h, variant=1)
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    np.testing.assert_array_equal(shep.cpu().numpy(), rshep)


# rows of 16, 4 and 1 lanes, with a last workgroup that is not full
@pytest.mark.parametrize("nside", [33, 91, 131, 363, 481])
@pytest.mark.parametrize("state", ["plain", "switch", "odd", "rest"])
def test_near_kernels_equal_general_kernels(nside, state):
    """The uniform-support kernels give the bits of the general ones (reached
    by passing the same support per particle), also for operands out of
    their fast range: zero, tiny and huge densities, infinities, NaN, pairs
    closer than 2^-48; at rest the own density meets no other operand."""
    print(f"case {nside} {state}", flush=True)
    rng = np.random.default_rng(3)
    pos, dx = sampling.sample_regular(nside)
    pos = sampling.jitter(pos, dx, 0.3, 5).astype(np.float32)
    n = pos.shape[0]
    vel = rng.standard_normal((n, 2)).astype(np.float32)
    rho = (1.0 + 0.01 * rng.standard_normal(n)).astype(np.float32)
    if state == "rest":
        vel[:] = 0.0
        rho[rng.permutation(n)[:6]] = [3e38, np.inf, 1e-30, -3e38, 2e37, 1e25]
    if state == "odd":
        pos[0] = (1e-16, 1e-17)
        pos[1] = (1e-16, 3e-16)
        pick = rng.permutation(n)[:12]
        rho[pick[:6]] = [0.0, 1e-30, 1e30, np.inf, np.nan, -1.0]
        vel[pick[6:11], 0] = [np.inf, np.nan, 1e25, 0.0, -np.inf]
    h = sampling.volume_to_support(dx * dx, 50.0)
    dev = torch.device("cuda:0")
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(dev)  # noqa: E731
    cfg = DeltaSPHConfig(support=h, dx=dx, viscosity="deltaSPH_inviscid" if state == "switch" else "deltaSPH_viscid",
                         pi_switch=state == "switch")
    sv = DeltaSPHSolver(T(pos), T(vel), T(np.full(n, dx * dx)), T(rho), cfg)
    nl, pr, wpos, grid = sv.neighbors(sv.pos)
    L, st = _lib.lib(), _lib.stream_handle(dev)
    hs = torch.full((n,), h, dtype=torch.float32, device=dev)
    out = []
    for general in (False, True):
        pr.qh = pr.rh = _lib.ptr(hs) if general else None
        vol, g, m = torch.empty(n, device=dev), torch.empty(n, 2, device=dev), torch.empty(n, 4, device=dev)
        g2, du, dr = torch.empty(n, 2, device=dev), torch.empty(n, 2, device=dev), torch.empty(n, device=dev)
        tm = torch.empty(n, 8, device=dev)
        P = _lib.ptr
        _lib.check(L.dsph_volume(n, P(sv.mass), P(sv.rho), P(vol), st), "volume")
        _lib.check(L.dsph_deltasph_normalization_v(C.byref(pr), None, P(sv.mass), P(sv.rho), P(vol), P(m), None, P(g),
                                                   st), "normalization")
        _lib.check(L.dsph_deltasph_normalization_v(C.byref(pr), None, P(sv.mass), P(sv.rho), None, None, None, P(g2),
                                                   st), "normalization")
        gr = torch.zeros_like(g) if state == "rest" else g
        _lib.check(L.dsph_deltasph_rhs(C.byref(pr), None, C.byref(sv.prm), P(sv.vel), P(sv.mass), P(sv.rho), P(gr),
                                       P(du), P(dr), P(tm), st), "rhs")
        out.append([t.cpu().numpy() for t in (m, g, g2, du, dr, tm)])
    for name, a, b in zip(("L", "grad", "grad, no volumes", "dudt", "drhodt", "terms"), *out):
        np.testing.assert_array_equal(a, b, err_msg=name)
