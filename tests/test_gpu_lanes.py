"""The force passes past the particle numbers of the small tests: spheres on four lanes and on one lane per particle,
polyhedra on four. The feature tests (rolling stiffness, triangle mesh, cylinder and moving drivers) run a few hundred
to a few thousand particles, which take eight; here the same features run at sizes that take the others, in the engine
and at the end of a run (the pass without integration), against the CPU oracle.

Bars: FP64 state, forces, moments and histories equal the oracle's bit for bit (drivers with curved surfaces within
1e-12 relative, as in the small tests); the FP32-force form's forces within its stated 1e-5 of the FP64 form's.
"""
import numpy as np
import pytest

from exadem_amd import inputs, native, stl
from exadem_amd.sim import PolySim, SphereSim, scheme
import pyoracle as po

import driver_cases as dcs
from helpers import by_id, force, interaction_table, pos, rel_err, vel

pytestmark = pytest.mark.gpu

STATE = ("rx", "ry", "rz", "vx", "vy", "vz", "qw", "qx", "qy", "qz", "vrotx", "vroty", "vrotz", "fx", "fy", "fz", "momx",
         "momy", "momz")
# spheres in a list of six rows per particle: four lanes in both forms; one lane in both forms (the limits are 45,000
# and 49,152)
SIZES = [40001, 65601]


def floor_mesh(edge, spacing):
    """A flat triangulated floor of [0, edge]^2."""
    g = np.linspace(0.0, edge, max(2, int(edge // spacing) + 1))
    x, y = np.meshgrid(g, g, indexing="ij")
    p = np.stack([x, y, np.zeros_like(x)], -1)
    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
    tri = np.stack([np.stack([a, b, c], -2), np.stack([a, c, d], -2)], -3).reshape(-1, 3, 3)
    v, e, f = stl.build_shape(tri)
    return {"mesh_id": 3, "vertices": v, "edges": e, "faces": f, "minkowski": 0.01}


def bed(n, kr=0.0, mesh=False):
    side = int(np.ceil((n / 1.5) ** (1.0 / 3.0)))
    edge = 0.98 * (side - 1) + 0.96
    w = inputs.deposition(n=n, spacing=0.98, seed=n, start=0.48, box=(edge, edge, 2 * edge + 2))
    rng = np.random.default_rng(n)
    for k in ("vx", "vy", "vz", "vrotx", "vroty", "vrotz"):
        w.particles[k] = rng.normal(0, 0.3, n)
    w.cp = w.cpd = native.contact_params(kn=1e5, kt=8e4, kr=kr, mu=0.3, damp_rate=0.9)
    m = None
    if mesh:  # a triangulated floor in place of the plane
        w.walls = [x for x in w.walls if x["offset"] != 0.0 or x["normal"][2] == 0.0]
        m = floor_mesh(edge, 0.9)
    return w, m


def oracle_for(w, m):
    o = po.Oracle(w.particles, w.domain, w.walls)
    if m is not None:
        o.set_mesh(m["mesh_id"], m["vertices"], m["edges"], m["faces"], m["minkowski"])
    return o


def same_histories(s, o, m):
    oi, oj, ot, of, _ = o.interactions()
    keep = ot < 7
    kg, fg = interaction_table(*s.ctx.interactions())
    ko, fo = interaction_table(oi[keep], oj[keep], ot[keep], of[keep])
    assert np.array_equal(kg, ko) and np.array_equal(fg, fo) and np.count_nonzero(fo) > 0
    if m is not None:
        kg, fg = interaction_table(*s.ctx.mesh_interactions()[:4])
        ko, fo = interaction_table(*o.mesh_interactions()[:4])
        assert np.array_equal(kg, ko) and np.array_equal(fg, fo) and np.count_nonzero(fo) > 0


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("kr,mesh", [(2e3, False), (0.0, True), (2e3, True)])
def test_rolling_and_mesh_match_oracle(gpu_ok, n, kr, mesh):
    w, m = bed(n, kr, mesh)
    s = SphereSim(w, mesh=m)
    s.first_iteration()
    s.run(5, poll=3)
    s.step()
    o = oracle_for(w, m)
    o.first_iteration(scheme(w))
    o.run_steps(scheme(w), 6)
    a, b = by_id(s.ctx.download()), by_id(o.particles())
    for k in STATE:
        assert np.array_equal(a[k], b[k]), k
    same_histories(s, o, m)
    f = SphereSim(w, form=native.XDEM_FORM_FP32, mesh=m)
    f.first_iteration()
    f.run(6, poll=3)
    c = by_id(f.ctx.download())
    assert rel_err(force(c), force(a), 9.81) <= 1e-5
    assert float(np.max(np.abs(pos(c) - pos(a)))) / float(np.max(np.abs(pos(a)))) <= 1e-9


def drum(n, R, depth):
    """The lower half of a spinning, shaking drum of radius R, n spheres."""
    box = (2 * R + 1.0, depth, 2 * R + 1.0)
    c = np.array([R + 0.5, 0.0, R + 0.5])
    p = dcs.lattice_inside(lambda x, y, z: (np.hypot(x - c[0], z - c[2]) < R - 0.49) & (z < c[2] + 0.5), box)
    assert p["rx"].size >= n
    p = {k: np.ascontiguousarray(v[:n]) for k, v in p.items()}
    assert dcs.settle_onto(p, c, (1, 0, 1), R - 0.49, 0.45) > 500
    walls = [{"kind": "cylinder", "radius": R, "axis": (1.0, 0.0, 1.0), "center": tuple(c), "vrot": (0.0, 1.5, 0.0),
              "motion": {"motion_type": "SHAKER", "amplitude": 0.02, "omega": 100.0, "shaker_dir": (1.0, 0.0, 0.0)}},
             {"offset": 0.0, "normal": (0.0, 1.0, 0.0)}, {"offset": depth, "normal": (0.0, 1.0, 0.0)}]
    return dcs.workload("drum", p, box, walls)


def piston(n):
    """The walled bed with a wall that moves inward by 8e-3 a step: a rebuild that the driver triggers, inside the
    chain."""
    w, _ = bed(n)
    w.dt = 1e-4
    w.walls = [dict(x) for x in w.walls]
    w.walls[1]["motion"] = {"motion_type": "LINEAR_MOTION", "motion_vector": (1.0, 0.0, 0.0), "const_vel": -80.0}
    return w


@pytest.mark.parametrize("case,n", [("drum", 40001), ("drum", 65601), ("piston", 40001), ("piston", 65601)])
def test_moving_drivers_match_oracle(gpu_ok, case, n):
    w = piston(n) if case == "piston" else drum(n, 25.0 if n < 50000 else 30.0, 46.0 if n < 50000 else 52.0)
    sch = scheme(w)
    o = po.Oracle(w.particles, w.domain, w.walls)
    o.first_iteration(sch)
    orb = o.run_steps(sch, 12)
    q = by_id(o.particles())
    assert orb >= (1 if case == "piston" else 0)
    for form, tol in ((native.XDEM_FORM_FP64, 1e-12), (native.XDEM_FORM_FP32, 1e-7)):
        s = SphereSim(w, form=form)
        s.first_iteration()
        st = s.run(12, poll=5)
        g = by_id(s.ctx.download())
        assert st["rebuilds"] == orb
        assert float(np.max(np.abs(pos(g) - pos(q)))) / float(np.max(np.abs(pos(q)))) <= tol
        if form == native.XDEM_FORM_FP64:
            assert float(np.max(np.abs(vel(g) - vel(q)))) <= tol * float(np.max(np.abs(vel(q))))
            assert rel_err(force(g), force(q), q["mass"] * 9.81) <= tol
            same_histories(s, o, None)


@pytest.mark.parametrize("kr,mesh", [(2e3, False), (0.0, True), (2e3, True)])
def test_polyhedra_on_four_lanes_match_oracle(gpu_ok, kr, mesh):
    """Past 32,768 polyhedra the gather takes four lanes per particle: rolling stiffness and a triangulated floor in
    place of the plane, in the engine and the operator step."""
    n = 32900
    w = inputs.polyhedra(density=2500.0, n=n, spacing=1.35, jitter=0.05, seed=n, dt=2e-4, sigma_v=1.0, z0=0.5,
                         periodic=(False, False, False))
    w.cp = w.cpd = native.contact_params(kn=1e5, kt=8e4, kr=kr, mu=0.3, damp_rate=0.9)
    m = None
    if mesh:
        w.walls = w.walls[1:]
        m = dict(floor_mesh(w.domain.hi[0], 1.7), max_candidates=128)
    s = PolySim(w, mesh=m)
    o = po.Oracle(w.particles, w.domain, w.walls)
    o.set_shapes(w.shapes)
    if mesh:
        o.set_mesh(m["mesh_id"], m["vertices"], m["edges"], m["faces"], m["minkowski"])
    s.first_iteration()
    o.first_iteration_poly(scheme(w))
    s.run(7, poll=4)
    s.step()
    o.run_steps_poly(scheme(w), 8)
    a, b = by_id(s.ctx.download()), by_id(o.particles())
    for k in STATE:
        assert np.array_equal(a[k], b[k]), k

    def table(rows):
        ii, jj, tt, sw, si, sj, fr = rows
        key = np.stack([x.astype(np.int64) for x in (ii, jj, tt, sw, si, sj)], 1)
        order = np.argsort(ii, kind="stable")
        return key[order], fr[order]
    kg, fg = table(s.ctx.poly_interactions())
    ko, fo = table(o.poly_interactions())
    assert np.array_equal(kg, ko) and np.array_equal(fg, fo)
    wall = kg[:, 2] >= (7 if mesh else 4)
    assert np.count_nonzero(fg[wall]) > 0 and np.count_nonzero(fg[~wall]) > 0


def test_recorded_pass_of_polyhedra_on_four_lanes(gpu_ok):
    """With contact recording on, the engine's passes are not integrating; the recorded rows hold the friction of the
    histories and add up to the particles' forces."""
    n = 32900
    w = inputs.polyhedra(density=2500.0, n=n, spacing=1.35, jitter=0.05, seed=n, dt=2e-4, sigma_v=1.0, z0=0.5)
    a, b = PolySim(w), PolySim(w)
    b.ctx.set_contact_record(True)
    for s in (a, b):
        s.first_iteration()
        s.run(6, poll=4)
    pa, pb = by_id(a.ctx.download()), by_id(b.ctx.download())
    for k in STATE:
        assert np.array_equal(pa[k], pb[k]), k
    b.ctx.reset_force_moment()
    b.compute_force()
    p = by_id(b.ctx.download())
    ii, jj, tt, v = b.ctx.contact_state()
    F = p["mass"][:, None] * np.asarray(w.gravity)[None, :]
    f = v[:, 4:7] + v[:, 7:10]
    np.add.at(F, ii.astype(np.int64), f)
    pair = tt < 4
    np.add.at(F, jj[pair].astype(np.int64), -f[pair])
    assert np.count_nonzero(~pair) > 0 and np.count_nonzero(pair) > 0
    assert rel_err(F, force(p), p["mass"] * 9.81) <= 1e-12
