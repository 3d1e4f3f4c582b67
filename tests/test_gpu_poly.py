"""Parity of the HIP polyhedra path (through the C ABI) with the CPU oracle, on seeded inputs.

Cubes (edge 1) and octahedra (circumradius 0.8), Minkowski radius 0.02, random orientations.
Bars: the feature interaction lists (owner, partner, type, swap, sub-features, order per owner)
bit-exact; friction history bit-exact; forces and moments within 1e-12 relative (floor m|g|);
trajectories within 1e-10 relative. The fused engine must equal the operator-by-operator path.
"""
import numpy as np
import pytest

from exadem_amd import inputs, native
from exadem_amd import shapes as shp
from exadem_amd.sim import PolySim, scheme
import pyoracle as po

from helpers import by_id, force, pos, rel_err, vec, vel

pytestmark = pytest.mark.gpu

FORCE_TOL = 1e-12
TRAJ_TOL = 1e-10


def poly_case(name):
    if name == "periodic":
        return inputs.polyhedra(density=2500.0, n=2000, spacing=1.45, jitter=0.08, seed=21, dt=2e-4, sigma_v=1.0, z0=0.75)
    if name == "walls":
        return inputs.polyhedra(density=2500.0, n=1500, spacing=1.5, jitter=0.05, seed=5, dt=2e-4, sigma_v=0.5, z0=0.6,
                                periodic=(False, False, False))
    raise KeyError(name)


def oracle_for(w):
    o = po.Oracle(w.particles, w.domain, w.walls)
    o.set_shapes(w.shapes)
    return o


def feature_table(ii, jj, tt, sw, si, sj, fr):
    """Stable sort by owner id: keeps each owner's list in storage order."""
    order = np.argsort(ii, kind="stable")
    keys = np.stack([ii.astype(np.int64), jj.astype(np.int64), tt.astype(np.int64), sw.astype(np.int64),
                     si.astype(np.int64), sj.astype(np.int64)], axis=1)
    return keys[order], fr[order]


def force_floor(w):
    p = by_id(w.particles)
    return p["mass"] * 9.81


def compare_state(g, o, floor, what):
    g, o = by_id(g), by_id(o)
    assert np.array_equal(g["id"], o["id"]), what
    L = max(1.0, float(np.max(np.abs(pos(o)))))
    dpos = float(np.max(np.abs(pos(g) - pos(o)))) / L
    vs = max(1e-3, float(np.max(np.abs(vel(o)))))
    dvel = float(np.max(np.abs(vel(g) - vel(o)))) / vs
    dq = float(np.max(np.abs(np.stack([g[k] - o[k] for k in ("qw", "qx", "qy", "qz")]))))
    ef = rel_err(force(g), force(o), floor)
    mscale = np.maximum(np.linalg.norm(vec(o, "mom"), axis=1), 1e-6 * float(np.max(floor)))
    em = float(np.max(np.linalg.norm(vec(g, "mom") - vec(o, "mom"), axis=1) / mscale))
    assert dpos <= TRAJ_TOL, f"{what}: positions differ by {dpos:.3e}"
    assert dvel <= TRAJ_TOL, f"{what}: velocities differ by {dvel:.3e}"
    assert dq <= TRAJ_TOL, f"{what}: orientations differ by {dq:.3e}"
    assert ef <= FORCE_TOL, f"{what}: forces differ by {ef:.3e} relative"
    assert em <= FORCE_TOL, f"{what}: moments differ by {em:.3e} relative"
    return dpos, dvel, ef, em


@pytest.mark.parametrize("case", ["periodic", "walls"])
def test_feature_lists_bit_exact(gpu_ok, case):
    w = poly_case(case)
    o = oracle_for(w)
    o.rebuild_poly(w.rcut_inc)
    s = PolySim(w)
    s.rebuild()
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert len(gk) == len(ok) and len(gk) > 100
    assert np.array_equal(gk, ok)
    assert np.array_equal(gf, of)
    types = np.bincount(gk[:, 2], minlength=6)
    assert types[0] + types[1] > 0 and types[2] > 0 and types[3] > 0, types
    if case == "walls":
        assert types[5] > 0


def aligned_cubes(n=1000, gap=0.01, jitter=0.002):
    """Axis-aligned cubes on a simple-cubic lattice, faces `gap` apart between the Minkowski shells (well
    inside rVerlet): face-to-face neighbours share about 28 features (4 VV, 16 VE, 8 VF)."""
    w = inputs.polyhedra(density=2500.0, n=n, spacing=1.0 + 2 * 0.02 + gap, jitter=jitter, seed=9, dt=2e-4)
    cube = w.shapes[0]
    assert cube.nv == 8
    p = w.particles
    p["type"] = np.zeros(w.n, dtype=np.uint32)
    p["radius"] = np.full(w.n, float(np.max(p["radius"])))
    p["mass"] = np.full(w.n, 2500.0 * cube.volume)
    for a in ("inx", "iny", "inz"):
        p[a] = p["mass"] * cube.inertia_on_mass[0]
    p["qw"], p["qx"], p["qy"], p["qz"] = np.ones(w.n), np.zeros(w.n), np.zeros(w.n), np.zeros(w.n)
    return w


@pytest.mark.parametrize("pool_words", [None, 2 * 232])
def test_feature_lists_through_overflow_paths(gpu_ok, monkeypatch, pool_words):
    """Aligned cubes face to face, whose pairs have more than the 24 features a list slot keeps during the
    enumeration: with the default pool their extra features come from pool chunks; with a pool of two
    chunks most of them are enumerated again, straight into place. The lists stay bit-exact with the
    oracle either way."""
    if pool_words is None:
        monkeypatch.delenv("XDEM_FEAT_POOL_WORDS", raising=False)
    else:
        monkeypatch.setenv("XDEM_FEAT_POOL_WORDS", str(pool_words))
    w = aligned_cubes()
    o = oracle_for(w)
    o.rebuild_poly(w.rcut_inc)
    s = PolySim(w)
    s.rebuild()
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert len(gk) == len(ok) and np.array_equal(gk, ok) and np.array_equal(gf, of)
    feat = gk[gk[:, 2] < 4]
    _, per_pair = np.unique(feat[:, :2], axis=0, return_counts=True)
    big = int(np.sum(per_pair > 24))
    print(f"pool {pool_words}: {len(per_pair)} pairs, {big} with more than 24 features, max {per_pair.max()}",
          flush=True)
    assert big >= 100


@pytest.mark.parametrize("case", ["periodic", "walls"])
def test_first_force_pass(gpu_ok, case):
    w = poly_case(case)
    sch = scheme(w)
    o = oracle_for(w)
    o.first_iteration_poly(sch)
    s = PolySim(w)
    s.first_iteration()
    g, q = by_id(s.ctx.download()), by_id(o.particles())
    floor = force_floor(w)
    assert rel_err(force(g), force(q), floor) <= FORCE_TOL
    mscale = np.maximum(np.linalg.norm(vec(q, "mom"), axis=1), 1e-6 * float(np.max(floor)))
    assert float(np.max(np.linalg.norm(vec(g, "mom") - vec(q, "mom"), axis=1) / mscale)) <= FORCE_TOL
    # some particles are in contact: the force differs from gravity alone
    fg = np.abs(force(q)[:, 2] + q["mass"] * 9.81)
    assert np.count_nonzero(fg > 1e-6 * q["mass"]) > 20
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert np.array_equal(gk, ok) and np.array_equal(gf, of)
    assert np.count_nonzero(np.abs(of).sum(axis=1)) > 10


@pytest.mark.parametrize("case", ["periodic", "walls"])
def test_run_steps_match_oracle(gpu_ok, case):
    """120 steps of the fused engine against the oracle's scheme, with vertex-displacement rebuilds."""
    w = poly_case(case)
    sch = scheme(w, poll=8)
    o = oracle_for(w)
    o.first_iteration_poly(sch)
    orb = o.run_steps_poly(sch, 120)
    s = PolySim(w)
    s.first_iteration()
    st = s.run(120, poll=8)
    assert st["rebuilds"] == orb and orb >= 1
    compare_state(s.ctx.download(), o.particles(), force_floor(w), case)
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert np.array_equal(gk, ok)
    assert np.array_equal(gf, of)


def test_engine_equals_operator_path(gpu_ok):
    w = poly_case("periodic")
    a = PolySim(w)
    a.first_iteration()
    for _ in range(40):
        a.step()
    b = PolySim(w)
    b.first_iteration()
    b.run(40, poll=4)
    assert a.rebuilds == b.rebuilds
    pa, pb = by_id(a.ctx.download()), by_id(b.ctx.download())
    for k in ("rx", "ry", "rz", "vx", "vy", "vz", "qw", "qx", "qy", "qz", "fx", "fy", "fz", "momx", "vrotx"):
        assert np.array_equal(pa[k], pb[k]), k
    ka, fa = feature_table(*a.ctx.poly_interactions())
    kb, fb = feature_table(*b.ctx.poly_interactions())
    assert np.array_equal(ka, kb) and np.array_equal(fa, fb)


def test_vertex_displ_over(gpu_ok):
    w = poly_case("periodic")
    s = PolySim(w)
    s.first_iteration()
    assert not s.ctx.vertex_displ_over(0.05)
    o = oracle_for(w)
    o.first_iteration_poly(scheme(w))
    for k in range(6):
        s.ctx.combined_compute_prolog(0.02)
        o.prolog(0.02)
        assert s.ctx.vertex_displ_over(0.05) == o.vertex_displ_over(0.05), k


def test_contact_state_dump(gpu_ok, tmp_path):
    """Recorded contact state of a polyhedron force pass (the reference functor's analysis tuple with
    the positions): one row per feature in contact and per vertex-wall contact; the vertex side comes
    first, as the reference's swapped pairs store it; ft is the feature's friction history; the rows'
    forces add up to each particle's force; the dump file reads back."""
    from exadem_amd import itools
    w = poly_case("walls")
    s = PolySim(w)
    s.ctx.set_contact_record(True)
    s.first_iteration()
    ii, jj, si, sj, tt, v = s.ctx.contact_state(subs=True)
    assert np.all(np.diff(tt.astype(np.int64)) >= 0)  # one block per type, as the reference writes
    feat, wall = tt < 4, tt == 5
    assert np.count_nonzero(feat) > 0 and np.count_nonzero(wall) > 0
    assert np.all(v[feat, 0] < 0)
    assert np.all(sj[wall] == 0xffffffff)
    fi, fj, ftp, fsw, fsi, fsj, ffr = s.ctx.poly_interactions()
    hist = {(int(a), int(b), int(t), int(x), int(y), int(z)): f
            for a, b, t, x, y, z, f in zip(fi, fj, ftp, fsw, fsi, fsj, ffr)}
    p = by_id(s.ctx.download())
    F = p["mass"][:, None] * np.asarray(w.gravity)[None, :]
    for k in range(len(ii)):
        a, b, t = int(ii[k]), int(jj[k]), int(tt[k])
        if t == 5:
            key = (a, b, 5, 0, int(si[k]), 0xffffffff)
        else:
            key = (a, b, t, 0, int(si[k]), int(sj[k]))
            if key not in hist:  # a swapped feature: the owner is the second particle
                key = (b, a, t, 1, int(sj[k]), int(si[k]))
        assert np.array_equal(v[k, 7:10], hist[key]), key
        assert np.array_equal(v[k, 10:13], pos(p)[a])
        f = v[k, 4:7] + v[k, 7:10]
        F[a] += f
        if t != 5:
            F[b] -= f
    assert rel_err(F, force(p), p["mass"] * 9.81) <= 1e-12
    path, rows = itools.write_dump(s.ctx, str(tmp_path), "InteractionOutputDir-", 0)
    keys, vals = itools.read_dump(path)
    assert rows == len(ii)
    assert np.array_equal(keys[:, 2], si.astype(np.int64)) and np.array_equal(keys[:, 3], sj.astype(np.int64))
    assert np.allclose(vals, v, rtol=1e-5, atol=1e-300)


def test_checkpoint_restart_with_history(gpu_ok, tmp_path):
    """Polyhedra restart with interaction history: a run checkpointed after 60 steps and restarted
    (particles uploaded, feature lists rebuilt, feature and vertex-wall histories handed over by key)
    is, bit for bit, the uninterrupted run with a neighbour rebuild at the checkpoint step, which is what
    a restart is: right after the restart the history equals the saved one, and 60 steps later
    positions, velocities and the active features with their history are identical. (A rebuild
    re-enumerates the features at the new positions, so a polyhedra run with an extra rebuild differs
    from one without it.) Without the history the state differs."""
    w = poly_case("walls")
    a = PolySim(w)
    a.first_iteration()
    a.run(60)
    ck = str(tmp_path / "restart.npz")
    a.checkpoint(ck)
    saved = np.load(ck)
    assert np.count_nonzero(np.any(saved["fr"] != 0, axis=1)) > 0
    a.rebuild()
    b = PolySim.restart(w, ck)
    c = PolySim.restart(w, ck, history=False)

    def active(sim):
        keys, fr = feature_table(*sim.ctx.poly_interactions())
        act = np.any(fr != 0, axis=1)
        k, f = keys[act], fr[act]
        order = np.lexsort(k.T[::-1])
        return k[order], f[order]

    ka, fa = active(a)
    kb, fb = active(b)
    assert len(ka) > 0 and np.array_equal(ka, kb) and np.array_equal(fa, fb)
    for sim in (a, b, c):
        sim.run(60)
    ka, fa = active(a)
    kb, fb = active(b)
    kc, fc = active(c)
    assert len(ka) > 0 and np.array_equal(ka, kb) and np.array_equal(fa, fb)
    pa, pb = by_id(a.ctx.download()), by_id(b.ctx.download())
    for k in ("rx", "ry", "rz", "vx", "vy", "vz", "qw", "qx", "vrotx", "fx", "momx"):
        assert np.array_equal(pa[k], pb[k]), k
    assert not np.array_equal(kc, ka) or not np.array_equal(fc, fa)


def test_simulation_state(gpu_ok):
    """simulation_state of polyhedra: energies and mass as the downloaded fields give them, interactions
    as the feature lists hold them (features twice, vertex-wall candidates once), the active ones (with
    history), and the smallest dn equal to the smallest dn the recorded contact state of the same pass
    holds."""
    w = poly_case("walls")
    s = PolySim(w)
    s.ctx.set_contact_record(True)
    s.first_iteration()
    st = s.ctx.simulation_state()
    p = by_id(s.ctx.download())
    m = p["mass"]
    ke = float(np.sum(0.5 * p["vx"] * p["vx"] * m))
    assert abs(st["kinetic_energy"][0] - ke) <= 1e-12 * max(ke, 1e-300)
    assert abs(st["mass"] - float(np.sum(m))) <= 1e-12 * float(np.sum(m))
    ii, jj, tt, sw, si, sj, fr = s.ctx.poly_interactions()
    coef = np.where(tt == 5, 1, 2)
    assert st["n_interactions"] == int(np.sum(coef))
    act = np.any(fr != 0, axis=1)
    assert st["n_active"] == int(np.sum(coef[act])) and st["n_active"] > 0
    _, _, _, v = s.ctx.contact_state()
    assert st["min_dn"] == min(0.0, float(np.min(v[:, 0]))) and st["min_dn"] < 0
    print(f"polyhedra: {st['n_interactions']} interactions, {st['n_active']} active, min dn {st['min_dn']:.6g}")


def test_classifier_waves(gpu_ok):
    """classify_interactions on the GPU (classify_interactions.cpp:52-136): the feature interactions split
    into one wave per type (VV, VE, VF, EE). Wave sizes equal the oracle's feature counts by type and the
    vertex-wall candidates its type-5 items; each wave holds exactly the list's rows of its type (owner,
    partner, swap, sub-features), in increasing list index; the waves together hold every feature once.
    The contact pass refuses lists that were not classified."""
    w = poly_case("walls")
    s = PolySim(w)
    s.first_iteration()
    o = oracle_for(w)
    o.first_iteration_poly(scheme(w))
    sizes = s.ctx.classifier_waves()
    ii, jj, tt, sw, si, sj, fr = s.ctx.poly_interactions()
    ot = o.poly_interactions()[2]
    assert np.array_equal(sizes[:4], np.bincount(ot[ot < 4], minlength=4))
    assert sizes[5] == int(np.count_nonzero(ot == 5)) and sizes[5] > 0
    assert np.all(sizes[:4] > 0) and np.all(sizes[6:] == 0) and sizes[4] == 0
    every = []
    for t in range(4):
        a, b, wsw, wsi, wsj, idx = s.ctx.classifier_wave(t)
        assert len(a) == sizes[t]
        assert np.all(np.diff(idx.astype(np.int64)) > 0)
        sel = tt == t
        got = sorted(zip(a.tolist(), b.tolist(), wsw.tolist(), wsi.tolist(), wsj.tolist()))
        ref = sorted(zip(ii[sel].tolist(), jj[sel].tolist(), sw[sel].tolist(), si[sel].tolist(), sj[sel].tolist()))
        assert got == ref, t
        every.append(idx)
    every = np.sort(np.concatenate(every).astype(np.int64))
    assert np.array_equal(every, np.arange(int(np.sum(sizes[:4]))))
    print(f"waves VV {sizes[0]}, VE {sizes[1]}, VF {sizes[2]}, EE {sizes[3]}, vertex-wall {sizes[5]}")
    # operator path: nbh_polyhedron without classify_interactions is refused by the contact pass
    c = s.ctx
    c.move_particles()
    c.chunk_neighbors_contact(w.rcut_inc)
    c.nbh_polyhedron(w.rcut_inc)
    c.reset_force_moment()
    with pytest.raises(native.XdemError, match="classify_interactions"):
        c.contact_polyhedron(w.cp, w.cpd, w.dt)
    c.classify_interactions()
    c.contact_polyhedron(w.cp, w.cpd, w.dt)


@pytest.mark.parametrize("n", [33, 1000, 32769])
def test_integrating_gather_matches_oracle(gpu_ok, n):
    """The engine's integrating gather (eight lanes per particle, four past 32,768) at block edges, with pair and wall
    contacts: the state after a chain of steps equals the oracle's bit for bit."""
    w = inputs.polyhedra(density=2500.0, n=n, spacing=1.35, jitter=0.05, seed=n, dt=2e-4, sigma_v=1.0, z0=0.5,
                         periodic=(n > 500, n > 500, False))
    s = PolySim(w)
    s.first_iteration()
    s.run(12, poll=5)
    o = oracle_for(w)
    o.first_iteration_poly(scheme(w))
    o.run_steps_poly(scheme(w), 12)
    a, b = by_id(s.ctx.download()), by_id(o.particles())
    for k in ("rx", "ry", "rz", "vx", "vy", "vz", "qw", "qx", "qy", "qz", "vrotx", "vroty", "vrotz", "fx", "fy", "fz",
              "momx", "momy", "momz"):
        assert np.array_equal(a[k], b[k]), k
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert np.array_equal(gk, ok) and np.array_equal(gf, of) and np.count_nonzero(gf) > 0


@pytest.mark.parametrize("n", [2, 9, 77, 1203])
def test_feature_enumeration_of_mixed_shapes(gpu_ok, n):
    """Sixteen lanes per pair: shapes that fill all vertex, edge and face lanes (cube, octahedron) and shapes that leave
    most of them idle (a rod: two vertices, one edge, no face; a sphere: one vertex), with numbers of pairs below and
    beyond a block: the feature lists equal the oracle's, word for word and in order."""
    rod, ball = shp.ShapeDef("rod"), shp.ShapeDef("sphere")
    rod.vertices, rod.edges = [(-0.6, 0.0, 0.0), (0.6, 0.0, 0.0)], [(0, 1)]
    ball.vertices = [(0.0, 0.0, 0.0)]
    for d, r in ((rod, 0.05), (ball, 0.4)):
        d.radius, d.volume, d.inertia_on_mass = r, 0.2, (0.1, 0.1, 0.1)
    w = inputs.polyhedra(density=2500.0, n=n, spacing=1.1, jitter=0.05, seed=n, dt=2e-4, z0=0.8,
                         periodic=(n > 500, n > 500, False))
    w.shapes = list(w.shapes) + [rod.to_record(), ball.to_record()]
    w.particles["type"] = (np.arange(n) * 7 // 3 % 4).astype(np.uint32)
    o = oracle_for(w)
    o.rebuild_poly(w.rcut_inc)
    s = PolySim(w)
    s.rebuild()
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert np.array_equal(gk, ok) and np.array_equal(gf, of)
    if n > 500:
        assert {0, 1, 2, 3} <= set(gk[:, 2]) and set(gk[gk[:, 2] > 0, 3]) == {0, 1}


@pytest.mark.parametrize("n", [7, 1203])
@pytest.mark.parametrize("kinds", [("ball",), ("rod",), ("rod", "ball"), ("tetra",), ("plate", "rod"), ("tetra", "ball")])
def test_feature_enumeration_of_small_shapes(gpu_ok, kinds, n):
    """Two, four and eight lanes per pair: particles of shapes without cubes and octahedra (registered with them, which
    does not count), whose vertices, edges and faces fill the lanes or leave some idle: the feature lists equal the
    oracle's, word for word and in order."""
    defs = {k: shp.ShapeDef(k) for k in ("rod", "ball", "tetra", "plate")}
    defs["rod"].vertices, defs["rod"].edges = [(-0.6, 0.0, 0.0), (0.6, 0.0, 0.0)], [(0, 1)]
    defs["ball"].vertices = [(0.0, 0.0, 0.0)]
    defs["tetra"].vertices = [(0.5, 0.5, 0.5), (-0.5, -0.5, 0.5), (-0.5, 0.5, -0.5), (0.5, -0.5, -0.5)]
    defs["tetra"].edges = [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]
    defs["tetra"].faces = [(0, 1, 2), (0, 3, 1), (0, 2, 3), (1, 3, 2)]
    defs["plate"].vertices = [(0.5, 0.5, 0.0), (-0.5, 0.5, 0.0), (-0.5, -0.5, 0.0), (0.5, -0.5, 0.0)]
    defs["plate"].edges, defs["plate"].faces = [(0, 1), (1, 2), (2, 3), (3, 0)], [(0, 1, 2, 3)]
    for k, d in defs.items():
        d.radius, d.volume, d.inertia_on_mass = 0.4 if k == "ball" else 0.05, 0.2, (0.1, 0.1, 0.1)
    w = inputs.polyhedra(density=2500.0, n=n, spacing=0.85 if kinds == ("ball",) else 1.0, jitter=0.05, seed=n, dt=2e-4,
                         z0=0.8, periodic=(n > 500, n > 500, False))
    w.shapes = list(w.shapes) + [defs[k].to_record() for k in kinds]
    w.particles["type"] = (2 + np.arange(n) * 7 // 3 % len(kinds)).astype(np.uint32)
    o = oracle_for(w)
    o.rebuild_poly(w.rcut_inc)
    s = PolySim(w)
    s.rebuild()
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert np.array_equal(gk, ok) and np.array_equal(gf, of)
    if n > 500:
        types = set(gk[:, 2])
        assert 0 in types
        if "rod" in kinds or "tetra" in kinds:
            assert {1, 3} <= types
        if "tetra" in kinds:
            assert 2 in types


@pytest.mark.parametrize("n", [41, 1203])
def test_histories_carried_over_rebuilds(gpu_ok, n):
    """Histories found again by feature: after several rebuilds with pairs in contact the lists and friction histories
    equal the oracle's bit for bit, over more or fewer features than a block."""
    w = inputs.polyhedra(density=2500.0, n=n, spacing=1.3, jitter=0.05, seed=n, dt=5e-4, sigma_v=3.0, z0=0.7,
                         periodic=(n > 500, n > 500, False))
    s = PolySim(w)
    s.first_iteration()
    st = s.run(60, poll=16)
    o = oracle_for(w)
    o.first_iteration_poly(scheme(w))
    o.run_steps_poly(scheme(w), 60)
    gk, gf = feature_table(*s.ctx.poly_interactions())
    ok, of = feature_table(*o.poly_interactions())
    assert st["rebuilds"] >= 2
    assert np.array_equal(gk, ok) and np.array_equal(gf, of) and np.count_nonzero(gf) > 0
