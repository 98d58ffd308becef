"""The launches that take a size or a form of their own: the fused step of engines
without bonded groups, its two contact kernels, the line to the two-launch step, the pair search's and the summation
runs' group sizes, the queries' order, the servo's two ways to its force sum, and
the calibration engine's gathers and tapes.  Sizes are the edges of waves, of the
64-particle groups, of the runs a group of lanes holds and of the dispatch rules.

Tolerances: events and lists bit-exact; a step's arithmetic is the oracle's up to
the order of a particle's sum, so positions after the few dozen steps here agree to
1e-9 of a radius (sums of up to 500 forces at 2^-53 each, grown by the contacts)."""
import ctypes
import importlib
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-9


@pytest.fixture(scope="module")
def spm(pkg):
    return importlib.import_module("esys_particle_amd.specimens")


def follow(pkg, orc, spm, spec, steps, names, batch=32, extra=None, lists=True):
    g = pkg.LsmMpi(stepsPerBatch=batch)
    o = orc.oracle_lsm_class(pkg)()
    for sim in (g, o):
        spm.apply(sim, spec)
        if extra:
            extra(sim)
    print("case: n=%d steps=%d batch=%d" % (len(spec["ids"]), steps, batch), flush=True)
    g.runTimeSteps(steps)
    o.runTimeSteps(steps)
    assert g.engine.rebuild_steps().tolist() == o.engine.rebuild_steps().tolist()
    if lists:
        np.testing.assert_array_equal(g.engine.neighbour_pairs(), o.engine.neighbour_pairs())
        for name in names:
            np.testing.assert_array_equal(g.getInteractionPairs(name), o.getInteractionPairs(name))
    r = float(np.mean(spec["rad"]))
    po = o.getParticleData("pos")
    assert np.max(np.abs(g.getParticleData("pos") - po)) <= TOL * r
    vo = o.getParticleData("vel")
    assert np.max(np.abs(g.getParticleData("vel") - vo)) <= TOL * max(np.abs(vo).max(), 1e-300)
    return g, o


def cloud(spm, n, seed=5):
    """n particles packed in a box with some moving into each other."""
    L = max(1.6, (n * 0.9) ** (1.0 / 3.0))
    spec = spm.gravity_settling(n=n, seed=seed, box=(L, 2.0 * L, L), dt=2e-3, k=100.0, wall_k=100.0)
    spec["vel"] = np.random.default_rng(seed).normal(0.0, 2.0, (n, 3))
    return spec


def hub(n_small=420, seed=3):
    """One large particle under a shell of small ones that overlap it: a run of
    more than 400 touching pairs in one group."""
    rng = np.random.default_rng(seed)
    k = np.arange(n_small) + 0.5
    phi, th = np.arccos(1.0 - 2.0 * k / n_small), np.pi * (1.0 + 5.0 ** 0.5) * k
    d = np.stack([np.cos(th) * np.sin(phi), np.sin(th) * np.sin(phi), np.cos(phi)], 1)
    R, r = 3.0, 0.12
    pos = np.concatenate([np.zeros((1, 3)), d * (R + 0.97 * r)]) + 5.0
    rad = np.concatenate([[R], np.full(n_small, r)])
    n = len(rad)
    return {"ptype": "RotSphere", "grid": 2 * R + 0.1, "alpha": 0.1, "dt": 1e-4,
            "domain": ((-3.0, -3.0, -3.0), (13.0, 13.0, 13.0)),
            "ids": np.arange(n, dtype=np.int32), "pos": pos, "rad": rad, "density": 1.0,
            "vel": rng.normal(0.0, 0.5, (n, 3)), "walls": []}


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257])
def test_elastic_step_sizes(pkg, orc, spm, n):
    g, o = follow(pkg, orc, spm, cloud(spm, n), 80, ["elastic"])
    np.testing.assert_allclose(g.engine.wall_force_history("bottom", 80),
                               o.engine.wall_force_history("bottom", 80), rtol=TOL, atol=1e-9)


def test_elastic_step_searches_and_queue_depth(pkg, orc, spm):
    """Several searches within a queue, with the same bits step by step."""
    spec = cloud(spm, 300)
    g, o = follow(pkg, orc, spm, spec, 200, ["elastic"], batch=64)
    assert len(o.engine.rebuild_steps()) >= 4
    s = pkg.LsmMpi(stepsPerBatch=1)
    spm.apply(s, spec)
    s.runTimeSteps(200)
    for f in ("pos", "vel"):
        assert s.getParticleData(f).tobytes() == g.getParticleData(f).tobytes()


def add_groups(pkg, form):
    def add(sim):
        if form in ("friction", "mixed"):
            sim.createInteractionGroup(pkg.RotFrictionPrms("fr", 200.0, 0.4, 0.4, 100.0))
        if form == "rigid":
            sim.createInteractionGroup(pkg.RotFrictionPrms("fr", 200.0, 0.4, 0.4, 100.0, rigid=True))
        if form in ("rotelastic", "mixed"):
            sim.createInteractionGroup(pkg.RotElasticPrms("el", 50.0))
        if form == "two":
            sim.createInteractionGroup(pkg.NRotElasticPrms("el", 50.0))
            sim.createInteractionGroup(pkg.NRotElasticPrms("fr", 25.0))
        if form == "nrot":
            sim.createInteractionGroup(pkg.NRotElasticPrms("el", 50.0))
    return add


NAMES = {"friction": ["fr"], "rigid": ["fr"], "rotelastic": ["el"], "mixed": ["fr", "el"],
         "two": ["el", "fr"], "nrot": ["el"]}


@pytest.mark.parametrize("form", ["friction", "rigid", "rotelastic", "mixed", "two"])
@pytest.mark.parametrize("n", [63, 65, 300])
def test_contact_block_forms(pkg, orc, spm, form, n):
    spec = cloud(spm, n, seed=n)
    spec["ptype"] = "RotSphere"
    spec["elastic"] = []
    g, o = follow(pkg, orc, spm, spec, 80, NAMES[form], extra=add_groups(pkg, form))
    assert np.max(np.abs(g.getParticleData("angvel") - o.getParticleData("angvel"))) <= \
        TOL * max(np.abs(o.getParticleData("angvel")).max(), 1e-300)
    if "fr" in NAMES[form] and form != "two":
        np.testing.assert_array_equal(g.engine.friction_state("fr")[1],
                                      o.engine.friction_state("fr")[1])


def launches(sim):
    """(steps in two launches, steps in all) since kernel timing was turned on."""
    kt = sim.engine.kernel_times()
    return kt["forces"][1], kt["gather_integrate"][1]


def skin(spec, alpha):
    spec["ptype"], spec["elastic"] = "RotSphere", []
    spec["alpha"], spec["grid"] = alpha, 1.0 + alpha
    return spec


@pytest.mark.parametrize("form,n,alpha,fused", [
    ("friction", 300, 0.8, True), ("friction", 300, 1.2, False),
    ("rigid", 300, 0.8, True), ("rigid", 300, 1.2, False),
    ("mixed", 300, 0.2, True), ("mixed", 300, 0.8, False),
    ("rotelastic", 300, 0.8, True), ("rotelastic", 300, 1.2, False),
    ("two", 300, 0.2, True), ("two", 300, 1.2, False),
    ("nrot", 300, 1.6, True), ("nrot", 300, 2.0, False), ("nrot", 2000, 2.0, True)])
def test_one_launch_or_two(pkg, orc, spm, form, n, alpha, fused):
    """Skins to both sides of the pairs a particle up to which a step is one launch."""
    g, o = follow(pkg, orc, spm, skin(cloud(spm, n, seed=n), alpha), 40, NAMES[form],
                  extra=add_groups(pkg, form))
    g.engine.set_kernel_timing(True)
    for sim in (g, o):
        sim.runTimeSteps(10)
    assert launches(g) == (0 if fused else 10, 10)
    g.engine.check_state()
    assert np.max(np.abs(g.getParticleData("pos") - o.getParticleData("pos"))) <= TOL


def test_form_changes_during_a_run(pkg, orc, spm):
    """A cloud that contracts: one launch a step while it is loose, two once it is
    dense, with the oracle's lists, history and walls throughout."""
    spec = skin(cloud(spm, 300, seed=300), 0.8)
    mid = spec["pos"].mean(0)
    spec["vel"] = -4.0 * (spec["pos"] - mid)
    g, o = pkg.LsmMpi(stepsPerBatch=32), orc.oracle_lsm_class(pkg)()
    for sim in (g, o):
        spm.apply(sim, spec)
        add_groups(pkg, "friction")(sim)
    g.engine.set_kernel_timing(True)
    print("case: contracting cloud", flush=True)
    for _ in range(4):
        for sim in (g, o):
            sim.runTimeSteps(30)
        g.engine.check_state()
        assert np.max(np.abs(g.getParticleData("pos") - o.getParticleData("pos"))) <= TOL
        np.testing.assert_array_equal(g.getInteractionPairs("fr"), o.getInteractionPairs("fr"))
        np.testing.assert_array_equal(g.engine.friction_state("fr")[1],
                                      o.engine.friction_state("fr")[1])
        np.testing.assert_allclose(list(g.getWallForce("bottom")), list(o.getWallForce("bottom")),
                                   rtol=1e-9, atol=1e-9)
    assert g.engine.rebuild_steps().tolist() == o.engine.rebuild_steps().tolist()
    two, every = launches(g)
    assert 0 < two < every


@pytest.mark.parametrize("form", ["nrot", "friction", "mixed"])
def test_long_runs(pkg, orc, spm, form):
    """More pairs of one particle than a search run (192) or a block's packed
    entries (320 touching, 512) hold."""
    g, o = follow(pkg, orc, spm, hub(), 20, NAMES[form], extra=add_groups(pkg, form))
    assert len(o.engine.neighbour_pairs()) > 400


@pytest.mark.parametrize("n_small", [190, 191, 192, 193, 1000])
def test_search_around_one_large_particle(pkg, orc, spm, n_small):
    """The large particle's partners around the 192 that are placed by counting, and
    far past them.  A search around the 1,000 takes 20 ms, 170 where they are placed
    by counting, too: the bound lies between."""
    spec = hub(n_small)
    spec["vel"][:] = (600.0, 0.0, 0.0)  # past half the skin in every step
    follow(pkg, orc, spm, spec, 4, ["el"], extra=add_groups(pkg, "nrot"))
    g = pkg.LsmMpi(stepsPerBatch=32)
    spm.apply(g, spec)
    add_groups(pkg, "nrot")(g)
    g.runTimeSteps(4)
    before, t = g.getStats()["num_rebuilds"], time.perf_counter()
    g.runTimeSteps(30)
    ms = (time.perf_counter() - t) * 1e3 / (g.getStats()["num_rebuilds"] - before)
    print("case: %d around one, %.2f ms a search" % (n_small, ms), flush=True)
    assert ms < 60.0


@pytest.mark.parametrize("tagged", [False, True])
def test_long_search_runs_with_large_skin(pkg, orc, spm, tagged):
    """A search cutoff that gives every particle hundreds of neighbours, with and
    without a tag mask on the group."""
    spec = cloud(spm, 500)
    spec["alpha"], spec["grid"] = 6.0, 7.0
    spec["elastic"] = [] if tagged else spec["elastic"]
    spec["tags"] = (np.arange(500) % 2).astype(np.int32)

    def add(sim):
        if tagged:
            sim.createInteractionGroupTagged(pkg.NRotElasticPrms("elastic", 100.0), 1, 1, 0, 1)
    follow(pkg, orc, spm, spec, 30, ["elastic"], extra=add)


@pytest.mark.parametrize("n", [8191, 8193, 16385, 33000])
def test_search_at_scan_sizes(pkg, orc, spm, n):
    spec = spm.gravity_settling(n=n, seed=n, box=(30.0, 90.0, 30.0))
    follow(pkg, orc, spm, spec, 3, ["elastic"])


def test_queries_with_sparse_ids(pkg, orc, spm):
    spec = cloud(spm, 130)
    rng = np.random.default_rng(4)
    spec["ids"] = np.sort(rng.choice(10 ** 6, 130, replace=False)).astype(np.int32)[
        rng.permutation(130)]
    g, o = follow(pkg, orc, spm, spec, 40, ["elastic"])
    np.testing.assert_array_equal(g.getParticleData("rad"), o.getParticleData("rad"))


def test_servo_with_untagged_particle_at_the_wall(pkg, orc, spm):
    """A wall's untagged particles are not bonded to it but may touch it: the servo
    then iterates over the candidates instead of one pass of sums."""
    spec = spm.shear_cell(n=600, seed=3, phi=0.35, dt=5e-4, wall_speed=10.0)
    spec["vel"] = np.random.default_rng(3).normal(0.0, 2.0, (600, 3))
    tags = np.array(spec["tags"])
    tag = spec["bonded_walls"][1][4]
    mine = np.flatnonzero(tags == tag)
    assert len(mine) > 4
    tags[mine[::2]] = 1
    spec["tags"] = tags
    g, o = follow(pkg, orc, spm, spec, 60, ["friction"])
    np.testing.assert_allclose(list(g.getWallPosition("top")), list(o.getWallPosition("top")),
                               rtol=1e-12, atol=1e-12)


def column(spm, flyers=40):
    """4 x 40 x 4 spheres apart from each other between two bonded walls, most
    64-particle groups away from both; some of the middle ones fly out of the domain
    in the first step."""
    k = np.stack(np.meshgrid(np.arange(4), np.arange(40), np.arange(4), indexing="ij"), -1)
    pos = 1.2 * k.reshape(-1, 3) + 0.6
    n = len(pos)
    tags = np.ones(n, np.int32)
    tags[pos[:, 1] < 2.0] = 2
    tags[pos[:, 1] > 46.0] = 3
    mid = np.flatnonzero(np.abs(pos[:, 1] - 20.0) < 5.0)[:flyers]
    vel = np.random.default_rng(8).normal(0.0, 0.5, (n, 3))
    vel[mid, 2] = 4e4  # 20 diameters a step
    v = 1e-3
    return {"ptype": "RotSphere", "grid": 1.4, "alpha": 0.2, "dt": 5e-4,
            "domain": ((-1.0, -2.0, -1.0), (6.0, 50.0, 6.0)),
            "ids": np.random.default_rng(9).permutation(n).astype(np.int32), "pos": pos,
            "rad": np.full(n, 0.5), "tags": tags, "vel": vel, "density": 1.0,
            "friction": ("friction", 1e3, 0.5, 0.5, 1e3), "walls": [],
            "bonded_walls": [("bottom", (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 1e3, 2, (v, 0.0, 0.0)),
                             ("top", (0.0, 48.0, 0.0), (0.0, -1.0, 0.0), 1e3, 3, (0.0, 0.0, 0.0))]}


@pytest.mark.parametrize("noalloc", [False, True])
def test_servo_after_checkpoint_that_erased_particles(pkg, orc, spm, tmp_path, noalloc):
    """A checkpoint's search erases the particles outside the domain and moves the
    slots of those behind them; a servo call before the next step still sums over
    every candidate of its wall."""
    spec = column(spm)
    n = len(spec["ids"])
    g, o = pkg.LsmMpi(stepsPerBatch=32), orc.oracle_lsm_class(pkg)()
    for sim in (g, o):
        spm.apply(sim, spec)
        sim.runTimeSteps(1)
    # (the oracle erases them at its next step's search: no wall candidate is among them)
    g.engine.save_checkpoint(str(tmp_path / "cp"), 0, 12)
    assert g.getNumParticles() == n - 40
    force = [0.0, -30.0, 4.0]
    print("case: servo after a checkpoint, n=%d, noalloc=%d" % (n, noalloc), flush=True)
    g.engine.check_state()
    for _ in range(3):  # before the step after the checkpoint, and between later steps
        if noalloc:
            g.engine.apply_force_to_wall_noalloc("top_bonds", force)
        else:
            g.applyForceToWall("top_bonds", force)
        o.applyForceToWall("top_bonds", force)
        np.testing.assert_allclose(list(g.getWallPosition("top")), list(o.getWallPosition("top")),
                                   rtol=1e-12, atol=1e-12)
        for sim in (g, o):
            sim.runTimeSteps(4)
        g.engine.check_state()
    r = 0.5
    assert np.max(np.abs(g.getParticleData("pos") - o.getParticleData("pos"))) <= TOL * r


# ---- the calibration engine ----
@pytest.fixture(scope="module")
def cal(pkg):
    return importlib.import_module("esys_particle_amd.calibration")


@pytest.fixture(scope="module")
def weak(spm):
    return spm.dense_bonded_compression(n=1500, seed=9, coh_mean=2.0, coh_sd=0.2, wall_speed=20.0)


THETA = np.array([1e5, 3e4, 2.0, 0.3])


@pytest.mark.parametrize("K", [1, 37, 100])
def test_tape_equals_checkpoints(cal, weak, K):
    """A plain run keeps every state, a tangent run checkpoints: the sweeps over
    both give the same bits, over neighbour searches and broken bonds."""
    # the small skin makes the run search for neighbours again and again
    m = cal.DiffModel.from_specimens([weak], 200, 20, checkpoint_every=K, alpha=0.02)
    target = np.full((1, m.nsamples), 5.0)
    st, loss = m.forward(THETA, target)
    g = m.backward()
    pos = m.particle_data("pos")
    assert len(m.bond_breaks()) > 100 and len(m.rebuild_steps()) > 1
    st2, loss2, _ = m.forward_tangent(THETA, np.ones((1, 4)), target)
    np.testing.assert_array_equal(st2, st)
    np.testing.assert_array_equal(m.particle_data("pos"), pos)
    for _ in range(2):  # the second sweep starts from what the first left
        np.testing.assert_array_equal(m.backward(), g)
        np.testing.assert_array_equal(m.particle_data("pos"), pos)


def pairs_within(spec, alpha):
    """Neighbour pairs a search of the specimen lists."""
    spatial = pytest.importorskip("scipy.spatial")
    pos, rad = np.asarray(spec["pos"]), np.asarray(spec["rad"])
    a, b = spatial.cKDTree(pos).query_pairs(2 * rad.max() + alpha, output_type="ndarray").T
    return int(np.sum(np.linalg.norm(pos[a] - pos[b], axis=1) <= rad[a] + rad[b] + alpha))


def test_tape_limit(cal, weak):
    """Past its limit a tape is given back, before the run, in the middle of it (a
    later search lists more pairs than the first) or between a run and its gradient;
    losses, gradients and the final state keep their bits."""
    steps, n = 200, len(weak["rad"])
    target = np.full((1, 10), 5.0)
    states = 32 * 4 * n * (steps + 1)
    first = 32 * steps * pairs_within(weak, 0.02)
    ref = None
    for limit, kept in ((24 << 30, True), (states + first, False), (states, False), (0, False)):
        m = cal.DiffModel.from_specimens([weak], steps, 20, checkpoint_every=37, alpha=0.02)
        m.set_tape_limit(limit)
        for rep in range(2):
            out = m.forward(THETA, target) + (m.backward(), m.particle_data("pos"))
            assert (m.tape_bytes() > 0) == kept and m.tape_bytes() <= limit
            ref = out if ref is None else ref
            for a, b in zip(out, ref):
                np.testing.assert_array_equal(a, b)
        if kept:
            assert m.tape_bytes() > states + first  # the searches do list more pairs
    m = cal.DiffModel.from_specimens([weak], steps, 20, checkpoint_every=37, alpha=0.02)
    m.forward(THETA, target)
    m.set_tape_limit(states)
    assert m.tape_bytes() == 0
    # of the next forward run, not of the run whose gradient follows
    m.lib.esp_diff_set_gravity(m.h, (ctypes.c_double * 3)(0.0, -50.0, 0.0))
    for _ in range(2):
        np.testing.assert_array_equal(m.particle_data("pos"), ref[3])
        np.testing.assert_array_equal(m.backward(), ref[2])


@pytest.mark.parametrize("copies", [1, 25])
def test_checkpointed_batch_equals_tape(cal, weak, copies):
    """Forward runs stepped in place and segments recomputed for the sweep, in a row
    of lanes a particle and (37,500 particles) in quads, against the tape; segments
    shorter and longer than the run."""
    th = np.tile(THETA, (copies, 1))
    ref = None
    for K, limit in ((9, 24 << 30), (9, 0), (64, 0)):
        m = cal.DiffModel.from_specimens([weak] * copies, 40, 10, checkpoint_every=K, alpha=0.05)
        m.set_tape_limit(limit)
        out = m.forward(th, np.full((copies, 4), 3.0)) + (m.backward(), m.particle_data("quat"))
        ref = out if ref is None else ref
        for a, b in zip(out, ref):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("copies", [7, 25])
def test_wide_batch_equals_single(cal, weak, copies):
    """Past the sizes where a particle's row of lanes becomes a quad (8,192 in the
    forward gather, 32,768 in the adjoint) a specimen keeps its bits."""
    mb = cal.DiffModel.from_specimens([weak] * copies, 40, 10)
    th = np.tile(THETA, (copies, 1))
    target = np.full((copies, mb.nsamples), 3.0)
    _, lb = mb.forward(th, target)
    gb = mb.backward()
    for s in (0, copies - 1):
        ms = cal.DiffModel.from_specimens([weak], 40, 10, x_start=mb.starts[s])
        _, ls = ms.forward(THETA, target[:1])
        assert lb[s] == ls[0]
        np.testing.assert_array_equal(gb[s], ms.backward()[0])


@pytest.mark.parametrize("nx", [31, 33])
def test_bonded_gather_sizes(pkg, orc, spm, nx):
    """Below and past 32,768 particles the bonded gather keeps three active slots of
    a particle in flight a lane, or one."""
    spec = spm.lattice_block(nx=nx, ny=32, nz=32, dt=1e-4, vel_sd=0.05)
    g, o = follow(pkg, orc, spm, spec, 12, ["bonded", "friction"], lists=False)
    np.testing.assert_array_equal(g.getBondBreaks(), o.getBondBreaks())
