"""A step's launch variants give one result: what a rule on sizes, options or
the launch's scenes picks between must not change a bit of it."""
import numpy as np
import pytest

from sph_amd import configs, sphg

pytestmark = pytest.mark.gpu

METHODS = [sphg.WCSPH, sphg.PCISPH, sphg.DFSPH]
FORCES = {
    "none": {},
    "xsph": dict(viscosity_method=sphg.VISCOSITY_XSPH, viscosity=0.02, boundary_viscosity=0.01),
    "cohesion": dict(surface_tension_method=sphg.SURFACE_TENSION_AKINCI, surface_tension=0.05),
    "adhesion": dict(adhesion_method=sphg.ADHESION_AKINCI, adhesion=0.1),
    "standard": dict(viscosity_method=sphg.VISCOSITY_STANDARD, viscosity=0.01),
}
FORCES["xsph_cohesion"] = {**FORCES["xsph"], **FORCES["cohesion"]}
FORCES["all"] = {**FORCES["xsph_cohesion"], **FORCES["adhesion"]}


def fields(scene):
    out = [scene.get(sphg.FIELD_X), scene.get(sphg.FIELD_V), scene.get(sphg.FIELD_A), scene.get(sphg.FIELD_DRHO)]
    if scene.params.method == sphg.DFSPH:
        out += [scene.get(sphg.FIELD_K), scene.get(sphg.FIELD_KV)]
    return out


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(fields(a), fields(b)))


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("forces", sorted(FORCES))
def test_forces_kernel_of_one_and_of_mixed_options(ctx, method, forces):
    """Alone, a scene's forces run in the kernel compiled for its options; in
    a batch with a scene of other options, in the general one.  The ragged
    size leaves the last wavefront partly empty."""
    other = "standard" if forces != "standard" else "xsph"
    specs = [configs.small_scene(method, n_side=(9, 7, 8), box=(1.2, 0.55, 0.8), **FORCES[f]) for f in (forces, other)]
    alone, mixed, extra = [sphg.Scene(ctx, s.params, s.fluid, s.boundary) for s in (specs[0], specs[0], specs[1])]
    alone.step(4)
    ctx.batch_step([mixed, extra], 4)
    assert same(alone, mixed)
    for s in (alone, mixed, extra):
        s.close()


def scalars(scene):
    s = scene.scalars()
    return [(n, getattr(s, n)) for n, _ in s._fields_]


def moving(spec, seed=5, speed=1.0):
    """Random velocities: iteration counts that change from step to step, so
    that steps launched ahead need more iterations than were predicted."""
    return np.random.default_rng(seed).uniform(-speed, speed, spec.fluid.shape).astype(np.float32)


LOOPS = {
    "plain": {},
    "none_at_least": dict(min_iterations=0, min_iterations_v=0),
    "one_at_least": dict(min_iterations=1),
    "many_at_least": dict(min_iterations=5, min_iterations_v=3),
    "to_the_cap": dict(eta=0.0, eta_v=0.0, max_iterations=7),
    "cap_below_minimum": dict(min_iterations=4, min_iterations_v=4, max_iterations=2),
    "no_iterations": dict(max_iterations=0),
    "loose": dict(eta=10.0, eta_v=1e6),
}


@pytest.mark.parametrize("method", [sphg.DFSPH, sphg.PCISPH])
@pytest.mark.parametrize("loops", sorted(LOOPS))
@pytest.mark.parametrize("size", [(3, 3, 3), (9, 7, 8), (31, 17, 9)])
def test_lone_scene_steps_like_one_of_a_batch(ctx, method, loops, size):
    """A lone scene decides its loops in the sweeps and launches its steps
    ahead; in a batch the host asks after finalize kernels.  Uneven calls, so
    that predictions are carried over, and single steps."""
    spec = configs.small_scene(method, n_side=size, box=tuple(0.05 * (s + 4) for s in size), **LOOPS[loops])
    v = moving(spec)
    alone, mixed, extra = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(3)]
    for steps in (1, 6, 2, 9):
        a, b = alone.step(steps), ctx.batch_step([mixed, extra], steps)
        assert 2 * a.iterations == b.iterations and 2 * a.iterations_v == b.iterations_v
        assert scalars(alone) == scalars(mixed)
    assert same(alone, mixed)
    for s in (alone, mixed, extra):
        s.close()


@pytest.mark.parametrize("method", [sphg.DFSPH, sphg.PCISPH])
def test_loops_decided_by_finalize_kernels_in_a_large_lone_scene(ctx, method):
    """2,048 chunks of 256 are the most whose partials every block adds up."""
    for size in ((128, 64, 64), (129, 64, 64)):
        spec = configs.small_scene(method, n_side=size, spacing=0.02, box=tuple(0.02 * (s + 4) for s in size))
        other = configs.small_scene(method, n_side=5)
        v = moving(spec, speed=0.3)
        alone, mixed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(2)]
        extra = sphg.Scene(ctx, other.params, other.fluid, other.boundary)
        alone.step(5)
        ctx.batch_step([mixed, extra], 5)
        assert scalars(alone) == scalars(mixed) and same(alone, mixed)
        for s in (alone, mixed, extra):
            s.close()


@pytest.mark.parametrize("method", [sphg.DFSPH, sphg.PCISPH])
def test_lone_scene_with_replay_schedules_and_timing(ctx, method):
    """Captured segments, launch schedules and kernel timing change which
    launches are made ahead, not what they compute."""
    spec = configs.small_scene(method, n_side=(12, 9, 8), box=(0.9, 0.65, 0.6))
    v = moving(spec)
    base, replay, timed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(3)]
    base.step(24)
    ctx.set_graphs(True)
    for steps in (1, 3, 10, 10):
        replay.step(steps)
    ctx.set_graphs(False)
    timed.step(3)
    ctx.kernel_timing(True)
    timed.step(4)
    launches = ctx.kernel_time("build")[0]
    ctx.kernel_timing(False)
    timed.step(17)
    assert launches == 4
    assert scalars(base) == scalars(replay) == scalars(timed)
    assert same(base, replay) and same(base, timed)
    for s in (base, replay, timed):
        s.close()


@pytest.mark.parametrize("cells", [31 * 1024 + 1, 32 * 1024, 33 * 1024, 90 * 1024])
def test_cell_scan_in_one_and_two_launches(ctx, cells):
    """Up to 32 scan chunks of 1,024 cells the counts are scanned in one
    launch.  A domain stretched along z keeps every cell's index."""
    from dataclasses import replace
    spec = configs.small_scene(sphg.WCSPH, n_side=(9, 7, 8), box=(0.9, 0.55, 0.8))
    pts = np.concatenate([spec.fluid, spec.boundary]).astype(np.float64)
    lo, hi = pts.min(axis=0), pts.max(axis=0)
    g = sphg.Scene(ctx, replace(spec.params, domain_min=tuple(lo), domain_max=tuple(hi)), spec.fluid, spec.boundary)
    h = spec.params.support_radius
    layer = np.prod([np.floor(hi[a] / h) - np.floor(lo[a] / h) + 5 for a in (0, 1)])
    tall = replace(spec.params, domain_min=tuple(lo), domain_max=(hi[0], hi[1], h * np.ceil(cells / layer)))
    t = sphg.Scene(ctx, tall, spec.fluid, spec.boundary)
    assert g.info()["ncells"] <= 32 * 1024 and abs(t.info()["ncells"] - cells) <= 8 * layer
    g.step(6)
    t.step(6)
    assert same(g, t)
    g.close()
    t.close()


def build_fields(scene):
    out = fields(scene) + [scene.get(sphg.FIELD_NNB), scene.get(sphg.FIELD_NGRAD)]
    if scene.params.method == sphg.DFSPH:
        out += [scene.get(sphg.FIELD_ALPHA), scene.get(sphg.FIELD_DIVERR)]
    if scene.params.method == sphg.PCISPH:
        out += [scene.get(sphg.FIELD_NSH)]
    counts, ids = scene.neighbors(((scene.params.max_neighbors or 96) + 3) & ~3)
    return out + [counts, np.where(np.arange(ids.shape[1])[None, :] < counts[:, None], ids, 0)]


def block_of(n, spacing, jitter, seed, at=0.06):
    side = int(np.ceil(n ** (1.0 / 3.0)))
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    rng = np.random.default_rng(seed)
    return ((grid + rng.uniform(-jitter, jitter, grid.shape)) * spacing + at).astype(np.float32)


@pytest.fixture(scope="module")
def crowd(ctx):
    """For each method a scene that brings a launch past the sizes at which a
    particle has 4 lanes in the list build and the PCISPH density sweep."""
    out = {}
    for m in METHODS:
        spec = configs.small_scene(m, n_side=59, spacing=0.02)
        out[m] = sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary)
    yield out
    for s in out.values():
        s.close()


BUILDS = {
    # name: (particles, spacing in 2r, jitter, boundary sampling in h, more)
    "one": (1, 1.0, 0.0, 1.0, {}),
    "group_less_one": (63, 1.0, 0.2, 1.0, {}),
    "group": (64, 1.0, 0.2, 1.0, {}),
    "group_and_one": (65, 1.0, 0.2, 1.0, {}),
    "chunk_and_one": (257, 1.0, 0.3, 1.0, {}),
    "disordered": (3000, 0.9, 0.5, 1.0, FORCES["adhesion"]),
    "sparse": (700, 3.0, 0.9, 1.0, FORCES["adhesion"]),
    # rows that do not fit the stage, boundary candidates that do not, lists
    # of several hundred
    "half_spacing": (1500, 0.5, 0.1, 1.0, dict(max_neighbors=500)),
    "dense_walls": (1200, 1.0, 0.1, 0.25, FORCES["adhesion"]),
    "few_slots": (500, 1.3, 0.1, 1.0, dict(max_neighbors=29)),
}


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("name", sorted(BUILDS))
def test_list_build_with_four_lanes_a_particle(ctx, crowd, method, name):
    """A small scene's lists are built with 4 lanes a particle, in a large
    launch with one: the same lists, sums and steps, bit for bit."""
    n, gap, jitter, walls, more = BUILDS[name]
    r = 0.01
    p = configs.small_scene(method, n_side=2, spacing=2 * r, **more).params
    p.domain_min, p.domain_max = (-0.1, -0.1, -0.1), (0.5, 0.4, 0.4)   # some leave it: cells clamped
    x = block_of(n, gap * 2 * r, jitter, 11)
    v = np.random.default_rng(2).uniform(-0.5, 0.5, x.shape).astype(np.float32)
    b = sphg.sample_box((0.02, 0.02, 0.02), (0.6, 0.4, 0.45), walls * 4 * r)
    alone, mixed = [sphg.Scene(ctx, p, x, b, v) for _ in range(2)]
    most = 0
    for _ in range(3):
        alone.step(1)
        ctx.batch_step([mixed, crowd[method]], 1)
        for a, m in zip(build_fields(alone), build_fields(mixed)):
            assert np.array_equal(a, m, equal_nan=True)
        most = max(most, alone.get(sphg.FIELD_NNB).max())
    assert most > (12 if name in ("disordered", "half_spacing", "dense_walls") else -1)
    alone.close()
    mixed.close()


@pytest.mark.parametrize("method", METHODS)
def test_four_lane_build_with_overflow_and_nan(ctx, crowd, method):
    """Too many neighbors are refused alike, and a NaN position stays its own
    particle's."""
    r = 0.01
    p = configs.small_scene(method, n_side=2, spacing=2 * r, max_neighbors=40).params
    b = sphg.sample_box((0.0, 0.0, 0.0), (0.4, 0.4, 0.4), 4 * r)
    x = block_of(700, 0.7 * 2 * r, 0.1, 3)
    alone, mixed = [sphg.Scene(ctx, p, x, b) for _ in range(2)]
    for step in (lambda: alone.step(1), lambda: ctx.batch_step([mixed, crowd[method]], 1)):
        with pytest.raises(sphg.SphgError) as err:
            step()
        assert err.value.code == sphg.EOVERFLOW
    assert alone.scalars().neighbor_overflow == mixed.scalars().neighbor_overflow > 40
    assert np.array_equal(alone.get(sphg.FIELD_NNB), mixed.get(sphg.FIELD_NNB))
    alone.close()
    mixed.close()
    p.max_neighbors = 0
    x = block_of(300, 2 * r, 0.1, 4)
    alone, mixed = [sphg.Scene(ctx, p, x, b) for _ in range(2)]
    x = x.copy()
    x[77, 1] = np.nan
    for s in (alone, mixed):
        s.set_state(x, np.zeros_like(x))
    alone.step(1)
    ctx.batch_step([mixed, crowd[method]], 1)
    assert all(np.array_equal(a, m, equal_nan=True) for a, m in zip(build_fields(alone), build_fields(mixed)))
    assert np.isfinite(np.delete(alone.get(sphg.FIELD_X), 77, 0)).all()
    alone.close()
    mixed.close()


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("forces", ["none", "xsph", "cohesion", "xsph_cohesion"])
@pytest.mark.parametrize("n", [1, 63, 65, 257, 3000])
def test_sweeps_with_four_lanes_a_particle(ctx, crowd, method, forces, n):
    """The sweeps of a small launch, of one scene and of a batch, give a
    particle 4 lanes, those of a large one give it one: the same sums."""
    r = 0.01
    p = configs.small_scene(method, n_side=2, spacing=2 * r, **FORCES[forces]).params
    x = block_of(n, 2 * r, 0.3, 7)
    v = np.random.default_rng(8).uniform(-0.5, 0.5, x.shape).astype(np.float32)
    b = sphg.sample_box((0.02, 0.02, 0.02), (0.6, 0.4, 0.45), 4 * r)
    alone, pair, twin, mixed = [sphg.Scene(ctx, p, x, b, v) for _ in range(4)]
    for _ in range(4):
        alone.step(1)
        ctx.batch_step([pair, twin], 1)
        ctx.batch_step([mixed, crowd[method]], 1)
        assert scalars(alone) == scalars(pair) == scalars(twin) == scalars(mixed)
        assert same(alone, pair) and same(alone, twin) and same(alone, mixed)
    for s in (alone, pair, twin, mixed):
        s.close()


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("side", [32, 33, 36, 37, 40, 41, 46, 47])
def test_lines_of_the_four_lane_sweeps(ctx, crowd, method, side):
    """Both sides of 128, 192, 256 and 384 chunks of 256 particles."""
    spec = configs.small_scene(method, n_side=side, spacing=0.02, **FORCES["xsph_cohesion"])
    v = moving(spec, speed=0.3)
    alone, mixed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(2)]
    alone.step(3)
    ctx.batch_step([mixed, crowd[method]], 3)
    assert scalars(alone) == scalars(mixed) and same(alone, mixed)
    alone.close()
    mixed.close()


@pytest.mark.parametrize("method", [sphg.DFSPH, sphg.PCISPH])
def test_large_lone_scene_with_kernel_timing(ctx, method):
    """While kernels are timed the host asks after the predicted iterations;
    in a large scene those are decided one by one as well, so that a step
    ends where its loop does."""
    spec = configs.small_scene(method, n_side=(129, 64, 64), spacing=0.02, box=tuple(0.02 * (s + 4) for s in (129, 64, 64)))
    v = moving(spec, speed=0.3)
    plain, timed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(2)]
    plain.step(8)
    ctx.kernel_timing(True)
    timed.step(8)
    ctx.kernel_timing(False)
    assert scalars(plain) == scalars(timed) and same(plain, timed)
    plain.close()
    timed.close()


@pytest.mark.parametrize("method", [sphg.DFSPH, sphg.PCISPH])
@pytest.mark.parametrize("loops", sorted(LOOPS))
def test_large_lone_scene_loop_limits(ctx, method, loops):
    """The loop limits of test_lone_scene_steps_like_one_of_a_batch where a
    kernel of its own decides the loops."""
    spec = configs.small_scene(method, n_side=(129, 64, 64), spacing=0.02, box=tuple(0.02 * (s + 4) for s in (129, 64, 64)),
                               **LOOPS[loops])
    other = configs.small_scene(method, n_side=5)
    v = moving(spec, speed=0.3)
    alone, mixed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v) for _ in range(2)]
    extra = sphg.Scene(ctx, other.params, other.fluid, other.boundary)
    for steps in (1, 5, 2):
        alone.step(steps)
        ctx.batch_step([mixed, extra], steps)
        assert scalars(alone) == scalars(mixed)
    assert same(alone, mixed)
    for s in (alone, mixed, extra):
        s.close()


def inflow(method, budget, fluid=None, start=3.5, **kw):
    """A scene with room for `budget` more particles, the first of which enter
    after `start` steps; without `fluid` it begins empty."""
    spec = configs.small_scene(method, n_side=4, **kw)
    em = sphg.Emitter(type=sphg.EMITTER_CIRCLE, num_particles=budget, position=(0.5, 0.26, 0.5), velocity=5.0,
                      rotation=(0.0, 1.0, 0.0, 0.0), start_time=start * spec.params.time_step, width=0.1, spacing=1.0)
    return spec.params, np.zeros((0, 3), np.float32) if fluid is None else fluid, spec.boundary, [em]


def test_pcisph_densities_without_active_particles(ctx):
    """A group without an active particle, among them those of a scene that is
    still empty, reads none and has an error of zero: the loop takes its
    minimum of iterations."""
    p, x, b, em = inflow(sphg.PCISPH, 600)
    other = configs.small_scene(sphg.PCISPH, n_side=5)
    alone, mixed = [sphg.Scene(ctx, p, x, b, emitters=em) for _ in range(2)]
    extra = sphg.Scene(ctx, other.params, other.fluid, other.boundary)
    empty = 0
    for _ in range(30):
        before = alone.n
        alone.step(1)
        ctx.batch_step([mixed, extra], 1)
        assert alone.n == mixed.n and scalars(alone) == scalars(mixed) and same(alone, mixed)
        if before == 0:
            empty += 1
            assert alone.scalars().iterations == p.min_iterations and alone.scalars().max_density_error == 0.0
    assert empty >= 3 and alone.n > 7 and np.isfinite(alone.get(sphg.FIELD_X)).all()
    for s in (alone, mixed, extra):
        s.close()


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("start", ["empty", "few"])
def test_list_build_of_an_inflow_in_a_large_launch(ctx, crowd, method, start):
    """Chunks cover a scene's capacity: those past its active particles, the
    first one of an empty scene among them, have no cell to start from.  Alone
    the lists are built with 4 lanes a particle, beside the crowd with one."""
    fluid = None if start == "empty" else block_of(40, 0.05, 0.1, 9, at=0.1)
    p, x, b, em = inflow(method, 1500, fluid)
    alone, mixed = [sphg.Scene(ctx, p, x, b, emitters=em) for _ in range(2)]
    first = alone.n
    for _ in range(25):
        alone.step(1)
        ctx.batch_step([mixed, crowd[method]], 1)
        assert alone.n == mixed.n and scalars(alone) == scalars(mixed)
        if alone.n:
            assert all(np.array_equal(a, m, equal_nan=True) for a, m in zip(build_fields(alone), build_fields(mixed)))
    assert alone.n >= first + 7 and alone.capacity > 5 * 256 and np.isfinite(alone.get(sphg.FIELD_X)).all()
    alone.close()
    mixed.close()


@pytest.mark.parametrize("method", METHODS)
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_nan_position_of_either_sign_stays_its_own_particles(ctx, crowd, method, sign):
    """The list build's FP32 test by the sign of d^2 - h^2 lets a NaN with its
    sign bit set through to the FP64 test, which rejects it: no other
    particle's sums hold a trace of it, with 4 lanes a particle or one."""
    r = 0.01
    p = configs.small_scene(method, n_side=2, spacing=2 * r).params
    b = sphg.sample_box((0.0, 0.0, 0.0), (0.4, 0.4, 0.4), 4 * r)
    x = block_of(300, 2 * r, 0.1, 4, at=0.02)
    v = np.random.default_rng(6).uniform(-0.3, 0.3, x.shape).astype(np.float32)
    alone, mixed = [sphg.Scene(ctx, p, x, b) for _ in range(2)]
    x = x.copy()
    # the grid clamps it to the cells of the domain's corner, where the block is
    x[77] = np.copysign(np.float32(np.nan), np.float32(sign))
    for s in (alone, mixed):
        s.set_state(x, v)
    for _ in range(3):
        alone.step(1)
        ctx.batch_step([mixed, crowd[method]], 1)
        assert all(np.array_equal(a, m, equal_nan=True) for a, m in zip(build_fields(alone), build_fields(mixed)))
        assert all(np.isfinite(np.delete(f, 77, 0)).all() for f in fields(alone))
    alone.close()
    mixed.close()


@pytest.mark.parametrize("speed", [np.inf, -np.nan])
def test_velocity_of_a_rejected_candidate(ctx, speed):
    """A candidate just past h passes the FP32 test and not the FP64 one: its
    velocity, which may be anything, is in no divergence."""
    r, side = 0.01, 10
    p = configs.small_scene(sphg.DFSPH, n_side=2, spacing=2 * r).params
    b = sphg.sample_box((0.0, 0.0, 0.0), (0.4, 0.4, 0.4), 4 * r)
    x = block_of(side ** 3, 0.8, 0.0, 4, at=0.0) * 2 * r + np.float32(0.06)
    face = ((side - 1) * side + side // 2) * side + side // 2
    past = x[face] + np.array([p.support_radius * (1 + 2e-5), 0, 0])
    x = np.concatenate([x, past[None]]).astype(np.float32)
    v = np.random.default_rng(6).uniform(-0.3, 0.3, x.shape).astype(np.float32)
    v[face] = (-1.0, 0.0, 0.0)   # into its neighbors
    s = sphg.Scene(ctx, p, x, b)
    out = []
    for u in (0.0, speed):
        v[-1] = u
        s.set_state(x, v)
        out.append([s.get(f)[:-1] for f in (sphg.FIELD_ALPHA, sphg.FIELD_DIVERR)])
    assert out[0][1][face] > 0.0 and all(np.array_equal(a, c) for a, c in zip(*out))
    s.close()


STALLS = {
    # the loop that needs more iterations than were launched ahead; the other one stays at its minimum
    "density": (sphg.DFSPH, dict(eta_v=1e9)),
    "divergence": (sphg.DFSPH, dict(eta=1e3)),
    "pressure": (sphg.PCISPH, {}),
}


@pytest.mark.parametrize("loop", sorted(STALLS))
@pytest.mark.parametrize("where", ["small", "replayed", "large"])
def test_lone_scene_that_needs_more_iterations_than_predicted(ctx, loop, where):
    """At rest a loop takes a few iterations; with velocities that compress the
    fluid it takes more, so that the steps launched ahead stop behind it and
    the host adds iterations (the only waits that host_syncs counts once there
    is a prediction): the same steps as in a batch."""
    method, more = STALLS[loop]
    if where == "large":
        size = (129, 64, 64)
        spec = configs.small_scene(method, n_side=size, spacing=0.02, box=tuple(0.02 * (s + 4) for s in size), **more)
    else:
        spec = configs.small_scene(method, n_side=(12, 9, 8), box=(0.9, 0.65, 0.6), **more)
    other = configs.small_scene(method, n_side=5)
    center = spec.fluid.mean(0)
    speed = 300.0 * spec.params.particle_radius   # the same strain in both sizes
    inward = ((center - spec.fluid) / np.abs(center - spec.fluid).max() * speed).astype(np.float32)
    alone, mixed = [sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary) for _ in range(2)]
    extra = sphg.Scene(ctx, other.params, other.fluid, other.boundary)
    ctx.set_graphs(where == "replayed")
    try:
        for steps in (1, 4):
            alone.step(steps)
        before = alone.scalars()
        ctx.batch_step([mixed, extra], 5)
        for s in (alone, mixed):
            s.set_state(spec.fluid, inward)
        stats = alone.step(4)
        ctx.batch_step([mixed, extra], 4)
    finally:
        ctx.set_graphs(False)
    after = alone.scalars()
    assert stats.host_syncs > 0
    if loop == "divergence":
        assert after.sum_iterations_v - before.sum_iterations_v > 4 * spec.params.min_iterations_v
        assert after.sum_iterations - before.sum_iterations == 4 * spec.params.min_iterations
    else:
        assert after.sum_iterations - before.sum_iterations > 4 * spec.params.min_iterations
        assert after.sum_iterations_v - before.sum_iterations_v == (4 if method == sphg.DFSPH else 0)
    assert scalars(alone) == scalars(mixed) and same(alone, mixed)
    for s in (alone, mixed, extra):
        s.close()


def test_shell_width_after_a_new_state(ctx):
    """The shell of a PCISPH step is as wide as the previous step's predicted
    displacements ask for, also where a new state (with its iteration count at
    zero) came between: no step of a fluid at speed falls back to the walk
    over 27 cells for it."""
    spec = configs.small_scene(sphg.PCISPH, n_side=(9, 7, 8), box=(2.0, 0.55, 0.8))
    v = np.zeros_like(spec.fluid)
    v[:, 0] = 0.08 * spec.params.support_radius / spec.params.time_step
    s = sphg.Scene(ctx, spec.params, spec.fluid, spec.boundary, v)
    s.step(3)
    before = s.scalars()
    assert before.pcisph_walk_steps == 1 and before.pcisph_shell_steps == 2
    s.set_state(spec.fluid, v)
    s.step(1)
    s.set_state(spec.fluid, v, last_iterations=3)
    s.step(2)
    after = s.scalars()
    assert after.pcisph_walk_steps == 1 and after.pcisph_shell_steps == 5
    s.close()
