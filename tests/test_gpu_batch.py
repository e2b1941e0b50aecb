"""GPU: many instances stepped together (sb_batch_*) against each instance stepped alone.

Bar: bit-identical results and wake states per instance and per step, in
EXACT and FAST mode, over uneven instances (strips, wings, wake rows, time
steps, free and convected wakes, symmetry), across the first step (wake
initialisation), the start of the free-wake self-induction and several
replays of the captured step graph.  One instance is also held to the
oracle directly.
"""
import numpy as np
import pytest

import stormbird_amd as sb
from stormbird_amd import setups as S

from test_gpu_parity import compare_results, same

pytestmark = pytest.mark.gpu


def mixed_setups(seed=7, n=10):
    rng = np.random.default_rng(seed)
    setups, cases = [], []
    for _ in range(n):
        js, case = S.polar_sweep_instance(rng, max_panels=40, min_panels=6)
        setups.append(js)
        cases.append(case)
    # a free-wake instance and a symmetric one (self-induction and mirror paths)
    js, case = S.polar_sweep_instance(rng, max_panels=30, min_panels=20)
    d = __import__("json").loads(js)
    d["simulation_settings"]["Dynamic"]["wake"]["ratio_of_wake_affected_by_induced_velocities"] = 1.0
    setups.append(__import__("json").dumps(d))
    cases.append(case)
    js, case = S.polar_sweep_instance(rng, max_panels=25, min_panels=10)
    d = __import__("json").loads(js)
    d["simulation_settings"]["Dynamic"]["wake"]["symmetry_condition"] = "Z"
    setups.append(__import__("json").dumps(d))
    cases.append(case)
    return setups, cases


def run_pair(mode, steps):
    setups, cases = mixed_setups()
    batch = sb.Batch(setups, mode=mode)
    alone = [sb.Simulation(js, mode=mode) for js in setups]
    fs_parts = [S.uniform_freestream(s.nr_freestream_points(), c["velocity"]) for s, c in zip(alone, cases)]
    fs_all = np.concatenate(fs_parts)
    assert fs_all.shape[0] == batch.nr_freestream_points
    dts = np.array([c["time_step"] for c in cases])
    for k in range(steps):
        print(f"batch step {k} mode {mode}", flush=True)
        rb = batch.do_step(times=k * dts, time_steps=dts, freestream_velocity=fs_all)
        for i, sim in enumerate(alone):
            ra = sim.do_step(time=k * dts[i], time_step=dts[i], freestream_velocity=fs_parts[i])
            compare_results(rb[i], ra, exact=True, where=f"step {k} instance {i}")
        if k in (0, 3, steps - 1):
            for i, sim in enumerate(alone):
                wb, wa = batch.instances[i].get_wake_state(), sim.get_wake_state()
                for key in ("points", "velocities", "strengths"):
                    assert same(wb[key], wa[key]), f"step {k} instance {i}: wake {key}"
    return batch


def test_batch_equals_alone_exact():
    batch = run_pair(sb.MODE_EXACT, 9)
    assert batch.last_step_ms() > 0.0


def test_batch_equals_alone_fast():
    run_pair(sb.MODE_FAST, 6)


@pytest.mark.parametrize("neglect", [False, True])
@pytest.mark.parametrize("symmetry", [None, "Z"])
def test_fixed_velocity_jobs_at_their_edges(neglect, symmetry):
    """Control points below, at and above a job's 16, wakes from 2 rows (fewer panels than a block of
    the fixed-velocity kernel) up: the batch gives the bits of the instances alone, in every variant."""
    import json

    setups = []
    for sails, strips, rows in [(1, 1, 2), (1, 15, 3), (1, 16, 9), (1, 17, 6), (3, 5, 12), (2, 17, 8), (4, 4, 2)]:
        js, case = S.four_sail_free_wake(nr_panels=rows, nr_strips=strips, ratio=0.0)
        d = json.loads(js)
        d["line_force_model"]["wing_builders"] = d["line_force_model"]["wing_builders"][:sails]
        wake = d["simulation_settings"]["Dynamic"]["wake"]
        if neglect:
            wake["neglect_self_induced_velocities"] = True
        if symmetry:
            wake["symmetry_condition"] = symmetry
        setups.append(json.dumps(d))
    batch, alone = sb.Batch(setups), [sb.Simulation(js) for js in setups]
    parts = [S.uniform_freestream(a.nr_freestream_points(), case["velocity"]) for a in alone]
    for k in range(13):
        batch.set_tuning(1 + k % 3, 64)
        rb = batch.do_step(times=0.2 * k, time_steps=0.2, freestream_velocity=np.concatenate(parts))
        for i, a in enumerate(alone):
            ra = a.do_step(time=0.2 * k, time_step=0.2, freestream_velocity=parts[i])
            compare_results(rb[i], ra, exact=True, where=f"step {k} instance {i}")


@pytest.mark.parametrize("mode", [sb.MODE_EXACT, sb.MODE_FAST])
def test_self_induction_kernels_on_both_sides_of_their_rules(mode):
    """16 wake points per workgroup or 256 (single instances: at most 384 workgroups of 256 on 256 CUs;
    batches: 768 in EXACT): the same wake step through every route gives the same bits.  A target map
    keeps a single instance on the 256-point kernel."""
    rows = 590  # 4 x 41 x 591 points: 379 workgroups of 256
    js, case = S.four_sail_free_wake(nr_panels=rows)
    alone = sb.Simulation(js, mode=mode)
    tiled = sb.Simulation(js, mode=mode)
    tiled.target_tiling = 8
    batches = [sb.Batch([js] * n, mode=mode) for n in (1, 2, 3)]  # 379, 758, 1,137 workgroups
    data = np.load(S.DEVELOPED_FOUR_SAIL)
    p = data["points"].reshape(2001, -1, 3)[:rows + 1].astype(np.float64).reshape(-1, 3)
    g = data["strengths"].reshape(2000, -1)[:rows].astype(np.float64)
    u = np.tile(np.asarray(case["velocity"]), (p.shape[0], 1))
    fs = S.uniform_freestream(alone.nr_freestream_points(), case["velocity"])

    def load(sim):
        sim.set_wake_state(p, u, g.ravel(), rows)
        sim.previous_circulation_strength = g[0]

    for sim in (alone, tiled):
        load(sim)
        sim.do_step(time=1.0, time_step=0.2, freestream_velocity=fs)
    want = alone.get_wake_state()
    got = [tiled.get_wake_state()]
    for b in batches:
        b.do_step(times=0.0, time_steps=0.2, freestream_velocity=np.concatenate([fs] * len(b.instances)))
        for sim in b.instances:
            load(sim)
        b.do_step(times=1.0, time_steps=0.2, freestream_velocity=np.concatenate([fs] * len(b.instances)))
        got += [sim.get_wake_state() for sim in b.instances]
    for i, w in enumerate(got):
        for key in ("points", "velocities", "strengths"):
            assert same(w[key], want[key]), f"route {i}: wake {key}"


def test_batch_instance_matches_oracle(oracle):
    rng = np.random.default_rng(11)
    setups, cases = [], []
    for _ in range(3):
        js, case = S.polar_sweep_instance(rng, max_panels=20, min_panels=8)
        setups.append(js)
        cases.append(case)
    batch = sb.Batch(setups)
    orc = oracle.Simulation(setups[1], variant="pm")
    parts = [S.uniform_freestream(s.nr_freestream_points(), c["velocity"]) for s, c in zip(batch.instances, cases)]
    dts = np.array([c["time_step"] for c in cases])
    for k in range(8):
        rb = batch.do_step(times=k * dts, time_steps=dts, freestream_velocity=np.concatenate(parts))
        ro = orc.do_step(time=k * dts[1], time_step=dts[1], freestream_velocity=parts[1])
        compare_results(rb[1], ro, exact=True, where=f"step {k}")


def test_batch_rejects_bad_input():
    js, _ = S.polar_sweep_instance(np.random.default_rng(1), max_panels=10, min_panels=5)
    with pytest.raises(ValueError):
        sb.Batch([js, "{not json"])
    batch = sb.Batch([js, js])
    with pytest.raises(RuntimeError):
        batch.do_step(times=None, time_steps=0.1, freestream_velocity=np.zeros((3, 3)))


def test_route_simulation_batch_equals_alone(oracle):
    """Rolling ships in gusty wind with free wakes: the batch's freestream is the reference's
    WindEnvironment at every point (the oracle's restatement, bit for bit: power-law profile,
    gusts along and across the wind, ship speed), and the batched steps equal each ship
    stepped alone with that freestream."""
    import oracle_csm

    from stormbird_amd.route import RouteSimulation, wind_environment

    route = RouteSimulation(n_ships=3, n_conditions=2, seed=5, nr_strips=8, nr_panels=12, nr_freqs=50)
    alone = [sb.Simulation(js, mode=sb.MODE_EXACT) for js in route.setups]
    m = oracle_csm.Libm("pm")
    env = oracle_csm.WindEnvironment(wind_environment(), m)
    conds = [oracle_csm.WindCondition(wc, m) for wc in route.wind_conditions]
    off = route.batch.freestream_offsets
    for k in range(7):
        print(f"route step {k}", flush=True)
        pts = []
        for i, sim in enumerate(alone):
            dt = float(route.dt[i])
            sim.set_translation_and_rotation_with_finite_difference_for_the_velocity(
                dt, [0.0, 0.0, 0.0], [route.roll(route.k * dt), 0.0, 0.0])
            pts.append(sim.get_freestream_velocity_points())
        t = route.k * route.dt
        rb = route.step()
        fs_all = route.batch.get_freestream()
        for i, sim in enumerate(alone):
            fs = fs_all[off[i]:off[i + 1]]
            linear = oracle_csm.scale(env.zero, float(route.ship_speed[i]))
            want = np.array([env.unsteady_apparent(conds[i], tuple(p), linear, float(t[i])) for p in pts[i]])
            assert same(fs, want), f"step {k} ship {i}: freestream"
            ra = sim.do_step(time=float(t[i]), time_step=float(route.dt[i]), freestream_velocity=fs)
            compare_results(rb[i], ra, exact=True, where=f"step {k} ship {i}")
    # a judged warm start (untrained network) changes only the initial guess
    net = sb.Mlp(seed=1)
    route.batch.set_warm_start(net, 3)
    res = route.step()
    assert route.batch.last_warm_taken() + route.batch.last_fallbacks() <= 3
    for r in res:
        assert np.all(np.isfinite(r.force_input.circulation_strength))
    with pytest.raises(ValueError):
        route.batch.set_wind(wind_environment(), route.wind_conditions[:2])


@pytest.mark.parametrize("solver", [None, {"start_with_linearized_solution": True,
                                           "max_iterations_per_time_step": 400}])
def test_quasi_steady_batch_matches_single_instances(oracle, solver):
    """A batch of quasi-steady instances (horseshoe wake; Linearized, or SimpleIterative from
    the Linearized start) equals every instance stepped alone, bit for bit, over several steps;
    two instances are held to the oracle too."""
    rng = np.random.default_rng(11)
    setups, cases = zip(*[S.quasi_steady_polar_instance(rng, solver=solver) for _ in range(12)])
    batch = sb.Batch(list(setups))
    alone = [sb.Simulation(js) for js in setups]
    orcs = {0: oracle.Simulation(setups[0], "pm"), 5: oracle.Simulation(setups[5], "pm")}
    assert batch.nr_freestream_points == sum(s.nr_ctrl_points for s in alone)
    dts = np.array([c["time_step"] for c in cases])
    for k in range(3):
        print(f"quasi batch step {k}", flush=True)
        parts = [S.uniform_freestream(s.nr_freestream_points(), np.array(c["velocity"]) * (1.0 + 0.05 * k))
                 for s, c in zip(alone, cases)]
        rb = batch.do_step(times=k * dts, time_steps=dts, freestream_velocity=np.concatenate(parts))
        for i, sim in enumerate(alone):
            ra = sim.do_step(time=k * dts[i], time_step=dts[i], freestream_velocity=parts[i])
            compare_results(rb[i], ra, exact=True, where=f"step {k} instance {i}")
            if i in orcs:
                ro = orcs[i].do_step(time=k * dts[i], time_step=dts[i], freestream_velocity=parts[i])
                compare_results(rb[i], ro, exact=True, where=f"oracle step {k} instance {i}")


def test_batch_rejects_mixed_and_warm_quasi():
    rng = np.random.default_rng(3)
    q, _ = S.quasi_steady_polar_instance(rng)
    d, _ = S.polar_sweep_instance(rng, max_panels=10, min_panels=5)
    with pytest.raises(ValueError, match="either quasi-steady or dynamic"):
        sb.Batch([q, d])
    b = sb.Batch([q, q])
    m = sb.Mlp(seed=1)
    with pytest.raises(RuntimeError, match="dynamic batches"):
        b.set_warm_start(m, 1)


@pytest.mark.parametrize("symmetric", [False, True])
def test_autotuner_and_every_variant_keep_results(tmp_path, symmetric):
    """The autotuner times the kernel variants on the batch's own state without changing
    it; every variant (fours of panels per wave of the fixed-velocity kernel, LDS tile length of
    the self-induction kernel, which this small wake does not reach:
    test_every_self_induction_kernel_gives_the_same_bits) gives the same bits; the choice is
    cached per device and shape class in a JSON file and reused by a batch of the same shape."""
    import json

    setups, cases = mixed_setups()
    if not symmetric:
        setups, cases = setups[:-1], cases[:-1]
    ref, tuned = sb.Batch(setups), sb.Batch(setups)
    fs_all = np.concatenate([S.uniform_freestream(s.nr_freestream_points(), c["velocity"])
                             for s, c in zip(ref.instances, cases)])
    dts = np.array([c["time_step"] for c in cases])

    def step_both(k):
        print(f"tuning step {k}", flush=True)
        ra = ref.do_step(times=k * dts, time_steps=dts, freestream_velocity=fs_all)
        rb = tuned.do_step(times=k * dts, time_steps=dts, freestream_velocity=fs_all)
        for i in range(len(setups)):
            compare_results(rb[i], ra[i], exact=True, where=f"step {k} instance {i}")

    for k in range(5):  # the free wake's self-induction runs from the fourth step on
        step_both(k)
    cache = str(tmp_path / "tuning.json")
    cached, choice, t = tuned.autotune(cache)
    assert not cached and choice[0] in (1, 2, 3) and choice[1] in (64, 128, 256)
    assert np.all(t > 0.0), t  # both kernels had work
    for i in range(len(setups)):  # the state is unchanged
        wa, wb = ref.instances[i].get_wake_state(), tuned.instances[i].get_wake_state()
        for key in ("points", "velocities", "strengths"):
            assert same(wa[key], wb[key]), f"instance {i}: wake {key} after tuning"
    k = 5
    for variant in (choice, (1, 64), (2, 128), (3, 256)):
        tuned.set_tuning(*variant)
        assert tuned.get_tuning() == variant
        step_both(k)
        k += 1
    entries = json.load(open(cache))["entries"]
    assert len(entries) == 1 and entries[0]["fixed_per"] == choice[0] and entries[0]["targets_tile"] == choice[1]
    other = sb.Batch(setups)
    for j in range(5):
        other.do_step(times=j * dts, time_steps=dts, freestream_velocity=fs_all, want_result=False)
    hit, choice2, t2 = other.autotune(cache)
    assert hit and choice2 == choice and np.allclose(t2, t, atol=1e-4)
    with pytest.raises(RuntimeError):
        other.set_tuning(4, 256)
    fresh = sb.Batch(setups)
    with pytest.raises(RuntimeError, match="take a step"):
        fresh.autotune(None)


def test_residual_warm_start_with_a_zero_network_is_the_default_guess():
    """In residual mode the network predicts the change from the previous circulation: a
    network whose every parameter is zero predicts no change, and the steps then equal the
    steps without a warm start bit for bit."""
    from stormbird_amd.route import RouteSimulation

    a = RouteSimulation(n_ships=3, n_conditions=2, seed=6, nr_strips=8, nr_panels=12, nr_freqs=50)
    b = RouteSimulation(n_ships=3, n_conditions=2, seed=6, nr_strips=8, nr_panels=12, nr_freqs=50)
    net = sb.Mlp(seed=2)
    net.set_params(np.zeros(net.nr_params, dtype=np.float32))
    b.batch.set_warm_start(net, 2, residual=True)
    for k in range(6):
        print(f"residual warm start step {k}", flush=True)
        ra, rb = a.step(), b.step()
        for i in range(3):
            compare_results(rb[i], ra[i], exact=True, where=f"step {k} ship {i}")
    assert b.batch.last_fallbacks() == 0


def wide_route(batch):
    """1 when the batch's last fixed velocities ran in jobs of 64 control points, 0 in jobs of 16."""
    import ctypes

    L = sb.lib()
    L.sb_debug_batch_fixed_wide.argtypes = [ctypes.c_void_p]
    return L.sb_debug_batch_fixed_wide(batch._h)


@pytest.mark.parametrize("neglect", [False, True])
@pytest.mark.parametrize("mode,symmetry", [(sb.MODE_FAST, None), (sb.MODE_FAST, "Z"), (sb.MODE_EXACT, "Z"),
                                           (sb.MODE_EXACT, None)])
def test_fixed_velocity_jobs_of_64_control_points(mode, symmetry, neglect):
    """Sixty copies of twelve instances fill the GPU in jobs of 64 control points, which FAST arithmetic and
    symmetry planes then take.  Control points below, at and above a job's
    64, wakes from 2 rows (fewer panels than a block) up: the bits of the instances alone and of one
    copy of each (jobs of 16), and the tuner times the one kernel once and leaves its parameter."""
    import json

    setups = []
    for sails, strips, rows in [(1, 1, 2), (1, 15, 3), (1, 16, 9), (1, 17, 6), (1, 63, 8), (1, 64, 8), (1, 65, 3),
                                (3, 5, 12), (2, 17, 8), (4, 4, 2), (1, 64, 9), (2, 32, 9)]:
        js, case = S.four_sail_free_wake(nr_panels=rows, nr_strips=strips, ratio=0.0)
        d = json.loads(js)
        d["line_force_model"]["wing_builders"] = d["line_force_model"]["wing_builders"][:sails]
        wake = d["simulation_settings"]["Dynamic"]["wake"]
        if neglect:
            wake["neglect_self_induced_velocities"] = True
        if symmetry:
            wake["symmetry_condition"] = symmetry
        setups.append(json.dumps(d))
    n = len(setups)
    many, once = sb.Batch(setups * 60, mode=mode), sb.Batch(setups, mode=mode)
    alone = [sb.Simulation(js, mode=mode) for js in setups]
    parts = [S.uniform_freestream(a.nr_freestream_points(), case["velocity"]) for a in alone]
    for k in range(13):
        rm = many.do_step(times=0.2 * k, time_steps=0.2, freestream_velocity=np.concatenate(parts * 60))
        ro = once.do_step(times=0.2 * k, time_steps=0.2, freestream_velocity=np.concatenate(parts))
        assert wide_route(once) == 0
        if k > 3:
            assert wide_route(many) == (1 if mode == sb.MODE_FAST or symmetry else 0)
        for i, a in enumerate(alone):
            ra = a.do_step(time=0.2 * k, time_step=0.2, freestream_velocity=parts[i])
            compare_results(ro[i], ra, exact=True, where=f"step {k} instance {i}")
            for j in (0, 23, 59):
                compare_results(rm[j * n + i], ra, exact=True, where=f"step {k} instance {i}, copy {j}")
    many.set_tuning(2, 256)
    _, choice, t = many.autotune(None)
    if wide_route(many):
        assert choice[0] == 2 and t[0] == t[1] == t[2] > 0.0
    else:
        assert len(set(t[:3])) > 1 and np.all(t[:3] > 0.0)


def few_route(batch):
    """1 when the batch's last self-induction took the kernel for few wake points, else 0."""
    import ctypes

    L = sb.lib()
    L.sb_debug_batch_targets_few.argtypes = [ctypes.c_void_p]
    return L.sb_debug_batch_targets_few(batch._h)


def free_wake_setup(rows, strips, symmetry=None):
    import json

    js, case = S.four_sail_free_wake(nr_panels=rows, nr_strips=strips)
    d = json.loads(js)
    if symmetry:
        d["simulation_settings"]["Dynamic"]["wake"]["symmetry_condition"] = symmetry
    return json.dumps(d), np.asarray(case["velocity"])


def shed_every_row(sim, rows, strips, seed):
    """A stepped simulation's straight wake with noise, every row shed, strengths decaying downstream."""
    rng = np.random.default_rng(seed)
    w = sim.get_wake_state()
    g = -40.0 * np.exp(-np.arange(rows) / rows)[:, None] * rng.uniform(0.5, 1.0, (rows, 4 * strips))
    sim.set_wake_state(w["points"] + rng.normal(0.0, 0.05, w["points"].shape), w["velocities"], g.ravel(), rows)
    sim.previous_circulation_strength = g[0]


def free_wake_batch(copies, rows, strips, mode, symmetry=None):
    """`copies` of a four-sail free wake with every row shed, after one step with self-induction;
    (batch, step)."""
    js, u = free_wake_setup(rows, strips, symmetry)
    batch = sb.Batch([js] * copies, mode=mode)
    fs = np.tile(u, (batch.nr_freestream_points, 1))

    def step():
        return batch.do_step(times=0.0, time_steps=0.2, freestream_velocity=fs)

    step()
    for i, sim in enumerate(batch.instances):
        shed_every_row(sim, rows, strips, i)
    step()
    return batch, step


@pytest.mark.parametrize("symmetry", [None, "Z"])
@pytest.mark.parametrize("mode", [sb.MODE_EXACT, sb.MODE_FAST])
def test_every_self_induction_kernel_gives_the_same_bits(mode, symmetry):
    """A wake of 141 workgroups of 256 points on the kernel for few points (alone and in a batch), on the
    256-point kernel of single instances (a target map keeps it there) and on the batched 256-point
    kernel with each tile (seven copies), with and without a symmetry plane: equal wakes."""
    rows, strips = 271, 32
    js, u = free_wake_setup(rows, strips, symmetry)
    alone, tiled = sb.Simulation(js, mode=mode), sb.Simulation(js, mode=mode)
    tiled.target_tiling = 8
    fs = np.tile(u, (alone.nr_freestream_points(), 1))
    few, step_few = free_wake_batch(1, rows, strips, mode, symmetry)
    many, step_many = free_wake_batch(7, rows, strips, mode, symmetry)
    assert few_route(few) == 1 and few_route(many) == 0
    for sim in (alone, tiled):
        sim.do_step(time=0.0, time_step=0.2, freestream_velocity=fs)
        shed_every_row(sim, rows, strips, 0)
        sim.do_step(time=0.0, time_step=0.2, freestream_velocity=fs)
    for tile in (256, 64, 128):
        want = alone.get_wake_state()
        for where, sim in (("tiled", tiled), ("few", few.instances[0]), ("many", many.instances[0])):
            got = sim.get_wake_state()
            for key in ("points", "velocities", "strengths"):
                assert same(got[key], want[key]), f"{where}, tile before {tile}: wake {key}"
        many.set_tuning(3, tile)
        step_many()
        step_few()
        for sim in (alone, tiled):
            sim.do_step(time=0.0, time_step=0.2, freestream_velocity=fs)
    want, got = alone.get_wake_state(), many.instances[0].get_wake_state()
    for key in ("points", "velocities", "strengths"):
        assert same(got[key], want[key]), f"tile 128: wake {key}"


@pytest.mark.parametrize("mode,symmetry,copies,few", [
    (sb.MODE_EXACT, None, 5, 1), (sb.MODE_EXACT, None, 6, 0),   # 705 and 846 workgroups of 256; 768 of 256 CUs
    (sb.MODE_EXACT, "Z", 2, 1), (sb.MODE_EXACT, "Z", 3, 0),     # 282 and 423; 304
    (sb.MODE_FAST, None, 2, 1), (sb.MODE_FAST, None, 3, 0),     # 282 and 423; 384
    (sb.MODE_FAST, "Z", 1, 1), (sb.MODE_FAST, "Z", 2, 0),       # 141 and 282; 160
])
def test_self_induction_kernel_of_a_batch(mode, symmetry, copies, few):
    """The rule between the two kernels on both sides of its measured lines: by the workgroups, and by the
    panels in the first steps, where the wake has many points and few shed rows."""
    import json

    batch, _ = free_wake_batch(copies, 271, 32, mode, symmetry)
    assert few_route(batch) == few
    if mode != sb.MODE_EXACT:
        return
    d = json.loads(free_wake_setup(2000, 8, symmetry)[0])
    d["line_force_model"]["wing_builders"] = d["line_force_model"]["wing_builders"][:1]
    start = sb.Batch([json.dumps(d)] * (4 if symmetry else 8), mode=mode)  # 71 workgroups of 256 points each
    fs = np.tile([10.0, 3.0, 0.0], (start.nr_freestream_points, 1))
    for k in range(5):  # 40 panels
        start.do_step(times=0.2 * k, time_steps=0.2, freestream_velocity=fs)
    assert few_route(start) == 0


def test_autotuner_keeps_the_self_induction_kernels_apart(tmp_path):
    """The kernel for few wake points has no tile: one time for all three, and the tile stays.  Batches of
    one size class (2 and 3 instances, equal powers of two of both pair counts) on the two sides of the
    rule don't share a cache entry, and a limit on the timed jobs does not change the kernel."""
    import json

    cache = str(tmp_path / "tuning.json")
    few, _ = free_wake_batch(2, 271, 32, sb.MODE_FAST)   # 282 workgroups of 256 on 256 CUs
    many, step = free_wake_batch(3, 271, 32, sb.MODE_FAST)  # 423
    assert few_route(few) == 1 and few_route(many) == 0
    few.set_tuning(2, 128)
    cached, choice, t = few.autotune(cache)
    assert not cached and choice[1] == 128 and np.all(t > 0.0)
    assert t[3] == t[4] == t[5]
    cached, choice, t = many.autotune(cache, max_jobs=200)
    assert not cached and np.all(t > 0.0) and len(set(t[3:])) > 1
    assert few_route(many) == 0
    step()
    assert few_route(many) == 0
    entries = json.load(open(cache))["entries"]
    assert len(entries) == 2 and [e["targets_tile"] for e in entries] == [128, choice[1]]
    assert len({e["key"].replace("|few1", "|few0") for e in entries}) == 1  # one size class otherwise
