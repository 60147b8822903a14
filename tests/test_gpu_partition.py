"""The sweep loops over a spatial partition of the bodies (pd_parts.hpp) against the CPU oracle:
every substep's state, counters and ledger, at partitions from one workgroup to one row per few."""
import numpy as np
import pytest

from test_gpu_parity import run_pair

# rows per workgroup: one workgroup for all rows, a few, and many of a chunk (32 rows) or less
ROWS = [100000, 200, 33, 9]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bed", "bed_periodic", "gas", "bed_walls"])
@pytest.mark.parametrize("rows", ROWS)
def test_partition_sizes(hip_lib, kind, rows):
    h, _ = run_pair(kind, 500, 12, tuning={"partition_rows": rows})
    paths = h.debug_paths()
    print(paths, flush=True)
    assert paths["vel_parts"] + paths["vel_one"] == 12
    assert (paths["refused"], paths["alone"], paths["global"]) == (0, 0, 0)
    # (position loops: from 20 x rows on, after a loop of more than two sweeps; the gas thins out)
    gas = kind == "gas"
    vel, pos = {100000: (0, 0), 200: (0 if gas else 3, 0), 33: (1 if gas else 11, 0 if gas else 10),
                9: (3 if gas else 12, 3 if gas else 10)}[rows]
    assert paths["vel_parts"] >= vel and paths["pos_parts"] >= pos
    assert vel or paths["vel_parts"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,steps", [("column_small_box", 64, 8), ("boxes", 48, 8),
                                          ("cylinders", 48, 8), ("bed_small_box", 60, 8),
                                          ("big_among_small", 4000, 3)])
@pytest.mark.parametrize("rows", [200, 9])
def test_partition_shapes_and_twins(hip_lib, kind, n, steps, rows):
    # several points per manifold, every sphere with images of its neighbours, and (the big sphere)
    # colourings whose last class keeps the loops off the partition
    h, _ = run_pair(kind, n, steps, tuning={"partition_rows": rows, "partition_bodies": 8})
    paths = h.debug_paths()
    print(paths, flush=True)
    assert (paths["refused"], paths["alone"]) == (0, 0)
    if kind == "big_among_small":
        assert (paths["vel_parts"], paths["vel_block"], paths["pos_parts"]) == (2, 1, 0)
    elif rows == 9:
        assert paths["vel_parts"] >= (1 if kind in ("boxes", "cylinders") else steps)
        # (the contacts of the cylinders are not all coloured)
        assert paths["pos_parts"] >= {"cylinders": 0, "boxes": 1}.get(kind, steps - 1)
    else:
        assert paths["vel_one"] == steps


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bed", "bed_periodic", "gas"])
@pytest.mark.parametrize("tuning", [{"velocity_loop_lds_bodies": 3}, {"velocity_loop_lds_keys": 16},
                                    {"partition_workgroups": 2}],
                         ids=["lds-and-global", "refused-check-in", "two-workgroups"])
def test_partition_storage_and_check_in(hip_lib, kind, tuning):
    # parts with more bodies than LDS slots; workgroups that agree to leave at the check-in, so that
    # one of them runs the loop; more rows per workgroup than asked for
    h, _ = run_pair(kind, 300, 10, tuning={"partition_rows": 20, **tuning})
    paths = h.debug_paths()
    print(paths, flush=True)
    assert paths["vel_parts"] >= (1 if kind == "gas" else 6)
    assert paths["global"] == (10 if "velocity_loop_lds_bodies" in tuning else 0)
    if "velocity_loop_lds_keys" in tuning:
        assert paths["alone"] >= (3 if kind == "gas" else 10)
    else:
        assert paths["alone"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("over", [{"material": (0.3, 0.0, 0.5)}, {"material": (0.6, 0.4, 0.0)},
                                  {"stab": "off"}, {"iters": (1, 1)}, {"iters": (0, 3)}],
                         ids=["no-tangential", "frictionless", "no-stabilization", "one-sweep",
                              "no-position-loop"])
def test_partition_options(hip_lib, over):
    h, _ = run_pair("bed_periodic", 400, 10, tuning={"partition_rows": 60}, **over)
    paths = h.debug_paths()
    # (a position loop of one sweep does not repay a partition)
    assert paths["vel_parts"] == 10 and paths["pos_parts"] == (0 if "iters" in over else 9)


def bodies(sim):
    return [sim.get_positions(), sim.get_velocities(), sim.get_angular_velocities(),
            *sim.debug_ledger()]


def assert_same_bodies(a, b, tag):
    for k, (x, y) in enumerate(zip(bodies(a), bodies(b))):
        assert np.array_equal(x, y), (tag, k)


@pytest.mark.gpu
@pytest.mark.parametrize("block_rows", [16384, 100], ids=["alone", "launches"])
def test_check_in_that_times_out(hip_lib, block_rows):
    # one workgroup keeps away: the others agree to leave, and the loop runs in one workgroup, or,
    # above block_solver_rows rows, in launches per colour; the partition is then left alone for 4
    # substeps
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    scene = make_scene("bed_periodic", 1500, 2)
    scene["vel"][:, 2] -= 0.5
    h, plain = (apply_scene(Simulation(1500), scene) for _ in range(2))
    plain.set_tuning("block_solver_rows", 0)
    h.set_tuning("partition_rows", 20)
    h.set_tuning("block_solver_rows", block_rows)
    h.set_tuning("partition_absent", 1)
    for k in range(3):
        h.step(scene["dt"])
        plain.step(scene["dt"])
        assert h.get_stats() == plain.get_stats()
        assert_same_bodies(h, plain, k)
    paths = h.debug_paths()
    assert (paths["alone"], paths["refused"]) == ((1, 0) if block_rows == 16384 else (0, 1))
    assert paths["vel_parts"] == (1 if block_rows == 16384 else 0)
    h.set_tuning("partition_absent", 0)
    h.step_n(scene["dt"], 2)
    plain.step_n(scene["dt"], 2)
    assert h.debug_paths()["vel_parts"] == paths["vel_parts"]
    h.step_n(scene["dt"], 10)
    plain.step_n(scene["dt"], 10)
    after = h.debug_paths()
    print(paths, after, flush=True)
    assert after["vel_parts"] == paths["vel_parts"] + 10 and after["refused"] == paths["refused"]
    assert_same_bodies(h, plain, "after")
    h.close()
    plain.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,form", [("bed_walls", 500, "pos_block"),
                                         ("big_among_small", 600, "pos_block"),
                                         ("bed_walls", 4000, "pos_parts"),
                                         ("big_among_small", 2000, "pos_block"),
                                         ("sphere_in_shell", 201, "pos_block"),
                                         ("boxes", 512, "chain")])
def test_form_of_the_position_loop(hip_lib, kind, n, form):
    # loops of fewer than 5,120 rows run in one workgroup from global memory, the form that is the
    # shorter one there; so do loops of up to 16,384 whose last class is that of one large body
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    scene = make_scene(kind, n, 5)
    h = apply_scene(Simulation(len(scene["pos"])), scene)
    h.step_n(scene["dt"], 12)
    before = h.debug_paths()
    h.step_n(scene["dt"], 8)
    after = h.debug_paths()
    print(kind, n, h.get_stats()["num_contacts"], before, after, flush=True)
    assert kind == "sphere_in_shell" or h.get_stats()["sweeps_pos"] > 2
    assert after[form] == before[form] + 8
    assert form == "chain" or after["chain"] == 0
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("block_rows", [16384, 1000])
@pytest.mark.parametrize("far", ["one-body", "half"])
def test_bodies_far_apart(hip_lib, far, block_rows):
    # a sphere a thousand bed widths from its bed: the partition is that of the bed.  Two beds as far
    # from each other: a few parts hold all rows, which the loops notice before they start
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    n = 9000
    scene = make_scene("bed", n, 5)
    width = scene["domain"][0]
    if far == "one-body":
        scene["pos"][-1] = [1000.0 * width, 0.5 * width, 0.02]
    else:
        scene["pos"][n // 2:] = scene["pos"][:n - n // 2] + np.array([1000.0 * width, 0.0, 0.0])
    h, plain = (apply_scene(Simulation(n), scene) for _ in range(2))
    plain.set_tuning("block_solver_rows", 0)
    h.set_tuning("block_solver_rows", block_rows)
    for k in range(3):
        h.step(scene["dt"])
        plain.step(scene["dt"])
        assert h.get_stats() == plain.get_stats()
        assert_same_bodies(h, plain, k)
    paths = h.debug_paths()
    print(far, h.get_stats(), paths, flush=True)
    if far == "one-body":
        assert (paths["vel_parts"], paths["alone"], paths["refused"]) == (3, 0, 0)
    else:
        # (the loops of one substep, then the pause)
        assert 1 <= paths["alone"] + paths["refused"] <= 2
        assert block_rows == 16384 or paths["alone"] == 0
    h.close()
    plain.close()


@pytest.mark.gpu
def test_parts_of_bodies_with_one_row_each(hip_lib):
    # a dense block (about 18 contacts a sphere) and as many spheres in pairs: a part of pairs holds
    # several times the average number of bodies, and still has LDS slots for all of them
    from peclet.dem import Simulation

    r, rng = 1e-3, np.random.default_rng(4)
    g = np.stack(np.meshgrid(*[np.arange(12)] * 3, indexing="ij"), -1).reshape(-1, 3)
    dense = (g + 1.0) * 1.4 * r + rng.uniform(-0.01, 0.01, g.shape) * r
    m = np.stack(np.meshgrid(*[np.arange(10)] * 3, indexing="ij"), -1).reshape(-1, 3)[:864]
    pairs = np.array([0.0, 0.0, 0.03]) + (m + 1.0) * 6.0 * r
    pairs = np.concatenate([pairs, pairs + np.array([1.9 * r, 0.0, 0.0])])
    pos = np.concatenate([dense, pairs])
    n = len(pos)

    def system(**tuning):
        h = Simulation(n)
        h.set_sphere_shape(r)
        h.set_domain(0.08, 0.08, 0.12, False, False, False)
        h.set_positions(pos)
        h.set_velocities(np.random.default_rng(5).normal(0.0, 0.05, (n, 3)))
        h.set_gravity(0.0, 0.0, -9.81)
        h.set_material_params(0.3, 0.2, 0.5)
        h.set_solver_iterations(6, 6)
        for key, value in tuning.items():
            h.set_tuning(key, value)
        return h

    h, plain = system(), system(block_solver_rows=0)
    for k in range(4):
        h.step(1e-5)
        plain.step(1e-5)
        assert h.get_stats() == plain.get_stats()
        assert_same_bodies(h, plain, k)
    paths = h.debug_paths()
    print(h.get_stats(), paths, flush=True)
    assert paths["vel_parts"] == 4 and paths["pos_parts"] == 3
    assert (paths["alone"], paths["refused"], paths["global"]) == (0, 0, 0)
    h.close()
    plain.close()


@pytest.mark.gpu
def test_very_large_loops_are_launches_per_colour(hip_lib):
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    n = 1600000
    scene = make_scene("bed_periodic", n, 1)
    h = apply_scene(Simulation(n), scene)
    h.step_n(scene["dt"], 3)
    paths, stats = h.debug_paths(), h.get_stats()
    print(stats, paths, flush=True)
    assert stats["active_manifolds"] > 1000000 and stats["num_contacts"] > 1 << 22
    assert stats["sweeps_pos"] > 2
    assert (paths["vel_colours"], paths["pos_colours"]) == (3, 3)
    h.close()


@pytest.mark.gpu
def test_two_large_systems_at_once(hip_lib):
    # each takes more than half of the compute units: loops that cannot have all their workgroups
    # running become launches per colour, and either system's states are those of a run by itself
    import threading

    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    n, steps = 90000, 12
    scenes = [make_scene("bed_periodic", n, seed) for seed in (1, 2)]
    alone = []
    for sc in scenes:
        h = apply_scene(Simulation(n), sc)
        h.step_n(sc["dt"], steps)
        alone.append(bodies(h))
        h.close()
    pair = [apply_scene(Simulation(n), sc) for sc in scenes]
    threads = [threading.Thread(target=h.step_n, args=(sc["dt"], steps))
               for h, sc in zip(pair, scenes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for h, want in zip(pair, alone):
        paths = h.debug_paths()
        print(paths, flush=True)
        assert paths["alone"] == 0 and paths["vel_parts"] + paths["vel_colours"] == steps
        for x, y in zip(bodies(h), want):
            assert np.array_equal(x, y)
        h.close()


def set_state(sim, scene):
    sim.set_positions(scene["pos"])
    sim.set_scales(scene["scale"])
    sim.set_inv_mass(scene["inv_mass"])
    sim.set_inv_inertia(scene["inv_inertia"])
    sim.set_velocities(scene["vel"])
    sim.set_angular_velocities(scene["angvel"])


@pytest.mark.gpu
@pytest.mark.parametrize("loop", ["velocity", "position"])
def test_a_wait_that_runs_out_fails_the_handle_until_it_is_set_again(hip_lib, loop):
    # one workgroup leaves after the check-in, the others' waits run out: the step raises, the
    # handle refuses to go on from the half-updated state, and a new state steps like a new handle
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    scene = make_scene("bed_periodic", 400, 2)
    scene["vel"][:, 2] -= 0.5
    h = apply_scene(Simulation(400), scene)
    h.set_tuning("partition_rows", 20)
    h.set_tuning("velocity_loop_lds", 1 if loop == "velocity" else 0)
    for _ in range(4):
        h.step(scene["dt"])
    assert h.get_stats()["sweeps_pos"] > 2
    h.set_tuning("partition_wait_polls", 256)
    h.set_tuning("partition_absent", 2)
    with pytest.raises(RuntimeError, match="waited too long"):
        h.step(scene["dt"])
    h.set_tuning("partition_absent", 0)
    for step in (h.step, lambda dt: h.step_n(dt, 2), lambda dt: h.step_hertz(dt, 1)):
        with pytest.raises(RuntimeError, match="state was lost"):
            step(scene["dt"])
    set_state(h, scene)
    other = apply_scene(Simulation(400), scene)
    for _ in range(4):
        h.step(scene["dt"])
        other.step(scene["dt"])
    for name in ("get_positions", "get_velocities", "get_angular_velocities"):
        assert np.array_equal(getattr(h, name)(), getattr(other, name)()), name
    h.close()
    other.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,tunings", [
    # enough rows for more than a hundred workgroups of several chunks per colour
    ("bed_periodic", 20000, [{}, {"partition_workgroups": 7}]),
    # the most workgroups, of several times partition_rows rows each
    ("bed_periodic", 140000, [{}]),
    # a sphere wider than its box: rows of a body and its own image
    ("big_among_small", 300, [{}, {"partition_rows": 10}])])
def test_partition_equals_the_launches_per_colour(hip_lib, kind, n, tunings):
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    scene = make_scene(kind, n, 5)
    runs = []
    for tuning in [{"block_solver_rows": 0}] + tunings:
        print(tuning, flush=True)
        h = apply_scene(Simulation(n), scene)
        for key, value in tuning.items():
            h.set_tuning(key, value)
        h.step_n(scene["dt"], 6)
        runs.append((h.get_positions(), h.get_velocities(), h.get_angular_velocities(),
                     *h.debug_ledger(), h.get_stats()))
        paths = h.debug_paths()
        print(paths, flush=True)
        if "block_solver_rows" in tuning:
            assert paths["vel_parts"] + paths["vel_one"] + paths["pos_parts"] == 0
        else:
            assert paths["vel_parts" if n > 1000 else "vel_one"] == 6
            assert paths["pos_parts"] == (5 if n > 1000 or "partition_rows" in tuning else 0)
            assert (paths["refused"], paths["alone"]) == (0, 0)
        h.close()
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert np.array_equal(a, b) if isinstance(a, np.ndarray) else a == b


@pytest.mark.gpu
@pytest.mark.parametrize("tuning", [{}, {"partition_bodies": 20},
                                    {"partition_bodies": 20, "partition_absent": 1},
                                    {"partition_rows": 0}],
                         ids=["chain", "more-parts", "refused", "launches"])
def test_last_contact_class_as_a_chain(hip_lib, tuning):
    # packed hollow cylinders with a dense shell: hundreds of rows in the contact class whose rows
    # share bodies, walked by one wavefront beside the other classes' partition, or in launches
    from oracle_binding import oracle_sim
    from peclet.dem import Simulation
    from peclet.dem.workloads import cylinder_pack, setup_cylinder_bed

    n = 300
    bed = cylinder_pack(n, 0.0274, 3)
    h = setup_cylinder_bed(Simulation(n), bed, 5e-6, 0.4, 0.2)
    for key, value in tuning.items():
        h.set_tuning(key, value)
    r = setup_cylinder_bed(oracle_sim(n), bed, 5e-6, 0.4, 0.2)
    for k in range(2):
        print(n, tuning, k, flush=True)
        h.step(5e-6)
        r.step(5e-6)
        for name in ("get_positions", "get_velocities", "get_angular_velocities"):
            assert np.array_equal(getattr(h, name)(), getattr(r, name)()), (k, name)
        assert h.get_stats()["sweeps_pos"] == r.get_stats()["sweeps_pos"]
        colours = h.debug_contact_colors()
        assert np.array_equal(colours, r.debug_contact_colors())
    assert (colours == 62).sum() > 64
    paths = h.debug_paths()
    if "partition_rows" in tuning:
        assert paths["chain"] == 0 and paths["chain_parts"] == 0
    else:
        assert paths["chain"] == 2
        # (a refusal in the first substep's first sweep keeps the second substep off the partition)
        absent = "partition_absent" in tuning
        assert paths["chain_parts"] == (1 if absent else 2)
        assert paths["refused"] == (1 if absent else 0) and paths["alone"] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("skin", [100, 1])
def test_candidate_list_left_out_after_failures(hip_lib, skin):
    # images that come and go, and a skin that every step outruns: lists that fail at their first
    # reuse, the substeps that go without one, and the next list
    h, _ = run_pair("bed_periodic", 300, 50, tuning={"candidate_skin_permille": skin})
    paths = h.debug_paths()
    # (after two lists in vain 8 substeps without, then 16, 32: all 50 in vain, 2 + 2 lists)
    assert paths["list_rebuilt"] >= 4 and paths["list_left_out"] >= 8
    assert (paths["list_reused"] > 0) == (skin == 100)
    assert skin == 100 or paths["list_rebuilt"] == 4


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["skin", "bodies", "autotune"])
def test_candidate_list_returns_after_a_change(hip_lib, change):
    # a skin that every step outruns, until the list is left out; a new skin, another number of
    # bodies or the autotuner's trials start with a list at once
    from peclet.dem import Simulation
    from scenes import apply_scene, make_scene

    scene = make_scene("bed_periodic", 300, 3)
    scene["vel"] = scene["vel"] + np.array([3.0, 2.0, 0.0])
    h = apply_scene(Simulation(300), scene)
    h.set_tuning("candidate_skin_permille", 1)
    for _ in range(24):  # (two lists in vain, eight substeps without, a third, sixteen without)
        h.step(scene["dt"])
        if h.debug_paths()["list_left_out"] >= 10:
            break
    before = h.debug_paths()
    assert before["list_left_out"] >= 10
    if change == "autotune":
        cfg, ms = h.autotune(scene["dt"], substeps=2, use_cache=False)
        # every trial with a skin of its own builds one: the current, four tried, the choice
        assert h.debug_paths()["list_rebuilt"] >= before["list_rebuilt"] + 4
    else:
        if change == "skin":
            h.set_tuning("candidate_skin_permille", 400)
        else:
            h.set_positions(scene["pos"][:280])
        h.step(scene["dt"])
        after = h.debug_paths()
        assert after["list_rebuilt"] == before["list_rebuilt"] + 1
        assert after["list_left_out"] == before["list_left_out"]
    h.close()
