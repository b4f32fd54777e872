"""The single world's solve: over the GPU (colouring and data-flow sweeps) where its paths change: more
items than waves and an item per wave, bodies whose pairs exceed what a thread keeps (32), what a workgroup
counts in LDS (64 colours) and the colour starts kept there (1024), joints beside contacts; in one
workgroup (small worlds) with its rows in LDS, in memory, and where pairs or colours outgrow it.  Colour classes
equal the oracle's; velocities and impulses are the oracle's colour-order solve's within the 1e-5 the
other solver tests use (both sides round the same operations; the contact points differ by an ulp of
atan2f at most)."""
import numpy as np
import pytest

from helpers import impulse_error

pytestmark = pytest.mark.gpu

REL, ABS = 1e-5, 1e-6


def _close(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.all(np.abs(a - b) <= ABS + REL * np.abs(b))


def plate_scene(spheres):
    """A dynamic plate on the ground under `spheres` spheres, each resting on the plate alone: the plate is in
    every contact but one, so its pairs all take different colours."""
    from pe_amd.scenes import SHAPE_BOX, SHAPE_SPHERE, SceneBuilder
    b = SceneBuilder()
    side = int(np.ceil(np.sqrt(spheres)))
    w = 0.5 * side + 1.0
    b.add(SHAPE_BOX, (2 * w, 1.0, 2 * w), 1.0, (0.0, -0.5, 0.0), kin=1)
    b.add(SHAPE_BOX, (w, 0.4, w), 50.0 * spheres, (0.0, 0.199, 0.0))
    for k in range(spheres):
        x, z = (k % side - side / 2 + 0.5) * 0.45, (k // side - side / 2 + 0.5) * 0.45
        b.add(SHAPE_SPHERE, (0.2,), 10.0 + k % 7, (x, 0.598 - 0.0001 * (k % 3), z))
    return b.scene(name=f"plate{spheres}")


@pytest.mark.parametrize("spheres,blocks,mode", [(20, 0, 0), (80, 0, 0), (80, 1, 2), (80, 0, 1), (150, 0, 0), (1100, 0, 2), (1100, 3, 2)])
def test_one_body_in_many_pairs(spheres, blocks, mode):
    import pe_amd
    from pyoracle import OracleWorld
    sc = plate_scene(spheres)
    g, o = pe_amd.World(sc, max_pairs=40 * sc.n), OracleWorld(sc, 32)
    g.set_solver_blocks(blocks)
    g.set_colouring(mode)
    print(f"[plate] {spheres} spheres, blocks {blocks}, colouring {mode}", flush=True)
    for step in range(3):
        for stage in ("integrate", "broadphase", "narrowphase", "solve"):
            getattr(g, stage)()
            getattr(o, stage)()
        g.sync()
        gp = g.pairs()
        assert np.array_equal(gp, o.pairs())
        order, cs = g.solve_order()
        col = np.full(len(gp), -1)
        for c in range(len(cs) - 1):
            col[order[cs[c]:cs[c + 1]]] = c
        assert np.array_equal(col, o.color_of()), f"colour classes step {step}"
        assert len(cs) - 1 >= spheres
        _, _, gv, gw = g.state()
        _, _, ov, ow = o.state()
        assert _close(gv, ov) and _close(gw, ow), f"velocities step {step}"
        npts, _ = g.contacts()
        err, _ = impulse_error(g.impulses(), o.impulses(), npts)
        assert err <= REL, f"impulses step {step}: {err:.3e}"
        o.set_state(*[np.asarray(x, np.float64) for x in g.state()])
    g.close()


@pytest.mark.parametrize("blocks", [1, 2, 7, 0])
def test_results_do_not_depend_on_the_workgroups(blocks):
    """A pile in contact, and joint chains whose ends strike the ground: the same bits with one workgroup
    (many items per wave) as with the default's."""
    import pe_amd
    from pe_amd import scenes
    for sc, steps in ((scenes.grid_world(700, seed=5, p_sphere=0.3), 90), (scenes.joint_chain_scene(30, 9, seed=3), 60)):
        ref, w = pe_amd.World(sc), pe_amd.World(sc)
        w.set_colouring(2)
        w.set_solver_blocks(blocks)
        ref.set_colouring(2)
        ref.set_solver_blocks(16)
        print(f"[workgroups] {sc.name}, blocks {blocks}", flush=True)
        ref.step(steps)
        w.step(steps)
        w.sync()
        for a, b in zip(w.state(), ref.state()):
            assert np.array_equal(a.view(np.int32), b.view(np.int32))
        assert np.array_equal(w.impulses(), ref.impulses())
        ref.close()
        w.close()


def cluster_scene(n, size, seed=9):
    """n overlapping spheres in a cube of edge `size`: many pairs in contact per body."""
    from pe_amd.scenes import SHAPE_BOX, SHAPE_SPHERE, SceneBuilder
    rng = np.random.default_rng(seed)
    b = SceneBuilder()
    b.add(SHAPE_BOX, (60.0, 1.0, 60.0), 1.0, (0.0, -0.5, 0.0), kin=1)
    for x in rng.uniform(-0.5, 0.5, (n, 3)) * size + (0.0, 0.5 * size, 0.0):
        b.add(SHAPE_SPHERE, (0.3,), 100.0, x)
    return b.scene(name=f"cluster{n}")


@pytest.mark.parametrize("name", ["pair", "mixed", "boxes", "limit", "chains", "joint_demo", "cluster"])
def test_one_workgroup_equals_the_flow(name):
    """The solve of a small world in one workgroup and over the GPU: the same bits, the same colour classes.  (Two
    other worlds crowd the GPU, so that all of these up to 600 bodies are solved in one workgroup.)"""
    import pe_amd
    from pe_amd import scenes
    sc, steps = {"pair": lambda: (scenes.grid_world(1, seed=2), 70),
                 "mixed": lambda: (scenes.grid_world(350, seed=5), 90),
                 "boxes": lambda: (scenes.grid_world(560, seed=6, p_sphere=0.0), 100),
                 "limit": lambda: (scenes.grid_world(599, seed=7, p_sphere=0.2), 80),
                 "chains": lambda: (scenes.joint_chain_scene(30, 9, seed=3), 60),
                 "joint_demo": lambda: (scenes.joint_demo_scene(), 60),
                 "cluster": lambda: (cluster_scene(590, 2.6), 1)}[name]()
    a, b = pe_amd.World(sc, max_pairs=200 * sc.n), pe_amd.World(sc, max_pairs=200 * sc.n)
    b.set_colouring(2)
    crowd = [pe_amd.World(scenes.grid_world(700, seed=1)) for _ in range(2)]
    for w in crowd:
        w.set_solver_blocks(200)
    print(f"[one workgroup] {name}: {sc.n} bodies", flush=True)
    for part in (steps, 2 if steps > 1 else 3):
        a.step(part)
        b.step(part)
        a.sync()
        b.sync()
        for x, y in zip(a.state(), b.state()):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
        assert np.array_equal(a.impulses(), b.impulses())
        (oa, ca), (ob, cb) = a.solve_order(), b.solve_order()
        assert np.array_equal(ca, cb)
        for k in range(len(ca) - 1):
            assert np.array_equal(np.sort(oa[ca[k]:ca[k + 1]]), np.sort(ob[ca[k]:ca[k + 1]]))
        print(f"[one workgroup] {name}: {a.counts()}", flush=True)
        assert a.counts()["colour_rounds"] == 0 and (len(oa) == 0 or b.counts()["colour_rounds"] > 0)
        if name == "cluster" and part == steps:
            assert len(oa) * 28 + sc.n * 56 > 152 * 1024   # beyond the LDS the kernel works in
    for w in crowd:
        w.close()
    a.close()
    b.close()


@pytest.mark.parametrize("name", ["mixed", "boxes", "limit", "beyond", "cluster", "chains"])
def test_one_workgroup_up_to_its_limits(name):
    """As test_one_workgroup_equals_the_flow, at the sizes to which one workgroup is the default: 280 bodies, 600 with
    few contact points; a pile beyond; a cluster whose pairs outgrow its LDS."""
    import pe_amd
    from pe_amd import scenes
    sc, steps = {"mixed": lambda: (scenes.grid_world(200, seed=5), 90),
                 "boxes": lambda: (scenes.grid_world(275, seed=6, p_sphere=0.0), 100),
                 "limit": lambda: (scenes.grid_world(279, seed=7, p_sphere=0.2), 80),
                 "beyond": lambda: (scenes.grid_world(330, seed=7, p_sphere=0.2), 110),
                 "cluster": lambda: (cluster_scene(279, 0.9), 1),
                 "chains": lambda: (scenes.joint_chain_scene(66, 8, seed=3), 60)}[name]()
    a, b = pe_amd.World(sc, max_pairs=200 * sc.n), pe_amd.World(sc, max_pairs=200 * sc.n)
    b.set_colouring(2)
    print(f"[one workgroup] {name}: {sc.n} bodies", flush=True)
    for part in (steps, 2):
        a.step(part)
        a.sync()
        a.step(1)   # by now the contact points of the steps before are known
        b.step(part + 1)
        for x, y in zip(a.state(), b.state()):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
        assert np.array_equal(a.impulses(), b.impulses())
        (oa, ca), (ob, cb) = a.solve_order(), b.solve_order()
        assert np.array_equal(ca, cb)
        for k in range(len(ca) - 1):
            assert np.array_equal(np.sort(oa[ca[k]:ca[k + 1]]), np.sort(ob[ca[k]:ca[k + 1]]))
        if len(oa):   # the flow counts its tries, one workgroup does not
            assert (a.counts()["colour_rounds"] > 0) == (name == "beyond") and b.counts()["colour_rounds"] > 0
        if name == "cluster" and part == steps:
            assert len(oa) * 28 + sc.n * 56 > 152 * 1024   # beyond the LDS the kernel works in
    a.close()
    b.close()


def test_a_pile_that_lands_changes_the_route():
    """400 bodies: in one workgroup as they fall, over the GPU once they lie (by the contact points and colours of a step
    before), and again in one workgroup when they are set back into the air: the same bits as over the GPU throughout."""
    import pe_amd
    from pe_amd import scenes
    sc = scenes.grid_world(400, seed=9, p_sphere=0.2)
    a, b = pe_amd.World(sc), pe_amd.World(sc)
    b.set_colouring(2)
    start = a.state()
    routes = []
    print(f"[route] {sc.n} bodies", flush=True)
    for part in range(14):
        if part == 12:
            for w in (a, b):
                w.set_state(*start)
        for w in (a, b):
            w.step(10)
            w.sync()
        points = a.counts()["points"]
        if points:
            routes.append((points, a.counts()["colour_rounds"] > 0))
        for x, y in zip(a.state(), b.state()):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
    print(f"[route] {routes}", flush=True)
    assert not routes[0][1]
    assert any(r for _, r in routes) and not all(r for _, r in routes)
    a.close()
    b.close()


def heavy_scene(name):
    """Bodies in more than 32 pairs in contact beside each other: two plates on each other under spheres; a cluster
    whose bodies are all heavy; a plate in so many pairs that, beside the cluster, the colour sets outgrow
    their memory (max_pairs is the number of pairs)."""
    from pe_amd import scenes
    from pe_amd.scenes import SHAPE_BOX
    far = lambda sc, x: (sc.position.__iadd__(np.array([x, 0.0, 0.0])), sc)[1]
    if name == "plates":
        a, b = plate_scene(70), plate_scene(200)
        b.shape_param[1, :3] = (11.0, 0.4, 30.0)       # reaches over the smaller plate's spheres and plate
        return scenes.concat([a, far(b, 9.0)], "plates")
    if name == "cluster":
        return cluster_scene(300, 1.2)
    return scenes.concat([plate_scene(6000), far(cluster_scene(400, 2.0), 200.0)], "hub")


@pytest.mark.parametrize("name,blocks", [("plates", 0), ("plates", 1), ("cluster", 0), ("cluster", 3), ("hub", 0), ("hub", 2)])
def test_heavy_bodies_are_coloured_alike(name, blocks):
    """Pairs of bodies in many pairs, coloured over the GPU by the sets of their colours (a pair per thread and several,
    both bodies heavy, sets that do not fit), and by claims in one workgroup: the same classes, the same bits."""
    import pe_amd
    sc = heavy_scene(name)
    probe = pe_amd.World(sc, max_pairs=400 * sc.n)
    probe.step(1)
    cap = len(probe.pairs()) if name == "hub" else 400 * sc.n
    probe.close()
    a, b = pe_amd.World(sc, max_pairs=cap), pe_amd.World(sc, max_pairs=cap)
    a.set_colouring(2)
    a.set_solver_blocks(blocks)
    b.set_colouring(1)
    print(f"[heavy] {name}: {sc.n} bodies, {cap} pairs at most, blocks {blocks}", flush=True)
    for step in range(1 if name == "hub" else 3):
        a.step(1)
        b.step(1)
        (oa, ca), (ob, cb) = a.solve_order(), b.solve_order()
        assert np.array_equal(ca, cb) and len(ca) > 33
        for k in range(len(ca) - 1):
            assert np.array_equal(np.sort(oa[ca[k]:ca[k + 1]]), np.sort(ob[ca[k]:ca[k + 1]]))
        for x, y in zip(a.state(), b.state()):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
        assert np.array_equal(a.impulses(), b.impulses())
        print(f"[heavy] {name}: {a.counts()}", flush=True)
        assert (a.counts()["colour_rounds"] == 0) == (name == "hub")   # (claims, where the sets do not fit, count no tries)
    a.close()
    b.close()


def test_launch_called_off_solves_the_same():
    """Workgroups that do not wait for each other call the solve over the GPU off, and the last of them solves
    alone (any world whose workgroups could not be had at once): the same bits, also with more workgroups
    than the GPU holds beside other worlds' and with joints."""
    import ctypes
    import pe_amd
    from pe_amd import scenes
    from pe_amd._lib import check, lib
    for sc, steps in ((scenes.grid_world(900, seed=5, p_sphere=0.3), 90), (scenes.joint_chain_scene(80, 9, seed=3), 60)):
        a, b = pe_amd.World(sc), pe_amd.World(sc)
        b.set_solver_blocks(200)
        check(lib().pe_internal_set_flow_patience(b.h, ctypes.c_int64(0)))
        print(f"[called off] {sc.name}", flush=True)
        a.step(steps)
        b.step(steps)
        b.sync()
        for x, y in zip(a.state(), b.state()):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
        assert np.array_equal(a.impulses(), b.impulses())
        # the solve over the GPU counts its tries, one workgroup does not
        assert a.counts()["points"] > 0 and a.counts()["colour_rounds"] > 0 and b.counts()["colour_rounds"] == 0
        a.close()
        b.close()


def test_worlds_on_their_own_streams_and_threads():
    """More worlds than the GPU holds solves over it at once, stepped from several threads on their own streams:
    each as it is alone."""
    import threading
    import pe_amd
    from pe_amd import scenes
    sc = scenes.grid_world(900, seed=15, p_sphere=0.3)
    ref = pe_amd.World(sc)
    ref.step(80)
    want = ref.state()
    ws = [pe_amd.World(sc) for _ in range(6)]
    for w in ws:
        w.set_solver_blocks(256)
    print("[threads] 6 worlds", flush=True)
    ts = [threading.Thread(target=lambda w=w: [w.step(20) for _ in range(4)]) for w in ws]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for w in ws:
        w.sync()
        for x, y in zip(w.state(), want):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
        w.close()
    ref.close()


def test_worlds_that_come_and_go_change_the_route():
    """A world between the limits is solved over the GPU, in one workgroup while others crowd the GPU, and over it again
    when they are gone: each step as a world stepped alone."""
    import pe_amd
    from pe_amd import scenes
    sc = scenes.grid_world(400, seed=15, p_sphere=0.3)
    ref, w = pe_amd.World(sc), pe_amd.World(sc)
    big = scenes.grid_world(900, seed=5, p_sphere=0.3)
    print("[crowd] 401 bodies", flush=True)
    ref.step(120)
    w.step(120)
    w.sync()
    assert w.counts()["points"] > 700
    others = []
    for crowd in (False, True, False, True):
        if crowd:
            others = [pe_amd.World(big) for _ in range(2)]
            for o in others:
                o.set_solver_blocks(200)
        else:
            for o in others:
                o.close()
        w.step(3)
        w.sync()
        assert (w.counts()["colour_rounds"] > 0) == (not crowd)
    for o in others:
        o.close()
    ref.step(12)
    for x, y in zip(w.state(), ref.state()):
        assert np.array_equal(x.view(np.int32), y.view(np.int32))
    w.close()
    ref.close()


def test_velocities_nothing_updates_are_solved_alike():
    """A removed body, which no contact updates, has the solver's velocities after a solve on every path, also where
    the caller has set others since (the solver's are those of its last step): in one workgroup, over the GPU, and
    with the launch called off."""
    import ctypes
    import pe_amd
    from pe_amd import scenes
    from pe_amd._lib import check, lib
    sc = scenes.grid_world(150, seed=8, p_sphere=0.3)
    gone = 5
    print("[untouched] 151 bodies", flush=True)
    states = []
    for mode, patience in ((0, None), (2, None), (2, 0)):
        w = pe_amd.World(sc)
        w.set_colouring(mode)
        if patience is not None:
            check(lib().pe_internal_set_flow_patience(w.h, ctypes.c_int64(patience)))
        w.step(60)
        w.remove_body(gone)
        w.step(1)
        before = w.state()
        assert w.counts()["points"] > 0
        set_v = np.full((sc.n, 3), 3.25, np.float32)
        out = []
        for call in (w.solve, lambda: w.step(1)):
            w.set_state(v=set_v, w=set_v)
            call()
            w.sync()
            out.append(w.state())
            assert np.array_equal(out[-1][2][gone], before[2][gone]) and np.array_equal(out[-1][3][gone], before[3][gone])
        states.append(out)
        w.close()
    for other in states[1:]:
        for a, b in zip(states[0], other):
            for x, y in zip(a, b):
                assert np.array_equal(x.view(np.int32), y.view(np.int32))


def test_worlds_on_callers_streams_take_turns():
    """Worlds that crowd the GPU, stepped on streams of the caller's that come and go (a new stream may have the handle
    of a destroyed one): each as it is alone."""
    import pe_amd
    from pe_amd import scenes
    from pe_amd.hip import Stream
    sc = scenes.grid_world(900, seed=15, p_sphere=0.3)
    ref = pe_amd.World(sc)
    ref.step(60)
    want = ref.state()
    ws = [pe_amd.World(sc) for _ in range(4)]
    for w in ws:
        w.set_solver_blocks(256)
    print("[streams] 4 worlds", flush=True)
    for _ in range(6):
        streams = [Stream() for _ in ws]
        for w, st in zip(ws, streams):
            w.step_async(10, st.handle.value)
        for st in streams:
            st.close()
    for w in ws:
        w.sync()
        for x, y in zip(w.state(), want):
            assert np.array_equal(x.view(np.int32), y.view(np.int32))
        w.close()
    ref.close()


def test_more_than_1024_colours_with_joints():
    """Colours beyond those whose starts a workgroup keeps, and joints after them: the same bits as coloured by claims in
    one workgroup."""
    import pe_amd
    from pe_amd import scenes
    sc = scenes.concat([plate_scene(1100), scenes.joint_chain_scene(6, 5, seed=2)], "plate_chains")
    off = plate_scene(1100).n
    sc.position[off:] += np.array([150.0, 0.0, 0.0])
    joints = scenes.joint_chain_scene(6, 5, seed=2).joints
    for j in joints:
        j.body_a += off
        j.body_b += off
    a, b = pe_amd.World(sc, max_pairs=40 * sc.n), pe_amd.World(sc, max_pairs=40 * sc.n)
    print(f"[colours] {sc.n} bodies, {len(joints)} joints", flush=True)
    for w, mode in ((a, 2), (b, 1)):
        w.add_joints(joints)
        w.set_colouring(mode)
        w.step(2)
        w.sync()
    assert a.counts()["colors"] > 1024
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x.view(np.int32), y.view(np.int32))
    assert np.array_equal(a.impulses(), b.impulses())
    a.close()
    b.close()
