"""Raycasts on the device (pe_world_raycast) against the oracle's DefaultRaycastSolver restatement,
which is pinned bit for bit to the compiled reference (test_oracle_vs_ref.py::test_raycast_bit_exact).

The device world and the oracle step in lock-step for 30 steps (the poses and AABBs after integrate
are bit-identical), then a few hundred rays go to both: hit flag, body, distance, hit point and
normal bit-identical -- boxes, spheres, cylinders, a convex hull and the heightfield, rays with
ignore sets, rays from inside bodies, and queries the reference ends early at a mesh body whose
AABB the ray misses."""
import numpy as np
import pytest

from helpers import small_rain

pytestmark = pytest.mark.gpu


def _lockstep(sc, steps):
    import pe_amd
    from pyoracle import OracleWorld
    g, o = pe_amd.World(sc), OracleWorld(sc, 32, color_order=True)
    for _ in range(steps):
        g.integrate(); o.integrate()
        g.broadphase(); o.broadphase()
        g.narrowphase(); o.narrowphase()
        g.solve(); o.solve()
        g.sync()
        o.set_state(*[np.asarray(x, np.float64) for x in g.state()])
    return g, o


def _rays(sc, pos, rng, k, aim=None):
    lo, hi = pos.min(0) - 1, pos.max(0) + 1
    out = []
    for i in range(k):
        if aim is not None and i % 2 == 0:
            s = pos[aim] + rng.uniform(-0.4, 0.4, 3) + np.array([0.0, 8.0, 0.0])
            d = np.array([0.0, -1.0, 0.0]) + rng.normal(size=3) * 0.01
            length, ig = 20.0, []
        else:
            s = rng.uniform(lo, hi)
            d = rng.normal(size=3) if i % 3 else np.array([rng.normal() * 0.2, -1.0, rng.normal() * 0.2])
            if i % 7 == 0:
                d = np.array([0.0, -1.0, 0.0])
            length = float(rng.uniform(0.5, 40.0))
            ig = rng.choice(sc.n, 3, replace=False).tolist() if i % 5 == 0 else []
        d = d / np.linalg.norm(d)
        out.append((s.astype(np.float32), d.astype(np.float32), np.float32(length), ig))
    return out


@pytest.mark.parametrize("name", ["rain", "hull", "mix"])
def test_raycast_matches_oracle(name):
    from pe_amd import scenes
    mix = scenes.shape_mix_scene(160, seed=23, volume=(10, 6, 10), grid=12, ground_size=(14, 14))
    conv = np.nonzero(mix.shape_type == scenes.SHAPE_CONVEX)[0]
    keep = sorted([i for i in range(mix.n) if mix.shape_type[i] != scenes.SHAPE_CONVEX] + [int(conv[0])])
    sc = {"rain": small_rain(150, seed=2), "hull": mix.subset(keep), "mix": mix}[name]
    print(f"[raycast] {name}: n={sc.n}", flush=True)
    g, o = _lockstep(sc, 30)
    pos = np.asarray(g.state()[0], np.float64)
    rays = _rays(sc, pos, np.random.default_rng(7), 300, aim=keep.index(int(conv[0])) if name == "hull" else None)
    hits = partial = mesh = 0
    for k, (s, d, length, ig) in enumerate(rays):
        gh, gb, gd, gp, gn = g.raycast([s], [d], [length], ig)
        oh, ob, od, op, on = o.raycast(s.astype(np.float64), d.astype(np.float64), float(length), ig)
        assert bool(gh[0]) == oh and int(gb[0]) == ob, f"ray {k}: device {(gh[0], gb[0])} oracle {(oh, ob)}"
        assert gd[0] == np.float32(od), f"ray {k} distance"
        assert np.array_equal(gp[0], op.astype(np.float32)) and np.array_equal(gn[0], on.astype(np.float32)), f"ray {k}"
        hits += oh
        partial += (not oh) and ob >= 0
        mesh += oh and sc.shape_type[ob] >= scenes.SHAPE_CONVEX
    # the same rays in one call (one workgroup per ray)
    st = np.stack([r[0] for r in rays if not r[3]])
    dr = np.stack([r[1] for r in rays if not r[3]])
    ln = np.array([r[2] for r in rays if not r[3]], np.float32)
    bh, bb, bd, _, _ = g.raycast(st, dr, ln)
    for i, (s, d, length) in enumerate(zip(st, dr, ln)):
        oh, ob, od, _, _ = o.raycast(s.astype(np.float64), d.astype(np.float64), float(length))
        assert bool(bh[i]) == oh and int(bb[i]) == ob and bd[i] == np.float32(od), f"batched ray {i}"
    print(f"[raycast] {name}: {hits} hits ({mesh} on meshes), {partial} queries ended early with a partial "
          f"result, of {len(rays)}", flush=True)
    g.close()


@pytest.mark.parametrize("count", [1023, 1024, 1027])
@pytest.mark.parametrize("basis", ["turned", "scaled"])
def test_many_rays_sharing_a_pass_match_oracle(count, basis):
    """From 1024 rays on several share a workgroup, and boxes a ray passes well clear of are left out by a bound:
    grazing rays, rays along the axes, directions of other lengths than 1, starts far off and bases that
    are no rotations (where the bound does not hold and is not used) give the oracle's results."""
    import pe_amd
    from pyoracle import OracleWorld
    sc = small_rain(90, seed=11)
    rng = np.random.default_rng(count)
    g, o = pe_amd.World(sc), OracleWorld(sc, 32)
    pos, rot, v, w = (np.array(x, np.float32) for x in g.state())
    if basis == "scaled":
        rot[::2] = rot[::2] * np.float32(1.7)
        rot[1::4] = rot[1::4] * np.float32(0.4)
    g.set_state(pos, rot, v, w)
    o.set_state(*[x.astype(np.float64) for x in (pos, rot, v, w)])
    body = rng.integers(0, sc.n, count)
    far = rng.choice([0.0, 3.0, 60.0], count)[:, None]
    at = pos[body] + rng.uniform(-0.8, 0.8, (count, 3))      # past, along and through the faces and corners
    d = rng.normal(size=(count, 3))
    axis = rng.random(count) < 0.3
    d[axis] = np.eye(3)[rng.integers(0, 3, axis.sum())] * rng.choice([-1.0, 1.0], axis.sum())[:, None]
    d /= np.linalg.norm(d, axis=1)[:, None]
    st = (at - far * d).astype(np.float32)
    d = (d * rng.choice([1.0, 1.0, 0.05, 0.5, 4.0], count)[:, None]).astype(np.float32)
    ln = rng.uniform(0.5, 300.0, count).astype(np.float32)
    print(f"[raycast] {count} rays at once, {basis}", flush=True)
    gh, gb, gd, gp, gn = g.raycast(st, d, ln)
    hits = 0
    for k in range(count):
        oh, ob, od, op, on = o.raycast(st[k].astype(np.float64), d[k].astype(np.float64), float(ln[k]))
        assert bool(gh[k]) == oh and int(gb[k]) == ob and gd[k] == np.float32(od), f"ray {k}"
        assert np.array_equal(gp[k], op.astype(np.float32)) and np.array_equal(gn[k], on.astype(np.float32)), f"ray {k}"
        hits += oh
    assert hits > count // 4
    g.close()


@pytest.mark.parametrize("count", [1, 300, 1027])
def test_rays_through_many_meshes_match_oracle(count):
    """260 concentric hulls of several trees' sizes among boxes and spheres, every ray through the boxes of all
    of them: each thread of a workgroup walks a mesh at the same time (a stack row each), over
    every place a body can have in it."""
    import pe_amd
    from pe_amd import scenes
    from pe_amd.scenes import SHAPE_BOX, SHAPE_CONVEX, SHAPE_SPHERE, SceneBuilder
    from pyoracle import OracleWorld
    rng = np.random.default_rng(31)
    b = SceneBuilder()
    ids = [b.add_mesh(scenes.gaussian_hull(rng, int(k), r)) for k, r in ((8, 2.0), (20, 1.0), (60, 1.5), (200, 1.2), (400, 1.8))]
    rots = scenes.quat_to_matrix(scenes.random_quaternions(rng, 300))
    for k in range(300):
        if k % 15 == 0:
            b.add(SHAPE_BOX, rng.uniform(0.2, 1.0, 3), 1.0, rng.uniform(-2.0, 2.0, 3), rot=rots[k], kin=1)
        elif k % 15 == 1:
            b.add(SHAPE_SPHERE, (0.3,), 1.0, rng.uniform(-2.0, 2.0, 3), kin=1)
        else:
            b.add(SHAPE_CONVEX, (), 1.0, rng.uniform(-0.05, 0.05, 3), rot=rots[k], kin=1, mesh=ids[int(rng.integers(0, len(ids)))])
    sc = b.scene(name="nested")
    g, o = pe_amd.World(sc), OracleWorld(sc, 32)
    g.integrate()   # (all kinematic: this makes their AABBs)
    o.integrate()
    way = rng.normal(size=(count, 3))
    way /= np.linalg.norm(way, axis=1)[:, None]
    st = (rng.uniform(-0.1, 0.1, (count, 3)) - 6.0 * way).astype(np.float32)
    d, ln = way.astype(np.float32), rng.uniform(3.0, 9.0, count).astype(np.float32)
    print(f"[raycast] {count} rays through {sc.n} bodies", flush=True)
    gh, gb, gd, gp, gn = g.raycast(st, d, ln)
    mesh = 0
    for k in range(count):
        oh, ob, od, op, on = o.raycast(st[k].astype(np.float64), d[k].astype(np.float64), float(ln[k]))
        assert bool(gh[k]) == oh and int(gb[k]) == ob and gd[k] == np.float32(od), f"ray {k}"
        assert np.array_equal(gp[k], op.astype(np.float32)) and np.array_equal(gn[k], on.astype(np.float32)), f"ray {k}"
        mesh += oh and sc.shape_type[ob] == SHAPE_CONVEX
    assert mesh > count // 4
    g.close()
