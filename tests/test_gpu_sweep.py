"""The sweep-and-prune stage at the sizes where its paths change: the edges of the counting sort's workgroups (64
bodies) and key tiles (2048), the change to the radix sort (beyond 16 384 bodies), the edges of the sweep's
workgroups (16 bodies), bodies whose run is everything, with tied keys, signed zeros, kinematic,
ignoring and removed bodies.  Pairs in order, bit for bit, against a stable sort and a sweep in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def records(n, seed, wide=0):
    """AABB records [n, 8]: minima on a grid of 1/4 (ties), extents up to 1.5; `wide` bodies span everything."""
    rng = np.random.default_rng(seed)
    side = max(2.0, 1.3 * n ** (1.0 / 3.0))
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = np.round(rng.uniform(-side, side, (n, 3)) * 4.0) / 4.0 * (1.0, 0.6, 1.4)
    r[:, 0:3][r[:, 0:3] == 0.0] *= np.float32(-1.0)
    r[:, 4:7] = r[:, 0:3] + np.round(rng.uniform(0.25, 1.5, (n, 3)) * 8.0) / 8.0
    for k in rng.permutation(n)[:wide]:
        r[k, 0:3], r[k, 4:7] = -5.0 * side, 5.0 * side
    r[:, 3] = rng.random(n) < 0.1
    r[:, 7] = rng.choice([0.0, 0.0, 0.0, 0.0, 0.0, 1.0], n)
    if n > 40:   # bodies that have left the world
        for k in rng.permutation(n)[:3]:
            r[k] = (np.inf, np.inf, np.inf, 0.0, -np.inf, -np.inf, -np.inf, 1.0)
    return r


def sweep(r, axis):
    key = r[:, axis] + np.float32(0.0)
    order = np.argsort(key, kind="stable")
    R, sk = r[order], key[order]
    end = np.searchsorted(sk, R[:, 4 + axis], side="right")
    pa, pb = [], []
    for q in range(len(r)):
        j = np.arange(q + 1, max(q + 1, end[q]))
        ok = (R[q, 7] != 1.0) & (R[j, 7] != 1.0) & ~((R[q, 3] != 0) & (R[j, 3] != 0))
        for k in range(3):
            ok &= (R[q, k] <= R[j, 4 + k]) & (R[j, k] <= R[q, 4 + k])
        j = j[ok]
        pa.append(np.full(len(j), order[q]))
        pb.append(order[j])
    c = ((r[:, 0:3] + r[:, 4:7]) * np.float32(0.5))[r[:, 0] <= r[:, 4]]
    var = (c.astype(np.float64) * c).sum(0) - c.astype(np.float64).sum(0) ** 2 / len(c)
    return np.concatenate(pa), np.concatenate(pb), int(np.argmax(var))


@pytest.mark.parametrize("n,wide", [(2, 0), (3, 1), (15, 0), (16, 1), (17, 2), (63, 0), (64, 1), (65, 5), (257, 40), (2047, 1),
                                    (2048, 0), (2049, 3), (6000, 2), (16384, 1), (16385, 1), (20000, 2)])
def test_sweep_equals_a_stable_sort_and_sweep(n, wide):
    from pe_amd.hip import DeviceArray
    from pe_amd.stage import Stage
    r = records(n, seed=n)
    if wide:
        r = records(n, n, wide)
    cap = 40 * n + 4 * wide * n + 64
    st = Stage(n, cap)
    buf = DeviceArray.from_numpy(r)
    for axis in range(3) if n <= 6000 else (0, 2):
        print(f"[sweep] n={n} wide={wide} axis {axis}", flush=True)
        pa, pb, res = st.broadphase(buf, axis, cap)
        a, b, nxt = sweep(r, axis)
        got = res.numpy()
        assert list(got) == [len(a), nxt, 0]
        assert np.array_equal(pa.numpy()[:len(a)], a) and np.array_equal(pb.numpy()[:len(a)], b)
    few = max(1, len(a) // 2)   # the output's capacity cuts the same list short
    pa, pb, res = st.broadphase(buf, axis, few)
    assert res.numpy()[0] == len(a) and (res.numpy()[2] & 1) == (1 if len(a) > few else 0)
    few = min(few, len(a))
    assert np.array_equal(pa.numpy()[:few], a[:few])
    st.close()


@pytest.mark.parametrize("n,wide", [(2111, 1), (2112, 0), (2113, 2), (60011, 1)])
def test_sweep_in_blocks_of_64(n, wide):
    """The sweep's blocks beyond 2048 bodies at their edges, and over more blocks than a workgroup has threads."""
    test_sweep_equals_a_stable_sort_and_sweep(n, wide)
