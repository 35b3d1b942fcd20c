"""The walk over child pairs (crt_intersect and crt_intersect_primary of a stackless context) against the walk of the
stackless array itself (crt_trace over the context's scene view), record for record."""
import numpy as np
import pytest

from oracle_cases import axis_aligned_rays, random_rays

pytestmark = pytest.mark.gpu


def bits(a):
    return np.asarray(a, np.int32).view(np.float32)


def chain(crt, depth, right, per_leaf=1, box=1e3):
    """A tree of `depth` inner nodes one below the other, on the left or the right side, every box the same, with
    triangles that lie apart from the origin's z axis, but for the last."""
    count = 2 * depth + 1
    nodes = np.zeros(count, crt.node_dtype(crt.FORMAT_STACKLESS))
    nodes["min"][:, :3], nodes["max"][:, :3] = -box, box
    kind, link = np.zeros(count, np.int32), np.zeros(count, np.int32)
    if right:       # inner, leaf, inner, leaf, ..., leaf
        inner = np.arange(0, 2 * depth, 2)
        kind[inner] = -1
        link[:] = -1
        link[inner + 1] = inner + 2
        leaves = np.append(inner + 1, 2 * depth)
    else:           # inner, inner, ..., leaf, leaf, ...
        kind[:depth] = -1
        link[:depth] = np.append(-1, np.arange(2 * depth, depth + 1, -1))[:depth]
        link[depth:] = np.arange(depth + 1, count + 1)
        link[-1] = -1
        leaves = np.arange(depth, count)
    kind[leaves] = (np.arange(leaves.size) * per_leaf) << 4 | per_leaf
    nodes["min"][:, 3], nodes["max"][:, 3] = bits(kind), bits(link)
    ntri = max(1, leaves.size * per_leaf)
    pos = np.zeros((ntri, 3, 3), np.float32)
    pos[:, 0], pos[:, 1], pos[:, 2] = (5, 5, 0), (6, 5, 0), (5, 6, 0)
    pos[-1] = (-1, -1, 7), (1, -1, 7), (0, 1, 7)
    verts = np.zeros(3 * ntri, crt.VERTEX_DTYPE)
    verts["position"][:, :3] = pos.reshape(-1, 3)
    tris = np.zeros(ntri, crt.TRIANGLE_DTYPE)
    tris["packed"][:, :3] = np.arange(3 * ntri).reshape(-1, 3)
    tris["packed"][:, 3] = 3
    return nodes, tris, verts


def context(crt, objects, entities):
    r = crt.RayIntersector(crt.FORMAT_STACKLESS)
    for k, (n, t, v) in enumerate(objects):
        r.add_object_prebuilt(k, n, t, v)
    for e in entities:
        r.push_entity(e)
    r.buffer_entities()
    r.buffer_data()
    return r


def same_as_array_walk(crt, r, rays, flags=0):
    d = crt.DeviceArray.from_host(rays)
    for query in (crt.QUERY_CLOSEST, crt.QUERY_ANY):
        a, b = crt.DeviceArray(crt.HIT_DTYPE, rays.size), crt.DeviceArray(crt.HIT_DTYPE, rays.size)
        r.intersect(query, d, a, flags=flags)
        crt.trace(r.scene(), query, d, b, flags=flags)
        crt.lib().crt_device_sync()
        got, want = a.download(), b.download()
        assert got.tobytes() == want.tobytes(), f"query {query}: {np.count_nonzero(got != want)} records differ"
    return want


def along_z(crt, n):
    rays = random_rays(n, [-0.2, -0.2, -2], [0.2, 0.2, -1], seed=n)
    rays["dir"][::2] = (0, 0, 1)
    return rays


@pytest.mark.parametrize("right", [False, True], ids=["left", "right"])
@pytest.mark.parametrize("depth", [1, 9, 10, 11, 12, 13, 40, 64, 65, 200])
def test_depths(crt, depth, right):
    """Around the stack's LDS part, its end and the depth from which the array itself is walked."""
    r = context(crt, [chain(crt, depth, right)], [0])
    hits = same_as_array_walk(crt, r, along_z(crt, 130))
    assert (hits["t"] > 0).any()


def balanced(crt, leaves, per_leaf):
    """A complete tree over `leaves` (a power of two) copies of the chain's triangles."""
    nodes, tris, verts = chain(crt, leaves - 1, False, per_leaf)
    kind, link = nodes["min"][:, 3].view(np.int32), nodes["max"][:, 3].view(np.int32)
    kind, link = kind.copy(), link.copy()

    def place(at, first, n, escape):
        link[at] = escape
        kind[at] = -1 if n > 1 else (first * per_leaf) << 4 | per_leaf
        if n > 1:
            right = at + n                     # a left subtree of n / 2 leaves has n - 1 nodes
            place(at + 1, first, n // 2, right)
            place(right, first + n // 2, n // 2, escape)
    place(0, 0, leaves, -1)
    nodes["min"][:, 3], nodes["max"][:, 3] = bits(kind), bits(link)
    return nodes, tris, verts


@pytest.mark.parametrize("leaves,per_leaf", [(2, 3), (256, 0), (512, 1), (512, 2), (1024, 1), (4096, 3)])
def test_iteration_cap(crt, leaves, per_leaf):
    """1,023 nodes stay below the cap of 1,024 visits, 2,047 and 8,191 exceed it, with empty and odd leaves too."""
    r = context(crt, [balanced(crt, leaves, per_leaf), chain(crt, 5, True)], [0, 1, 0])
    hits = same_as_array_walk(crt, r, along_z(crt, 200))
    assert ((hits["status"] & crt.STATUS_ITER_CAP) != 0).any() == (leaves > 512)


def patchy(crt, leaves, seed):
    """A complete tree whose boxes each cover a part of x at random, the middle always: rays visit from a few hundred
    to all of its nodes.  The triangles cover every ray, each nearer than those before it."""
    nodes, tris, verts = balanced(crt, leaves, 1)
    rng = np.random.default_rng(seed)
    nodes["min"][1:, 0] = rng.uniform(-0.2, 0.0, nodes.size - 1)
    nodes["max"][1:, 0] = rng.uniform(0.0, 0.2, nodes.size - 1)
    corners = np.array([(-9, -9, 0), (9, -9, 0), (0, 18, 0)], np.float32)
    pos = np.repeat(corners[None], leaves, axis=0)
    pos[:, :, 2] = 7 - np.arange(leaves, dtype=np.float32)[:, None] / leaves
    verts["position"][:, :3] = pos.reshape(-1, 3)
    return nodes, tris, verts


@pytest.mark.parametrize("entities", [[0], [1, 0, 1]], ids=["one", "several"])
def test_iteration_cap_in_full_waves(crt, entities):
    """Rays below and above the cap side by side, 64 to a wave: a ray that starts again to count each visit in its turn
    leaves its neighbours' records alone."""
    r = context(crt, [patchy(crt, 2048, 1), chain(crt, 9, True)], entities)
    rays = random_rays((6144 << 6) // 2 + 777, [-0.04, -0.2, -2], [0.04, 0.2, -1], seed=5)
    rays["dir"] = (0, 0, 1)
    rays["dir"][::2, :2] = np.random.default_rng(6).uniform(-1e-3, 1e-3, (len(rays[::2]), 2))
    hits = same_as_array_walk(crt, r, rays)
    assert ((hits["status"] & 0xFFFFFF) > 0).all()
    closest = crt.DeviceArray(crt.HIT_DTYPE, rays.size)
    r.intersect(crt.QUERY_CLOSEST, crt.DeviceArray.from_host(rays), closest)
    crt.lib().crt_device_sync()
    capped = (closest.download()["status"] & crt.STATUS_ITER_CAP) != 0
    assert 0.2 < capped.mean() < 0.8


@pytest.mark.parametrize("log2", range(7))
def test_rays_per_wave(crt, log2):
    """Batches on both sides of each change of the rays that a wave takes."""
    from candela_amd import scenes
    r = crt.RayIntersector(crt.FORMAT_STACKLESS)
    r.add_object(0, scenes.icosphere_cloud(count=30, subdivisions=2, seed=log2, box=20.0))
    r.push_entity(0)
    r.buffer_entities()
    r.buffer_data()
    for n in ((6144 << log2) - 1, 6144 << log2, (6144 << log2) + 1):
        assert (same_as_array_walk(crt, r, random_rays(n, [-2, -2, -2], [22, 22, 22], seed=n))["t"] > 0).any()


def test_one_leaf_object_and_empty_scene(crt):
    nodes, tris, verts = chain(crt, 1, True)
    nodes = nodes[1:2].copy()
    nodes["max"][:, 3], nodes["min"][:, 3] = bits([-1]), bits([1 << 4 | 1])
    assert (same_as_array_walk(crt, context(crt, [(nodes, tris, verts)], [0, 0]), along_z(crt, 65))["t"] > 0).any()
    same_as_array_walk(crt, context(crt, [(nodes, tris, verts)], []), along_z(crt, 65))


def test_other_trees_walk_the_array(crt):
    """Nodes behind the tree, a link that skips a subtree, leaves beyond the triangles' end (in a box that no ray
    meets): the array's own walk answers."""
    nodes, tris, verts = chain(crt, 20, False)
    longer = np.concatenate([nodes, nodes[-1:]])
    skip = nodes.copy()
    skip["max"][20, 3] = bits([23])[0]
    beyond = nodes.copy()
    beyond["min"][25, :3] = beyond["max"][25, :3] = 5e3
    beyond["min"][25, 3] = bits([1000 << 4 | 2])[0]
    for n in (longer, skip, beyond):
        same_as_array_walk(crt, context(crt, [(n, tris, verts), chain(crt, 3, True)], [0, 1]), along_z(crt, 100))


def test_many_objects(crt):
    """Trees of sizes around a workgroup's 256 nodes, one behind the other at any offset, and between them arrays that are
    no trees (an even number of nodes, inner nodes alone, a leaf beyond the triangles), which no entity names."""
    trees = [balanced(crt, k, 1) for k in (2, 64, 128, 256)]
    trees += [chain(crt, d, right) for d in (1, 20, 126, 127, 128, 129, 300) for right in (False, True)]
    nodes, tris, verts = chain(crt, 130, True)
    only_inner, beyond = nodes[:200].copy(), nodes.copy()
    only_inner["min"][:, 3], only_inner["max"][:, 3] = bits([-1]), bits([-1])
    beyond["min"][-1, 3] = bits([100000 << 4 | 1])[0]
    others = [(n, tris, verts) for n in (nodes[:-1], only_inner, beyond, nodes[:2])]
    objects, named = [], []
    for k, t in enumerate(trees):
        named.append(len(objects))
        objects += [t, others[k % len(others)]]
    rays = along_z(crt, 130)
    for k in named:
        assert (same_as_array_walk(crt, context(crt, objects, [k]), rays)["t"] > 0).any()
    same_as_array_walk(crt, context(crt, objects, named), rays)
    named.append(1)       # an entity that names such an array: all walk the array
    same_as_array_walk(crt, context(crt, objects, named), rays)


def test_buffering_costs_what_it_copies(crt):
    """A stackless context, with child pairs, against the stack layout's of the same scene, which copies more."""
    import time

    from candela_amd import scenes
    mesh = scenes.icosphere_cloud(count=500, subdivisions=3, seed=2, box=63.0)
    best = []
    for fmt in (crt.FORMAT_STACK, crt.FORMAT_STACKLESS):
        r = crt.RayIntersector(fmt)
        r.add_object(0, mesh)
        took = []
        for _ in range(8):
            crt.lib().crt_device_sync()
            t = time.perf_counter()
            r.buffer_data()
            took.append(time.perf_counter() - t)
        best.append(min(took))
    assert best[1] < 1.6 * best[0], best


def test_rebuffered_data_and_cleared_copies(crt):
    """An object that took another's id beside the entities of the first, then the host copies gone."""
    r = context(crt, [chain(crt, 6, True), chain(crt, 9, False)], [1, 0])
    rays = along_z(crt, 70)
    first = same_as_array_walk(crt, r, rays)
    r.add_object_prebuilt(0, *chain(crt, 70, True))
    r.buffer_data()
    assert same_as_array_walk(crt, r, rays).tobytes() == first.tobytes()
    r.push_entity(0)
    r.push_entity(1)
    r.buffer_entities()
    same_as_array_walk(crt, r, rays)      # an entity of 71 levels: all walk the array
    r.push_entity(1)
    r.buffer_entities()
    last = same_as_array_walk(crt, r, rays)
    r.buffer_data(clear_cpu_data=True)
    assert same_as_array_walk(crt, r, rays).tobytes() == last.tobytes()


@pytest.mark.parametrize("flags", [0, 1, 2, 3])
def test_degenerate_rays(crt, flags):
    from candela_amd import scenes
    r = crt.RayIntersector(crt.FORMAT_STACKLESS)
    r.add_object(0, scenes.boxes_scene())
    r.push_entity(0)
    r.push_entity(0, np.diag([1, -1, 2, 1]).astype(np.float32), translucency=0.5)
    r.buffer_entities()
    r.buffer_data()
    rays = axis_aligned_rays(4000, [-2, -1, -2], [18, 6, 18], seed=4)
    rays["org"][::3] = np.round(rays["org"][::3])       # on the planes of the boxes: 0 * inf
    rays["tmax"][::5], rays["tmax"][1::5], rays["tmax"][2::5] = np.nan, np.inf, 0.5
    rays["tmax"][3::25] = -1.0
    rays["dir"][7::40], rays["org"][9::40] = np.nan, np.inf
    same_as_array_walk(crt, r, rays, flags)


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("width,height", [(1, 1), (8, 8), (7, 300), (300, 7), (9, 17), (129, 255), (640, 487)])
def test_primary_images(crt, fmt, width, height):
    from candela_amd import scenes
    r = crt.RayIntersector(fmt)
    r.add_object(0, scenes.boxes_scene())
    r.push_entity(0)
    r.buffer_entities()
    r.buffer_data()
    iv, ip = scenes.camera_inverses(aspect=width / height, **scenes.BOXES_CAMERA)
    rays, hits = r.intersect_primary(width, height, iv, ip)
    again = crt.DeviceArray(crt.HIT_DTYPE, rays.count)
    crt.trace(r.scene(), crt.QUERY_CLOSEST, rays, again)
    crt.lib().crt_device_sync()
    assert np.array_equal(rays.download()["id"], np.arange(width * height, dtype=np.uint32))
    assert hits.download().tobytes() == again.download().tobytes()
