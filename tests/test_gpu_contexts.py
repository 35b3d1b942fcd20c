"""A context's own calls (crt_intersect, crt_intersect_primary) over the stack layout and over several entities, against
crt_trace over the context's scene view, record for record."""
import time

import numpy as np
import pytest

from oracle_cases import axis_aligned_rays, crafted_stack_chain, random_rays
from test_gpu_pair import along_z, balanced, chain, patchy, same_as_array_walk

pytestmark = pytest.mark.gpu


def to_stack(crt, nodes):
    """The stack layout of a pre-order tree."""
    kind, link = nodes["min"][:, 3].view(np.int32), nodes["max"][:, 3].view(np.int32)
    inner = np.flatnonzero(kind == -1)
    entry = np.zeros(nodes.size, np.int32)
    entry[inner] = np.arange(inner.size)
    out = np.zeros(inner.size, crt.node_dtype(crt.FORMAT_STACK))
    for side, child in (("left", inner + 1), ("right", link[inner + 1])):
        out[side]["min"], out[side]["max"] = nodes["min"][child], nodes["max"][child]
        out[side]["max"][:, 3] = np.where(kind[child] == -1, entry[child], 0).astype(np.int32).view(np.float32)
    return out


def stack_context(crt, objects, entities):
    r = crt.RayIntersector(crt.FORMAT_STACK)
    for k, (n, t, v) in enumerate(objects):
        r.add_object_prebuilt(k, n, t, v)
    for e in entities:
        r.push_entity(e)
    r.buffer_entities()
    r.buffer_data()
    return r


def as_stack(crt, tree):
    return (to_stack(crt, tree[0]),) + tree[1:]


@pytest.mark.parametrize("entities", [[0], [0, 0, 1]], ids=["one", "several"])
@pytest.mark.parametrize("depth", [2, 15, 16, 17, 18, 19, 40, 63, 64, 65, 70])
def test_stack_depths(crt, depth, entities):
    """Around the stack's LDS part and its end, where the walk stops with the overflow flag."""
    _, tris, verts = chain(crt, 3, True)
    r = stack_context(crt, [(crafted_stack_chain(depth), tris, verts), as_stack(crt, chain(crt, 9, True))], entities)
    rays = along_z(crt, 130)
    rays["org"] += np.float32(0.3)
    hits = same_as_array_walk(crt, r, rays)
    closest = crt.DeviceArray(crt.HIT_DTYPE, rays.size)
    r.intersect(crt.QUERY_CLOSEST, crt.DeviceArray.from_host(rays), closest)
    crt.lib().crt_device_sync()
    assert ((closest.download()["status"] & crt.STATUS_STACK_OVERFLOW) != 0).any() == (depth > 64)
    assert hits.size == 130


@pytest.mark.parametrize("entities", [[0], [1, 0, 1]], ids=["one", "several"])
@pytest.mark.parametrize("leaves,per_leaf,count", [(2, 3, 200), (512, 2, 200), (4096, 0, 200), (4096, 3, 200),
                                                   (2048, 1, 200000)])
def test_stack_iteration_cap(crt, leaves, per_leaf, count, entities):
    """Trees of fewer and of more than 1,024 inner nodes; at the largest count rays of different visits side by side."""
    tree = patchy(crt, leaves, 1) if count > 1000 else balanced(crt, leaves, per_leaf)
    r = stack_context(crt, [as_stack(crt, tree), as_stack(crt, chain(crt, 5, True))], entities)
    rays = random_rays(count, [-0.04, -0.2, -2], [0.04, 0.2, -1], seed=count)
    rays["dir"] = (0, 0, 1)
    rays["dir"][::2, :2] = np.random.default_rng(6).uniform(-1e-3, 1e-3, (len(rays[::2]), 2))
    same_as_array_walk(crt, r, rays)


@pytest.mark.parametrize("log2", range(7))
@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
def test_rays_per_wave_over_instances(crt, fmt, log2):
    """Batches on both sides of each change of the rays that a wave takes, over one entity and over several."""
    from candela_amd import scenes
    rng = np.random.default_rng(log2)
    for count in (1, 7):
        r = crt.RayIntersector(fmt)
        r.add_object(0, scenes.icosphere_cloud(count=30, subdivisions=2, seed=log2, box=20.0))
        for k in range(count):
            m = np.eye(4)
            m[:3, 3] = rng.uniform(-15, 15, 3) if k else 0
            r.push_entity(0, m, translucency=0.5 if k == 3 else 0.0)
        r.buffer_entities()
        r.buffer_data()
        for n in ((6144 << log2) - 1, (6144 << log2) + 1):
            rays = random_rays(n, [-2, -2, -2], [22, 22, 22], seed=n)
            assert (same_as_array_walk(crt, r, rays, flags=n % 2)["t"] > 0).any()


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("flags", [0, 1, 2, 3])
def test_degenerate_rays_and_flags(crt, fmt, flags):
    from candela_amd import scenes
    for turned in (None, np.diag([1, -1, 2, 1]).astype(np.float32)):
        r = crt.RayIntersector(fmt)
        r.add_object(0, scenes.boxes_scene())
        r.push_entity(0)
        if turned is not None:
            r.push_entity(0, turned, translucency=0.5)
            r.push_entity(0, turned)
        r.buffer_entities()
        r.buffer_data()
        rays = axis_aligned_rays(4000, [-2, -1, -2], [18, 6, 18], seed=4)
        rays["org"][::3] = np.round(rays["org"][::3])       # on the planes of the boxes: 0 * inf
        rays["tmax"][::5], rays["tmax"][1::5], rays["tmax"][2::5] = np.nan, np.inf, 0.5
        rays["tmax"][3::25] = -1.0
        rays["dir"][7::40], rays["org"][9::40] = np.nan, np.inf
        same_as_array_walk(crt, r, rays, flags)


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("entities", [1, 5, 130])
@pytest.mark.parametrize("width,height,flags", [(1, 1, 0), (9, 17, 1), (7, 300, 2), (129, 255, 1), (640, 487, 0)])
def test_images_of_instances(crt, fmt, entities, width, height, flags):
    from candela_amd import scenes
    rng = np.random.default_rng(entities)
    r = crt.RayIntersector(fmt)
    r.add_object(0, scenes.icosphere_cloud(count=3, subdivisions=2, seed=4, box=4.0))
    for k in range(entities):
        m = np.eye(4)
        m[:3, 3] = rng.uniform(-8, 8, 3)
        r.push_entity(0, m, translucency=0.5 if k % 4 == 1 else 0.0)
    r.buffer_entities()
    r.buffer_data()
    iv, ip = scenes.camera_inverses(eye=(2.0, 3.0, -22.0), center=(0.0, 0.0, 0.0), fovy_deg=60.0, aspect=width / height)
    rays, hits = r.intersect_primary(width, height, iv, ip, flags=flags)
    again = crt.DeviceArray(crt.HIT_DTYPE, rays.count)
    crt.trace(r.scene(), crt.QUERY_CLOSEST, rays, again, flags=flags)
    crt.lib().crt_device_sync()
    assert np.array_equal(rays.download()["id"], np.arange(width * height, dtype=np.uint32))
    assert hits.download().tobytes() == again.download().tobytes()
    assert width < 100 or (hits.download()["t"] > 0).any()


def test_stack_rebuffered_data_and_cleared_copies(crt):
    first, second = (as_stack(crt, chain(crt, d, True)) for d in (6, 9))
    r = stack_context(crt, [first, second], [1, 0])
    rays = along_z(crt, 70)
    before = same_as_array_walk(crt, r, rays)
    r.add_object_prebuilt(0, *as_stack(crt, chain(crt, 70, True)))
    r.buffer_data()
    assert same_as_array_walk(crt, r, rays).tobytes() == before.tobytes()
    r.push_entity(0)
    r.push_entity(1)
    r.buffer_entities()
    last = same_as_array_walk(crt, r, rays)
    r.buffer_data(clear_cpu_data=True)
    assert same_as_array_walk(crt, r, rays).tobytes() == last.tobytes()


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
def test_images_of_many_instances_take_no_longer_than_a_thread_per_ray(crt, fmt):
    """64 instances that most rays pass by: waves whose lanes each went from entity to entity alone took 1.3 to 1.6 times
    as long."""
    from candela_amd import scenes
    rng = np.random.default_rng(1)
    r = crt.RayIntersector(fmt)
    r.add_object(0, scenes.icosphere_cloud(count=1, subdivisions=5, seed=2, box=1.0))
    for _ in range(64):
        m = np.diag([3.0, 3.0, 3.0, 1.0])
        m[:3, 3] = rng.uniform(-20, 20, 3)
        r.push_entity(0, m)
    r.buffer_entities()
    r.buffer_data()
    iv, ip = scenes.camera_inverses(eye=(0.0, 0.0, -24.0), center=(0.0, 0.0, 0.0), fovy_deg=60.0, aspect=640 / 480)
    rays, hits = r.intersect_primary(640, 480, iv, ip)
    flat = [np.ascontiguousarray(a.T.reshape(16), np.float32) for a in (iv, ip)]
    view = r.scene()

    def primary():
        crt.check(crt.lib().crt_intersect_primary(r.handle, rays.ptr, hits.ptr, 640, 480, flat[0].ctypes.data,
                                                  flat[1].ctypes.data, 0, None))

    def best(call):
        took = []
        for _ in range(6):
            crt.lib().crt_device_sync()
            t = time.perf_counter()
            for _ in range(10):
                call()
            crt.lib().crt_device_sync()
            took.append(time.perf_counter() - t)
        return min(took)

    alone = best(lambda: crt.trace(view, crt.QUERY_CLOSEST, rays, hits, kernel=crt.KERNEL_THREAD_PER_RAY))
    assert best(primary) < 1.2 * alone
