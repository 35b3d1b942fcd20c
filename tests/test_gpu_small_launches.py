"""Launches of the speculative walks around the sizes where a wave takes fewer rays, and where the refilling presets
take rays from the queue: every ray's record is that of one large launch."""
import numpy as np
import pytest

from oracle_cases import random_rays

pytestmark = pytest.mark.gpu

LARGE = 400000                      # more than the waves of an idle device take at once
COUNTS = [1, 2, 63, 2048, 2049, 4100, 32768, 32769, 65536, 65537, 70001, 131073, 327680, 327681]


@pytest.fixture(scope="module")
def wide(crt):
    from candela_amd import scenes
    r = crt.RayIntersector(crt.FORMAT_STACKLESS)
    r.add_object(0, scenes.boxes_scene())
    r.push_entity(0)
    r.buffer_entities()
    r.buffer_data()
    return {w: crt.upload_wide(crt.FORMAT_STACKLESS, r.host_buffers(), w, 2) for w in (4, 8)}


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("kernel,variant,query", [("SPECULATIVE", 5, 1), ("SPECULATIVE", 4, 0),
                                                  ("SPECULATIVE_REFILL", 4, 0), ("SPECULATIVE_REFILL", 5, 1)])
def test_traces(crt, wide, width, kernel, variant, query):
    k = getattr(crt, "KERNEL_" + kernel)
    rays = crt.DeviceArray.from_host(random_rays(LARGE, [-4, 0, -4], [20, 8, 20], seed=6))
    scene = wide[width].scene

    def trace(n):
        from candela_amd import workloads
        hits = crt.DeviceArray(crt.HIT_DTYPE, n)
        hits.fill_bytes(255)
        crt.trace(scene, query, workloads.DeviceSpan(rays, 0, n), hits, kernel=k, variant=variant)
        crt.lib().crt_device_sync()
        return hits.download()

    whole = trace(LARGE)
    assert (whole["t"] > 0).mean() > 0.2
    for n in COUNTS:
        assert trace(n).tobytes() == whole[:n].tobytes(), n


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("variant", [6, 7])
def test_paths(crt, wide, width, variant):
    from candela_amd import scenes
    iv, ip = scenes.camera_inverses(aspect=1.0, **scenes.BOXES_CAMERA)
    albedo = crt.DeviceArray.from_host(np.full(6, 0.6, np.float32))
    camera = [np.ascontiguousarray(m.T.reshape(16)) for m in (iv, ip)]

    def paths(height):
        out = crt.DeviceArray(crt.PATH_SAMPLE_DTYPE, 641 * height)
        out.fill_bytes(255)
        p = crt.path_params(641, LARGE // 641, 1, *camera, albedo=albedo, seed=5)
        crt.trace_paths(wide[width].scene, p, out, variant=variant)
        crt.lib().crt_device_sync()
        return out.download()

    whole = paths(LARGE // 641)
    for height in (1, 3, 4, 7, 100, 205, 511, 512):
        assert paths(height).tobytes() == whole[:641 * height].tobytes(), height


def test_half_of_the_rays_take_no_longer(crt):
    """40,000 rays over eight overlapping entities against 80,000: in waves of 32 they took 1.25 times as long."""
    import time

    from candela_amd import scenes, workloads
    rng = np.random.default_rng(1)
    r = crt.RayIntersector(crt.FORMAT_STACKLESS)
    r.add_object(0, scenes.boxes_scene())
    for _ in range(8):
        m = np.eye(4)
        m[:3, 3] = rng.uniform(-20, 20, 3)
        r.push_entity(0, m)
    r.buffer_entities()
    r.buffer_data()
    scene = crt.upload_wide(crt.FORMAT_STACKLESS, r.host_buffers(), 4, 2, None, None, crt.COLLAPSE_SAH, 0.0, 0.3)
    rays = crt.DeviceArray.from_host(random_rays(80000, [-25] * 3, [25] * 3, seed=40000))
    best = {}
    for n in (40000, 80000):
        span, hits = workloads.DeviceSpan(rays, 0, n), crt.DeviceArray(crt.HIT_DTYPE, n)
        took = []
        for _ in range(8):
            crt.lib().crt_device_sync()
            t = time.perf_counter()
            for _ in range(20):
                crt.trace(scene.scene, crt.QUERY_CLOSEST, span, hits, kernel=crt.KERNEL_SPECULATIVE, variant=0)
            crt.lib().crt_device_sync()
            took.append(time.perf_counter() - t)
        best[n] = min(took)
    assert best[40000] < 1.1 * best[80000], best
