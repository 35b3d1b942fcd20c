"""Shading over 64-pixel tiles whose rays the waves of a workgroup share: visibility per ray and sums over many tiles."""
import numpy as np
import pytest

from shade_terms import order_bounds

pytestmark = pytest.mark.gpu


def problem(crt, fmt, pixels, lights, entities, seed=3):
    from candela_amd import scenes
    rng = np.random.default_rng(seed)
    r = crt.RayIntersector(fmt)
    r.add_object(0, scenes.boxes_scene())
    for k in range(entities):
        m = np.eye(4, dtype=np.float32)
        m[:3, 3] = (3.0 * k, 0.25 * k, -2.0 * k)
        r.push_entity(0, m)
    r.buffer_entities()
    r.buffer_data()
    height = 64
    width = -(-pixels // height)
    iv, ip = scenes.camera_inverses(aspect=1.0, **scenes.BOXES_CAMERA)
    rays, hits = r.intersect_primary(width, height, iv, ip)
    crt.lib().crt_device_sync()
    # any pixels in any order, so that a tile holds many triangles
    pick = rng.permutation(rays.count)[:pixels]
    rays = crt.DeviceArray.from_host(rays.download()[pick])
    hits = crt.DeviceArray.from_host(hits.download()[pick])
    ntri = r.host_buffers()["triangles"].size
    light = rng.uniform([-4.0, 6.0, -4.0], [20.0, 14.0, 20.0], size=(lights, 3)).astype(np.float32)
    model = crt.ShadingModel(rng.uniform(0.05, 0.95, (ntri, 3)), rng.uniform(0.05, 1.0, ntri), light,
                             rng.uniform(1.0, 10.0, lights))
    color = crt.DeviceArray(np.float32, 3 * pixels)
    rec = crt.DeviceArray(crt.SHADE_RECORD_DTYPE, pixels)
    model.forward(r.scene(), rays, hits, color, rec)
    crt.lib().crt_device_sync()
    return r, model, light, hits, color, rec


def traced_visibility(crt, r, x, n, light):
    rays = np.zeros(len(x), crt.RAY_DTYPE)
    rays["org"] = x + n * np.float32(1e-4)
    d = light - rays["org"]
    rays["tmax"] = np.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2])
    rays["dir"] = d * (np.float32(1.0) / rays["tmax"])[:, None]
    dr, dh = crt.DeviceArray.from_host(rays), crt.DeviceArray(crt.HIT_DTYPE, len(x))
    crt.trace(r.scene(), crt.QUERY_ANY, dr, dh, kernel=crt.KERNEL_THREAD_PER_RAY)
    crt.lib().crt_device_sync()
    return ~(dh.download()["t"] > 0)


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("pixels,lights,entities", [(1, 1, 1), (64, 16, 1), (65, 3, 2), (700, 16, 3), (5000, 8, 0)])
def test_visibility_equals_traced_shadow_rays(crt, fmt, pixels, lights, entities):
    r, _, light, hits, color, rec = problem(crt, fmt, pixels, lights, entities)
    got = rec.download()
    hit = hits.download()
    assert np.array_equal(got["tri0"], np.where(hit["t"] > 0, hit["tri"], -1))
    assert (color.download().reshape(-1, 3)[got["tri0"] < 0] == 0).all() and (got["vis"][got["tri0"] < 0] == 0).all()
    for base, x, n, live in ((0, "p", "n", got["tri0"] >= 0), (16, "q", "nq", got["tri1"] >= 0)):
        for l in range(lights):
            bit = (got["vis"] >> np.uint32(base + l)) & 1
            assert not bit[~live].any()
            if live.any():
                want = traced_visibility(crt, r, got[x][live], got[n][live], light[l])
                assert np.array_equal(bit[live].astype(bool), want)


def gradients(crt, r, model, rec, color, target, lo, n):
    from candela_amd import workloads
    g = [crt.DeviceArray(np.float32, k) for k in (3 * model.ntri, model.ntri, model.nl)]
    for d in g:
        d.fill_bytes(0)
    model.backward(r.scene(), workloads.DeviceSpan(rec, lo, n), workloads.DeviceSpan(color, 3 * lo, 3 * n),
                   workloads.DeviceSpan(target, 3 * lo, 3 * n), *g)
    crt.lib().crt_device_sync()
    return [d.download().astype(np.float64) for d in g]


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("pixels", [640, 40000, 300000])
def test_gradients_are_the_sum_over_tiles(crt, fmt, pixels):
    """One launch against the sum of launches over parts: several tiles per workgroup at the larger sizes, triangles
    that share an LDS entry at all."""
    r, model, _, _, color, rec = problem(crt, fmt, pixels, 8, 1)
    target = crt.DeviceArray(np.float32, 3 * pixels)
    target.fill_bytes(0)
    whole = gradients(crt, r, model, rec, color, target, 0, pixels)
    part = max(64, pixels // 30 // 64 * 64)
    parts = [gradients(crt, r, model, rec, color, target, lo, min(part, pixels - lo)) for lo in range(0, pixels, part)]
    assert np.count_nonzero(whole[1]) > 50
    bounds = order_bounds(model, rec.download(), color.download(), target.download())
    for k, got in enumerate(whole):
        want = sum(p[k] for p in parts)
        assert (np.abs(got - want) <= bounds[k]).all(), (k, np.flatnonzero(np.abs(got - want) > bounds[k]))


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("pixels", [192, 40000, 120000])
def test_triangles_of_one_lds_entry(crt, fmt, pixels):
    """Triangles 128 apart, several pixels of each in every wave, so that they keep pushing each other out of the entry
    they share, against launches over one triangle's pixels at a time."""
    r, model, _, _, color, rec = problem(crt, fmt, pixels, 4, 1)
    target = crt.DeviceArray(np.float32, 3 * pixels)
    target.fill_bytes(0)
    host = rec.download()
    rng = np.random.default_rng(pixels)
    tris = 5 + 128 * np.arange(6)
    live = host["tri0"] >= 0
    pick = rng.choice(tris, pixels).astype(np.int32)
    host["tri0"] = np.where(live, pick, -1)
    host["tri1"] = np.where(live & (host["tri1"] >= 0), rng.choice(tris + 1, pixels), -1)
    rec.upload(host)
    whole = gradients(crt, r, model, rec, color, target, 0, pixels)
    bounds = order_bounds(model, host, color.download(), target.download())
    want = [np.zeros_like(w) for w in whole]
    for t in tris:
        one = host.copy()
        one["tri0"] = np.where(live & (pick == t), t, -1)
        rec.upload(one)
        for w, g in zip(want, gradients(crt, r, model, rec, color, target, 0, pixels)):
            w += g
    assert (whole[1][tris] != 0).all()
    for k, got in enumerate(whole):
        assert (np.abs(got - want[k]) <= bounds[k]).all(), (k, np.flatnonzero(np.abs(got - want[k]) > bounds[k]))
