"""Ray generation at the edges of its tiles and of the scanned form, and attributes of every half-precision pattern."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def context(crt):
    from candela_amd import scenes
    r = crt.RayIntersector(crt.FORMAT_STACKLESS)
    r.add_object(0, scenes.boxes_scene())
    r.push_entity(0)
    r.buffer_entities()
    r.buffer_data()
    return r


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1023, 1024, 1025, 262144, 262145, 4096 * 1024, 4096 * 1024 + 1])
@pytest.mark.parametrize("share", [0.0, 0.6, 1.0])
def test_raygen_keeps_order(crt, n, share):
    rng = np.random.default_rng(n)
    hits = np.zeros(n, crt.HIT_DTYPE)
    live = rng.random(n) < share
    hits["t"] = np.where(live, 2.0, -1.0)
    hits["tri"] = rng.integers(0, 3074, n)
    rays = np.zeros(n, crt.RAY_DTYPE)
    rays["dir"] = (0.0, -1.0, 0.0)
    rays["id"] = rng.permutation(n)
    r = context(crt)
    d_rays, d_hits = crt.DeviceArray.from_host(rays), crt.DeviceArray.from_host(hits)
    out = [crt.DeviceArray(crt.RAY_DTYPE, n) for _ in range(2)]
    for o in out:
        o.fill_bytes(0)
    gen = crt.RayGen(n)
    gen.diffuse(r.scene(), d_rays, d_hits, crt.raygen_params(seed=1), *out)
    assert gen.last_count() == live.sum()
    for o in out:
        got = o.download()
        assert np.array_equal(got["id"][:live.sum()], rays["id"][live])
        assert not got["tmax"][live.sum():].any()


def test_half_patterns(crt):
    """Normals of every finite half, denormals among them, against numpy's conversion (exact in both)."""
    h = np.arange(65536, dtype=np.uint32)
    h = h[np.isfinite(h.astype(np.uint16).view(np.float16))]
    other, third = np.roll(h, 7), np.roll(h, 29)
    r = context(crt)
    n = h.size
    verts = np.zeros(3 * n, crt.VERTEX_DTYPE)
    verts["normal_tangent_data"][0::3, 0] = h | other << 16
    verts["normal_tangent_data"][0::3, 1] = third
    tris = np.zeros(n, crt.TRIANGLE_DTYPE)
    tris["packed"][:, :3] = np.arange(3 * n).reshape(-1, 3)
    hits = np.zeros(n, crt.HIT_DTYPE)
    hits["t"], hits["u"] = 1.0, 1.0
    hits["tri"] = np.arange(n)
    d_v, d_t = crt.DeviceArray.from_host(verts), crt.DeviceArray.from_host(tris)
    view = r.scene()
    scene = crt.SceneView(view.format, view.entity_count, view.total_nodes, view.nodes, d_t.ptr, d_v.ptr, view.entities)
    out = crt.DeviceArray(crt.HIT_ATTR_DTYPE, n)
    for refs in (0, 1):       # without materials, and with one of no texture
        table = np.zeros(refs, crt.TEXTURE_REF_DTYPE)
        table["albedo"], table["model_color"] = -1, 0.25
        crt.hit_attributes(scene, crt.MaterialTable(table, []), crt.DeviceArray.from_host(hits), out)
        crt.lib().crt_device_sync()
        got = out.download()
        v = np.stack([x.astype(np.uint16).view(np.float16).astype(np.float32) for x in (h, other, third)], 1)
        with np.errstate(all="ignore"):
            il = np.float32(1.0) / np.sqrt(v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1] + v[:, 2] * v[:, 2])
            want = v * il[:, None]
        assert np.array_equal(got["normal"], want, equal_nan=True)
        assert (got["albedo"] == 0.25 * refs).all()
