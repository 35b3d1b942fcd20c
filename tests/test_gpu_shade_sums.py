"""Rounding of the shading adjoint's light gradients, which every pixel of an image adds to: on average no more than that
of 128-pixel sums added one after the other, whatever the image's size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIGHTS, VALUES, RUNS = 16, 64, 24


def sum_128(terms, rng):
    """FP32 sums over the columns: 64 at a time as a wave adds them, two of those, then one after the other."""
    t = np.zeros((terms.shape[0], -(-terms.shape[1] // 128) * 128), np.float32)
    t[:, :terms.shape[1]] = terms
    t = t.reshape(len(t), -1, 2, 64)
    while t.shape[-1] > 1:
        half = t.shape[-1] // 2
        t = t[..., :half] + t[..., half:]
    t = t[..., 0, 0] + t[..., 1, 0]
    return np.cumsum(t[:, rng.permutation(t.shape[1])], axis=1, dtype=np.float32)[:, -1]


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("size", [64, 112, 181, 182, 250, 260, 330])
def test_light_gradients_round_no_more_than_128_pixel_sums(crt, fmt, size):
    from candela_amd import scenes, workloads
    rng = np.random.default_rng(size)
    n = size * size
    r = crt.RayIntersector(fmt)
    r.add_object(0, scenes.boxes_scene())
    r.push_entity(0)
    r.buffer_entities()
    r.buffer_data()
    ntri = r.host_buffers()["triangles"].size
    light = rng.uniform([-4.0, 90.0, -4.0], [20.0, 120.0, 20.0], size=(LIGHTS, 3)).astype(np.float32)
    model = crt.ShadingModel(np.full((ntri, 3), 0.5), np.full(ntri, 0.6), light, rng.uniform(1.0, 10.0, LIGHTS))
    # every pixel is the same point above the scene, in sight of every light; a pixel's terms differ by the residual alone
    host = np.zeros(n, crt.SHADE_RECORD_DTYPE)
    host["p"], host["n"], host["eye"], host["tri1"] = (8, 50, 8), (0, 1, 0), (0, 80, 3), -1
    rec = crt.DeviceArray.from_host(host)
    color, target = crt.DeviceArray(np.float32, 3 * n), crt.DeviceArray(np.float32, 3 * n)
    target.fill_bytes(0)
    g = [crt.DeviceArray(np.float32, k) for k in (3 * ntri, ntri, LIGHTS)]

    def gradient(lo, count):
        for d in g:
            d.fill_bytes(0)
        model.backward(r.scene(), workloads.DeviceSpan(rec, lo, count), workloads.DeviceSpan(color, 3 * lo, 3 * count),
                       workloads.DeviceSpan(target, 3 * lo, 3 * count), *g)
        crt.lib().crt_device_sync()
        return g[2].download()

    palette = rng.uniform(0.5, 1.0, VALUES).astype(np.float32)
    values = np.zeros((n, 3), np.float32)
    values[:VALUES, 0] = palette
    color.upload(values.reshape(-1))
    terms = np.stack([gradient(k, 1) for k in range(VALUES)], axis=1)     # one pixel: its terms themselves
    assert (terms > 0).all()
    got, model_error = [], []
    for _ in range(RUNS):
        pick = rng.integers(0, VALUES, n)
        values[:, 0] = palette[pick]
        color.upload(values.reshape(-1))
        exact = terms.astype(np.float64)[:, pick].sum(1)
        got.append(np.abs(gradient(0, n) - exact) / exact)
        model_error.append(np.abs(sum_128(terms[:, pick], rng) - exact) / exact)
    # means of LIGHTS * RUNS = 384 errors, a few percent apart by chance; twice as many additions give 1.4 times the error
    print("mean relative error", np.mean(got), "of 128-pixel sums", np.mean(model_error))
    assert np.mean(got) <= 1.2 * np.mean(model_error), (np.mean(got), np.mean(model_error))
