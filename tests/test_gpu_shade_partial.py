"""The shading adjoint over record counts that are no whole number of its 128-pixel tiles.

The records behind the requested ones are valid pixels of the same image, so a lane past the end that read its
record would add that pixel's gradient (and stay in bounds).  The expected gradients are those of the same call over
the whole buffer with every record behind the requested ones marked as a miss.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZE = 32


@pytest.mark.parametrize("fmt", [0, 1], ids=["stackless", "stack"])
@pytest.mark.parametrize("count", [1, 63, 65, 127, 129, 700, SIZE * SIZE - 1, SIZE * SIZE])
def test_backward_stops_at_the_count(fmt, count):
    import candela_amd as crt
    from candela_amd import workloads
    n = SIZE * SIZE
    pb = workloads.shading_problem(crt, size=SIZE, fmt=fmt)
    color, target = crt.DeviceArray(np.float32, 3 * n), crt.DeviceArray(np.float32, 3 * n)
    rec = crt.DeviceArray(crt.SHADE_RECORD_DTYPE, n)
    pb.model.forward(pb.scene, pb.rays, pb.hits, color, rec)
    crt.lib().crt_device_sync()
    target.fill_bytes(0)

    def gradients(records):
        g = [crt.DeviceArray(np.float32, k) for k in (3 * pb.roughness.size, pb.roughness.size, pb.intensity.size)]
        for d in g:
            d.fill_bytes(0)
        pb.model.backward(pb.scene, records, color, target, *g)
        crt.lib().crt_device_sync()
        return [d.download() for d in g]

    got = gradients(workloads.DeviceSpan(rec, 0, count))
    host = rec.download()
    assert (host["tri0"] >= 0).mean() > 0.5          # what lies behind the requested records is not empty
    host["tri0"][count:] = -1
    rec.upload(host)
    want = gradients(rec)
    for a, b in zip(got, want):
        # the same terms in another order: at most n additions of 2^-24 relative error each, on the sum of
        # magnitudes, which cancellation between the three channels' residuals leaves within 16 of the largest sum
        assert np.abs(a - b).max() <= 16 * n * 2.0 ** -24 * max(np.abs(b).max(), 1e-30)
