"""The shading adjoint over record counts that are no whole number of its 64-pixel tiles.

The records behind the requested ones are valid pixels of the same image, so a lane past the end that read its
record would add that pixel's gradient (and stay in bounds).  The expected gradients are those of the same call over
the whole buffer with every record behind the requested ones marked as a miss.
"""
import numpy as np
import pytest

from shade_terms import order_bounds

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
    # the same terms in another order; an element that none of the requested records adds to stays exactly 0
    bounds = order_bounds(pb.model, host, color.download(), target.download())
    for a, b, bound in zip(got, want, bounds):
        assert (np.abs(a.astype(np.float64) - b) <= bound).all()
        assert not a[bound == 0].any() and not b[bound == 0].any()
    assert (bounds[1] == 0).any()
