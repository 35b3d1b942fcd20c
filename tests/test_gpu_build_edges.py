"""The device builder at the edges of its tiles: sort tiles of 2,048 codes and their super-tiles, chunks of 512
leaves, groups of 64 and super-groups of 4,096, all against the host twin byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _soup(n, seed, cells):
    """n small triangles whose centroids take at most `cells` places per axis (few cells: many equal codes)."""
    from candela_amd import scenes
    rng = np.random.default_rng(seed)
    c = rng.integers(0, cells, size=(n, 1, 3)) / max(1, cells - 1) * 100.0
    p = (c + np.array([[0.0, 0.0, 0.0], [0.02, 0.0, 0.01], [0.0, 0.02, -0.01]]) +
         rng.uniform(-1e-4, 1e-4, (n, 3, 3))).astype(np.float32)
    return scenes.make_vertices(p.reshape(-1, 3)), np.arange(3 * n, dtype=np.uint32)


@pytest.mark.parametrize("cells", [2, 40, 100000])
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 66, 255, 256, 257, 258, 511, 512, 513, 514, 1023, 1024, 1025,
                               2047, 2048, 2049, 4095, 4096, 4097,
                               4352, 8191, 32767, 32769, 65537, 262145, 1100001])
def test_build_edges(n, cells):
    import candela_amd as crt
    import oracle
    if cells != 100000 and n > 300000:
        pytest.skip("equal codes are covered at the smaller sizes")
    verts, idx = _soup(n, n + cells, cells)
    b = crt.GpuBVH(verts, idx, None, mesh_id=7, t_offset=11)
    crt.lib().crt_device_sync()
    for d in (b.nodes, b.triangles):
        d.fill_bytes(0xCD)
    b.workspace.fill_bytes(0xEE)          # what the workspace holds does not matter
    b.build()
    crt.lib().crt_device_sync()
    nodes, tris = oracle.build_lbvh(verts, idx, None, 7, 11)
    assert b.nodes.download()[: nodes.size].tobytes() == nodes.tobytes()
    assert b.triangles.download().tobytes() == tris.tobytes()
