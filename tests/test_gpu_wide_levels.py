"""The device collapse's level passes at their edges: levels of one workgroup and of several, of more workgroups than
are launched, trees of few and of many levels, both widths, against crt_wide_build's layout renumbered breadth-first."""
import numpy as np
import pytest

from test_gpu_build import _bfs_renumber

pytestmark = pytest.mark.gpu


def _soup(n, seed, same):
    from candela_amd import scenes
    rng = np.random.default_rng(seed)
    c = np.zeros((n, 1, 3)) if same else rng.uniform(-50, 50, size=(n, 1, 3))
    d = np.array([[0.0, 0.0, 0.0], [0.3, 0.0, 0.1], [0.0, 0.2, -0.1]])
    p = (c + (d if same else rng.normal(scale=0.3, size=(n, 3, 3)))).astype(np.float32)
    return scenes.make_vertices(p.reshape(-1, 3)), np.arange(3 * n, dtype=np.uint32)


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("n,same", [(2, False), (3, False), (4, False), (5, True), (37, False), (129, True), (400, False),
                                    (900, False), (2500, True), (9000, False), (330000, False)])
def test_levels_match_host_collapse(n, same, width):
    import candela_amd as crt
    import oracle
    verts, idx = _soup(n, n, same)
    b = crt.GpuBVH(verts, idx)
    a = crt.GpuWide(b, width, max_levels=48)
    crt.lib().crt_device_sync()
    a.workspace.fill_bytes(0x5A)          # what the workspace holds does not matter
    a.groups.fill_bytes(0xCD)
    a.build()
    total, status = a.result()
    assert status == 0
    nodes, tris = b.nodes.download()[: n - 1], b.triangles.download()
    h = crt.wide_build(1, nodes, tris, verts, oracle.identity_entity(nodes.size), width, 2)
    ref, reached = _bfs_renumber(h.groups, width, int(h.entities["node_offset"][0]))
    assert total == reached == h.stats["node_count"]
    assert a.groups.download()[: total * (width // 4)].tobytes() == ref.tobytes()
    rec = a.records.download()
    assert rec.tobytes() == h.records.tobytes()
    depth = a.levels
    for levels in {1, max(1, depth - 1), max(1, depth), depth + 1}:     # a budget that ends the passes early says so
        w = crt.GpuWide(b, width, max_levels=levels)
        got, st = w.result()
        assert st == (0 if levels >= depth else crt.WIDE_GPU_TOO_DEEP), (levels, depth)
        assert got == total or levels < depth
