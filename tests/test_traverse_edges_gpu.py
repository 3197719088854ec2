"""BVH traversal at the sizes where its bookkeeping can go wrong: waves with
one ray or one ray too many, trees of one leaf, rays with an interval that
starts behind the origin or never ends, ties between coincident triangles,
and stacks that move to private memory and back more than once.  Hits equal
the brute-force loop bit for bit."""
import numpy as np
import pytest

from test_trace_gpu import _gpu_trace, _onion

pytestmark = pytest.mark.gpu


def _soup(n, seed, copies=1):
    """n random triangles, each present `copies` times (coincident: ties go to the lowest id)."""
    from violet_amd import scene

    rng = np.random.default_rng(seed)
    c = rng.uniform(-1.0, 1.0, (n, 1, 3))
    pos = np.tile(c + rng.normal(0, 0.4, (n, 3, 3)), (copies, 1, 1)).reshape(-1, 3).astype(np.float32)
    m = n * copies
    return scene.Mesh(positions=pos, normals=np.tile(np.array([0, 0, 1], np.float32), (3 * m, 1)),
                      indices=np.arange(3 * m, dtype=np.uint32).reshape(m, 3), tri_material=np.zeros(m, np.uint32),
                      albedo=np.full((1, 3), 0.5), metallic=np.zeros(1), roughness=np.full(1, 0.5))


def _check(vgi, mesh, rays):
    import oracle
    from violet_amd import scene

    sc = scene.Scene(mesh)
    g_thv, g_id = _gpu_trace(sc, rays, False)
    o_thv, o_id = oracle.trace(32, mesh.positions, mesh.indices, rays, brute=True)
    assert np.array_equal(g_id, o_id), f"hit ids differ on {np.mean(g_id != o_id):.3%} of rays"
    hit = g_id != 0xFFFFFFFF
    assert np.array_equal(g_thv[hit].view(np.uint32), o_thv[hit].astype(np.float32).view(np.uint32))
    assert np.array_equal(_gpu_trace(sc, rays, True)[1] != 0xFFFFFFFF, hit)
    return hit


@pytest.mark.parametrize("n_rays", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("n_tris,copies", [(1, 1), (2, 1), (5, 1), (3, 6), (300, 2)])
@pytest.mark.parametrize("interval", [(5e-4, 1000.0), (-3.0, 1000.0), (0.0, np.inf), (0.5, 1.5)])
def test_edges(vgi, n_tris, copies, n_rays, interval):
    rng = np.random.default_rng(n_tris + n_rays)
    mesh = _soup(n_tris, 3, copies)
    o = rng.uniform(-2.0, 2.0, (n_rays, 3))
    d = rng.uniform(-1.0, 1.0, (n_rays, 3)) - o
    # every other ray from one unit off a triangle's middle, about along its normal: a sure hit in all intervals
    aimed = np.arange(n_rays) % 2 == 0
    tri = mesh.positions[mesh.indices[rng.integers(0, len(mesh.indices), n_rays)]].astype(np.float64)
    normal = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    normal /= np.linalg.norm(normal, axis=1, keepdims=True)
    d[aimed] = (normal * rng.choice([-1, 1], (n_rays, 1)) + rng.uniform(-0.3, 0.3, (n_rays, 3)))[aimed]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o[aimed] = (tri.mean(1) - d)[aimed]
    one = np.ones((n_rays, 1))
    rays = np.concatenate([o, interval[0] * one, d, interval[1] * one], 1).astype(np.float32)
    assert _check(vgi, mesh, rays)[aimed].all()


def test_stack_leaves_lds_twice(vgi):
    """200,000 stacked quads: every box on a ray's way is hit, three children
    stay on the stack per level, about 30 entries: two moves of eight
    (test_traverse_replay.py checks that there are as many)."""
    rng = np.random.default_rng(8)
    m = 256
    o = np.column_stack([rng.uniform(-0.5, 0.5, (m, 2)), np.where(rng.random(m) < 0.5, -1.0, 11.0)])
    d = np.column_stack([rng.normal(0, 0.02, (m, 2)), np.where(o[:, 2] < 0, 1.0, -1.0)])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([o, np.full((m, 1), 5e-4), d, np.full((m, 1), 1000.0)], 1).astype(np.float32)
    assert _check(vgi, _onion(200_000, 4), rays).all()
    # any hit from inside the pile: early exits while entries wait in private memory
    rays[:, 2] = rng.uniform(0.0, 10.0, m)
    _check(vgi, _onion(200_000, 4), rays)


@pytest.mark.parametrize("n_tris", [16384, 16385, 40000])
def test_scene_built_in_pieces(vgi, n_tris):
    """Scenes at and past the size from which subtrees are built apart and put together."""
    rng = np.random.default_rng(n_tris)
    m = 300
    o = rng.uniform(-2.0, 2.0, (m, 3))
    d = rng.uniform(-1.0, 1.0, (m, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([o, np.full((m, 1), 5e-4), d, np.full((m, 1), 1000.0)], 1).astype(np.float32)
    assert _check(vgi, _soup(n_tris, 5), rays).any()


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("width,far", [(1.0, -900.0), (4.0, -4000.0)])
def test_mixed_scales_lose_no_hit(vgi, width, far, axis):
    """A small tiled surface at the edge of a node that spans a far triangle: the node's
    rounding exceeds the surface's own padding, and the node's margin covers it."""
    from test_traverse_replay import mixed_scale

    from violet_amd import scene

    pos, idx, rays = mixed_scale(width, far, axis, 60000, seed=2)
    mesh = scene.Mesh(positions=pos, normals=np.tile(np.array([0, 0, 1], np.float32), (len(pos), 1)), indices=idx,
                      tri_material=np.zeros(len(idx), np.uint32), albedo=np.full((1, 3), 0.5), metallic=np.zeros(1),
                      roughness=np.full(1, 0.5))
    assert _check(vgi, mesh, rays).mean() > 0.99
