"""The traversal on the CPU, over the nodes of the scene builder: waves of 64
rays in lockstep with the device's stack and the slab test's float operations.

* The closest hit is a brute-force loop's bit for bit on scenes that mix
  scales (a small tiled surface near the origin and one triangle far away),
  where a node's rounding errors are larger than the padding of a child near
  the origin.
* Stacks move to private memory when they are full and at no other step, and a
  lane whose LDS part is empty goes on with what it moved without waiting for
  the rest of its wave: its waves take about as many steps as with unbounded
  stacks.  The scenes of the GPU tests that mean to do so do
  leave LDS."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
ROCM = Path("/opt/rocm")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not (ROCM / "include" / "hip").exists(),
                                reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    d = tmp_path_factory.mktemp("replay")
    csrc = ROOT / "violet_amd" / "csrc"
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-pthread", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}",
           f"-I{ROOT / 'include'}", f"-I{csrc}", str(ROOT / "tests" / "host" / "traverse_replay.cpp"),
           str(csrc / "vgi_bvh.cpp"), str(csrc / "vgi_runtime.cpp"), f"-L{ROCM / 'lib'}", "-lamdhip64",
           f"-Wl,-rpath,{ROCM / 'lib'}", "-o", str(d / "traverse_replay")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]

    def run(positions, indices, rays):
        with open(d / "in.bin", "wb") as f:
            f.write(np.array([len(positions), len(indices), len(rays)], np.uint32).tobytes())
            for a, t in ((positions, np.float32), (indices, np.uint32), (rays, np.float32)):
                f.write(np.ascontiguousarray(a, t).tobytes())
        p = subprocess.run([str(d / "traverse_replay"), str(d / "in.bin")], capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, p.stderr
        w = p.stdout.split()
        return dict(zip(w[::2], map(int, w[1::2])))

    return run


def mixed_scale(width, far, axis, n_rays, seed, away=0.0):
    """A square of 16 x 16 tiles of edge width / 16 across `axis` through the
    origin, one triangle about `far` units away, and rays at the square from
    within two widths of it (`away` further back): grazing it, or across it
    along the axes."""
    rng = np.random.default_rng(seed)
    n = 16
    g = np.linspace(-width / 2, width / 2, n + 1)
    u, v = np.meshgrid(g, g, indexing="ij")
    pos = np.stack([u, v, np.zeros_like(u)], -1).reshape(-1, 3)
    i = (np.arange(n)[:, None] * (n + 1) + np.arange(n)).reshape(-1)
    c = np.array([1.0, 0.7, 0.9]) * far
    idx = np.concatenate([np.stack([i, i + n + 1, i + n + 2], 1), np.stack([i, i + n + 2, i + 1], 1),
                          [[len(pos), len(pos) + 1, len(pos) + 2]]])
    pos = np.concatenate([pos, [c, c + [1, 0, 0], c + [0, 1, 0]]])
    target = np.column_stack([rng.uniform(-width / 2, width / 2, (n_rays, 2)), np.zeros(n_rays)])
    phi = rng.uniform(0, 2 * np.pi, n_rays)
    tilt = 10 ** rng.uniform(-4.0, -1.5, n_rays) * rng.choice([-1, 1], n_rays)
    d = np.column_stack([np.cos(phi) * np.cos(tilt), np.sin(phi) * np.cos(tilt), np.sin(tilt)])
    k = n_rays // 8  # straight down onto the square, at tile borders too
    d[:k] = [0, 0, 1]
    target[: k // 2, 0] = rng.choice(g, k // 2)
    o = target - d * (away + 2 * width * rng.uniform(0.2, 1.0, (n_rays, 1)))
    one = np.ones((n_rays, 1))
    rays = np.concatenate([np.roll(o, axis, 1), 5e-4 * one, np.roll(d, axis, 1), (1000.0 + 2 * away) * one], 1)
    return np.roll(pos, axis, 1).astype(np.float32), idx.astype(np.uint32), rays.astype(np.float32)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("width,far", [(1.0, -900.0), (1.0, 300.0), (4.0, -4000.0)])
def test_mixed_scales_lose_no_hit(replay, width, far, axis):
    r = replay(*mixed_scale(width, far, axis, 60000, seed=2))
    assert r["hits"] > 0.99 * r["rays"]
    assert r["lost"] == 0 and r["any"] == 0, r


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_a_thousand_units_away(replay, axis):
    """Rays from far outside, whose errors go with their distance: the outermost planes of a node have
    room for them."""
    r = replay(*mixed_scale(1.0, -900.0, axis, 100000, seed=axis, away=1000.0))
    assert r["hits"] > 0.99 * r["rays"]
    assert r["lost"] == 0 and r["any"] == 0, r


def soup(n, seed):
    rng = np.random.default_rng(seed)
    pos = (rng.uniform(-1.0, 1.0, (n, 1, 3)) + rng.normal(0, 0.4 / n ** (1 / 3), (n, 3, 3))).reshape(-1, 3)
    return pos.astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(n, 3)


def test_only_full_stacks_move(replay):
    """A wave's node steps look into its stacks only when a lane's is full, not whenever one of
    its lanes is done."""
    rng = np.random.default_rng(3)
    m = 6400
    o = rng.uniform(-2.0, 2.0, (m, 3))
    d = rng.uniform(-1.0, 1.0, (m, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([o, np.full((m, 1), 5e-4), d, np.full((m, 1), 1000.0)], 1)
    r = replay(*soup(2000, 7), rays)
    assert r["lost"] == 0 and r["any"] == 0 and r["max_moves"] == 0
    assert r["steps"] > 0 and r["move_steps"] == r["needed_steps"] == 0, r


def piled_rays(m, seed, kind):
    """Rays at a pile of quads over z in [0, 10]: along it from both ends, or from inside in all directions."""
    rng = np.random.default_rng(seed)
    up = rng.random(m) < 0.5
    o = np.column_stack([rng.uniform(-0.5, 0.5, (m, 2)), np.where(up, -1.0, 11.0)])
    d = np.column_stack([rng.normal(0, 0.02, (m, 2)), np.where(up, 1.0, -1.0)])
    if kind == "inside":
        o[:, 2] = rng.uniform(0.0, 10.0, m)
        d = rng.standard_normal((m, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([o, np.full((m, 1), 5e-4), d, np.full((m, 1), 1000.0)], 1)


@pytest.mark.parametrize("kind", ["along", "inside"])
@pytest.mark.parametrize("quads,moves", [(25_000, 1), (200_000, 2)])
def test_deep_stacks_go_on_alone(replay, quads, moves, kind):
    """The piles of test_deep_traversal_stack_spills_exactly and test_stack_leaves_lds_twice."""
    from test_trace_gpu import _onion

    mesh = _onion(quads, 4)
    r = replay(mesh.positions, mesh.indices, piled_rays(256, 8, kind))
    assert r["lost"] == 0 and r["any"] == 0
    assert r["max_entries"] > 14 and r["max_moves"] >= moves, r
    assert r["move_steps"] == r["needed_steps"] > 0
    assert r["steps"] <= 1.1 * r["unbounded_steps"], r
