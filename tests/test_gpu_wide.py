"""The 6-wide traversal tree (csrc/bvh_wide.hip) and the ray batches of its
kernel at the sizes where they can go wrong, hits bit-exact against the
oracle's brute-force loop:
- triangle counts around a node's six children, a leaf's sixteen triangles
  and the fifteen a leaf may be offset by, distinct and all alike (median
  splits: full leaves side by side, merged into one);
- ray counts around a batch (8 to 64 rays a wave) and a wave;
- rays that start far away (their box intervals widen past whole nodes),
  that lie in the planes of boxes, and with infinite or NaN components (always
  a miss).
"""
import numpy as np
import pytest

from test_gpu_bvh_sah import _assert_hits_equal, _ctx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_mod():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


def _rays(mipt_mod, rng, n, V, I):
    """Random rays towards random triangles, some from far away, some axis-aligned
    from a vertex's height, some not finite."""
    rays = np.zeros(n, mipt_mod.RAY_DTYPE)
    tri = V[I[rng.integers(0, I.shape[0], n)]]
    target = tri.mean(axis=1)
    kind = rng.integers(0, 8, n)
    scale = np.where(kind == 0, 1.0e5, 2.0)[:, None]
    o = target + rng.normal(size=(n, 3)) * scale
    flat = kind == 1
    o[flat, 1:] = tri[flat, 0, 1:]
    rays["o"] = o.astype(np.float32)
    d = target - rays["o"]
    rays["d"] = (d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)).astype(np.float32)
    rays["d"][flat] = [1, 0, 0]
    rays["last_prim"] = np.where(kind == 2, rng.integers(0, I.shape[0], n), -1)
    rays["tmax"] = np.where(kind == 3, rng.uniform(0.0, 4.0, n), np.inf)
    bad = np.nonzero(kind == 4)[0]
    for j in bad:
        rays[rng.choice(["o", "d"])][j, rng.integers(0, 3)] = rng.choice([np.nan, np.inf, -np.inf])
    rays["tmax"][kind == 5] = rng.choice([-1.0, 0.0, np.nan])
    return rays


@pytest.mark.parametrize("builder", ["lbvh", "sah"])
@pytest.mark.parametrize("alike", [False, True])
@pytest.mark.parametrize("triangles", [1, 2, 5, 6, 7, 12, 13, 16, 17, 31, 32, 33, 64, 97, 515])
def test_wide_tree(mipt_mod, oracle_mod, torch_mod, triangles, alike, builder):
    rng = np.random.default_rng(triangles)
    if alike:
        V = np.tile(np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.5]], np.float32), (triangles, 1))
    else:
        c = rng.uniform(-4, 4, (triangles, 1, 3))
        V = (c + rng.uniform(-0.6, 0.6, (triangles, 3, 3))).astype(np.float32).reshape(-1, 3)
    I = np.arange(3 * triangles, dtype=np.int32).reshape(triangles, 3)
    ctx = _ctx(mipt_mod, mipt_mod.Scene(V, I),
               mipt_mod.MIPT_BVH_SAH_BINNED if builder == "sah" else mipt_mod.MIPT_BVH_LBVH)
    for n in (1, 8, 9, 64, 65, 2000):
        rays = _rays(mipt_mod, rng, n, V, I)
        with np.errstate(all="ignore"):
            want = oracle_mod.trace_brute(V, I, rays)
        got = ctx.trace_closest_host(rays)
        _assert_hits_equal(got, want)
        assert np.array_equal(ctx.trace_any_host(rays).astype(bool), want["prim"] >= 0)
    ctx.close()


@pytest.mark.parametrize("block,stack", [(64, 8), (128, 16), (256, 32)])
@pytest.mark.parametrize("n", [7, 8, 2047, 16385, 131073, 400001])
def test_ray_batches(mipt_mod, oracle_mod, torch_mod, scene1, n, block, stack):
    """Ray counts on both sides of the rules that deal rays to waves: every
    ray's hit is the same as in one large launch (each is checked there)."""
    ctx = _ctx(mipt_mod, scene1, mipt_mod.MIPT_BVH_SAH_BINNED)
    rng = np.random.default_rng(3)
    rays = np.zeros(400001, mipt_mod.RAY_DTYPE)
    rays["o"] = rng.uniform(-0.9, 0.9, (rays.size, 3))
    d = rng.normal(size=(rays.size, 3))
    rays["d"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    rays["last_prim"] = -1
    rays["tmax"] = np.inf
    want = ctx.trace_closest_host(rays)
    some = rng.integers(0, rays.size, 200)
    _assert_hits_equal(want[some], oracle_mod.trace_brute(scene1.vertices, scene1.indices, rays[some]))
    ctx.set_trace_config(block, stack)
    _assert_hits_equal(ctx.trace_closest_host(rays[:n]), want[:n])
    ctx.close()


@pytest.mark.parametrize("crowd", [False, True])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 17, 63, 64, 129])
def test_last_rays(mipt_mod, oracle_mod, torch_mod, n, crowd):
    """The rays that eight lanes share: slivers through one point, whose boxes
    all overlap (stacks past the LDS entries, in the columns of the lanes that
    the rays began in), alone in their waves and as the rest of larger batches
    (`crowd`: the others miss at once); with the triangle that each hits
    excluded, so that the next one of its leaf counts."""
    rng = np.random.default_rng(n)
    k = 3000
    d = rng.normal(size=(k, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    off = rng.normal(size=(k, 3)) * 0.02
    V = np.stack([-3 * d + off, 3 * d + off, 3 * d - off + rng.normal(size=(k, 3)) * 0.05], 1).astype(np.float32)
    V = V.reshape(-1, 3)
    I = np.arange(3 * k, dtype=np.int32).reshape(k, 3)
    ctx = _ctx(mipt_mod, mipt_mod.Scene(V, I), mipt_mod.MIPT_BVH_SAH_BINNED)
    rays = np.zeros(n, mipt_mod.RAY_DTYPE)
    o = rng.normal(size=(n, 3))
    o = (4 * o / np.linalg.norm(o, axis=1, keepdims=True)).astype(np.float32)
    aim = rng.normal(size=(n, 3)) * 0.3 - o
    rays["o"] = o
    rays["d"] = (aim / np.linalg.norm(aim, axis=1, keepdims=True)).astype(np.float32)
    rays["last_prim"] = -1
    rays["tmax"] = np.inf
    rays["last_prim"] = oracle_mod.trace_brute(V, I, rays)["prim"]
    want = oracle_mod.trace_brute(V, I, rays)
    at = np.arange(n)
    if crowd:
        many = np.zeros(40 * n, mipt_mod.RAY_DTYPE)
        many["o"] = (50, 50, 50)
        many["d"] = (1, 0, 0)
        many["last_prim"] = -1
        many["tmax"] = np.inf
        at = np.sort(rng.choice(many.size, n, replace=False))
        many[at] = rays
        rays = many
    got = ctx.trace_closest_host(rays)
    _assert_hits_equal(got[at], want)
    assert np.all(np.delete(got["prim"], at) == -1)
    assert np.array_equal(ctx.trace_any_host(rays)[at].astype(bool), want["prim"] >= 0)
    ctx.close()
