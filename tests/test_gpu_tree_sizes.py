"""Trees at the sizes where a builder changes its way of working: whole
subtrees by one wave up to 64 triangles, tasks of one block up to 2048, chunked
tasks above; trees checked and laid out by one block up to 4096 triangles; equal centroids (median splits) and mixed sizes. Checked on the
copied tree: each triangle in one leaf, conservative boxes, depth-first order
(first child next to its parent), and the reported counts, depth and SAH cost
against a walk in float64; two builds are equal."""
import numpy as np
import pytest

from test_gpu_bvh_sah import _check_tree, _ctx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_mod():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


def _area(lo, hi):
    d = hi.astype(np.float64) - lo.astype(np.float64)
    return float(d[0] * d[1] + d[1] * d[2] + d[2] * d[0])


def _walk(nodes):
    """(leaves, depth, largest leaf, SAH cost) of a copied tree; checks the order of its nodes."""
    refs = nodes[:, 12:14].copy().view(np.int32)
    boxes = [(nodes[:, 0:3], nodes[:, 3:6]), (nodes[:, 6:9], nodes[:, 9:12])]
    leaves, depth, largest, cost, next_node = 0, 0, 0, 0.0, 0
    stack = [(0, 0)]
    while stack:
        i, d = stack.pop()
        assert i == next_node, "nodes are not in depth-first order"
        next_node += 1
        push = []
        for s in range(2):
            a = _area(boxes[s][0][i], boxes[s][1][i])
            r = int(refs[i, s])
            if r >= 0:
                push.append((r, d + 1))
                cost += a
            else:
                n = ((~r) & 15) + 1
                leaves, depth, largest, cost = leaves + 1, max(depth, d + 1), max(largest, n), cost + n * a
        stack.extend(reversed(push))
    assert next_node == len(nodes)
    root = _area(np.minimum(boxes[0][0][0], boxes[1][0][0]), np.maximum(boxes[0][1][0], boxes[1][1][0]))
    return leaves, depth, largest, (cost + root) / root


@pytest.mark.parametrize("builder", ["lbvh", "sah"])
@pytest.mark.parametrize("triangles,alike", [(2, 0), (16, 0), (17, 16), (63, 0), (64, 64), (65, 0), (65, 65), (129, 40),
                                             (700, 0), (2048, 0), (2049, 300), (6000, 0), (4500, 4500)])
def test_tree_sizes(mipt_mod, torch_mod, triangles, alike, builder):
    rng = np.random.default_rng(triangles + alike)
    c = rng.uniform(-8, 8, (triangles, 1, 3)) * np.array([1.0, 0.3, 1.0])
    V = (c + rng.uniform(-0.3, 0.3, (triangles, 3, 3)) * rng.choice([0.05, 1.0, 6.0], (triangles, 1, 1))).astype(np.float32)
    V[:alike] = V[0]
    V = V[rng.permutation(triangles)].reshape(-1, 3)
    scene = mipt_mod.Scene(V, np.arange(3 * triangles, dtype=np.int32).reshape(triangles, 3))
    b = mipt_mod.MIPT_BVH_SAH_BINNED if builder == "sah" else mipt_mod.MIPT_BVH_LBVH
    ctx = _ctx(mipt_mod, scene, b)
    nodes, tris = ctx.read_bvh()
    sizes = _check_tree(scene, nodes, tris)
    leaves, depth, largest, cost = _walk(nodes)
    info = ctx.bvh_info()
    assert (info.leaf_count, info.max_depth, info.max_leaf_size) == (leaves, depth, largest)
    assert info.node_count == len(nodes) == leaves - 1 and sum(sizes) == triangles
    # double sums of the same terms in another order
    assert abs(info.sah_cost - cost) <= 1e-12 * len(nodes) * cost
    ctx.build_bvh(b)
    n2, t2 = ctx.read_bvh()
    assert n2.tobytes() == nodes.tobytes() and t2.tobytes() == tris.tobytes()
    ctx.close()


@pytest.mark.parametrize("builder", ["lbvh", "sah"])
@pytest.mark.parametrize("triangles,size,alike", [(3, 0.01, 0), (4095, 0.01, 0), (4096, 0.01, 0), (4096, 3.0, 0), (4096, 0.01, 4000),
                                                  (4097, 0.01, 0), (4097, 3.0, 900), (30011, 0.01, 0)])
def test_trees_of_one_block(mipt_mod, oracle_mod, torch_mod, triangles, size, alike, builder):
    """Trees around the size that one block checks and collapses, of small triangles (leaves of
    one: levels of more wide nodes than the block has groups), of overlapping ones and of equal
    ones: statistics and order of the binary tree, hits through the wide one."""
    rng = np.random.default_rng(triangles)
    c = rng.uniform(-1, 1, (triangles, 1, 3))
    V = (c + rng.uniform(-size, size, (triangles, 3, 3))).astype(np.float32)
    V[:alike] = V[0]
    V = V.reshape(-1, 3)
    I = np.arange(3 * triangles, dtype=np.int32).reshape(triangles, 3)
    scene = mipt_mod.Scene(V, I)
    ctx = _ctx(mipt_mod, scene, mipt_mod.MIPT_BVH_SAH_BINNED if builder == "sah" else mipt_mod.MIPT_BVH_LBVH)
    nodes, tris = ctx.read_bvh()
    sizes = _check_tree(scene, nodes, tris)
    leaves, depth, largest, cost = _walk(nodes)
    info = ctx.bvh_info()
    assert (info.leaf_count, info.max_depth, info.max_leaf_size) == (leaves, depth, largest)
    assert info.node_count == len(nodes) == leaves - 1 and sum(sizes) == triangles
    assert abs(info.sah_cost - cost) <= 1e-12 * len(nodes) * cost
    n = 2000
    rays = np.zeros(n, mipt_mod.RAY_DTYPE)
    rays["o"] = rng.uniform(-1.2, 1.2, (n, 3))
    d = V[I[rng.integers(0, triangles, n)]].mean(axis=1) - rays["o"]
    rays["d"] = d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)
    rays["last_prim"] = -1
    rays["tmax"] = np.inf
    want = oracle_mod.trace_brute(V, I, rays)
    got = ctx.trace_closest_host(rays)
    assert np.array_equal(got["prim"], want["prim"]) and (got["prim"] >= 0).mean() > 0.5
    assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
    ctx.close()


@pytest.mark.parametrize("builder,triangles,most", [("lbvh", 1000, 1.75), ("lbvh", 5000, 2.75)])
def test_small_builds_are_quick(mipt_mod, torch_mod, scene1, builder, triangles, most):
    """Small trees take few launches and waits. Wall time of a build over that of one triangle's
    (a single block that kept its nodes in scratch memory: 1.9 to 2.0 and 3.0 to 3.3, slower
    than host passes over a copied tree; now 1.4 to 1.5 and 2.0 to 2.15)."""
    import time

    rng = np.random.default_rng(0)

    def wall(count):
        keep = np.sort(rng.choice(scene1.triangle_count, count, replace=False))
        ctx = mipt_mod.Context(0)
        ctx.set_scene(mipt_mod.Scene(scene1.vertices, scene1.indices[keep]))
        times = []
        for _ in range(41):
            t = time.perf_counter()
            ctx.build_bvh(mipt_mod.MIPT_BVH_SAH_BINNED if builder == "sah" else mipt_mod.MIPT_BVH_LBVH)
            times.append(time.perf_counter() - t)
        ctx.close()
        return sorted(times)[20]

    ratio = wall(triangles) / wall(1)
    print(f"{builder} of {triangles} triangles: {ratio:.2f} of one triangle's")
    assert ratio <= most
