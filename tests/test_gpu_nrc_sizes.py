"""The radiance cache's kernels at the sizes where they change their way of
working.

- Inference: a row's answer does not depend on the rows beside it, so row
  counts around a wave's 64 rows and a block's 256 give the same bits as one
  large call.
- Encoded rows: one launch up to 49,152 rows, planes and a copy past it; the same bits.
- Grid and weight gradients: from 4096 rows on (16 levels; 15,360 with one) the corner
  updates are binned, below they are added by atomics. A batch's gradient is the row-weighted mean
  of its halves' (the terms are the same 32-bit products, up to the scale
  1 / (3 rows) and the order of the sums): with at most 2^17 addends of random
  sign per entry the two agree to 1e-5 in the 2-norm.
"""
import numpy as np
import pytest

from test_gpu_nrc import _infer, _make, _queries, _randomize_grid

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_mod():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    return torch


@pytest.mark.parametrize("levels", [1, 7, 16])
def test_rows_are_independent(mipt_mod, torch_mod, scene1, levels):
    rng = np.random.default_rng(levels)
    ctx, cs = _make(mipt_mod, scene1, grid_levels=levels, grid_log2_table=13)
    _randomize_grid(ctx, cs, rng)
    q = _queries(rng, scene1, 70001)
    want = _infer(mipt_mod, torch_mod, ctx, q)
    assert np.isfinite(want).all() and (want[:, 3] == 0.0).all()
    for n in (1, 2, 63, 64, 65, 255, 256, 257, 4097, 49153):
        assert _infer(mipt_mod, torch_mod, ctx, q[:n]).tobytes() == want[:n].tobytes(), n
    ctx.close()


@pytest.mark.parametrize("offset", [1, 2, 3])
def test_output_rows_at_any_float(mipt_mod, torch_mod, scene1, offset):
    """Rows of an array of floats that does not begin at a multiple of 16 bytes."""
    rng = np.random.default_rng(offset)
    ctx, cs = _make(mipt_mod, scene1, grid_levels=16, grid_log2_table=13)
    _randomize_grid(ctx, cs, rng)
    n = 1003
    d_q = mipt_mod.to_device(_queries(rng, scene1, n))
    want = torch_mod.empty(4 * n, device="cuda")
    ctx.cache_infer(d_q, n, want)
    buf = torch_mod.full((4 * n + 8,), -7.0, device="cuda")
    ctx.cache_infer(d_q, n, buf[offset:])
    assert torch_mod.equal(buf[offset:offset + 4 * n], want)
    assert (buf[:offset] == -7.0).all() and (buf[offset + 4 * n:] == -7.0).all()
    ctx.close()


@pytest.mark.parametrize("levels", [1, 7, 8, 9, 16])
def test_encoded_rows_are_independent(mipt_mod, torch_mod, scene1, levels):
    rng = np.random.default_rng(levels)
    ctx, cs = _make(mipt_mod, scene1, grid_levels=levels, grid_log2_table=13)
    _randomize_grid(ctx, cs, rng)
    n = 49153
    d_q = mipt_mod.to_device(_queries(rng, scene1, n))
    want = torch_mod.empty(n, 64, dtype=torch_mod.int16, device="cuda")
    ctx.cache_encode(d_q, n, want)
    assert (want[:, 2 * levels + 28:] == 0).all()
    for k in (1, 2, 255, 256, 257, 16385, 49152):
        got = torch_mod.full((k + 1, 64), -1, dtype=torch_mod.int16, device="cuda")
        ctx.cache_encode(d_q, k, got)
        assert torch_mod.equal(got[:k], want[:k]), k
        assert (got[k] == -1).all(), "written past the last row"
    ctx.close()


FEW_LEVELS = [(4827, 7, 14), (7168, 3, 21), (15360, 1, 10)]  # the first binned batch of 7, 3 and 1 levels


@pytest.mark.parametrize("rows,levels,log2_table", [(r, *c) for c in [(16, 4), (16, 7), (16, 9), (16, 10), (7, 14), (16, 15), (16, 19), (3, 21)]
                                                    for r in (4096, 4097, 6000)] + FEW_LEVELS)
def test_binned_gradient_is_the_mean_of_its_halves(mipt_mod, torch_mod, scene1, rows, levels, log2_table):
    rng = np.random.default_rng(rows + log2_table)
    ctx, cs = _make(mipt_mod, scene1, grid_levels=levels, grid_log2_table=log2_table)
    _randomize_grid(ctx, cs, rng)
    q = _queries(rng, scene1, rows)
    q[: rows // 3, 0:3] = q[0, 0:3]  # many rows in one cell: full bins, shares of a bin
    y = np.zeros((rows, 4), np.float32)
    y[:, :3] = rng.uniform(0.0, 2.0, (rows, 3))
    a = rows // 2

    def grad(lo, hi):
        return ctx.cache_gradients(mipt_mod.to_device(q[lo:hi]), mipt_mod.to_device(y[lo:hi]), hi - lo)

    whole, first, second = grad(0, rows), grad(0, a), grad(a, rows)
    for g, g1, g2 in zip(whole[:2], first[:2], second[:2]):
        want = (g1.astype(np.float64) * a + g2.astype(np.float64) * (rows - a)) / rows
        assert np.linalg.norm(want) > 0.0
        assert np.linalg.norm(g - want) <= 1e-5 * np.linalg.norm(want)
    ctx.close()


@pytest.mark.parametrize("rows", [65536, 65537, 140000])
def test_binned_gradient_in_passes(mipt_mod, torch_mod, scene1, rows):
    """More rows than are binned at a time (2^16)."""
    rng = np.random.default_rng(rows)
    ctx, cs = _make(mipt_mod, scene1, grid_log2_table=14, batch_size=1 << 18)
    _randomize_grid(ctx, cs, rng)
    q = _queries(rng, scene1, rows)
    y = np.zeros((rows, 4), np.float32)
    y[:, :3] = rng.uniform(0.0, 2.0, (rows, 3))
    d_q, d_y = mipt_mod.to_device(q), mipt_mod.to_device(y)
    whole = ctx.cache_gradients(d_q, d_y, rows)
    total = None
    for lo in range(0, rows, 4000):
        n = min(4000, rows - lo)
        g = ctx.cache_gradients(mipt_mod.to_device(q[lo:lo + n]), mipt_mod.to_device(y[lo:lo + n]), n)
        part = [x.astype(np.float64) * n for x in g[:2]]
        total = part if total is None else [t + x for t, x in zip(total, part)]
    for g, t in zip(whole[:2], total):
        assert np.linalg.norm(g - t / rows) <= 1e-5 * np.linalg.norm(t / rows)
    ctx.close()
