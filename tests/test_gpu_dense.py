"""Dense SwiGLU FFN of the first layers (MLP::forward_gpu, layer.cu:1231-1269)
through the C-ABI (moe_dense_*), against the oracle's restatement.

Bar: y within rtol 1e-3 / atol 1e-4 in fp32.  The HIP path cuts the
intermediate dimension into 4 chunks and adds their partial down-projections,
so its k-sums are ordered differently from the reference's single chains;
only the tolerance is expected, not bit equality.
"""
import sys

import numpy as np
import pytest

RTOL, ATOL = 1e-3, 1e-4
H, I = 2048, 7168


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def dense_weights():
    rng = np.random.default_rng(2024)
    w1 = rng.standard_normal((I, H), dtype=np.float32) * np.float32(0.02)
    w3 = rng.standard_normal((I, H), dtype=np.float32) * np.float32(0.02)
    w2 = rng.standard_normal((H, I), dtype=np.float32) * np.float32(0.02)
    return w1, w3, w2


@pytest.fixture(scope="module")
def mlp(dense_weights):
    from final_amd import DenseMLP
    m = DenseMLP(H, I, max_tokens=2048)
    m.set_weights(*dense_weights)
    yield m
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 8, 31, 32, 48, 64, 100, 150, 192, 256, 1000, 2048])
def test_dense_matches_oracle(T, mlp, dense_weights, oracle_mod):
    from final_amd import workloads as W
    say(f"[dense] T={T} plan={mlp.plan(T)}")
    if T <= 192:
        # K-split tiles on the 4 chunks of 1792
        assert mlp.plan(T) == 0
    x = W.gen_x(T, seed=31)
    y = mlp.forward(x)
    ref = oracle_mod.dense_mlp(x, *dense_weights)
    np.testing.assert_allclose(y, ref, rtol=RTOL, atol=ATOL)


@pytest.mark.gpu
def test_dense_residual_in_place(mlp, dense_weights, oracle_mod):
    from final_amd import hip
    from final_amd import workloads as W
    T = 40
    x = W.gen_x(T, seed=32)
    r = W.gen_x(T, seed=33)
    ref = oracle_mod.dense_mlp(x, *dense_weights, residual=r)
    dx = hip.DeviceArray.from_numpy(x)
    dr = hip.DeviceArray.from_numpy(r)
    mlp.forward_gpu(dx, dr, T, residual=dr)
    hip.synchronize()
    mlp.check_device()
    np.testing.assert_allclose(dr.download(), ref, rtol=RTOL, atol=ATOL)


# Edges of the K-split tiles that serve up to 192 tokens: 16-, 32- and 48-row
# gate/up tiles, one and two column blocks in the down tiles.
@pytest.mark.gpu
@pytest.mark.parametrize("T", [2, 15, 16, 17, 33, 37, 47, 49, 65, 97, 191])
def test_dense_few_tokens_edges(T, mlp, dense_weights, oracle_mod):
    from final_amd import _native, hip
    from final_amd import workloads as W
    say(f"[dense edges] T={T}")
    x, r = W.gen_x(T, seed=T), W.gen_x(T, seed=T + 1)
    dx, dr, dy = (hip.DeviceArray.from_numpy(a) for a in (x, r, np.zeros_like(x)))
    mlp.forward_gpu(dx, dy, T, residual=dr)
    hip.synchronize()
    ref = oracle_mod.dense_mlp(x, *dense_weights, residual=r)
    np.testing.assert_allclose(dy.download(), ref, rtol=RTOL, atol=ATOL)
    # the fixed routing a forward reports, whichever kernels it ran
    idx, w, counts = np.empty((T, 4), np.int32), np.empty((T, 4), np.float32), np.empty(32, np.int32)
    rc = _native.lib().moe_last_routing(mlp._ctx, idx.ctypes.data, w.ctypes.data, counts.ctypes.data,
                                        None, T, None)
    assert rc == 0
    assert (idx == np.arange(4)).all() and (w == 1.0).all()
    assert (counts[:4] == T).all() and not counts[4:].any()


@pytest.mark.gpu
def test_dense_nonfinite_rows(mlp, dense_weights):
    """Infinities and NaN stay in their rows, to the last bit of the others."""
    from final_amd import hip
    from final_amd import workloads as W
    for T in (20, 300, 700):
        x = W.gen_x(T, seed=5)
        y0 = mlp.forward(x)
        x[3, 7], x[11, 0] = np.inf, np.nan
        y = mlp.forward(x)
        assert not np.isfinite(y[3]).any() and np.isnan(y[11]).all()
        keep = np.setdiff1d(np.arange(T), [3, 11])
        np.testing.assert_array_equal(y[keep].view(np.uint32), y0[keep].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("h,i", [(256, 1024), (512, 3072), (1024, 1024), (2304, 6144)])
def test_dense_other_shapes(h, i, oracle_mod):
    """K-split tiles for few tokens whatever the shape, against the oracle and the 64-row plan."""
    from final_amd import DenseMLP, _native
    r = np.random.default_rng(h + i)
    w = [np.float32(0.04) * r.standard_normal(s, dtype=np.float32) for s in ((i, h), (i, h), (h, i))]
    m = DenseMLP(h, i, max_tokens=200)
    try:
        m.set_weights(*w)
        for T in (1, 16, 17, 33, 48, 65, 192):
            say(f"[dense shapes] {h} x {i} T={T}")
            x = r.standard_normal((T, h), dtype=np.float32)
            assert m.plan(T) == 0 and m.plan(193) == 64
            y = m.forward(x)
            assert _native.lib().moe_force_tile_rows(m._ctx, 64) == 0
            y64 = m.forward(x)
            assert _native.lib().moe_force_tile_rows(m._ctx, -1) == 0
            np.testing.assert_allclose(y, oracle_mod.dense_mlp(x, *w), rtol=RTOL, atol=ATOL)
            np.testing.assert_allclose(y, y64, rtol=RTOL, atol=ATOL)
        # compiled for no such shape: the forced streaming plan stays refused
        assert _native.lib().moe_force_tile_rows(m._ctx, 0) != 0
    finally:
        m.close()


@pytest.mark.gpu
def test_dense_plan_by_work():
    from final_amd import DenseMLP
    m = DenseMLP(4096, 16384, max_tokens=64)
    assert [m.plan(T) for T in (1, 42, 43, 64)] == [0, 0, 64, 64]
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [100, 300, 700])
def test_dense_small_inputs(T):
    """Inputs near the smallest normal value against weights that undo them: as the same block unscaled."""
    from final_amd import DenseMLP
    h, i = 256, 1024
    r = np.random.default_rng(T)
    w = [np.float32(0.05) * r.standard_normal(s, dtype=np.float32) for s in ((i, h), (i, h), (h, i))]
    x = r.uniform(1.0, 2.0, (T, h)).astype(np.float32)
    ys = []
    for e in (0, 124):
        m = DenseMLP(h, i, max_tokens=T)
        m.set_weights(np.ldexp(w[0], e), np.ldexp(w[1], e), w[2])
        ys.append(m.forward(np.ldexp(x, -e)))
        m.close()
    # every product is the same number on both sides; each side's sums take at
    # most h and i roundings of 2^-24, those of gate and up carried through the
    # product and the down rows: (2 h + i) 2^-24 in the norm, and far less when
    # roundings cancel, as they do for all but a constant sign
    assert np.linalg.norm(ys[1] - ys[0]) <= 2 * (2 * h + i) * 2.0 ** -24 / np.sqrt(h) * np.linalg.norm(ys[0])


@pytest.mark.gpu
def test_dense_context_rejects_moe_calls(mlp):
    from final_amd import _native
    L = _native.lib()
    assert L.moe_forward(mlp._ctx, None, None, None, 1, None) == _native.MOE_ERR_INVALID_ARG
    assert L.moe_route(mlp._ctx, None, 1, None) == _native.MOE_ERR_INVALID_ARG
    assert L.moe_dense_forward(mlp._ctx, None, None, None, 0, None) == 0  # T = 0: no-op
