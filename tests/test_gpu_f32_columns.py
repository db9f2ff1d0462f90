"""Several f32 columns, staged in LDS or read from global memory, and one column of short
matrices whose workgroups add waves that only stage.

The bar is the GEMVs' (1e-5 relative L2 against the f64 product of the
oracle's decode): f32 x is split into hi + lo f16 (22 bits), products are
exact, the sums f32.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TIGHT = 1e-5


def rel_l2(got, want):
    return float(np.linalg.norm(np.asarray(got, np.float64) - want) / max(np.linalg.norm(want), 1e-300))


def gemv(sm, dev, data, x, rows, accumulate=None):
    import torch
    dc = sm.DeviceContainer(data)
    y = torch.full((x.shape[0], rows), float("nan") if accumulate is None else accumulate, device=dev)
    dc.gemv(torch.from_numpy(x).to(dev), y, ncols=x.shape[0], accumulate=accumulate is not None)
    torch.cuda.synchronize()
    return y.cpu().numpy()


# (rows, cols, columns, codebook): units of 2, 4, 5 and 10 steps, 13-bit
# indices, the widest call, ragged rows, a K (9 steps) that keeps the staged
# ring kernel, and two whose 2-step units would take several rounds of workgroups
F32_COLUMNS = [(6160, 2560, 8, 4096), (300, 2560, 16, 4096), (2560, 10240, 5, 4096), (33, 2560, 8, 4096), (24, 256, 2, 4096), (40, 10240, 16, 4096),
               (64, 4096, 3, 4096), (48, 4096, 8, 8192), (130, 2560, 7, 4096), (57, 1152, 4, 4096),
               (5400, 3328, 3, 4096), (5744, 2816, 8, 4096), (504, 2304, 4, 4096)]


@pytest.mark.parametrize("rows,cols,ncol,nc", F32_COLUMNS)
def test_f32_columns_against_oracle(sm, ref, dev, rows, cols, ncol, nc):
    data = sm.synth_container(rows + ncol, rows, cols, 4, nc, 2, 1)
    W = ref.decode(data).astype(np.float64)
    x = np.random.default_rng(cols + ncol).standard_normal((ncol, cols)).astype(np.float32)
    want = x.astype(np.float64) @ W.T
    got = gemv(sm, dev, data, x, rows)
    for n in range(ncol):
        assert rel_l2(got[n], want[n]) <= TIGHT, n
    assert np.array_equal(got, gemv(sm, dev, data, x, rows))
    assert rel_l2(gemv(sm, dev, data, x, rows, accumulate=2.0), want + 2.0) <= TIGHT


@pytest.mark.parametrize("scale", [-140, -30, -12, 12, 20, 100])
@pytest.mark.parametrize("cols", [2560, 10240], ids=["staged", "global"])
def test_f32_columns_out_of_f16_range(sm, ref, dev, scale, cols):
    """All columns scaled far out of f16's range, or, where x is read from
    global memory (whose range is checked per column), one of them."""
    rows, ncol = 64, 4
    data = sm.synth_container(5, rows, cols)
    W = ref.decode(data).astype(np.float64)
    x0 = np.random.default_rng(3).standard_normal((ncol, cols)).astype(np.float32)
    for which in (slice(0, ncol), slice(2, 3))[:1 if cols == 2560 else 2]:
        x = x0.copy()
        x[which] = np.ldexp(x[which], scale)
        got = gemv(sm, dev, data, x, rows)
        for n in range(ncol):
            want = x[n].astype(np.float64) @ W.T
            # x of 2^-140 holds 9 bits and y its own last bits only
            assert rel_l2(got[n], want) <= (2.0 ** -6 if scale < -126 and (which.start <= n < which.stop) else TIGHT), n


@pytest.mark.parametrize("cols", [2560, 10240], ids=["staged", "global"])
def test_f32_columns_spike_and_non_finite(sm, ref, dev, cols):
    rows, ncol = 33, 5
    data = sm.synth_container(6, rows, cols)
    W = ref.decode(data).astype(np.float64)
    x = np.random.default_rng(4).standard_normal((ncol, cols)).astype(np.float32)
    x[0, 7] = 3.0e5
    x[1, 9] = np.inf
    x[2, 1000] = np.nan
    x[3] = 0.0
    got = gemv(sm, dev, data, x, rows)
    assert rel_l2(got[0], x[0].astype(np.float64) @ W.T) <= TIGHT
    assert not np.isfinite(got[1][W[:, 9] != 0]).any() and np.isnan(got[2]).all()
    assert np.array_equal(got[3], np.zeros(rows, np.float32))
    assert rel_l2(got[4], x[4].astype(np.float64) @ W.T) <= TIGHT


@pytest.mark.parametrize("f32", [False, True], ids=["bf16x", "f32x"])
@pytest.mark.parametrize("rows,cols,nc", [(1024, 2560, 4096), (8, 256, 4096), (520, 10240, 4096), (16, 10240, 4096),
                                          (1024, 4096, 4096), (600, 1152, 4096), (300, 8192, 8192), (40, 2560, 4094),
                                          (64, 2560, 1 << 12), (2304, 2304, 4096), (600, 1792, 4096), (70, 1152, 4096), (96, 1152, 8192),
                                          (4300, 9856, 4096), (1984, 2688, 8192)])
def test_one_column_of_a_short_matrix(sm, ref, dev, rows, cols, nc, f32):
    import torch
    data = sm.synth_container(rows + cols, rows, cols, 4, nc, 2, 1)
    W = ref.decode(data).astype(np.float64)
    xt = torch.from_numpy(np.random.default_rng(cols).standard_normal((1, cols)).astype(np.float32)).to(dev)
    xt = xt if f32 else xt.to(torch.bfloat16)
    y = torch.full((1, rows), float("nan"), device=dev)
    sm.DeviceContainer(data).gemv(xt, y)
    torch.cuda.synchronize()
    assert rel_l2(y[0].cpu().numpy(), W @ xt[0].double().cpu().numpy()) <= TIGHT


def launches(stream, call):
    """Kernels that call() puts on the stream, from a capture of it."""
    import ctypes
    hip, graph, n = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p(), ctypes.c_size_t()
    at = ctypes.c_void_p(stream.cuda_stream)
    assert hip.hipStreamBeginCapture(at, ctypes.c_int(2)) == 0
    try:
        call()
    finally:
        assert hip.hipStreamEndCapture(at, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return n.value


@pytest.mark.parametrize("rows", [40, 300, 1024])
@pytest.mark.parametrize("cols,want", [(5376, 1), (5504, 1), (6144, 1), (6656, 1), (6784, 2), (7552, 2), (7680, 2)])
def test_waves_that_stage_leave_x_its_room(sm, ref, dev, rows, cols, want):
    """Two 13-bit codebooks fill 128 of 160 KB of LDS: one f32 column stays one
    launch, with the staging waves that fit beside it, unless few do and units are long."""
    import torch
    data = sm.synth_container(rows + cols, rows, cols, 4, 8192, 2, 1)
    x = torch.from_numpy(np.random.default_rng(cols).standard_normal((1, cols)).astype(np.float32)).to(dev)
    dc, y, stream = sm.DeviceContainer(data), torch.full((1, rows), float("nan"), device=dev), torch.cuda.Stream()
    dc.gemv(x, y)
    torch.cuda.synchronize()
    assert rel_l2(y[0].cpu().numpy(), ref.decode(data).astype(np.float64) @ x[0].double().cpu().numpy()) <= TIGHT
    assert launches(stream, lambda: dc.gemv(x, y, stream=stream)) == want
