"""th_capture_begin / th_capture_end / th_graph_launch: a capture whose
recorded call fails its argument checks raises that error and leaves the
device stream usable (the capture is ended, its graph freed); a replay of a
q4 GEMV graph matches the eager call bit for bit."""
import numpy as np
import pytest

from tang_amd import capi

pytestmark = pytest.mark.gpu


def test_failed_capture_leaves_stream_usable(dev):
    rows, cols = 64, 256
    nib, sc16 = capi.synth_q4(5, rows, cols)
    w = dev.q4_upload_packed(nib, sc16, rows, cols, capi.F16)
    x = dev.upload(capi.synth_normal(6, cols, 1.0, capi.BF16), capi.BF16)
    short = dev.alloc(3)
    with pytest.raises(capi.TangHipError):
        dev.capture(lambda: dev.gemm_q4(x, 1, w, short))  # y too short: rejected before any launch
    eager = dev.gemm_q4(x, 1, w).to_numpy()
    y = dev.alloc(rows)
    g = dev.capture(lambda: dev.gemm_q4(x, 1, w, y))
    try:
        for _ in range(3):
            y.upload(np.zeros(rows, np.float32))
            g.launch()
            dev.sync()
            assert np.array_equal(y.to_numpy(), eager)
    finally:
        g.free()


@pytest.mark.parametrize("m", [6, 20])
def test_captured_gemm_splits_before_any_call(m):
    """A q8 GEMM captured as a device's first call splits K in the workspace the
    device starts with: every replay matches the eager call bit for bit."""
    dev = capi.HipComputeDevice(0)
    rows, cols = 1000, 1096
    rng = np.random.default_rng(m)
    w = dev.q8_upload_rowwise(rng.integers(-128, 128, (rows, cols), np.int8),
                              rng.uniform(0.005, 0.02, rows).astype(np.float32), rows, cols)
    x = dev.upload(rng.standard_normal(m * cols).astype(np.float32))
    y = dev.alloc(m * rows)
    g = dev.capture(lambda: dev.gemv_q8(x, m, w, y))
    try:
        eager = dev.gemv_q8(x, m, w).to_numpy()
        for _ in range(3):
            y.upload(np.zeros(m * rows, np.float32))
            g.launch()
            dev.sync()
            assert np.array_equal(y.to_numpy(), eager)
    finally:
        g.free()


@pytest.mark.parametrize("grown", [False, True])
@pytest.mark.parametrize("m,k,n,bd", [(5, 4000, 700, capi.F32), (100, 2100, 1000, capi.BF16), (130, 4096, 8000, capi.F32)])
def test_captured_matmul_matches_eager(grown, m, k, n, bd):
    """A matmul captured as a device's first call, or after calls that outgrew the
    first workspace, gives the eager call's bits on every replay."""
    dev = capi.HipComputeDevice(0)
    rng = np.random.default_rng(m)
    if grown:
        kv = dev.alloc(3000 * 16 * 256, capi.F16)
        q, o = dev.alloc(496 * 64 * 256), dev.alloc(496 * 64 * 256)
        for b in (kv, q):
            dev.zero_buffer(b)
        capi.check(capi.lib().th_kv_attention(dev.handle, q.handle, kv.handle, kv.handle, 2504, 496, 64, 16, 256, o.handle))
    a = dev.upload(rng.standard_normal(m * k))
    b = dev.convert(dev.upload(rng.standard_normal(k * n)), bd)
    c = dev.alloc(m * n)
    call = lambda: capi.check(capi.lib().th_matmul_ex(dev.handle, a.handle, b.handle, m, k, n, 0, 0, 0, c.handle))
    g = dev.capture(call)
    other = capi.HipComputeDevice(0)  # its workspace holds what a new device's does
    a2 = other.upload(a.to_numpy())
    b2 = other.convert(other.upload(dev.convert(b, capi.F32).to_numpy()), bd)
    eager = other.matmul(a2, b2, m, k, n).to_numpy()
    call()
    assert np.array_equal(c.to_numpy(), eager)
    for _ in range(3):
        dev.zero_buffer(c)
        g.launch()
        dev.sync()
        assert np.array_equal(c.to_numpy(), eager)
    g.free()


def test_replay_after_workspaces_grew():
    """A graph names the workspaces that its calls used.  Larger calls afterwards
    outgrow them (and other buffers take whatever is freed): every replay still
    gives the eager result, and the outgrown memory comes back with the graph."""
    dev = capi.HipComputeDevice(0)
    rng = np.random.default_rng(3)
    heads, hd, n = 16, 256, 3000
    kv = [dev.upload(rng.standard_normal(n * heads * hd).astype(np.float16).view(np.uint16), capi.F16) for _ in range(2)]
    q = dev.upload(rng.standard_normal(heads * hd).astype(np.float32))
    nib, sc = capi.synth_q4(5, 512, 1024)
    w4 = dev.q4_upload_packed(nib, sc, 512, 1024, capi.F16)
    w8 = dev.q8_upload_rowwise(rng.integers(-128, 128, (1000, 4096), np.int8),
                               rng.uniform(0.005, 0.02, 1000).astype(np.float32), 1000, 4096)
    x4, x8 = dev.upload(rng.standard_normal(40 * 1024)), dev.upload(rng.standard_normal(20 * 4096))
    out = [dev.alloc(heads * hd), dev.alloc(40 * 512), dev.alloc(20 * 1000)]

    def calls():  # K splits' records and arrival counters, prepared activations, K splits' partial sums
        capi.check(capi.lib().th_kv_attention(dev.handle, q.handle, kv[0].handle, kv[1].handle, n - 1, 1, heads, heads, hd,
                                              out[0].handle))
        dev.gemm_q4(x4, 40, w4, out[1])
        dev.gemv_q8(x8, 20, w8, out[2])

    calls()
    eager = [o.to_numpy() for o in out]
    g = dev.capture(calls)
    big_q = dev.alloc(496 * 64 * hd)  # 64 heads on 16, two splits: records of 65 MB
    dev.zero_buffer(big_q)
    big_out = dev.alloc(496 * 64 * hd)
    big_x, big_y = dev.alloc(4096 * 1024), dev.alloc(4096 * 512)
    dev.zero_buffer(big_x)
    for _ in range(2):
        capi.check(capi.lib().th_kv_attention(dev.handle, big_q.handle, kv[0].handle, kv[1].handle, n - 496, 496, 64, heads, hd,
                                              big_out.handle))
        dev.gemm_q4(big_x, 4096, w4, big_y)
        held = [dev.upload(np.full(k << 18, np.nan, np.float32)) for k in (1, 2, 4, 8, 16, 32)]
        for i in range(3):
            for o in out:
                dev.zero_buffer(o)
            g.launch()
            dev.sync()
            for o, e in zip(out, eager):
                assert np.array_equal(o.to_numpy(), e)
    free = dev.memory_info()[0]
    g.free()
    assert dev.memory_info()[0] >= free + (32 << 20)  # the blocks that only the graph named
    calls()
    assert all(np.array_equal(o.to_numpy(), e) for o, e in zip(out, eager))
    for b in held + [big_q, big_out, big_x, big_y, q, x4, x8] + kv + out:
        b.free()
    dev.close()
