"""Dense ComputeDevice operators on the device against the oracle
(crates/tang-compute/src/cpu.rs naive_matmul :760, transpose_2d :317,
reduce_sum :169, add_assign :650; device.rs bias_add :378) and the
run-time compiled element-wise kernels of ComputeDevice::elementwise
(device.rs:93) against numpy.

Bars: transpose, reduce_sum (same summation order), bias_add and
add_assign bit-exact; matmul within 1e-5 max-abs-rel of the oracle's f32
sums (f32 MFMA products, f32 accumulation in another order; the north-star
bar for f32 is 1e-3); element-wise kernels within 1e-6 max-abs-rel of
numpy's float32 evaluation (the device's sin/exp2/log2/atan2/sqrt differ
from numpy's in the last bits)."""
import numpy as np
import pytest

import oracle
from conftest import max_abs_rel
from tang_amd import capi

pytestmark = pytest.mark.gpu


def _bf16_round(x):
    return oracle.bf16_to_f32(oracle.f32_to_bf16(x))


@pytest.mark.parametrize("m,k,n", [(1, 2, 1), (2, 3, 2), (37, 100, 71), (64, 64, 64), (256, 1024, 384),
                                   (5, 4096, 11)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_variants(dev, m, k, n, ta, tb):
    print(f"matmul m={m} k={k} n={n} ta={ta} tb={tb}", flush=True)
    rng = np.random.default_rng(m * 7 + k + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    ref = oracle.matmul(a, b, m, k, n)
    da = dev.upload((a.T if ta else a).reshape(-1).copy())
    db = dev.upload((b.T if tb else b).reshape(-1).copy())
    c = dev.matmul(da, db, m, k, n, trans_a=ta, trans_b=tb).to_numpy().reshape(m, n)
    err = max_abs_rel(c, ref)
    print("max_abs_rel", err)
    assert err < 1e-5


@pytest.mark.parametrize("m,k,n", [(1, 1, 3), (16, 31, 64), (17, 33, 65), (64, 32, 128), (65, 130, 129), (3, 1000, 70),
                                   (130, 515, 260), (1, 100, 1), (33, 200, 100), (610, 100, 1210)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("ad,bd", [("f32", "bf16"), ("bf16", "f32"), ("bf16", "bf16"), ("f32", "f32")])
def test_matmul_tiles_and_types(dev, m, k, n, ta, tb, ad, bd):
    """Edges of the 16- and 64-row tiles, the 32-deep steps and the K splits,
    for every operand type and order, added to C.  Products of bf16 parts are
    exact (f32 x f32 leaves out under 2^-30 of one), sums are f32: an output
    is off by at most (k + 4) roundings of its terms' magnitudes."""
    rng = np.random.default_rng(m * 7 + k + n)
    a = (rng.standard_normal((m, k)) * 10.0 ** rng.uniform(-8, 8, (m, 1))).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    c0 = rng.standard_normal((m, n)).astype(np.float32)

    def up(x, t, dt):
        x = (x.T if t else x).reshape(-1).copy()
        return dev.upload(oracle.f32_to_bf16(x), capi.BF16) if dt == "bf16" else dev.upload(x)

    if ad == "bf16":
        a = _bf16_round(a.reshape(-1)).reshape(m, k)
    if bd == "bf16":
        b = _bf16_round(b.reshape(-1)).reshape(k, n)
    c = dev.upload(c0)
    dev.matmul(up(a, ta, ad), up(b, tb, bd), m, k, n, trans_a=ta, trans_b=tb, accumulate_into=c)
    a, b = a.astype(np.float64), b.astype(np.float64)
    ref, mag = c0 + a @ b, np.abs(c0) + np.abs(a) @ np.abs(b)
    assert np.all(np.abs(c.to_numpy().reshape(m, n) - ref) <= (k + 4) * 2.0 ** -24 * mag)


def _spread(rng, shape, exps):
    """Random signs and mantissas, a power of two per row (exps) down to f32's
    subnormals."""
    x = rng.uniform(1, 2, shape) * rng.choice([-1.0, 1.0], shape) * np.exp2(np.asarray(exps, np.float64))[:, None]
    return x.astype(np.float32)


@pytest.mark.parametrize("m,k,n", [(9, 70, 50), (80, 515, 140), (620, 70, 1160)])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
@pytest.mark.parametrize("ad,bd", [("f32", "bf16"), ("bf16", "f32"), ("f32", "f32")])
@pytest.mark.parametrize("big", [False, True])
def test_matmul_exponent_range(dev, m, k, n, ta, tb, ad, bd, big):
    """Rows of f32's smallest numbers, subnormals among them, against large
    partners keep f32's bits, and (big) so do sums near its largest: as many
    roundings as anywhere else."""
    rng = np.random.default_rng(m + k + big)
    ea = rng.integers(90, 117, m) if big else rng.integers(-149, -95, m)
    a = _spread(rng, (m, k), ea if ad == "f32" else rng.integers(90, 110, m))
    b = _spread(rng, (n, k), (rng.integers(-4, 1, n) if big else rng.integers(95, 105, n)) if ad == "f32" else
                (rng.integers(-9, 4, n) if big else rng.integers(-149, -95, n)))

    def up(x, t, dt):
        x = (x.T if t else x).reshape(-1).copy()
        return dev.upload(oracle.f32_to_bf16(x), capi.BF16) if dt == "bf16" else dev.upload(x)

    if ad == "bf16":
        a = _bf16_round(a.reshape(-1)).reshape(m, k)
    if bd == "bf16":
        b = _bf16_round(b.reshape(-1)).reshape(n, k)
    c = dev.alloc(m * n)
    dev.zero_buffer(c)
    dev.matmul(up(a, ta, ad), up(b, not tb, bd), m, k, n, trans_a=ta, trans_b=tb, accumulate_into=c)
    a, b = a.astype(np.float64), b.astype(np.float64).T
    mag = np.abs(a) @ np.abs(b)
    assert np.all(mag > 2.0 ** -70) and np.all(mag < 2.0 ** 128)
    assert np.all(np.abs(c.to_numpy().reshape(m, n) - a @ b) <= (k + 4) * 2.0 ** -24 * mag)


@pytest.mark.parametrize("ad,bd", [("f32", "f32"), ("f32", "bf16"), ("bf16", "f32")])
@pytest.mark.parametrize("m,k", [(5, 1), (40, 1), (40, 2), (40, 32), (40, 45)])
def test_matmul_full_mantissas(dev, m, k, ad, bd):
    """Significands that truncate worst in parts, all of one sign: one product is
    rounded once, as in f32.  A sum's bound is two roundings for its steps and
    one of an eighth of the terms for each of them."""
    worst = {"f32": 0x3F80FFFF, "bf16": 0x3FFF0000}
    rng = np.random.default_rng(k)
    a = np.full((m, k), worst[ad], np.uint32).view(np.float32)
    b = np.full((k, 30), worst[bd], np.uint32).view(np.float32)
    if ad == "f32":
        a[1:] = rng.uniform(1, 2, (m - 1, k)).astype(np.float32)
    if bd == "f32":
        b[:, 1:] = rng.uniform(1, 2, (k, 29)).astype(np.float32)
    up = lambda x, dt: dev.upload(oracle.f32_to_bf16(x.reshape(-1)), capi.BF16) if dt == "bf16" else dev.upload(x)
    c = dev.matmul(up(a, ad), up(b, bd), m, k, 30).to_numpy().reshape(m, 30).astype(np.float64)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    err = (c - ref) / ref * 2.0 ** 24
    assert np.max(np.abs(err)) <= (1 if k == 1 else k / 8 + 2)


@pytest.mark.parametrize("m,k", [(5, 200), (70, 200), (5, 400), (70, 400)])
@pytest.mark.parametrize("bd", ["f32", "bf16"])
def test_matmul_infinities(dev, m, k, bd):
    """An infinity times finite values gives infinities, times zero NaN, and
    reaches no other row or column."""
    n = 40
    rng = np.random.default_rng(m)
    a = rng.integers(1, 9, (m, k)).astype(np.float32)
    b = rng.integers(1, 9, (k, n)).astype(np.float32)
    a[1, 7], a[2, 150], b[7, 3], b[90, 5] = np.inf, -np.inf, 0.0, np.inf
    db = dev.upload(oracle.f32_to_bf16(b.reshape(-1)), capi.BF16) if bd == "bf16" else dev.upload(b)
    c = dev.matmul(dev.upload(a), db, m, k, n).to_numpy().reshape(m, n)
    with np.errstate(invalid="ignore"):
        ref = np.stack([(a[:, [i]].astype(np.float64) * b[[i]]) for i in range(k)]).sum(0)
    assert np.isnan(ref[1, 3]) and np.isnan(ref[2, 5]) and np.isinf(ref[1, 0])
    assert np.array_equal(c, ref.astype(np.float32), equal_nan=True)


def test_matmul_kats_and_accumulate(dev):
    """cpu.rs:785-822 known answers; matmul_accumulate (device.rs:391) adds."""
    c = dev.matmul(dev.upload(np.array([1, 0, 0, 1], np.float32)), dev.upload(np.array([1, 2, 3, 4], np.float32)),
                   2, 2, 2)
    assert c.to_numpy().tolist() == [1, 2, 3, 4]
    c = dev.matmul(dev.upload(np.array([1, 2, 3, 4, 5, 6], np.float32)),
                   dev.upload(np.array([7, 8, 9, 10, 11, 12], np.float32)), 2, 3, 2)
    assert c.to_numpy().tolist() == [58, 64, 139, 154]
    dev.matmul(dev.upload(np.array([1, 2, 3, 4, 5, 6], np.float32)),
               dev.upload(np.array([7, 8, 9, 10, 11, 12], np.float32)), 2, 3, 2, accumulate_into=c)
    assert c.to_numpy().tolist() == [116, 128, 278, 308]


def test_linear_forward_2d_bf16_weight(dev):
    """Linear::forward_2d (modules.rs:56) on the device: x . W^T with W
    [out][in] in bf16, then bias_add."""
    rng = np.random.default_rng(9)
    m, k, n = 48, 320, 200
    x = rng.standard_normal((m, k)).astype(np.float32)
    w = _bf16_round(rng.standard_normal((n, k)).astype(np.float32) * 0.05)
    bias = rng.standard_normal(n).astype(np.float32)
    y = dev.matmul_b_transposed(dev.upload(x.reshape(-1)), dev.upload(oracle.f32_to_bf16(w).reshape(-1), capi.BF16),
                                m, k, n)
    y = dev.bias_add(y, dev.upload(bias), m * n, n).to_numpy().reshape(m, n)
    ref = oracle.bias_add(oracle.matmul(x, w.T.copy(), m, k, n), bias, m * n, n).reshape(m, n)
    assert max_abs_rel(y, ref) < 1e-5


@pytest.mark.parametrize("rows,cols", [(2, 3), (1, 1000), (33, 65), (1024, 700)])
def test_transpose_exact(dev, rows, cols):
    x = np.random.default_rng(rows).standard_normal(rows * cols).astype(np.float32)
    got = dev.transpose_2d(dev.upload(x), rows, cols).to_numpy()
    assert np.array_equal(got, oracle.transpose_2d(x, rows, cols))


@pytest.mark.parametrize("shape", [[2, 3], [7, 300, 5], [4096, 3], [3, 1, 9], [1000]])
def test_reduce_sum_bit_exact(dev, shape):
    x = np.random.default_rng(len(shape)).standard_normal(int(np.prod(shape))).astype(np.float32)
    dx = dev.upload(x)
    for axis in range(len(shape)):
        got = dev.reduce_sum(dx, shape, axis).to_numpy()
        assert np.array_equal(got, oracle.reduce_sum(x, shape, axis)), axis
    # reduce_sum_accumulate (device.rs:451): dst + reduce_sum
    acc = dev.upload(np.ones(int(np.prod(shape[1:])), np.float32))
    dev.reduce_sum(dx, shape, 0, accumulate_into=acc)
    assert np.array_equal(acc.to_numpy(), (np.float32(1) + oracle.reduce_sum(x, shape, 0)).astype(np.float32))


def test_bias_add_and_add_assign_exact(dev):
    rng = np.random.default_rng(5)
    m = rng.standard_normal(30 * 17).astype(np.float32)
    b = rng.standard_normal(17).astype(np.float32)
    got = dev.bias_add(dev.upload(m), dev.upload(b), m.size, 17).to_numpy()
    assert np.array_equal(got, oracle.bias_add(m, b, m.size, 17))
    a = dev.upload(np.array([1.0, 2.0, 3.0], np.float32))  # cpu.rs:1152-1158
    dev.add_assign(a, dev.upload(np.array([0.5, 1.0, 1.5], np.float32)))
    assert a.to_numpy().tolist() == [1.5, 3.0, 4.5]
    with pytest.raises(capi.TangHipError):
        dev.add_assign(a, dev.upload(np.zeros(4, np.float32)))


def _expr_kernel(n_inputs, body, result):
    """A kernel in the form tang-expr generates for ComputeDevice::elementwise:
    inputs in0.., output `outputs`, element count, one thread per element,
    inputs loaded as x<i>, SSA temporaries, one output."""
    params = "".join("const float* __restrict__ in%d,\n    " % i for i in range(n_inputs))
    loads = "".join("    float x%d = in%d[gid];\n" % (i, i) for i in range(n_inputs))
    return ('extern "C" __global__ void k0(' + params + "float* __restrict__ outputs,\n"
            "    const unsigned int count) {\n"
            "    unsigned int gid = blockIdx.x * blockDim.x + threadIdx.x;\n"
            "    if (gid >= count) { return; }\n\n" + loads + "\n" +
            "".join("    float %s;\n" % line for line in body) + "\n"
            "    outputs[gid * 1 + 0] = %s;\n}\n" % result)


def test_elementwise_runtime_kernels(dev):
    rng = np.random.default_rng(8)
    n = 100003
    x = rng.uniform(0.1, 3.0, n).astype(np.float32)
    y = rng.standard_normal(n).astype(np.float32)
    dx, dy = dev.upload(x), dev.upload(y)
    cases = [
        # (x*y) + sin(x)
        (2, ["t2 = (x0 * x1)", "t3 = sin(x0)", "t4 = (t2 + t3)"], "t4",
         lambda: (x * y + np.sin(x)).astype(np.float32)),
        # select(y, sqrt(x), -1/x), exp2, log2
        (2, ["t2 = sqrt(x0)", "t3 = (1.0f / x0)", "t4 = (-t3)", "t5 = (x1 > 0.0f ? t2 : t4)",
             "t6 = exp2(x1)", "t7 = log2(x0)", "t8 = (t5 + t6)", "t9 = (t8 * t7)"], "t9",
         lambda: ((np.where(y > 0, np.sqrt(x), -1 / x) + np.exp2(y)) * np.log2(x)).astype(np.float32)),
        # atan2(y, x) with one input only used twice
        (2, ["t2 = atan2(x1, x0)"], "t2", lambda: np.arctan2(y, x).astype(np.float32)),
    ]
    for n_in, body, res, ref in cases:
        k = dev.compile_kernel(_expr_kernel(n_in, body, res))
        try:
            got = dev.run_kernel(k, [dx, dy][:n_in], n).to_numpy()
        finally:
            capi.lib().th_kernel_free(k)
        want = ref()
        err = max_abs_rel(got, want)
        print(res, "max_abs_rel", err)
        assert err < 1e-6


def test_elementwise_compile_error_reported(dev):
    with pytest.raises(capi.TangHipError) as e:
        dev.compile_kernel('extern "C" __global__ void k0(float* outputs, const unsigned int count) { oops; }')
    assert "compile" in str(e.value)


def _graphs():
    """(n_inputs, builder, exact): graphs over x in [0.1, 3) and y ~ N(0, 1).
    exact: only +, *, neg, 1/x, sqrt, select and literals, whose f64 results
    are IEEE-determined, so the device must give the CPU backend's bits."""
    def hypot_sel(g, v):
        x, y = v
        return g.select(y, g.sqrt(g.add(g.mul(x, x), g.mul(y, y))), g.neg(g.recip(x)))

    def poly(g, v):
        x, y = v
        t = g.add(g.mul(g.lit(0.1), x), g.lit(-2.5))
        return g.add(g.mul(t, t), g.mul(g.lit(1.0 / 3.0), g.mul(x, y)))

    def sigmoid_ish(g, v):  # the reference's softplus/sigmoid shapes go through exp2 and recip
        x, y = v
        e = g.exp2(g.mul(g.lit(-1.4426950408889634), y))
        return g.mul(x, g.recip(g.add(g.lit(1.0), e)))

    def trig(g, v):
        x, y = v
        return g.add(g.mul(g.sin(x), g.atan2(y, x)), g.log2(x))

    def one_input(g, v):
        (x,) = v
        return g.mul(g.add(x, g.lit(1.0)), g.add(x, g.lit(1.0)))

    return [(2, hypot_sel, True), (2, poly, True), (2, sigmoid_ish, False), (2, trig, False), (1, one_input, True)]


@pytest.mark.parametrize("n", [1, 3, 4, 1027, 100003])
def test_elementwise_graph_matches_cpu_backend(dev, n):
    """ComputeDevice::elementwise from a tang-expr graph: bit-identical to the
    CPU backend's f64 evaluation (oracle.expr_eval) for the IEEE-exact ops;
    within one f32 rounding step for sin/atan2/exp2/log2 (device math
    library against the host's libm, both f64).  n covers the 4-wide tail."""
    import oracle
    rng = np.random.default_rng(n)
    x = rng.uniform(0.1, 3.0, n).astype(np.float32)
    y = rng.standard_normal(n).astype(np.float32)
    dx, dy = dev.upload(x), dev.upload(y)
    for n_in, build, exact in _graphs():
        print("expr", build.__name__, n, flush=True)
        got = dev.elementwise([dx, dy][:n_in], n, build).to_numpy()
        g = capi.ExprGraph()
        out = build(g, [g.var(i) for i in range(n_in)])
        want = oracle.expr_eval(g.array(), out, [x, y][:n_in])
        if exact:
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), build.__name__
        else:
            ulp = np.abs(got.view(np.int32).astype(np.int64) - want.view(np.int32).astype(np.int64))
            assert ulp.max() <= 1, (build.__name__, ulp.max())


def test_elementwise_graph_cache_and_special_values(dev):
    """The same graph twice (second call from the device's compiled cache),
    and IEEE special values: 1/0 = inf, sqrt(-1) = NaN, select on NaN takes
    the else branch, as the CPU backend's closure does."""
    x = np.array([0.0, -1.0, np.nan, 4.0, -0.0], np.float32)
    dx = dev.upload(x)
    build = lambda g, v: g.add(g.recip(v[0]), g.select(v[0], g.sqrt(v[0]), g.lit(7.0)))
    a = dev.elementwise([dx], len(x), build).to_numpy()
    b = dev.elementwise([dx], len(x), build).to_numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert np.isposinf(a[0]) and a[1] == 6.0 and np.isnan(a[2]) and a[3] == 2.25 and np.isneginf(a[4])
