"""GPU parity of the softmax kernels against the CPU oracle and the golden fixtures.

Tolerances: f32 outputs rel 1e-5; f16/bf16 outputs rel 2e-2 / abs 1e-2 (and, tighter,
within one f16 ulp of the oracle)."""
import numpy as np
import pytest
import torch

import intent_amd as intent
import oracle
from intent_amd.examples import inputs
from intent_amd.examples.kernels.backward.softmax import softmax_backward, softmax_backward_f16
from intent_amd.examples.kernels.normalization.softmax import (chunked_softmax_bf16, stable_softmax,
                                                               stable_softmax_f16)
from intent_amd.runtime.hip import library as hiplib
from tests.gpu_util import (announce, assert_16bit, assert_f32_rel, bf16_tensor_bits, bf16_to_f32,
                            f16_ulp_distance, to_bf16_tensor)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4096, 1024), (7, 1000), (5, 5000), (3, 4097), (2, 64), (1, 3), (64, 4096)])
def test_softmax_f32_matches_oracle(device, shape):
    announce("softmax_f32", shape)
    x = inputs.normal(np.random.default_rng(shape[1]), shape, "f32", 4)
    y = intent.jit(stable_softmax, backend="hip").run(torch.from_numpy(x).to(device))
    assert_f32_rel(y.cpu().numpy(), oracle.softmax_fwd(x))


def test_softmax_f32_config1_seed0(device):
    announce("softmax_f32 config 1")
    x = inputs.softmax_f32()
    y = intent.jit(stable_softmax, backend="hip").run(torch.from_numpy(x).to(device)).cpu().numpy()
    assert_f32_rel(y, oracle.softmax_fwd(x))
    assert np.allclose(y.astype(np.float64).sum(axis=1), 1.0, atol=1024 * 2 ** -24)


def test_softmax_golden(device, golden):
    announce("softmax golden")
    g = golden("softmax")
    run32 = intent.jit(stable_softmax, backend="hip")
    y = run32.run(torch.from_numpy(g["softmax_f32_x"]).to(device)).cpu().numpy()
    assert_f32_rel(y, g["softmax_f32_y"])
    assert (y[2, ::3] == 0).all() and y[3, 17] == 1.0
    y2 = run32.run(torch.from_numpy(g["softmax_pow2_x"]).to(device)).cpu().numpy()
    assert (y2 == np.float32(1 / 1024)).all()
    y16 = intent.jit(stable_softmax_f16, backend="hip").run(torch.from_numpy(g["softmax_f16_x"]).to(device))
    assert_16bit(y16.cpu().numpy(), g["softmax_f16_y"])
    yb = intent.jit(chunked_softmax_bf16, backend="hip").run(to_bf16_tensor(g["softmax_bf16_x"], device))
    assert_16bit(bf16_to_f32(bf16_tensor_bits(yb)), g["softmax_bf16_y"])


@pytest.mark.parametrize("shape", [(16384, 4096), (9, 8200), (4, 12), (33, 2048), (3, 1001)])
def test_softmax_f16_matches_oracle(device, shape):
    announce("softmax_f16", shape)
    x = inputs.normal(np.random.default_rng(shape[0]), shape, "f16", 3)
    y = intent.jit(stable_softmax_f16, backend="hip").run(torch.from_numpy(x).to(device)).cpu().numpy()
    want = oracle.softmax_fwd(x)
    assert_16bit(y, want)
    ulps = f16_ulp_distance(y, want)
    assert ulps.max() <= 1
    if ulps.size >= 10000:
        assert (ulps == 0).mean() > 0.98


def test_softmax_bf16_matches_oracle(device):
    announce("softmax_bf16")
    x = inputs.normal(np.random.default_rng(3), (129, 3000), "bf16", 3)
    y = intent.jit(chunked_softmax_bf16, backend="hip").run(to_bf16_tensor(x, device))
    want = oracle.softmax_fwd(x, storage="bf16")
    assert_16bit(bf16_to_f32(bf16_tensor_bits(y)), bf16_to_f32(want))
    assert np.abs(bf16_tensor_bits(y).astype(np.int32) - want.astype(np.int32)).max() <= 1


def test_softmax_special_values(device):
    announce("softmax special values")
    x = np.random.default_rng(4).standard_normal((6, 4096)).astype(np.float32)
    x[0, 5] = np.nan
    x[1, :] = -np.inf
    x[2, 9] = np.inf
    x[3, ::2] = -np.inf
    y = intent.jit(stable_softmax, backend="hip").run(torch.from_numpy(x).to(device)).cpu().numpy()
    want = oracle.softmax_fwd(x)
    assert np.isnan(y[:3]).all()
    assert_f32_rel(y, want)
    y16 = intent.jit(stable_softmax_f16, backend="hip").run(torch.from_numpy(x.astype(np.float16)).to(device))
    assert (np.isnan(y16.cpu().numpy()) == np.isnan(oracle.softmax_fwd(x.astype(np.float16)))).all()


def test_softmax_layouts_and_explicit_outputs(device):
    announce("softmax layouts")
    rng = np.random.default_rng(5)
    base = torch.from_numpy(inputs.normal(rng, (300, 512), "f16", 3)).to(device)
    kernel = intent.jit(stable_softmax_f16, backend="hip")
    transposed = base.t()                                  # inner stride 512: staged through a copy
    y = kernel.run(transposed)
    assert_16bit(y.cpu().numpy(), oracle.softmax_fwd(np.ascontiguousarray(transposed.cpu().numpy())))
    sliced = base[:, 100:400]                              # row stride 512, misaligned start
    out = torch.empty(300, 300, dtype=torch.float16, device=device)
    kernel(sliced, out)
    assert_16bit(out.cpu().numpy(), oracle.softmax_fwd(np.ascontiguousarray(sliced.cpu().numpy())))
    strided_out = torch.empty(300, 600, dtype=torch.float16, device=device)[:, ::2]  # inner stride 2
    kernel.prepare(sliced, outputs=(strided_out,)).launch()
    assert_16bit(strided_out.cpu().numpy(), oracle.softmax_fwd(np.ascontiguousarray(sliced.cpu().numpy())))
    inplace = base.clone()
    kernel(inplace, inplace)                               # exact alias: each row is read before written
    assert_16bit(inplace.cpu().numpy(), oracle.softmax_fwd(base.cpu().numpy()))
    with pytest.raises(ValueError):
        kernel(base[:, 1:], base[:, :-1])                 # partial overlap is rejected


def test_softmax_bwd_f32_static(device):
    announce("softmax_bwd_f32 4096x4097")
    rng = np.random.default_rng(6)
    p = oracle.softmax_fwd(inputs.normal(rng, (4096, 4097), "f32", 2))
    dy = inputs.normal(rng, (4096, 4097), "f32")
    dx = intent.jit(softmax_backward, backend="hip").run(torch.from_numpy(p).to(device),
                                                        torch.from_numpy(dy).to(device)).cpu().numpy()
    want = oracle.softmax_bwd(p, dy)
    # cancelling sum: |err| <= 1e-5 * p * (|dy| + sum|p dy|)
    scale = np.abs(p.astype(np.float64)) * (np.abs(dy) + np.sum(np.abs(p * dy), axis=1, keepdims=True))
    assert np.all(np.abs(dx.astype(np.float64) - want) <= 1e-5 * scale + 1e-37)


@pytest.mark.parametrize("shape", [(16384, 4096), (5, 9000), (17, 1000), (3, 8)])
def test_softmax_bwd_f16(device, shape):
    announce("softmax_bwd_f16", shape)
    x, dy = inputs.softmax_f16_fwd_bwd(seed=shape[1], rows=shape[0], cols=shape[1])
    fwd = intent.jit(stable_softmax_f16, backend="hip")
    bwd = intent.jit(softmax_backward_f16, backend="hip")
    y = fwd.run(torch.from_numpy(x).to(device))
    dx = bwd.run(y, torch.from_numpy(dy).to(device)).cpu().numpy()
    p = y.cpu().numpy()
    want = oracle.softmax_bwd(p, dy)
    assert_16bit(dx, want)
    # within two f16 roundings, plus the projection's reassociation error 1e-5 * p * sum|p dy|
    p64 = p.astype(np.float64)
    spread = 1e-5 * np.abs(p64) * np.sum(np.abs(p64 * dy.astype(np.float64)), axis=1, keepdims=True)
    assert np.all(np.abs(dx.astype(np.float64) - want) <= 2 ** -9 * np.abs(want.astype(np.float64)) + spread + 6e-8)


def test_softmax_bwd_f16_rounds_like_the_definition(device):
    """Inputs on which every product, the whole projection sum and dy - proj are exact in f32
    (p = k 2^-12 with k < 2048 at 128 places per row, dy = j 2^-3 with |j| < 32), so the
    summation order cannot matter and dx must equal the oracle bit for bit. The definition
    rounds p * (dy - proj) to f32 and then casts to f16; on these rows 31 elements differ from
    a single rounding straight to f16 (a multiply fused with the conversion), so such a fusion
    fails here."""
    announce("softmax_bwd_f16 exact-rounding rows")
    rng = np.random.default_rng(7)
    rows, cols, nz = 4096, 4096, 128
    k = np.zeros((rows, cols), np.int64)
    for r in range(rows):
        k[r, rng.choice(cols, nz, replace=False)] = rng.integers(1, 2048, nz)
    p = (k * 2.0 ** -12).astype(np.float16)
    dy = (rng.integers(-31, 32, (rows, cols)) * 2.0 ** -3).astype(np.float16)
    p64 = p.astype(np.float64)
    product = p64 * (dy.astype(np.float64) - (p64 * dy.astype(np.float64)).sum(axis=1, keepdims=True))
    once = product.astype(np.float16)
    want = oracle.softmax_bwd(p, dy)
    assert np.array_equal(want.view(np.uint16), product.astype(np.float32).astype(np.float16).view(np.uint16))
    assert (want.view(np.uint16) != once.view(np.uint16)).sum() > 0     # the rows discriminate
    dx = intent.jit(softmax_backward_f16, backend="hip").run(torch.from_numpy(p).to(device),
                                                            torch.from_numpy(dy).to(device)).cpu().numpy()
    assert np.array_equal(dx.view(np.uint16), want.view(np.uint16))


def test_softmax_bwd_golden(device, golden):
    announce("softmax_bwd golden")
    g = golden("softmax_bwd")
    dx = intent.jit(softmax_backward_f16, backend="hip").run(
        torch.from_numpy(g["softmax_bwd_f16_p"]).to(device), torch.from_numpy(g["softmax_bwd_f16_dy"]).to(device))
    w = g["softmax_bwd_f16_dx"]
    assert np.all(np.abs(dx.cpu().numpy() - w) <= 2e-2 * np.abs(w) + 1e-2 * np.abs(w).max())


def test_softmax_config2_seed0_fwd_bwd(device):
    """The exact pair the bench times: x, dy of config 2 drawn from seed 0, the forward's y fed to
    the backward through prepared calls, as bench.py's step does."""
    announce("softmax config 2 seed 0 fwd+bwd")
    x, dy = inputs.softmax_f16_fwd_bwd(seed=0, rows=16384, cols=4096)
    fwd = intent.jit(stable_softmax_f16, backend="hip").prepare(torch.from_numpy(x).to(device))
    bwd = intent.jit(softmax_backward_f16, backend="hip").prepare(fwd.result(), torch.from_numpy(dy).to(device))
    fwd.launch()
    bwd.launch()
    y = fwd.result().cpu().numpy()
    want_y = oracle.softmax_fwd(x)
    assert_16bit(y, want_y)
    ulps = f16_ulp_distance(y, want_y)
    assert ulps.max() <= 1 and (ulps == 0).mean() > 0.98
    dx = bwd.result().cpu().numpy()
    want = oracle.softmax_bwd(y, dy)
    assert_16bit(dx, want)
    p64 = y.astype(np.float64)
    spread = 1e-5 * np.abs(p64) * np.sum(np.abs(p64 * dy.astype(np.float64)), axis=1, keepdims=True)
    assert np.all(np.abs(dx.astype(np.float64) - want) <= 2 ** -9 * np.abs(want.astype(np.float64)) + spread + 6e-8)


# Rows of a workgroup: both sides of every step of threads and chunks (16-bit 8192, 16384, 32768, 65536, 131072
# elements; f32 half of that), ragged ends, ragged rows that are a wave's in these numbers (up to 1024 16-bit and 2048 f32
# columns; many of them below), rows longer than any workgroup's registers.
@pytest.mark.parametrize("rows,cols", [(5, 255), (5, 257), (9, 505), (3, 513), (7, 1017), (3, 2049), (2, 4095), (2, 4104),
                                       (3, 8185), (2, 8192), (2, 8200), (3, 16384), (2, 16392), (2, 32768), (2, 32776),
                                       (1, 65533), (2, 65544), (1, 131065), (1, 131072), (2, 131080), (1, 140001)])
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_softmax_workgroup_rows(device, rows, cols, kind):
    """Forward (and for f32 and f16 backward) against the oracle, with the output inside a buffer whose other elements must
    not change, and the operands' rows at a stride and start that leave them ragged and differently aligned."""
    announce("softmax workgroup rows", rows, cols, kind)
    dtype = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    rng = np.random.default_rng(rows * cols)
    fwd = {"f32": stable_softmax, "f16": stable_softmax_f16, "bf16": chunked_softmax_bf16}[kind]
    x = rng.standard_normal((rows, cols), dtype=np.float32) * 3
    dy = rng.standard_normal((rows, cols), dtype=np.float32)
    as_f64 = lambda t: t.float().cpu().numpy().astype(np.float64)  # noqa: E731
    for pad, offsets in ((0, (0, 0, 0)), (3, (1, 1, 1)), (5, (0, 2, 3))):
        def view(data, offset):
            base = torch.full((rows * (cols + pad) + 16,), 7.0, dtype=dtype, device=device)
            v = base[offset:offset + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
            if data is not None:
                v.copy_(torch.from_numpy(data).to(device).to(dtype))
            return base, v

        def untouched(base, v):
            v.fill_(7.0)
            return bool((base == 7.0).all())

        _, xv = view(x, offsets[0])
        y_base, yv = view(None, offsets[1])
        intent.jit(fwd, backend="hip")(xv, yv)
        want = torch.softmax(xv.double(), dim=1)
        if kind == "f32":
            assert_f32_rel(as_f64(yv), want.cpu().numpy())
        else:
            assert_16bit(as_f64(yv), want.cpu().numpy(), rel=2.0 ** (-10 if kind == "f16" else -7), abs_=2.0 ** -24)
        p = yv.clone()
        assert untouched(y_base, yv)
        if kind != "bf16":       # through the C ABI: the f32 definition's extents are fixed
            _, pv = view(as_f64(p).astype(np.float32), offsets[0])
            _, gv = view(dy, offsets[2])
            d_base, dv = view(None, offsets[1])
            lib, stride = hiplib.library(), cols + pad
            lib.check(lib.fn["softmax_bwd"](hiplib.F32 if kind == "f32" else hiplib.F16, pv.data_ptr(), gv.data_ptr(),
                                            dv.data_ptr(), rows, cols, stride, stride, stride,
                                            torch.cuda.current_stream().cuda_stream))
            p64, g64 = as_f64(pv), as_f64(gv)
            proj = (p64 * g64).sum(1, keepdims=True)
            # f32: the projection's sum in another order, at most 160 roundings deep (137 elements of a lane,
            # then lanes and waves), and the roundings of the difference and the product; f16 adds its cast
            bound = p64 * 2.0 ** -24 * (160 * np.abs(p64 * g64).sum(1, keepdims=True) + 4 * np.abs(g64 - proj))
            if kind == "f16":
                bound = bound + 2.0 ** -11 * np.abs(p64 * (g64 - proj)) + 2.0 ** -25
            assert (np.abs(as_f64(dv) - p64 * (g64 - proj)) <= bound + 1e-40).all()
            assert untouched(d_base, dv)


# A wave's rows, a workgroup's (one to four waves' worth and more, aligned and ragged), and rows read again in each pass.
@pytest.mark.parametrize("cols", [255, 257, 1003, 4104, 9001, 40000, 131072, 140001])
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_softmax_specials_on_every_kernel(device, cols, kind):
    """NaN, infinities, masks of the type's lowest value and wholly masked rows: NaN where the float64 softmax is NaN (a NaN or
    +inf in the row, or every element -inf), and its values elsewhere; a row's specials stay in the row."""
    announce("softmax specials", cols, kind)
    dtype = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    fwd = {"f32": stable_softmax, "f16": stable_softmax_f16, "bf16": chunked_softmax_bf16}[kind]
    x = torch.randn(9, cols, generator=torch.Generator(device=device).manual_seed(cols), device=device).to(dtype)
    lowest = torch.finfo(dtype).min
    x[1, cols - 1], x[2, 0], x[3, :] = float("nan"), float("inf"), float("-inf")
    x[4, ::2], x[5, 1:], x[6, :], x[7, :cols - 1] = float("-inf"), lowest, lowest, float("-inf")
    y, want = intent.jit(fwd, backend="hip").run(x), torch.softmax(x.double(), dim=1)
    assert bool((y.isnan() == want.isnan()).all()) and bool(y[1:4].isnan().all()) and not bool(y[4:].isnan().any())
    got, want = (v.nan_to_num(0.0).double().cpu().numpy() for v in (y, want))
    if kind == "f32":
        assert_f32_rel(got, want, floor=1e-30)
    else:
        assert_16bit(got, want, rel=2.0 ** (-10 if kind == "f16" else -7), abs_=2.0 ** -24)


WAVE, ROW = ("softmax_{}_wave", 128), lambda threads: ("softmax_{}_block", threads)  # noqa: E731


@pytest.mark.parametrize("kind,rows,cols,pad,fwd,bwd", [
    ("f16", 3, 1024, 0, ("softmax_fwd_pipe", 256), WAVE), ("f16", 3, 1016, 3, ROW(256), ROW(256)), ("f16", 3, 255, 0, WAVE, WAVE),
    ("f16", 3, 4104, 0, ROW(256), ROW(256)), ("f16", 3, 40000, 1, ROW(1024), ROW(1024)),
    ("f16", 3, 140000, 0, ("softmax_fwd_stream", 1024), ("softmax_bwd_stream", 1024)),
    ("f16", 116000, 383, 0, WAVE, WAVE), ("f16", 117000, 383, 0, ROW(256), ROW(256)), ("f16", 6200, 505, 0, WAVE, WAVE),
    ("f16", 6300, 505, 0, ROW(256), ROW(256)), ("f16", 17000, 506, 0, WAVE, WAVE), ("f16", 3, 641, 0, ROW(256), ROW(256)),
    ("f16", 6100, 1022, 0, WAVE, WAVE), ("f16", 6200, 1022, 0, ROW(256), ROW(256)), ("f16", 3, 1025, 0, ROW(256), ROW(256)),
    ("f16", 90000, 510, 0, ROW(256), ROW(256)), ("f16", 80000, 510, 0, WAVE, WAVE),
    ("f16", 180000, 257, 0, ROW(256), ROW(256)), ("f32", 80000, 512, 1, WAVE, WAVE), ("f32", 16400, 2047, 0, ROW(256), ROW(256)),
    ("f32", 3, 4000, 0, ROW(256), WAVE), ("f32", 2622, 4000, 0, WAVE, WAVE), ("f32", 8400, 4000, 0, ROW(256), WAVE),
    ("f32", 10900, 2047, 0, WAVE, WAVE), ("f32", 10940, 2047, 0, WAVE, ROW(256)), ("f32", 3, 2049, 0, ROW(256), ROW(256)),
    ("f32", 2047, 4095, 0, ROW(512), ROW(512)), ("f32", 2048, 4095, 0, WAVE, WAVE), ("f32", 3, 4096, 0, ROW(256), WAVE),
    ("f32", 3, 4100, 0, ROW(512), ROW(512))])
def test_softmax_observes_the_kernel_that_ran(device, kind, rows, cols, pad, fwd, bwd):
    """Each line of the dispatch from both sides, and rows at a stride that leaves them unaligned."""
    announce("softmax observation", kind, rows, cols, pad)
    dtype = torch.float16 if kind == "f16" else torch.float32
    p, dy, out = (torch.zeros(rows, cols + pad, dtype=dtype, device=device)[:, :cols] for _ in range(3))
    lib, code, stride = hiplib.library(), getattr(hiplib, kind.upper()), cols + pad
    at = [v.data_ptr() for v in (p, dy, out)]
    if kind == "f16":
        call = intent.jit(stable_softmax_f16, backend="hip").prepare(p, outputs=(out,))
        call.launch()
        facts = {r.name: r.value for r in call.observation.resources} | {"kernel": call.observation.kernel}
    else:
        facts = lib.call_resources(hiplib.OP_SOFTMAX_FWD, code, at[0], at[2], rows, cols, stride, stride)
    assert (facts["kernel"], facts["block_threads"]) == (fwd[0].format("fwd"), fwd[1])
    facts = lib.call_resources(hiplib.OP_SOFTMAX_BWD, code, *at, rows, cols, stride, stride, stride)
    assert (facts["kernel"], facts["block_threads"]) == (bwd[0].format("bwd"), bwd[1])


def test_softmax_ragged_f32_rows_past_the_mall_go_four_to_a_workgroup(device):
    """Up to 2048 columns a wave holds the row (no shared memory for partial results): one workgroup a row is bound by their
    launches (91500 x 550: 185 us, 65)."""
    announce("softmax f32 waves of a workgroup")
    lib, x = hiplib.library(), torch.zeros(61100, 1101, device=device)
    for cols, rows in ((550, 61100), (1021, 34000), (1101, 61100)):
        at = (x.data_ptr(), x.data_ptr(), x.data_ptr())
        for op, args in ((hiplib.OP_SOFTMAX_FWD, at[:2]), (hiplib.OP_SOFTMAX_BWD, at)):
            facts = lib.call_resources(op, hiplib.F32, *args, rows, cols, *[1101] * len(args))
            assert (facts["block_threads"], facts["lds_bytes"]) == (256, 0)


# Many ragged rows: the sizes at which a workgroup takes rows that a wave takes when there are fewer, and their neighbours.
@pytest.mark.parametrize("kind,rows,cols", [("f16", 32641, 257), ("f16", 17000, 505), ("f16", 17000, 515), ("f16", 6200, 1021), ("f16", 9000, 1001),
                                            ("bf16", 17000, 450), ("bf16", 9000, 1001), ("f32", 43000, 521), ("f32", 22400, 1001), ("f32", 33600, 1001), ("f32", 2700, 4000), ("f32", 8400, 4000),
                                            ("f32", 11000, 2045), ("f32", 2500, 4095), ("f32", 5500, 4095)])
def test_softmax_many_ragged_rows(device, kind, rows, cols):
    """Forward and backward against float64 on the device, to the roundings of the sums (as above) and of the result."""
    announce("softmax many ragged rows", kind, rows, cols)
    dtype = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]
    lib, code, stream = hiplib.library(), getattr(hiplib, kind.upper()), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=device).manual_seed(cols)
    x, dy = ((torch.randn(rows, cols, generator=g, device=device) * s).to(dtype) for s in (3, 1))
    y, dx = torch.full_like(x, 7.0), torch.full_like(x, 7.0)
    lib.check(lib.fn["softmax_fwd"](code, x.data_ptr(), y.data_ptr(), rows, cols, cols, cols, stream))
    lib.check(lib.fn["softmax_bwd"](code, y.data_ptr(), dy.data_ptr(), dx.data_ptr(), rows, cols, cols, cols, cols, stream))
    unit = {"f32": 1e-5, "f16": 2.0 ** -10, "bf16": 2.0 ** -7}[kind]
    tiny = {"f32": 1e-37, "f16": 2.0 ** -24, "bf16": 1e-37}[kind]
    for at in range(0, rows, 4096):
        s = slice(at, at + 4096)
        want, p, d = torch.softmax(x[s].double(), dim=1), y[s].double(), dy[s].double()
        assert bool(((p - want).abs() <= unit * want + tiny).all())
        proj = (p * d).sum(1, keepdim=True)
        bound = p * 2.0 ** -24 * (160 * (p * d).abs().sum(1, keepdim=True) + 4 * (d - proj).abs())
        if kind != "f32":
            bound = bound + unit * (p * (d - proj)).abs() + tiny
        assert bool(((dx[s].double() - p * (d - proj)).abs() <= bound + 1e-40).all())


def test_softmax_longest_row(device):
    """2^31 - 1 columns, the most an entry takes: the last 16-byte chunk reaches past 2^31 elements, and what follows the row
    in the result's buffer stays as it was."""
    cols, tail = 2 ** 31 - 1, 24
    announce("softmax longest row", cols)
    lib, stream = hiplib.library(), torch.cuda.current_stream().cuda_stream
    step = torch.arange(tail, device=device, dtype=torch.float32)
    x, buffer = torch.zeros(cols, dtype=torch.bfloat16, device=device), torch.full((cols + 9,), 7.0, dtype=torch.bfloat16,
                                                                                   device=device)
    # The maximum is 0, so that almost every exponential is 1 and a thread's 2^21 terms add up without rounding (a sum of
    # 2^21 other f32 terms may be off by 2^21 x 2^-24).
    x[-tail:] = -step / 8
    lib.check(lib.fn["softmax_fwd"](hiplib.BF16, x.data_ptr(), buffer.data_ptr(), 1, cols, cols, cols, stream))
    total = cols - tail + float(torch.exp(-step.double() / 8).sum())
    assert bool((buffer[cols:] == 7.0).all())
    assert_16bit(buffer[cols - tail:cols].double().cpu().numpy(), torch.exp(-step.double() / 8).cpu().numpy() / total,
                 rel=2.0 ** -7, abs_=0)
    first = buffer[:1].clone()
    assert abs(float(first) * total - 1) <= 2.0 ** -8 and bool((buffer[:cols - tail] == first).all())
    del x, buffer

    p = torch.zeros(cols, dtype=torch.float16, device=device)
    dy, dx = torch.ones_like(p), torch.full((cols + 9,), 7.0, dtype=torch.float16, device=device)
    p[-tail:], dy[-tail:] = 1 / 32, step.half()
    lib.check(lib.fn["softmax_bwd"](hiplib.F16, p.data_ptr(), dy.data_ptr(), dx.data_ptr(), 1, cols, cols, cols, cols, stream))
    assert bool((dx[cols:] == 7.0).all()) and bool((dx[:cols - tail] == 0).all())
    assert torch.equal(dx[cols - tail:cols], ((step - step.sum() / 32) / 32).half())      # exact in f32
    del p, dy, dx
    torch.cuda.empty_cache()


def test_softmax_more_rows_than_a_launch_has_workgroups(device):
    """Rows of one workgroup each, more of them than a launch may have (2^32 threads), all reading one row of x."""
    rows, cols = (1 << 24) + 5, 4097
    announce("softmax most rows", rows, cols)
    if torch.cuda.mem_get_info(device)[0] < 160e9:
        pytest.skip("the result takes 137 GB of device memory")
    x = torch.randn(cols, generator=torch.Generator(device=device).manual_seed(3), device=device).bfloat16()
    y = torch.empty((rows, cols), dtype=torch.bfloat16, device=device)
    lib = hiplib.library()
    lib.check(lib.fn["softmax_fwd"](hiplib.BF16, x.data_ptr(), y.data_ptr(), rows, cols, 0, cols,
                                    torch.cuda.current_stream().cuda_stream))
    want = torch.softmax(x.double(), dim=0)
    assert_16bit(y[0].double().cpu().numpy(), want.cpu().numpy(), rel=2.0 ** -7, abs_=2.0 ** -24)
    for at in range(0, rows, 1 << 20):
        assert bool((y[at:at + (1 << 20)] == y[0]).all())
    del y
    torch.cuda.empty_cache()
