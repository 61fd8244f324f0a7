"""GPU parity of the bf16 GEMM.

Bars: bf16 outputs within rel 2e-2 / abs 1e-2 of the fp32-accumulated reference (the oracle,
and hipBLASLt through torch in float32 on the full 8192^3 config); bit-exact on inputs whose
products and partial sums are exact in f32 (small integers, permutation matrices)."""
import numpy as np
import pytest
import torch

import intent_amd as intent
import oracle
from intent_amd.examples import inputs
from intent_amd.examples.kernels.contraction.gemm import Activation, bf16_gemm, gemm, gemm_f32, quantized_gemm
from tests.gpu_util import announce, assert_16bit, bf16_tensor_bits, bf16_to_f32, to_bf16_tensor

pytestmark = pytest.mark.gpu


def run(device, a_bits, b_bits):
    c = intent.jit(bf16_gemm, backend="hip").run(to_bf16_tensor(a_bits, device), to_bf16_tensor(b_bits, device))
    return bf16_tensor_bits(c)


def test_gemm_golden(device, golden):
    announce("gemm golden")
    g = golden("gemm")
    c = bf16_to_f32(run(device, g["gemm_a"], g["gemm_b"]))
    assert_16bit(c, g["gemm_c64"])
    assert (run(device, g["gemm_int_a"], g["gemm_int_b"]) == g["gemm_int_c"]).all()


@pytest.mark.parametrize("m,n,k", [(256, 256, 64), (300, 520, 72), (1, 8, 8), (513, 264, 1000), (33, 17, 19),
                                   (64, 24, 4096), (1024, 2048, 512), (7, 3, 0)])
def test_gemm_shapes(device, m, n, k):
    announce("gemm", m, n, k)
    a, b = inputs.gemm_bf16(seed=m + n + k, m=m, n=n, k=k)
    c = run(device, a, b)
    want = oracle.gemm_bf16(a, b)
    assert_16bit(bf16_to_f32(c), bf16_to_f32(want))
    diff = np.abs(c.astype(np.int32) - want.astype(np.int32))
    assert (diff <= 2).mean() > 0.999 if diff.size else True


def test_gemm_exact_cases(device):
    announce("gemm exact")
    rng = np.random.default_rng(11)
    a = inputs._bf16_bits(rng.integers(-8, 9, (512, 768)).astype(np.float32))
    b = inputs._bf16_bits(rng.integers(-8, 9, (768, 256)).astype(np.float32))
    assert (run(device, a, b) == oracle.gemm_bf16(a, b)).all()          # exact integer sums
    perm = rng.permutation(512)
    p = inputs._bf16_bits(np.eye(512, dtype=np.float32)[perm])
    x = inputs.uniform(rng, (512, 264), -1, 1, "bf16")
    assert (run(device, p, x) == x[perm]).all()                          # rows permuted exactly
    perm2 = rng.permutation(264)
    q = inputs._bf16_bits(np.eye(264, dtype=np.float32)[perm2])
    assert (run(device, x, q) == x[:, np.argsort(perm2)]).all()         # columns permuted exactly


def test_gemm_strided_views(device):
    announce("gemm strided")
    a, b = inputs.gemm_bf16(seed=3, m=384, n=640, k=512)
    big_a = torch.zeros(384, 1024, dtype=torch.bfloat16, device=device)
    big_a[:, 256:768] = to_bf16_tensor(a, device)
    ta = big_a[:, 256:768]                                 # row stride 1024
    tb = to_bf16_tensor(np.ascontiguousarray(b.T), device).t()   # inner stride 512: staged copy
    c = intent.jit(bf16_gemm, backend="hip").run(ta, tb)
    assert (bf16_tensor_bits(c) == run(device, a, b)).all()
    out = torch.empty(640, 384, dtype=torch.bfloat16, device=device).t()   # strided output
    intent.jit(bf16_gemm, backend="hip")(ta, to_bf16_tensor(b, device), out)
    assert (bf16_tensor_bits(out.contiguous()) == run(device, a, b)).all()


def test_gemm_config3_full(device):
    announce("gemm config 3 8192^3")
    a, b = inputs.gemm_bf16()
    ta, tb = to_bf16_tensor(a, device), to_bf16_tensor(b, device)
    c = intent.jit(bf16_gemm, backend="hip").run(ta, tb)
    ref = torch.matmul(ta.float(), tb.float())             # fp32-accumulated library reference
    err = (c.float() - ref).abs()
    assert bool((err <= 1e-2 + 2e-2 * ref.abs()).all())
    rows = np.array([0, 1, 255, 256, 1000, 4095, 4096, 5555, 8190, 8191])
    want = oracle.gemm_bf16(np.ascontiguousarray(a[rows]), b)
    got = bf16_tensor_bits(c)[rows]
    assert_16bit(bf16_to_f32(got), bf16_to_f32(want))
    assert (np.abs(got.astype(np.int32) - want.astype(np.int32)) <= 2).mean() > 0.999


def check_product(device, m, n, k, workspace):
    """Against the oracle, and exact on small integers whose sums f32 holds (an element read from the wrong place,
    twice or not at all shows); rows of NaN in A and columns of NaN in B stay in their own row and
    column of C, so no padding row, column or K group reaches a result."""
    announce("gemm", m, n, k, workspace)
    kernel = intent.jit(bf16_gemm, backend="hip", backend_options={"workspace": workspace})
    call = lambda a, b: bf16_tensor_bits(kernel.run(to_bf16_tensor(a, device), to_bf16_tensor(b, device)))  # noqa: E731
    a, b = inputs.gemm_bf16(seed=m + n + k, m=m, n=n, k=k)
    got, want = call(a, b), oracle.gemm_bf16(a, b)
    assert_16bit(bf16_to_f32(got), bf16_to_f32(want))
    assert (np.abs(got.astype(np.int32) - want.astype(np.int32)) <= 2).mean() > 0.999
    rng = np.random.default_rng(m * n + k)
    ints = [inputs._bf16_bits(rng.integers(-2, 3, shape).astype(np.float32)) for shape in ((m, k), (k, n))]
    assert (call(*ints) == oracle.gemm_bf16(*ints)).all()
    a[m - 1, k - 1] = b[0, n - 1] = 0x7FC0
    nan = np.isnan(bf16_to_f32(call(a, b)))
    expected = np.zeros((m, n), bool)
    expected[m - 1, :] = expected[:, n - 1] = True
    assert (nan == expected).all()


# 64 x 64 and 128 x 128 tiles (up to 128, 256 and 512 of the latter) and 256 x 256 ones, each with its last row and column
# of tiles partly filled, K below one step, off it by every multiple of 8, and divided over workgroups;
# then operands the DMA does not take: odd extents, one below and above a tile, every K remainder class.
@pytest.mark.parametrize("m,n,k", [(129, 8, 8), (200, 72, 56), (192, 64, 64), (130, 1000, 136), (300, 264, 1032),
                                   (257, 136, 2056), (1500, 1400, 72), (1409, 1416, 192), (2300, 2200, 40),
                                   (2310, 2304, 128), (3000, 3080, 8), (2900, 3088, 104), (2900, 3072, 192),
                                   (1, 1, 1), (63, 65, 7), (65, 63, 9), (130, 129, 63), (64, 200, 65), (129, 77, 1027),
                                   (200, 131, 2049), (33, 8, 17)])
@pytest.mark.parametrize("workspace", ["prepare", "static"])
def test_gemm_tiles(device, m, n, k, workspace):
    """As test_gemm_few_rows; the last element of each operand and of the result lies at its buffer's end."""
    check_product(device, m, n, k, workspace)


@pytest.mark.parametrize("lda,ldb,ldc,offset", [(8, 0, 0, 0), (3, 0, 0, 0), (0, 5, 0, 0), (0, 0, 1, 0), (0, 0, 4, 0),
                                                (0, 0, 0, 1), (8, 8, 4, 8), (1, 2, 3, 3)])
@pytest.mark.parametrize("m,n,k", [(40, 64, 72), (200, 136, 72), (1500, 1400, 64)])
def test_gemm_strides_and_offsets(device, m, n, k, lda, ldb, ldc, offset):
    """Row strides `lda`, `ldb`, `ldc` elements past the row, and operands `offset` elements into their buffers: whichever
    kernel takes a layout, the result is that of the contiguous operands up to the order of the f32 sums,
    and the result's buffer is unchanged outside it."""
    announce("gemm layouts", m, n, k, lda, ldb, ldc, offset)
    rng = np.random.default_rng(m + n + k)
    ints = [rng.integers(-2, 3, shape).astype(np.float32) for shape in ((m, k), (k, n))]

    def place(data, rows, cols, pad):
        base = torch.full((rows * (cols + pad) + offset,), 9.0, dtype=torch.bfloat16, device=device)
        view = base[offset:].view(rows, cols + pad)[:, :cols]
        if data is not None:
            view.copy_(torch.from_numpy(data).to(device))
        return base, view

    (_, a), (_, b), (base, c) = place(ints[0], m, k, lda), place(ints[1], k, n, ldb), place(None, m, n, ldc)
    intent.jit(bf16_gemm, backend="hip")(a, b, c)
    want = torch.from_numpy(ints[0] @ ints[1]).to(device).to(torch.bfloat16)     # exact in f32
    assert torch.equal(c, want)
    c.fill_(9.0)
    assert bool((base == 9.0).all())


# The few-row kernel: row blocks of 16, 32 and 64 and their edges, two row blocks (m > 64), column
# counts below and past one 64-column workgroup, K below one 64-deep unit, past it by every multiple
# of 8, and long enough that K is divided over workgroups (from 2048 rows on; 2056 leaves a tail).
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (15, 64, 24), (16, 72, 40), (17, 56, 64), (32, 520, 56), (33, 136, 72),
                                   (64, 64, 120), (65, 200, 1000), (128, 72, 520), (1, 24, 2048), (31, 1000, 2056),
                                   (100, 136, 4104), (128, 8, 2048), (3, 16384, 2048)])
@pytest.mark.parametrize("workspace", ["prepare", "static"])
def test_gemm_few_rows(device, m, n, k, workspace):
    check_product(device, m, n, k, workspace)


# f16 on every kernel (few rows, 64 x 64 tiles, both with K divided; 128 x 128 with four and two stages; 256 x 256; through
# registers, with K divided too), the activation applied after the whole sum.
@pytest.mark.parametrize("m,n,k", [(32, 1000, 2056), (100, 72, 4104), (257, 136, 2056), (1500, 1400, 72), (2300, 2200, 40),
                                   (3000, 3080, 40), (200, 131, 2049)])
@pytest.mark.parametrize("activation", [Activation.NONE, Activation.RELU])
def test_gemm_f16_kernels_and_activation(device, m, n, k, activation):
    """Against the oracle and exact on small integers, half of whose sums are negative; NaN in the last row of A and the last column
    of B passes the activation and stays in its own row and column."""
    announce("gemm f16 kernels", m, n, k, activation.name)
    kernel = intent.jit(gemm, backend="hip", constexprs={"ACTIVATION": activation})
    call = lambda x, y: kernel.run(torch.from_numpy(x).to(device), torch.from_numpy(y).to(device)).cpu().numpy()  # noqa: E731
    rng = np.random.default_rng(m + n + k)
    relu = activation == Activation.RELU
    a, b = inputs.normal(rng, (m, k), "f16"), inputs.normal(rng, (k, n), "f16")
    got, want = call(a, b), oracle.gemm16(a, b, relu=relu)
    assert_16bit(got, want)
    assert (np.abs(got.view(np.int16).astype(np.int32) - want.view(np.int16).astype(np.int32))[np.abs(want) > 1e-2] <= 2).mean() > 0.999
    ints = [rng.integers(-2, 3, shape).astype(np.float16) for shape in ((m, k), (k, n))]
    got = call(*ints)
    assert np.array_equal(got, oracle.gemm16(*ints, relu=relu)) and (got < 0).any() == (not relu)
    a[m - 1, k - 1] = b[0, n - 1] = np.nan
    expected = np.zeros((m, n), bool)
    expected[m - 1, :] = expected[:, n - 1] = True
    assert (np.isnan(call(a, b)) == expected).all()


# (m, n, k): the kernel, its threads and its LDS, on both sides of each line of the dispatch.
KERNELS = {(16, 72, 64): ("gemm_skinny", 512, 8 * 16 * 68 * 4), (17, 72, 64): ("gemm_skinny", 512, 8 * 32 * 68 * 4),
           (128, 72, 64): ("gemm_skinny", 512, 8 * 64 * 68 * 4), (129, 72, 64): ("gemm_small", 256, 4 * 16384),
           (129, 72, 65): ("gemm_small", 256, 2 * 16384), (1, 1, 1): ("gemm_small", 256, 2 * 16384),
           (1024, 2048, 64): ("gemm_small", 256, 4 * 16384), (1025, 2048, 64): ("gemm_small", 512, 4 * 32768),
           (2048, 2048, 64): ("gemm_small", 512, 4 * 32768), (2049, 2048, 64): ("gemm_small", 256, 2 * 32768),
           (4096, 2048, 8): ("gemm_small", 256, 2 * 32768), (4097, 2048, 8): ("gemm_mfma", 512, 5 * 32768),
           (4097, 2048, 64): ("gemm_mfma", 512, 5 * 32768), (4097, 2049, 64): ("gemm_small", 256, 2 * 16384)}


@pytest.mark.parametrize("m,n,k", KERNELS)
@pytest.mark.parametrize("kind", ["bf16", "f16", "quantize"])
def test_gemm_observes_the_kernel_that_ran(device, m, n, k, kind):
    announce("gemm observation", m, n, k, kind)
    dtype = torch.bfloat16 if kind == "bf16" else torch.float16
    args = [torch.zeros(shape, dtype=dtype, device=device) for shape in ((m, k), (k, n))]
    if kind == "quantize":
        args += [torch.zeros(n, device=device), torch.zeros(m, n, dtype=dtype, device=device), torch.ones(n, device=device)]
    kernel = intent.jit({"bf16": bf16_gemm, "f16": gemm, "quantize": quantized_gemm}[kind], backend="hip",
                        **({"constexprs": {"ACTIVATION": Activation.RELU}} if kind == "f16" else {}))
    call = kernel.prepare(*args)
    call.launch()
    facts = {r.name: r.value for r in call.observation.resources}
    name, threads, lds = KERNELS[m, n, k]
    assert call.observation.kernel == name + {"bf16": "<bf16>", "f16": "<f16>", "quantize": "<f16,quantize>"}[kind]
    assert facts["block_threads"] == threads and facts["lds_bytes"] == lds


def split_product(device, kind):
    """A prepared product whose K is divided over workgroups, its result's buffer, the exact result, and its workspace's bytes."""
    g = torch.Generator(device=device).manual_seed(5)
    a, b = (torch.randint(-3, 4, shape, generator=g, device=device).float() for shape in ((16, 4096), (4096, 640)))
    want, c = a @ b, torch.zeros(16, 640, device=device)          # exact: whole sums below 2^24
    if kind == "bf16":
        a, b, c, want = a.bfloat16(), b.bfloat16(), c.bfloat16(), want.bfloat16()
    kernel = intent.jit(bf16_gemm if kind == "bf16" else gemm_f32, backend="hip")
    call = kernel.prepare(a, b, outputs=(c,))
    size = dict(call.inspect_configurations()[0].configuration)["workspace_bytes"]
    assert size > 0
    return call, (a, b), c, want, size


@pytest.mark.parametrize("kind", ["bf16", "f32"])
def test_split_gemm_on_another_stream(device, kind):
    """A prepared call launched on another stream and dropped before that stream comes to it: the memory it gives back is
    another tensor's by then and stays that tensor's."""
    announce("split gemm, other stream", kind)
    call, operands, c, want, size = split_product(device, kind)
    busy = torch.randn(4096, 4096, device=device)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(20):
            busy = busy @ busy * 1e-3
        call.launch()
        call.launch()
    del call
    others = [torch.full((size,), 77, dtype=torch.uint8, device=device) for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(c, want) and all(bool((o == 77).all()) for o in others)


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("kind", ["bf16", "f32"])
def test_split_gemm_graph_outlives_its_call(device, kind, own_stream):
    """A graph that captured a prepared call, whether the call was prepared on the capturing stream or not, is replayed after
    the call was dropped and its memory given away."""
    announce("split gemm, graph", kind, own_stream)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream if own_stream else torch.cuda.current_stream()):
        call, (a, b), c, want, size = split_product(device, kind)
        call.launch()
    torch.cuda.synchronize()
    assert torch.equal(c, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            call.launch()
        del call
        others = [torch.full((size,), 77, dtype=torch.uint8, device=device) for _ in range(3)]
    others += [torch.full((size,), 77, dtype=torch.uint8, device=device) for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(3):
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want) and all(bool((o == 77).all()) for o in others)


# One row against more columns, and one column against more rows, than workgroups of one tile each fit one axis of a launch
# (2^32 threads): the few-row kernel, and 64 x 64 tiles through registers.
@pytest.mark.parametrize("m,n,k", [(1, (1 << 29) + 72, 8), ((1 << 30) - 1, 1, 1)])
def test_gemm_longest_extents(device, m, n, k):
    announce("gemm longest extents", m, n, k)
    g = torch.Generator(device=device).manual_seed(11)
    small = lambda *shape: torch.randint(-3, 4, shape, generator=g, device=device, dtype=torch.int8)  # noqa: E731
    a, b = small(m, k), small(k, n)
    c = intent.jit(bf16_gemm, backend="hip").run(a.bfloat16(), b.bfloat16())
    step = 1 << 26
    for at in range(0, max(m, n), step):        # small integers: exact
        rows, columns = (a[at:at + step], b) if m > n else (a, b[:, at:at + step])
        want = sum(rows[:, i:i + 1] * columns[i:i + 1] for i in range(k))
        assert torch.equal(c[at:at + step] if m > n else c[:, at:at + step], want.bfloat16())
