"""Differential tests: the HIP library (through the C ABI) against the CPU oracle on identical
seeded bytes, in the manner of crates/forja-metal/tests/*.rs (CpuBackend = reference,
candidate = device backend).  Integer results are bit-exact; float results meet the elementwise
rel 1e-2 / abs 1e-2 bar and the reference's normwise bound for the dtype."""
import math

import numpy as np
import pytest

from forja_amd import programs
from forja_amd.core import (BackendError, BinOp, CommandList, DType, Inst, Layout, Op, Program,
                            ProgramBuilder, ProgramKind, RedOp, Slice, Status, UnOp, ValueType,
                            INTO_PAGES, OUT_OF_PAGES)
from oracle import cpu_backend as orc
from tests.helpers import (Quantised, assert_close, from_f32, normal_bf16, to_f32, upload,
                           upload_raw)
from tests.test_oracle_golden import paged_case, top_k_case

pytestmark = pytest.mark.gpu


def run(backend, commands):
    backend.submit(commands).wait()


def coarser(*dtypes):
    """The dtype whose tolerance judges an attention output: the reference holds f32 outputs
    computed from f16 or bf16 pools to the pools' tolerance (crates/forja-metal/tests/paged.rs:982-988)."""
    return max(dtypes, key=[DType.F32, DType.F16, DType.BF16].index)


def compare(cpu, hip, cpu_tensor, hip_tensor, bar=None, **kw):
    """`bar`: the dtype whose tolerance applies to float outputs (their own when not given)."""
    dtype = cpu_tensor.dtype
    a, b = cpu.read(cpu_tensor), hip.read(hip_tensor)
    if dtype in (DType.U32, DType.I32):
        assert a == b
    else:
        assert_close(to_f32(b, dtype), to_f32(a, dtype), coarser(dtype, bar or dtype), **kw)


def differential(cpu, hip, build, expect_error=None, **kw):
    """build(backend) -> (commands, [outputs]); runs on both and compares every output."""
    results = []
    for backend in (cpu, hip):
        commands, outputs = build(backend)
        error = None
        try:
            run(backend, commands)
        except BackendError as e:
            error = e
        results.append((outputs, error))
    (cpu_out, cpu_err), (hip_out, hip_err) = results
    if expect_error is None:
        assert cpu_err is None and hip_err is None, (cpu_err, hip_err)
    else:
        assert cpu_err is not None and hip_err is not None
        assert hip_err.status in expect_error
    for a, b in zip(cpu_out, hip_out):
        compare(cpu, hip, a, b, **kw)
    return results


# ------------------------------------------------------------------ device info / storage

def test_device_is_gfx950_and_storage_round_trips(hip):
    info = hip.device_info()
    assert info["family"].startswith("gfx950"), info
    assert info["wavefront"] == 64
    t = hip.alloc(DType.U32, (5, 7))
    assert hip.read(t) == bytes(5 * 7 * 4)                      # zero-initialised
    data = np.arange(35, dtype=np.uint32)
    hip.write(t, data.tobytes())
    assert np.frombuffer(hip.read(t), np.uint32).tolist() == data.tolist()
    view = t.slice([Slice(1, 2, 2), Slice(0, 3, 3)]).permute([1, 0])
    assert np.frombuffer(hip.read(view), np.uint32).tolist() == data.reshape(5, 7)[1::2, 0::3][:2, :3].T.ravel().tolist()
    with pytest.raises(BackendError):
        hip.write(view, bytes(24))                              # non-contiguous write refused
    hip.release(t)
    with pytest.raises(BackendError):
        hip.read(t)                                             # released allocation


@pytest.mark.parametrize("first,length", [(0, 16), (4, 20), (1, 16), (16, 3), (7, 16377), (0, 16384), (0, 16385), (4, 24572),
                                          (8, 65528), (0, 65536), (3, 65537)])
def test_bytes_moved_to_and_from_a_buffer(hip, first, length):
    """Pieces of 16, 4 and 1 bytes by alignment, and both sides of the sizes that a kernel moves."""
    t = hip.alloc(DType.U32, (1 << 15,))
    rng = np.random.default_rng(length)
    expected = bytearray(rng.bytes(1 << 17))
    hip.write(t, bytes(expected))
    data = rng.bytes(length)
    assert hip._lib.fh_write(hip._handle, t.buffer, first, data, length) == 0
    expected[first:first + length] = data
    assert hip.read_buffer_range(t.buffer, first, first + length) == data
    assert hip.read_buffer_range(t.buffer, 0, 1 << 17) == bytes(expected)
    view = t.narrow(0, first, (length + 3) // 4)   # (gathered on the device)
    assert hip.read(view) == bytes(expected[4 * first:4 * (first + (length + 3) // 4)])
    hip.release(t)


def test_error_records_are_clear_again_after_an_error(hip):
    """Records of a submission without an error are used again as they are, those of one that raised one are cleared."""
    ids, out, table = hip.alloc(DType.U32, (1,)), hip.alloc(DType.BF16, (1, 64)), Quantised(68, 0, (4, 64)).upload(hip)
    commands = CommandList()
    for _ in range(3):
        commands.dispatch(Op.quant_embed(4, 64), [*table, ids], out)
    for index in (3, 9, 2, 1, 7, 8, 0):
        hip.write_array(ids, np.array([index], np.uint32))
        if index < 4:
            run(hip, commands)
            continue
        with pytest.raises(BackendError) as info:
            run(hip, commands)
        assert info.value.status == Status.INDEX_OUT_OF_RANGE and info.value.index == index and info.value.dispatch == 0


def test_submit_refuses_foreign_tensors_and_bad_shapes(hip):
    x = hip.alloc(DType.BF16, (4, 64))
    out = hip.alloc(DType.BF16, (4, 8))
    packed = hip.alloc(DType.U32, (8, 8))
    scales, biases = hip.alloc(DType.BF16, (8, 1)), hip.alloc(DType.BF16, (8, 1))
    wrong = hip.alloc(DType.BF16, (4, 9))
    commands = CommandList()
    commands.dispatch(Op.quant_matmul(4, 64), [x, packed, scales, biases], wrong)
    with pytest.raises(BackendError) as info:
        hip.submit(commands)
    assert info.value.status == Status.INVALID_INPUT
    hip.release(scales)
    commands = CommandList()
    commands.dispatch(Op.quant_matmul(4, 64), [x, packed, scales, biases], out)
    with pytest.raises(BackendError):
        hip.submit(commands)


def test_seeded_fill_matches_the_host_generator_bit_for_bit(cpu, hip):
    def build(backend):
        words = backend.alloc(DType.U32, (3, 1000))
        uniform = backend.alloc(DType.BF16, (777,))
        normal = backend.alloc(DType.BF16, (5, 999))
        normal32 = backend.alloc(DType.F32, (4096,))
        commands = CommandList()
        commands.dispatch(Op.fill_seeded(0, 0x1234_5678_9abc, 3, first=17), [], words)
        commands.dispatch(Op.fill_seeded(1, 99, 4, lo=0.001, hi=0.02), [], uniform)
        commands.dispatch(Op.fill_seeded(2, 99, 5, first=1 << 20), [], normal)
        commands.dispatch(Op.fill_seeded(2, 7, 6), [], normal32)
        return commands, [words, uniform, normal, normal32]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    for a, b in zip(cpu_out, hip_out):
        assert cpu.read(a) == hip.read(b)


def test_kernel_timers_follow_the_selected_classes(hip):
    """fh_profile_select: only the selected kernel classes are timed (class 6 = the kernels of a
    dense quantised product)."""
    weights = Quantised(20, 1, (64, 256))
    x = upload(hip, normal_bf16(20, 2, (8, 256)), DType.BF16)
    out = hip.alloc(DType.BF16, (8, 64))
    commands = CommandList()
    commands.dispatch(Op.quant_matmul(4, 64), [x, *weights.upload(hip)], out)
    try:
        hip.profile_enable(1)
        for mask, expected in ((1 << 4, 0), (1 << 6, 1), (0xffffffff, 1)):
            hip.profile_select(mask)
            hip.profile_reset()
            run(hip, commands)
            nanoseconds, launches = hip.profile_read(6)
            assert launches == expected and (nanoseconds > 0) == (expected > 0)
        # fh_profile_sample: one launch in three is timed
        hip.profile_sample(3)
        hip.profile_reset()
        for _ in range(7):
            run(hip, commands)
        assert hip.profile_read(6)[1] == 3
    finally:
        hip.profile_sample(1)
        hip.profile_select(0xffffffff)
        hip.profile_enable(0)


# ------------------------------------------------------------------ quantised matmul

QMM_CASES = [
    # rows, N, K, bits, group, activation dtype
    (1, 64, 64, 4, 64, DType.F32),
    (7, 48, 128, 4, 64, DType.BF16),
    (33, 40, 256, 4, 64, DType.BF16),
    (4, 4096, 1024, 4, 64, DType.BF16),     # C0 stacked qkv
    (4, 1024, 3072, 4, 64, DType.BF16),     # C0 down
    (128, 160, 2048, 4, 64, DType.BF16),    # C3 row count, narrow N
    (128, 128, 2048, 8, 64, DType.BF16),    # router (q8 in the reference engine)
    (5, 24, 256, 4, 32, DType.F16),
    (3, 24, 256, 8, 128, DType.F32),
    (40, 72, 192, 4, 64, DType.BF16),
    (1, 2048, 2048, 4, 64, DType.BF16),
    (64, 100, 512, 4, 64, DType.BF16),      # column tail inside a wave
    (130, 96, 768, 4, 64, DType.BF16),      # row tail across row blocks
    (8, 512, 4096, 4, 64, DType.BF16),
    (128, 5120, 2048, 4, 64, DType.BF16),   # C3 stacked qkv: packed-activation path, 2 splits
    (128, 2048, 4096, 4, 64, DType.BF16),   # C3 o_proj: 4 splits
    (100, 130, 2048, 4, 64, DType.BF16),    # row and column tails, 8 splits
    (64, 96, 256, 4, 64, DType.BF16),       # a single group per wave, no split
    (65, 32, 3072, 4, 64, DType.BF16),      # 12 splits
    (192, 4096, 2048, 4, 64, DType.BF16),   # more rows than the decode path takes: tiled GEMM
    (257, 300, 512, 4, 64, DType.BF16),     # GEMM with row and column tails
    (1000, 96, 256, 4, 64, DType.BF16),     # GEMM, a single column tile, four row tiles
    (512, 1024, 2048, 4, 64, DType.BF16),   # GEMM, whole tiles
    # f32 / f16 activations and 8-bit weights: the f32 vector-ALU kernel
    (8, 5120, 2048, 4, 64, DType.F32),      # the qwen3-coder engine's decode batch: stacked qkv
    (8, 128, 2048, 8, 64, DType.F32),       # its 8-bit router
    (128, 2048, 4096, 4, 64, DType.F32),    # o_proj on a full decode batch
    (19, 130, 1056, 4, 32, DType.F16),      # row, column and wave tails; 33 pieces over 8 waves
    (70, 200, 384, 8, 128, DType.F16),
    (3, 70, 32, 4, 32, DType.F32),          # a single piece: one wave
    (300, 96, 256, 8, 32, DType.BF16),      # prefill rows with 8-bit weights
]


@pytest.mark.parametrize("rows,n,k,bits,group,dtype", QMM_CASES)
def test_quant_matmul(cpu, hip, rows, n, k, bits, group, dtype):
    weights = Quantised(21, 100 + n + k, (n, k), bits=bits, group=group)
    x_values = normal_bf16(21, 7, (rows, k))

    def build(backend):
        x = upload(backend, x_values, dtype)
        packed, scales, biases = weights.upload(backend)
        out = backend.alloc(dtype, (rows, n))
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(bits, group), [x, packed, scales, biases], out)
        return commands, [out]
    differential(cpu, hip, build)


@pytest.mark.parametrize("rows,n,k,residual", [(8, 5120, 2048, False), (1, 2048, 768, False), (16, 768, 2048, True),
                                               (20, 2048, 1024, True), (31, 96, 512, False),
                                               (8, 2048, 4096, True), (24, 512, 4096, False)])   # o_proj: two K ranges
def test_quant_matmul_on_f32_activations_that_use_their_whole_mantissa(cpu, hip, rows, n, k, residual):
    """The engines' activations are f32 (engines/qwen3-coder/src/lib.rs:296-437) and carry 24
    significant bits, unlike the bf16-valued inputs of the cases above: a kernel that rounded them
    to bf16, or to two bf16 pieces, on its way to the matrix cores would miss the f32 bar."""
    weights = Quantised(25, n + k, (n, k))
    x_values = orc.fill_normal_f32(25, 1, rows * k).reshape(rows, k)
    extra_values = orc.fill_normal_f32(25, 2, rows * n).reshape(rows, n)

    def build(backend):
        x = upload(backend, x_values, DType.F32)
        out = backend.alloc(DType.F32, (rows, n))
        commands = CommandList()
        if residual:
            extra = upload(backend, extra_values, DType.F32)
            add = backend.prepare_epilogue(programs.add_elements())
            commands.dispatch_epilogue(Op.quant_matmul(4, 64), [x, *weights.upload(backend)], out, add, [extra])
        else:
            commands.dispatch(Op.quant_matmul(4, 64), [x, *weights.upload(backend)], out)
        return commands, [out]
    differential(cpu, hip, build)


@pytest.mark.parametrize("rows,k,experts,n,inner", [(8, 8, 128, 768, 2048), (3, 4, 16, 512, 1024), (40, 2, 64, 256, 512)])
def test_routed_products_on_f32_activations_that_use_their_whole_mantissa(cpu, hip, rows, k, experts, n, inner):
    """The MoE block of a small decode batch in the engine's dtypes: gate/up pair with SwiGLU, the
    down projection as a weighted sum with the residual, all f32."""
    gate = Quantised(26, 1, (n, inner), experts=experts)
    up = Quantised(26, 11, (n, inner), experts=experts)
    down = Quantised(26, 21, (inner, n), experts=experts)
    indices = routed_case(26, rows, k, experts, n, inner)
    x_values = orc.fill_normal_f32(26, 40, rows * inner).reshape(rows, inner)
    logits = orc.fill_normal_f32(26, 41, rows * k).reshape(rows, k)
    w_values = np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True)
    residual_values = orc.fill_normal_f32(26, 42, rows * inner).reshape(rows, inner)

    def build(backend):
        x = upload(backend, x_values, DType.F32)
        idx = upload(backend, indices, DType.U32)
        g, u, d = gate.upload(backend), up.upload(backend), down.upload(backend)
        plain = backend.alloc(DType.F32, (rows, k, n))
        activated = backend.alloc(DType.F32, (rows, k, n))
        combined = backend.alloc(DType.F32, (rows, inner))
        weights = upload(backend, w_values, DType.F32)
        residual = upload(backend, residual_values, DType.F32)
        swiglu = backend.prepare_epilogue(programs.silu_mul_elements())
        add = backend.prepare_epilogue(programs.add_elements())
        commands = CommandList()
        commands.dispatch(Op.gather_quant_matmul(4, 64), [x, *g, idx], plain)
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [x, *g, *u, idx], activated, swiglu, [])
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [activated, *d, idx, weights], combined,
                                   add, [residual])
        return commands, [plain, activated, combined]
    differential(cpu, hip, build)


@pytest.mark.parametrize("rows,n,k,bits,dtype,padded", [
    # row tiles of 16, 32, 48 and 64 and their remainders; 16-column tiles past a block's edge; K ranges
    # of an odd number of 256-value quads; K that no other matrix-core kernel for few rows takes
    (1, 8224, 1280, 4, DType.BF16, False), (9, 144, 1280, 4, DType.BF16, True),
    (17, 272, 6400, 4, DType.BF16, False), (33, 16, 256, 4, DType.BF16, True),
    (48, 400, 3328, 4, DType.BF16, False), (49, 128, 1280, 4, DType.BF16, False),
    (64, 144, 2304, 4, DType.BF16, True), (127, 256, 3840, 4, DType.BF16, False),
    # f32 rows: tiles of 32, 4- and 8-bit weights
    (33, 272, 256, 4, DType.F32, True), (65, 528, 1280, 4, DType.F32, False),
    (9, 16, 768, 8, DType.F32, False), (70, 272, 2048, 8, DType.F32, True),
])
def test_quant_matmul_in_row_tiles(cpu, hip, rows, n, k, bits, dtype, padded):
    """`padded`: results into rows that no 16-byte store fits.  f32 inputs use their whole mantissa."""
    weights = Quantised(27, 300 + n + k, (n, k), bits=bits)
    x_values = orc.fill_normal_f32(27, 1, rows * k).reshape(rows, k) if dtype == DType.F32 else normal_bf16(27, 1, (rows, k))
    extra_values = normal_bf16(27, 2, (rows, n))

    def build(backend):
        x, extra = upload(backend, x_values, dtype), upload(backend, extra_values, dtype)
        plain, whole = backend.alloc(dtype, (rows, n)), upload(backend, np.zeros((rows, n + 3)), dtype)
        added = whole.narrow(1, 1, n) if padded else whole.narrow(1, 0, n)
        triple = weights.upload(backend)
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(bits, 64), [x, *triple], plain)
        commands.dispatch_epilogue(Op.quant_matmul(bits, 64), [x, *triple], added,
                                   backend.prepare_epilogue(programs.add_elements()), [extra])
        return commands, [plain, whole]
    differential(cpu, hip, build)


@pytest.mark.parametrize("rows,dtype", [(1, DType.BF16), (9, DType.BF16), (24, DType.BF16), (41, DType.BF16), (57, DType.BF16),
                                        (97, DType.BF16), (9, DType.F32), (40, DType.F32)])
def test_row_tiles_of_rows_with_something_between_them(cpu, hip, rows, dtype):
    """Rows of a wider tensor: NaNs behind each row's values and in the rows that follow (tiles of 16 to 64 rows, each with
    rows past the last one in its first or second eight)."""
    n = 8224 if rows == 1 else 1040     # (less for one row is a single tile product)
    weights = Quantised(27, 5, (n, 1280))
    values = np.full((rows + 64, 1280 + 64), np.nan, np.float32)
    values[:rows, :1280] = normal_bf16(27, 3, (rows, 1280))

    def build(backend):
        x = upload(backend, values, dtype).narrow(0, 0, rows).narrow(1, 0, 1280)
        out = backend.alloc(dtype, (rows, n))
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(4, 64), [x, *weights.upload(backend)], out)
        return commands, [out]
    _, (hip_out, _) = differential(cpu, hip, build)
    assert np.isfinite(to_f32(hip.read(hip_out[0]), dtype)).all()


@pytest.mark.parametrize("rows,n,k,dtype", [(17, 272, 6400, DType.BF16), (64, 400, 3328, DType.BF16),
                                            (33, 16, 256, DType.BF16), (40, 272, 1280, DType.F32)])
def test_row_tiles_under_an_epilogue_that_is_not_fused(cpu, hip, rows, n, k, dtype):
    """The product itself stays f32, of bf16 rows too: added up from several K ranges, and from one."""
    weights = Quantised(27, 300 + n + k, (n, k))
    x_values, extra_values = normal_bf16(27, 1, (rows, k)), normal_bf16(27, 2, (rows, n))
    builder = ProgramBuilder(ProgramKind.MAP)
    builder.output(0, builder.mul(builder.input(0), builder.input(1)))
    program = builder.finish()

    def build(backend):
        out = backend.alloc(dtype, (rows, n))
        commands = CommandList()
        commands.dispatch_epilogue(Op.quant_matmul(4, 64), [upload(backend, x_values, dtype), *weights.upload(backend)], out,
                                   backend.prepare_epilogue(program), [upload(backend, extra_values, dtype)])
        return commands, [out]
    differential(cpu, hip, build)


@pytest.mark.parametrize("rows,k,experts,n,inner,dtype", [
    (60, 8, 8, 144, 256, DType.BF16),      # 60 routes per expert: a 64-row tile and its remainder
    (130, 2, 5, 272, 512, DType.BF16),     # 52: columns past a block's edge, two quads
    (45, 4, 7, 784, 768, DType.BF16),      # odd numbers of quads
    (17, 8, 8, 144, 256, DType.F32), (70, 4, 7, 272, 768, DType.F32),
])
def test_routed_products_in_row_tiles(cpu, hip, rows, k, experts, n, inner, dtype):
    """More routes per expert than the K-split kernels take, with bad routes among them."""
    gate, up = (Quantised(28, 1 + i, (n, inner), experts=experts) for i in range(2))
    down = Quantised(28, 21, (512, inner), experts=experts)
    indices = routed_case(28, rows, k, experts, n, inner, bad=((3, 1, experts), (rows - 1, 0, experts + 7)))
    x_values, wide_values = normal_bf16(28, 40, (rows, inner)), normal_bf16(28, 43, (rows, k, inner))
    if dtype == DType.F32:
        x_values = orc.fill_normal_f32(28, 40, rows * inner).reshape(rows, inner)
    logits = orc.fill_normal_f32(28, 41, rows * k).reshape(rows, k)
    w_values = np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True)

    def pair(backend):
        x, idx = upload(backend, x_values, dtype), upload(backend, indices, DType.U32)
        activated = backend.alloc(dtype, (rows, k, n))
        commands = CommandList()
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [x, *gate.upload(backend), *up.upload(backend), idx],
                                   activated, backend.prepare_epilogue(programs.silu_mul_elements()), [])
        return commands, [activated]

    def summed(backend):
        x, idx = upload(backend, wide_values, dtype), upload(backend, indices, DType.U32)
        combined = backend.alloc(dtype, (rows, 512))
        commands = CommandList()
        commands.dispatch(Op.gather_quant_matmul(4, 64),
                          [x, *down.upload(backend), idx, upload(backend, w_values, dtype)], combined)
        return commands, [combined]

    for build in (pair, summed):
        differential(cpu, hip, build, expect_error={Status.INDEX_OUT_OF_RANGE, Status.DEVICE_ERROR_FLAG})


def rows_with_infinities(seed, rows, k, dtype):
    """Rows 1 to 5: an infinity of either sign, two that agree, two that do not, a NaN; row 6 (f32 only):
    values next to the largest of f32, whose sum over a group by 128 is past it."""
    values = orc.fill_normal_f32(seed, 1, rows * k).reshape(rows, k) if dtype == DType.F32 else normal_bf16(seed, 1, (rows, k))
    values[1, 7], values[2, k - 1], values[3, [0, 70]] = np.inf, -np.inf, np.inf
    values[4, 5], values[4, 200], values[5, 64] = np.inf, -np.inf, np.nan
    if dtype == DType.F32:
        values[6] *= np.float32(2.0 ** 120)
    return values


def same_kinds(expected, actual, dtype):
    """The same infinities and NaNs; elsewhere sums of the same products: f32 ones that differ by their order
    (1e-5 of the row's typical value, as in assert_close), rounded once more to bf16."""
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(expected), kind(actual))
    finite = np.isfinite(expected)
    assert finite.any() and not finite.all()
    e, a = (np.where(finite, v, 0).astype(np.float64) for v in (expected, actual))
    rel, of_row = (1e-4, 1e-5) if dtype == DType.F32 else (1e-2, 1e-2)
    typical = np.sqrt(np.mean(np.square(e), axis=tuple(range(1, e.ndim)), keepdims=True))
    assert np.all(np.abs(a - e) <= of_row * typical + rel * np.abs(e))


@pytest.mark.parametrize("rows,n,k,bits,dtype", [(40, 272, 1280, 4, DType.F32), (9, 4112, 2048, 4, DType.F32),
                                                 (40, 272, 768, 8, DType.F32), (48, 400, 3328, 4, DType.BF16)])
def test_infinities_in_row_tiles_reach_the_results_as_the_products_give_them(cpu, hip, rows, n, k, bits, dtype):
    weights, values = Quantised(27, 300 + n + k, (n, k), bits=bits), rows_with_infinities(29, rows, k, dtype)
    results = []
    for backend in (cpu, hip):
        out = backend.alloc(dtype, (rows, n))
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(bits, 64), [upload(backend, values, dtype), *weights.upload(backend)], out)
        run(backend, commands)
        results.append(to_f32(backend.read(out), dtype).reshape(rows, n))
    same_kinds(*results, dtype)


@pytest.mark.parametrize("dtype", [DType.F32, DType.BF16])
def test_infinities_in_routed_row_tiles(cpu, hip, dtype):
    rows, k, experts, n, inner = 70, 4, 7, 272, 768
    gate, up = (Quantised(28, 1 + i, (n, inner), experts=experts) for i in range(2))
    indices, values = routed_case(28, rows, k, experts, n, inner), rows_with_infinities(29, rows, inner, dtype)
    results = []
    for backend in (cpu, hip):
        x, idx = upload(backend, values, dtype), upload(backend, indices, DType.U32)
        plain, activated = backend.alloc(dtype, (rows, k, n)), backend.alloc(dtype, (rows, k, n))
        g, u = gate.upload(backend), up.upload(backend)
        commands = CommandList()
        commands.dispatch(Op.gather_quant_matmul(4, 64), [x, *g, idx], plain)
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [x, *g, *u, idx], activated,
                                   backend.prepare_epilogue(programs.silu_mul_elements()), [])
        run(backend, commands)
        results.append([to_f32(backend.read(out), dtype).reshape(rows, k, n) for out in (plain, activated)])
    for expected, actual in zip(*results):
        same_kinds(expected, actual, dtype)


def rows_of_every_magnitude(seed, rows, k):
    """Rows at 2^-130 to 2^120, a row of zeros, rows with groups of zeros, of values far below the row's
    others, and of 1e6 beside 1e-3; every value uses its whole mantissa."""
    values = orc.fill_normal_f32(seed, 1, rows * k).reshape(rows, k)
    exponents = (-130, -126, -120, -112, -100, -90, -60, 60, 100, 118)
    for row, exponent in enumerate(exponents):
        values[row] = np.ldexp(values[row], exponent)
    values[10], values[11, :64], values[12, 64:192] = 0, 0, values[12, 64:192] * np.float32(2.0 ** -120)
    values[13, ::2] *= np.float32(1e6)
    values[13, 1::2] *= np.float32(1e-3)
    values[14] = np.ldexp(np.abs(values[14]), -126)
    return values


def close_row_by_row(actual, values, dense, k):
    """Against 64 bits.  f32 sums of K products: K roundings of 2^-24 of the running sum, which add up like sqrt(K) in
    the 2-norm over a row of results.  The running sum is at most about the larger of the sum itself (terms of one
    sign) and the root of its squared terms; and every addition below 2^-126 rounds to 2^-149."""
    expected = values.astype(np.float64) @ np.swapaxes(dense, -1, -2)
    size = np.maximum(np.abs(expected), np.sqrt(values.astype(np.float64) ** 2 @ np.swapaxes(dense, -1, -2) ** 2))
    error = np.linalg.norm(actual - expected, axis=-1)
    bound = math.sqrt(k) * 2.0 ** -24 * np.linalg.norm(size, axis=-1) + 2.0 ** -149 * k ** 0.5 * dense.shape[-2] ** 0.5
    assert np.all(error <= bound), (error / bound).max()


@pytest.mark.parametrize("rows,n,k,bits", [(40, 272, 1280, 4), (16, 4112, 2048, 4), (40, 272, 768, 8)])
def test_f32_rows_of_every_magnitude_in_row_tiles(hip, rows, n, k, bits):
    weights, values = Quantised(27, 300 + n + k, (n, k), bits=bits), rows_of_every_magnitude(29, rows, k)
    out = hip.alloc(DType.F32, (rows, n))
    commands = CommandList()
    commands.dispatch(Op.quant_matmul(bits, 64), [upload(hip, values, DType.F32), *weights.upload(hip)], out)
    run(hip, commands)
    close_row_by_row(to_f32(hip.read(out), DType.F32).reshape(rows, n).astype(np.float64), values, weights.dequantised(), k)


def test_f32_rows_of_every_magnitude_in_routed_row_tiles(hip):
    rows, k, experts, n, inner = 70, 4, 7, 272, 768
    weights = Quantised(28, 1, (n, inner), experts=experts)
    indices, values = routed_case(28, rows, k, experts, n, inner), rows_of_every_magnitude(29, rows, inner)
    out = hip.alloc(DType.F32, (rows, k, n))
    commands = CommandList()
    commands.dispatch(Op.gather_quant_matmul(4, 64), [upload(hip, values, DType.F32), *weights.upload(hip),
                                                      upload(hip, indices, DType.U32)], out)
    run(hip, commands)
    actual, dense = to_f32(hip.read(out), DType.F32).reshape(rows, k, n).astype(np.float64), weights.dequantised()
    for slot in range(k):
        for row in range(rows):
            close_row_by_row(actual[row:row + 1, slot], values[row:row + 1], dense[indices[row, slot]], inner)


@pytest.mark.parametrize("dtype,bits,group", [(DType.F32, 4, 64), (DType.F16, 8, 32), (DType.BF16, 4, 128)])
def test_quant_matmul_with_f16_scales_and_a_residual_in_other_dtypes(cpu, hip, dtype, bits, group):
    """f16 affine parameters (the reference allows f16 or bf16, quantized.rs:78-121) and the
    residual-add epilogue on activations that are not bf16, plus an unrecognised epilogue."""
    rows, n, k = 40, 200, 768
    weights = Quantised(24, n + k, (n, k), bits=bits, group=group)
    x_values = normal_bf16(24, 1, (rows, k))
    extra_values = normal_bf16(24, 2, (rows, n))

    def build(backend):
        x = upload(backend, x_values, dtype)
        extra = upload(backend, extra_values, dtype)
        plain, added, scaled = (backend.alloc(dtype, (rows, n)) for _ in range(3))
        triple = weights.upload(backend, scale_dtype=DType.F16)
        b = ProgramBuilder(ProgramKind.MAP)
        b.output(0, b.mul(b.input(0), b.input(1)))
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(bits, group), [x, *triple], plain)
        commands.dispatch_epilogue(Op.quant_matmul(bits, group), [x, *triple], added,
                                   backend.prepare_epilogue(programs.add_elements()), [extra])
        commands.dispatch_epilogue(Op.quant_matmul(bits, group), [x, *triple], scaled,
                                   backend.prepare_epilogue(b.finish()), [extra])
        return commands, [plain, added, scaled]
    differential(cpu, hip, build)


@pytest.mark.parametrize("rows,n,k", [
    (129, 72, 512),       # the fewest K steps a part of the split takes, a column tile nearly empty
    (300, 200, 1536),     # ragged rows and columns
    (130, 70, 17408),     # more columns of group sums than a slot of LDS holds at a time
    (200, 8264, 512),     # 128 x 128 tiles, the fewest K steps
    (257, 5700, 2560),
    # rows held by 64, 128 and 256 threads, in four, ten and sixteen pieces each
    (133, 72, 2048), (133, 72, 4096), (131, 72, 8192), (129, 72, 8704), (129, 72, 20992),
])
@pytest.mark.parametrize("residual", [False, True])
def test_prefill_products_of_few_tiles(hip, rows, n, k, residual):
    """Products whose waves split K: against 64 bits.  A result is rounded once to bf16 (2^-9 of all of them together);
    what the products' operands are held to is in the test of their exactness."""
    weights, values, extra = Quantised(62, n + k, (n, k)), normal_bf16(62, 1, (rows, k)), normal_bf16(62, 2, (rows, n))
    out = hip.alloc(DType.BF16, (rows, n))
    commands, operands = CommandList(), [upload(hip, values, DType.BF16), *weights.upload(hip)]
    if residual:
        commands.dispatch_epilogue(Op.quant_matmul(4, 64), operands, out, hip.prepare_epilogue(programs.add_elements()),
                                   [upload(hip, extra, DType.BF16)])
    else:
        commands.dispatch(Op.quant_matmul(4, 64), operands, out)
    run(hip, commands)
    reference = values.astype(np.float64) @ weights.dequantised().T + (extra if residual else 0.0)
    error = to_f32(hip.read(out), DType.BF16).reshape(rows, n) - reference
    assert np.linalg.norm(error) <= (2.0 ** -9 + 2.0 ** -12) * np.linalg.norm(reference)
    # (element by element: the sums' own rounding is that of f16 products of k random values)
    scale = np.sqrt(np.mean(reference ** 2))
    assert np.all(np.abs(error) <= 2.0 ** -8 * np.abs(reference) + 2.0 ** -9 * scale)


@pytest.mark.parametrize("rows,n,k", [
    (140, 72, 512), (140, 136, 17408),      # 128 x 64 tiles, K over four parts of a workgroup's waves
    (600, 5120, 1024),                      # 128 x 128 tiles, two parts
    (1030, 5120, 512),                      # 128 x 128 tiles of four waves
    (2100, 6200, 512),                      # 256 x 256 tiles
    (140, 72, 768), (2100, 6200, 256),      # fp16 weights written once
])
def test_prefill_products_hold_weights_and_rows_exactly(hip, rows, n, k):
    """What is left of a product beside the bf16 numbers nearest to it in 64 bits (added before the one rounding, of at most
    2^-8 of what is left, itself at most 2^-8 of the product).  Rows and weights are exact; group sums and the biases against
    them are held to 2^-22, and the sums are those of f32.  Weights rounded to f16 would be off by 2^-12.3 of the
    product."""
    weights, values = Quantised(64, n + k, (n, k)), normal_bf16(64, 1, (rows, k))
    centred = -7.5 * orc.bf16_to_f32(weights.scales)    # weights of no common sign
    weights.biases = orc.f32_to_bf16(centred.ravel()).reshape(centred.shape)
    reference = values.astype(np.float64) @ weights.dequantised().T
    nearest = orc.bf16_to_f32(orc.f32_to_bf16(-reference.astype(np.float32).ravel())).reshape(rows, n)
    out = hip.alloc(DType.BF16, (rows, n))
    commands = CommandList()
    commands.dispatch_epilogue(Op.quant_matmul(4, 64), [upload(hip, values, DType.BF16), *weights.upload(hip)], out,
                               hip.prepare_epilogue(programs.add_elements()), [upload(hip, nearest, DType.BF16)])
    run(hip, commands)
    left = reference + nearest
    error = to_f32(hip.read(out), DType.BF16).reshape(rows, n) - left
    assert np.linalg.norm(error) <= 2.0 ** -16 * np.linalg.norm(reference)
    assert np.linalg.norm(left) >= 2.0 ** -10 * np.linalg.norm(reference)


def test_quant_gemm_with_scales_outside_the_fp16_range_and_huge_activations(cpu, hip):
    """Prefill-sized product whose affine parameters are not fp16 normal numbers (tiny scales, a
    zero bias, a large scale) and whose activations exceed the fp16 range in some rows: the
    f32 dequantisation path and the per-row power-of-two scaling."""
    rows, n, k = 300, 200, 512
    weights = Quantised(61, 3, (n, k))
    scales = orc.bf16_to_f32(weights.scales).copy()
    biases = orc.bf16_to_f32(weights.biases).copy()
    scales[::3, 0] = 3.0e-6
    scales[1::7, 1] = 7000.0
    biases[::5, 2] = 0.0
    biases[2::5, 3] = 1.0e-7
    weights.scales = orc.f32_to_bf16(scales.ravel()).reshape(scales.shape)
    weights.biases = orc.f32_to_bf16(biases.ravel()).reshape(biases.shape)
    x_values = orc.bf16_to_f32(normal_bf16(61, 9, (rows, k))).copy()
    x_values[5] *= 3.0e6
    x_values[17, 3] = 1.0e9
    x_values[40] *= 1.0e-6

    def build(backend):
        x = upload(backend, x_values, DType.BF16)
        packed, sc, bi = weights.upload(backend)
        out = backend.alloc(DType.BF16, (rows, n))
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(4, 64), [x, packed, sc, bi], out)
        return commands, [out]
    differential(cpu, hip, build)


@pytest.mark.parametrize("k,scale,bias,taken", [
    # words unpacked in the GEMM (whole blocks of eight groups): 24 scale within fp16, the scale a normal number of it
    (512, 2688.0, -8.0, True), (512, 2704.0, -8.0, False), (512, -2688.0, -8.0, True),
    (512, 2.0 ** -14, -8.0, True), (512, 2.0 ** -14 - 2.0 ** -22, -8.0, False), (512, 0.0, 0.0, True),
    (512, 1792.0, -7.5, True), (512, 1920.0, -7.5, False),      # 64 (bias + 8 scale) within fp16
    # fp16 weights written once
    (768, 2704.0, -8.0, True), (768, 4000.0, -8.0, True), (768, 4016.0, -8.0, False), (768, 2.0 ** -15, -8.0, True),
    (768, 1792.0, -7.5, True), (768, 1920.0, -7.5, False),
])
def test_prefill_products_at_the_limits_of_a_scale(k, scale, bias, taken):
    """One group's scale and bias (a multiple of it) at either side of what the GEMM takes.  Refused weights go to the
    kernel of any range, and no operand of theirs is kept.  Each column against 64 bits: results are rounded once, by at
    most 2^-8 of each; what the sums themselves and one group of weights below fp16's normal numbers add is far less."""
    from forja_amd.hip_backend import HipBackend
    own = HipBackend(0)
    try:
        rows, n = 140, 80
        weights, values = Quantised(63, k, (n, k)), normal_bf16(63, 1, (rows, k))
        for held, value in ((weights.scales, scale), (weights.biases, bias * scale)):
            raw = orc.f32_to_bf16(np.array([value], np.float32))
            assert orc.bf16_to_f32(raw)[0] == value
            held[37, 5] = raw[0]
        out = own.alloc(DType.BF16, (rows, n))
        commands, x, triple = CommandList(), upload(own, values, DType.BF16), weights.upload(own)
        commands.dispatch(Op.quant_matmul(4, 64), [x, *triple], out)
        prepared = n * (64 if k == 512 else 832) * 2    # 3 columns a group (or all with them), in whole steps of 64
        held = []
        for _ in range(2):      # the first product prepares, the second knows
            run(own, commands)
            held.append(own.memory_usage())
            reference = values.astype(np.float64) @ weights.dequantised().T
            error = to_f32(own.read(out), DType.BF16).reshape(rows, n) - reference
            assert np.all(np.linalg.norm(error, axis=0) <= 2.0 ** -8 * np.linalg.norm(reference, axis=0))
        assert held[0] == held[1]
        for tensor in triple:   # releasing the weights gives back what was kept of them
            own.release(tensor)
        kept = held[1] - own.memory_usage() - sum(t.layout.buffer_len for t in triple)
        assert kept == (prepared + 256 if taken else 0)
    finally:
        own.close()


def test_quant_matmul_on_strided_views_with_bias_epilogue(cpu, hip):
    """Every operand sliced with step 2 (crates/forja-metal/tests/quant_matmul/shared.rs:95-107)
    plus a fused epilogue that adds a broadcast bias."""
    rows, n, k = 6, 32, 128
    weights = Quantised(22, 5, (2 * n, 2 * k), bits=4, group=64)
    x_values = normal_bf16(22, 8, (2 * rows, 2 * k))
    bias_values = normal_bf16(22, 9, (n,))

    def build(backend):
        x = upload(backend, x_values, DType.BF16).slice([Slice(0, rows, 2), Slice(0, k)])
        packed, scales, biases = weights.upload(backend)
        packed = packed.slice([Slice(1, n, 2), Slice(0, k // 8)])
        scales = scales.slice([Slice(1, n, 2), Slice(0, k // 64)])
        biases = biases.slice([Slice(1, n, 2), Slice(0, k // 64)])
        big = backend.alloc(DType.BF16, (rows, 2 * n))
        out = big.slice([Slice(0, rows), Slice(1, n, 2)])
        bias = upload(backend, bias_values, DType.BF16).broadcast((rows, n))
        epilogue = backend.prepare_epilogue(programs.add_elements())
        commands = CommandList()
        commands.dispatch_epilogue(Op.quant_matmul(4, 64), [x, packed, scales, biases], out, epilogue, [bias])
        return commands, [big]
    differential(cpu, hip, build)


def test_prefill_products_follow_weights_that_are_rewritten(cpu, hip):
    """Products of more than 128 rows keep a prepared copy of their weights from one product to the
    next.  The copy must go when any of the three tensors is written: by the host, by a dispatch,
    or when the allocation is released and its memory taken by other weights."""
    rows, n, k = 200, 320, 512
    first, second, third = (Quantised(27, seed, (n, k)) for seed in (1, 2, 3))
    x_values = normal_bf16(27, 9, (rows, k))

    def build(backend):
        x = upload(backend, x_values, DType.BF16)
        packed, scales, biases = first.upload(backend)
        outs = [backend.alloc(DType.BF16, (rows, n)) for _ in range(5)]
        op = Op.quant_matmul(4, 64)

        def product(out, triple):
            commands = CommandList()
            commands.dispatch(op, [x, *triple], out)
            run(backend, commands)
        product(outs[0], (packed, scales, biases))
        product(outs[1], (packed, scales, biases))                      # the kept copy serves
        backend.write(scales, np.ascontiguousarray(second.scales).tobytes())   # written by the host
        product(outs[2], (packed, scales, biases))
        commands = CommandList()                                        # written by a dispatch
        commands.dispatch(Op.copy(), [upload_raw(backend, third.packed, DType.U32, third.packed.shape)], packed)
        commands.dispatch(op, [x, packed, scales, biases], outs[3])
        run(backend, commands)
        for tensor in (packed, scales, biases):                         # released: the memory may come back
            backend.release(tensor)
        product(outs[4], second.upload(backend))
        return CommandList(), outs
    differential(cpu, hip, build)


def test_prefill_products_without_kept_weights(cpu, monkeypatch):
    """FORJA_HIP_PREPARED_MB=0: nothing is kept, every product prepares its weights into the
    workspace and stands by with the conditioned second kernel, as it does when the memory set
    aside for kept weights is used up."""
    from forja_amd.hip_backend import HipBackend
    monkeypatch.setenv("FORJA_HIP_PREPARED_MB", "0")
    frugal = HipBackend(0)
    try:
        rows, n, k = 300, 520, 512
        weights = Quantised(28, 1, (n, k))
        x_values = normal_bf16(28, 2, (rows, k))

        def build(backend):
            x = upload(backend, x_values, DType.BF16)
            triple = weights.upload(backend)
            outs = [backend.alloc(DType.BF16, (rows, n)) for _ in range(2)]
            commands = CommandList()
            for out in outs:
                commands.dispatch(Op.quant_matmul(4, 64), [x, *triple], out)
            return commands, outs
        differential(cpu, frugal, build)
    finally:
        frugal.close()


def test_memory_limit_counts_and_evicts_what_the_library_keeps(cpu):
    """`Backend::set_memory_limit` (crates/forja-core/src/backend.rs:683-686) covers the caller's
    allocations and the operands the library keeps for prefill products; `memory_usage` counts
    both.  An allocation that would pass the limit drops the kept operands first and succeeds;
    one that cannot fit is refused with QuotaExceeded; results do not depend on any of it."""
    from forja_amd.hip_backend import HipBackend
    own = HipBackend(0)     # its own backend: the shared one holds other tests' allocations
    try:
        rows, n, k = 200, 2048, 512
        weights = Quantised(29, 1, (n, k))
        x_values = normal_bf16(29, 2, (rows, k))
        kept = n * 64 * 2 + 256     # fp16 bias columns (3 per group of 64, padded to 64 a row) + flag
        names = ("kept", "served by the kept operand", "prepared into workspace", "kept again")
        x = upload(own, x_values, DType.BF16)
        triple = weights.upload(own)
        outs = {name: own.alloc(DType.BF16, (rows, n)) for name in names}
        allocated = sum(t.layout.buffer_len for t in (x, *triple, *outs.values()))

        def product(backend, x, triple, out):
            commands = CommandList()
            commands.dispatch(Op.quant_matmul(4, 64), [x, *triple], out)
            run(backend, commands)
        before = own.memory_usage()
        assert before >= allocated
        product(own, x, triple, outs["kept"])
        held = own.memory_usage()
        assert held >= before + kept                       # the kept operand is counted (and the workspace)
        product(own, x, triple, outs["served by the kept operand"])
        assert own.memory_usage() == held
        # room for half the kept operand more: an allocation of its size fits only once it is dropped
        own.set_memory_limit(allocated + kept + kept // 2)
        extra = own.alloc(DType.U32, ((kept - 256) // 4,))
        assert own.memory_usage() == held - kept + (kept - 256)
        product(own, x, triple, outs["prepared into workspace"])     # no room to keep anything
        assert own.memory_usage() <= held + (kept - 256)
        with pytest.raises(BackendError) as refused:
            own.alloc(DType.U32, (kept,))
        assert refused.value.status == Status.QUOTA_EXCEEDED
        own.set_memory_limit(0)
        own.release(extra)
        product(own, x, triple, outs["kept again"])
        assert own.memory_usage() >= held
        expected = cpu.alloc(DType.BF16, (rows, n))
        product(cpu, upload(cpu, x_values, DType.BF16), weights.upload(cpu), expected)
        for name in names:
            compare(cpu, own, expected, outs[name])
    finally:
        own.close()


def test_profiled_submission_reports_an_ordered_timeline(hip):
    """`submit_profiled_retained` / `Submission::profile` (crates/forja-core/src/backend.rs:455-579):
    one entry per executed dispatch, in order, intervals that do not overlap, inside the
    submission's device time."""
    weights = Quantised(30, 1, (512, 1024))
    x = upload(hip, normal_bf16(30, 2, (8, 1024)), DType.BF16)
    triple = weights.upload(hip)
    outs = [hip.alloc(DType.BF16, (8, 512)) for _ in range(3)]
    total = hip.alloc(DType.BF16, (8, 512))
    commands = CommandList()
    for out in outs:
        commands.dispatch(Op.quant_matmul(4, 64), [x, *triple], out)
    commands.dispatch(Op.copy(), [outs[0]], total)
    plain = hip.submit(commands)
    plain.wait()
    assert plain.profile() == []                       # not asked for: nothing recorded
    submission = hip.submit_profiled(commands)
    with pytest.raises(BackendError):
        submission.profile()                           # the timeline exists after the wait
    submission.wait()
    timeline = submission.profile()
    assert [entry[0] for entry in timeline] == [0, 1, 2, 3]
    assert [entry[1] for entry in timeline] == [1, 1, 1, 1]
    assert [entry[2] for entry in timeline] == [int(d.op.kind) for d in commands.dispatches]
    previous_end = 0
    for _, _, _, start, end in timeline:
        assert previous_end <= start <= end
        previous_end = end
    assert sum(end - start for _, _, _, start, end in timeline) <= submission.gpu_time_ns() * 1.05 + 2000
    assert previous_end <= submission.gpu_time_ns() * 1.05 + 2000


@pytest.mark.parametrize("rows,n,k,kind", [
    (128, 256, 1024, "add"),    # decode rows: the add joins the slab sum
    (8, 64, 256, "add"),        # a single K slab: accumulators + epilogue program
    (300, 520, 512, "add"),     # prefill rows: the add joins the tiled GEMM's store
    (300, 130, 512, "add"),     # residual rows not 8-byte aligned: accumulators + epilogue program
    (700, 768, 1024, "mul"),    # unrecognised epilogue over a GEMM of several tiles
    (96, 512, 2048, "mul"),     # unrecognised epilogue over the slab kernels
])
def test_quant_matmul_with_elementwise_epilogue(cpu, hip, rows, n, k, kind):
    """out = epilogue(f32 accumulator, extra) with a full [rows, N] extra operand: the residual add
    after the dense down projection (crates/forja-sdk/src/nn/blocks.rs:408-411) and a product."""
    weights = Quantised(23, n + k, (n, k))
    x_values = normal_bf16(23, 1, (rows, k))
    extra_values = normal_bf16(23, 2, (rows, n))

    def build(backend):
        x = upload(backend, x_values, DType.BF16)
        extra = upload(backend, extra_values, DType.BF16)
        out = backend.alloc(DType.BF16, (rows, n))
        if kind == "add":
            program = programs.add_elements()
        else:
            b = ProgramBuilder(ProgramKind.MAP)
            b.output(0, b.mul(b.input(0), b.input(1)))
            program = b.finish()
        epilogue = backend.prepare_epilogue(program)
        commands = CommandList()
        commands.dispatch_epilogue(Op.quant_matmul(4, 64), [x, *weights.upload(backend)], out, epilogue,
                                   [extra])
        return commands, [out]
    differential(cpu, hip, build)


# ------------------------------------------------------------------ routed projections

def routed_case(seed, rows, k, experts, n, inner, bad=()):
    rng = np.random.default_rng(seed)
    indices = np.stack([rng.permutation(experts)[:k] for _ in range(rows)]).astype(np.uint32)
    for (r, s, value) in bad:
        indices[r, s] = value
    return indices


@pytest.mark.parametrize("rows,k,experts,n,inner", [(24, 4, 16, 128, 128), (256, 8, 128, 64, 128),
                                                   (5, 2, 3, 64, 64), (40, 8, 8, 192, 256),
                                                   (64, 8, 16, 256, 256), (33, 4, 7, 512, 256),
                                                   (256, 8, 128, 768, 2048)])   # last
def test_gather_projection_pair_and_weighted_sum(cpu, hip, rows, k, experts, n, inner):
    gate = Quantised(31, 1, (n, inner), experts=experts)
    up = Quantised(31, 11, (n, inner), experts=experts)
    down = Quantised(31, 21, (inner, n), experts=experts)
    indices = routed_case(31, rows, k, experts, n, inner)
    x_values = normal_bf16(31, 40, (rows, inner))
    logits = orc.fill_normal_f32(31, 41, rows * k).reshape(rows, k)
    w_values = np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True)
    residual_values = normal_bf16(31, 42, (rows, inner))

    def build(backend):
        x = upload(backend, x_values, DType.BF16)
        idx = upload(backend, indices, DType.U32)
        g, u, d = gate.upload(backend), up.upload(backend), down.upload(backend)
        plain = backend.alloc(DType.BF16, (rows, k, n))
        activated = backend.alloc(DType.BF16, (rows, k, n))
        combined = backend.alloc(DType.BF16, (rows, inner))
        summed = backend.alloc(DType.BF16, (rows, inner))
        weights = upload(backend, w_values, DType.BF16)
        residual = upload(backend, residual_values, DType.BF16)
        swiglu = backend.prepare_epilogue(programs.silu_mul_elements())
        add = backend.prepare_epilogue(programs.add_elements())
        commands = CommandList()
        commands.dispatch(Op.gather_quant_matmul(4, 64), [x, *g, idx], plain)
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [x, *g, *u, idx], activated, swiglu, [])
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [activated, *d, idx, weights], combined,
                                   add, [residual])
        commands.dispatch(Op.gather_quant_matmul(4, 64), [activated, *d, idx, weights], summed)
        return commands, [plain, activated, combined, summed]
    differential(cpu, hip, build)


@pytest.mark.parametrize("form", ["plain", "residual", "norm_into_residual", "norm_of_a_slice",
                                  "weights_in_the_sum"])
@pytest.mark.parametrize("rows,k,experts,n,inner", [(128, 8, 128, 768, 2048), (19, 4, 7, 256, 256)])
def test_weighted_sum_followed_by_the_normalisation_of_its_rows(cpu, hip, rows, k, experts, n, inner, form):
    """A decoder layer ends with the routed weighted sum and the next begins by normalising those
    rows (engines/qwen3-coder/src/lib.rs): the backend may run the two as one kernel.  The result
    must be that of the two dispatches, also where the second is not what the first can absorb: a
    normalisation that overwrites the sum's residual, one that reads only part of the rows, one
    whose weights are the rows themselves."""
    down = Quantised(33, 21, (inner, n), experts=experts)
    indices = routed_case(33, rows, k, experts, n, inner)
    activated_values = normal_bf16(33, 40, (rows, k, n))
    logits = orc.fill_normal_f32(33, 41, rows * k).reshape(rows, k)
    w_values = np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True)
    residual_values = normal_bf16(33, 42, (rows, inner))
    norm_values = normal_bf16(33, 43, (inner,))

    def build(backend):
        activated = upload(backend, activated_values, DType.BF16)
        idx = upload(backend, indices, DType.U32)
        d = down.upload(backend)
        weights = upload(backend, w_values, DType.BF16)
        residual = upload(backend, residual_values, DType.BF16)
        norm_weight = upload(backend, norm_values, DType.BF16).broadcast((rows, inner))
        summed = backend.alloc(DType.BF16, (rows, inner))
        normed = backend.alloc(DType.BF16, (rows, inner))
        add = backend.prepare_epilogue(programs.add_elements())
        norm = backend.prepare_program(programs.rms_norm_rows(1e-6))
        commands = CommandList()
        outputs = [summed, normed]
        if form == "plain":
            commands.dispatch(Op.gather_quant_matmul(4, 64), [activated, *d, idx, weights], summed)
        else:
            commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [activated, *d, idx, weights], summed,
                                       add, [residual])
        if form == "norm_into_residual":
            commands.dispatch_kernel(norm, [summed, norm_weight], [residual])
            outputs = [summed, residual]
        elif form == "norm_of_a_slice":
            half = rows // 2
            commands.dispatch_kernel(norm, [summed.narrow(0, 0, half), norm_weight.narrow(0, 0, half)],
                                     [normed.narrow(0, 0, half)])
            commands.dispatch(Op.copy(), [summed.narrow(0, half, rows - half)], normed.narrow(0, half, rows - half))
        elif form == "weights_in_the_sum":
            commands.dispatch_kernel(norm, [summed, summed], [normed])
        else:
            commands.dispatch_kernel(norm, [summed, norm_weight], [normed])
        return commands, outputs
    # rows normalised by themselves square the one-ulp differences the sums may have: twice the bar
    differential(cpu, hip, build, **({"rel": 3e-2} if form == "weights_in_the_sum" else {}))


@pytest.mark.parametrize("rows,n,k", [(1, 1024, 1024), (8, 96, 512), (16, 64, 768), (17, 160, 1536), (32, 256, 2048),
                                      (5, 32768, 1024), (33, 64, 1024), (3, 72, 1024), (4, 128, 3072)])
@pytest.mark.parametrize("form", ["norm", "residual_norm", "residual_norm_silu", "silu", "norm_add",
                                  "sum_added", "over_the_rows", "other_rows", "other_halves"])
def test_dense_products_with_the_row_programs_around_them(cpu, hip, rows, n, k, form):
    """A normalisation, the product of its rows and silu of the product's halves, next to each other:
    the backend may run them as one kernel (up to 32 rows; the last three sizes are beyond what it takes) and the
    results must be those of the dispatches one by one, also where they are not to be joined: a product
    that adds the sum the normalisation has just written, one stored over the rows that are normalised,
    one that reads other rows, halves taken the other way round."""
    weights = Quantised(35, 1, (n, k))
    x_values, u_values = normal_bf16(35, 10, (rows, k)), normal_bf16(35, 11, (rows, k))
    norm_values = 0.02 + 0.002 * normal_bf16(35, 12, (k,))

    def build(backend):
        x, u = upload(backend, x_values, DType.BF16), upload(backend, u_values, DType.BF16)
        norm_weight = upload(backend, norm_values, DType.BF16).broadcast((rows, k))
        added, normed = (backend.alloc(DType.BF16, (rows, k)) for _ in range(2))
        out, activated = backend.alloc(DType.BF16, (rows, n)), backend.alloc(DType.BF16, (rows, n // 2))
        commands = CommandList()
        outputs = [normed, out]
        if form != "silu":
            if "residual" in form or form == "sum_added":
                commands.dispatch_kernel(backend.prepare_program(programs.residual_norm_rows(1e-6)), [x, u, norm_weight],
                                         [added, normed])
                outputs.append(added)
            else:
                commands.dispatch_kernel(backend.prepare_program(programs.rms_norm_rows(1e-6)), [x, norm_weight], [normed])
        product = [u if form == "other_rows" else x if form == "silu" else normed, *weights.upload(backend)]
        if form in ("norm_add", "sum_added"):   # something as wide as the result is added to it
            extra = upload(backend, normal_bf16(35, 13, (rows, n)), DType.BF16)
            if form == "sum_added" and n <= k:
                extra = added.narrow(1, 0, n)
            commands.dispatch_epilogue(Op.quant_matmul(4, 64), product, out,
                                       backend.prepare_epilogue(programs.add_elements()), [extra])
        elif form == "over_the_rows" and n <= k:
            commands.dispatch(Op.quant_matmul(4, 64), product, x.narrow(1, 0, n))
            outputs[1] = x
        else:
            commands.dispatch(Op.quant_matmul(4, 64), product, out)
        if form in ("residual_norm_silu", "silu", "other_halves"):
            halves = [out.narrow(1, 0, n // 2), out.narrow(1, n // 2, n // 2)]
            commands.dispatch_kernel(backend.prepare_program(programs.silu_mul_elements()),
                                     halves[::-1] if form == "other_halves" else halves, [activated])
            outputs.append(activated)
        return commands, outputs if form != "silu" else outputs[1:]
    # silu of halves multiplies two results of one ulp each
    differential(cpu, hip, build, rel=2e-2, abs_=2e-2)
    # dispatches that run as one share an entry of the profile
    takes_rows = (rows, n, k) in ((1, 1024, 1024), (16, 64, 768), (5, 32768, 1024))
    takes_silu = (rows, n, k) in ((1, 1024, 1024), (32, 256, 2048), (5, 32768, 1024))
    groups = {"norm": [2] if takes_rows else [1, 1], "residual_norm": [2] if takes_rows else [1, 1],
              "residual_norm_silu": [3] if takes_rows and takes_silu else [1, 2] if takes_silu else [2, 1] if takes_rows
              else [1, 1, 1],
              "silu": [2] if takes_silu else [1, 1], "norm_add": [2] if takes_rows else [1, 1], "sum_added": [2] if takes_rows and n > k else [1, 1],
              "over_the_rows": [2] if takes_rows and n > k else [1, 1], "other_rows": [1, 1],
              "other_halves": [2, 1] if takes_rows else [1, 1, 1]}
    submission = hip.submit_profiled(build(hip)[0])
    submission.wait()
    assert [entry[1] for entry in submission.profile()] == groups[form]


@pytest.mark.parametrize("rows,n", [(1, 2048), (8, 2048), (16, 96), (17, 96), (3, 40)])
@pytest.mark.parametrize("product_first", [False, True])
def test_f32_product_of_long_rows_and_the_residual_normalisation_behind_it(cpu, hip, rows, n, product_first):
    """A product over K = 4096, whose two halves the normalisation adds: the oracle's results, and bit for bit
    those of the two dispatches submitted one by one; 17 rows and columns of no whole batch take the launches apart."""
    k, weights = 4096, Quantised(75, n, (n, 4096))
    x_values = orc.fill_normal_f32(75, 1, rows * k).reshape(rows, k)
    other_values = orc.fill_normal_f32(75, 2, rows * n).reshape(rows, n)
    norm_values = orc.fill_normal_f32(75, 3, n)

    def record(backend):
        x, other = upload(backend, x_values, DType.F32), upload(backend, other_values, DType.F32)
        norm_weight = upload(backend, norm_values, DType.F32).broadcast((rows, n))
        product, summed, normed = (backend.alloc(DType.F32, (rows, n)) for _ in range(3))
        first, second = CommandList(), CommandList()
        terms = [product, other] if product_first else [other, product]
        program = backend.prepare_program(programs.residual_norm_rows(1e-6))
        operands = [x, *weights.upload(backend)]
        joined = CommandList()
        for product_list, norm_list in ((first, second), (joined, joined)):
            product_list.dispatch(Op.quant_matmul(4, 64), operands, product)
            norm_list.dispatch_kernel(program, [*terms, norm_weight], [summed, normed])
        return joined, [first, second], [product, summed, normed]

    differential(cpu, hip, lambda backend: record(backend)[::2])
    joined, apart, tensors = record(hip)
    run(hip, joined)
    together = [hip.read(t) for t in tensors]
    for commands in apart:
        run(hip, commands)
    assert together == [hip.read(t) for t in tensors]
    submission = hip.submit_profiled(joined)
    submission.wait()
    assert [entry[1] for entry in submission.profile()] == ([1, 1] if (rows, n) in ((17, 96), (3, 40)) else [2])


@pytest.mark.parametrize("with_residual", [False, True])
def test_f32_weighted_sum_followed_by_the_normalisation_of_its_rows(cpu, hip, with_residual):
    """The same pair in the engine's dtypes: an 8-row decode batch, everything f32."""
    rows, k, experts, n, inner = 8, 8, 128, 768, 2048
    down = Quantised(34, 21, (inner, n), experts=experts)
    indices = routed_case(34, rows, k, experts, n, inner)
    activated_values = orc.fill_normal_f32(34, 40, rows * k * n).reshape(rows, k, n)
    logits = orc.fill_normal_f32(34, 41, rows * k).reshape(rows, k)
    w_values = np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True)
    residual_values = orc.fill_normal_f32(34, 42, rows * inner).reshape(rows, inner)
    norm_values = orc.fill_normal_f32(34, 43, inner)

    def build(backend):
        activated = upload(backend, activated_values, DType.F32)
        idx = upload(backend, indices, DType.U32)
        weights = upload(backend, w_values, DType.F32)
        residual = upload(backend, residual_values, DType.F32)
        norm_weight = upload(backend, norm_values, DType.F32).broadcast((rows, inner))
        summed = backend.alloc(DType.F32, (rows, inner))
        normed = backend.alloc(DType.F32, (rows, inner))
        commands = CommandList()
        if with_residual:
            add = backend.prepare_epilogue(programs.add_elements())
            commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [activated, *down.upload(backend), idx, weights],
                                       summed, add, [residual])
        else:
            commands.dispatch(Op.gather_quant_matmul(4, 64), [activated, *down.upload(backend), idx, weights], summed)
        commands.dispatch_kernel(backend.prepare_program(programs.rms_norm_rows(1e-6)), [summed, norm_weight], [normed])
        return commands, [summed, normed]
    differential(cpu, hip, build)


@pytest.mark.parametrize("dtype,bits,group,scale_dtype", [
    (DType.F32, 4, 64, DType.BF16),      # the qwen3-coder engine: f32 activations
    (DType.F16, 8, 32, DType.F16),
    (DType.BF16, 4, 128, DType.BF16),    # a group size the matrix-core kernels do not take
])
@pytest.mark.parametrize("rows,k,experts,n,inner", [(8, 8, 128, 768, 2048), (37, 3, 5, 96, 256),
                                                   (70, 8, 16, 192, 512)])   # ≈35 routes per expert: two tiles
def test_gather_in_other_dtypes_bits_and_groups(cpu, hip, rows, k, experts, n, inner, dtype, bits, group,
                                                scale_dtype):
    """The routed forms through the f32 vector-ALU kernels (route by route for the first case, grouped
    by expert for the others), with two bad routes: the valid routes
    agree with the oracle, the lowest bad expert is reported, bad projection rows read zero and bad
    routes are left out of the weighted sum."""
    gate = Quantised(35, 1, (n, inner), bits=bits, group=group, experts=experts)
    up = Quantised(35, 11, (n, inner), bits=bits, group=group, experts=experts)
    down = Quantised(35, 21, (inner, n), bits=bits, group=group if n % group == 0 else 32, experts=experts)
    down_group = down.group
    indices = routed_case(35, rows, k, experts, n, inner, bad=[(1, 2, experts + 9), (rows - 1, 0, experts)])
    x_values = normal_bf16(35, 40, (rows, inner))
    logits = orc.fill_normal_f32(35, 41, rows * k).reshape(rows, k)
    w_values = np.exp(logits) / np.exp(logits).sum(axis=1, keepdims=True)
    residual_values = normal_bf16(35, 42, (rows, inner))

    def build(backend, good_only):
        x = upload(backend, x_values, dtype)
        idx = upload(backend, indices if not good_only else indices % experts, DType.U32)
        g, u, d = (w.upload(backend, scale_dtype=scale_dtype) for w in (gate, up, down))
        plain, activated = (backend.alloc(dtype, (rows, k, n)) for _ in range(2))
        combined, summed = (backend.alloc(dtype, (rows, inner)) for _ in range(2))
        weights = upload(backend, w_values, dtype)
        residual = upload(backend, residual_values, dtype)
        swiglu = backend.prepare_epilogue(programs.silu_mul_elements())
        add = backend.prepare_epilogue(programs.add_elements())
        first, second = CommandList(), CommandList()
        first.dispatch(Op.gather_quant_matmul(bits, group), [x, *g, idx], plain)
        second.dispatch_epilogue(Op.gather_quant_matmul(bits, group), [x, *g, *u, idx], activated, swiglu, [])
        second.dispatch_epilogue(Op.gather_quant_matmul(bits, down_group), [activated, *d, idx, weights],
                                 combined, add, [residual])
        second.dispatch(Op.gather_quant_matmul(bits, down_group), [activated, *d, idx, weights], summed)
        return (first, second), [plain, activated, combined, summed]

    # without bad routes: every output against the oracle
    outputs = []
    for backend in (cpu, hip):
        lists, tensors = build(backend, True)
        for commands in lists:
            run(backend, commands)
        outputs.append(tensors)
    for a, b in zip(*outputs):
        compare(cpu, hip, a, b)
    # with them: the lowest bad expert is reported by both, the projection's bad rows are zero
    for backend in (cpu, hip):
        lists, tensors = build(backend, False)
        with pytest.raises(BackendError) as info:
            run(backend, lists[0])
        assert info.value.index == experts
        if backend is hip:
            values = to_f32(hip.read(tensors[0]), dtype).reshape(rows, k, n)
            assert not values[1, 2].any() and not values[rows - 1, 0].any() and values[0, 0].any()
            with pytest.raises(BackendError) as info:
                run(backend, lists[1])
            assert info.value.index == experts


def test_gather_reports_lowest_bad_expert_and_zeroes_its_rows(cpu, hip):
    """lib.rs:2929-2950, crates/forja-metal/tests/gather_quant_matmul.rs:644-764"""
    rows, k, experts, n, inner = 6, 3, 4, 32, 64
    gate = Quantised(32, 1, (n, inner), experts=experts)
    indices = routed_case(32, rows, k, experts, n, inner, bad=[(1, 2, 99), (4, 0, 7)])
    x_values = normal_bf16(32, 40, (rows, inner))

    def build(backend):
        x = upload(backend, x_values, DType.BF16)
        idx = upload(backend, indices, DType.U32)
        out = upload(backend, np.full((rows, k, n), 3.0), DType.BF16)
        commands = CommandList()
        commands.dispatch(Op.gather_quant_matmul(4, 64), [x, *gate.upload(backend), idx], out)
        return commands, [out]
    results = differential(cpu, hip, build, expect_error={Status.INDEX_OUT_OF_RANGE, Status.DEVICE_ERROR_FLAG})
    (cpu_out, cpu_err), (hip_out, hip_err) = results
    assert cpu_err.index == 7 and hip_err.index == 7
    values = to_f32(hip.read(hip_out[0]), DType.BF16).reshape(rows, k, n)
    assert not values[1, 2].any() and not values[4, 0].any() and values[0, 0].any()


def test_gather_with_an_unrecognised_epilogue_uses_the_interpreter(cpu, hip):
    rows, k, experts, n, inner = 8, 2, 4, 32, 64
    gate, up = Quantised(33, 1, (n, inner), experts=experts), Quantised(33, 2, (n, inner), experts=experts)
    indices = routed_case(33, rows, k, experts, n, inner)
    x_values = normal_bf16(33, 3, (rows, inner))
    program = Program(ProgramKind.MAP, [
        Inst.input(0), Inst.input(1), Inst.unary(UnOp.TANH, 0), Inst.binary(BinOp.MAX, 1, 2),
        Inst.const(0.5), Inst.binary(BinOp.MUL, 3, 4)], [(0, 5)])

    def build(backend):
        x = upload(backend, x_values, DType.F32)
        idx = upload(backend, indices, DType.U32)
        out = backend.alloc(DType.F32, (rows, k, n))
        commands = CommandList()
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64),
                                   [x, *gate.upload(backend), *up.upload(backend), idx], out,
                                   backend.prepare_epilogue(program), [])
        return commands, [out]
    differential(cpu, hip, build, rel=1e-4, abs_=1e-4, norm_tol=1e-4)


@pytest.mark.parametrize("rows,k,experts,tile", [(256, 8, 128, 16), (128, 8, 128, 32), (7, 3, 5, 2),
                                                (1, 1, 1, 1), (300, 8, 128, 32), (64, 2, 200, 8),
                                                (100, 8, 512, 32), (333, 8, 3, 32),
                                                (2081, 8, 128, 64),     # 17 steps of a wave, the last runs short
                                                (5003, 8, 40, 32)])     # more routes than LDS puts together
def test_route_pack_is_bit_exact(cpu, hip, rows, k, experts, tile):
    rng = np.random.default_rng(rows * 31 + k)
    indices = rng.integers(0, experts, (rows, k)).astype(np.uint32)
    if experts == 3:
        indices[:] = 1      # every route names the same expert: one long run across rounds
        indices[5, 2] = 0

    def build(backend):
        idx = upload(backend, indices, DType.U32)
        max_blocks = experts + rows * k // tile + 1
        outs = [backend.alloc(DType.U32, (experts,)), backend.alloc(DType.U32, (experts + 1,)),
                backend.alloc(DType.U32, (rows * k,)), backend.alloc(DType.U32, (max_blocks, 3))]
        commands = CommandList()
        commands.dispatch_many(Op.route_pack(tile), [idx], outs)
        return commands, outs
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    flat = indices.ravel().astype(np.int64)
    order = np.argsort(flat, kind="stable")
    assert np.frombuffer(hip.read(hip_out[2]), np.uint32).tolist() == order.tolist()


def test_route_pack_skips_bad_routes_and_reports_the_lowest(cpu, hip):
    indices = np.array([[0, 9, 2], [7, 1, 1], [2, 2, 50]], dtype=np.uint32)

    def build(backend):
        idx = upload(backend, indices, DType.U32)
        outs = [backend.alloc(DType.U32, (3,)), backend.alloc(DType.U32, (4,)),
                backend.alloc(DType.U32, (9,)), backend.alloc(DType.U32, (8, 3))]
        commands = CommandList()
        commands.dispatch_many(Op.route_pack(2), [idx], outs)
        return commands, outs[:2]
    results = differential(cpu, hip, build, expect_error={Status.INDEX_OUT_OF_RANGE})
    assert results[1][1].index == 7


# ------------------------------------------------------------------ selection

@pytest.mark.parametrize("width,k", [(1, 1), (64, 8), (100, 8), (128, 8), (300, 16), (512, 64),
                                     (2050, 64)])
def test_top_k_edge_widths_ties_and_nans(cpu, hip, width, k):
    values = top_k_case(width)

    def build(backend):
        x = upload_raw(backend, values, DType.F32, (1, width))
        outs = [backend.alloc(DType.F32, (1, k)), backend.alloc(DType.U32, (1, k))]
        commands = CommandList()
        commands.dispatch_many(Op.top_k(k, False), [x], outs)
        return commands, outs
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[0]) == hip.read(hip_out[0])       # values copied bit for bit


@pytest.mark.parametrize("dtype", [DType.BF16, DType.F32])
def test_router_top_k_is_bit_exact_in_order_and_close_in_weight(cpu, hip, dtype):
    logits = orc.fill_normal_f32(41, 1, 256 * 128).reshape(256, 128)

    def build(backend):
        x = upload(backend, logits, dtype)
        outs = [backend.alloc(dtype, (256, 8)), backend.alloc(DType.U32, (256, 8))]
        commands = CommandList()
        commands.dispatch_many(Op.top_k(8, True), [x], outs)
        return commands, outs
    differential(cpu, hip, build)


@pytest.mark.parametrize("case", ["chain", "indices_rewritten", "fewer_logits_than_experts", "one_allocation"])
@pytest.mark.parametrize("rows,dtype", [(1, DType.BF16), (8, DType.BF16), (16, DType.F32), (17, DType.BF16)])
def test_top_k_of_a_small_batch_feeds_the_routed_products(cpu, hip, rows, dtype, case):
    """A small decode batch: router logits -> top-k -> routed gate/up + SwiGLU -> routed down with
    the weighted sum, the two products sharing the route plan packed from the selected indices.
    The result is the oracle's, also where the indices are overwritten before the products read
    them, the products know more experts than there were logits, or values and indices live in
    one allocation."""
    k, experts, n, inner = 8, 128, 128, 256
    width = 64 if case == "fewer_logits_than_experts" else experts
    gate = Quantised(47, 1, (n, inner), experts=experts)
    up = Quantised(47, 11, (n, inner), experts=experts)
    down = Quantised(47, 21, (inner, n), experts=experts)
    logits = orc.fill_normal_f32(47, 31, rows * width).reshape(rows, width)
    other = routed_case(47, rows, k, experts, n, inner)
    x_values = normal_bf16(47, 40, (rows, inner))

    def build(backend):
        x = upload(backend, x_values, DType.BF16)
        g, u, d = gate.upload(backend), up.upload(backend), down.upload(backend)
        router = upload(backend, logits, dtype)
        if case == "one_allocation":      # u32 indices behind the weights in the same allocation
            both = backend.alloc(DType.U32, (2 * rows, k))
            span = both.layout.buffer_len
            weights = both.with_layout(Layout.contiguous(dtype, 0, (rows, k), span))
            idx = both.with_layout(Layout.contiguous(DType.U32, rows * k, (rows, k), span))
        else:
            weights, idx = backend.alloc(dtype, (rows, k)), backend.alloc(DType.U32, (rows, k))
        activated = backend.alloc(DType.BF16, (rows, k, n))
        summed = backend.alloc(DType.BF16, (rows, inner))
        bf16_weights = backend.alloc(DType.BF16, (rows, k))
        swiglu = backend.prepare_epilogue(programs.silu_mul_elements())
        commands = CommandList()
        commands.dispatch_many(Op.top_k(k, True), [router], [weights, idx])
        if case == "indices_rewritten":
            commands.dispatch(Op.copy(), [upload(backend, other, DType.U32)], idx)
        commands.dispatch(Op.copy(), [weights], bf16_weights)
        commands.dispatch_epilogue(Op.gather_quant_matmul(4, 64), [x, *g, *u, idx], activated, swiglu, [])
        commands.dispatch(Op.gather_quant_matmul(4, 64), [activated, *d, idx, bf16_weights], summed)
        return commands, [weights, idx, activated, summed]
    differential(cpu, hip, build)


def test_argmax_ties_and_vocabulary_width(cpu, hip):
    rng = np.random.default_rng(3)
    logits = rng.standard_normal((4, 151936)).astype(np.float32)
    logits[1, 77] = logits[1, 150000] = 99.0            # tie: highest index wins
    logits[2, 5] = np.inf
    logits[3, 100] = np.nan                             # +NaN is the maximum under total order
    small = np.array([[1.0, 9.0, 2.0, 9.0, 3.0]], dtype=np.float32)

    def build(backend):
        a, b = upload(backend, logits, DType.BF16), upload(backend, small, DType.F32)
        c = upload(backend, logits, DType.F32)             # the engine's f32 logits
        outs = [backend.alloc(DType.U32, (4,)), backend.alloc(DType.U32, (1,)), backend.alloc(DType.U32, (4,))]
        commands = CommandList()
        commands.dispatch(Op.argmax(), [a], outs[0])
        commands.dispatch(Op.argmax(), [b], outs[1])
        commands.dispatch(Op.argmax(), [c], outs[2])
        return commands, outs
    (_, _), (hip_out, _) = differential(cpu, hip, build)
    assert np.frombuffer(hip.read(hip_out[1]), np.uint32).tolist() == [3]
    assert np.frombuffer(hip.read(hip_out[0]), np.uint32).tolist()[1:] == [150000, 5, 100]


# ------------------------------------------------------------------ paged storage

def test_paged_copy_round_trip_with_conversion(cpu, hip):
    values = np.arange(21, dtype=np.float32) / 8.0

    def build(backend):
        source = upload(backend, values.reshape(7, 3), DType.F32)
        pool = backend.alloc(DType.F16, (3, 4, 3))
        table = upload(backend, np.array([[2, 5], [0, 7]]), DType.U32)
        generations = upload(backend, np.array([7, 0, 5]), DType.U32)
        output = backend.alloc(DType.F32, (7, 3))
        commands = CommandList()
        commands.dispatch(Op.paged_copy(INTO_PAGES, 1, 4), [source, table, generations], pool)
        commands.dispatch(Op.paged_copy(OUT_OF_PAGES, 1, 4), [pool, table, generations], output)
        return commands, [pool, output]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[0]) == hip.read(hip_out[0]) and cpu.read(cpu_out[1]) == hip.read(hip_out[1])


def test_paged_copy_refuses_stale_entries_without_writing(hip):
    """crates/forja-metal/tests/paged.rs:239-277: rejected rows are not written, others are."""
    source = upload(hip, np.arange(16, dtype=np.float32).reshape(8, 2) + 1.0, DType.F32)
    pool = hip.alloc(DType.F32, (3, 4, 2))
    generations = upload(hip, np.array([7, 8, 9]), DType.U32)
    table = upload(hip, np.array([[1, 8], [2, 1]]), DType.U32)     # second entry is stale
    commands = CommandList()
    commands.dispatch(Op.paged_copy(INTO_PAGES, 0, 4), [source, table, generations], pool)
    with pytest.raises(BackendError) as info:
        run(hip, commands)
    assert info.value.status == Status.DEVICE_ERROR_FLAG and info.value.index == 1
    values = to_f32(hip.read(pool), DType.F32).reshape(3, 4, 2)
    assert values[1].ravel().tolist() == list(np.arange(8) + 1.0) and not values[2].any()


PAGED_CASES = [
    # hq, hkv, sq, key_length, q_start, causal, pool dtype, page_tokens
    (16, 8, 1, 18, 17, True, DType.BF16, 16),
    (16, 8, 1, 65, 64, True, DType.BF16, 16),
    (16, 8, 1, 131, 130, True, DType.BF16, 16),
    (16, 8, 1, 512, 511, True, DType.BF16, 16),
    (32, 4, 1, 1000, 999, True, DType.BF16, 16),
    (32, 4, 1, 300, 299, True, DType.BF16, 64),
    (4, 2, 5, 37, 32, True, DType.BF16, 16),
    (4, 4, 3, 33, 0, False, DType.F16, 16),
    (2, 1, 4, 20, 16, True, DType.F32, 4),
    (40, 8, 77, 177, 100, True, DType.BF16, 16),     # prefill chunk through the single-lane op
    (16, 8, 50, 90, 0, False, DType.BF16, 16),       # non-causal: every row attends key_length
    (32, 4, 130, 130, 0, True, DType.BF16, 16),
]


@pytest.mark.parametrize("hq,hkv,sq,key_length,q_start,causal,dtype,pt", PAGED_CASES)
def test_paged_sdpa(cpu, hip, hq, hkv, sq, key_length, q_start, causal, dtype, pt):
    scale = 1.0 / math.sqrt(128)

    def build(backend):
        t, _ = paged_case(backend, hq, hkv, sq, key_length, pt, q_start, pool_dtype=dtype)
        commands = CommandList()
        commands.dispatch(Op.paged_sdpa(scale, causal, q_start, key_length, pt),
                          [t["q"], t["keys"], t["values"], t["table"], t["generations"]], t["out"])
        return commands, [t["out"]]
    differential(cpu, hip, build)


@pytest.mark.parametrize("sq,key_length,q_start", [(1, 300, 299), (77, 177, 100)])
@pytest.mark.parametrize("q_dtype", [DType.F32, DType.F16])
def test_paged_sdpa_and_append_with_f16_pools(cpu, hip, q_dtype, sq, key_length, q_start):
    """The qwen3-coder engine's dtypes: f32 activations against an f16 KV cache
    (engines/qwen3-coder/src/lib.rs: the pools are allocated as F16, the rows arrive as F32)."""
    hq, hkv, pt = 32, 4, 64
    scale = 1.0 / math.sqrt(128)
    k_new = normal_bf16(52, 1, (sq, hkv, 128)) * 1.001      # not representable in f16 as they stand
    v_new = normal_bf16(52, 2, (sq, hkv, 128)) * 1.001

    def build(backend):
        t, _ = paged_case(backend, hq, hkv, sq, key_length, pt, q_start, pool_dtype=DType.F16, q_dtype=q_dtype)
        appended = backend.alloc(q_dtype, (hq, sq, 128))
        commands = CommandList()
        commands.dispatch(Op.paged_sdpa(scale, True, q_start, key_length, pt),
                          [t["q"], t["keys"], t["values"], t["table"], t["generations"]], t["out"])
        if sq == 1:       # the appending form takes a single query row (check_paged_append, ops.rs:2266)
            commands.dispatch_many(Op.paged_sdpa_append(scale, q_start, pt),
                                   [t["q"], upload(backend, k_new, q_dtype), upload(backend, v_new, q_dtype),
                                    t["table"], t["generations"]], [appended, t["keys"], t["values"]])
        return commands, [t["out"], appended, t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build, bar=DType.F16)
    assert cpu.read(cpu_out[2]) == hip.read(hip_out[2]) and cpu.read(cpu_out[3]) == hip.read(hip_out[3])


def test_paged_sdpa_through_a_permuted_query_view(cpu, hip):
    """Engines pass q as a permuted [Hq,Sq,D] view of [Sq,Hq,D] storage and read the output the
    same way (crates/forja-host/src/lib.rs:6223-6333)."""
    hq, hkv, sq, key_length, q_start = 8, 2, 3, 40, 37
    scale = 0.1

    def build(backend):
        t, host = paged_case(backend, hq, hkv, sq, key_length, 16, q_start)
        stored_q = upload(backend, np.transpose(host["q"], (1, 0, 2)), DType.BF16)
        stored_out = backend.alloc(DType.BF16, (sq, hq, 128))
        commands = CommandList()
        commands.dispatch(Op.paged_sdpa(scale, True, q_start, key_length, 16),
                          [stored_q.permute([1, 0, 2]), t["keys"], t["values"], t["table"], t["generations"]],
                          stored_out.permute([1, 0, 2]))
        return commands, [stored_out]
    differential(cpu, hip, build)


def test_paged_append_then_attend(cpu, hip):
    hq, hkv, q_start = 16, 8, 130
    scale = 1.0 / math.sqrt(128)
    k_new = normal_bf16(51, 1, (1, hkv, 128))
    v_new = normal_bf16(51, 2, (1, hkv, 128))

    def build(backend):
        t, _ = paged_case(backend, hq, hkv, 1, q_start + 1, 16, q_start)
        kn, vn = upload(backend, k_new, DType.BF16), upload(backend, v_new, DType.BF16)
        commands = CommandList()
        commands.dispatch_many(Op.paged_sdpa_append(scale, q_start, 16),
                               [t["q"], kn, vn, t["table"], t["generations"]],
                               [t["out"], t["keys"], t["values"]])
        return commands, [t["out"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)


def test_inactive_lane_is_zero_and_touches_nothing(hip):
    query = upload(hip, np.ones((2, 1, 4)), DType.F32)
    key = upload(hip, np.ones((1, 1, 4)), DType.F32)
    value = upload(hip, np.ones((1, 1, 4)), DType.F32)
    table = upload(hip, np.array([[0, 0xffffffff]]), DType.U32)
    generations = upload(hip, np.array([1]), DType.U32)
    activity = upload(hip, np.array([0]), DType.U32)
    key_pages, value_pages = hip.alloc(DType.F32, (1, 4, 1, 4)), hip.alloc(DType.F32, (1, 4, 1, 4))
    output = upload(hip, np.full((2, 1, 4), 5.0), DType.F32)
    commands = CommandList()
    commands.dispatch_many(Op.paged_sdpa_append(1.0, 0, 4), [query, key, value, table, generations, activity],
                           [output, key_pages, value_pages])
    run(hip, commands)
    assert not any(hip.read(output)) and not any(hip.read(key_pages)) and not any(hip.read(value_pages))


def test_stale_generation_is_reported_and_never_dereferenced(hip):
    t, _ = paged_case(hip, 4, 2, 1, 40, 16, 39)
    generations = np.frombuffer(hip.read(t["generations"]), np.uint32).copy()
    table = np.frombuffer(hip.read(t["table"]), np.uint32).reshape(-1, 2)
    generations[table[1, 0]] += 1                       # logical page 1 is now stale
    hip.write(t["generations"], generations.tobytes())
    commands = CommandList()
    commands.dispatch(Op.paged_sdpa(0.1, True, 39, 40, 16),
                      [t["q"], t["keys"], t["values"], t["table"], t["generations"]], t["out"])
    with pytest.raises(BackendError) as info:
        run(hip, commands)
    assert info.value.status == Status.DEVICE_ERROR_FLAG and info.value.index == 1
    assert not any(hip.read(t["out"]))


# ------------------------------------------------------------------ ragged batch

def ragged_case(backend, contexts, counts, hq, hkv, pt, seed, activity=None, dtype=DType.BF16,
                corrupt=None, pool_dtype=None, out_dtype=None):
    """Lanes with `contexts[l]` tokens already cached and `counts[l]` new queries each.  Shuffled
    physical pages shared by all lanes, generations 11+page, poisoned table tails.  `dtype` is
    that of the query and of the new rows; pools and output follow it unless named."""
    width = 128
    pool_dtype = dtype if pool_dtype is None else pool_dtype
    out_dtype = dtype if out_dtype is None else out_dtype
    lanes = len(contexts)
    pages_needed = [(c + n + pt - 1) // pt for c, n in zip(contexts, counts)]
    table_pages = max(pages_needed) + 2
    physical = sum(pages_needed) + 5
    rng = np.random.default_rng(seed)
    free = list(rng.permutation(physical))
    tables = np.zeros((lanes, table_pages, 2), np.uint32)
    tables[:, :, 1] = 0xffffffff
    for lane, need in enumerate(pages_needed):
        for logical in range(need):
            page = free.pop()
            tables[lane, logical] = (page, 11 + page)
    if corrupt is not None:
        lane, logical = corrupt
        tables[lane, logical, 1] += 1
    pool_k = orc.bf16_to_f32(orc.fill_normal_bf16(seed, 1, physical * pt * hkv * width))
    pool_v = orc.bf16_to_f32(orc.fill_normal_bf16(seed, 2, physical * pt * hkv * width))
    total = sum(counts)
    cu = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    tensors = dict(
        q=upload(backend, normal_bf16(seed, 3, (total, hq, width)), dtype),
        k_new=upload(backend, normal_bf16(seed, 4, (total, hkv, width)), dtype),
        v_new=upload(backend, normal_bf16(seed, 5, (total, hkv, width)), dtype),
        tables=upload(backend, tables, DType.U32),
        generations=upload(backend, 11 + np.arange(physical), DType.U32),
        cu=upload(backend, cu, DType.U32),
        starts=upload(backend, np.array(contexts), DType.U32),
        out=backend.alloc(out_dtype, (total, hq, width)),
        keys=upload(backend, pool_k.reshape(physical, pt, hkv, width), pool_dtype),
        values=upload(backend, pool_v.reshape(physical, pt, hkv, width), pool_dtype))
    inputs = [tensors[n] for n in ("q", "k_new", "v_new", "tables", "generations", "cu", "starts")]
    if activity is not None:
        inputs.append(upload(backend, np.array(activity), DType.U32))
    return tensors, inputs


RAGGED_CASES = [
    # contexts, new tokens per lane, hq, hkv, page_tokens
    ([17, 64, 130, 511], [1, 1, 1, 1], 16, 8, 16),
    ([300, 1, 2047, 700, 15, 16, 0], [1, 1, 1, 1, 1, 1, 1], 32, 4, 16),
    ([40, 0, 100], [1, 5, 3], 8, 2, 16),                           # decode + prefill chunks
    ([100, 257], [1, 1], 32, 4, 64),                               # engine page size
    ([0, 130, 33, 900], [70, 1, 45, 1], 40, 8, 16),                # prefill chunks of a 5-head group + decode rows
    ([0, 64], [200, 37], 16, 8, 16),                               # 16 tokens per query group, ragged tails
    ([500], [96], 32, 4, 16),                                      # a chunk continuing a long context
    ([0, 5], [33, 31], 4, 4, 16),                                  # one head per kv head: 32 tokens per group
    # decode lanes of very different lengths: the split length is the shortest that gives every
    # work item a place on the device at once
    ([5000, 100, 2500, 3100, 33, 4000, 777, 1500, 6000, 9000, 7000, 8990], [1] * 12, 8, 8, 16),
    # more decode lanes than the device holds workgroups, two of them long: split at the even
    # share of a place, up to the split limit of so many tokens
    ([3000 if i == 5 else 2000 if i == 200 else (37 * i) % 60 for i in range(300)], [1] * 300, 8, 8, 16),
]


@pytest.mark.parametrize("contexts,counts,hq,hkv,pt", RAGGED_CASES)
def test_ragged_attention_equals_the_per_lane_sequence(cpu, hip, contexts, counts, hq, hkv, pt):
    scale = 1.0 / math.sqrt(128)

    def build(backend):
        t, inputs = ragged_case(backend, contexts, counts, hq, hkv, pt, seed=61)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(scale, pt), inputs, [t["out"], t["keys"], t["values"]])
        return commands, [t["out"], t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    # block-table gather and append placement are pure addressing: pools must match bit for bit
    assert cpu.read(cpu_out[1]) == hip.read(hip_out[1]) and cpu.read(cpu_out[2]) == hip.read(hip_out[2])


def keep_only_keys(backend, t, contexts, pt, hkv):
    """Every slot of the pools that holds no key of `contexts` becomes a NaN."""
    tables = np.frombuffer(backend.read(t["tables"]), np.uint32).reshape(t["tables"].shape)
    for name in ("keys", "values"):
        pool = np.frombuffer(backend.read(t[name]), np.uint16).reshape(-1, pt, hkv * 128)
        held = np.full_like(pool, 0x7fff)
        for lane, keys in enumerate(contexts):
            for first in range(0, keys, pt):
                page, rows = tables[lane, first // pt, 0], min(pt, keys - first)
                held[page, :rows] = pool[page, :rows]
        backend.write(t[name], held.tobytes())


@pytest.mark.parametrize("pt,hq,hkv,dtype", [(16, 16, 8, DType.BF16), (48, 5, 1, DType.F16), (64, 32, 2, DType.F32)])
def test_decode_reads_no_slot_past_its_keys(cpu, hip, pt, hq, hkv, dtype):
    """Every length of a last tile, one split and several (of one or two tiles, most of them); all slots that hold no key
    are NaNs (bf16 and f16 pools; f32 queries read an f16 one)."""
    contexts = list(range(0, 66)) + [94, 95, 96, 127, 128, 159, 160, 161, 64 * pt - 2, 64 * pt, 64 * pt + 33, 4000]
    pool_dtype = DType.F16 if dtype is DType.F32 else dtype
    pools = {}

    def build(backend):
        t, inputs = ragged_case(backend, contexts, [1] * len(contexts), hq, hkv, pt, seed=67, dtype=dtype,
                                pool_dtype=pool_dtype)
        keep_only_keys(backend, t, contexts, pt, hkv)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, pt), inputs, [t["out"], t["keys"], t["values"]])
        pools[backend] = t["keys"], t["values"]
        return commands, [t["out"]]
    _, (hip_out, _) = differential(cpu, hip, build, bar=pool_dtype)
    assert np.isfinite(to_f32(hip.read(hip_out[0]), dtype)).all()
    for want, got in zip(pools[cpu], pools[hip]):
        assert cpu.read(want) == hip.read(got)


@pytest.mark.parametrize("pt,hq,hkv,dtype", [(16, 4, 2, DType.BF16), (48, 5, 1, DType.F16), (64, 4, 1, DType.F32)])
def test_decode_items_of_many_tiles_read_no_slot_past_their_keys(cpu, hip, pt, hq, hkv, dtype):
    """Items of one to seven tiles of 32 keys, so that either of the kernel's two tiles in flight ends one, with last tiles
    of one key to all of them; all slots that hold no key are NaNs.  A batch of so many rows has room for one split a lane
    (16384 // rows), whatever length splits have: an item is a lane's keys."""
    rows = 8200
    assert 16384 // rows == 1
    contexts = [32 * tiles + last - 1 for tiles in range(7) for last in (1, 15, 16, 17, 31, 32)]
    lanes = len(contexts)
    pool_dtype = DType.F16 if dtype is DType.F32 else dtype
    pools = {}

    def build(backend):
        t, inputs = ragged_case(backend, contexts + [0], [1] * lanes + [rows - lanes], hq, hkv, pt, seed=72, dtype=dtype,
                                pool_dtype=pool_dtype)
        keep_only_keys(backend, t, contexts, pt, hkv)
        tables = np.frombuffer(backend.read(t["tables"]), np.uint32).reshape(t["tables"].shape)
        inputs[3] = upload(backend, tables[:lanes], DType.U32)     # the other rows belong to no lane
        inputs[5] = upload(backend, np.arange(lanes + 1), DType.U32)
        inputs[6] = upload(backend, np.array(contexts), DType.U32)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, pt, one_row_per_lane=True), inputs,
                               [t["out"], t["keys"], t["values"]])
        pools[backend] = t["keys"], t["values"]
        return commands, [t["out"]]
    _, (hip_out, _) = differential(cpu, hip, build, bar=pool_dtype)
    assert np.isfinite(to_f32(hip.read(hip_out[0]), dtype)).all()
    for want, got in zip(pools[cpu], pools[hip]):
        assert cpu.read(want) == hip.read(got)


@pytest.mark.parametrize("contexts,counts", [
    # six tokens to a group of five heads, eight kv heads: 63 and 64 groups, the second with decode rows
    # in items of the longest group's length, the third with groups shorter than the shortest items
    ([0, 1500, 513], [381, 1, 1]), ([0, 1500, 513], [382, 1, 1]), ([0] * 8 + [1500, 31], [48] * 8 + [1, 1])])
def test_decode_rows_beside_prefill_groups_that_fill_the_device(cpu, hip, contexts, counts):
    def build(backend):
        t, inputs = ragged_case(backend, contexts, counts, 40, 8, 16, seed=62)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(1.0 / math.sqrt(128), 16), inputs,
                               [t["out"], t["keys"], t["values"]])
        return commands, [t["out"], t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[1]) == hip.read(hip_out[1]) and cpu.read(cpu_out[2]) == hip.read(hip_out[2])


@pytest.mark.parametrize("contexts,counts,hq,hkv,pt,scale", [
    # groups of 128 query rows, waves of 32, tiles of 64 keys: one row less, the edge, one more
    ([0, 1, 63, 64], [63, 64, 65, 2], 16, 8, 16, 0.09),      # 64 tokens to a group
    ([31, 0, 960], [25, 26, 51], 40, 8, 16, 0.09),           # 25 tokens, rows that share a wave unevenly
    ([0, 32], [17, 130], 24, 3, 48, -0.09),                  # three kv heads, a negative scale
    ([5], [130], 4, 4, 16, 0.0),                             # 128 tokens to a group, every key alike
    ([1100, 2048, 3070], [70, 3, 2], 32, 2, 16, 0.09),       # page numbers in rounds of 64, two splits
    ([3071, 3100], [40, 9], 16, 8, 48, 0.09)])
def test_prefill_attention_at_the_edges_of_its_tiles(cpu, hip, contexts, counts, hq, hkv, pt, scale):
    def build(backend):
        t, inputs = ragged_case(backend, contexts, counts, hq, hkv, pt, seed=63)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(scale, pt), inputs, [t["out"], t["keys"], t["values"]])
        return commands, [t["out"], t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[1]) == hip.read(hip_out[1]) and cpu.read(cpu_out[2]) == hip.read(hip_out[2])


def test_a_value_without_a_number_reaches_later_rows_only(cpu, hip):
    """Token 69 of a chunk stores a value row of NaNs: rows whose 16-key blocks end before it (here: the
    first 64 tokens, four waves of a group) do not meet it."""
    def build(backend):
        t, inputs = ragged_case(backend, [0], [70], 16, 8, 16, seed=64)
        values = normal_bf16(64, 5, (70, 8, 128)).astype(np.float32)
        values[69] = np.nan
        inputs[2] = upload(backend, values, DType.BF16)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 16), inputs, [t["out"], t["keys"], t["values"]])
        backend.submit(commands).wait()
        return to_f32(backend.read(t["out"]), DType.BF16).reshape(70, 16, 128)
    want, got = build(cpu), build(hip)
    assert np.isfinite(want[:69]).all() and np.isnan(want[69]).all()
    # both round a sum of at most 70 weighted values to bf16; weights are rounded to bf16 on the device
    assert np.abs(got[:64] - want[:64]).max() <= 2.0 ** -7 * np.abs(want[:64]).max()
    assert np.isnan(got[69]).all()


@pytest.mark.parametrize("pool", [DType.F16, DType.BF16])
@pytest.mark.parametrize("lead", [1.3, 4.7, 5.9])
def test_prefill_weight_of_the_largest_score_is_not_rounded(hip, pool, lead):
    """Key 64, the first of a second tile, leads key 0 by 2^lead and all others by far more; only its value is not
    zero.  Weights are relative to the largest score, so that its own is 1 in any format and a row's result has the
    errors of 32-bit sums alone: of the score (2^-24 of at most 8, doubled by the scale's rounding) and the division."""
    tokens = 130
    t, inputs = ragged_case(hip, [0], [tokens], 2, 2, 16, seed=66, dtype=DType.F32, pool_dtype=pool)
    q, keys, values = (np.zeros((tokens, 2, 128), np.float32) for _ in range(3))
    q[:, :, 0] = 1.0
    keys[:, :, 0] = -60.0
    keys[0, :, 0], keys[64, :, 0] = 0.0, to_f32(from_f32(np.array([lead]), pool), pool)[0]
    values[64] = 1.0
    inputs[:3] = [upload(hip, v, DType.F32) for v in (q, keys, values)]
    commands = CommandList()
    commands.dispatch_many(Op.paged_attention_ragged(float(np.log(2.0)), 16), inputs, [t["out"], t["keys"], t["values"]])
    run(hip, commands)
    got = to_f32(hip.read(t["out"]), DType.F32).reshape(tokens, 2, 128).astype(np.float64)
    scores = keys[:, 0, 0].astype(np.float64)
    for row in range(64, tokens):
        weights = np.exp2(scores[:row + 1])
        assert np.abs(got[row] / (weights[64] / weights.sum()) - 1.0).max() <= 2.0 ** -18


@pytest.mark.parametrize("dtype,pool", [(DType.BF16, DType.BF16), (DType.F32, DType.F16)])
def test_prefill_with_a_zero_scale_keeps_queries_without_a_number(cpu, hip, dtype, pool):
    """Every finite score is zero; zero times a NaN or an infinity is a NaN, and so is that row of that head.  (f32
    queries beyond the f16 range of their pool are held at its largest number, infinities too: only the NaN there.)"""
    infinities = dtype == pool
    def build(backend):
        t, inputs = ragged_case(backend, [3], [70], 16, 8, 16, seed=67, dtype=dtype, pool_dtype=pool)
        queries = normal_bf16(67, 3, (70, 16, 128)).astype(np.float32)
        queries[5, 2, 17] = np.nan
        if infinities:
            queries[40, 9, 126], queries[69, 0, 0] = np.inf, -np.inf
        inputs[0] = upload(backend, queries, dtype)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.0, 16), inputs, [t["out"], t["keys"], t["values"]])
        return commands, [t["out"]]
    (cpu_out, _), _ = differential(cpu, hip, build, bar=DType.F16 if dtype == DType.F32 else None)
    nan = np.isnan(to_f32(cpu.read(cpu_out[0]), dtype).reshape(70, 16, 128))
    assert nan[5, 2].all() and nan.sum() == (3 if infinities else 1) * 128


DTYPE_MIXES = [
    # query and new rows, pools, output
    (DType.F32, DType.F16, DType.F32),      # the qwen3-coder engine
    (DType.F16, DType.F16, DType.F16),
    (DType.F16, DType.F16, DType.BF16),
    (DType.BF16, DType.BF16, DType.F32),
    (DType.F32, DType.BF16, DType.F32),     # f32 activations against a bf16 cache
    (DType.F32, DType.BF16, DType.BF16),
]


@pytest.mark.parametrize("dtype,pool_dtype,out_dtype", DTYPE_MIXES)
@pytest.mark.parametrize("contexts,counts,hq,hkv,pt,promise", [
    ([300, 1, 2047, 700, 15, 16, 0], [1] * 7, 32, 4, 16, True),
    ([300, 1, 2047, 700, 15, 16, 0], [1] * 7, 32, 4, 64, False),
    ([0, 130, 33, 900], [70, 1, 45, 1], 40, 8, 16, False),
    (list(range(0, 520, 13)), [1] * 40, 16, 8, 16, True)])
def test_ragged_attention_across_activation_and_pool_dtypes(cpu, hip, dtype, pool_dtype, out_dtype, contexts,
                                                            counts, hq, hkv, pt, promise):
    """f16 or bf16 pools fed by rows of their own dtype or by f32 rows, any float output: the
    stored rows are rounded once, exactly as the oracle rounds them, so the pools match bit for
    bit; a second layer reuses the work plan on other pools."""
    scale = 1.0 / math.sqrt(128)

    def build(backend):
        t, inputs = ragged_case(backend, contexts, counts, hq, hkv, pt, seed=69, dtype=dtype,
                                pool_dtype=pool_dtype, out_dtype=out_dtype)
        # new rows with more significand bits than the pools hold
        rows = sum(counts)
        inputs[1] = upload(backend, normal_bf16(69, 6, (rows, hkv, 128)) * 1.001, dtype)
        inputs[2] = upload(backend, normal_bf16(69, 7, (rows, hkv, 128)) * 1.001, dtype)
        physical = t["keys"].shape[0]
        other_k = upload(backend, normal_bf16(69, 8, (physical, pt, hkv, 128)), pool_dtype)
        other_v = upload(backend, normal_bf16(69, 9, (physical, pt, hkv, 128)), pool_dtype)
        out2 = backend.alloc(out_dtype, t["out"].shape)
        op = Op.paged_attention_ragged(scale, pt, one_row_per_lane=promise)
        commands = CommandList()
        commands.dispatch_many(op, inputs, [t["out"], t["keys"], t["values"]])
        commands.dispatch_many(op, inputs, [out2, other_k, other_v])
        return commands, [t["out"], out2, t["keys"], t["values"], other_k, other_v]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build, bar=pool_dtype)
    for index in (2, 3, 4, 5):
        assert cpu.read(cpu_out[index]) == hip.read(hip_out[index])


def test_f32_queries_beyond_the_f16_range_stay_finite(cpu, hip):
    """An f32 query element no f16 holds: the oracle's scores are huge but finite, and so are the
    device's (the element is held at the largest finite f16); the winner of such a softmax is
    one key on both sides."""
    def build(backend):
        t, inputs = ragged_case(backend, [40, 7], [1, 1], 8, 2, 16, seed=70, dtype=DType.F32,
                                pool_dtype=DType.F16)
        values = normal_bf16(70, 3, (2, 8, 128)).astype(np.float32)
        values[0, 3, 5] = 3.0e6
        values[1, 0, 100] = -1.0e9
        inputs[0] = upload(backend, values, DType.F32)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 16), inputs, [t["out"], t["keys"], t["values"]])
        return commands, [t["out"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build, bar=DType.F16)
    assert np.isfinite(to_f32(hip.read(hip_out[0]), DType.F32)).all()


@pytest.mark.parametrize("contexts,counts,hq,hkv", [([300, 40, 2047, 700], [1, 1, 1, 1], 32, 4),
                                                    ([0, 130, 33], [70, 1, 45], 16, 8)])
def test_ragged_attention_layers_share_metadata_until_it_is_rewritten(cpu, hip, contexts, counts, hq, hkv):
    """One command list the way a model step records it: two layers (their own pools) attend with
    the same tables, starts and cu_seqlens, then the starts are overwritten on the device and a third
    dispatch must follow the new values."""
    scale, pt = 1.0 / math.sqrt(128), 16
    moved = [max(0, c - 5) for c in contexts]

    def build(backend):
        t, inputs = ragged_case(backend, contexts, counts, hq, hkv, pt, seed=64)
        physical = t["keys"].shape[0]
        other_k = upload(backend, normal_bf16(64, 8, (physical, pt, hkv, 128)), DType.BF16)
        other_v = upload(backend, normal_bf16(64, 9, (physical, pt, hkv, 128)), DType.BF16)
        out2, out3 = (backend.alloc(DType.BF16, t["out"].shape) for _ in range(2))
        new_starts = upload(backend, np.array(moved), DType.U32)
        op = Op.paged_attention_ragged(scale, pt)
        commands = CommandList()
        commands.dispatch_many(op, inputs, [t["out"], t["keys"], t["values"]])
        commands.dispatch_many(op, inputs, [out2, other_k, other_v])
        commands.dispatch(Op.copy(), [new_starts], t["starts"])
        commands.dispatch_many(op, inputs, [out3, t["keys"], t["values"]])
        return commands, [t["out"], out2, out3, t["keys"], other_k]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[3]) == hip.read(hip_out[3]) and cpu.read(cpu_out[4]) == hip.read(hip_out[4])


@pytest.mark.parametrize("contexts,hq,hkv,pt", [
    ([17, 64, 130, 511], 16, 8, 16), ([300, 1, 2047, 700, 15, 16, 0], 32, 4, 16), ([100, 257], 32, 4, 64),
    ([0], 8, 2, 16), (list(range(0, 520, 13)), 32, 4, 16)])
def test_decode_batch_with_the_one_row_promise_stores_the_new_rows_itself(cpu, hip, contexts, hq, hkv, pt):
    """With the recorder's promise of one query row per lane the attention kernel stores the new
    key/value rows itself: pools still match the oracle bit for bit (lanes at context 0 attend
    nothing but the row just stored), and so does a second layer that reuses the work plan."""
    scale = 1.0 / math.sqrt(128)

    def build(backend):
        t, inputs = ragged_case(backend, contexts, [1] * len(contexts), hq, hkv, pt, seed=66)
        physical = t["keys"].shape[0]
        other_k = upload(backend, normal_bf16(66, 8, (physical, pt, hkv, 128)), DType.BF16)
        other_v = upload(backend, normal_bf16(66, 9, (physical, pt, hkv, 128)), DType.BF16)
        out2 = backend.alloc(DType.BF16, t["out"].shape)
        op = Op.paged_attention_ragged(scale, pt, one_row_per_lane=True)
        commands = CommandList()
        commands.dispatch_many(op, inputs, [t["out"], t["keys"], t["values"]])
        commands.dispatch_many(op, inputs, [out2, other_k, other_v])
        return commands, [t["out"], out2, t["keys"], t["values"], other_k, other_v]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    for index in (2, 3, 4, 5):
        assert cpu.read(cpu_out[index]) == hip.read(hip_out[index])


def test_a_broken_one_row_promise_is_reported(cpu, hip):
    def build(backend):
        t, inputs = ragged_case(backend, [40, 0, 100], [1, 2, 1], 8, 2, 16, seed=67)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 16, one_row_per_lane=True), inputs,
                               [t["out"], t["keys"], t["values"]])
        return commands, []
    for backend in (cpu, hip):
        commands, _ = build(backend)
        with pytest.raises(BackendError) as info:
            run(backend, commands)
        assert info.value.status == Status.DEVICE_ERROR_FLAG and info.value.index == 1


def test_the_one_row_promise_keeps_inactive_lanes_and_stale_pages_unwritten(cpu, hip):
    def build(backend, corrupt):
        t, inputs = ragged_case(backend, [33, 70, 5], [1, 1, 1], 8, 4, 16, seed=68,
                                activity=[1, 0, 1], corrupt=corrupt)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 16, one_row_per_lane=True), inputs,
                               [t["out"], t["keys"], t["values"]])
        return commands, [t["out"], t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, lambda backend: build(backend, None))
    assert cpu.read(cpu_out[1]) == hip.read(hip_out[1]) and cpu.read(cpu_out[2]) == hip.read(hip_out[2])
    # lane 0 appends at position 33 = logical page 2: stale there, nothing of lane 0 is written
    commands, tensors = build(hip, (0, 2))
    before = hip.read(tensors[1])
    with pytest.raises(BackendError) as info:
        run(hip, commands)
    assert info.value.status == Status.DEVICE_ERROR_FLAG and info.value.index == 2
    # exactly one token row of the key pool changed: lane 2's (lane 1 is inactive, lane 0 refused)
    token_row = 4 * 128 * 2
    changed = np.frombuffer(hip.read(tensors[1]), np.uint8).reshape(-1, token_row) != \
        np.frombuffer(before, np.uint8).reshape(-1, token_row)
    assert changed.any(axis=1).sum() == 1
    assert not to_f32(hip.read(tensors[0]), DType.BF16).reshape(3, -1)[0].any()


@pytest.mark.parametrize("hq,hkv,pt,counts,cu", [
    (8, 4, 16, [1, 1, 1, 1], [0, 100, 4, 4, 4]),      # decode batch: lane 0 claims 100 rows of 4
    (8, 4, 16, [20, 30, 14], [0, 20, 10, 64]),        # prefill groups: lane 1 runs backwards
    (8, 4, 16, [20, 30, 14], [0, 20, 50, 4000]),      # the last lane runs past the packed batch
    (6, 2, 8, [3, 2, 1], [0, 3, 70, 6])])             # a page size only the generic kernels take
def test_ragged_attention_refuses_malformed_cu_seqlens(cpu, hip, hq, hkv, pt, counts, cu):
    """cu_seqlens is read on the device: ranges that run backwards or beyond the packed batch fail
    the dispatch (lowest offending lane reported), every output row reads zero, and neither the
    pools nor the allocations around q and out are touched.  Every kernel exits normally."""
    contexts = [40 + 3 * lane for lane in range(len(counts))]
    bad_lane = next(l for l in range(len(counts)) if cu[l + 1] < cu[l] or cu[l + 1] > sum(counts))
    for promise in (False, True) if max(counts) == 1 else (False,):
        for backend in (cpu, hip):
            guard_before = upload(backend, normal_bf16(72, 1, (4096,)), DType.BF16)
            t, inputs = ragged_case(backend, contexts, counts, hq, hkv, pt, seed=71)
            guard_after = upload(backend, normal_bf16(72, 2, (4096,)), DType.BF16)
            inputs[5] = upload(backend, np.array(cu), DType.U32)
            backend.write(t["out"], np.full(sum(counts) * hq * 128, 0x3f80, np.uint16).tobytes())
            pools = backend.read(t["keys"]), backend.read(t["values"])
            guards = backend.read(guard_before), backend.read(guard_after)
            commands = CommandList()
            commands.dispatch_many(Op.paged_attention_ragged(0.09, pt, one_row_per_lane=promise), inputs,
                                   [t["out"], t["keys"], t["values"]])
            with pytest.raises(BackendError) as info:
                run(backend, commands)
            assert info.value.status == Status.DEVICE_ERROR_FLAG and info.value.index == bad_lane
            assert not np.frombuffer(backend.read(t["out"]), np.uint16).any()
            assert (backend.read(t["keys"]), backend.read(t["values"])) == pools
            assert (backend.read(guard_before), backend.read(guard_after)) == guards
            # and the backend keeps working: the same batch with its real cu_seqlens succeeds
            inputs[5] = t["cu"]
            commands = CommandList()
            commands.dispatch_many(Op.paged_attention_ragged(0.09, pt), inputs, [t["out"], t["keys"], t["values"]])
            run(backend, commands)
            assert np.frombuffer(backend.read(t["out"]), np.uint16).any()


@pytest.mark.parametrize("promise", [False, True])
def test_rows_of_no_lane_leave_the_promised_rows_stored(cpu, hip, promise):
    """More rows than lanes, the last ones of no lane, under the promise of one row a lane: the lanes' new rows are stored
    and attended, the others read zeros."""
    def build(backend):
        t, inputs = ragged_case(backend, [33, 70, 5], [1, 1, 1], 8, 4, 16, seed=70)
        tables = np.frombuffer(backend.read(t["tables"]), np.uint32).reshape(3, -1, 2)
        inputs[3] = upload(backend, tables[:2], DType.U32)
        inputs[5] = upload(backend, np.array([0, 1, 2]), DType.U32)
        inputs[6] = upload(backend, np.array([33, 70]), DType.U32)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 16, one_row_per_lane=promise), inputs,
                               [t["out"], t["keys"], t["values"]])
        return commands, [t["out"], t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[1]) == hip.read(hip_out[1]) and cpu.read(cpu_out[2]) == hip.read(hip_out[2])
    assert not to_f32(hip.read(hip_out[0]), DType.BF16).reshape(3, -1)[2].any()


def test_decode_item_of_more_than_64_pages(cpu, hip):
    """Pages of an odd multiple of sixteen tokens: the 64 that a wave looks up at once may end within a tile of 32 keys, whose
    other half belongs to the next 64.  6000 rows leave a lane two items: the second begins at key 3232, its first page at
    3216, and its 64 pages end at 6288, in the middle of a tile.  Were that half read through the first page, the values of
    page 67, a hundred times the others, would count twice."""
    contexts = [6463, 80, 0]

    def build(backend):
        t, inputs = ragged_case(backend, contexts, [1, 1, 5998], 2, 1, 48, seed=71)
        tables = np.frombuffer(backend.read(t["tables"]), np.uint32).reshape(3, -1, 2)
        values = to_f32(backend.read(t["values"]), DType.BF16).reshape(-1, 48, 128).copy()
        values[tables[0, 67, 0]] *= 100.0
        backend.write(t["values"], orc.f32_to_bf16(values).tobytes())
        inputs[3] = upload(backend, tables[:2], DType.U32)
        inputs[5] = upload(backend, np.array([0, 1, 2]), DType.U32)
        inputs[6] = upload(backend, np.array(contexts[:2]), DType.U32)
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 48, one_row_per_lane=True), inputs,
                               [t["out"], t["keys"], t["values"]])
        return commands, [t["out"]]
    differential(cpu, hip, build)


def test_ragged_attention_skips_inactive_lanes(cpu, hip):
    def build(backend):
        t, inputs = ragged_case(backend, [33, 70, 5], [1, 1, 1], 8, 4, 16, seed=62, activity=[1, 0, 1])
        commands = CommandList()
        commands.dispatch_many(Op.paged_attention_ragged(0.09, 16), inputs, [t["out"], t["keys"], t["values"]])
        return commands, [t["out"], t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[1]) == hip.read(hip_out[1])
    assert not to_f32(hip.read(hip_out[0]), DType.BF16).reshape(3, -1)[1].any()


def test_ragged_attention_reports_a_stale_page(hip):
    t, inputs = ragged_case(hip, [33, 70, 5], [1, 1, 1], 8, 4, 16, seed=63, corrupt=(1, 2))
    commands = CommandList()
    commands.dispatch_many(Op.paged_attention_ragged(0.09, 16), inputs, [t["out"], t["keys"], t["values"]])
    with pytest.raises(BackendError) as info:
        run(hip, commands)
    assert info.value.status == Status.DEVICE_ERROR_FLAG and info.value.index == 2
    out = to_f32(hip.read(t["out"]), DType.BF16).reshape(3, -1)
    assert not out[1].any() and out[0].any() and out[2].any()


def test_empty_batches_are_accepted_and_change_nothing(cpu, hip):
    """Zero rows through the projections, the router and a program, and a ragged batch whose lanes
    bring no query tokens: both backends accept them, write nothing and report nothing."""
    weights = Quantised(81, 1, (64, 128))
    stacked = Quantised(81, 2, (64, 128), experts=4)

    def build(backend):
        x = backend.alloc(DType.BF16, (0, 128))
        out = backend.alloc(DType.BF16, (0, 64))
        logits = backend.alloc(DType.BF16, (0, 4))
        route_weights, route_ids = backend.alloc(DType.BF16, (0, 2)), backend.alloc(DType.U32, (0, 2))
        routed = backend.alloc(DType.BF16, (0, 2, 64))
        t, inputs = ragged_case(backend, [5, 9], [0, 0], 8, 4, 16, seed=82)
        commands = CommandList()
        commands.dispatch(Op.quant_matmul(4, 64), [x, *weights.upload(backend)], out)
        commands.dispatch_many(Op.top_k(2, True), [logits], [route_weights, route_ids])
        commands.dispatch(Op.gather_quant_matmul(4, 64), [x, *stacked.upload(backend), route_ids], routed)
        commands.dispatch_kernel(backend.prepare_program(programs.add_elements()), [out, out],
                                 [backend.alloc(DType.BF16, (0, 64))])
        commands.dispatch_many(Op.paged_attention_ragged(0.1, 16), inputs, [t["out"], t["keys"], t["values"]])
        return commands, [t["keys"], t["values"]]
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    assert cpu.read(cpu_out[0]) == hip.read(hip_out[0]) and cpu.read(cpu_out[1]) == hip.read(hip_out[1])


# ------------------------------------------------------------------ programs and glue

@pytest.mark.parametrize("dtype", [DType.BF16, DType.F32])
def test_engine_row_programs(cpu, hip, dtype):
    """The fused row-program kernels on bf16 and on f32 rows.  f32 results are held to the f16 bar:
    the rotation angle at position 32767 carries the few-ulp difference between the device's and
    the host's powf, about 3e-3 rad."""
    rows, hidden, heads, half = 6, 1024, 24, 64
    x_values = normal_bf16(71, 1, (rows, hidden))
    u_values = normal_bf16(71, 2, (rows, hidden))
    w_values = 1.0 + 0.1 * normal_bf16(71, 3, (hidden,))
    qk_values = normal_bf16(71, 4, (rows, heads, 2 * half))
    norm_values = 1.0 + 0.1 * normal_bf16(71, 5, (heads, 2 * half))
    positions = np.array([0, 1, 17, 511, 4095, 32767], dtype=np.float32)

    def build(backend):
        x, u = upload(backend, x_values, dtype), upload(backend, u_values, dtype)
        w = upload(backend, w_values, dtype).broadcast((rows, hidden))
        normed = backend.alloc(dtype, (rows, hidden))
        hidden_out, normed2 = backend.alloc(dtype, (rows, hidden)), backend.alloc(dtype, (rows, hidden))
        qk = upload(backend, qk_values, dtype)
        norm = upload(backend, norm_values, dtype).broadcast((rows, heads, 2 * half))
        pos = upload(backend, positions, DType.F32).reshape((rows, 1, 1)).broadcast((rows, heads, half))
        rotated = backend.alloc(dtype, (rows, heads, 2 * half))
        commands = CommandList()
        commands.dispatch_kernel(backend.prepare_program(programs.rms_norm_rows(1e-6)), [x, w], [normed])
        commands.dispatch_kernel(backend.prepare_program(programs.residual_norm_rows(1e-6)), [x, u, w],
                                 [hidden_out, normed2])
        commands.dispatch_kernel(
            backend.prepare_program(programs.qk_norm_rope_rows(128.0, 1e-6, 1e6)),
            [qk.narrow(2, 0, half), qk.narrow(2, half, half), norm.narrow(2, 0, half),
             norm.narrow(2, half, half), pos],
            [rotated.narrow(2, 0, half), rotated.narrow(2, half, half)])
        return commands, [normed, hidden_out, normed2, rotated]
    differential(cpu, hip, build, abs_=2e-2, bar=DType.F16 if dtype == DType.F32 else None)


@pytest.mark.parametrize("rows,heads", [(512, 3), (1029, 24)])
@pytest.mark.parametrize("dtype", [DType.BF16, DType.F32])
def test_head_norm_and_rotation_over_many_rows(cpu, hip, rows, heads, dtype):
    """From 512 rows on a workgroup takes a row and a wave two heads: an odd number of heads, rows that lie further apart
    than their heads.  f32 results are held to the f16 bar, as above."""
    half = 64
    qk_values, norm_values = normal_bf16(73, rows, (rows, heads + 1, 2 * half)), 1.0 + 0.1 * normal_bf16(73, 5, (heads, 2 * half))
    positions = (np.arange(rows) * 7 % 4099).astype(np.float32)

    def build(backend):
        qk = upload(backend, qk_values, dtype).narrow(1, 1, heads)   # (rows that lie further apart than their heads)
        norm = upload(backend, norm_values, dtype).broadcast((rows, heads, 2 * half))
        pos = upload(backend, positions, DType.F32).reshape((rows, 1, 1)).broadcast((rows, heads, half))
        rotated = backend.alloc(dtype, (rows, heads, 2 * half))
        commands = CommandList()
        commands.dispatch_kernel(
            backend.prepare_program(programs.qk_norm_rope_rows(128.0, 1e-6, 1e6)),
            [qk.narrow(2, 0, half), qk.narrow(2, half, half), norm.narrow(2, 0, half),
             norm.narrow(2, half, half), pos],
            [rotated.narrow(2, 0, half), rotated.narrow(2, half, half)])
        return commands, [rotated]
    differential(cpu, hip, build, abs_=2e-2, bar=DType.F16 if dtype == DType.F32 else None)


@pytest.mark.parametrize("rows,width", [(5, 64), (130, 1024), (3, 20)])
def test_engine_element_programs_on_the_halves_of_a_stacked_projection(cpu, hip, rows, width):
    """silu_mul_elements over the gate and up halves of one [rows, 2 * width] tensor and
    add_elements (crates/forja-sdk/src/nn/blocks.rs:408-416); the last width is not a multiple of
    eight."""
    stacked_values = 3.0 * normal_bf16(72, 1, (rows, 2 * width))
    residual_values = normal_bf16(72, 2, (rows, width))

    def build(backend):
        stacked = upload(backend, stacked_values, DType.BF16)
        residual = upload(backend, residual_values, DType.BF16)
        activated, summed = (backend.alloc(DType.BF16, (rows, width)) for _ in range(2))
        commands = CommandList()
        commands.dispatch_kernel(backend.prepare_program(programs.silu_mul_elements()),
                                 [stacked.narrow(1, 0, width), stacked.narrow(1, width, width)], [activated])
        commands.dispatch_kernel(backend.prepare_program(programs.add_elements()), [residual, activated],
                                 [summed])
        return commands, [activated, summed]
    differential(cpu, hip, build)


def test_map_programs_casts_index_select(cpu, hip):
    values = np.array([[-1.5, 3.7, np.nan, 5e9, 0.25, -0.0, 7.0, 1e-3]], dtype=np.float32).repeat(3, axis=0)
    b = ProgramBuilder(ProgramKind.MAP)
    v, w = b.input(0), b.input(1)
    as_u32 = b.cast(ValueType.U32, v)
    b.output(0, b.cast(ValueType.F32, as_u32))
    column = b.cast(ValueType.F32, b.index(1))
    big = b.binary(BinOp.GT, column, b.const(3.5))
    b.output(1, b.select(big, b.binary(BinOp.MAX, v, b.const(0.0)), b.unary(UnOp.ABS, v)))
    b.output(2, b.cast(ValueType.F32, b.binary(BinOp.ADD, w, b.extent(1))))
    program = b.finish()

    def build(backend):
        x = upload_raw(backend, values, DType.F32, values.shape)
        ids = upload(backend, np.arange(24).reshape(3, 8), DType.U32)
        outs = [backend.alloc(DType.F32, values.shape) for _ in range(3)]
        commands = CommandList()
        commands.dispatch_kernel(backend.prepare_program(program), [x, ids], outs)
        return commands, outs
    (cpu_out, _), (hip_out, _) = differential(cpu, hip, build)
    for a, b_ in zip(cpu_out, hip_out):
        assert cpu.read(a) == hip.read(b_)


def random_program(rng, kind, inputs, length, exact):
    """A typed random SSA program over `inputs` = [ValueType of input slot ...]: every operand is
    drawn from earlier values of the right type, the way the reference's proptest generator does
    (crates/forja-metal/tests/map_programs.rs).  `exact` keeps to operations IEEE fixes bit for bit
    (no division, roots or transcendentals, no sum reduction)."""
    b = ProgramBuilder(kind)
    of_type = {ValueType.F32: [], ValueType.U32: [], ValueType.BOOL: []}
    for slot, value_type in enumerate(inputs):
        of_type[value_type].append(b.input(slot))
    of_type[ValueType.F32].append(b.const(float(rng.choice([0.0, -1.5, 2.0, 0.3, 1e-3]))))
    of_type[ValueType.U32].append(b.index(1))
    of_type[ValueType.U32].append(b.extent(1))
    pick = lambda t: int(rng.choice(of_type[t]))
    reductions = 0
    exact_unary = [UnOp.NEG, UnOp.ABS, UnOp.FLOOR]
    loose_unary = [UnOp.NEG, UnOp.ABS, UnOp.TANH, UnOp.SIGMOID, UnOp.SIN, UnOp.COS]
    exact_binary = [BinOp.ADD, BinOp.SUB, BinOp.MUL, BinOp.MIN, BinOp.MAX]
    compare = [BinOp.LT, BinOp.LE, BinOp.EQ, BinOp.NE, BinOp.GE, BinOp.GT]
    for _ in range(length):
        # the loose set stays with continuous operations: a comparison, floor or integer cast of a
        # value that differs in its last bit may legitimately take the other branch
        choice = int(rng.integers(0, 9)) if exact else int(rng.choice([0, 1, 2, 7, 8]))
        if choice == 0:
            of_type[ValueType.F32].append(b.unary(rng.choice(exact_unary if exact else loose_unary),
                                                  pick(ValueType.F32)))
        elif choice in (1, 2):
            ops = exact_binary
            of_type[ValueType.F32].append(b.binary(rng.choice(ops), pick(ValueType.F32), pick(ValueType.F32)))
        elif choice == 3:
            of_type[ValueType.U32].append(b.binary(rng.choice(exact_binary), pick(ValueType.U32),
                                                   pick(ValueType.U32)))
        elif choice == 4:
            operand = ValueType.F32 if rng.integers(0, 2) else ValueType.U32
            of_type[ValueType.BOOL].append(b.binary(rng.choice(compare), pick(operand), pick(operand)))
        elif choice == 5 and of_type[ValueType.BOOL]:
            chosen = ValueType.F32 if rng.integers(0, 2) else ValueType.U32
            of_type[chosen].append(b.select(pick(ValueType.BOOL), pick(chosen), pick(chosen)))
        elif choice == 6:
            source = [t for t in of_type if of_type[t]][int(rng.integers(0, sum(1 for t in of_type if of_type[t])))]
            target = ValueType(int(rng.integers(0, 3)))
            of_type[target].append(b.cast(target, pick(source)))
        elif choice == 7 and kind == ProgramKind.ROW and reductions < 4:   # MAX_REDUCTIONS, program.rs:27
            reductions += 1
            ops = [RedOp.MAX, RedOp.MIN] if exact else [RedOp.MAX, RedOp.MIN, RedOp.SUM]
            of_type[ValueType.F32].append(b.reduce(rng.choice(ops), pick(ValueType.F32)))
        else:
            of_type[ValueType.F32].append(b.cast(ValueType.F32, pick(ValueType.U32)))
    for slot in range(2):
        b.output(slot, int(of_type[ValueType.F32][-1 - slot]))
    return b.finish()


@pytest.mark.parametrize("kind", [ProgramKind.MAP, ProgramKind.ROW])
@pytest.mark.parametrize("exact", [True, False])
def test_random_typed_programs_agree_with_the_interpreter(cpu, hip, kind, exact):
    """25 seeded random programs per case over a broadcast row, a strided view and an integer
    tensor: bit for bit where IEEE fixes the result, to 1e-5 where libm or the order of a sum does
    not."""
    rows, width = 5, 37
    rng = np.random.default_rng(1234 + 2 * int(kind) + int(exact))
    first = orc.fill_normal_f32(73, 1, rows * width).reshape(rows, width)
    second = orc.fill_normal_f32(73, 2, 2 * width).reshape(1, 2 * width)
    for case in range(25):
        program = random_program(rng, kind, [ValueType.F32, ValueType.F32, ValueType.U32],
                                 length=int(rng.integers(4, 24)), exact=exact)

        def build(backend):
            x = upload(backend, first, DType.F32)
            y = upload(backend, second, DType.F32).slice([Slice(0, 1), Slice(1, width, 2)]).broadcast(
                (rows, width))
            ids = upload(backend, (np.arange(rows * width) * 7919) % 1000, DType.U32).reshape((rows, width))
            outs = [backend.alloc(DType.F32, (rows, width)) for _ in range(2)]
            commands = CommandList()
            commands.dispatch_kernel(backend.prepare_program(program), [x, y, ids], outs)
            return commands, outs
        try:
            if exact:
                (cpu_out, _), (hip_out, _) = differential(cpu, hip, build, rel=0.0, abs_=0.0, norm_tol=0.0)
                for a, b_ in zip(cpu_out, hip_out):
                    assert cpu.read(a) == hip.read(b_), (case, program)
            else:
                differential(cpu, hip, build, rel=1e-5, abs_=1e-6, norm_tol=1e-5)
        except AssertionError as error:
            raise AssertionError(f"program {case}: {program}") from error


def test_program_limits_are_refused_when_prepared(cpu, hip):
    """Five reductions, a reduction in a map program, an operand that is not earlier
    (validate_structure, crates/forja-core/src/program.rs:1052-1094)."""
    five = ProgramBuilder(ProgramKind.ROW)
    value = five.input(0)
    for _ in range(5):
        value = five.reduce(RedOp.MAX, value)
    five.output(0, value)
    in_map = ProgramBuilder(ProgramKind.MAP)
    in_map.output(0, in_map.reduce(RedOp.SUM, in_map.input(0)))
    forward = Program(ProgramKind.MAP, [Inst.input(0), Inst.unary(UnOp.NEG, 2), Inst.const(1.0)], [(0, 1)])
    for backend in (cpu, hip):
        for program in (five.finish(), in_map.finish(), forward):
            with pytest.raises(BackendError) as info:
                backend.prepare_program(program)
            assert info.value.status == Status.INVALID_INPUT


def test_softmax_row_program_with_max_and_sum_reductions(cpu, hip):
    b = ProgramBuilder(ProgramKind.ROW)
    x = b.input(0)
    e = b.unary(UnOp.EXP, b.sub(x, b.reduce(RedOp.MAX, x)))
    b.output(0, b.div(e, b.reduce(RedOp.SUM, e)))
    program = b.finish()
    values = orc.fill_normal_f32(72, 1, 5 * 700).reshape(5, 700)

    def build(backend):
        x = upload(backend, values, DType.F32)
        out = backend.alloc(DType.F32, (5, 700))
        commands = CommandList()
        commands.dispatch_kernel(backend.prepare_program(program), [x], [out])
        return commands, [out]
    differential(cpu, hip, build, rel=1e-4, abs_=1e-6, norm_tol=1e-5)


def test_quant_embed_copy_matmul_rms_norm_rope(cpu, hip):
    table = Quantised(81, 1, (300, 128))
    ids_values = np.array([[5, 299, 0], [17, 100, 3]], dtype=np.uint32)
    experts_values = normal_bf16(81, 2, (6, 32, 4))
    weights_values = normal_bf16(81, 3, (6, 4, 1))
    x_values = normal_bf16(81, 4, (7, 16, 128))

    def build(backend):
        ids = upload(backend, ids_values, DType.U32)
        embedded = backend.alloc(DType.BF16, (2, 3, 128))
        experts = upload(backend, experts_values, DType.BF16)
        weights = upload(backend, weights_values, DType.BF16)
        combined = backend.alloc(DType.BF16, (6, 32, 1))
        x = upload(backend, x_values, DType.BF16)
        copied = backend.alloc(DType.F32, (16, 7, 128))
        normed = backend.alloc(DType.BF16, (7, 16, 128))
        w = upload(backend, np.linspace(0.5, 1.5, 128), DType.F32)
        roped = backend.alloc(DType.BF16, (7, 16, 128))
        pos = upload(backend, np.array([0, 1, 2, 100, 1000, 20000, 32767]), DType.U32)
        commands = CommandList()
        commands.dispatch(Op.quant_embed(4, 64), [*table.upload(backend), ids], embedded)
        commands.dispatch(Op.matmul(), [experts, weights], combined)     # MoE combine shape
        commands.dispatch(Op.copy(), [x.permute([1, 0, 2])], copied)
        commands.dispatch(Op.rms_norm(1e-6), [x, w], normed)
        commands.dispatch(Op.rope(1e6), [x, pos], roped)
        return commands, [embedded, combined, copied, normed, roped]
    differential(cpu, hip, build, abs_=2e-2)


@pytest.mark.parametrize("dtype", [DType.BF16, DType.F32])
def test_quant_embed_rows_of_every_alignment(cpu, hip, dtype):
    """Output rows that take the eight-value stores, dense and strided, and rows that start off them."""
    table, ids_values = Quantised(83, 1, (37, 320)), np.array([36, 0, 3, 5, 36, 11, 2], dtype=np.uint32)

    def build(backend):
        ids, triple = upload(backend, ids_values, DType.U32), table.upload(backend)
        plain = backend.alloc(dtype, (7, 320))
        whole = upload(backend, np.ones((7, 339)), dtype)
        wide = upload(backend, np.ones((7, 336)), dtype)
        commands = CommandList()
        for out in (plain, whole.narrow(1, 1, 320), wide.narrow(1, 8, 320)):
            commands.dispatch(Op.quant_embed(4, 64), [*triple, ids], out)
        return commands, [plain, whole, wide]
    differential(cpu, hip, build)


def test_quant_embed_zeroes_bad_rows_and_reports_the_lowest_bad_id(cpu, hip):
    """lib.rs:3020-3037 for the quantised table"""
    table = Quantised(82, 1, (300, 128))
    ids_values = np.array([5, 1000, 0, 999], dtype=np.uint32)

    def build(backend):
        ids = upload(backend, ids_values, DType.U32)
        embedded = upload(backend, np.ones((4, 128)), DType.BF16)
        commands = CommandList()
        commands.dispatch(Op.quant_embed(4, 64), [*table.upload(backend), ids], embedded)
        return commands, [embedded]
    results = differential(cpu, hip, build, expect_error={Status.INDEX_OUT_OF_RANGE})
    assert results[0][1].index == 999 and results[1][1].index == 999
