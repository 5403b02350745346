"""The prompt-chunk GEMM with weights decoded in registers, around the edges
of its tiles, against the oracle's half-operand product within the
reference's roundoff bound (matrix_precision.rs:119-142)."""
import ctypes

import numpy as np
import pytest

import oracle as O
import packers as P
from _util import Guarded, say
from test_gpu_skinny import product, weights

pytestmark = pytest.mark.gpu

# Partial row and column tiles, one to nine 256-column steps, on whichever
# kernel the choice takes; test_every_tile pins the tile and the K parts.
SHAPES = [(32, 260, 2304), (33, 1100, 256), (64, 256, 512), (65, 20004, 256), (97, 6144, 1280), (130, 516, 2048),
          (200, 132, 1280), (257, 8196, 512), (500, 12288, 256)]


@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, P.Q5_K, P.Q6_K, P.Q4_0, P.Q4_1])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_prompt_chunk(lib, fmt, m, n, k):
    from oco_amd import synth
    say("prompt chunk", fmt, m, n, k)
    w = weights(fmt, n, k, 11 + n)
    x = synth.bf16_bits(synth.activations(12, m * k)).reshape(m, k)
    rows = np.unique(np.r_[0:8, m // 2:m // 2 + 8, m - 9:m].clip(0, m - 1))
    half, mag = O.matmul_reference(fmt, w, x[rows], n, k, half_operands=True)
    got = product(lib, fmt, w, x, m, n, k, offset=7)[rows]
    assert np.all(np.abs(got - half) <= O.roundoff_bound(half, mag, k, False)), np.abs(got - half).max()


Q4 = (P.Q4_0, P.Q4_1, P.Q4_K)  # the formats of the wider tiles
TILES = [(fmt, mt, nt) for fmt in (P.Q8_0, P.Q4_K, P.Q5_K, P.Q6_K, P.Q4_0, P.Q4_1)
         for mt, nt in [(2, 1), (4, 1), (8, 1), (4, 2), (4, 3)] if (mt < 8 or fmt == P.Q6_K) and (nt == 1 or fmt in Q4)]


@pytest.mark.parametrize("fmt,mt,nt", TILES)
def test_every_tile(lib, fmt, mt, nt):
    """Each tile of each format (16 mt activation rows x 64 nt weight rows),
    pinned: one K part over an odd and an even number of 256-column steps and
    over one; two and four parts of unequal length; rows and columns one past
    and one short of whole tiles; rows that are not whole quads with one part
    and with several; f32 and bf16 outputs, bias, f16 activations."""
    from oco_amd import synth
    rows, cols = 16 * mt, 64 * nt
    for parts, m, n, k, options in [
            (1, rows + 1, cols + 4, 768, {}), (1, 2 * rows - 1, 2 * cols - 4, 512, dict(y_bf16=True)),
            (1, rows, cols, 256, dict(x_f16=True)), (1, 3 * rows - 5, cols + 1, 1024, dict(workspace=True)),
            (2, rows + 1, cols + 4, 768, dict(y_bf16=True)), (4, rows - 1, 2 * cols, 1280, {}),
            (4, rows + 3, cols - 1, 1280, dict(workspace=True)), (3, 2, 3 * cols + 3, 1024, dict(workspace=True, x_f16=True))]:
        say("tile", fmt, mt, nt, parts, m, n, k, options)
        w = weights(fmt, n, k, 51 + n)
        x = synth.activations(52, m * k).reshape(m, k)
        f16 = options.get("x_f16", False)
        x = x.astype(np.float16) if f16 else synth.bf16_bits(x).reshape(m, k)
        bias = np.random.default_rng(m + n).normal(size=n).astype(np.float32)
        half, mag = O.matmul_reference(fmt, w, x, n, k, half_operands=True)
        want = half + O.bf16_round(bias)
        with lib.overridden(lib.Knob.MATMUL_VENDOR, (2, mt, nt, parts)):
            route = lib.matmul_route(fmt, lib.Matrix(k, n, m, 0, 1, 1, 1), lib.DType.F16 if f16 else lib.DType.BF16)
            assert route == (lib.MatmulKernel.PANEL, mt, nt, parts)
            got = product(lib, fmt, w, x, m, n, k, bias=bias, offset=5, **options)
        bound = O.roundoff_bound(want, mag + np.abs(O.bf16_round(bias)), k, options.get("y_bf16", False))
        assert np.all(np.abs(got - want) <= bound), (parts, m, n, k, np.abs(got - want).max())


@pytest.mark.parametrize("fmt,n,k,choices", [
    (P.Q4_K, 12288, 4096, {32: (2, 1, 2), 128: (4, 1, 1), 256: (4, 3, 1), 320: (4, 2, 1), 512: (4, 3, 1), 640: None, 1024: None}),
    (P.Q4_K, 14336, 4096, {32: (2, 1, 2), 256: (4, 2, 1), 384: (4, 3, 1), 448: None, 512: None, 640: None}),
    (P.Q8_0, 4096, 4096, {64: (4, 1, 4), 256: (4, 1, 2), 512: None}), (P.Q6_K, 12288, 4096, {64: (4, 1, 4), 128: (8, 1, 1), 512: None}),
    (P.Q5_K, 4096, 4096, {64: (4, 1, 4), 448: (4, 1, 1), 1024: None}),
    (P.Q4_0, 12288, 4096, {64: (4, 2, 4), 128: (4, 3, 4), 512: (4, 3, 1), 640: None})])
def test_choice(lib, fmt, n, k, choices):
    """Tile and K parts, or the pass + GEMM (None), at row counts whose times
    on both are known (64 x 192 of 14336 x 4096 needs a third workgroup on some CUs
    from 448 rows on)."""
    for m, tile in choices.items():
        kernel, *got = lib.matmul_route(fmt, lib.Matrix(k, n, m, 0, 1, 1, 0), y_dtype=lib.DType.BF16)
        assert (kernel, *got) == ((lib.MatmulKernel.PANEL, *tile) if tile else (lib.MatmulKernel.GEMM, 0, 0, 0)), m


@pytest.mark.parametrize("fmt,values,m,k", [(P.Q4_K, (2, 3, 1, 1), 64, 512), (P.Q8_0, (2, 4, 2, 1), 64, 512), (P.Q4_K, (2, 8, 1, 1), 64, 512), (P.Q4_K, (2, 4, 1, 3), 40, 512),
                                            (P.Q4_K, (2, 4, 1, 2), 200, 512), (P.Q4_K, (2, 4, 1, 0), 64, 512), (P.Q4_K, (2,), 64, 512),
                                            (P.Q8_0, (2, 4, 1, 1), 64, 288), (1, (2, 4, 1, 1), 64, 512)])
def test_a_pinned_tile_that_cannot_run_is_refused(lib, fmt, values, m, k):
    """A tile that is not built, more parts than 256-column steps or than the
    workspace holds, no parts, a K that is not whole steps, another format."""
    say("tile refused", fmt, values, m, k)
    p, y = lib.Matrix(k, 128, m, 0, 1, 1, 0), lib.DeviceBuffer(m * 128 * 4)
    w, x = lib.DeviceBuffer.from_array(weights(fmt, 128, k, 61)), lib.DeviceBuffer(m * k * 2)
    with lib.overridden(lib.Knob.MATMUL_VENDOR, values):
        with pytest.raises(lib.OcoError, match="no panel tile"):
            lib.matmul(fmt, w, x, y, p)


@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, P.Q6_K, P.Q4_1])
@pytest.mark.parametrize("m,n,k", [(40, 132, 1280), (66, 2052, 256), (257, 8196, 512)])
def test_prompt_chunk_f16_input_bias_bf16_output(lib, fmt, m, n, k):
    from oco_amd import synth
    say("prompt chunk f16", fmt, m, n, k)
    w = weights(fmt, n, k, 13 + n)
    x = synth.activations(14, m * k).reshape(m, k).astype(np.float16)
    bias = np.random.default_rng(m).normal(size=n).astype(np.float32)
    got = product(lib, fmt, w, x, m, n, k, x_f16=True, y_bf16=True, bias=bias)
    half, mag = O.matmul_reference(fmt, w, x, n, k, half_operands=True)
    want = half + O.bf16_round(bias)
    assert np.all(np.abs(got - want) <= O.roundoff_bound(want, mag + np.abs(O.bf16_round(bias)), k, True))


def test_prompt_chunk_output_off_its_boundary(lib):
    """An output that is not 16-byte aligned takes the scalar stores."""
    from oco_amd import synth
    m, n, k = 65, 4100, 512
    w = weights(P.Q4_K, n, k, 23)
    x = synth.bf16_bits(synth.activations(24, m * k)).reshape(m, k)
    wb, xb = lib.DeviceBuffer.from_array(w), lib.DeviceBuffer.from_array(x)
    for dt, size, bits in ((lib.DType.F32, 4, np.uint32), (lib.DType.BF16, 2, np.uint16)):
        got = []
        for off in (0, size):
            y = Guarded(lib, m * n * size + 16)
            lib.matmul(P.Q4_K, wb, xb, y.ptr + off, lib.Matrix(k, n, m, 0, 1, 1, 0), y_dtype=dt)
            lib.synchronize()
            got.append(y.read(np.uint8)[off:off + m * n * size].view(bits))
        np.testing.assert_array_equal(*got)


def test_prompt_chunk_in_graph(lib):
    """K parts and their sum replay to the eager result."""
    from oco_amd import synth
    m, n, k = 48, 1024, 4096
    w = lib.DeviceBuffer.from_array(weights(P.Q4_K, n, k, 33))
    x = lib.DeviceBuffer.from_array(synth.bf16_bits(synth.activations(34, m * k)))
    p, y, eager = lib.Matrix(k, n, m, 0, 1, 1, 0), lib.DeviceBuffer(m * n * 2), lib.DeviceBuffer(m * n * 2)
    ws = lib.DeviceBuffer(lib.matmul_workspace(P.Q4_K, p))
    run = lambda out, s=None: lib.matmul(P.Q4_K, w, x, out, p, y_dtype=lib.DType.BF16, stream=s, workspace=ws, workspace_bytes=ws.nbytes)  # noqa: E731
    s = lib.Stream()
    g = lib.Graph(s, lambda: run(y, s))
    run(eager)
    lib.synchronize()
    want = eager.download(np.uint16)
    for _ in range(3):
        y.fill32(0)
        lib.synchronize()
        g.launch()
        s.sync()
        np.testing.assert_array_equal(y.download(np.uint16), want)
        run(eager)
        lib.synchronize()


def pool_high_water(reset=False):
    """Most bytes drawn at once from the device's stream-ordered pool."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    hip, pool, value = ctypes.CDLL(path), ctypes.c_void_p(), ctypes.c_uint64(0)
    assert hip.hipDeviceGetDefaultMemPool(ctypes.byref(pool), 0) == 0
    used_mem_high = 8  # hipMemPoolAttrUsedMemHigh
    if reset:
        assert hip.hipMemPoolSetAttribute(pool, used_mem_high, ctypes.byref(value)) == 0
    assert hip.hipMemPoolGetAttribute(pool, used_mem_high, ctypes.byref(value)) == 0
    return value.value


@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, 1])
def test_odd_rows_without_a_workspace_draw_no_memory(lib, fmt):
    """oco_matmul with n % 4 != 0 takes nothing from the stream-ordered pool
    (whole quads do), and its launch can be recorded and replayed."""
    from oco_amd import synth
    m, k = 40, 512
    say("odd rows draw no memory", fmt)
    x = lib.DeviceBuffer.from_array(synth.bf16_bits(synth.activations(36, m * k)))
    drawn = []
    for n in (1101, 1104):
        w, y = lib.DeviceBuffer.from_array(weights(fmt, n, k, 35)), lib.DeviceBuffer(m * n * 4)
        p = lib.Matrix(k, n, m, 0, 1, 1, 0)
        lib.synchronize()
        pool_high_water(reset=True)
        lib.matmul(fmt, w, x, y, p)
        lib.synchronize()
        drawn.append(pool_high_water())
        if n % 4:
            s, z = lib.Stream(), lib.DeviceBuffer(m * n * 4)
            g = lib.Graph(s, lambda: lib.matmul(fmt, w, x, z, p, stream=s))
            for _ in range(2):
                z.fill32(0)
                lib.synchronize()
                g.launch()
                s.sync()
                np.testing.assert_array_equal(z.download(np.uint32), y.download(np.uint32))
    assert drawn[0] == 0 and drawn[1] > 0


@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, P.Q4_0, 0, 1])
@pytest.mark.parametrize("m,n,k", [(33, 1101, 512), (140, 259, 1280), (520, 134, 256), (64, 130, 1184)])
def test_rows_that_are_not_whole_quads(lib, fmt, m, n, k):
    """n % 4 != 0 from 32 rows on: with the workspace the pass + GEMM or the
    panel kernel, without it the fused tiles as before; bias, both outputs."""
    from oco_amd import synth
    if fmt == P.Q4_K and k % 256:
        k = 1280
    say("odd rows", fmt, m, n, k)
    w = np.frombuffer(np.random.default_rng(n).normal(0, 0.05, n * k).astype(np.float32).tobytes(), np.uint8) if fmt == 0 \
        else weights(fmt, n, k, 15 + n)
    x = synth.bf16_bits(synth.activations(16, m * k)).reshape(m, k)
    bias = np.random.default_rng(m).normal(size=n).astype(np.float32)
    half, mag = O.matmul_reference(fmt, w, x, n, k, half_operands=True)
    want, size = half + O.bf16_round(bias), mag + np.abs(O.bf16_round(bias))
    for bf16 in (False, True):
        got = product(lib, fmt, w, x, m, n, k, y_bf16=bf16, bias=bias, workspace=True)
        assert np.all(np.abs(got - want) <= O.roundoff_bound(want, size, k, bf16))
    wb, xb, bb = (lib.DeviceBuffer.from_array(a) for a in (w, x, bias))
    y, ws = Guarded(lib, m * n * 4), lib.DeviceBuffer(64)
    lib.matmul(fmt, wb, xb, y.ptr, lib.Matrix(k, n, m, 0, 1, 1, 1), bias=bb, workspace=ws, workspace_bytes=0)
    lib.synchronize()
    assert np.all(np.abs(y.read(np.float32).reshape(m, n) - want) <= O.roundoff_bound(want, size, k, False))


@pytest.mark.parametrize("fmt,m,n,k,kernel", [(P.Q8_0, 500, 2047, 256, 3), (P.Q6_K, 500, 2047, 256, 3), (P.Q8_0, 200, 2047, 256, 4),
                                              (P.Q4_K, 500, 2047, 256, 4), (P.Q8_0, 300, 515, 480, 3), (P.Q8_0, 300, 515, 512, 4), (P.Q8_0, 300, 515, 992, 5),
                                              (P.Q8_0, 1000, 1030, 736, 3), (P.Q5_K, 300, 515, 512, 4), (P.Q6_K, 700, 4097, 1024, 5)])
def test_odd_rows_of_a_short_k(lib, fmt, m, n, k, kernel):
    """The fused tiles (3), the panel kernel (4) and the pass + GEMM (5) stand
    side by side at short K, and an override reaches the one it names."""
    from oco_amd import synth
    say("odd rows, short k", fmt, m, n, k)
    w = weights(fmt, n, k, 41)
    x = synth.bf16_bits(synth.activations(42, m * k)).reshape(m, k)
    half, mag = O.matmul_reference(fmt, w, x, n, k, half_operands=True)
    p = lib.Matrix(k, n, m, 0, 1, 1, 0)
    for values, want in (((), kernel), ((0,), 3), ((1,), 5)):
        with lib.overridden(lib.Knob.MATMUL_VENDOR, values):
            assert lib.matmul_route(fmt, p)[0] == want
            got = product(lib, fmt, w, x, m, n, k, workspace=True)
        assert np.all(np.abs(got - half) <= O.roundoff_bound(half, mag, k, False))
