"""The product of a few activation rows at the edges of its tiles, against
the oracle's half-operand product within the reference's roundoff bound
(matrix_precision.rs:119-142)."""
import numpy as np
import pytest

import oracle as O
import packers as P
from _util import Guarded, say, upload_at_offset

pytestmark = pytest.mark.gpu

F16 = 1


def weights(fmt, n, k, seed):
    if fmt == F16:
        return np.frombuffer(np.random.default_rng(seed).normal(0, 0.05, n * k).astype(np.float16).tobytes(), np.uint8)
    from oco_amd import synth
    return synth.weights(fmt, n, k, seed=seed)


def product(lib, fmt, w, x, m, n, k, x_f16=False, y_bf16=False, bias=None, offset=0, workspace=False):
    keep, wp = upload_at_offset(lib, w, offset)
    xb, bb = lib.DeviceBuffer.from_array(x), None if bias is None else lib.DeviceBuffer.from_array(bias)
    y = Guarded(lib, m * n * (2 if y_bf16 else 4))
    p, xt = lib.Matrix(k, n, m, 0, 1, 1, 0 if bias is None else 1), lib.DType.F16 if x_f16 else lib.DType.BF16
    need = lib.matmul_workspace(fmt, p, xt) if workspace else 0
    ws = lib.DeviceBuffer(need) if need else None
    lib.matmul(fmt, wp, xb, y.ptr, p, xt, lib.DType.BF16 if y_bf16 else lib.DType.F32, bb, workspace=ws, workspace_bytes=need)
    lib.synchronize()
    got = y.read(np.uint16 if y_bf16 else np.float32)
    return (O.bf16_to_f32(got) if y_bf16 else got).reshape(m, n)


# K units of 256: one, a partial one, nine (past one round of the eight
# wavefronts), seventeen and 33 (second and third refill of a wavefront's pair).
@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, P.Q5_K, P.Q6_K, P.Q4_0, P.Q4_1, F16])
@pytest.mark.parametrize("m,n,units", [(5, 1, 1), (16, 15, 9), (17, 17, 17), (31, 33, 33), (9, 6200, 1), (12, 10270, 1)])
def test_few_rows(lib, fmt, m, n, units):
    from oco_amd import synth
    say("few rows", fmt, m, n, units)
    for k in [256 * units] + ([] if fmt in (P.Q4_K, P.Q5_K, P.Q6_K) else [256 * units - 32, 256 * units - 224]):
        w = weights(fmt, n, k, 7 + n)
        x = synth.bf16_bits(synth.activations(8, m * k)).reshape(m, k)
        half, mag = O.matmul_reference(fmt, w, x, n, k, half_operands=True)
        if fmt in (P.Q4_0, P.Q4_1) and n > 1024:  # scaled rows: half(x gain) / gain, the same values but for subnormals
            mag = mag + 2.0 ** -12 * np.abs(half).max()
        got = product(lib, fmt, w, x, m, n, k, offset=7)
        assert np.all(np.abs(got - half) <= O.roundoff_bound(half, mag, k, False)), (k, np.abs(got - half).max())


@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, P.Q5_K, P.Q6_K, P.Q4_0, P.Q4_1, F16])
@pytest.mark.parametrize("m", [1, 3, 18])
def test_few_rows_f16_input_bias_bf16_output(lib, fmt, m):
    from oco_amd import synth
    n, k = 70, 768
    say("few rows f16", fmt, m)
    w = weights(fmt, n, k, 17)
    x = synth.activations(18, m * k).reshape(m, k).astype(np.float16)
    bias = np.random.default_rng(m).normal(size=n).astype(np.float32)
    got = product(lib, fmt, w, x, m, n, k, x_f16=True, y_bf16=True, bias=bias)
    half, mag = O.matmul_reference(fmt, w, x, n, k, half_operands=True)
    want = half + O.bf16_round(bias)
    assert np.all(np.abs(got - want) <= O.roundoff_bound(want, mag + np.abs(O.bf16_round(bias)), k, True))


@pytest.mark.parametrize("fmt", [P.Q8_0, P.Q4_K, P.Q6_K])
def test_few_rows_nonfinite_and_rows_apart(lib, fmt):
    """A NaN or infinite activation reaches its own row only; rows are
    independent of their number."""
    from oco_amd import synth
    m, n, k = 11, 40, 512
    say("few rows non-finite", fmt)
    w = weights(fmt, n, k, 27)
    x = synth.bf16_bits(synth.activations(28, m * k)).reshape(m, k)
    plain = product(lib, fmt, w, x, m, n, k)
    x2 = x.copy()
    x2[3, 300], x2[7, 511] = 0x7FC0, 0x7F80
    got = product(lib, fmt, w, x2, m, n, k)
    assert np.isnan(got[3]).all() and not np.isfinite(got[7]).any()
    keep = [r for r in range(m) if r not in (3, 7)]
    np.testing.assert_array_equal(got[keep], plain[keep])
    np.testing.assert_array_equal(product(lib, fmt, w, x[:5], 5, n, k), plain[:5])


@pytest.mark.parametrize("fmt,mid,top", [(P.Q4_0, 8, 15), (P.Q6_K, 32, 63), (P.Q8_0, 0, 127)])
@pytest.mark.parametrize("m,n,k", [(11, 40, 512), (65, 20004, 256)])  # the few-row kernel; the prompt-chunk GEMM
def test_infinite_block_scales(lib, fmt, mid, top, m, n, k):
    """A block's weights are scale * (code - middle): with an infinite scale
    +-Inf, NaN at the middle code only, whichever kernel decodes it."""
    from oco_amd import synth
    say("infinite block scales", fmt, m, n, k)
    unit, size = (256, 210) if fmt == P.Q6_K else (32, 34 if fmt == P.Q8_0 else 18)
    w = weights(fmt, n, k, 37).reshape(n, k // unit * size).copy()

    def block(scale_bits, code, first=None):
        """One block of equal codes, the first of them `first`."""
        c = np.full(unit, code, np.int64)
        c[0] = code if first is None else first
        d = np.array([scale_bits], np.uint16).view(np.uint8)
        if fmt == P.Q8_0:
            return np.r_[d, c.astype(np.int8).view(np.uint8)]
        if fmt == P.Q4_0:
            return np.r_[d, (c[:16] | (c[16:] << 4)).astype(np.uint8)]
        q = c.reshape(2, 4, 32)
        ql = np.concatenate([q[:, :2] & 15 | (q[:, 2:] & 15) << 4], 1).reshape(-1)
        hi = q >> 4
        qh = (hi[:, 0] | hi[:, 1] << 2 | hi[:, 2] << 4 | hi[:, 3] << 6).reshape(-1)
        return np.r_[ql.astype(np.uint8), qh.astype(np.uint8), np.full(16, 3, np.uint8), d]

    inf, ninf, nan = 0x7C00, 0xFC00, 0x7E00
    w[0, :size], w[1, :size], w[2, :size] = block(inf, top), block(inf, mid - 1), block(inf, top, mid)
    w[3, :size], w[4, :size], w[5, :size] = block(ninf, mid + 1), block(nan, top), block(inf, mid - 3)
    x = synth.bf16_bits(np.abs(synth.activations(38, m * k)) + 0.5).reshape(m, k)
    got = product(lib, fmt, w.reshape(-1), x, m, n, k)
    want = np.array([np.inf, -np.inf, np.nan, -np.inf, np.nan, -np.inf], np.float32)
    np.testing.assert_array_equal(got[:, :6], np.broadcast_to(want, (m, 6)))
    assert np.isfinite(got[:, 6:]).all()
