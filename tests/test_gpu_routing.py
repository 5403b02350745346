"""Routing kernels at the edges of their tiles, against the oracle."""
import numpy as np
import pytest

import oracle as O
from _util import Guarded, rel_l2, say

pytestmark = pytest.mark.gpu


def dev(oco, a):
    return oco.DeviceBuffer.from_array(np.ascontiguousarray(a))


@pytest.mark.parametrize("experts,k", [(1, 1), (8, 8), (63, 8), (64, 8), (65, 8), (127, 5), (128, 8), (129, 8), (255, 7), (256, 8)])
def test_route_select_lane_groups(lib, experts, k):
    """Selections around the 64 experts that a lane group holds: random rows,
    rows of few distinct values (ties within and across the groups go to the
    lowest index), both zeros, and a row whose maximum sits in the last place."""
    say("route_select lane groups", experts, k)
    rng = np.random.default_rng(experts * 10 + k)
    logits = rng.normal(size=(21, experts)).astype(np.float32)
    logits[5:13] = rng.integers(-2, 2, (8, experts)).astype(np.float32)
    logits[13] = np.where(np.arange(experts) % 2 == 0, -0.0, 0.0)
    logits[14, -1] = 9.0
    ids_b, probs_b = Guarded(lib, 21 * k * 4), Guarded(lib, 21 * k * 4)
    lib.route_select(dev(lib, logits), 21, experts, k, ids_b.ptr, probs_b.ptr)
    lib.synchronize()
    want_ids, want_probs = O.select_experts(logits, k)
    np.testing.assert_array_equal(ids_b.read(np.uint32).reshape(21, k), want_ids)
    # probabilities are bf16: equal up to one bf16 step (exp is not bit-pinned)
    np.testing.assert_allclose(probs_b.read(np.float32).reshape(21, k), want_probs, rtol=2 ** -7, atol=0)


@pytest.mark.parametrize("fmt,tokens", [(12, 16), (12, 17), (12, 33), (39, 17)])
def test_forward_selection_around_one_token_per_wavefront(lib, fmt, tokens):
    """oco_experts_forward selects up to 16 tokens beside the route plan and
    more in a launch of their own: both equal oco_router then
    oco_experts_apply bit for bit."""
    from oco_amd import synth
    E, hidden, ffn, k = 128, 256, 256, 8
    say("forward selection", fmt, tokens)
    ws = [dev(lib, synth.weights(fmt, E * 256, 256, 40 + i)) for i in range(3)]
    bank = lib.ExpertBank(fmt, hidden, ffn, E, k, *ws, activation=1, up_bias_one=False)
    rng = np.random.default_rng(tokens)
    x = dev(lib, O.f32_to_bf16(rng.normal(size=(tokens, hidden)).astype(np.float32)))
    rw = dev(lib, (rng.normal(size=(E, hidden)) / 16).astype(np.float32))
    rb = dev(lib, (rng.normal(size=E) * 0.1).astype(np.float32))
    resid = O.f32_to_bf16(rng.normal(size=(tokens, hidden)).astype(np.float32))
    got = []
    for whole in (True, False):
        out, ids, probs = dev(lib, resid), lib.DeviceBuffer(tokens * k * 4), lib.DeviceBuffer(tokens * k * 4)
        if whole:
            bank.forward(rw, rb, x, lib.DType.BF16, tokens, out, ids, probs)
        else:
            lib.router(x, lib.DType.BF16, rw, rb, tokens, hidden, E, k, lib.DeviceBuffer(tokens * E * 4), ids, probs)
            bank.apply(x, lib.DType.BF16, ids, probs, tokens, out)
        lib.synchronize()
        got.append((out.download(np.uint16), ids.download(np.uint32), probs.download(np.uint32)))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("tokens,hidden,experts,dtype", [(64, 2048, 128, "bf16"), (257, 2880, 32, "f32"), (8192, 32, 1, "bf16"),
                                                         (33, 1056, 255, "f32"), (500, 4096, 17, "bf16"), (37, 992, 256, "bf16")])
def test_router_logits_of_a_prompt(lib, tokens, hidden, experts, dtype):
    """tokens x experts past 8192: the matrix-core tiles at whole and partial
    tiles of 16 x 16, with K steps that do and do not fill the eight
    wavefronts.  Products of bf16 values are exact in f32; a 32-term sum in
    f32 is within 32 u of the sum of magnitudes, and what follows is 64-bit
    up to the result's own rounding."""
    say("router prompt", tokens, hidden, experts, dtype)
    rng = np.random.default_rng(hidden + experts)
    x = rng.normal(size=(tokens, hidden)).astype(np.float32)
    w = (rng.normal(size=(experts, hidden)) / np.sqrt(hidden)).astype(np.float32)
    b = rng.normal(size=experts).astype(np.float32)
    k = min(8, experts)
    bits = O.f32_to_bf16(x)
    logits = Guarded(lib, tokens * experts * 4)
    ids, probs = lib.DeviceBuffer(tokens * k * 4), lib.DeviceBuffer(tokens * k * 4)
    lib.router(dev(lib, bits if dtype == "bf16" else x), lib.DType.BF16 if dtype == "bf16" else lib.DType.F32, dev(lib, w),
               dev(lib, b), tokens, hidden, experts, k, logits.ptr, ids, probs)
    lib.synchronize()
    got = logits.read(np.float32).reshape(tokens, experts)
    as64 = lambda bits: (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)  # noqa: E731
    xr, wr, br = as64(bits), as64(O.f32_to_bf16(w)), as64(O.f32_to_bf16(b))
    want, mag = xr @ wr.T + br, np.abs(xr) @ np.abs(wr).T + np.abs(br)
    assert np.all(np.abs(got - want) <= 34 * 2.0 ** -24 * mag)
    np.testing.assert_array_equal(ids.download(np.uint32).reshape(tokens, k), O.select_experts(got, k)[0])


@pytest.mark.parametrize("routes,experts,tile", [(1, 1, 16), (64, 256, 16), (1025, 3, 48), (4096, 128, 32), (5000, 200, 64),
                                                 (65536, 256, 16), (65537, 256, 16), (300, 257, 32), (70, 7, 1 << 31)])
def test_route_plan_spread_and_single_workgroup(lib, routes, experts, tile):
    """The plan by one workgroup per expert (up to 256 experts and 65536
    routes) and past both limits by one workgroup, some ids >= experts."""
    say("route_plan edges", routes, experts, tile)
    rng = np.random.default_rng(routes)
    ids = rng.integers(0, experts, routes).astype(np.uint32)
    ids[rng.random(routes) < 0.03] = experts + 5
    words = lib.route_plan_words(routes, experts)
    out = Guarded(lib, words * 4)
    lib.route_plan(dev(lib, ids), routes, experts, tile, 3, 4, out.ptr)
    lib.synchronize()
    got = out.read(np.uint32)
    grouped = 6 + 2 * ((routes + 15) // 16 + experts)
    rows = grouped + experts * (routes + 1)
    tiles, offset = [], 0
    for e in range(experts):
        mine = np.nonzero(ids == e)[0]
        base = grouped + e * (routes + 1)
        assert got[base] == mine.size and got[rows + e] == offset
        np.testing.assert_array_equal(got[base + 1:base + 1 + mine.size], mine)
        np.testing.assert_array_equal(got[rows + experts + mine], offset + np.arange(mine.size))
        tiles += [(e, b) for b in range(0, mine.size, tile)]
        offset += mine.size
    np.testing.assert_array_equal(got[:6], [3, len(tiles), 1, 4, len(tiles), 1])
    np.testing.assert_array_equal(got[6:6 + 2 * len(tiles)].reshape(-1, 2), np.array(tiles, np.uint32).reshape(-1, 2))


@pytest.mark.parametrize("fmt,E", [(12, 65), (12, 128), (12, 256), (39, 128), (8, 64)])
def test_forward_one_token_over_many_experts(lib, fmt, E):
    """One token selects inside the gate/up kernel whatever the number of
    experts: ids, probabilities and rows equal oco_router then
    oco_experts_apply bit for bit."""
    from oco_amd import synth
    hidden, ffn, k = 256, 256, 8
    say("forward one token", fmt, E)
    ws = [dev(lib, synth.weights(fmt, E * 256, 256, 60 + i)) for i in range(3)]
    bank = lib.ExpertBank(fmt, hidden, ffn, E, k, *ws, activation=1, up_bias_one=False)
    rng = np.random.default_rng(E)
    x = dev(lib, O.f32_to_bf16(rng.normal(size=(1, hidden)).astype(np.float32)))
    rw = dev(lib, (rng.normal(size=(E, hidden)) / 16).astype(np.float32))
    rb = dev(lib, np.where(np.arange(E) == E - 1, 9.0, 0.0).astype(np.float32))  # the last expert is chosen first
    resid = O.f32_to_bf16(rng.normal(size=(1, hidden)).astype(np.float32))
    got = []
    for whole in (True, False):
        out, ids, probs = dev(lib, resid), dev(lib, np.zeros(k, np.uint32)), lib.DeviceBuffer(k * 4)
        if whole:
            bank.forward(rw, rb, x, lib.DType.BF16, 1, out, ids, probs)
        else:
            lib.router(x, lib.DType.BF16, rw, rb, 1, hidden, E, k, lib.DeviceBuffer(E * 4), ids, probs)
            bank.apply(x, lib.DType.BF16, ids, probs, 1, out)
        lib.synchronize()
        got.append((out.download(np.uint16), ids.download(np.uint32), probs.download(np.uint32)))
    assert got[0][1][0] == E - 1
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("fmt,tokens,E,k", [(12, 2, 128, 8), (12, 24, 128, 8), (12, 25, 128, 8), (14, 3, 65, 8), (8, 7, 256, 4),
                                            (39, 3, 32, 4), (12, 31, 8, 2),
                                            (8, 31, 4, 4)])
def test_decode_batches_route_by_route_and_in_tiles(lib, fmt, tokens, E, k):
    """Up to 1.5 routes per expert every route is a tile of its own and each
    workgroup selects its token's experts; beyond, tiles of four routes.  Both
    against the oracle, and the selection against oco_router."""
    from oco_amd import synth
    hidden, ffn = (64, 32) if E == 4 else (512, 256)  # short rows leave no room for descriptors
    say("decode batches", fmt, tokens, E, k)
    host = [synth.weights(fmt, E * n, kk, 80 + i) for i, (n, kk) in enumerate([(ffn, hidden), (ffn, hidden), (hidden, ffn)])]
    bank = lib.ExpertBank(fmt, hidden, ffn, E, k, *[dev(lib, h) for h in host], activation=1, up_bias_one=False)
    rng = np.random.default_rng(tokens + E)
    xs = rng.normal(size=(tokens, hidden)).astype(np.float32)
    x, rw = dev(lib, xs), dev(lib, (rng.normal(size=(E, hidden)) / 22).astype(np.float32))
    resid = O.f32_to_bf16(rng.normal(size=(tokens, hidden)).astype(np.float32))
    out, ids, probs = dev(lib, resid), dev(lib, np.zeros(tokens * k, np.uint32)), lib.DeviceBuffer(tokens * k * 4)
    routed = Guarded(lib, tokens * k * hidden * 4)
    bank.forward(rw, None, x, lib.DType.F32, tokens, out, ids, probs, routed=routed.ptr)
    ids2, probs2 = lib.DeviceBuffer(tokens * k * 4), lib.DeviceBuffer(tokens * k * 4)
    lib.router(x, lib.DType.F32, rw, None, tokens, hidden, E, k, lib.DeviceBuffer(tokens * E * 4), ids2, probs2)
    lib.synchronize()
    got = ids.download(np.uint32).reshape(tokens, k)
    np.testing.assert_array_equal(got, ids2.download(np.uint32).reshape(tokens, k))
    np.testing.assert_array_equal(probs.download(np.uint32), probs2.download(np.uint32))
    ref = O.experts_reference(fmt, hidden, ffn, *host, xs, got, probs.download(np.float32).reshape(tokens, k), resid, activation=1, up_one=False)
    assert rel_l2(routed.read(np.float32).reshape(-1, hidden), ref["down"]) <= 1e-5


@pytest.mark.parametrize("tokens,E", [(2, 64), (20, 16)])
def test_apply_leaves_out_ids_past_the_bank(lib, tokens, E):
    """Routes whose id is past the bank have no rows, one route per tile or
    four; the others' rows are as without them."""
    from oco_amd import synth
    hidden, ffn, k = 256, 256, 4
    say("ids past the bank", tokens, E)
    bank = lib.ExpertBank(12, hidden, ffn, E, k, *[dev(lib, synth.weights(12, E * 256, 256, 90 + i)) for i in range(3)],
                          activation=1, up_bias_one=False)
    rng = np.random.default_rng(tokens)
    x = dev(lib, rng.normal(size=(tokens, hidden)).astype(np.float32))
    good = np.stack([rng.permutation(E)[:k] for _ in range(tokens)]).astype(np.uint32)
    bad = good.copy()
    bad[1, 2] = E + 1000000
    probs, rows = dev(lib, np.full((tokens, k), 0.25, np.float32)), []
    for ids in (good, bad):
        routed = Guarded(lib, tokens * k * hidden * 4)
        out = dev(lib, np.zeros((tokens, hidden), np.uint16))
        bank.apply(x, lib.DType.F32, dev(lib, ids), probs, tokens, out, routed=routed.ptr)
        lib.synchronize()
        rows.append(routed.read(np.uint32).reshape(tokens * k, hidden))
    keep = np.arange(tokens * k) != k + 2
    np.testing.assert_array_equal(rows[0][keep], rows[1][keep])
    assert np.all(rows[1][k + 2] == 0x7FC12345)  # untouched


@pytest.mark.parametrize("fmt,ffn,hidden", [(12, 1024, 48 * 16 + 256), (12, 256, 256), (8, 1024, 992), (8, 32, 32), (14, 768, 1280)])
def test_down_rows_two_at_a_time(lib, fmt, ffn, hidden):
    """The routed down pass takes two rows per half-wavefront up to 32 pieces
    a row: the longest such rows, the shortest, and row counts that are not
    whole groups of sixteen."""
    from oco_amd import synth
    E, k, tokens = 16, 2, 3
    say("down rows", fmt, ffn, hidden)
    host = [synth.weights(fmt, E * n, kk, 70 + i) for i, (n, kk) in enumerate([(ffn, hidden), (ffn, hidden), (hidden, ffn)])]
    bank = lib.ExpertBank(fmt, hidden, ffn, E, k, *[dev(lib, h) for h in host], activation=1, up_bias_one=False)
    rng = np.random.default_rng(ffn + hidden)
    xs = rng.normal(size=(tokens, hidden)).astype(np.float32)
    ids, probs = O.select_experts(rng.normal(size=(tokens, E)).astype(np.float32), k)
    resid = O.f32_to_bf16(rng.normal(size=(tokens, hidden)).astype(np.float32))
    routed = Guarded(lib, tokens * k * hidden * 4)
    bank.apply(dev(lib, xs), lib.DType.F32, dev(lib, ids), dev(lib, probs), tokens, dev(lib, resid), routed=routed.ptr)
    lib.synchronize()
    ref = O.experts_reference(fmt, hidden, ffn, *host, xs, ids, probs, resid, activation=1, up_one=False)
    assert rel_l2(routed.read(np.float32).reshape(-1, hidden), ref["down"]) <= 1e-5
