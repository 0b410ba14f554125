"""Batched Q4_K x Q8_1 matmul at the edges of its integer fold.  The sums over the eight sub-blocks of a super-block are whole numbers of
2^-24 that start from a double's bit pattern while every activation scale of the tile lies in [0, 4); of 2^-24, or of 2^(s - 24) where one
reaches 2^(7 + s), converted at the end, for larger and negative ones; in double for non-finite scales, and where one reaches 2^(7 + s)
and another is below 2^(s - 14).  All must return the bits of the host loop."""
import numpy as np
import pytest

from bunker_amd import runtime as rt
from bunker_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    rt.cu(0)


def _same(y, ref):
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(y[~nan].view(np.uint32), ref[~nan].view(np.uint32)), int((y[~nan] != ref[~nan]).sum())


def _run(orc, W, xq, N, K, B):
    dW, dxq, dy = rt.to_device(W), rt.to_device(xq), rt.cuAlloc(B * N * 4)
    try:
        rt.cuMemset(dy, 0xff, B * N * 4)
        rt.gemm_q4k_q8_1(dW, dxq, dy, N, K, B)
        y = rt.from_device(dy, (B, N), np.float32)
    finally:
        for p in (dW, dxq, dy):
            rt.cuFree(p)
    with np.errstate(all="ignore"):
        ref = np.stack([orc.gemv_q4k_q8_1(W, xq[b], N, K) for b in range(B)])
    _same(y, ref)


SHAPES = [(100, 768, 32), (33, 2048, 9), (70, 1024, 33), (200, 512, 77), (130, 2304, 130), (257, 256, 260)]


@pytest.mark.parametrize("N,K,B", SHAPES)
@pytest.mark.parametrize("form", ["edge", "edge128", "shifted", "gap", "wide", "mixed", "negative", "infinite"])
def test_scales_on_both_sides_of_the_integer_fold(orc, N, K, B, form):
    print(f"matmul scales {form} N={N} K={K} B={B}", flush=True)
    g = synth.rng(1200 + N + K + B + len(form))
    W = synth.q4k_random(g, N, K)
    xq = np.stack([orc.pack_q8_1(r) for r in g.standard_normal((B, K)).astype(np.float32)]).reshape(B, K // 32, 36)
    scales = xq[:, :, 32:34].view(np.float16)[..., 0]
    tops = {"edge": 3.998, "edge128": 127.9, "shifted": 255.8, "gap": 255.8}
    if form in tops:              # the largest scale of a form (0x43ff; 0x57ff: 31 bits; s = 1) with the smallest ones that it takes, or (gap) just below
        low = {"shifted": 2.0**-13, "gap": 2.0**-13 - 2.0**-24}.get(form, 2.0**-24)
        pick = g.integers(0, 4, scales.shape)
        scales[pick == 0], scales[pick == 1], scales[pick == 2] = np.float16(tops[form]), np.float16(2.0**-13), np.float16(low)
        scales[(pick == 3) & (g.random(scales.shape) < 0.2)] = 0
        if form == "shifted":
            scales[(scales > 0) & (scales < np.float16(2.0**-13))] = 0
        xq[:, :, :32] = g.choice(np.array([-128, 127], np.int8), xq[:, :, :32].shape).view(np.uint8)
    elif form == "wide":          # scales of 4 to 32768 in every super-block
        scales[:] = np.exp2(g.integers(2, 16, scales.shape)).astype(np.float16)
    elif form == "mixed":         # one sub-block of a few rows: only some tiles and super-blocks leave the integer form
        for _ in range(3):
            scales[g.integers(0, B), g.integers(0, K // 32)] = np.float16(4.0)
    elif form == "negative":
        scales[g.integers(0, B)] *= np.float16(-1.0)
    else:
        scales[g.integers(0, B), g.integers(0, K // 32)] = np.float16(np.inf)
        scales[g.integers(0, B), g.integers(0, K // 32)] = np.float16(np.nan)
    xq[:, :, 32:34] = scales[..., None].view(np.uint8)
    _run(orc, W, np.ascontiguousarray(xq.reshape(B, -1)), N, K, B)


@pytest.mark.parametrize("top", [3.998, 127.9, 65504.0, -65504.0])
def test_largest_sums_of_the_integer_fold(orc, top):
    """Every weight 15 with scale 63 and every activation of one sign at the largest scale: the sums reach 8 * 32 * 945 * 128 * 4, * 128 and * 65504."""
    N, K, B = 64, 1024, 96
    g = synth.rng(77)
    W = synth.q4k_random(g, N, K).reshape(-1, 144)
    W[:, 4:16] = synth.pack_q4k_scales(np.full((W.shape[0], 8), 63), np.full((W.shape[0], 8), 63))
    W[:, 16:] = 0xFF
    xq = np.zeros((B, K // 32, 36), np.uint8)
    xq[:, :, :32] = np.where(np.arange(B) % 2 == 0, 0x80, 0x7F)[:, None, None]
    xq[:, :, 32:34] = np.float16(top).view(np.uint16).reshape(1).view(np.uint8)
    xq[:, :, 34:36] = np.float16(-1.0).view(np.uint16).reshape(1).view(np.uint8)
    _run(orc, W, xq.reshape(B, -1), N, K, B)


def _big(g, N, K, B):
    W = synth.q4k_centered(g, N, K, 0.05)
    x = g.standard_normal((B, K)).astype(np.float32)
    dx, dxq = rt.to_device(x), rt.cuAlloc(B * (K // 32) * 36)
    rt.quantize_q8_1(dx, dxq, K, B, rt.F32)
    rt.cuFree(dx)
    return W, rt.to_device(W), dxq


@pytest.mark.parametrize("K,B", [(1024, B) for B in (33, 65, 129, 257, 385, 449, 513, 641, 833, 961, 1025, 1153, 1217, 1345)]
                         + [(2048, 33), (2048, 1153), (5120, 833)])
def test_every_split_of_a_tile_gives_the_same_bits(orc, K, B):
    """The number of waves that share a tile follows from the tiles per CU (one to twelve over these batches: 66 tiles of rows, 256 CUs) and,
    where two choices are close, from the length of a row; eight share one from K = 2048.  Whichever it is, the sums are the host
    loop's."""
    N = 2085
    assert {-(-66 * -(-b // 32) // 256) for b in (33, 65, 129, 257, 385, 449, 513, 641, 833, 961, 1025, 1153, 1217, 1345)} == set(range(1, 13))
    print(f"split N={N} K={K} B={B}", flush=True)
    W, dW, dxq = _big(synth.rng(90 + B), N, K, B)
    dy = rt.cuAlloc(B * N * 4)
    try:
        outs = []
        for nw in (0, 1, 2, 4, 8):
            rt.tune_set("gemm_nw", nw)
            rt.cuMemset(dy, 0xff, B * N * 4)
            rt.gemm_q4k_q8_1(dW, dxq, dy, N, K, B)
            outs.append(rt.from_device(dy, (B, N), np.uint32))
        xq = rt.from_device(dxq, (B, K // 32 * 36), np.uint8)
    finally:
        rt.tune_set("gemm_nw", 0)
        for p in (dW, dxq, dy):
            rt.cuFree(p)
    for o in outs[1:]:
        assert np.array_equal(o, outs[0])
    for b in (0, B // 2, B - 1):
        assert np.array_equal(outs[0][b], orc.gemv_q4k_q8_1(W, xq[b], N, K).view(np.uint32)), b


@pytest.mark.parametrize("N,K,B,offset", [(32, 256, 9, 0), (96, 512, 33, 2), (160, 1024, 70, 0), (64, 2048, 31, 8)])
def test_swiglu_blocks_of_every_split(orc, N, K, B, offset):
    """Gate, up, SwiGLU and the Q8_1 blocks of the result with one wave a tile (a thread holds eight values of a block) and with two and
    four (one value a lane), the bf16 result at addresses of every alignment: the host's bytes."""
    print(f"swiglu split N={N} K={K} B={B} offset={offset}", flush=True)
    g = synth.rng(300 + N + B)
    Wg, dWg, dxq = _big(g, N, K, B)
    Wu = synth.q4k_centered(g, N, K, 0.05)
    dWu, dact, dq = rt.to_device(Wu), rt.cuAlloc(B * N * 2 + 16), rt.cuAlloc(B * (N // 32) * 36)
    k = rt.compileAndLoad(f"gemv_fused K={K} pro=0 G=2 swiglu=1 N0={N} N1={N} batch={B} q8out=1")
    try:
        xq = rt.from_device(dxq, (B, K // 32 * 36), np.uint8)
        for nw in (0, 1, 2, 4):
            rt.tune_set("gemm_nw", nw)
            rt.cuMemset(dact, 0, B * N * 2 + 16)
            assert rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [dxq, dWg, dWu, dact + offset, dq]) == 0, rt.last_error()
            raw = rt.from_device(dact, (B * N * 2 + 16,), np.uint8)
            act = raw[offset : offset + B * N * 2].view(np.uint16).reshape(B, N)
            assert not raw[:offset].any() and not raw[offset + B * N * 2 :].any()
            gq = rt.from_device(dq, (B, (N // 32) * 36), np.uint8)
            for b in range(B):
                ref = orc.swiglu(orc.gemv_q4k_q8_1(Wg, xq[b], N, K), orc.gemv_q4k_q8_1(Wu, xq[b], N, K))
                assert np.array_equal(act[b], ref), (nw, b)
                assert np.array_equal(gq[b], orc.pack_q8_1((ref.astype(np.uint32) << 16).view(np.float32))), (nw, b)
    finally:
        rt.tune_set("gemm_nw", 0)
        rt.unloadKernel(k)
        for p in (dWg, dWu, dxq, dact, dq):
            rt.cuFree(p)
