"""Batched Q4_K x Q8_1 matmul in workgroups of 64 weight rows x 64 activation rows (gemm_tiles.hip): every output equals the host loop's
bits at the edges of tiles and pairs of tiles, for every epilogue, and in every range of activation scales."""
import numpy as np
import pytest

from bunker_amd import runtime as rt
from bunker_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def tiles():
    rt.cu(0)
    rt.tune_set("gemm_tiles", 1)
    yield
    rt.tune_set("gemm_tiles", -1)


def _same(y, ref):
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(y[~nan].view(np.uint32), ref[~nan].view(np.uint32)), int((y[~nan] != ref[~nan]).sum())


def _activations(orc, g, B, K):
    return np.stack([orc.pack_q8_1(r) for r in g.standard_normal((B, K)).astype(np.float32)]).reshape(B, K // 32, 36)


@pytest.mark.parametrize("form", ["plain", "large", "shifted", "gap", "mixed", "negative", "infinite"])
@pytest.mark.parametrize("N,K,B", [(1, 256, 8), (33, 768, 33), (64, 512, 64), (97, 256, 65), (31, 1280, 31), (130, 512, 130),
                                   (163, 2048, 131), (33, 4096, 70), (97, 6144, 65)])
def test_outputs_equal_the_host_loop(orc, N, K, B, form):
    print(f"matmul tiles {form} N={N} K={K} B={B}", flush=True)
    g = synth.rng(4200 + N + K + B)
    W, xq = synth.q4k_random(g, N, K), _activations(orc, g, B, K)
    scales = xq[:, :, 32:34].view(np.float16)[..., 0]
    tops = {"large": (127.9, 2.0**-24), "shifted": (255.8, 2.0**-13), "gap": (255.8, 2.0**-13 - 2.0**-24)}
    if form in tops:
        scales[:] = g.choice(np.array(tops[form], np.float16), scales.shape)
        scales[g.random(scales.shape) < 0.05] = 0
    elif form == "mixed":
        scales[g.integers(0, B), g.integers(0, K // 32)] = np.float16(4.0)
    elif form == "negative":
        scales[g.integers(0, B)] *= np.float16(-1.0)
    elif form == "infinite":
        scales[g.integers(0, B), g.integers(0, K // 32)] = np.float16(np.inf)
    xq[:, :, 32:34] = scales[..., None].view(np.uint8)
    xq = np.ascontiguousarray(xq.reshape(B, -1))
    # activations at an address that is only a multiple of 4; nothing is written past the outputs
    raw = np.concatenate([np.zeros(4, np.uint8), xq.ravel()])
    dW, dxq, dy = rt.to_device(W), rt.to_device(raw), rt.cuAlloc(B * N * 4 + 64)
    try:
        rt.cuMemset(dy, 0xff, B * N * 4 + 64)
        rt.gemm_q4k_q8_1(dW, dxq + 4, dy, N, K, B)
        y = rt.from_device(dy, (B * N + 16,), np.float32)
    finally:
        for p in (dW, dxq, dy):
            rt.cuFree(p)
    with np.errstate(all="ignore"):
        ref = np.stack([orc.gemv_q4k_q8_1(W, xq[b], N, K) for b in range(B)])
    _same(y[: B * N].reshape(B, N), ref)
    assert (y[B * N :].view(np.uint32) == 0xFFFFFFFF).all()


@pytest.mark.parametrize("B", [33, 96, 100])
def test_four_matrices_in_one_launch_with_every_epilogue(orc, B):
    """Tiles of different matrices in one workgroup, bf16 outputs and the residual add: the bits of the launch for the same group with lone waves."""
    K, Ns = 512, [40, 16, 96, 33]
    print(f"matmul tiles group B={B}", flush=True)
    g = synth.rng(77 + B)
    Ws = [rt.to_device(synth.q4k_centered(g, n, K, 0.05)) for n in Ns]
    x = rt.to_device(g.standard_normal((B, K)).astype(np.float32))
    dxq = rt.cuAlloc(B * (K // 32) * 36)
    rt.quantize_q8_1(x, dxq, K, B, rt.F32)
    res = [rt.to_device((g.standard_normal((B, n)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)) for n in Ns]
    outs = [rt.cuAlloc(B * n * 4) for n in Ns]
    got = []
    try:
        for epis in ([0, 1, 1, 0], [1, 0, 0, 1]):
            spec = f"gemv_fused K={K} pro=0 G=4 batch={B} " + " ".join(f"N{i}={n} epi{i}={e}" for i, (n, e) in enumerate(zip(Ns, epis)))
            k = rt.compileAndLoad(spec)
            for tiles in (1, 0):
                rt.tune_set("gemm_tiles", tiles)
                for o, n in zip(outs, Ns):
                    rt.cuMemset(o, 0, B * n * 4)
                assert rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [dxq] + [p for pair in zip(Ws, outs) for p in pair]) == 0, rt.last_error()
                got.append([rt.from_device(o, (B, n * 2), np.uint16) for o, n in zip(outs, Ns)])
            rt.unloadKernel(k)
        for tiles in (1, 0):
            rt.tune_set("gemm_tiles", tiles)
            row = []
            for W, r, o, n in zip(Ws, res, outs, Ns):
                rt.cuMemset(o, 0, B * n * 4)
                rt.gemm_q4k_q8_1(W, dxq, o, n, K, B, out_dtype=rt.BF16, residual=r)
                row.append(rt.from_device(o, (B, n * 2), np.uint16))
            got.append(row)
    finally:
        for p in (*Ws, x, dxq, *res, *outs):
            rt.cuFree(p)
    for a, b in zip(got[::2], got[1::2]):
        for u, v in zip(a, b):
            assert v.any() and np.array_equal(u, v)


@pytest.mark.parametrize("N,K,B,offset", [(32, 256, 9, 0), (96, 512, 33, 2), (160, 1024, 70, 0), (64, 768, 64, 8), (32, 512, 129, 0), (160, 2048, 131, 0), (64, 6144, 33, 2)])
def test_swiglu_blocks(orc, N, K, B, offset):
    print(f"swiglu tiles N={N} K={K} B={B} offset={offset}", flush=True)
    g = synth.rng(500 + N + B)
    Wg, Wu = synth.q4k_centered(g, N, K, 0.05), synth.q4k_centered(g, N, K, 0.05)
    xq = np.ascontiguousarray(_activations(orc, g, B, K).reshape(B, -1))
    dWg, dWu, dxq, dact, dq = rt.to_device(Wg), rt.to_device(Wu), rt.to_device(xq), rt.cuAlloc(B * N * 2 + 16), rt.cuAlloc(B * (N // 32) * 36)
    k = rt.compileAndLoad(f"gemv_fused K={K} pro=0 G=2 swiglu=1 N0={N} N1={N} batch={B} q8out=1")
    try:
        rt.cuMemset(dact, 0, B * N * 2 + 16)
        assert rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [dxq, dWg, dWu, dact + offset, dq]) == 0, rt.last_error()
        raw, gq = rt.from_device(dact, (B * N * 2 + 16,), np.uint8), rt.from_device(dq, (B, (N // 32) * 36), np.uint8)
    finally:
        rt.unloadKernel(k)
        for p in (dWg, dWu, dxq, dact, dq):
            rt.cuFree(p)
    act = raw[offset : offset + B * N * 2].view(np.uint16).reshape(B, N)
    assert not raw[:offset].any() and not raw[offset + B * N * 2 :].any()
    for b in range(B):
        ref = orc.swiglu(orc.gemv_q4k_q8_1(Wg, xq[b], N, K), orc.gemv_q4k_q8_1(Wu, xq[b], N, K))
        assert np.array_equal(act[b], ref), b
        assert np.array_equal(gq[b], orc.pack_q8_1((ref.astype(np.uint32) << 16).view(np.float32))), b


@pytest.mark.parametrize("N,K,B", [(3072, 512, 1024), (8240, 256, 1000), (4063, 6144, 1000), (6113, 2048, 1023)])
def test_large_launches_choose_it_and_return_the_same_bits(orc, N, K, B):
    print(f"matmul tiles by shape N={N} K={K} B={B}", flush=True)
    g = synth.rng(N + B)
    W = synth.q4k_centered(g, N, K, 0.05)
    x = g.standard_normal((B, K)).astype(np.float32)
    dW, dx, dxq, dy = rt.to_device(W), rt.to_device(x), rt.cuAlloc(B * (K // 32) * 36), rt.cuAlloc(B * N * 4)
    try:
        rt.quantize_q8_1(dx, dxq, K, B, rt.F32)
        outs = []
        for tiles in (-1, 0, 1):
            rt.tune_set("gemm_tiles", tiles)
            rt.cuMemset(dy, 0xff, B * N * 4)
            rt.gemm_q4k_q8_1(dW, dxq, dy, N, K, B)
            outs.append(rt.from_device(dy, (B, N), np.uint32))
        xq = rt.from_device(dxq, (B, K // 32 * 36), np.uint8)
    finally:
        for p in (dW, dx, dxq, dy):
            rt.cuFree(p)
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    for b in (0, B // 2, B - 1):
        assert np.array_equal(outs[0][b], orc.gemv_q4k_q8_1(W, xq[b], N, K).view(np.uint32)), b
