"""GPU parity, through the C ABI, of the Q8_1 quantizer, the nibble dequant kernels and the
Q4_K GEMVs against the CPU oracle on the same seeded inputs.

Bars: integer / byte outputs bit-exact; f32 outputs |gpu - ref| <= 1e-4 * max(|ref|, rms(ref))."""
import numpy as np
import pytest

from bunker_amd import runtime as rt
from bunker_amd import synth

pytestmark = pytest.mark.gpu

REL = 1e-4


def _assert_rel(got, ref, rel=REL):
    ref = ref.astype(np.float64); got = got.astype(np.float64)
    lim = rel * np.maximum(np.abs(ref), np.sqrt(np.mean(ref * ref)))
    bad = np.abs(got - ref) > lim
    assert not bad.any(), f"{bad.sum()} of {bad.size} outside tolerance, worst {np.abs(got - ref).max():.3e}"


class Dev:
    """Uploads arrays and frees them at the end of a test."""

    def __init__(self):
        self.ptrs = []

    def up(self, a):
        p = rt.to_device(a); self.ptrs.append(p); return p

    def empty(self, nbytes):
        p = rt.cuAlloc(nbytes); self.ptrs.append(p); return p

    def close(self):
        for p in self.ptrs:
            rt.cuFree(p)


@pytest.fixture()
def dev():
    d = Dev()
    yield d
    d.close()


# ------------------------------------------------------------------ quantizer
@pytest.mark.parametrize("K,batch", [(2048, 1), (6144, 1), (2048, 8), (256, 3), (40, 2)])
def test_quantize_q8_1_bit_exact(orc, dev, K, batch):
    print(f"quantize K={K} batch={batch}", flush=True)
    g = synth.rng(100 + K + batch)
    x = g.standard_normal((batch, K)).astype(np.float32)
    x[0, :32] = 0.0
    if K >= 64:
        x[0, 32] = 127.0
        x[0, 33:41] = [0.5, -0.5, 1.5, -1.5, 2.5, -2.5, 0.49999997, -0.50000006]
        x[0, 41:64] = 0
    nb = (K + 31) // 32
    out = dev.empty(batch * nb * 36)
    rt.quantize_q8_1(dev.up(x), out, K, batch, rt.F32)
    got = rt.from_device(out, (batch, nb * 36), np.uint8)
    ref = np.stack([orc.pack_q8_1(r) for r in x])
    assert np.array_equal(got, ref)
    # bf16 activations are widened first
    xb = synth.f32_to_bf16(x)
    rt.quantize_q8_1(dev.up(xb), out, K, batch, rt.BF16)
    got = rt.from_device(out, (batch, nb * 36), np.uint8)
    ref = np.stack([orc.pack_q8_1(r) for r in synth.bf16_to_f32(xb)])
    assert np.array_equal(got, ref)


def test_quantize_q8_1_scale_sweep(orc, dev):
    """Magnitudes from 1e-6 to 1e4 and exact .5 quotients: rounding and fp16 truncation paths."""
    g = synth.rng(7)
    K = 32 * 512
    x = (g.standard_normal(K) * 10.0 ** g.uniform(-6, 4, K // 32).repeat(32)).astype(np.float32)
    half = (g.integers(-254, 254, K // 2) * 0.5).astype(np.float32)       # amax 127 -> d = 1
    half[::32] = 127.0
    x[: K // 2] = half
    out = dev.empty(K // 32 * 36)
    rt.quantize_q8_1(dev.up(x), out, K, 1, rt.F32)
    assert np.array_equal(rt.from_device(out, (K // 32 * 36,), np.uint8), orc.pack_q8_1(x))


# ------------------------------------------------------------------ dequant
def test_dequant_legacy_known_answer(orc, dev):
    g = synth.rng(8)
    nb = 128 * 32                                            # tests/test_dequant.ts:3-7 sizes
    lo = g.integers(0, 16, (nb, 16)); hi = g.integers(0, 16, (nb, 16))
    blocks = np.zeros((nb, 20), np.uint8)
    blocks[:, :16] = lo | (hi << 4)
    blocks[:, 16:] = g.integers(0, 256, (nb, 4))
    ref = np.empty((nb, 32), np.int8); ref[:, 0::2] = lo - 8; ref[:, 1::2] = hi - 8
    out = dev.empty(nb * 32)
    rt.dequant_legacy_i8(dev.up(blocks), out, nb)
    got = rt.from_device(out, (nb, 32), np.int8)
    assert np.array_equal(got, ref)
    assert np.array_equal(got.ravel(), orc.legacy_dequant_i8(blocks))


def test_q4k_unpack_bit_exact(orc, dev):
    g = synth.rng(9)
    N, K = 96, 2048
    W = synth.q4k_random(g, N, K)
    nblk = N * K // 256
    dW = dev.up(W)
    o1 = dev.empty(nblk * 256)
    rt.q4k_nibbles(dW, o1, nblk)
    assert np.array_equal(rt.from_device(o1, (nblk * 256,), np.uint8), orc.q4k_nibbles(W))
    o2 = dev.empty(nblk * 256 * 4)
    rt.q4k_dequant_f32(dW, o2, nblk)
    assert np.array_equal(rt.from_device(o2, (nblk * 256,), np.float32).view(np.uint32),
                          orc.q4k_dequant(W).view(np.uint32))


# ------------------------------------------------------------------ GEMV
DECODE_SHAPES = {"qkv": (6144, 2048), "gate_up": (12288, 2048), "down": (2048, 6144), "lm_head": (151936, 2048)}


@pytest.mark.parametrize("name", list(DECODE_SHAPES))
def test_gemv_q4k_q8_1_decode_shapes(orc, dev, name):
    N, K = DECODE_SHAPES[name]
    print(f"gemv {name} N={N} K={K}", flush=True)
    g = synth.rng(200 + N % 97)
    W = synth.q4k_random(g, N, K)
    x = g.standard_normal(K).astype(np.float32)
    dW, dx = dev.up(W), dev.up(x)
    dxq = dev.empty(K // 32 * 36)
    rt.quantize_q8_1(dx, dxq, K, 1, rt.F32)
    xq = rt.from_device(dxq, (K // 32 * 36,), np.uint8)
    assert np.array_equal(xq, orc.pack_q8_1(x))
    # exact integer sub-block dots
    dI = dev.empty(N * (K // 32) * 4)
    rt.q4k_q8_1_subdots(dW, dxq, dI, N, K)
    I = rt.from_device(dI, (N, K // 32), np.int32)
    assert np.array_equal(I, orc.q4k_q8_1_subdots(W, xq, N, K))
    # f32 output
    dy = dev.empty(N * 4)
    rt.gemv_q4k_q8_1(dW, dxq, dy, N, K)
    y = rt.from_device(dy, (N,), np.float32)
    ref = orc.gemv_q4k_q8_1(W, xq, N, K, acc64=True)
    _assert_rel(y, ref)
    # every term after the integer dots is exact in double, so the f32 result equals the host's to the bit
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), int((y != ref).sum())
    # run-to-run determinism (fixed reduction order, no atomics)
    rt.gemv_q4k_q8_1(dW, dxq, dy, N, K)
    assert np.array_equal(rt.from_device(dy, (N,), np.float32).view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("N,K", [(1001, 2048), (515, 4096), (258, 6144)])
def test_gemv_variants_return_the_same_bits(orc, dev, N, K):
    """Every kernel variant behind bk_gemv_q4k_q8_1 (rows through LDS; direct loads with 1, 2 or 4 rows per wave step;
    few or many workgroups per CU) returns the checker's bits: the arithmetic does not depend on the launch shape."""
    print(f"gemv variants N={N} K={K}", flush=True)
    g = synth.rng(350 + N)
    W = synth.q4k_random(g, N, K)
    xq = orc.pack_q8_1(g.standard_normal(K).astype(np.float32))
    ref = orc.gemv_q4k_q8_1(W, xq, N, K)
    dW, dxq, dy = dev.up(W), dev.up(xq), dev.empty(N * 4)
    try:
        for impl, rpi, cap in [(2, 0, 16), (2, 4, 16), (2, 2, 1), (0, 1, 16), (0, 2, 2), (0, 4, 1), (0, 4, 64)]:
            rt.tune_set("gemv_impl", impl); rt.tune_set("gemv_rpi", rpi); rt.tune_set("gemv_cap", cap)
            rt.cuMemset(dy, 0xCD, N * 4)
            rt.gemv_q4k_q8_1(dW, dxq, dy, N, K)
            y = rt.from_device(dy, (N,), np.float32)
            assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), (impl, rpi, cap, int((y != ref).sum()))
    finally:
        rt.tune_set("gemv_impl", 2); rt.tune_set("gemv_rpi", 0); rt.tune_set("gemv_cap", 16)


@pytest.mark.parametrize("N,K", [(64, 256), (33, 768), (100, 1792), (128, 4096), (77, 8192), (5, 2048)])
def test_gemv_q4k_q8_1_ragged_shapes(orc, dev, N, K):
    print(f"gemv ragged N={N} K={K}", flush=True)
    g = synth.rng(300 + N + K)
    W = synth.q4k_random(g, N, K)
    xq = orc.pack_q8_1(g.standard_normal(K).astype(np.float32))
    dW, dxq = dev.up(W), dev.up(xq)
    dy = dev.empty(N * 4)
    rt.gemv_q4k_q8_1(dW, dxq, dy, N, K)
    y = rt.from_device(dy, (N,), np.float32); ref = orc.gemv_q4k_q8_1(W, xq, N, K)
    _assert_rel(y, ref)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    dI = dev.empty(N * (K // 32) * 4)
    rt.q4k_q8_1_subdots(dW, dxq, dI, N, K)
    assert np.array_equal(rt.from_device(dI, (N, K // 32), np.int32), orc.q4k_q8_1_subdots(W, xq, N, K))


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 6, 9, 10, 11, 12, 13, 14, 15, 17, 18, 20, 21, 23])
def test_gemv_q4k_q8_1_rows_numbered_through(orc, dev, nb):
    """Rows that do not fill whole rounds of 64 slots, in the form that numbers the super-blocks of several rows through: every class of row length at both
    ends, fewer rows than a step has, one and several steps a wave, each epilogue, two batch rows, and a row with an infinite scale,
    which its neighbours in the same rounds do not see.  The bits of the host loop: a sum of exactly known terms in double, in whatever order, rounded once."""
    K = 256 * nb
    g = synth.rng(60 + nb)
    try:
        rt.tune_set("gemv_impl", 3)
        for N, steps in ((1, 0), (3, 0), (50, 0), (301, 3), (170, 8)):
            print(f"gemv flat nb={nb} N={N} steps={steps}", flush=True)
            rt.tune_set("gemv_steps", steps)
            W = synth.q4k_random(g, N, K)
            bad = N // 2
            if N > 1:
                W.reshape(N, nb, 144)[bad, (nb - 1) // 2, 0:2] = np.array([0x7C00], np.uint16).view(np.uint8)
            xq = np.stack([orc.pack_q8_1(g.standard_normal(K).astype(np.float32)) for _ in range(2)])
            res = synth.f32_to_bf16(g.standard_normal((2, N)).astype(np.float32))
            keep = np.arange(N) != bad if N > 1 else np.ones(N, bool)
            ref = np.ascontiguousarray(np.stack([orc.gemv_q4k_q8_1(W, xq[i], N, K) for i in range(2)])[:, keep])
            dW, dx, dr = dev.up(W), dev.up(xq), dev.up(res)
            dy = dev.empty(2 * N * 4 + 64)
            rt.cuMemset(dy, 0xCD, 2 * N * 4 + 64)
            rt.gemv_q4k_q8_1(dW, dx, dy, N, K, batch=2)
            raw = rt.from_device(dy, (2 * N + 16,), np.float32)
            got = raw[:2 * N].reshape(2, N)
            assert (raw[2 * N:].view(np.uint32) == 0xCDCDCDCD).all()
            assert np.isfinite(got[:, keep]).all() and (N == 1 or not np.isfinite(got[:, bad]).any())
            assert np.array_equal(np.ascontiguousarray(got[:, keep]).view(np.uint32), ref.view(np.uint32)), int((got[:, keep] != ref).sum())
            for r in (0, dr):
                db = dev.empty(2 * N * 2)
                rt.gemv_q4k_q8_1(dW, dx, db, N, K, batch=2, out_dtype=rt.BF16, residual=r)
                want = synth.f32_to_bf16(got)
                if r:
                    want = synth.f32_to_bf16(synth.bf16_to_f32(want) + synth.bf16_to_f32(res))
                assert np.array_equal(rt.from_device(db, (2, N), np.uint16)[:, keep], want[:, keep])
    finally:
        rt.tune_set("gemv_impl", 2)
        rt.tune_set("gemv_steps", 0)


def test_gemv_q4k_q8_1_epilogues_and_batch(orc, dev):
    g = synth.rng(11)
    N, K, B = 2048, 2048, 3
    W = synth.q4k_random(g, N, K)
    x = g.standard_normal((B, K)).astype(np.float32)
    xq = np.stack([orc.pack_q8_1(r) for r in x])
    res = synth.f32_to_bf16(g.standard_normal((B, N)).astype(np.float32))
    dW, dxq, dres = dev.up(W), dev.up(xq), dev.up(res)
    ref = np.stack([orc.gemv_q4k_q8_1(W, xq[b], N, K) for b in range(B)])
    dy = dev.empty(B * N * 4)
    rt.gemv_q4k_q8_1(dW, dxq, dy, N, K, batch=B)
    y = rt.from_device(dy, (B, N), np.float32)
    _assert_rel(y, ref)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    # bf16 output: exactly the RNE rounding of the kernel's own f32 result
    rt.gemv_q4k_q8_1(dW, dxq, dy, N, K, batch=B, out_dtype=rt.BF16)
    yb = rt.from_device(dy, (B, N), np.uint16)
    assert np.array_equal(yb, synth.f32_to_bf16(y))
    # cast then add: bf16(f32(bf16(acc)) + f32(res))  (src/model.ts:110-117 order)
    rt.gemv_q4k_q8_1(dW, dxq, dy, N, K, batch=B, out_dtype=rt.BF16, residual=dres)
    ya = rt.from_device(dy, (B, N), np.uint16)
    assert np.array_equal(ya, orc.add_bf16(yb.ravel(), res.ravel()).reshape(B, N))


def test_gemv_q4k_f32_config1(orc, dev):
    """W 4096x4096, d,dmin = |N(0,0.01)|, scales/mins 0..63, nibbles 0..15, x ~ N(0,1)."""
    g = synth.rng(12)
    N = K = 4096
    W = synth.q4k_random(g, N, K)
    x = g.standard_normal(K).astype(np.float32)
    dy = dev.empty(N * 4)
    rt.gemv_q4k_f32(dev.up(W), dev.up(x), dy, N, K)
    _assert_rel(rt.from_device(dy, (N,), np.float32), orc.gemv_q4k_f32(W, x, N, K, acc64=True))


@pytest.mark.parametrize("N,K", [(1, 256), (2049, 2048), (4097, 1280), (515, 3584), (8195, 4096), (3, 6144), (70, 6400)])
def test_gemv_q4k_f32_staged_rows(orc, dev, N, K):
    """Edges of the staged form: a lone row, one row past a wave step and past the one-row rule, rows that do not fill their
    rounds, several steps per wave, and the longer rows that run the generic form; nothing past y is written."""
    g = synth.rng(1300 + N + K)
    W = synth.q4k_random(g, N, K)
    x = g.standard_normal(K).astype(np.float32)
    dy = dev.up(np.full(N + 64, 7.5, np.float32))
    rt.gemv_q4k_f32(dev.up(W), dev.up(x), dy, N, K)
    y = rt.from_device(dy, (N + 64,), np.float32)
    _assert_rel(y[:N], orc.gemv_q4k_f32(W, x, N, K, acc64=True))
    assert np.all(y[N:] == 7.5)


@pytest.mark.parametrize("K,block", [(1280, 0), (1280, 4), (2304, 0), (2304, 8), (5376, 20), (6400, 0), (6400, 24)])
def test_gemv_q4k_f32_infinite_scale(orc, dev, K, block):
    """Lanes past the end of a row stand on a block of the row and must add nothing, also where its scale is infinite: the row's
    result is the infinity that its own elements give (nibbles, scales and activations of that block positive, min 0)."""
    g = synth.rng(1400 + K + block)
    N = 5
    W = synth.q4k_random(g, N, K)
    blk = W.reshape(N, K // 256, 144)[2, block]
    blk[0:4] = np.array([np.inf, 0.0], np.float16).view(np.uint8)
    blk[4:16] = 0x11
    blk[16:] = 0x73
    x = np.abs(g.standard_normal(K)).astype(np.float32) + 0.1
    dy = dev.empty(N * 4)
    rt.gemv_q4k_f32(dev.up(W), dev.up(x), dy, N, K)
    y, ref = rt.from_device(dy, (N,), np.float32), orc.gemv_q4k_f32(W, x, N, K, acc64=True)
    assert ref[2] == np.inf and y[2] == np.inf, (y[2], ref[2])
    rest = np.arange(N) != 2
    _assert_rel(y[rest], ref[rest])


@pytest.mark.parametrize("N,K", [(64, 2048), (50, 1024), (9, 6144)])
def test_gemv_q4k_f32_other_shapes(orc, dev, N, K):
    g = synth.rng(13 + K)
    W = synth.q4k_random(g, N, K)
    x = g.standard_normal(K).astype(np.float32)
    dy = dev.empty(N * 4)
    rt.gemv_q4k_f32(dev.up(W), dev.up(x), dy, N, K)
    _assert_rel(rt.from_device(dy, (N,), np.float32), orc.gemv_q4k_f32(W, x, N, K, acc64=True))


def test_gemv_integer_special_case_exact(orc, dev):
    """d = 1, dmin = 0, scales 1, x integers with d8 = 1: the GEMV is an exact integer dot."""
    g = synth.rng(14)
    N, K = 256, 2048
    W = synth.q4k_random(g, N, K)
    W[:, 0:2] = np.array([1.0], np.float16).view(np.uint8); W[:, 2:4] = 0
    W[:, 4:16] = synth.pack_q4k_scales(np.ones(8, np.uint8), np.zeros(8, np.uint8))
    x = g.integers(-100, 101, K).astype(np.float32)
    x[::32] = 127.0                                          # every block: amax 127 -> d8 = 1
    xq = orc.pack_q8_1(x)
    dy = dev.empty(N * 4)
    rt.gemv_q4k_q8_1(dev.up(W), dev.up(xq), dy, N, K)
    nib = orc.q4k_nibbles(W).reshape(N, K).astype(np.int64)
    assert np.array_equal(rt.from_device(dy, (N,), np.float32), (nib @ x.astype(np.int64)).astype(np.float32))


def test_gemm_op_launch_surface(orc, dev):
    """The graph's gemm node through compileAndLoad + cuLaunch: A bf16 -> Q8_1 -> GEMV, slots (A, B, out)."""
    g = synth.rng(15)
    N, K = 6144, 2048
    W = synth.q4k_random(g, N, K)
    a = synth.f32_to_bf16(g.standard_normal(K).astype(np.float32))
    k = rt.compileAndLoad(f"gemm N={N} K={K} cast=1")
    dout = dev.empty(N * 2)
    rc = rt.cuLaunch(k, [1, N // 64, 1], [128, 1, 1], [dev.up(a), dev.up(W), dout])
    assert rc == 0, rt.last_error()
    rt.cuSync()
    xq = orc.pack_q8_1(synth.bf16_to_f32(a))
    ref = orc.gemv_q4k_q8_1(W, xq, N, K)
    got = synth.bf16_to_f32(rt.from_device(dout, (N,), np.uint16))
    assert np.all(np.abs(got - ref) <= 2.0 ** -8 * np.abs(ref) + 1e-4 * np.sqrt(np.mean(ref ** 2)))
    # error paths: too few slots, unknown op, bad K
    assert rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [0, 0]) < 0 and "slots" in rt.last_error()
    with pytest.raises(rt.BunkerError, match="no kernel for op"):
        rt.compileAndLoad("nonsense N=1")
    with pytest.raises(rt.BunkerError, match="multiple of 256"):
        rt.compileAndLoad("gemm N=16 K=100")
    with pytest.raises(rt.BunkerError, match="multiple of 256"):
        rt.gemv_q4k_q8_1(1 << 20, 1 << 20, 1 << 20, 16, 100)


@pytest.mark.parametrize("N,K,B", [(6144, 2048, 32), (2048, 6144, 32), (16, 2048, 32), (100, 768, 7), (2048, 4096, 17),
                                   (4096, 2048, 40), (520, 512, 100)])
def test_gemm_mfma_equals_gemv_and_oracle(orc, dev, N, K, B):
    """Batched int8-MFMA matmul: same bits as the GEMV path and as the host loop in double, for every batch row."""
    print(f"gemm mfma N={N} K={K} B={B}", flush=True)
    g = synth.rng(700 + N + K + B)
    W = synth.q4k_random(g, N, K)
    x = g.standard_normal((B, K)).astype(np.float32)
    x[0] = 0.0                                              # an all-zero activation row
    xq = np.stack([orc.pack_q8_1(r) for r in x])
    res = synth.f32_to_bf16(g.standard_normal((B, N)).astype(np.float32))
    dW, dxq, dres = dev.up(W), dev.up(xq), dev.up(res)
    dy, dy2 = dev.empty(B * N * 4), dev.empty(B * N * 4)
    rt.gemm_q4k_q8_1(dW, dxq, dy, N, K, B)
    y = rt.from_device(dy, (B, N), np.float32)
    ref = np.stack([orc.gemv_q4k_q8_1(W, xq[b], N, K) for b in range(B)])
    _assert_rel(y, ref)
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), int((y != ref).sum())
    rt.gemv_q4k_q8_1(dW, dxq, dy2, N, K, batch=B)
    assert np.array_equal(rt.from_device(dy2, (B, N), np.float32).view(np.uint32), y.view(np.uint32))
    rt.gemm_q4k_q8_1(dW, dxq, dy, N, K, B, out_dtype=rt.BF16, residual=dres)
    ya = rt.from_device(dy, (B, N), np.uint16)
    assert np.array_equal(ya, orc.add_bf16(synth.f32_to_bf16(y).ravel(), res.ravel()).reshape(B, N))


@pytest.mark.parametrize("N,K,B", [(200, 2048, 70), (96, 1280, 32), (41, 3072, 19)])
def test_gemm_mfma_every_split_of_k_returns_the_same_bits(orc, dev, N, K, B):
    """1, 2, 4 or 8 wavefronts per tile (K split by super-block, partials joined in wave order): same bits as the host loop."""
    print(f"gemm mfma splits N={N} K={K} B={B}", flush=True)
    g = synth.rng(900 + N + K + B)
    W = synth.q4k_random(g, N, K)
    x = (g.standard_normal((B, K)) * np.exp(g.standard_normal((B, 1)))).astype(np.float32)
    xq = np.stack([orc.pack_q8_1(r) for r in x])
    ref = np.stack([orc.gemv_q4k_q8_1(W, xq[b], N, K) for b in range(B)])
    dW, dxq, dy = dev.up(W), dev.up(xq), dev.empty(B * N * 4)
    try:
        for r16 in (0, 1, 2):                  # tiles of 32, 16 or 8 weight rows (the narrow ones for a single batch tile only)
            rt.tune_set("gemm_r16", r16)
            for nw in (1, 2, 4, 8):
                rt.tune_set("gemm_nw", nw)
                rt.cuMemset(dy, 0xff, B * N * 4)
                rt.gemm_q4k_q8_1(dW, dxq, dy, N, K, B)
                y = rt.from_device(dy, (B, N), np.float32)
                assert np.array_equal(y.view(np.uint32), ref.view(np.uint32)), (r16, nw, int((y != ref).sum()))
    finally:
        rt.tune_set("gemm_nw", 0)
        rt.tune_set("gemm_r16", -1)


@pytest.mark.parametrize("exponent", [-139, -126, -100, -64, -62, 0, 60, 100])
@pytest.mark.parametrize("N,K", [(5, 256), (300, 1024), (1030, 2304), (2100, 2048), (9, 6144), (7, 6400)])
def test_gemv_q4k_f32_activations_of_any_magnitude(orc, dev, N, K, exponent):
    """The dots run on nibbles as subnormal halves, 2^-24 below their value; activations down to the smallest must keep their bits, in every form of the
    kernel (x shared by the workgroup or not, one to three rounds, rows of any length).  The same activations times a power of two give the
    same result times that power, unless it leaves the normal range: there half a unit of its last place (rows of more than 6144: of every lane's
    share of every round of 2048, which leave that range before they are added)."""
    print(f"gemv f32 magnitude N={N} K={K} 2^{exponent}", flush=True)
    g = synth.rng(9 + N + K)
    W = synth.q4k_random(g, N, K)
    x = (1 + g.random(K)).astype(np.float32) * g.choice(np.array([-1, 1], np.float32), K)
    if exponent < -126:      # subnormal activations: few significant bits, so that the scaling is exact
        x = np.round(x * 1024) / np.float32(1024)
    ys = []
    for e in (0, exponent):
        dy = dev.empty(N * 4)
        rt.gemv_q4k_f32(dev.up(W), dev.up((x.astype(np.float64) * 2.0**e).astype(np.float32)), dy, N, K)
        ys.append(rt.from_device(dy, (N,), np.float32))
    want = ys[0].astype(np.float64) * 2.0**exponent
    assert np.isfinite(ys[1]).all() and (np.abs(ys[1].astype(np.float64) - want) <= 2.0**-150 * (1 if K <= 6144 else 64 * -(-K // 2048))).all()
    _assert_rel(ys[0], orc.gemv_q4k_f32(W, x, N, K, acc64=True))


@pytest.mark.parametrize("loud,rest", [(0, -110), (0, -118), (0, -125), (97, -100), (98, -20), (110, -125)])
@pytest.mark.parametrize("N,K", [(5, 256), (300, 1024), (1030, 2304), (2100, 2048), (9, 6144), (7, 6400)])
def test_gemv_q4k_f32_small_activations_beside_a_large_one(orc, dev, N, K, loud, rest):
    """One activation of 2^loud under weights of zero (all rows but the first) among activations of about 2^rest, on both sides of the line where activations
    are no longer lifted: the small ones keep every bit of their products.  A term meets at most 33 roundings on its way (scale, a lane's sixteen FMAs or sums,
    the joins of its lane, rounds and wave, and three in the checker's weight) of half a unit each, 2^-24 of the sum of magnitudes, and below the normal
    range four per sixteen weights of 2^-150."""
    print(f"gemv f32 loud N={N} K={K} 2^{loud} 2^{rest}", flush=True)
    g = synth.rng(31 + N + K)
    W = synth.q4k_random(g, N, K, 1.0)
    quiet = W.reshape(N, K // 256, 144)[1:, K // 512]
    quiet[:, 4] &= 0xc0      # scale and min of its first sub-block
    quiet[:, 8] &= 0xc0
    x = ((1 + g.random(K)) * g.choice([-1.0, 1.0], K) * 2.0**rest).astype(np.float32)
    x[K // 512 * 256 + 5] = 2.0**loud
    dy = dev.empty(N * 4)
    rt.gemv_q4k_f32(dev.up(W), dev.up(x), dy, N, K)
    y = rt.from_device(dy, (N,), np.float32).astype(np.float64)
    parts = [W.copy(), W.copy()]      # the weights without their mins, and the mins alone
    parts[0][:, 2:4] = 0
    parts[1][:, 0:2] = 0
    terms = sum(np.abs(orc.gemv_q4k_f32(p, np.abs(x), N, K, acc64=True).astype(np.float64)) for p in parts)
    worst = np.abs(y - orc.gemv_q4k_f32(W, x, N, K, acc64=True)) / (33 * 2.0**-24 * terms + K / 4 * 2.0**-150)
    assert worst.max() <= 1.0, worst.max()
