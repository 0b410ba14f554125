"""The projections of 2 to 7 sequences that share one pass over the weights (csrc/gemv_rows.hip) against the CPU checker, to the
bit: every batch, row counts around the 16-row tiles and 32-row SwiGLU pieces, row lengths that leave waves without a
super-block, all epilogues, and the wave-per-tile form of a long matrix.  The small shapes here would run in the one-row forms,
which are faster for them, so the tests ask for gemv_rows wherever it serves ("rows" = 2)."""
import numpy as np
import pytest

from bunker_amd import runtime as rt
from bunker_amd import synth
from test_gpu_fused import Dev, bf, f32, launch, ref_activation

pytestmark = pytest.mark.gpu


@pytest.fixture()
def dev():
    d = Dev()
    yield d
    d.close()


@pytest.fixture(autouse=True)
def rows_wherever_served():
    rt.tune_set("rows", 2)
    yield
    rt.tune_set("rows", 1)


@pytest.mark.parametrize("K,batch,N,epi", [(1024, 2, 1, 0), (1024, 7, 33, 2), (1536, 5, 100, 1), (2048, 3, 17, 0), (2048, 7, 520, 2), (2560, 6, 48, 1),
                                           (3584, 5, 1024, 2), (4096, 4, 31, 2), (6144, 7, 2048, 2), (6144, 2, 15, 0),
                                           (1024, 5, 32773, 0), (2048, 7, 32768, 0), (1536, 3, 33000, 1), (2048, 2, 40001, 2)])
def test_one_matrix_over_q8_1_rows(orc, dev, K, batch, N, epi):
    print(f"gemv_rows pro=0 K={K} batch={batch} N={N} epi={epi}", flush=True)
    g = synth.rng(2100 + K + 10 * batch + N)
    W = synth.q4k_random(g, N, K)
    xq = [orc.pack_q8_1(f32(bf(g.standard_normal(K).astype(np.float32) * 10.0 ** b))) for b in range(batch)]      # rows of different sizes
    res = bf(g.standard_normal((batch, N)).astype(np.float32))
    size = 4 if epi == 0 else 2
    out = dev.empty(batch * N * size + 64)
    launch(f"gemv_fused K={K} pro=0 G=1 N0={N} epi0={epi} batch={batch}", [dev.up(np.stack(xq)), dev.up(W)] + ([dev.up(res)] if epi == 2 else []) + [out])
    raw = rt.from_device(out, (batch * N * size + 64,), np.uint8)
    assert np.all(raw[batch * N * size:] == 0xCD)
    got = raw[:batch * N * size].view(np.uint32 if epi == 0 else np.uint16).reshape(batch, N)
    for b in range(batch):
        y = orc.gemv_q4k_q8_1(W, xq[b], N, K)
        if epi == 0:
            ref = y.view(np.uint32)
        else:
            ref = orc.cast_bf16(y)
            if epi == 2:
                ref = orc.add_bf16(ref, res[b])
        assert np.array_equal(got[b], ref), (b, np.count_nonzero(got[b] != ref))


@pytest.mark.parametrize("K,batch", [(1024, b) for b in (2, 4, 5, 7)] + [(2048, b) for b in (2, 3, 6, 7)])
def test_norm_and_several_matrices(orc, dev, K, batch):
    """Tiles of one workgroup in different matrices, rows past the end of each."""
    print(f"gemv_rows pro=2 K={K} batch={batch}", flush=True)
    g = synth.rng(2200 + K + batch)
    Ns, epis = [49, 130, 16, 18], [1, 2, 0, 0]
    Ws = [synth.q4k_random(g, n, K) for n in Ns]
    x, w = bf(g.standard_normal((batch, K)).astype(np.float32)), bf((g.standard_normal(K) * 0.1).astype(np.float32))
    res = bf(g.standard_normal((batch, Ns[1])).astype(np.float32))
    xq = ref_activation(orc, 2, x, w)
    args, outs = [dev.up(x), dev.up(w)], []
    for i, n in enumerate(Ns):
        o = dev.empty(batch * n * (4 if epis[i] == 0 else 2)); outs.append(o)
        args += [dev.up(Ws[i])] + ([dev.up(res)] if epis[i] == 2 else []) + [o]
    launch(f"gemv_fused K={K} pro=2 G=4 batch={batch} " + " ".join(f"N{i}={n} epi{i}={e}" for i, (n, e) in enumerate(zip(Ns, epis))), args)
    for i, n in enumerate(Ns):
        got = rt.from_device(outs[i], (batch, n), np.uint32 if epis[i] == 0 else np.uint16)
        for b in range(batch):
            y = orc.gemv_q4k_q8_1(Ws[i], xq[b], n, K)
            ref = y.view(np.uint32) if epis[i] == 0 else orc.cast_bf16(y)
            assert np.array_equal(got[b], orc.add_bf16(ref, res[b]) if epis[i] == 2 else ref), (i, b)


def _silu_conv(orc, y, st, w):
    """Rows [B, C] (f32) through bf16 and the convolution step: outputs and new states."""
    return [np.stack(v) for v in zip(*(orc.conv1d_decode(orc.cast_bf16(y[b]), st[b], w) for b in range(len(y))))]


@pytest.mark.parametrize("K,batch,Ns", [(1024, 2, (50, 33, 16, 16)), (1024, 7, (6144, 2048, 32, 32)), (2048, 3, (70, 33, 16, 16)),
                                        (2048, 2, (6144, 2048, 16, 16)), (2048, 5, (6100, 2050, 17, 33)), (2048, 7, (6144, 2048, 16, 16))])
def test_norm_group_with_the_convolution(orc, dev, K, batch, Ns):
    """A GDN layer's projections with the convolution behind the first: two tiles a workgroup, and three where the group has more
    than 512 tiles (6144 + 2048 + 16 + 16 rows at K = 2048), with row counts that are and are not whole workgroups."""
    print(f"gemv_rows conv K={K} batch={batch} N={Ns}", flush=True)
    g = synth.rng(2700 + K + batch + Ns[0])
    Ws = [synth.q4k_centered(g, n, K, 0.5) for n in Ns]
    x, w = bf(g.standard_normal((batch, K)).astype(np.float32)), bf((g.standard_normal(K) * 0.1).astype(np.float32))
    st = bf(g.standard_normal((batch, 3, Ns[0])).astype(np.float32))
    cw = bf((g.standard_normal((Ns[0], 4)) * 0.5).astype(np.float32))
    xq = ref_activation(orc, 2, x, w)
    outs = [dev.empty(batch * n * s + 64) for n, s in zip(Ns, (2, 2, 4, 4))]
    dst = dev.up(st)                                             # the new state over the old one, as the decode step has it
    launch(f"gemv_fused K={K} pro=2 G=4 N0={Ns[0]} epi0=3 N1={Ns[1]} epi1=1 N2={Ns[2]} epi2=0 N3={Ns[3]} epi3=0 batch={batch}",
           [dev.up(x), dev.up(w), dev.up(Ws[0]), dst, dev.up(cw), outs[0], dst, dev.up(Ws[1]), outs[1], dev.up(Ws[2]), outs[2], dev.up(Ws[3]), outs[3]])
    ref = [np.stack([orc.gemv_q4k_q8_1(W, r, n, K) for r in xq]) for W, n in zip(Ws, Ns)]
    ro, rs = _silu_conv(orc, ref[0], st, cw)
    assert np.array_equal(rt.from_device(outs[0], (batch, Ns[0]), np.uint16), ro)
    assert np.array_equal(rt.from_device(dst, st.shape, np.uint16), rs)
    assert np.array_equal(rt.from_device(outs[1], (batch, Ns[1]), np.uint16), np.stack([orc.cast_bf16(r) for r in ref[1]]))
    for i in (2, 3):
        assert np.array_equal(rt.from_device(outs[i], (batch, Ns[i]), np.uint32), ref[i].view(np.uint32))
    for o, n, s in zip(outs, Ns, (2, 2, 4, 4)):
        assert np.all(rt.from_device(o, (batch * n * s + 64,), np.uint8)[batch * n * s:] == 0xCD)


@pytest.mark.parametrize("batch,Ns,epis", [(2, (8192, 512, 512), (1, 1, 1)), (6, (8192, 520, 33), (1, 0, 2)), (7, (8250,), (0,))])
def test_norm_groups_of_more_than_512_tiles(orc, dev, batch, Ns, epis):
    """K = 2048, three tiles a workgroup without the convolution: an attention layer's q, k, v and row counts past whole workgroups."""
    K = 2048
    print(f"gemv_rows pro=2 K={K} batch={batch} N={Ns}", flush=True)
    g = synth.rng(2800 + batch)
    Ws = [synth.q4k_random(g, n, K) for n in Ns]
    x, w = bf(g.standard_normal((batch, K)).astype(np.float32)), bf((g.standard_normal(K) * 0.1).astype(np.float32))
    xq = ref_activation(orc, 2, x, w)
    args, outs, ress = [dev.up(x), dev.up(w)], [], []
    for W, n, e in zip(Ws, Ns, epis):
        ress.append(bf(g.standard_normal((batch, n)).astype(np.float32)))
        outs.append(dev.empty(batch * n * 4))
        args += [dev.up(W)] + ([dev.up(ress[-1])] if e == 2 else []) + [outs[-1]]
    launch(f"gemv_fused K={K} pro=2 G={len(Ns)} batch={batch} " + " ".join(f"N{i}={n} epi{i}={e}" for i, (n, e) in enumerate(zip(Ns, epis))), args)
    for W, n, e, o, res in zip(Ws, Ns, epis, outs, ress):
        got = rt.from_device(o, (batch, n), np.uint32 if e == 0 else np.uint16)
        for b in range(batch):
            y = orc.gemv_q4k_q8_1(W, xq[b], n, K)
            ref = y.view(np.uint32) if e == 0 else orc.cast_bf16(y)
            assert np.array_equal(got[b], orc.add_bf16(ref, res[b]) if e == 2 else ref), (n, b)


@pytest.mark.parametrize("K,N,batch", [(1024, 96, 2), (1024, 3584, 5), (2048, 32, 7), (2048, 6144, 4), (1024, 100, 3), (2048, 52, 6)])
def test_swiglu_as_bf16_and_as_q8_1(orc, dev, K, N, batch):
    print(f"gemv_rows swiglu K={K} N={N} batch={batch}", flush=True)
    g = synth.rng(2300 + N + batch)
    Wg, Wu = synth.q4k_centered(g, N, K, 0.05), synth.q4k_centered(g, N, K, 0.05)
    x, w = bf(g.standard_normal((batch, K)).astype(np.float32)), bf((g.standard_normal(K) * 0.1).astype(np.float32))
    xq = ref_activation(orc, 2, x, w)
    ref = [orc.swiglu(orc.gemv_q4k_q8_1(Wg, r, N, K), orc.gemv_q4k_q8_1(Wu, r, N, K)) for r in xq]
    common = [dev.up(x), dev.up(w), dev.up(Wg), dev.up(Wu)]
    spec = f"gemv_fused K={K} pro=2 G=2 swiglu=1 N0={N} N1={N} batch={batch}"
    out = dev.empty(batch * N * 2)
    launch(spec, common + [out])
    assert np.array_equal(rt.from_device(out, (batch, N), np.uint16), np.stack(ref))
    if N % 32:
        with pytest.raises(rt.BunkerError, match="q8only"):
            rt.compileAndLoad(spec + " q8only=1")
        return
    q8 = dev.empty(batch * (N // 32) * 36)
    launch(spec + " q8only=1", common + [q8])
    got = rt.from_device(q8, (batch, (N // 32) * 36), np.uint8)
    for b in range(batch):
        assert np.array_equal(got[b], orc.pack_q8_1(f32(ref[b]))), b


@pytest.mark.parametrize("spec", ["gemv_fused K=2048 pro=2 G=2 swiglu=1 N0=64 N1=64 q8only=1", "gemv_fused K=2048 pro=2 G=2 swiglu=1 N0=64 N1=64 batch=8 q8only=1",
                                  "gemv_fused K=512 pro=2 G=2 swiglu=1 N0=64 N1=64 batch=3 q8only=1", "gemv_fused K=2048 pro=0 G=1 N0=64 batch=3 q8only=1"])
def test_q8only_is_refused_where_nothing_serves_it(spec):
    with pytest.raises(rt.BunkerError, match="q8only"):
        rt.compileAndLoad(spec)


@pytest.mark.parametrize("K,N,batch,epi", [(1536, 9000, 5, 0), (2560, 8192, 3, 1), (3072, 40, 7, 2), (4608, 100, 2, 0), (5120, 33, 4, 2), (5632, 17, 6, 1)])
def test_q8_1_rows_at_four_byte_alignment(orc, dev, K, N, batch, epi):
    """Row lengths that the one-row form serves from four-byte alignment on are served there for several rows too."""
    print(f"gemv_fused pro=0 K={K} N={N} batch={batch} epi={epi}, rows at +4 bytes", flush=True)
    g = synth.rng(2400 + K)
    W = synth.q4k_random(g, N, K)
    xq = np.stack([orc.pack_q8_1(f32(bf(g.standard_normal(K).astype(np.float32)))) for _ in range(batch)])
    res = bf(g.standard_normal((batch, N)).astype(np.float32))
    at = dev.up(np.concatenate([np.zeros(4, np.uint8), np.ascontiguousarray(xq).view(np.uint8).ravel()])) + 4
    out = dev.empty(batch * N * (4 if epi == 0 else 2))
    launch(f"gemv_fused K={K} pro=0 G=1 N0={N} epi0={epi} batch={batch}", [at, dev.up(W)] + ([dev.up(res)] if epi == 2 else []) + [out])
    got = rt.from_device(out, (batch, N), np.uint32 if epi == 0 else np.uint16)
    for b in range(batch):
        y = orc.gemv_q4k_q8_1(W, xq[b], N, K)
        ref = y.view(np.uint32) if epi == 0 else orc.cast_bf16(y)
        assert np.array_equal(got[b], orc.add_bf16(ref, res[b]) if epi == 2 else ref), b


def test_epilogue_2_without_a_residual_is_the_bf16_result(orc, dev):
    K, N, batch = 4608, 50, 3
    g = synth.rng(2500)
    W = synth.q4k_random(g, N, K)
    xq = np.stack([orc.pack_q8_1(f32(bf(g.standard_normal(K).astype(np.float32)))) for _ in range(batch)])
    out = dev.empty(batch * N * 2)
    launch(f"gemv_fused K={K} pro=0 G=1 N0={N} epi0=2 batch={batch}", [dev.up(xq), dev.up(W), 0, out])
    got = rt.from_device(out, (batch, N), np.uint16)
    for b in range(batch):
        assert np.array_equal(got[b], orc.cast_bf16(orc.gemv_q4k_q8_1(W, xq[b], N, K))), b


@pytest.mark.parametrize("K", [1024, 2048, 3584, 4096, 6144])
def test_misaligned_rows_of_the_fused_lengths_stay_refused(dev, K):
    out = dev.empty(3 * 64 * 4)
    k = rt.compileAndLoad(f"gemv_fused K={K} pro=0 G=1 N0=64 epi0=0 batch=3")
    x, w = dev.empty(3 * K // 32 * 36 + 16), dev.empty(64 * K // 256 * 144)
    assert rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [x + 4, w, out]) != 0 and "aligned" in rt.last_error()


@pytest.mark.parametrize("spec,Ks,Ns", [
    ("pro=0 G=1 N0={0} epi0=0", 1024, (4100, 4300)), ("pro=0 G=1 N0={0} epi0=1", 2048, (16300, 16400)), ("pro=0 G=1 N0={0} epi0=0", 1536, (7900, 8100)),
    ("pro=0 G=1 N0={0} epi0=1", 4096, (4090, 4230)), ("pro=0 G=1 N0={0} epi0=0", 2560, (4090, 4100)), ("pro=0 G=1 N0={0} epi0=0", 4608, (4090, 4100)),
    ("pro=2 G=2 N0={0} epi0=0 N1=33 epi1=1", 1024, (4100, 4300)), ("pro=2 G=1 N0={0} epi0=1", 2048, (6200, 6400)),
    ("pro=2 G=2 swiglu=1 N0={0} N1={0}", 1024, (2700, 2800)), ("pro=2 G=2 swiglu=1 N0={0} N1={0}", 2048, (8192, 8224))])
@pytest.mark.parametrize("batch", [2, 3])
def test_both_sides_of_the_rule_have_the_same_bits(dev, spec, Ks, Ns, batch):
    """gemv_rows_pays sends the longer of the two matrices here at batch 2 or 3; never, always and by the rule agree."""
    for N in Ns:
        print(f"K={Ks} N={N} batch={batch} {spec}", flush=True)
        g = synth.rng(2600 + N + Ks)
        ns = [N, N] if "swiglu" in spec else ([N, 33] if "N1=33" in spec else [N])
        W = [dev.up(synth.q4k_centered(g, n, Ks, 0.05)) for n in ns]
        x, nw = dev.up(bf(g.standard_normal((batch, Ks)).astype(np.float32))), dev.up(bf((g.standard_normal(Ks) * 0.1).astype(np.float32)))
        if "pro=0" in spec:
            xq = dev.empty(batch * Ks // 32 * 36)
            rt.quantize_q8_1(x, xq, Ks, batch, rt.BF16)
            head = [xq]
        else:
            head = [x, nw]
        got = []
        for rows in (0, 1, 2):
            rt.tune_set("rows", rows)
            outs = [dev.empty(batch * n * 4) for n in ns]
            args = head + W + [outs[0]] if "swiglu" in spec else head + [v for pair in zip(W, outs) for v in pair]
            launch(f"gemv_fused K={Ks} {spec.format(N)} batch={batch}", args)
            got.append([rt.from_device(o, (batch * n * 4,), np.uint8) for o, n in zip(outs, ns)])
        for other in got[1:]:
            assert all(np.array_equal(a, b) for a, b in zip(got[0], other)), N
