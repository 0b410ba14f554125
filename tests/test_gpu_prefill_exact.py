"""Causal prompt attention in double precision, 16 query rows a workgroup (fa2_prefill with enough tokens): every output must have
the bits of the one-token-a-workgroup form and of the checker, whatever lies in the cache behind a row's context."""
import ctypes as C

import numpy as np
import pytest

from bunker_amd import runtime as rt
from bunker_amd import synth

pytestmark = pytest.mark.gpu

bf = synth.f32_to_bf16
f32 = synth.bf16_to_f32
HD, HALF = 256, 32


@pytest.fixture(scope="module", autouse=True)
def gpu():
    rt.cu(0)


class _Case:
    def __init__(self, orc, seed, NH, NKV, T, pos, max_len):
        g = synth.rng(seed)
        self.NH, self.NKV, self.T, self.max_len, self.g = NH, NKV, T, max_len, g
        pages = max_len // 16
        r = lambda *s: bf(g.standard_normal(s).astype(np.float32))  # noqa: E731
        self.cos, self.sin = orc.rope_tables(max_len, 2 * HALF, 1e7)
        self.kc, self.vc = r(pages, NKV, 16, HD), r(pages, NKV, 16, HD)
        self.qgate, self.k, self.v = r(T, NH, 2, HD), r(T, NKV, HD), r(T, NKV, HD)
        self.qw, self.kw = (bf((g.standard_normal(HD) * 0.1).astype(np.float32)) for _ in range(2))
        self.table = g.permutation(pages).astype(np.int32)
        self.pos = np.asarray(pos, np.int32)

    def run(self, form, shift=0):
        """``shift``: bytes by which the query | gate and output addresses miss the allocation's alignment"""
        rt.tune_set("prefill_exact", form)
        try:
            qgate = np.concatenate([np.zeros(shift, np.uint8), self.qgate.ravel().view(np.uint8)])
            ptrs = [rt.to_device(a) for a in (qgate, self.k, self.v, self.qw, self.kw, self.cos, self.sin, self.pos, self.table, self.kc,
                                              rt.v_pages_to_device_layout(self.vc))]
            out = rt.cuAlloc(self.T * self.NH * HD * 2 + 16)
            rt.cuMemset(out, 0x5a, self.T * self.NH * HD * 2 + 16)
            k = rt.compileAndLoad(f"fa2_prefill HD={HD} NH={self.NH} NKV={self.NKV} MAX_LEN={self.max_len} ROT_HALF={HALF} T={self.T}")
            assert rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [ptrs[0] + shift, *ptrs[1:], out + shift]) == 0, rt.last_error()
            rt.cuSync()
            raw = rt.from_device(out, (self.T * self.NH * HD * 2 + 16,), np.uint8)
            assert (raw[:shift] == 0x5a).all() and (raw[raw.size - 16 + shift:] == 0x5a).all()
            y = raw[shift:raw.size - 16 + shift].view(np.uint16).reshape(self.T, self.NH, HD)
            rt.unloadKernel(k)
            for p in ptrs + [out]:
                rt.cuFree(p)
            return y
        finally:
            rt.tune_set("prefill_exact", -1)


def _same(a, b):
    fa, fb = f32(a), f32(b)
    nan = np.isnan(fa)
    assert np.array_equal(nan, np.isnan(fb))
    assert np.array_equal(a[~nan], b[~nan]), int((a[~nan] != b[~nan]).sum())


@pytest.mark.parametrize("NH,NKV,T,pos0", [(16, 2, 1, 0), (16, 2, 2, 14), (16, 2, 145, 0), (16, 2, 33, 700), (8, 2, 3, 15), (8, 2, 147, 30), (4, 2, 9, 1),
                                           (4, 2, 65, 250), (2, 2, 17, 0), (2, 2, 150, 13), (8, 1, 16, 47), (12, 2, 150, 5)])
def test_equals_one_token_a_workgroup(orc, NH, NKV, T, pos0):
    print(f"prefill exact NH={NH} NKV={NKV} T={T} pos0={pos0}", flush=True)
    c = _Case(orc, 1300 + NH + T + pos0, NH, NKV, T, pos0 + np.arange(T), 1024)
    c.vc[:] = np.where(c.g.random(c.vc.shape) < 0.01, 0x7fc0, c.vc) if pos0 == 0 else c.vc      # no cached token is a context token then
    _same(c.run(1), c.run(0))


@pytest.mark.parametrize("NH,NKV", [(2, 2), (4, 2), (12, 2), (8, 1)])
def test_first_launch_of_a_new_handle(orc, NH, NKV):
    """A handle's workspace starts with what the memory held before (here NaNs of both widths) and is launched right behind its creation: one
    to eight heads a KV head, the ones that leave columns of the query copy unused among them."""
    c = _Case(orc, 1370 + NH, NH, NKV, 9, 40 + np.arange(9), 1024)
    want = c.run(1)
    for _ in range(3):
        old = [rt.cuAlloc(n) for n in (1 << 20, 4 << 20, 16 << 20)]
        for p, n in zip(old, (1 << 20, 4 << 20, 16 << 20)):
            rt.cuMemset(p, 0xff, n)
        for p in old:
            rt.cuFree(p)
        _same(c.run(0), want)


@pytest.mark.parametrize("shift", [2, 4, 8])
def test_gate_and_output_at_any_address(orc, shift):
    c = _Case(orc, 1350, 16, 2, 37, 5 + np.arange(37), 64)
    want = c.run(0)
    _same(c.run(1), want)
    _same(c.run(1, shift), want)
    _same(c.run(0, shift), want)


@pytest.mark.parametrize("T,NKV,max_len,rows16", [
    (4096, 2, 4352, True), (2048, 8, 16384, True), (143, 2, 4352, False), (144, 2, 16384, True),
    # longer caches, cut into ranges: the one-token form keeps the launches of few tokens and those just past a workgroup per CU (512 pairs)
    (144, 2, 16400, False), (199, 2, 65536, False), (200, 2, 65536, True), (256, 2, 65536, True), (258, 2, 65536, False), (360, 2, 32768, False),
    (361, 2, 32768, True), (515, 2, 65536, False), (1024, 2, 65536, True)])
def test_a_handle_keeps_no_workspace_that_its_form_does_not_read(T, NKV, max_len, rows16):
    """The form follows from the shape, as the lines of the table say, and the memory from the form: the 16-row form needs the normalised queries (bf16) alone; a token a workgroup also their copy in double (4 bytes a value, eight
    columns a KV head) and the partial results of its cut."""
    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert rt.cu().hipMemGetInfo(C.byref(free), C.byref(total)) == 0      # (of the runtime that the library is linked against)
        return free.value

    NH = 16
    spec = f"fa2_prefill HD={HD} NH={NH} NKV={NKV} MAX_LEN={max_len} ROT_HALF={HALF} T={T}"
    rt.unloadKernel(rt.compileAndLoad(spec))
    rt.cuSync()
    free = free_bytes()
    k = rt.compileAndLoad(spec)
    used = free - free_bytes()
    rt.unloadKernel(k)
    queries, copy = T * NH * HD * 2, T * NKV * HD * 8 * 4
    assert used <= queries + (4 << 20) if rows16 else used >= queries + copy, (used, queries, copy)


def test_positions_in_any_order_and_outside_the_cache(orc):
    g = synth.rng(5)
    pos = g.permutation(256)[:40]
    pos[3], pos[17] = -1, 255
    c = _Case(orc, 1401, 16, 2, 40, pos, 256)
    _same(c.run(1), c.run(0))


@pytest.mark.parametrize("where", ["prompt", "cached", "key", "query"])
def test_values_that_are_no_numbers_reach_only_the_rows_that_see_them(orc, where):
    c = _Case(orc, 1500, 16, 2, 150, 37 + np.arange(150), 256)
    if where == "prompt":                     # a token of the prompt whose value overflowed: the rows before it must not notice
        c.v[9, 0, 5], c.v[64, 1, 200], c.v[65, 1, 3] = 0x7f80, 0x7fc0, 0xff80
    elif where == "cached":
        c.vc[c.table[1], 0, 3, 77] = 0x7f80
    elif where == "key":
        c.k[31, 1, 100], c.kc[c.table[0], 0, 2, 9] = 0x7fc0, 0x7f80
    else:
        c.qgate[12, 3, 0, 4] = 0x7fc0
    _same(c.run(1), c.run(0))


def test_a_wave_whose_pages_hold_only_scores_of_minus_infinity_adds_nothing(orc):
    """Page 1 (all that the second of the four waves sees before page 5) has an infinite key element and every query a negative one
    there: its 16 scores are -inf and their weights 0, and the rows are what the other pages make them."""
    T, NH, NKV, pos0 = 150, 16, 2, 32
    c = _Case(orc, 1650, NH, NKV, T, pos0 + np.arange(T), 256)
    c.kc[c.table[1], :, :, 100] = 0x7f80
    c.qgate[:, :, 0, 100] |= 0x8000
    out = c.run(1)
    _same(out, c.run(0))
    kc, vc = c.kc.copy(), c.vc.copy()
    for t in range(3):
        kn = orc.rope(orc.headnorm(c.k[t].ravel(), c.kw, NKV, HD, HD), c.cos, c.sin, c.pos[t], NKV, HD, HALF)
        orc.kv_append(kn.reshape(NKV, HD), c.v[t], kc, vc, c.table, c.pos[t], NKV, HD, 16)
        qn = orc.rope(orc.headnorm(c.qgate[t].ravel(), c.qw, NH, HD, 2 * HD), c.cos, c.sin, c.pos[t], NH, HD, HALF).reshape(1, NH, HD)
        ro, _ = orc.attn_decode_paged(qn, kc, vc, c.table[None], np.array([c.pos[t] + 1], np.int32), 1, NH, NKV, HD, 16,
                                      gate=c.qgate[t].ravel()[HD:], gate_bstride=0, gate_hstride=2 * HD)
        assert np.isfinite(f32(ro[0])).all() and np.abs(f32(ro[0])).max() > 0
        assert np.array_equal(f32(out[t]), f32(ro[0])), t


def test_large_scores_move_the_reference_exponent(orc):
    c = _Case(orc, 1600, 16, 2, 150, 200 + np.arange(150), 512)
    c.qw[:], c.kw[:] = bf(np.full(HD, 30.0, np.float32)), bf(np.full(HD, 20.0, np.float32))       # scores of several thousand
    _same(c.run(1), c.run(0))


@pytest.mark.parametrize("T", [1, 150])
def test_a_call_is_refused_whatever_the_number_of_tokens(T):
    """Caches that are not aligned to 16 bytes and a cut into ranges of more than 1024 pages, by the one-token form and by the
    16-row form alike (the buffers have room for what the preparation launch in front of the refusal writes)."""
    NH, NKV, ML = 16, 2, 16400
    sizes = [T * NH * 2 * HD * 2, T * NKV * HD * 2, T * NKV * HD * 2, HD * 2, HD * 2, ML * HALF * 4, ML * HALF * 4, T * 4, ML // 16 * 4,
             ML * NKV * HD * 2 + 64, ML * NKV * HD * 2 + 64, T * NH * HD * 2]
    ptrs = [rt.cuAlloc(n) for n in sizes]
    for p, n in zip(ptrs, sizes):
        rt.cuMemset(p, 0, n)
    spec = f"fa2_prefill HD={HD} NH={NH} NKV={NKV} MAX_LEN={ML} ROT_HALF={HALF} T={T}"
    for extra, moved in ((" splits=1", None), ("", 9), ("", 10), ("", None)):
        k = rt.compileAndLoad(spec + extra)
        rc = rt.cuLaunch(k, [1, 1, 1], [128, 1, 1], [p + 8 * (i == moved) for i, p in enumerate(ptrs)])
        rt.cuSync()
        rt.unloadKernel(k)
        assert (rc != 0) == (bool(extra) or moved is not None), (extra, moved, rc)
    for p in ptrs:
        rt.cuFree(p)


def test_the_default_route_has_the_checkers_bits(orc):
    T, NH, NKV, pos0 = 150, 16, 2, 21
    c = _Case(orc, 1700, NH, NKV, T, pos0 + np.arange(T), 192)
    out = c.run(-1)
    kc, vc = c.kc.copy(), c.vc.copy()
    for t in range(T):
        qn = orc.rope(orc.headnorm(c.qgate[t].ravel(), c.qw, NH, HD, 2 * HD), c.cos, c.sin, c.pos[t], NH, HD, HALF).reshape(1, NH, HD)
        kn = orc.rope(orc.headnorm(c.k[t].ravel(), c.kw, NKV, HD, HD), c.cos, c.sin, c.pos[t], NKV, HD, HALF)
        orc.kv_append(kn.reshape(NKV, HD), c.v[t], kc, vc, c.table, c.pos[t], NKV, HD, 16)
        ro, _ = orc.attn_decode_paged(qn, kc, vc, c.table[None], np.array([c.pos[t] + 1], np.int32), 1, NH, NKV, HD, 16,
                                      gate=c.qgate[t].ravel()[HD:], gate_bstride=0, gate_hstride=2 * HD)
        assert np.array_equal(f32(out[t]), ro[0].astype(np.float32) if ro.dtype != np.uint16 else f32(ro[0])), t
