// Causal attention of T prompt tokens in double precision (prototypes/fa2_vllm.ts:114-139 evaluated in doubles), on the
// double-precision matrix instruction.  Same contract as attn_exact.hip: bf16 x bf16 products are exact, every sum is carried
// in f64, one rounding to f32; the order of the additions only moves the ~1e-16 tail, so the outputs are the bits of T
// single-token launches.
//
// A decode step has 8 query heads per KV head, half of the 16 columns of v_mfma_f64_16x16x4_f64, and nothing is gained over
// vector FMAs (attn_exact.hip).  A prompt fills them: a workgroup takes 16 query rows, 16 / G consecutive tokens x the G heads
// of a KV head, and its four waves walk the pages (16 tokens each) w, w + 4, ...  Per page and wave:
//   S^T[16 keys x 16 rows] = K . Q^T      64 instructions, K converted once for 16 rows, Q^T as doubles in LDS (one
//                                         512-byte read each, in lane order)
//   p = exp(s - ref)                      lane (row, q) holds keys 4q .. 4q + 3: the key rows enter the product permuted so that
//                                         the result is the second product's operand as it lies in the registers
//   O^T[256 dims x 16 rows] += V^T . P^T  64 instructions, V read as its pages lie (dim-major, 4 keys = 8 bytes a lane)
// `ref` is a reference exponent per row and wave, moved only when a score exceeds it by more than 600.  The waves'
// partial results meet through LDS at the end.
//
// Bound: the double-precision unit, 128 matrix instructions of 27 ns per page and 16 rows (3.4 us of a SIMD); conversions and
// exponentials bring a page to 5 us (the vector unit stands still while that instruction runs).  The whole op for 1024 tokens x 16
// heads, a token a workgroup and here: from empty 413 / 197 us, behind 1024 cached 840 / 474, behind 15360 6873 / 4485; 8 heads (four
// tokens a workgroup) 348 / 134 and 778 / 280.  Eight waves a workgroup instead of two workgroups of four: 16 % and 9 % slower.
// Registers: 256, two workgroups a CU.  What the loop over the one-token passes would carry across the pages (addresses of the tail
// and of the query copy) is worked out where it is used, behind an index that the compiler cannot see through: with 30 registers
// in scratch the whole op took 213 us from empty and 493 behind 1024, now 201 and 478 (same box).
#include "attn_args.h"

namespace bk {

typedef __attribute__((ext_vector_type(4))) double d64x4_t;

struct PrefillExactArgs {
  const uint16_t *q, *kc, *vc, *gate;
  const int32_t *block_table, *pos;
  uint16_t* out;
  int64_t gate_bstride, gate_hstride;
  int T, NH, NKV, max_ctx, groups;       // groups of 16 / G tokens
  int wide;                              // gate and out at 8-byte alignment: four values at a time
  float scale;
};

__device__ __forceinline__ double pe_lo(uint32_t w) { return (double)__uint_as_float(w << 16); }
__device__ __forceinline__ double pe_hi(uint32_t w) { return (double)__uint_as_float(w & 0xffff0000u); }

constexpr double PE_REF_SLACK = 600.0;
constexpr int PE_PAD = 17;               // doubles per dim of the exchange buffer (16 rows, padded against bank conflicts)

template <int G>
__global__ __launch_bounds__(256, 2) void attn_prefill_exact_kernel(PrefillExactArgs A) {
  constexpr int TK = 16 / G, NW = 4;     // tokens and waves of a workgroup
  // Q^T [64 steps][4][16 rows] while the pages are walked, the exchange buffer [NW waves][64 dims][PE_PAD] afterwards
  __shared__ __align__(16) double lds[NW * 64 * PE_PAD];
  __shared__ double lds_m[NW][16], lds_l[NW][16];
  static_assert(NW * 64 * PE_PAD >= 64 * 64, "Q fits the exchange buffer");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, q4 = lane >> 4;
  // longest contexts first: the short ones fill the end of the launch
  const int kvh = blockIdx.x % A.NKV, t0 = (A.groups - 1 - (int)blockIdx.x / A.NKV) * TK;

  // the row's context and the longest and shortest of the workgroup
  const int tok = t0 + l16 / G;
  const int ctx = tok < A.T ? min(max(A.pos[tok], -1), A.max_ctx - 1) + 1 : 0;      // a position outside the cache reads as the nearest end
  int cmax = ctx, cmin = tok < A.T ? ctx : A.max_ctx;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    cmax = max(cmax, __shfl_xor(cmax, o));
    cmin = min(cmin, __shfl_xor(cmin, o));
  }
  cmax = __builtin_amdgcn_readfirstlane(cmax);
  cmin = __builtin_amdgcn_readfirstlane(cmin);
  // Keys that only some of the rows reach have weight 0 for the others.  Where one of them holds no number (0 * inf is none either), the
  // workgroup takes its tokens one after the other.
  bool odd = false;
  for (int pg = cmin / ATT_PAGE; pg * ATT_PAGE < cmax; pg++) {
    const uint4* p = (const uint4*)(A.vc + ((int64_t)A.block_table[pg] * A.NKV + kvh) * (ATT_PAGE * ATT_HD) + tid * ATT_PAGE);
    const uint4 a = p[0], b = p[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int k = pg * ATT_PAGE + i;
      odd |= k >= cmin && k < cmax && ((w[i >> 1] >> (16 * (i & 1))) & 0x7f80u) == 0x7f80u;
    }
  }
  const int passes = __syncthreads_or(odd) ? TK : 1;
  for (int pass = 0; pass < passes; pass++) {
  const int only = passes > 1 ? pass : -1;                       // the one token of this pass
  const int lim = only < 0 || l16 / G == only ? ctx : 0;
  const int lmax = only < 0 ? cmax : __builtin_amdgcn_readfirstlane(__shfl(ctx, only * G));
  const int npages = (lmax + ATT_PAGE - 1) / ATT_PAGE;
  if (pass) __syncthreads();

  // Q^T to LDS: thread (row, 16 dims)
  {
    int tq = tid;
    asm volatile("" : "+v"(tq));           // (worked out in every pass, as below the pages)
    const int row = tq & 15, part = tq >> 4, t = min(t0 + row / G, A.T - 1);
    const uint4* p = (const uint4*)(A.q + ((int64_t)t * A.NH + kvh * G + row % G) * ATT_HD + 16 * part);
    const uint4 a = p[0], b = p[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int dim = 16 * part + i;
      lds[((dim & 63) * 4 + (dim >> 6)) * 16 + row] = (i & 1) ? pe_hi(w[i >> 1]) : pe_lo(w[i >> 1]);
    }
  }
  __syncthreads();

  // K: lane (l16, q4) holds dims 64 q4 .. + 63 of key 4 (l16 % 4) + l16 / 4, so that row 4 v + q4 of the product is key 4 q4 + v
  const int key = ((l16 & 3) << 2) | (l16 >> 2);
  auto page_at = [&](int p) -> int64_t { return ((int64_t)A.block_table[min(p, npages - 1)] * A.NKV + kvh) * (ATT_PAGE * ATT_HD); };
  uint4 kr[8];
  auto load_k = [&](int64_t base) {
    const uint4* p = (const uint4*)(A.kc + base + key * ATT_HD + 64 * q4);
#pragma unroll
    for (int i = 0; i < 8; i++) kr[i] = p[i];
  };
  d64x4_t O[16];
#pragma unroll
  for (int n = 0; n < 16; n++) O[n] = (d64x4_t){0.0, 0.0, 0.0, 0.0};
  double mref = ATT_NO_REF, l = 0.0;

  int64_t base = 0;
  if (wave < npages) { base = page_at(wave); load_k(base); }
  for (int pg = wave; pg < npages; pg += NW) {
    // V of this page travels during the first product, K of the next during the second
    uint2 vr[16];
    {
      const uint16_t* p = A.vc + base + l16 * ATT_PAGE + 4 * q4;
#pragma unroll
      for (int n = 0; n < 16; n++) vr[n] = *(const uint2*)(p + n * 16 * ATT_PAGE);
    }
    base = page_at(pg + NW);
    int ln = lane;
    asm volatile("" : "+v"(ln));             // (Q does not change from page to page, but its 64 doubles have no registers to stay in)
    d64x4_t s0 = {0.0, 0.0, 0.0, 0.0}, s1 = s0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const uint32_t w[4] = {kr[i].x, kr[i].y, kr[i].z, kr[i].w};
      double qv[8];
#pragma unroll
      for (int e = 0; e < 8; e++) qv[e] = lds[(8 * i + e) * 64 + ln];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        s0 = __builtin_amdgcn_mfma_f64_16x16x4f64(pe_lo(w[e]), qv[2 * e], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f64_16x16x4f64(pe_hi(w[e]), qv[2 * e + 1], s1, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);     // (the conversions of a whole page would not fit the registers)
    }
    load_k(base);                          // (the last page again behind the end)
    double s[4], p[4];
    bool valid[4];
    float smax = -INFINITY;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      s[v] = (s0[v] + s1[v]) * (double)A.scale;
      valid[v] = pg * ATT_PAGE + 4 * q4 + v < lim;
      smax = fmaxf(smax, valid[v] ? (float)s[v] : -INFINITY);
    }
    if (__ballot(smax > -INFINITY && (double)smax > mref + PE_REF_SLACK) != 0) {     // the first page with a key of a row, rarely again
      smax = fmaxf(smax, __shfl_xor(smax, 16));
      smax = fmaxf(smax, __shfl_xor(smax, 32));
      if (smax > -INFINITY && (double)smax > mref + PE_REF_SLACK) {      // the same in the four lanes of a row
        const double alpha = exp(mref - (double)smax);                  // (0 the first time: only zeros have been added)
        mref = (double)smax;
        l *= alpha;
#pragma unroll
        for (int n = 0; n < 16; n++)
#pragma unroll
          for (int v = 0; v < 4; v++) O[n][v] *= alpha;
      }
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
      p[v] = valid[v] ? exp(s[v] - mref) : 0.0;
      l += p[v];
    }
    // a key past every row's context has weight 0, but what its slot holds need not be a number: it enters as 0
    if (__builtin_expect(pg * ATT_PAGE + ATT_PAGE > lmax, 0)) {
      const int k0 = pg * ATT_PAGE + 4 * q4;
#pragma unroll
      for (int n = 0; n < 16; n++)
        vr[n] = make_uint2((k0 < lmax ? vr[n].x & 0xffffu : 0u) | (k0 + 1 < lmax ? vr[n].x & 0xffff0000u : 0u),
                           (k0 + 2 < lmax ? vr[n].y & 0xffffu : 0u) | (k0 + 3 < lmax ? vr[n].y & 0xffff0000u : 0u));
    }
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int n = 0; n < 16; n++) {
        const uint32_t w = v < 2 ? vr[n].x : vr[n].y;
        O[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(v & 1 ? pe_hi(w) : pe_lo(w), p[v], O[n], 0, 0, 0);
        if (n % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
  }

  // ---- the waves' partial results: weights exp(ref_w - M) per row, then 64 dims at a time through LDS
  int tl = tid;
  asm volatile("" : "+v"(tl));             // (the rest works out its addresses here: carried across the pages they would have no registers)
  const int c16 = tl & 15, r4 = (tl >> 4) & 3, w4 = tl >> 6;
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (r4 == 0) { lds_m[w4][c16] = mref == ATT_NO_REF ? -INFINITY : mref; lds_l[w4][c16] = l; }
  __syncthreads();                         // (and every wave is done with Q)
  double M = lds_m[0][c16];
#pragma unroll
  for (int w = 1; w < NW; w++) M = fmax(M, lds_m[w][c16]);
  const double f = mref == ATT_NO_REF ? 0.0 : exp(mref - M);
  const int orow = tl >> 4, od = 4 * (tl & 15), ot = t0 + orow / G, head = kvh * G + orow % G;
  double L = 0.0;
  {
    double Mo = lds_m[0][orow];
#pragma unroll
    for (int w = 1; w < NW; w++) Mo = fmax(Mo, lds_m[w][orow]);
#pragma unroll
    for (int w = 0; w < NW; w++) L += lds_l[w][orow] * (lds_m[w][orow] == -INFINITY ? 0.0 : exp(lds_m[w][orow] - Mo));      // (sum of a wave without a reference: 0, or NaN)
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    if (c) __syncthreads();
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int v = 0; v < 4; v++) lds[(w4 * 64 + 16 * n + 4 * v + r4) * PE_PAD + c16] = O[4 * c + n][v] * f;
    __syncthreads();
    if (ot < A.T && (only < 0 || orow / G == only)) {
      uint16_t ob[4];
      uint2 gr = make_uint2(0, 0);
      if (A.gate) {
        const uint16_t* g = A.gate + (int64_t)ot * A.gate_bstride + (int64_t)head * A.gate_hstride + 64 * c + od;
        if (A.wide) gr = *(const uint2*)g;
        else gr = make_uint2((uint32_t)g[0] | ((uint32_t)g[1] << 16), (uint32_t)g[2] | ((uint32_t)g[3] << 16));
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const double* x = lds + (od + i) * PE_PAD + orow;
        double y = x[0];
#pragma unroll
        for (int w = 1; w < NW; w++) y += x[w * 64 * PE_PAD];
        float o = L > 0.0 ? (float)(y / L) : 0.0f;          // no context: zeros
        if (A.gate) o = __fmul_rn(o, sigmoid_f64(bf16_to_f32((uint16_t)((i < 2 ? gr.x : gr.y) >> (16 * (i & 1))))));
        ob[i] = f32_to_bf16(o);
      }
      uint16_t* op = A.out + ((int64_t)ot * A.NH + head) * ATT_HD + 64 * c + od;
      if (A.wide) *(uint2*)op = make_uint2((uint32_t)ob[0] | ((uint32_t)ob[1] << 16), (uint32_t)ob[2] | ((uint32_t)ob[3] << 16));
      else
#pragma unroll
        for (int i = 0; i < 4; i++) op[i] = ob[i];
    }
  }
  }
}

int g_tune_prefill_exact = -1;           // -1 = from the shape, 0 = one launch row per token (attn_exact.hip), 1 = always where it serves

// Groups of 1, 2, 4 or 8 heads (the other form takes any) and enough tokens, against one workgroup per (token, KV head) and range
// of the context, of which a CU holds one (0.054 us a key).
// One range a token (contexts of up to 16384 tokens): from 288 pairs of token and KV head there are two rounds of those workgroups, where
// this kernel takes 0.083 us a key while it has at most a workgroup per CU and 0.075 per workgroup on a CU beyond that.  us, there and
// here, 8 heads a KV head: 288 pairs from empty 48 / 34, behind 16000 tokens 1739 / 1343; 516 pairs behind 15000 2479 / 2226;
// 256 pairs, one round there, behind 1000 90 / 111; groups of 4, 2 and 1 alike (one head: 288 pairs from empty 24.5 / 20.4).
// Several ranges a token: the last round no longer has to be full to be short, and only the work counts, 0.054 us per 256 pairs and key
// there.  384 pairs behind 64000 tokens 5175 / 5257, 448 6030 / 5269; at two workgroups a CU here 704 pairs 9501 / 9628, 768 10374 / 9576;
// three, 1030 pairs 14688 / 14368.  (Below that line prompts that fill little of a long cache would be faster here, 265 / 196
// at 288 pairs behind 2000: how much of it they fill is known on the device alone.)
bool attn_prefill_exact_serves(int T, int NH, int NKV, int HD, int splits) {
  if (HD != ATT_HD || NKV < 1 || NH % NKV) return false;
  const int G = NH / NKV;
  if (G != 1 && G != 2 && G != 4 && G != 8) return false;
  if (g_tune_prefill_exact >= 0) return g_tune_prefill_exact != 0;
  const int64_t pairs = (int64_t)T * NKV;
  if (splits <= 1) return pairs >= 288;
  const int64_t per_cu = ((T + 16 / G - 1) / (16 / G) * (int64_t)NKV + num_cus() - 1) / num_cus();
  return 100 * pairs >= num_cus() * (per_cu == 1 ? 156 : 141 * per_cu);
}

int launch_attn_prefill_exact(const void* q, const void* kc, const void* vc, const int32_t* block_table, const int32_t* pos, int max_ctx,
                              const void* gate, int64_t gate_bstride, int64_t gate_hstride, void* out, int T, int NH, int NKV) {
  BK_REQUIRE(q && kc && vc && block_table && pos && out, "fa2_prefill (exact): null pointer");
  BK_REQUIRE(((uintptr_t)q & 15) == 0 && ((uintptr_t)kc & 15) == 0 && ((uintptr_t)vc & 15) == 0, "fa2_prefill (exact): q, K and V must be 16-byte aligned");
  BK_REQUIRE(T >= 1 && T <= 65535 && NKV >= 1 && max_ctx >= 1 && gate_bstride % 4 == 0 && gate_hstride % 4 == 0, "fa2_prefill (exact): bad shape");
  const int G = NH / NKV, TK = 16 / G;
  const PrefillExactArgs A{(const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, (const uint16_t*)gate, block_table, pos,
                           (uint16_t*)out, gate_bstride, gate_hstride, T, NH, NKV, max_ctx, (T + TK - 1) / TK,
                           (((uintptr_t)gate | (uintptr_t)out) & 7) == 0, 0.0625f};
  const dim3 grid((unsigned)(A.groups * NKV));
  if (G == 8) hipLaunchKernelGGL(attn_prefill_exact_kernel<8>, grid, dim3(256), 0, stream(), A);
  else if (G == 4) hipLaunchKernelGGL(attn_prefill_exact_kernel<4>, grid, dim3(256), 0, stream(), A);
  else if (G == 2) hipLaunchKernelGGL(attn_prefill_exact_kernel<2>, grid, dim3(256), 0, stream(), A);
  else hipLaunchKernelGGL(attn_prefill_exact_kernel<1>, grid, dim3(256), 0, stream(), A);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

}  // namespace bk
