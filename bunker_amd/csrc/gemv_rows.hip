// Q4_K x Q8_1 products of 2 to 7 activation rows (the decode step of a few sequences): the weight rows are read once for
// all of them, and a workgroup prepares the activation rows once for all its weight rows.
//
// What bounds these launches.  One workgroup per (weight rows, sequence), the form this replaces for these batches, repeats
// the RMSNorm / Q8_1 preparation of a row in hundreds of workgroups and unpacks every weight once per sequence: vector
// issue, growing by the whole batch-1 cost with each sequence.  Here the int32 sub-block dots come from the matrix cores
// and the vector work left is the fold in double.  Neither is the bound now: at five rows vector issue takes 26 to 44 % of a launch, the
// matrix pipe 2 to 11 %, and 38 to 55 % of the wave cycles wait in the chain round trip - norm - header unpack - fold - join.
//
// v_mfma_i32_16x16x64_i8 takes 64 elements of K: the two sub-blocks 2g and 2g+1 that share 32 bytes of a Q4_K super-block.
// Its 16 columns are 8 activation rows twice: columns 0..7 hold the rows' sub-block 2g and zeros where the weights have the
// high nibbles, columns 8..15 zeros and sub-block 2g+1.  The result is then the exact dot of one sub-block per lane, for eight activation
// rows and two sub-blocks at once, and no lane folds a column of padding beyond the eighth row.
//   Lane (q4 = lane / 16, col = lane % 8, p = lane / 8 % 2) holds weight rows 4 q4 + v (v = 0..3), activation row col, of the
//   sub-blocks of parity p:   S[v] = sum_g d8[2g+p] * (sc[2g+p] * I),   acc[v] += d * S[v]
// with the arithmetic of the other Q4_K x Q8_1 kernels: every product exact in double, one rounding of the total to f32, so
// the bits are those of the one-row GEMV.  The min term - sum_j dmin m_j s8_j goes through v_mfma_f64_16x16x4_f64 into its own
// accumulators: its result holds row 4 v + q4 where the integer one holds 4 q4 + v, so its weight operand carries the rows in
// that order.
#include "gemv_tile.h"

namespace bk {

typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(4))) double f64x4_t;

enum : int { RPRO_Q8 = 0, RPRO_RMSNORM = 2 };
enum : int { RMODE_PLAIN = 0, RMODE_CONV = 1, RMODE_SWIGLU = 2 };
enum : int { REPI_F32 = 0, REPI_BF16 = 1, REPI_BF16_ADD = 2, REPI_CONV = 3 };

constexpr int ROWS_MAX = 7, RW = 8;            // activation rows; waves per workgroup

struct RowsGroup {
  const uint8_t* W;
  void* out;
  const uint16_t* res;
  int N, epi;
};
struct RowsArgs {
  RowsGroup g[4];
  int first[4];            // first workgroup of each matrix (matrices past the last: the number of workgroups)
  const void* x;           // Q8_1 [B, K/32 blocks] or bf16 [B, K]
  const uint16_t* norm_w;
  int nb, B, xstride;
  uint32_t row_div, xrow_div;      // ceil(2^32 / (9 nb)), ceil(2^32 / (18 nb))
  const uint16_t* conv_st;
  uint16_t* conv_st_new;
  const uint16_t* conv_w;
  uint8_t* out_q8;         // SwiGLU: the result as Q8_1 blocks (then there is no bf16 output)
};
struct RowsArgs1 {         // one matrix: 64 bytes
  RowsGroup g0;
  const void* x;
  int nb, B, tiles, xstride;
};

// LDS: activation rows in the Q8_1 layout, xstride apart (8 dwords past a multiple of 64, so that the sixteen-byte reads of
// eight rows fall into different banks), then 240 zero bytes, then the weight rows, an odd number of 16-byte pieces apart
// (sixteen rows read at the same place fall into different banks).
constexpr int R_ZERO = 240;
__host__ __device__ constexpr int rows_xstride(int nb) { return (nb * 288 + 255) / 256 * 256 + 32; }
__host__ __device__ constexpr int rows_wpieces(int nb) { return (nb * 9) | 1; }

struct RowsX {             // one super-block of the activation rows
  i32x4_t b[4];
  double d[4], s0, s1;
};

struct RowsLane {
  const unsigned char *xl, *xh, *xd, *xs;     // LDS: the two halves of the dots' operand (zeros where the lane has none), d of parity p, s of sub-block q4
  bool low;
  int lane, q4, l16, p;
};
__device__ __forceinline__ RowsLane rows_lane(const unsigned char* xrows, const unsigned char* zeros, int xstride, int B) {
  RowsLane L;
  L.lane = threadIdx.x & 63;
  L.q4 = L.lane >> 4; L.l16 = L.lane & 15; L.p = L.l16 >> 3;
  L.low = L.p == 0;
  const unsigned char* const row = xrows + min(L.l16 & 7, B - 1) * xstride;      // rows past B: row B - 1 again, not stored
  L.xl = L.low ? row + 8 * L.q4 : zeros;
  L.xh = L.low ? zeros : row + 36 + 8 * L.q4;
  L.xd = row + L.p * 36 + 32;
  L.xs = row + L.q4 * 36 + 34;
  return L;
}
__device__ __forceinline__ void rows_load_x(RowsX& x, const RowsLane& L, int blk) {
  const unsigned char* const pl = L.xl + (L.low ? blk * 288 : 0);
  const unsigned char* const ph = L.xh + (L.low ? 0 : blk * 288);
  const unsigned char* const pd = L.xd + blk * 288;
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const uint32_t *l = (const uint32_t*)(pl + 72 * g), *h = (const uint32_t*)(ph + 72 * g);
    x.b[g] = (i32x4_t){(int)l[0], (int)l[1], (int)h[0], (int)h[1]};
    x.d[g] = (double)half_to_f32(*(const uint16_t*)(pd + 72 * g));
  }
  const unsigned char* const ps = L.xs + blk * 288;
  x.s0 = (double)half_to_f32(*(const uint16_t*)ps);
  x.s1 = (double)half_to_f32(*(const uint16_t*)(ps + 144));
}

// What the fold reads of the block headers, unpacked once per workgroup (the eight columns of a row would each do it again:
// 179 vector instructions per super-block and wave, 114 this way): for every (tile, super-block, row) the 6-bit scales of the
// even sub-blocks, those of the odd ones and d, and the products -dmin * m_j (17 bits, exact).
struct RowsScale {
  uint32_t sc[2];
  double d;
};
__device__ __forceinline__ void rows_unpack_header(const uint4& h, RowsScale* __restrict__ sc, float* __restrict__ mins, int i) {
  const uint32_t lo = h.y & 0x3f3f3f3fu, hi = (h.w & 0x0f0f0f0fu) | (((h.y >> 6) & 0x03030303u) << 4);
  const uint32_t ml = h.z & 0x3f3f3f3fu, mh = ((h.w >> 4) & 0x0f0f0f0fu) | (((h.z >> 6) & 0x03030303u) << 4);
  RowsScale r;
  r.sc[0] = __builtin_amdgcn_perm(hi, lo, 0x06040200u);
  r.sc[1] = __builtin_amdgcn_perm(hi, lo, 0x07050301u);
  r.d = (double)half_to_f32((uint16_t)(h.x & 0xffffu));
  sc[i] = r;
  const float dmin_neg = -half_to_f32((uint16_t)(h.x >> 16));
  float* const m = mins + (i >> 4) * 128 + (i & 15);        // [tile, super-block][8 sub-blocks][16 rows]
#pragma unroll
  for (int j = 0; j < 8; j++) m[16 * j] = dmin_neg * (float)(((j < 4 ? ml : mh) >> (8 * (j & 3))) & 0xffu);
}

// One super-block of 16 weight rows: `w` points at it in the tile's first row, rows are wstride bytes apart; `ti` counts
// (tile, super-block).
__device__ __forceinline__ void rows_fold(f64x4_t& acc, f64x4_t& accm, const unsigned char* w, int wstride, const RowsScale* sct, const float* mins,
                                          int ti, const RowsX& x, const RowsLane& L) {
  const unsigned char* const wr = w + L.l16 * wstride + 16 + 8 * L.q4;
  i32x4_t c[4];
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const uint2 q = *(const uint2*)(wr + 32 * g);
    const i32x4_t a = {(int)(q.x & 0x0f0f0f0fu), (int)(q.y & 0x0f0f0f0fu), (int)((q.x >> 4) & 0x0f0f0f0fu), (int)((q.y >> 4) & 0x0f0f0f0fu)};
    c[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, x.b[g], (i32x4_t){0, 0, 0, 0}, 0, 0, 0);
  }
  const float* const m = mins + ti * 128 + 16 * L.q4 + 4 * (L.l16 & 3) + (L.l16 >> 2);
  accm = __builtin_amdgcn_mfma_f64_16x16x4f64((double)m[0], x.s0, accm, 0, 0, 0);
  accm = __builtin_amdgcn_mfma_f64_16x16x4f64((double)m[64], x.s1, accm, 0, 0, 0);
  const RowsScale* const sc = sct + ti * 16 + 4 * L.q4;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const uint32_t k = sc[v].sc[L.p];
    double S = x.d[0] * (double)__mul24(c[0][v], (int)(k & 0xffu));
    S = fma(x.d[1], (double)__mul24(c[1][v], (int)((k >> 8) & 0xffu)), S);
    S = fma(x.d[2], (double)__mul24(c[2][v], (int)((k >> 16) & 0xffu)), S);
    S = fma(x.d[3], (double)__mul24(c[3][v], (int)(k >> 24)), S);
    acc[v] = fma(sc[v].d, S, acc[v]);
  }
}

// columns col and col + 8 hold the two halves of one activation row's first sum, and each its whole min term
__device__ __forceinline__ void rows_join(f64x4_t& acc, const f64x4_t& accm) {
#pragma unroll
  for (int v = 0; v < 4; v++) acc[v] = (acc[v] + dpp_f64<0x128>(acc[v])) + accm[v];      // row_ror:8
}

// The matrix of a workgroup (wave-uniform).  Every matrix starts a workgroup of its own.
struct RowsSel {
  const uint8_t* W;
  void* out;
  const uint16_t* res;
  int N, epi, n0;
};
template <int ROWS>
__device__ __forceinline__ RowsSel rows_matrix(const RowsArgs& A, int wg) {
  const bool s1 = wg >= A.first[1], s2 = wg >= A.first[2], s3 = wg >= A.first[3];
  RowsSel r;
  r.W = s3 ? A.g[3].W : s2 ? A.g[2].W : s1 ? A.g[1].W : A.g[0].W;
  r.out = s3 ? A.g[3].out : s2 ? A.g[2].out : s1 ? A.g[1].out : A.g[0].out;
  r.res = s3 ? A.g[3].res : s2 ? A.g[2].res : s1 ? A.g[1].res : A.g[0].res;
  r.N = s3 ? A.g[3].N : s2 ? A.g[2].N : s1 ? A.g[1].N : A.g[0].N;
  r.epi = s3 ? A.g[3].epi : s2 ? A.g[2].epi : s1 ? A.g[1].epi : A.g[0].epi;
  r.n0 = ROWS * (wg - (s3 ? A.first[3] : s2 ? A.first[2] : s1 ? A.first[1] : 0));
  return r;
}

__device__ __forceinline__ void rows_store(void* out, const uint16_t* res, int epi, int64_t o, float v) {
  if (epi == REPI_F32) store_out<EPI_F32>(out, res, o, v);
  else if (epi == REPI_BF16) store_out<EPI_BF16>(out, res, o, v);
  else store_out<EPI_BF16_ADD>(out, res, o, v);
}

// Loads go through buffer resources: what lies past the end is not fetched and reads as zero (weights that are not stored anywhere),
// with nothing to clamp.  The range check covers the lane's offset and not the instruction's scalar offset, so the whole offset is
// the lane's: requests past the end are common (the last workgroup of a matrix, rows shorter than KP).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00027000);
}
template <int AUX>
__device__ __forceinline__ uint4 rows_load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, AUX));
}
constexpr int AUX_NT = 2;

// Q8_1 rows as given -> LDS, 16 bytes a piece.  NP: pieces per thread (requested together).
template <int NP>
struct RowsCopy {
  uint4 v[NP];
};
template <int NP>
__device__ __forceinline__ void rows_copy_load(RowsCopy<NP>& c, const void* xq, int pieces) {
  const __amdgpu_buffer_rsrc_t r = rows_rsrc(xq, pieces * 16);
#pragma unroll
  for (int i = 0; i < NP; i++) c.v[i] = rows_load16<0>(r, threadIdx.x * 16 + 64 * RW * 16 * i);
}
// row_div: ceil(2^32 / pieces per row), so that the high half of p * row_div is p / (pieces per row)
template <int NP>
__device__ __forceinline__ void rows_copy_park(const RowsCopy<NP>& c, unsigned char* xrows, int row_pieces, uint32_t row_div, int pieces, int xstride) {
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int p = threadIdx.x + 64 * RW * i, row = (int)__umulhi((uint32_t)p, row_div);
    if (p < pieces) *(uint4*)(xrows + row * (xstride - row_pieces * 16) + p * 16) = c.v[i];
  }
}

// RMSNorm -> bf16 -> Q8_1 of up to seven rows of KP elements: KP / 8 threads per row, 4096 / KP rows at a time, the sums of
// squares of all of them in front of one barrier.  Operation for operation (and lane for lane) glue.hip's rmsnorm_kernel.
template <int KP>
struct RowsNorm {
  static constexpr int TPR = KP / 8, RPP = 64 * RW / TPR, PASSES = (ROWS_MAX + RPP - 1) / RPP;
  uint4 xv[PASSES], wv;
};
template <int KP>
__device__ __forceinline__ void rows_norm_load(RowsNorm<KP>& r, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int B) {
  constexpr int TPR = RowsNorm<KP>::TPR;
  const int i = (threadIdx.x % TPR) * 8;
  r.wv = *(const uint4*)(w + i);
#pragma unroll
  for (int p = 0; p < RowsNorm<KP>::PASSES; p++)
    r.xv[p] = *(const uint4*)(x + (int64_t)min(p * RowsNorm<KP>::RPP + (int)threadIdx.x / TPR, B - 1) * KP + i);
}
template <int KP>
__device__ __forceinline__ void rows_norm_stage(const RowsNorm<KP>& r, unsigned char* xrows, int xstride, double* red, int B) {
  constexpr int TPR = RowsNorm<KP>::TPR, RPP = RowsNorm<KP>::RPP, PASSES = RowsNorm<KP>::PASSES, WPR = TPR / 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = (threadIdx.x % TPR) * 8, rsub = wave / WPR;
#pragma unroll
  for (int p = 0; p < PASSES; p++) {
    if (p * RPP + rsub < B) {
      const uint32_t u[4] = {r.xv[p].x, r.xv[p].y, r.xv[p].z, r.xv[p].w};
      double ss = 0.0;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float a = __uint_as_float(u[j] << 16), b = __uint_as_float(u[j] & 0xffff0000u);
        ss += (double)(a * a) + (double)(b * b);
      }
      ss = wave_sum_f64(ss);
      if ((threadIdx.x & 63) == 0) red[p * RW + wave] = ss;
    }
  }
  __syncthreads();
  const uint32_t uw[4] = {r.wv.x, r.wv.y, r.wv.z, r.wv.w};
#pragma unroll
  for (int p = 0; p < PASSES; p++) {
    const int row = p * RPP + rsub;
    if (row < B) {
      double ss = 0.0;
#pragma unroll
      for (int k = 0; k < WPR; k++) ss += red[p * RW + rsub * WPR + k];
      const float rstd = rsqrt_f64(ss / (double)KP + 1e-6);
      const uint32_t u[4] = {r.xv[p].x, r.xv[p].y, r.xv[p].z, r.xv[p].w};
      float f[8];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float a = __uint_as_float(u[j] << 16), b = __uint_as_float(u[j] & 0xffff0000u);
        const float wa = __uint_as_float(uw[j] << 16), wb = __uint_as_float(uw[j] & 0xffff0000u);
        f[2 * j] = bf16_to_f32(f32_to_bf16(__fmul_rn(__fmul_rn(a, rstd), __fadd_rn(1.0f, wa))));
        f[2 * j + 1] = bf16_to_f32(f32_to_bf16(__fmul_rn(__fmul_rn(b, rstd), __fadd_rn(1.0f, wb))));
      }
      uint32_t pk[2];
      const uint32_t ds = quad_q8_1(f, pk);
      unsigned char* ob = xrows + row * xstride + (i / 32) * 36;
      uint32_t* oq = (uint32_t*)(ob + (i & 31));
      oq[0] = pk[0]; oq[1] = pk[1];
      if ((i & 31) == 0) *(uint32_t*)(ob + 32) = ds;
    }
  }
}

// A workgroup owns SLOTS = RW / WPT * TPG tiles of 16 weight rows.  Their rows are contiguous in memory: every 128-byte line is
// requested once, all of them before the activation rows are prepared, and parked in LDS behind that.  (Operands loaded
// straight from memory, a row per lane, touch every line from several instructions: SwiGLU of 12288 x 2048 at four rows
// 13.4 us against 11.7, 15.5 with nontemporal loads.)  WPT waves split the super-blocks of a tile (wave w takes w, w + WPT, ...), each for TPG
// tiles.  The partial sums meet in LDS, in wave order.  SwiGLU: four slots = gate rows r..r+31, up rows r..r+31.
//   KP: the row length, for Q8_1 rows the largest.
template <int PRO, int KP, int MODE, int WPT, int TPG>
__global__ __launch_bounds__(64 * RW, TPG > 1 || KP > 2048 ? 2 : 4) void gemv_rows_kernel(RowsArgs A) {
  constexpr int NG = RW / WPT, SLOTS = NG * TPG;
  constexpr bool FIXED = PRO == RPRO_RMSNORM;        // the row length is known here
  static_assert(MODE != RMODE_SWIGLU || SLOTS == 4, "SwiGLU: 32 rows of gate and up");
  static_assert(MODE != RMODE_CONV || SLOTS * 128 <= 64 * RW, "conv: one output per thread");
  constexpr int NBX = KP / 256, XBYTES = ROWS_MAX * rows_xstride(NBX), WBYTES = SLOTS * 16 * rows_wpieces(NBX) * 16;
  constexpr int WLOADS = (SLOTS * 16 * NBX * 9 + 64 * RW - 1) / (64 * RW);
  __shared__ __align__(16) unsigned char lds_rows[XBYTES + R_ZERO + WBYTES];
  __shared__ __align__(16) double part[SLOTS * WPT * 128];
  __shared__ RowsScale sct[SLOTS * NBX * 16];
  __shared__ float mins[SLOTS * NBX * 128];
  static_assert(SLOTS * NBX * 16 <= 64 * RW, "a header per thread");
  __shared__ double red[FIXED ? RowsNorm<FIXED ? KP : 2048>::PASSES * RW : 1];
  unsigned char* const xrows = lds_rows;
  unsigned char* const zeros = lds_rows + XBYTES;
  unsigned char* const wrows = zeros + R_ZERO;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int gi = wave / WPT, kw = wave % WPT;
  const int nb = FIXED ? NBX : A.nb, rp = nb * 9, wstride = rows_wpieces(nb) * 16;
  const int xstride = FIXED ? rows_xstride(NBX) : A.xstride;
  const RowsLane L = rows_lane(xrows, zeros, xstride, A.B);

  [[maybe_unused]] RowsNorm<FIXED ? KP : 2048> nr;
  [[maybe_unused]] RowsCopy<(ROWS_MAX * NBX * 18 + 64 * RW - 1) / (64 * RW)> cp;
  if constexpr (FIXED) rows_norm_load<FIXED ? KP : 2048>(nr, (const uint16_t*)A.x, A.norm_w, A.B);
  else rows_copy_load(cp, A.x, A.B * nb * 18);

  // the convolution's operands of this thread's output
  [[maybe_unused]] uint16_t cs0 = 0, cs1 = 0, cs2 = 0;
  [[maybe_unused]] uint2 cw = make_uint2(0, 0);
  const int slot_t = threadIdx.x >> 7, col_t = (threadIdx.x >> 4) & 7, row_t = threadIdx.x & 15;
  if constexpr (MODE == RMODE_CONV) {
    const int C = A.g[0].N, ch = min((int)((blockIdx.x * SLOTS + slot_t) * 16 + row_t), C - 1);      // other matrices' workgroups: any channel
    const uint16_t* sb = A.conv_st + (int64_t)min(col_t, A.B - 1) * 3 * C;
    cs0 = sb[ch]; cs1 = sb[C + ch]; cs2 = sb[2 * C + ch];
    cw = *(const uint2*)(A.conv_w + 4 * (int64_t)ch);
  }

  // weight rows: SLOTS * 16 * rp pieces, one run of memory, or one of the gate matrix and one of the up matrix
  RowsSel M;
  if (MODE == RMODE_SWIGLU) { M.W = A.g[0].W; M.N = A.g[0].N; M.n0 = blockIdx.x * 32; }
  else M = rows_matrix<SLOTS * 16>(A, blockIdx.x);
  uint4 wreg[WLOADS];
  {
    constexpr int RUN = SLOTS * 8 * NBX * 9;          // SwiGLU: pieces of either matrix
    static_assert(MODE != RMODE_SWIGLU || RUN % 64 == 0, "a wave's pieces belong to one matrix");
    const int64_t at = (int64_t)M.n0 * rp * 16;
    const int bytes = min(MODE == RMODE_SWIGLU ? 32 : SLOTS * 16, M.N - M.n0) * rp * 16;
#pragma unroll
    for (int i = 0; i < WLOADS; i++) {
      const int p = wave * 64 + 64 * RW * i;
      const bool up = MODE == RMODE_SWIGLU && p >= RUN;
      wreg[i] = rows_load16<AUX_NT>(rows_rsrc((up ? A.g[1].W : M.W) + at, bytes), L.lane * 16 + (up ? p - RUN : p) * 16);
    }
  }
  const int tp = 16 * rp;
  if (threadIdx.x < R_ZERO / 4) ((uint32_t*)zeros)[threadIdx.x] = 0;
  if constexpr (FIXED) rows_norm_stage<FIXED ? KP : 2048>(nr, xrows, xstride, red, A.B);
  else rows_copy_park(cp, xrows, nb * 18, A.xrow_div, A.B * nb * 18, xstride);
#pragma unroll
  for (int i = 0; i < WLOADS; i++) {
    const int p = threadIdx.x + 64 * RW * i;
    const int row = FIXED ? p / (NBX * 9) : (int)__umulhi((uint32_t)p, A.row_div);      // counted over all slots
    if (p < SLOTS * tp) *(uint4*)(wrows + row * (wstride - rp * 16) + p * 16) = wreg[i];
  }
  __syncthreads();
  if ((int)threadIdx.x < SLOTS * nb * 16) {      // this thread's header: (tile, super-block) ti, row threadIdx % 16
    const int ti = threadIdx.x >> 4, tile = FIXED ? ti / NBX : (SLOTS > 1 && ti >= nb ? 1 : 0);
    rows_unpack_header(*(const uint4*)(wrows + (tile * 16 + (threadIdx.x & 15)) * wstride + (ti - tile * nb) * 144), sct, mins, threadIdx.x);
  }
  __syncthreads();

  auto leave = [&](int t, f64x4_t& acc, const f64x4_t& accm) {
    rows_join(acc, accm);
    if (L.low) {
      double2* p = (double2*)(part + ((gi * TPG + t) * WPT + kw) * 128 + L.l16 * 16 + 4 * L.q4);
      p[0] = make_double2(acc[0], acc[1]);
      p[1] = make_double2(acc[2], acc[3]);
    }
  };
  if constexpr (FIXED) {
    static_assert(!FIXED || NBX == WPT, "a super-block per wave and tile");
    RowsX x;
    rows_load_x(x, L, kw);
#pragma unroll
    for (int t = 0; t < TPG; t++) {
      f64x4_t acc = {0.0, 0.0, 0.0, 0.0}, accm = acc;
      rows_fold(acc, accm, wrows + (gi * TPG + t) * 16 * wstride + kw * 144, wstride, sct, mins, (gi * TPG + t) * NBX + kw, x, L);
      leave(t, acc, accm);
    }
  } else {
    static_assert(FIXED || TPG == 1, "one tile per wave");
    f64x4_t acc = {0.0, 0.0, 0.0, 0.0}, accm = acc;
    for (int blk = kw; blk < nb; blk += WPT) {
      RowsX x;
      rows_load_x(x, L, blk);
      rows_fold(acc, accm, wrows + gi * 16 * wstride + blk * 144, wstride, sct, mins, gi * nb + blk, x, L);
    }
    leave(0, acc, accm);
  }
  __syncthreads();
  auto total = [&](int slot, int e) {
    const double* p = part + slot * WPT * 128 + e;
    double t = p[0];
#pragma unroll
    for (int w = 1; w < WPT; w++) t += p[w * 128];
    return (float)t;
  };

  if constexpr (MODE == RMODE_SWIGLU) {
    if (threadIdx.x >= 256) return;
    const int col = threadIdx.x >> 5, r = threadIdx.x & 31, e = col * 16 + (r & 15), N = A.g[0].N;
    const float g = total(r >> 4, e), v = total(2 + (r >> 4), e);
    const uint16_t a = f32_to_bf16(__fmul_rn(__fmul_rn(g, sigmoid_f64(g)), v));
    const int row = blockIdx.x * 32 + r;
    if (A.out_q8) lane32_q8_1_store(bf16_to_f32(a), A.out_q8 + ((int64_t)col * (N / 32) + blockIdx.x) * 36, r, col < A.B);
    else if (col < A.B && row < N) ((uint16_t*)A.g[0].out)[(int64_t)col * N + row] = a;
  } else {
    static_assert(SLOTS * 128 <= 64 * RW, "an output per thread");
    const int row = M.n0 + 16 * slot_t + row_t, N = M.N;
    if (slot_t < SLOTS && col_t < A.B && row < N) {
      const float y = total(slot_t, col_t * 16 + row_t);
      const int64_t o = (int64_t)col_t * N + row;
      if (MODE == RMODE_CONV && M.epi == REPI_CONV) {
        // 4-tap causal convolution + SiLU of this channel and its new state rows (src/emitters.ts:48-72), as gemv_fused does it
        const uint16_t xb = f32_to_bf16(y);
        const float w0 = __uint_as_float(cw.x << 16), w1 = __uint_as_float(cw.x & 0xffff0000u);
        const float w2 = __uint_as_float(cw.y << 16), w3 = __uint_as_float(cw.y & 0xffff0000u);
        const float rr = __fadd_rn(__fadd_rn(w0 * bf16_to_f32(cs0), w1 * bf16_to_f32(cs1)),
                                   __fadd_rn(w2 * bf16_to_f32(cs2), w3 * bf16_to_f32(xb)));
        uint16_t* nbuf = A.conv_st_new + (int64_t)col_t * 3 * N;
        nbuf[row] = cs1; nbuf[N + row] = cs2; nbuf[2 * N + row] = xb;
        ((uint16_t*)M.out)[o] = f32_to_bf16(__fmul_rn(rr, sigmoid_f64(rr)));
      } else {
        rows_store(M.out, M.res, M.epi, o, y);
      }
    }
  }
}

// One matrix whose tiles alone fill the chip many times over (lm_head): a workgroup walks pairs of tiles, the next pair's rows
// on their way during the arithmetic of this one (registers, then the other half of the LDS buffer).
template <int NB>
__global__ __launch_bounds__(64 * RW, 2) void gemv_rows_stream_kernel(RowsArgs1 A) {
  constexpr int WPT = NB, NG = RW / NB, SLOTS = 2 * NG, TPG = 2, RP = NB * 9, TP = 16 * RP, WS = rows_wpieces(NB) * 16;
  static_assert(NB == 4 || NB == 8, "rows of 1024 or 2048");
  constexpr int XS = rows_xstride(NB), XBYTES = ROWS_MAX * XS, WBYTES = SLOTS * 16 * WS, WLOADS = (SLOTS * TP + 64 * RW - 1) / (64 * RW);
  __shared__ __align__(16) unsigned char lds_rows[XBYTES + R_ZERO + 2 * WBYTES];
  __shared__ __align__(16) double part[SLOTS * WPT * 128];
  __shared__ RowsScale sct[SLOTS * NB * 16];
  __shared__ float mins[SLOTS * NB * 128];
  static_assert(SLOTS * NB * 16 <= 64 * RW, "a header per thread");
  unsigned char* const zeros = lds_rows + XBYTES;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), gi = wave / WPT, kw = wave % WPT;
  const int N = A.g0.N, pieces = A.B * NB * 18;
  const RowsLane L = rows_lane(lds_rows, zeros, XS, A.B);
  RowsCopy<(ROWS_MAX * NB * 18 + 64 * RW - 1) / (64 * RW)> cp;
  rows_copy_load(cp, A.x, pieces);
  uint4 wreg[WLOADS];
  const int ti = threadIdx.x >> 4;
  auto request = [&](int chunk) {
    const int n0 = chunk * SLOTS * 16;
    const __amdgpu_buffer_rsrc_t r = rows_rsrc(A.g0.W + (int64_t)n0 * (NB * 144), min(SLOTS * 16, N - n0) * (NB * 144));
#pragma unroll
    for (int i = 0; i < WLOADS; i++) wreg[i] = rows_load16<AUX_NT>(r, threadIdx.x * 16 + 64 * RW * 16 * i);
  };
  int chunk = blockIdx.x;
  const int chunks = (A.tiles + SLOTS - 1) / SLOTS;
  request(chunk);
  if (threadIdx.x < R_ZERO / 4) ((uint32_t*)zeros)[threadIdx.x] = 0;
  rows_copy_park(cp, lds_rows, NB * 18, (uint32_t)((0x100000000ull + NB * 18 - 1) / (NB * 18)), pieces, XS);
  __syncthreads();
  RowsX x;
  rows_load_x(x, L, kw);                         // a super-block per wave: the same one for every tile
  for (int it = 0; chunk < chunks; it ^= 1, chunk += gridDim.x) {
    unsigned char* const wrows = zeros + R_ZERO + it * WBYTES;
#pragma unroll
    for (int i = 0; i < WLOADS; i++) {
      const int p = threadIdx.x + 64 * RW * i, row = p / RP;
      if (p < SLOTS * TP) *(uint4*)(wrows + row * (WS - RP * 16) + p * 16) = wreg[i];
    }
    if (chunk + (int)gridDim.x < chunks) request(chunk + gridDim.x);
    __syncthreads();
    if (threadIdx.x < SLOTS * NB * 16)
      rows_unpack_header(*(const uint4*)(wrows + (ti / NB * 16 + (threadIdx.x & 15)) * WS + ti % NB * 144), sct, mins, threadIdx.x);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TPG; t++) {
      f64x4_t acc = {0.0, 0.0, 0.0, 0.0}, accm = acc;
      rows_fold(acc, accm, wrows + (gi * TPG + t) * 16 * WS + kw * 144, WS, sct, mins, (gi * TPG + t) * NB + kw, x, L);
      rows_join(acc, accm);
      if (L.low) {
        double2* p = (double2*)(part + ((gi * TPG + t) * WPT + kw) * 128 + L.l16 * 16 + 4 * L.q4);
        p[0] = make_double2(acc[0], acc[1]);
        p[1] = make_double2(acc[2], acc[3]);
      }
    }
    __syncthreads();
    // 16 SLOTS consecutive rows of each activation row, along the threads
    for (int e = threadIdx.x; e < SLOTS * 128; e += 64 * RW) {
      const int r = e % (16 * SLOTS), col = e / (16 * SLOTS), row = chunk * 16 * SLOTS + r;
      const double* p = part + (r >> 4) * WPT * 128 + col * 16 + (r & 15);
      double t = p[0];
#pragma unroll
      for (int w = 1; w < WPT; w++) t += p[w * 128];
      if (col < A.B && row < N) rows_store(A.g0.out, A.g0.res, A.g0.epi, (int64_t)col * N + row, (float)t);
    }
  }
}

int g_tune_rows = 1;      // 0: these launches take the one-row forms, 1: gemv_rows_pays decides, 2: gemv_rows wherever it serves

bool gemv_rows_serves(int pro, int K, int batch, int ngroups, bool swiglu) {
  if (batch < 2 || batch > ROWS_MAX) return false;
  if (pro == RPRO_RMSNORM) return K == 1024 || K == 2048;
  return pro == RPRO_Q8 && !swiglu && ngroups == 1 && K >= 1024 && K <= 6144 && K % 512 == 0;
}

// Whether a served launch takes less time here than in the one-row forms; `rows`: weight rows of all its matrices.
// One-row forms (gemv_fused; gemv for the lengths that it has no kernel for) cost about 3 us and then grow with rows * batch.
// Here the batch costs little, but a launch starts later (a workgroup stages its weights, unpacks their headers and prepares
// every activation row before the first product) and, where only one workgroup fits a CU (KP = 6144: 131 KB of LDS, K = 2048 with
// the norm: 115), grows in whole rounds of the chip.  Measured on cold weights over 512 to 248320 rows and 2 to 7 sequences
// (one-row form -> here, us; the lines below lie where the two meet, no measured launch is sent to a form 10 % slower):
//   norm, K = 1024: 2048 rows x 5 5.0 -> 5.3, 5120 x 2 5.6 -> 4.6, 9216 x 7 16.9 -> 8.4; SwiGLU of 1024 x 7 6.5 -> 7.0, 3584 x 2 6.9 -> 5.8
//   norm, K = 2048: 5120 rows x 2 5.9 -> 6.3, 9216 x 2 8.2 -> 7.7, two rounds: 18432 x 2 10.9 -> 13.9, x 4 18.1 -> 16.0;
//                   SwiGLU of 6144 x 2 8.7 -> 9.2, x 3 12.1 -> 9.5
//   Q8_1 rows, K = 1024: 2048 x 4 3.4 -> 3.8, x 7 4.3 -> 4.0; K = 1536: 4096 x 3 4.0 -> 4.8, x 5 5.8 -> 5.0;
//              K = 2048: 8192 x 2 5.2 -> 5.5, 4096 x 4 4.9 -> 4.2; K = 4096: 1024 x 7 4.9 -> 5.2, 2048 x 5 6.0 -> 5.4, 12288 x 2 13.1 -> 15.1,
//              x 3 18.1 -> 15.2; K = 6144: 2048 x 2 4.9 -> 6.2, x 4 7.8 -> 6.2; K = 3072: 49152 x 2 38.8 -> 44.9, x 3 55.8 -> 46.0
bool gemv_rows_pays(int pro, int K, int batch, int64_t rows, bool swiglu) {
  const int64_t work = rows * batch;
  const auto rounds = [&](int64_t rows_per_wg) { return (rows + rows_per_wg * num_cus() - 1) / (rows_per_wg * num_cus()); };
  if (pro == RPRO_RMSNORM) {
    if (K == 1024) return work >= (swiglu ? 8000 + 1500 * batch : 6500 + 1000 * batch);
    if (swiglu && batch == 2) return false;
    const int64_t r = rounds(swiglu ? 64 : 48);
    return work >= (r > 1 ? 34000 * r : swiglu ? 14000 + 2200 * batch : 9000 + 1800 * batch);
  }
  if (K <= 2048) {
    if (batch == 2 && K > 1024) return work >= 32768;
    return work >= (K == 1536 ? 16000 : 6500 + 1000 * batch);        // six super-blocks occupy four waves twice
  }
  const int64_t r = rounds(16);
  if (gemv_fused_fast_path(K, batch, false)) return r == 1 ? work >= (K <= 4096 ? 8448 : 6656) : batch >= 3 && work >= 8192 * r;
  return r == 1 || batch >= 3 || K >= 4608;
}

template <int PRO, int KP, int MODE, int TPG>
static void launch_rows_one(int ngroups, RowsArgs& A) {
  constexpr int WPT = KP >= 2048 ? 8 : 4, ROWS = MODE == RMODE_SWIGLU ? 32 : 16 * RW / WPT * TPG;
  int wgs = 0;
  for (int i = 0; i < 4; i++) {
    A.first[i] = wgs;
    if (i < (MODE == RMODE_SWIGLU ? 1 : ngroups)) wgs += (A.g[i].N + ROWS - 1) / ROWS;
  }
  hipLaunchKernelGGL((gemv_rows_kernel<PRO, KP, MODE, WPT, TPG>), dim3(wgs), dim3(64 * RW), 0, stream(), A);
}
template <int KP>
static void launch_rows_norm(int mode, int ngroups, int tiles, RowsArgs& A) {
  // K = 2048: three tiles a workgroup where two would give some CUs a second workgroup, which then decides the time
  // (8192 + 512 + 512 rows at four sequences 11.8 us with two, 8.9 with three)
  constexpr int T1 = KP == 2048 ? 2 : 1, T2 = KP == 2048 ? 3 : 1;
  const bool three = T2 != T1 && tiles > 2 * num_cus();
  if (mode == RMODE_SWIGLU) launch_rows_one<RPRO_RMSNORM, KP, RMODE_SWIGLU, KP == 2048 ? 4 : 2>(ngroups, A);
  else if (mode == RMODE_CONV && three) launch_rows_one<RPRO_RMSNORM, KP, RMODE_CONV, T2>(ngroups, A);
  else if (mode == RMODE_CONV) launch_rows_one<RPRO_RMSNORM, KP, RMODE_CONV, T1>(ngroups, A);
  else if (three) launch_rows_one<RPRO_RMSNORM, KP, RMODE_PLAIN, T2>(ngroups, A);
  else launch_rows_one<RPRO_RMSNORM, KP, RMODE_PLAIN, T1>(ngroups, A);
}

int launch_gemv_rows(int pro, const void* x, const void* norm_w, int K, int batch, int ngroups, const void* const* W,
                     void* const* out, const void* const* res, const int* N, const int* epi, bool swiglu, const FusedConv* conv,
                     void* out_q8) {
  BK_REQUIRE(gemv_rows_serves(pro, K, batch, ngroups, swiglu), "gemv_rows: pro=%d K=%d batch=%d is not served", pro, K, batch);
  BK_REQUIRE(x && (pro != RPRO_RMSNORM || norm_w) && ((uintptr_t)x & 15) == 0 && ((uintptr_t)norm_w & 15) == 0,
             "gemv_rows: activation and norm weight must be given and 16-byte aligned");
  BK_REQUIRE(ngroups >= 1 && ngroups <= 4 && (!swiglu || ngroups == 2), "gemv_rows: bad number of matrices %d", ngroups);
  BK_REQUIRE(!out_q8 || (swiglu && N[0] % 32 == 0), "gemv_rows: the Q8_1 result exists for SwiGLU with N a multiple of 32");
  RowsArgs A{};
  A.x = x; A.norm_w = (const uint16_t*)norm_w; A.nb = K / 256; A.B = batch; A.xstride = rows_xstride(A.nb); A.out_q8 = (uint8_t*)out_q8;
  int tiles = 0;
  for (int i = 0; i < 4; i++) {
    const int j = i < ngroups ? i : ngroups - 1;
    BK_REQUIRE(W[j] && N[j] > 0 && ((uintptr_t)W[j] & 15) == 0, "gemv_rows: matrix %d: null, misaligned or N <= 0", j);
    A.g[i].W = (const uint8_t*)W[j]; A.g[i].N = N[j];
    if (swiglu) {
      BK_REQUIRE(N[j] == N[0] && (out[0] || out_q8), "gemv_rows: gate and up must have the same number of rows, and an output");
      A.g[i].out = out[0];
      continue;
    }
    BK_REQUIRE(out[j] && (epi[j] == REPI_F32 || epi[j] == REPI_BF16 || (epi[j] == REPI_BF16_ADD && res[j]) || (epi[j] == REPI_CONV && j == 0 && conv)),
               "gemv_rows: matrix %d: no output, bad epilogue %d or no residual", j, epi[j]);
    A.g[i].out = out[j]; A.g[i].res = (const uint16_t*)res[j]; A.g[i].epi = epi[j];
    if (i < ngroups) tiles += (N[j] + 15) / 16;
  }
  if (conv) {
    BK_REQUIRE(conv->st && conv->st_new && conv->w && ((uintptr_t)conv->w & 7) == 0 && pro == RPRO_RMSNORM && !swiglu, "gemv_rows: bad conv operands");
    A.conv_st = (const uint16_t*)conv->st; A.conv_st_new = (uint16_t*)conv->st_new; A.conv_w = (const uint16_t*)conv->w;
  }
  A.row_div = (uint32_t)((0x100000000ull + A.nb * 9 - 1) / (A.nb * 9));
  A.xrow_div = (uint32_t)((0x100000000ull + A.nb * 18 - 1) / (A.nb * 18));
  const int mode = swiglu ? RMODE_SWIGLU : conv ? RMODE_CONV : RMODE_PLAIN;
  if (pro == RPRO_RMSNORM) {
    if (K == 1024) launch_rows_norm<1024>(mode, ngroups, tiles, A);
    else launch_rows_norm<2048>(mode, ngroups, tiles, A);
  } else if (tiles >= 8 * num_cus() && (K == 1024 || K == 2048)) {
    const RowsArgs1 P{A.g[0], A.x, A.nb, A.B, tiles, A.xstride};
    if (K == 1024) hipLaunchKernelGGL((gemv_rows_stream_kernel<4>), dim3(num_cus()), dim3(64 * RW), 0, stream(), P);
    else hipLaunchKernelGGL((gemv_rows_stream_kernel<8>), dim3(num_cus()), dim3(64 * RW), 0, stream(), P);
  } else if (K < 2048) launch_rows_one<RPRO_Q8, 1536, RMODE_PLAIN, 1>(1, A);
  else if (K == 2048) launch_rows_one<RPRO_Q8, 2048, RMODE_PLAIN, 1>(1, A);
  else launch_rows_one<RPRO_Q8, 6144, RMODE_PLAIN, 1>(1, A);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

}  // namespace bk
