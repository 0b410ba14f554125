// Batched decode matmul: C[B, N] = Xq[B, K] . W[N, K]^T for tiles of up to 32 activation rows in
// Q8_1 and W in Q4_K, on the int8 matrix cores.  Precedent in the reference:
// int8MatmulTTIR (src/kernel.ts:397-417), i8 x i8 -> i32 exact, and its documented
// post-scale (experiments/q4k_q81_final.ts:214-217).
//
// One v_mfma_i32_32x32x32_i8 consumes exactly one 32-element sub-block of K for a tile
// of 32 weight rows (M) x 32 activation rows (N), so the matrix core produces the exact
// int32 sub-block dots I_j[n, b].  A lane owns activation row b = lane % 32 and 16 of the 32
// weight rows; it folds the dots with the scales in double, in the same way the GEMV does
// (every term exact, ~1e-16 accumulation error, one rounding to f32), so the batched
// path returns the same bits as the batch-1 path:
//   y[b, n] = sum_blk ( d * sum_j d8_j[b] * (sc_j * I_j) - dmin * sum_j m_j * s8_j[b] )
// The first sum is folded on the vector unit: per dot one 24-bit integer multiply by the 6-bit scale (a byte the
// lane's 16 rows share with its half of the wave, fetched from LDS 16 at a time) and one 64-bit integer multiply-add with
// the lane's own activation scale, a whole number of 2^-24; d comes in once per super-block.  (With the sum in double the dot
// took a conversion and an FMA, 4.4 ns of a SIMD against 2.6 for v_mad_i64_i32: 77 rows x 12288 x 2048 25.2 -> 24.3 us, a
// prompt of 2048 tokens 31.1 -> 30.3 ms.)  The second sum is a small dense product over
// the sub-blocks of K and runs on the double-precision matrix instruction (v_mfma_f64_16x16x4_f64), in its own
// accumulators that join the others once, at the end.
//
// Batches of more than 32 rows are cut into 32-row tiles (one launch, every (weight tile, batch tile) its own workgroup).
// A workgroup owns one 32 x 32 output tile; its NW wavefronts split K by super-block (wave w takes
// blocks w, w + NW, ...) and add their double partials in wave order through LDS at the end.
// Each wave copies the 32 x 144 weight bytes and the 32 x 288 activation bytes of its super-block into its own
// part of LDS with loads in which four neighbouring lanes cover 64 contiguous bytes (a lane-per-row load touches 64
// cache lines per instruction and leaves the kernel bound by the rate of the L1's address path), one super-block
// ahead of the arithmetic, and every operand is then read from LDS.
#include "ops.h"
#include <algorithm>
#include <type_traits>

namespace bk {

typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(16))) int i32x16_t;
typedef __attribute__((ext_vector_type(4))) double f64x4_t;

constexpr int64_t GM_MAGIC = 0x41B8000000000000;      // the bits of 1.5 * 2^28

// rows of the 32x32 accumulator held by a lane: r = 0..15 -> 8*(r/4) + 4*(lane/32) + r%4
__device__ __forceinline__ int mfma32_row(int r, int half) { return 8 * (r >> 2) + 4 * half + (r & 3); }

// Up to four matrices that share the activation rows run as one launch: their 32-row tiles are laid end to end.
struct MfmaGroup {
  const uint8_t* W;
  void* out;
  const uint16_t* res;
  int N, epi;
};
struct MfmaArgs {
  MfmaGroup g[4];
  int tile_first[5];      // first tile of each matrix; tile_first[i >= ngroups] = number of tiles
  const uint8_t* xq;
  int nb, B, tiles, btiles;
  uint8_t* out_q8;        // SwiGLU form: g[0] = gate (out = bf16 activation or null), g[1] = up; Q8_1 blocks of the activation
};

// Compact argument blocks (a launch pays for every 64-byte line of kernel arguments, about a quarter of a microsecond;
// MfmaArgs has three lines): one matrix in 56 bytes, the SwiGLU pair in 60.  The kernel rebuilds MfmaArgs in registers.
struct MfmaArgs1 {
  const uint8_t* W; void* out; const uint16_t* res; const uint8_t* xq;
  int N, epi, nb, B, tiles, btiles;
};
struct MfmaArgsSw {
  const uint8_t *Wg, *Wu; void* act; uint8_t* act_q8; const uint8_t* xq;
  int N, nb, B, tiles, btiles;
};
__device__ __forceinline__ const MfmaArgs& mfma_args_full(const MfmaArgs& A) { return A; }
__device__ __forceinline__ MfmaArgs mfma_args_full(const MfmaArgs1& P) {
  MfmaArgs A;
  const MfmaGroup g{P.W, P.out, P.res, P.N, P.epi};
  A.g[0] = g; A.g[1] = g; A.g[2] = g; A.g[3] = g;
  A.tile_first[0] = 0; A.tile_first[1] = A.tile_first[2] = A.tile_first[3] = A.tile_first[4] = P.tiles;
  A.xq = P.xq; A.nb = P.nb; A.B = P.B; A.tiles = P.tiles; A.btiles = P.btiles; A.out_q8 = nullptr;
  return A;
}
__device__ __forceinline__ MfmaArgs mfma_args_full(const MfmaArgsSw& P) {
  MfmaArgs A;
  const MfmaGroup g0{P.Wg, P.act, nullptr, P.N, 0}, g1{P.Wu, nullptr, nullptr, P.N, 0};
  A.g[0] = g0; A.g[1] = g1; A.g[2] = g1; A.g[3] = g1;
  A.tile_first[0] = 0; A.tile_first[1] = A.tile_first[2] = A.tile_first[3] = A.tile_first[4] = P.tiles;
  A.xq = P.xq; A.nb = P.nb; A.B = P.B; A.tiles = P.tiles; A.btiles = P.btiles; A.out_q8 = P.act_q8;
  return A;
}

enum : int { GX_ROW = 292, GW_ROW = 144, GX_BYTES = 32 * GX_ROW, GW_BYTES = 32 * GW_ROW, G_WAVE_LDS = GX_BYTES + GW_BYTES + 512 };

// Two waves a SIMD, 256 registers; lone waves and narrow tiles get there by themselves, and told so are scheduled 1 to 3 % slower.
// SWIGLU: the workgroup holds 2 NW waves; waves 0..NW-1 form the tile of 32 gate rows, waves NW..2NW-1 the tile of the
// same 32 up rows, and the last step writes act = bf16(silu(g) * u) and its Q8_1 block instead of g and u.
// TR: weight rows of the tile.  16 or 8 (the other rows of the matrix instruction repeat them and are ignored) for launches
// with so few tiles that the time is the length of one wave's instruction stream: a half or a quarter of the fold per
// super-block, two or four times the tiles.
template <int NW, bool SWIGLU, int TR = 32, typename ARGS = MfmaArgs>
__global__ __launch_bounds__(64 * NW * (SWIGLU ? 2 : 1), NW == 1 || TR < 32 ? 1 : 2) void gemm_q4k_q8_1_mfma_kernel(ARGS A_in) {
  const auto& A = mfma_args_full(A_in);
  static_assert(TR == 32 || TR == 16 || TR == 8, "tiles of 32, 16 or 8 weight rows");
  static_assert(!(SWIGLU && TR != 32), "the SwiGLU form quantizes 32 outputs at a time");
  constexpr int WAVES = NW * (SWIGLU ? 2 : 1);
  constexpr int RF = TR / 2;               // weight rows per lane
  constexpr int TN = TR >= 16 ? TR / 16 : 1;   // 16-row groups (min term; a tile of 8 fills half of one, the rest repeats it)
  // Per wave: the activation rows of the current super-block as they lie in memory (288 bytes, rows 292 apart so that
  // the lanes of a read fall into different banks), the weight rows (144 bytes each), and 512 bytes of weight scales
  // in the order the fold reads them (the 6-bit scales as bytes [8 sub-blocks][2 halves][16 rows], then d as doubles
  // [2 halves][16 rows]).  After the K loop the same memory holds the waves' partial sums [WAVES][16][64].
  __shared__ __align__(16) unsigned char lds_raw[WAVES * G_WAVE_LDS];
  static_assert(G_WAVE_LDS >= 16 * 64 * 8 && G_WAVE_LDS % 16 == 0, "the partial sums share the staging memory");

  // Workgroup -> (weight tile, batch tile).  With several batch tiles the workgroups that share a weight tile run next
  // to each other on one XCD (consecutive workgroup ids go round the 8 XCDs), batch tile fastest: the weight tile comes
  // from memory once and its other readers find it in that XCD's L2, where the activation rows stay resident.
  int tile = blockIdx.x, btile = 0;
  if (A.btiles > 1) {
    const int per_xcd = (A.tiles * A.btiles + 7) >> 3;
    const int v = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (v >= A.tiles * A.btiles) return;
    tile = v / A.btiles;
    btile = v - tile * A.btiles;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kw = SWIGLU ? wave % NW : wave;           // this wave's place in the split of K
  const bool s1 = !SWIGLU && tile >= A.tile_first[1], s2 = !SWIGLU && tile >= A.tile_first[2], s3 = !SWIGLU && tile >= A.tile_first[3];
  const uint8_t* __restrict__ W = SWIGLU ? (wave >= NW ? A.g[1].W : A.g[0].W) : s3 ? A.g[3].W : s2 ? A.g[2].W : s1 ? A.g[1].W : A.g[0].W;
  void* __restrict__ out = s3 ? A.g[3].out : s2 ? A.g[2].out : s1 ? A.g[1].out : A.g[0].out;
  const uint16_t* __restrict__ res = s3 ? A.g[3].res : s2 ? A.g[2].res : s1 ? A.g[1].res : A.g[0].res;
  const int N = s3 ? A.g[3].N : s2 ? A.g[2].N : s1 ? A.g[1].N : A.g[0].N;
  const int EPI = s3 ? A.g[3].epi : s2 ? A.g[2].epi : s1 ? A.g[1].epi : A.g[0].epi;
  const int nb = A.nb;
  const int b0 = btile * 32;                          // first batch row of this tile
  const int B = min(32, A.B - b0);
  const int64_t wrow_bytes = (int64_t)nb * 144, xrow_bytes = (int64_t)nb * 8 * 36;
  const uint8_t* __restrict__ xq = A.xq + (int64_t)b0 * xrow_bytes;

  const int half = lane >> 5, col = lane & 31, q4 = lane >> 4, l16 = lane & 15;
  const int n0 = (tile - (s3 ? A.tile_first[3] : s2 ? A.tile_first[2] : s1 ? A.tile_first[1] : 0)) * TR;
  unsigned char* const ldsX = lds_raw + wave * G_WAVE_LDS;
  unsigned char* const ldsW = ldsX + GX_BYTES;
  unsigned char* const stage = ldsW + GW_BYTES;

  // Copy maps.  Activations: instruction i = 2c + h covers bytes 64c.. of rows 16h + lane/4, 16 bytes per lane (the
  // last chunk has 32 bytes per row: lanes 2, 3 of a quad repeat lane 1's piece and store it where lane 1 does).  Rows past B
  // re-read row B-1 (their results are not stored).  Weights: piece p = lane + 64 i of the 288 16-byte pieces, row p / 9
  // (past the last piece: that piece again, to the same place); rows past N re-read row N-1.  Every lane stores in every
  // round: a store behind a lane test costs four scalar instructions and a branch.
  const int rq = lane >> 2, k4 = lane & 3;
  const uint8_t* xsrc[2] = {xq + (int64_t)min(rq, B - 1) * xrow_bytes + 16 * k4, xq + (int64_t)min(16 + rq, B - 1) * xrow_bytes + 16 * k4};
  const int xtail = 16 * min(k4, 1) - 16 * k4;                 // moves lanes 2, 3 back onto piece 17 in the last chunk
  unsigned char* const xdst[2] = {ldsX + rq * GX_ROW + 16 * k4, ldsX + (16 + rq) * GX_ROW + 16 * k4};
  unsigned char* const wlast = ldsW + min(lane + 64 * (TR * 9 / 64), TR * 9 - 1) * 16;      // the last, partial round of the weight pieces
  const uint8_t* const wbase = W + (int64_t)n0 * wrow_bytes;
  uint32_t woff[5];
#pragma unroll
  for (int i = 0; i < 5; i++) {
    const int p = min(lane + 64 * i, TR * 9 - 1), row = p / 9;
    woff[i] = (uint32_t)((min(n0 + row, N - 1) - n0) * (int)wrow_bytes + (p - 9 * row) * 16);
  }
  uint4 xr[10], wr0, wr1, wr2, wr3, wr4;
#define GM_FETCH(BLK)                                                                                                  \
  {                                                                                                                    \
    const int fb_ = (BLK);                                                                                             \
    _Pragma("unroll") for (int i = 0; i < 10; i++) {                                                                   \
      const uint32_t* p_ = (const uint32_t*)(xsrc[i & 1] + (int64_t)fb_ * 288 + 64 * (i >> 1) + (i >= 8 ? xtail : 0)); \
      xr[i] = make_uint4(p_[0], p_[1], p_[2], p_[3]); /* 4-byte aligned 16-byte load */                                \
    }                                                                                                                  \
    wr0 = *(const uint4*)(wbase + (int64_t)fb_ * 144 + woff[0]);                                                       \
    wr1 = *(const uint4*)(wbase + (int64_t)fb_ * 144 + woff[1]);                                                       \
    if (TR >= 16) wr2 = *(const uint4*)(wbase + (int64_t)fb_ * 144 + woff[2]);                                         \
    if (TR == 32) {                                                                                                    \
      wr3 = *(const uint4*)(wbase + (int64_t)fb_ * 144 + woff[3]);                                                     \
      wr4 = *(const uint4*)(wbase + (int64_t)fb_ * 144 + woff[4]);                                                     \
    }                                                                                                                  \
  }

  // where the lane's own weight row sits among the rows of its half: row = 8g + 4h + v  ->  [h][4g + v]
  const int wcol = col & (TR - 1);
  const uint32_t scmask = half ? 0x0f0f0f0fu : 0x3f3f3f3fu;
  const int stage_slot = ((wcol >> 2) & 1) * 16 + 4 * (wcol >> 3) + (wcol & 3);
  const unsigned char* const myW = ldsW + wcol * GW_ROW;        // int8 operands: weight row col, batch row col,
  const unsigned char* const myX = ldsX + col * GX_ROW;         // bytes 16*half.. of every sub-block
  // The fold's operands; opaque, so that the two forms of the fold share the addresses instead of each working them out in every super-block
  // (1 % on launches of 4 to 10 us; the gate/up form is 0.5 % faster without).
  int off_w = (int)(myW - lds_raw) + 16 * half, off_x = (int)(myX - lds_raw), off_s = (int)(stage - lds_raw) + 16 * half;
  if (!SWIGLU) asm volatile("" : "+v"(off_w), "+v"(off_x), "+v"(off_s));
  const unsigned char *const foldW = lds_raw + off_w, *const foldX = lds_raw + off_x, *const foldS = lds_raw + off_s;

  double acc[RF];
#pragma unroll
  for (int r = 0; r < RF; r++) acc[r] = 0.0;
  f64x4_t accm[TN][2];
#pragma unroll
  for (int t = 0; t < 2 * TN; t++) accm[t >> 1][t & 1] = (f64x4_t){0.0, 0.0, 0.0, 0.0};

  GM_FETCH(min(kw, nb - 1));            // requests are unconditional (clamped): the waits stay countable
  for (int blk = kw; blk < nb; blk += NW) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();     // the previous super-block has been consumed by every lane
#pragma unroll
    for (int i = 0; i < 10; i++) {
      uint32_t* p = (uint32_t*)(xdst[i & 1] + 64 * (i >> 1) + (i >= 8 ? xtail : 0));
      p[0] = xr[i].x; p[1] = xr[i].y; p[2] = xr[i].z; p[3] = xr[i].w;
    }
    *(uint4*)(ldsW + lane * 16) = wr0;
    if (TR == 8) {
      *(uint4*)wlast = wr1;
    } else if (TR == 16) {
      *(uint4*)(ldsW + (lane + 64) * 16) = wr1;
      *(uint4*)wlast = wr2;
    } else {
      *(uint4*)(ldsW + (lane + 64) * 16) = wr1;
      *(uint4*)(ldsW + (lane + 128) * 16) = wr2;
      *(uint4*)(ldsW + (lane + 192) * 16) = wr3;
      *(uint4*)wlast = wr4;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // the next super-block's bytes travel while this one is folded.  Waves that split K have one to three blocks each: their
    // last pass requests nothing (a clamped request would double the loads of a one-block wave; out_proj at batch 32
    // 6.7 -> 6.2 us); a lone wave walks all of K and keeps the branch-free clamped request (1 % faster at 1024 rows)
    if (NW == 1 || blk + NW < nb) GM_FETCH(min(blk + NW, nb - 1));

    // the 6-bit scales of the lane's weight row (half 0 stages sub-blocks 0..3, half 1 sub-blocks 4..7) and its d
    {
      const uint4 hdr = *(const uint4*)myW;
      // low bits from the word of the half's own sub-blocks, high bits (half 1) from the top of the first; the halves differ in
      // masks, not in a branch
      const uint32_t scw = ((half ? hdr.w : hdr.y) & scmask) | ((hdr.y >> 2) & ~scmask & 0x30303030u);
#pragma unroll
      for (int i = 0; i < 4; i++) stage[(4 * half + i) * 32 + stage_slot] = (unsigned char)(scw >> (8 * i));
      ((double*)(stage + 256))[stage_slot] = (double)half_to_f32((uint16_t)(hdr.x & 0xffffu));      // (both halves the same)
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // A = weights (M = weight row), B = activations (N = batch row): result[r] = I_j[n = mfma32_row(r), b = col]
    auto unpack = [](const uint4 q, int odd) {
      if (odd) return (i32x4_t){(int)((q.x >> 4) & 0x0f0f0f0fu), (int)((q.y >> 4) & 0x0f0f0f0fu), (int)((q.z >> 4) & 0x0f0f0f0fu),
                                (int)((q.w >> 4) & 0x0f0f0f0fu)};
      return (i32x4_t){(int)(q.x & 0x0f0f0f0fu), (int)(q.y & 0x0f0f0f0fu), (int)(q.z & 0x0f0f0f0fu), (int)(q.w & 0x0f0f0f0fu)};
    };
    auto load_x = [&](const unsigned char* mX, int j) {
      const uint32_t* xp = (const uint32_t*)(mX + j * 36 + 16 * half);
      return (i32x4_t){(int)xp[0], (int)xp[1], (int)xp[2], (int)xp[3]};
    };
    auto mfma = [](i32x4_t wb, i32x4_t xa) {
      i32x16_t z;
#pragma unroll
      for (int r = 0; r < 16; r++) z[r] = 0;
      return __builtin_amdgcn_mfma_i32_32x32x32_i8(wb, xa, z, 0, 0, 0);
    };
    // The sum over the eight sub-blocks is an integer: with every d8_j below 4 (rows whose largest value is below 508), d8_j * 2^24
    // is a whole number below 2^26 (fp16 has nothing finer than 2^-24), so one 64-bit multiply-add per dot holds the sum exactly
    // where the double form takes a conversion and an FMA.  It starts from the bit pattern of 1.5 * 2^28, whose last bit
    // is worth 2^-24: |sum| < 8 * 2^21.9 * 2^26 < 2^51, so the bits are the double 1.5 * 2^28 + sum * 2^-24 and one
    // subtraction, exact, gives the double.  Units with a larger d8 in any row of the tile run the same fold from 0 and convert its
    // sum in two halves (rounded once): below 128 (values below 16256) d8_j * 2^24 still fits 31 bits, above that the fold
    // takes d8_j * 2^(24 - s) as long as these are whole numbers, which scales of 2^(s - 14) and more are.  What is left (non-finite
    // scales, and one of 2^(7 + s) beside one below 2^(s - 14)) is folded in double, one sub-block after the other.  us for
    // 77 rows x 12288 x 2048 and for gate + up of 1024 x 6144 x 2048, every unit of a kind: scales below 4 24.0 and 154, up to 128 24.9
    // and 163, above 26.1 and 179, non-finite 30.4 and 217; everything in double, pipelined over the sub-blocks: 25.3 and 184.  (That
    // form beside this one takes more than the 256 registers of two waves a SIMD.)
    double S1[RF];
    auto fold = [&](auto small_scales, const unsigned char* mW, const unsigned char* mX, const unsigned char* mS, int s) __attribute__((always_inline)) {
      constexpr bool SMALL = decltype(small_scales)::value;
      const float to_whole = SMALL ? 16777216.0f : __builtin_bit_cast(float, (151 - s) << 23);      // 2^(24 - s): d8_j times this is the whole number
      // The fold runs as a pipeline over the sub-blocks: the operands and scale bytes of sub-block j+1 are requested from
      // LDS before sub-block j is folded and its matrix instruction is issued halfway through that fold, when they have
      // arrived; the second half of the fold covers the matrix instruction's latency.
      int64_t S[RF];
      uint4 q = *(const uint4*)(mW + 16), qn = q;
      // a narrow tile reads the scales of its own rows alone (of a wider read it would wait for the part that it has no use for)
      using scales_t = std::conditional_t<RF == 16, uint4, std::conditional_t<RF == 8, uint2, uint32_t>>;
      scales_t scb = *(const scales_t*)mS, scn = scb;
      uint32_t dsw = *(const uint16_t*)(mX + 32), dsn = dsw;
      i32x4_t xn = load_x(mX, 0);
      i32x16_t c = mfma(unpack(q, 0), xn), cn = c;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (j + 1 < 8) {
          scn = *(const scales_t*)(mS + (j + 1) * 32);
          dsn = *(const uint16_t*)(mX + (j + 1) * 36 + 32);
          xn = load_x(mX, j + 1);
          if (j & 1) qn = *(const uint4*)(mW + 16 + 32 * ((j + 1) >> 1));
        }
        __builtin_amdgcn_sched_barrier(0);
        const int m8 = (int)fma(half_to_f32((uint16_t)dsw), to_whole, 0.0f);      // (one instruction with the conversion; exact)
        uint32_t scv[RF / 4];
        __builtin_memcpy(scv, &scb, sizeof scv);
        // Four rows: their scales are the four bytes of one word.  (The sums are instructions, not C expressions: integer sums have
        // no order of their own, and the compiler gathers all eight matrix results in front of them; four in a block, because
        // it puts an idle cycle between neighbouring blocks that it cannot look into.  The products stay in C: only there does
        // the compiler keep the distance that a matrix instruction's result needs before it is read.)
        auto fold4 = [&](int r) {
          int t[4];
#pragma unroll
          for (int i = 0; i < 4; i++) t[i] = __mul24(c[r + i], (int)((scv[r >> 2] >> (8 * i)) & 0xffu));
          // A narrow tile ignores half of the matrix instruction's results or more.  All their registers stay taken up to the first use
          // of the results: a sum of the sub-block before, placed in one of them, would be overwritten when the instruction ends
          // (the compiler keeps its own instructions at a distance, but does not see what the blocks write).
          if (RF < 16 && r == 0) asm volatile("" :: "v"(c));
          if (j == 0)
            asm volatile("v_mad_i64_i32 %0, vcc, %4, %8, %9\n\tv_mad_i64_i32 %1, vcc, %5, %8, %9\n\t"
                         "v_mad_i64_i32 %2, vcc, %6, %8, %9\n\tv_mad_i64_i32 %3, vcc, %7, %8, %9"
                         : "=&v"(S[r]), "=&v"(S[r + 1]), "=&v"(S[r + 2]), "=&v"(S[r + 3])
                         : "v"(t[0]), "v"(t[1]), "v"(t[2]), "v"(t[3]), "v"(m8), "s"(SMALL ? GM_MAGIC : (int64_t)0) : "vcc");
          else
            asm volatile("v_mad_i64_i32 %0, vcc, %4, %8, %0\n\tv_mad_i64_i32 %1, vcc, %5, %8, %1\n\t"
                         "v_mad_i64_i32 %2, vcc, %6, %8, %2\n\tv_mad_i64_i32 %3, vcc, %7, %8, %3"
                         : "+&v"(S[r]), "+&v"(S[r + 1]), "+&v"(S[r + 2]), "+&v"(S[r + 3])
                         : "v"(t[0]), "v"(t[1]), "v"(t[2]), "v"(t[3]), "v"(m8) : "vcc");
        };
        // (the first half before the matrix instruction: two blocks of the sixteen rows, one of eight, none of four)
        constexpr int FIRST = RF / 8 * 4;
#pragma unroll
        for (int r = 0; r < FIRST; r += 4) fold4(r);
        __builtin_amdgcn_sched_barrier(0);
        if (j + 1 < 8) {
          if (j & 1) q = qn;
          cn = mfma(unpack(q, (j + 1) & 1), xn);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = FIRST; r < RF; r += 4) fold4(r);
        __builtin_amdgcn_sched_barrier(0);
        c = cn; scb = scn; dsw = dsn;
      }
#pragma unroll
      for (int r = 0; r < RF; r++)
        S1[r] = SMALL ? __builtin_bit_cast(double, S[r]) - 0x1.8p28
                      : ldexp(fma((double)(int)(S[r] >> 32), 4294967296.0, (double)(uint32_t)S[r]), s - 24);
    };
    uint32_t dmax = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) dmax = max(dmax, (uint32_t)*(const uint16_t*)(myX + j * 36 + 32));
    if (__builtin_expect(__ballot(dmax >= 0x4400u) == 0, 1)) {
      fold(std::true_type{}, foldW, foldX, foldS, 0);
    } else {
      int ln = lane;
      asm volatile("" : "+v"(ln));         // (addresses worked out here, not kept in registers around the loop over K)
      const int hf = ln >> 5;
      const unsigned char *const mW = ldsW + (ln & (TR - 1)) * GW_ROW + 16 * hf, *const mX = ldsX + (ln & 31) * GX_ROW, *const mS = stage + 16 * hf;
      int s = 0;
      bool in_double = false;
      if (__ballot(dmax >= 0x5800u) != 0) {
        uint32_t top = 0, low = 0xffffu;   // the largest scale and the smallest that is not zero, less one
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const uint32_t d = *(const uint16_t*)(mX + j * 36 + 32) & 0x7fffu;
          top = max(top, d);
          low = min(low, d - 1u);
        }
        const int wtop = __builtin_amdgcn_readfirstlane((int)wave_max((float)top)), wlow = 1 - __builtin_amdgcn_readfirstlane((int)wave_max(-(float)low));
        s = max((wtop >> 10) - 21, 0);
        in_double = wtop >= 0x7c00 || (s > 0 && wlow < ((s + 1) << 10));
      }
      if (!in_double) {
        fold(std::false_type{}, foldW, foldX, foldS, s);
      } else {
#pragma unroll
        for (int r = 0; r < RF; r++) S1[r] = 0.0;
#pragma unroll 1
        for (int j = 0; j < 8; j++) {
          const i32x16_t c = mfma(unpack(*(const uint4*)(mW + 16 + 32 * (j >> 1)), j & 1), load_x(mX, j));
          const double d8 = (double)half_to_f32(*(const uint16_t*)(mX + j * 36 + 32));
          const uint4 scb = *(const uint4*)(mS + j * 32);
          const uint32_t scv[4] = {scb.x, scb.y, scb.z, scb.w};
#pragma unroll
          for (int r = 0; r < RF; r++) S1[r] = fma(d8, (double)__mul24(c[r], (int)((scv[r >> 2] >> (8 * (r & 3))) & 0xffu)), S1[r]);
        }
      }
    }
    {
      const double2* dd = (const double2*)(stage + 256 + 128 * half);
#pragma unroll
      for (int r = 0; r < RF; r += 2) {
        const double2 v = dd[r >> 1];
        acc[r] = fma(v.x, S1[r], acc[r]);
        acc[r + 1] = fma(v.y, S1[r + 1], acc[r + 1]);
      }
    }
    // min term: accm[tn][tb] += (-dmin * m_j)[16 rows x 4 sub-blocks] . s8_j[4 sub-blocks x 16 batch rows], for the
    // sub-blocks 0..3 and then 4..7; a lane supplies row 16 t + l16 of either side at sub-blocks q4 and 4 + q4
    double am[TN][2], bm[2][2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      if (t < TN) {
        const uint4 hm = *(const uint4*)(ldsW + ((16 * t + l16) & (TR - 1)) * GW_ROW);
        const float dmin_neg = -half_to_f32((uint16_t)(hm.x >> 16));
        const uint32_t zb = (hm.z >> (8 * q4)) & 0xffu, wb = (hm.w >> (8 * q4)) & 0xffu;
        am[t][0] = (double)(dmin_neg * (float)(zb & 63u));
        am[t][1] = (double)(dmin_neg * (float)((wb >> 4) | ((zb >> 6) << 4)));
      }
      const unsigned char* xs = ldsX + (16 * t + l16) * GX_ROW + q4 * 36 + 34;
      bm[t][0] = (double)half_to_f32(*(const uint16_t*)xs);
      bm[t][1] = (double)half_to_f32(*(const uint16_t*)(xs + 144));
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int t = 0; t < 2 * TN; t++)
        accm[t >> 1][t & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(am[t >> 1][k], bm[t & 1][k], accm[t >> 1][t & 1], 0, 0, 0);
  }

  // The min-term accumulators hold element (n = 16 tn + 4 v + q4, b = 16 tb + l16); they reach the lanes that own those
  // outputs through this wave's part of the buffer.  Slot (r, lane) of a wave's part sits at r*64 + (lane ^ (r + 16*half)):
  // the swizzle keeps the transposed reads of the last step free of bank conflicts.
  double* part = (double*)lds_raw + wave * 16 * 64;
  __syncthreads();                         // all waves are done with the scales that share the buffer
#pragma unroll
  for (int t = 0; t < 2 * TN; t++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int n = 16 * (t >> 1) + 4 * v + q4, b = 16 * (t & 1) + l16;
      const int rr = 4 * (n >> 3) + (n & 3), hh = (n >> 2) & 1;
      part[rr * 64 + ((b + 32 * hh) ^ (rr + 16 * hh))] = accm[t >> 1][t & 1][v];
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int r = 0; r < RF; r++) acc[r] += part[r * 64 + (lane ^ (r + 16 * half))];

  // Last step: every wave leaves its 16 partial sums per lane in LDS; the threads then finish the outputs with the
  // weight row along the lanes (contiguous stores): thread (wave w, lane) takes row lane % 32 and batch rows
  // 2 (w R + i) + lane / 32, and adds the waves' partials in wave order.
  __builtin_amdgcn_wave_barrier();         // slot (r, lane) was read above by this lane only
#pragma unroll
  for (int r = 0; r < RF; r++) part[r * 64 + (lane ^ (r + 16 * half))] = acc[r];
  __syncthreads();
  const double* all = (const double*)lds_raw;
  if (SWIGLU && NW == 1) {
    // Prompts: a thread takes eight consecutive weight rows of one batch row, four neighbouring lanes a Q8_1 block, so that the
    // block's maximum, scale and sum are formed once per eight values and the lanes' eight sigmoids are independent.  (With a
    // value per lane and the block across 32 lanes, every value paid for them: this step was 27 of 169 us at 1024 rows x
    // 2 x 6144 x 2048.)  With this form 154 us.
    const int g8 = lane & 3, b = 16 * wave + (lane >> 2);
    float f[8];
    uint32_t a2[4];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int rr = 4 * g8 + (i & 3), hh = i >> 2, slot = rr * 64 + ((b + 32 * hh) ^ (rr + 16 * hh));
      const float gv = (float)all[slot], uv = (float)all[16 * 64 + slot];
      const uint16_t a16 = f32_to_bf16(__fmul_rn(__fmul_rn(gv, sigmoid_f64(gv)), uv));
      f[i] = bf16_to_f32(a16);
      a2[i >> 1] = i & 1 ? a2[i >> 1] | ((uint32_t)a16 << 16) : a16;
    }
    uint32_t pk[2];
    const uint32_t ds = quad_q8_1(f, pk);
    if (b < B) {
      if (uint16_t* act = (uint16_t*)A.g[0].out) {
        act += (int64_t)(b0 + b) * N + n0 + 8 * g8;
        if (((uintptr_t)act & 15) == 0) *(uint4*)act = make_uint4(a2[0], a2[1], a2[2], a2[3]);
        else
#pragma unroll
          for (int i = 0; i < 8; i++) act[i] = (uint16_t)(a2[i >> 1] >> (16 * (i & 1)));
      }
      uint32_t* q = (uint32_t*)(A.out_q8 + ((int64_t)(b0 + b) * (N / 32) + (n0 >> 5)) * 36);
      q[2 * g8] = pk[0];
      q[2 * g8 + 1] = pk[1];
      if (g8 == 0) q[8] = ds;
    }
    return;
  }
  // the thread's output row fn of the tile and its batch rows fb0 + FB * (wave R + i): 32 rows -> (lane % 32, lane / 32),
  // 16 rows -> (lane % 16, lane / 16), 8 rows -> (lane % 8, lane / 8)
  constexpr int R = TR / 2 / WAVES > 0 ? TR / 2 / WAVES : 1, FB = 64 / TR;
  if (wave * R * FB >= 32) return;         // (a 16-row tile gives each of eight waves one batch-row pair; an 8-row tile is finished by four waves)
  const int fn = lane & (TR - 1), fb0 = lane / TR;
  const int rr = 4 * (fn >> 3) + (fn & 3), hh = (fn >> 2) & 1;
  float y[SWIGLU ? 1 : R], u_[SWIGLU ? R : 1], g_[SWIGLU ? R : 1];
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int b = FB * (wave * R + i) + fb0;
    const int slot = rr * 64 + ((b + 32 * hh) ^ (rr + 16 * hh));
    if (SWIGLU) {
      double gd = all[slot], ud = all[NW * 16 * 64 + slot];
#pragma unroll
      for (int w = 1; w < NW; w++) { gd += all[w * 16 * 64 + slot]; ud += all[(NW + w) * 16 * 64 + slot]; }
      g_[i] = (float)gd; u_[i] = (float)ud;
    } else {
      double t = all[slot];
#pragma unroll
      for (int w = 1; w < NW; w++) t += all[w * 16 * 64 + slot];
      y[i] = (float)t;
    }
  }
  if (SWIGLU) {
    // g and u were rounded to f32 like the matmul's own outputs; the 32 lanes of a half hold one Q8_1 block of the activation
    uint16_t* act = (uint16_t*)A.g[0].out;
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int b = FB * (wave * R + i) + fb0;
      const uint16_t a16 = f32_to_bf16(__fmul_rn(__fmul_rn(g_[i], sigmoid_f64(g_[i])), u_[i]));
      const bool valid = b < B;
      if (valid && act) act[(int64_t)(b0 + b) * N + n0 + col] = a16;
      lane32_q8_1_store(bf16_to_f32(a16), A.out_q8 + ((int64_t)(b0 + b) * (N / 32) + (n0 >> 5)) * 36, col, valid);
    }
    return;
  }
  const bool n_ok = n0 + fn < N;
  const int64_t o0 = (int64_t)b0 * N + n0 + fn;
  if (EPI == GEPI_F32) {
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int b = FB * (wave * R + i) + fb0;
      if (n_ok && b < B) ((float*)out)[o0 + (int64_t)b * N] = y[i];
    }
  } else if (EPI == GEPI_BF16) {
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int b = FB * (wave * R + i) + fb0;
      if (n_ok && b < B) ((uint16_t*)out)[o0 + (int64_t)b * N] = f32_to_bf16(y[i]);
    }
  } else {
    uint16_t rv[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int b = FB * (wave * R + i) + fb0;
      rv[i] = (n_ok && b < B) ? res[o0 + (int64_t)b * N] : (uint16_t)0;
    }
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int b = FB * (wave * R + i) + fb0;
      if (n_ok && b < B) ((uint16_t*)out)[o0 + (int64_t)b * N] = f32_to_bf16(bf16_to_f32(f32_to_bf16(y[i])) + bf16_to_f32(rv[i]));
    }
  }
}

#undef GM_FETCH

int g_tune_gemm_nw = 0;      // waves per tile (1, 2, 4, 8); 0 = chosen from the shape
int g_tune_gemm_r16 = -1;    // narrow tiles (single batch tile only): 0 off, 1 = 16 weight rows, 2 = 8, -1 = from the shape

// Waves that share a tile.  A CU holds eight waves of this kernel (their registers; 115 KB of LDS), so w tiles on it run in rounds of
// 8 / nw: more waves a tile make a round shorter and leave fewer waves idle in the last one, but every wave brings a fixed part (first
// loads, the sums through LDS), and two waves on a SIMD hide each other's waits.  Which one wins depends on how full the last round
// is, and where two are close on the length of a row, whose stream outweighs the fixed part; us on the sizes in brackets, by tiles per CU,
// rounded up, nw = 1 / 2 / 4, each at K = 1024, 2048 and 6144:
//   up to one: eight (K >= 2048; 2048 x 6144 at 128 rows 40.8 / 23.6 / 15.5, eight 13.9);
//   two (N = 1024 at 512 rows): 10.9 / 9.8 / 8.0, 17.2 / 14.9 / 11.5, 42.5 / 35.6 / 23.8; three (1536): 11.3 / 10.4 / 10.6, 18.1 / 16.0 / 15.6, 44.3 / 37.9 / 33.1;
//   four (2048): 11.5 / 11.2 / 12.8, 18.8 / 17.5 / 19.2, 45.4 / 39.7 / 41.0; five (2560): 15.7 / 15.3 / 15.4, 26.5 / 23.5 / 22.4, 66.8 / 55.9 / 49.9;
//   six (3072): 16.3 / 19.0 / 17.9, 27.1 / 29.9 / 25.8, 68.2 / 72.3 / 59.2;
//   seven (3584): 17.1 / 19.7 / 20.3, 28.4 / 30.9 / 29.3, 70.9 / 73.0 / 67.3 (13312 x 3584 at 128 rows 45.9 / 46.9 / 45.6, x 4096 51.7 / 52.9 / 49.1, 3584 x 4096 at 512 53.0 / - / 53.3);
//   eight (4096): 17.9 / 21.5 / 22.8, 28.8 / 33.0 / 32.8, 72.3 / 81.8 / 75.7; nine (4608): 24.3 / 23.3 / 25.4, 40.4 / 36.0 / 36.2, 103.3 / 88.6 / 84.7;
//   ten (5120): 24.7 / 25.8 / 27.8, 40.6 / 40.4 / 40.0 (4900 rows 39.7 / 39.1 / -), 104.1 / 100.1 / 92.9; eleven (5376): 25.0 / 26.9 / 30.3, 40.6 / 42.2 / 43.1, 104.5 / 106.0 / 101.2;
//   twelve (6144): 25.3 / 28.8 / 32.8, 41.6 / 45.6 / 46.6, 109.7 / 116.0 / 111.0.
// (Left to two and one although four is 3 to 7 % faster: nine to eleven at K = 6144.  Six at K = 1024 would be 9 % faster with one.)
static int waves_per_tile(int64_t tiles, int nb) {
  const int64_t per_cu = (tiles + num_cus() - 1) / num_cus();
  int nw;
  if (per_cu <= 1 && nb >= 8) nw = 8;
  else if (per_cu <= 3) nw = 4;
  else if (per_cu == 4) nw = 2;
  else if (per_cu <= 6) nw = 4;
  else if (per_cu == 7) nw = nb >= 20 ? 4 : 1;
  else if (per_cu == 8) nw = 1;
  else if (per_cu == 9 || (per_cu == 10 && nb >= 8)) nw = 2;
  else nw = 1;
  return nb >= 4 ? nw : std::min(nw, nb >= 2 ? 2 : 1);       // no more than a row has super-blocks
}

// The SwiGLU form, by pairs of tiles per CU (a CU holds four pairs of lone waves), nw = 1 / 2 / 4 in us at K = 1024, 2048 and 6144 (N of gate and up in
// brackets, at 512 rows):
// one (512): 12.4 / 10.8 / 9.5, 18.8 / 14.4 / 12.7, 43.9 / 28.1 / 24.7; two (1024): 18.1 / 14.8 / 16.7, 26.9 / 20.1 / 22.4, 65.3 / 42.4 / 44.3;
// three (1536): 18.4 / 19.7 / 22.3, 28.7 / 28.2 / 32.0, 69.7 / 60.8 / 65.0 (5120 x 3584 at 128 rows 44.9 / 40.8 / 48.1, x 4096 50.1 / 45.0 / 49.3);
// four (2048): 19.6 / 23.7 / 28.9, 31.1 / 35.1 / 41.7, 77.5 / 76.5 / 85.9; five (2560): 26.8 / 28.7 / 35.4, 42.8 / 41.7 / 51.6, 105.8 / 95.4 / 106.3;
// six (3072): 34.5 / 33.8 / 42.5, 55.3 / 49.0 / 61.3, 136.9 / 112.2 / 127.7; seven (3328): 34.9 / 38.2 / 48.6, 56.0 / 55.3 / 70.7, 139.3 / 127.2 / 148.4;
// eight (4096): 37.9 / 42.4 / 55.4, 62.2 / 62.8 / 80.8, 153.6 / 145.2 / 169.3.  (Left to one although two is 6 to 10 % faster: five, seven and eight at 6144.)
static int waves_per_tile_swiglu(int64_t pairs, int nb) {
  const int64_t per_cu = (pairs + num_cus() - 1) / num_cus();
  const int nw = per_cu <= 1 ? 4 : (per_cu == 2 || per_cu == 6 || (per_cu == 3 && nb >= 12) ? 2 : 1);
  return nb >= 4 ? nw : std::min(nw, nb >= 2 ? 2 : 1);
}

template <typename ARGS>
static void launch_mfma_plain(int tr, int nw, dim3 grid, const ARGS& A) {
  if (tr == 16) {
    if (nw >= 8) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<8, false, 16, ARGS>), grid, dim3(512), 0, stream(), A);
    else hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<4, false, 16, ARGS>), grid, dim3(256), 0, stream(), A);
  } else if (tr == 8) {
    if (nw >= 8) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<8, false, 8, ARGS>), grid, dim3(512), 0, stream(), A);
    else hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<4, false, 8, ARGS>), grid, dim3(256), 0, stream(), A);
  } else if (nw == 8) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<8, false, 32, ARGS>), grid, dim3(512), 0, stream(), A);
  else if (nw == 4) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<4, false, 32, ARGS>), grid, dim3(256), 0, stream(), A);
  else if (nw == 2) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<2, false, 32, ARGS>), grid, dim3(128), 0, stream(), A);
  else hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<1, false, 32, ARGS>), grid, dim3(64), 0, stream(), A);
}

int launch_gemm_group_mfma(const void* xq, int K, int batch, int ngroups, const void* const* W, void* const* out,
                           const void* const* res, const int* N, const int* epi) {
  BK_REQUIRE(xq && ngroups >= 1 && ngroups <= 4, "gemm_q4k_q8_1_mfma: bad arguments");
  BK_REQUIRE(K > 0 && K % 256 == 0, "gemm_q4k_q8_1_mfma: K=%d must be a positive multiple of 256", K);
  BK_REQUIRE(batch >= 1 && batch <= 32 * 65535, "gemm_q4k_q8_1_mfma: bad batch=%d", batch);
  BK_REQUIRE(((uintptr_t)xq & 3) == 0, "gemm_q4k_q8_1_mfma: xq must be 4-byte aligned");
  MfmaArgs A{};
  A.xq = (const uint8_t*)xq; A.nb = K / 256; A.B = batch;
  int tiles = 0;
  for (int i = 0; i < ngroups; i++) {
    BK_REQUIRE(W[i] && out[i] && N[i] > 0 && ((uintptr_t)W[i] & 15) == 0, "gemm_q4k_q8_1_mfma: matrix %d: null, misaligned or N <= 0", i);
    BK_REQUIRE(epi[i] == GEPI_F32 || epi[i] == GEPI_BF16 || epi[i] == GEPI_BF16_ADD, "gemm_q4k_q8_1_mfma: bad epilogue %d", epi[i]);
    BK_REQUIRE(epi[i] != GEPI_BF16_ADD || res[i], "gemm_q4k_q8_1_mfma: the add epilogue needs a residual");
    A.g[i].W = (const uint8_t*)W[i]; A.g[i].out = out[i]; A.g[i].res = (const uint16_t*)res[i]; A.g[i].N = N[i]; A.g[i].epi = epi[i];
    A.tile_first[i] = tiles;
    tiles += (N[i] + 31) / 32;
  }
  if (g_tune_gemm_nw == 0 && gemm_tiles_pay(tiles, batch, A.nb, false)) return launch_gemm_tiles(xq, A.nb, batch, ngroups, W, out, res, N, epi);
  // One batch tile and so few weight tiles that CUs would stay empty: tiles of 16 weight rows (twice as many
  // workgroups, half the fold per wave) when that still leaves half of them empty... of 8 when a quarter.  Measured on the
  // 64-tile shapes at batch 32.
  int tr = 32;
  if (batch <= 32) {
    if (g_tune_gemm_r16 >= 0) tr = g_tune_gemm_r16 == 0 ? 32 : (g_tune_gemm_r16 == 1 ? 16 : 8);
    else if (A.nb >= 4) tr = 4 * tiles <= num_cus() ? 8 : (2 * tiles <= num_cus() ? 16 : 32);
  }
  if (tr != 32) {
    tiles = 0;
    for (int i = 0; i < ngroups; i++) { A.tile_first[i] = tiles; tiles += (N[i] + tr - 1) / tr; }
  }
  for (int i = ngroups; i < 5; i++) A.tile_first[i] = tiles;
  const int btiles = (batch + 31) / 32;
  const int64_t wgs = (int64_t)tiles * btiles;
  int nw = g_tune_gemm_nw > 0 ? g_tune_gemm_nw : waves_per_tile(wgs, A.nb);
  nw = nw >= 8 ? 8 : (nw >= 4 ? 4 : (nw >= 2 ? 2 : 1));
  A.tiles = tiles; A.btiles = btiles;
  const dim3 grid(btiles > 1 ? (unsigned)(8 * ((wgs + 7) / 8)) : (unsigned)tiles);
  if (ngroups == 1) {
    const MfmaArgs1 P{A.g[0].W, A.g[0].out, A.g[0].res, A.xq, A.g[0].N, A.g[0].epi, A.nb, A.B, tiles, btiles};
    launch_mfma_plain(tr, nw, grid, P);
  } else {
    launch_mfma_plain(tr, nw, grid, A);
  }
  BK_LAUNCH_CHECK();
  return BK_OK;
}

int launch_gemm_q4k_q8_1_mfma(const void* W, const void* xq, void* y, int N, int K, int batch, int out_dtype,
                              const void* residual) {
  BK_REQUIRE(W && xq && y, "gemm_q4k_q8_1_mfma: null pointer");
  BK_REQUIRE(out_dtype == DT_F32 || out_dtype == DT_BF16, "gemm_q4k_q8_1_mfma: out_dtype must be 0 (f32) or 1 (bf16)");
  BK_REQUIRE(!(residual && out_dtype != DT_BF16), "gemm_q4k_q8_1_mfma: a residual needs bf16 output");
  const int epi = out_dtype == DT_F32 ? GEPI_F32 : (residual ? GEPI_BF16_ADD : GEPI_BF16);
  return launch_gemm_group_mfma(xq, K, batch, 1, &W, &y, &residual, &N, &epi);
}

}  // namespace bk

namespace bk {

// gate and up projections with the SwiGLU and the Q8_1 quantization of its result in the last step of the matmul:
// act[b, n] = bf16(silu(g) * u) (src/fusion.ts:324-330 on the two matmuls' f32 outputs), written as bf16 (if `act` is
// given) and as the Q8_1 blocks the down projection reads.
int launch_gemm_swiglu_mfma(const void* xq, int K, int batch, const void* Wg, const void* Wu, int N, void* act, void* act_q8) {
  BK_REQUIRE(xq && Wg && Wu && act_q8, "gemm_swiglu_mfma: null pointer");
  BK_REQUIRE(K > 0 && K % 256 == 0, "gemm_swiglu_mfma: K=%d must be a positive multiple of 256", K);
  BK_REQUIRE(N > 0 && N % 32 == 0, "gemm_swiglu_mfma: N=%d must be a positive multiple of 32", N);
  BK_REQUIRE(batch >= 1 && batch <= 32 * 65535, "gemm_swiglu_mfma: bad batch=%d", batch);
  BK_REQUIRE(((uintptr_t)xq & 3) == 0 && ((uintptr_t)Wg & 15) == 0 && ((uintptr_t)Wu & 15) == 0 && ((uintptr_t)act_q8 & 3) == 0,
             "gemm_swiglu_mfma: misaligned pointer");
  MfmaArgs A{};
  A.xq = (const uint8_t*)xq; A.nb = K / 256; A.B = batch;
  A.g[0].W = (const uint8_t*)Wg; A.g[0].out = act; A.g[0].N = N;
  A.g[1].W = (const uint8_t*)Wu; A.g[1].N = N;
  A.out_q8 = (uint8_t*)act_q8;
  if (g_tune_gemm_nw == 0 && gemm_tiles_pay(N / 32, batch, A.nb, true)) return launch_gemm_swiglu_tiles(xq, A.nb, batch, Wg, Wu, N, act, act_q8);
  const int tiles = N / 32, btiles = (batch + 31) / 32;
  for (int i = 0; i < 5; i++) A.tile_first[i] = i ? tiles : 0;
  A.tiles = tiles; A.btiles = btiles;
  const int64_t wgs = (int64_t)tiles * btiles;
  int nw = g_tune_gemm_nw > 0 ? g_tune_gemm_nw : waves_per_tile_swiglu(wgs, A.nb);
  nw = nw >= 4 ? 4 : (nw >= 2 ? 2 : 1);
  const dim3 grid(btiles > 1 ? (unsigned)(8 * ((wgs + 7) / 8)) : (unsigned)tiles);
  const MfmaArgsSw P{A.g[0].W, A.g[1].W, act, (uint8_t*)act_q8, A.xq, N, A.nb, A.B, tiles, btiles};
  if (nw == 4) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<4, true, 32, MfmaArgsSw>), grid, dim3(512), 0, stream(), P);
  else if (nw == 2) hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<2, true, 32, MfmaArgsSw>), grid, dim3(256), 0, stream(), P);
  else hipLaunchKernelGGL((gemm_q4k_q8_1_mfma_kernel<1, true, 32, MfmaArgsSw>), grid, dim3(128), 0, stream(), P);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

}  // namespace bk
