// Batched matmul for prompts: the product of gemm_mfma.hip, C[B, N] = Xq[B, K] . W[N, K]^T with the same sums and the same bits,
// where a launch has so many tiles that its time is throughput and not the length of one wave's stream.
//
// A workgroup of four waves owns 64 weight rows x 64 activation rows, a wave 32 x 32 of them.  The super-block that all four work on is
// copied to LDS once, by all of them (a lone wave copies 32 rows of either side for itself: twice the loads, and 45 stores where
// this takes 22), and what every wave would work out for itself is worked out on the way: activation scales as whole
// numbers, weight scales as bytes in the order of the fold, -dmin m.  With the copy shared, and with the accumulators
// of the two sums in one set of registers, a wave gets by with 168 registers, so that three waves share a SIMD where the other kernel has two.
//
// One set of accumulators: the tile is four 16 x 16 products.  v_mfma_i32_16x16x32_i8 leaves row 4 q + v of its tile in register v of lanes 16 q..,
// v_mfma_f64_16x16x4_f64 row 4 v + q; the weight rows of the first are handed over in the order (4 (i % 4) + i / 4) that makes the two agree, and
// the min term is added to the sums of the fold where they are.  (The 32 x 32 form takes half the matrix time, but its rows
// cannot be made to agree.  With it, 227 registers and two waves a SIMD: 1024 rows x 12288 x 2048 137 us where this took 123.)
//
// What bounds it: vector issue and the matrix unit together.  A unit (32 x 32 x 256) is 1900 cycles of vector instructions (1024 of them the fold: a
// multiply and a 64-bit multiply-add per dot), 512 of the f64 matrix instruction, which runs on the vector unit, and 512 of the int8 one,
// of which about 300 hide behind the others: 2600 of the 2900 that pass.  us, gemm_mfma.hip -> here, 1024 rows:
//   12288 x 2048: 139 -> 120; 6144 x 2048: 73.1 -> 64.2; 4096 x 6144: 135 -> 127; gate + up 2 x 6144 x 2048 with SwiGLU: 154 -> 126.
#include "ops.h"
#include <algorithm>
#include <type_traits>

namespace bk {

typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(4))) double f64x4_t;

constexpr int64_t GT_MAGIC = 0x41B8000000000000;      // the bits of 1.5 * 2^28

// Up to four matrices that share the activation rows; their 32-row tiles are laid end to end.  SwiGLU: g[0] = gate (out = bf16 activation or
// null), g[1] = up, out_q8 = Q8_1 blocks of the activation.
struct TileGroup {
  const uint8_t* W;
  void* out;
  const uint16_t* res;
  int N, epi;
};
struct TileArgs {
  TileGroup g[4];
  int tile_first[4];      // first tile of each matrix; past the last one: the number of tiles
  const uint8_t* xq;
  int nb, B, tiles, mtiles;
  uint8_t* out_q8;
};

// LDS of a workgroup: the 64 weight and 64 activation rows of one super-block.
enum : int {
  GT_PLANE = 264,                      // 32 rows of 8 bytes, and 8 more (the copy's stores fall into different banks)
  GT_WORDS = 160,                      // 32 rows of 4 bytes, and 32 more
  GT_XT = 32 * GT_PLANE,               // activations of 32 rows: [8 sub-blocks][4 quarters of 8 bytes][row]
  GT_WT = 16 * GT_PLANE,               // weights: [4 pairs of sub-blocks][4 quarters][row]
  GT_X = 0, GT_W = GT_X + 2 * GT_XT,
  GT_RAW = GT_W + 2 * GT_WT,           // (d, s) halves of the activation blocks: [2 tiles][8][row]
  GT_M8 = GT_RAW + 16 * GT_WORDS,      // d as a whole number of 2^-24
  GT_MIN = GT_M8 + 16 * GT_WORDS,      // -dmin * m: [2 tiles][8][row]
  GT_D = GT_MIN + 16 * GT_WORDS,       // d of the weight rows as doubles, in the order the fold reads them
  GT_SC = GT_D + 512,                  // 6-bit scales as bytes, the same order: [2 tiles][8][32]
  GT_FLAG = GT_SC + 512,               // per wave: its share of the activation scales has one outside [0, 4) (1), outside (-128, 128) (3)
  GT_LDS = GT_FLAG + 16,
  GT_PITCH = 33,                       // the results pass through the same memory
};
static_assert(4 * 32 * GT_PITCH * 4 <= GT_LDS, "results share the staging memory");

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gt_rsrc(const void* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, -1, 0x00027000); }
__device__ __forceinline__ uint4 gt_load16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, int off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, off, 0));
}

// Four rows of a 16 x 16 tile: S[v] += (c[v] * byte v of w) * m.  (Instructions for the reasons given in gemm_mfma.hip.  The first product stays in C: at
// it the compiler keeps the distance that the results of a matrix instruction need before they are read, and the block, which reads the
// other three, comes behind it.  Carries go to four different places: into one place they wait for each other, 3.7 ns a multiply-add for a wave alone instead of 2.6.)
template <bool FIRST, bool SMALL>
__device__ __forceinline__ void gt_fold4(int64_t (&S)[4], const i32x4_t& c, uint32_t w, int m) {
  int p = __mul24(c[0], (int)(w & 0xffu)), q;
  uint64_t k0, k1, k2;
#define GT_MUL(P, C, BY) "v_mul_i32_i24_sdwa %[" P "], %[" C "], %[w] dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_" BY "\n\t"
#define GT_MAD(D, K, P, FROM) "v_mad_i64_i32 %[" D "], " K ", %[" P "], %[m], %[" FROM "]\n\t"
  if constexpr (FIRST)
    asm volatile(GT_MUL("q", "c1", "1") GT_MAD("s0", "vcc", "p", "z") GT_MUL("p", "c2", "2") GT_MAD("s1", "%[k0]", "q", "z")
                 GT_MUL("q", "c3", "3") GT_MAD("s2", "%[k1]", "p", "z") GT_MAD("s3", "%[k2]", "q", "z")
                 : [s0] "=&v"(S[0]), [s1] "=&v"(S[1]), [s2] "=&v"(S[2]), [s3] "=&v"(S[3]), [p] "+&v"(p), [q] "=&v"(q), [k0] "=&s"(k0), [k1] "=&s"(k1), [k2] "=&s"(k2)
                 : [c1] "v"(c[1]), [c2] "v"(c[2]), [c3] "v"(c[3]), [w] "v"(w), [m] "v"(m), [z] "s"(SMALL ? GT_MAGIC : (int64_t)0) : "vcc");
  else
    asm volatile(GT_MUL("q", "c1", "1") GT_MAD("s0", "vcc", "p", "s0") GT_MUL("p", "c2", "2") GT_MAD("s1", "%[k0]", "q", "s1")
                 GT_MUL("q", "c3", "3") GT_MAD("s2", "%[k1]", "p", "s2") GT_MAD("s3", "%[k2]", "q", "s3")
                 : [s0] "+&v"(S[0]), [s1] "+&v"(S[1]), [s2] "+&v"(S[2]), [s3] "+&v"(S[3]), [p] "+&v"(p), [q] "=&v"(q), [k0] "=&s"(k0), [k1] "=&s"(k1), [k2] "=&s"(k2)
                 : [c1] "v"(c[1]), [c2] "v"(c[2]), [c3] "v"(c[3]), [w] "v"(w), [m] "v"(m) : "vcc");
}

template <bool SWIGLU>
__global__ __launch_bounds__(256, 3) void gemm_q4k_q8_1_tiles_kernel(TileArgs A) {
  __shared__ __align__(16) unsigned char lds[GT_LDS];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);

  // Workgroup -> (pair of weight tiles, pair of batch tiles), as in gemm_mfma.hip: the workgroups that share weights run next to each other on one XCD.
  const int ngroups = SWIGLU ? A.tiles : (A.tiles + 1) >> 1, mgroups = (A.mtiles + 1) >> 1;
  const int per_xcd = (ngroups * mgroups + 7) >> 3;
  const int v = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || v >= ngroups * mgroups) return;
  const int ng = v / mgroups, mg = v - ng * mgroups;
  const int nb = A.nb, b0 = mg * 64, rows = min(64, A.B - b0), wrow = nb * 144, xrow = nb * 288;

  // weight tile i of the workgroup: its first row and how many rows of the matrix there are from there on
  const uint8_t* wbase[2];
  int wn[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int tile = SWIGLU ? ng : min(2 * ng + i, A.tiles - 1);
    const int m = SWIGLU ? i : tile >= A.tile_first[3] ? 3 : tile >= A.tile_first[2] ? 2 : tile >= A.tile_first[1] ? 1 : 0;
    const int n0 = (SWIGLU ? tile : tile - A.tile_first[m]) * 32;
    wbase[i] = A.g[m].W + (int64_t)n0 * wrow;
    wn[i] = A.g[SWIGLU ? 0 : m].N - n0;
  }
  const __amdgpu_buffer_rsrc_t xres = gt_rsrc(A.xq + (int64_t)b0 * xrow), wres0 = gt_rsrc(wbase[0]), wres1 = gt_rsrc(wbase[1]),
                               hres = wave >= 2 ? wres1 : wres0;
  // Copy maps.  Activations: 16 threads take the 16-byte pieces of a row (288 contiguous bytes with the scales), four rounds of 16 rows; the (d, s)
  // words eight threads a row, two rounds.  Weights: eight threads a row, a tile a round; its header four threads a row.  Rows past
  // the end repeat the last one (their results are not stored).
  const uint32_t xlane = ((t & 15) >> 1) * 36 + (t & 1) * 16, dlane = (t & 7) * 36 + 32;
  uint32_t xoff[4], doff[2];
#pragma unroll
  for (int i = 0; i < 4; i++) xoff[i] = min((t >> 4) + 16 * i, rows - 1) * xrow + xlane;
#pragma unroll
  for (int i = 0; i < 2; i++) doff[i] = min((t >> 3) + 32 * i, rows - 1) * xrow + dlane;
  const uint32_t woff0 = min(t >> 3, wn[0] - 1) * wrow + (t & 7) * 16 + 16, woff1 = min(t >> 3, wn[1] - 1) * wrow + (t & 7) * 16 + 16,
                 hoff = min((t >> 2) & 31, (wave >= 2 ? wn[1] : wn[0]) - 1) * wrow;
  uint4 xr0, xr1, xr2, xr3, wr0, wr1, hr;
  uint32_t dr0, dr1;
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const int xs = s * 288, ws = s * 144;
    xr0 = gt_load16(xres, xoff[0], xs);
    xr1 = gt_load16(xres, xoff[1], xs);
    xr2 = gt_load16(xres, xoff[2], xs);
    xr3 = gt_load16(xres, xoff[3], xs);
    wr0 = gt_load16(wres0, woff0, ws);
    wr1 = gt_load16(wres1, woff1, ws);
    dr0 = __builtin_amdgcn_raw_buffer_load_b32(xres, (int)doff[0], xs, 0);
    dr1 = __builtin_amdgcn_raw_buffer_load_b32(xres, (int)doff[1], xs, 0);
    hr = gt_load16(hres, hoff, ws);
  };
  const int xdst = GT_X + (t & 15) * 2 * GT_PLANE + (t >> 4) * 8, wdst = GT_W + (t & 7) * 2 * GT_PLANE + (t >> 3) * 8;
  const int rdst = GT_RAW + (t & 7) * GT_WORDS + (t >> 3) * 4;
  const int hrow = (t >> 2) & 31, part = t & 3, htile = wave >> 1;
  const int slot = (hrow & 3) * 8 + (hrow >> 4) * 4 + ((hrow >> 2) & 3);      // row 16 tn + 4 v + q -> [q][tn][v]
  const int sdst = GT_SC + htile * 256 + part * 64 + slot, mdst = GT_MIN + (htile * 8 + part * 2) * GT_WORDS + hrow * 4, ddst = GT_D + htile * 256 + slot * 8;
  auto stage = [&]() __attribute__((always_inline)) {
    auto put = [&](int at, const uint4& w) __attribute__((always_inline)) {
      *(uint2*)(lds + at) = make_uint2(w.x, w.y);
      *(uint2*)(lds + at + GT_PLANE) = make_uint2(w.z, w.w);
    };
    put(xdst, xr0);
    put(xdst + 128, xr1);
    put(xdst + GT_XT, xr2);
    put(xdst + GT_XT + 128, xr3);
    put(wdst, wr0);
    put(wdst + GT_WT, wr1);
    *(uint32_t*)(lds + rdst) = dr0;
    *(uint32_t*)(lds + rdst + 8 * GT_WORDS) = dr1;
    *(int*)(lds + rdst + GT_M8 - GT_RAW) = (int)fma(half_to_f32((uint16_t)dr0), 16777216.0f, 0.0f);
    *(int*)(lds + rdst + GT_M8 - GT_RAW + 8 * GT_WORDS) = (int)fma(half_to_f32((uint16_t)dr1), 16777216.0f, 0.0f);
    const bool outside = __ballot((dr0 & 0xffffu) >= 0x4400u) != 0 || __ballot((dr1 & 0xffffu) >= 0x4400u) != 0;
    const bool large = __ballot((dr0 & 0x7fffu) >= 0x5800u) != 0 || __ballot((dr1 & 0x7fffu) >= 0x5800u) != 0;
    *(int*)(lds + GT_FLAG + wave * 4) = large ? 3 : outside;
    const int sh = 16 * (part & 1);
    const uint32_t y = hr.y >> sh, z = hr.z >> sh, w = hr.w >> sh, low = part >= 2 ? 0x0f0fu : 0x3f3fu, high = 0x3f3fu ^ low;
    const uint32_t sc = ((part >= 2 ? w : y) & low) | ((y >> 2) & high), mn = ((part >= 2 ? w >> 4 : z) & low) | ((z >> 2) & high);
    const float dneg = -half_to_f32((uint16_t)(hr.x >> 16));
    lds[sdst] = (unsigned char)sc;
    lds[sdst + 32] = (unsigned char)(sc >> 8);
    *(float*)(lds + mdst) = dneg * (float)(mn & 0xffu);
    *(float*)(lds + mdst + GT_WORDS) = dneg * (float)((mn >> 8) & 0xffu);
    *(double*)(lds + ddst) = (double)half_to_f32((uint16_t)(hr.x & 0xffffu));
  };

  const int nt = wave >> 1, mt = wave & 1;
  const bool active = (SWIGLU || 2 * ng + nt < A.tiles) && b0 + 32 * mt < A.B;
  const int half = lane >> 5, col = lane & 31, q4 = lane >> 4, l16 = lane & 15;
  f64x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i >> 1][i & 1] = (f64x4_t){0.0, 0.0, 0.0, 0.0};
  const unsigned char* const pw = lds + GT_W + nt * GT_WT + q4 * GT_PLANE + (4 * (l16 & 3) + (l16 >> 2)) * 8;
  const unsigned char* const px = lds + GT_X + mt * GT_XT + q4 * GT_PLANE + l16 * 8;
  const unsigned char* const ps = lds + GT_SC + nt * 256 + q4 * 8;
  const unsigned char* const pm = lds + GT_M8 + mt * 8 * GT_WORDS + l16 * 4;
  auto load_x = [&](int j, int tb) __attribute__((always_inline)) { return *(const int64_t*)(px + j * 4 * GT_PLANE + tb * 128); };
  auto load_w = [&](int p, int tn) __attribute__((always_inline)) { return *(const int64_t*)(pw + p * 4 * GT_PLANE + tn * 128); };
  auto load_s = [&](int j) __attribute__((always_inline)) { return *(const uint2*)(ps + j * 32); };
  auto load_m = [&](int j, int tb) __attribute__((always_inline)) { return *(const int*)(pm + j * GT_WORDS + tb * 64); };
  auto load_d = [&](int j, int tb) __attribute__((always_inline)) { return half_to_f32(*(const uint16_t*)(pm + GT_RAW - GT_M8 + j * GT_WORDS + tb * 64)); };
  auto nibbles = [](int64_t w, int odd) __attribute__((always_inline)) {
    uint32_t a = (uint32_t)w, b = (uint32_t)((uint64_t)w >> 32);
    if (odd) { a >>= 4; b >>= 4; }
    return (int64_t)(((uint64_t)(b & 0x0f0f0f0fu) << 32) | (a & 0x0f0f0f0fu));
  };
  auto mfma = [](int64_t w, int64_t x) __attribute__((always_inline)) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(w, x, (i32x4_t){0, 0, 0, 0}, 0, 0, 0); };
#define GT_SB __builtin_amdgcn_sched_barrier(0)

  // One super-block from LDS.  The fold, its ranges of scales and its forms for large ones are those of gemm_mfma.hip.  us for gate + up of 1024 x 6144 x 2048,
  // every unit of a kind: scales below 4 126 (there 154), up to 128 132 (163), above 174 (179), non-finite 201 (217).
  auto compute = [&]() __attribute__((always_inline)) {
    const int4 fl = *(const int4*)(lds + GT_FLAG);
    f64x4_t S1[2][2];
    // MODE 0: every scale in [0, 4), the sums start as a double's bits; 1: in (-128, 128); 2: d * 2^(24 - s) has to be formed first
    auto fold = [&](auto mode, int s) __attribute__((always_inline)) {
      constexpr int MODE = decltype(mode)::value;
      constexpr bool SMALL = MODE == 0;
      const float to_whole = MODE == 2 ? __builtin_bit_cast(float, (151 - s) << 23) : 0.0f;
      auto load_whole = [&](int j, int tb) __attribute__((always_inline)) { return MODE == 2 ? (int)(load_d(j, tb) * to_whole) : load_m(j, tb); };
      int64_t S[2][2][4];
      int64_t x0 = load_x(0, 0), x1 = load_x(0, 1), w0 = load_w(0, 0), w1 = load_w(0, 1), wn0 = 0, wn1 = 0;
      uint2 sc = load_s(0), scn = sc;
      int m0 = load_whole(0, 0), m1 = load_whole(0, 1), mn0 = 0, mn1 = 0;
      int64_t a = nibbles(w0, 0);
      i32x4_t c00 = mfma(a, x0), c01 = mfma(a, x1);
      a = nibbles(w1, 0);
      i32x4_t c10 = mfma(a, x0), c11 = mfma(a, x1);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (j < 7) {
          x0 = load_x(j + 1, 0); x1 = load_x(j + 1, 1);
          scn = load_s(j + 1);
          mn0 = load_whole(j + 1, 0); mn1 = load_whole(j + 1, 1);
          if (j % 2 == 0 && j < 6) { wn0 = load_w(j / 2 + 1, 0); wn1 = load_w(j / 2 + 1, 1); }
        }
        GT_SB;
        i32x4_t n00, n01, n10, n11;
        if (j == 0) { gt_fold4<true, SMALL>(S[0][0], c00, sc.x, m0); gt_fold4<true, SMALL>(S[0][1], c01, sc.x, m1); }
        else { gt_fold4<false, SMALL>(S[0][0], c00, sc.x, m0); gt_fold4<false, SMALL>(S[0][1], c01, sc.x, m1); }
        GT_SB;
        if (j < 7) { a = j & 1 ? nibbles(wn0, 0) : nibbles(w0, 1); n00 = mfma(a, x0); n01 = mfma(a, x1); }
        GT_SB;
        if (j == 0) { gt_fold4<true, SMALL>(S[1][0], c10, sc.y, m0); gt_fold4<true, SMALL>(S[1][1], c11, sc.y, m1); }
        else { gt_fold4<false, SMALL>(S[1][0], c10, sc.y, m0); gt_fold4<false, SMALL>(S[1][1], c11, sc.y, m1); }
        GT_SB;
        if (j < 7) {
          a = j & 1 ? nibbles(wn1, 0) : nibbles(w1, 1);
          n10 = mfma(a, x0); n11 = mfma(a, x1);
          c00 = n00; c01 = n01; c10 = n10; c11 = n11; sc = scn; m0 = mn0; m1 = mn1;
          if (j & 1) { w0 = wn0; w1 = wn1; }
        }
        GT_SB;
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int64_t T = S[i >> 1][i & 1][u];
          S1[i >> 1][i & 1][u] = SMALL ? __builtin_bit_cast(double, T) - 0x1.8p28 : ldexp(fma((double)(int)(T >> 32), 4294967296.0, (double)(uint32_t)T), s - 24);
        }
    };
    const int kind = __builtin_amdgcn_readfirstlane(fl.x | fl.y | fl.z | fl.w);
    if (__builtin_expect(kind == 0, 1)) {
      fold(std::integral_constant<int, 0>{}, 0);
    } else if (kind == 1) {
      fold(std::integral_constant<int, 1>{}, 0);
    } else {
      uint32_t top = 0, low = 0xffffu;      // the largest scale and the smallest that is not zero, less one
#pragma unroll 1
      for (int i = 0; i < 16; i++) {
        const uint32_t d = *(const uint16_t*)(pm + GT_RAW - GT_M8 + (i >> 1) * GT_WORDS + (i & 1) * 64) & 0x7fffu;
        top = max(top, d);
        low = min(low, d - 1u);
      }
      const int wtop = __builtin_amdgcn_readfirstlane((int)wave_max((float)top)), wlow = 1 - __builtin_amdgcn_readfirstlane((int)wave_max(-(float)low));
      const int s = max((wtop >> 10) - 21, 0);
      const bool in_double = wtop >= 0x7c00 || (s > 0 && wlow < ((s + 1) << 10));
      if (!in_double) {
        fold(std::integral_constant<int, 2>{}, s);
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) S1[i >> 1][i & 1] = (f64x4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
        for (int j = 0; j < 8; j++) {
          const uint2 sc = load_s(j);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const i32x4_t c = mfma(nibbles(load_w(j >> 1, i >> 1), j & 1), load_x(j, i & 1));
            const double d8 = (double)load_d(j, i & 1);
#pragma unroll
            for (int u = 0; u < 4; u++)
              S1[i >> 1][i & 1][u] = fma(d8, (double)__mul24(c[u], (int)(((i >> 1 ? sc.y : sc.x) >> (8 * u)) & 0xffu)), S1[i >> 1][i & 1][u]);
          }
        }
      }
    }
    const double2* dd = (const double2*)(lds + GT_D + nt * 256 + q4 * 64);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const double2 w = dd[i];
      const int tn = i >> 1, u = 2 * (i & 1);
#pragma unroll
      for (int tb = 0; tb < 2; tb++) {
        acc[tn][tb][u] = fma(w.x, S1[tn][tb][u], acc[tn][tb][u]);
        acc[tn][tb][u + 1] = fma(w.y, S1[tn][tb][u + 1], acc[tn][tb][u + 1]);
      }
    }
    double am[2][2], bm[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        am[i][k] = (double)*(const float*)(lds + GT_MIN + (nt * 8 + q4 + 4 * k) * GT_WORDS + (16 * i + l16) * 4);
        bm[i][k] = (double)half_to_f32(*(const uint16_t*)(lds + GT_RAW + (mt * 8 + q4 + 4 * k) * GT_WORDS + (16 * i + l16) * 4 + 2));
      }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int i = 0; i < 4; i++) acc[i >> 1][i & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(am[i >> 1][k], bm[i & 1][k], acc[i >> 1][i & 1], 0, 0, 0);
  };

  fetch(0);
  for (int s = 0; s < nb; s++) {
    stage();
    GT_SB;
    __syncthreads();
    if (s + 1 < nb) fetch(s + 1);
    GT_SB;
    if (active) compute();
    GT_SB;
    __syncthreads();
  }

  float* const tile = (float*)lds + wave * 32 * GT_PITCH;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int u = 0; u < 4; u++) tile[(16 * (i & 1) + l16) * GT_PITCH + 16 * (i >> 1) + 4 * u + q4] = (float)acc[i >> 1][i & 1][u];
  __syncthreads();
  if (SWIGLU) {
    // a thread takes eight consecutive weight rows of one batch row, four neighbouring lanes a Q8_1 block (gemm_mfma.hip)
    const int g8 = lane & 3, b = t >> 2, N = A.g[0].N, n0 = ng * 32;
    const float *const gate = (const float*)lds + b * GT_PITCH + 8 * g8, *const up = gate + 64 * GT_PITCH;
    float f[8];
    uint32_t a2[4];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float gv = gate[i], uv = up[i];
      const uint16_t a16 = f32_to_bf16(__fmul_rn(__fmul_rn(gv, sigmoid_f64(gv)), uv));
      f[i] = bf16_to_f32(a16);
      a2[i >> 1] = i & 1 ? a2[i >> 1] | ((uint32_t)a16 << 16) : a16;
    }
    uint32_t pk[2];
    const uint32_t ds = quad_q8_1(f, pk);
    if (b < rows) {
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
  if (!active) return;
  const int wt = 2 * ng + nt, m = wt >= A.tile_first[3] ? 3 : wt >= A.tile_first[2] ? 2 : wt >= A.tile_first[1] ? 1 : 0;
  void* const out = A.g[m].out;
  const uint16_t* const res = A.g[m].res;
  const int N = A.g[m].N, epi = A.g[m].epi, n0 = (wt - A.tile_first[m]) * 32, first = b0 + 32 * mt, B = min(32, A.B - first);
  const bool n_ok = n0 + col < N;
  const int64_t o0 = (int64_t)first * N + n0 + col;
  float y[16];
#pragma unroll
  for (int i = 0; i < 16; i++) y[i] = tile[(2 * i + half) * GT_PITCH + col];
  if (epi == GEPI_F32) {
#pragma unroll
    for (int i = 0; i < 16; i++)
      if (n_ok && 2 * i + half < B) ((float*)out)[o0 + (int64_t)(2 * i + half) * N] = y[i];
  } else if (epi == GEPI_BF16) {
#pragma unroll
    for (int i = 0; i < 16; i++)
      if (n_ok && 2 * i + half < B) ((uint16_t*)out)[o0 + (int64_t)(2 * i + half) * N] = f32_to_bf16(y[i]);
  } else {
    uint16_t rv[16];
#pragma unroll
    for (int i = 0; i < 16; i++) rv[i] = n_ok && 2 * i + half < B ? res[o0 + (int64_t)(2 * i + half) * N] : (uint16_t)0;
#pragma unroll
    for (int i = 0; i < 16; i++)
      if (n_ok && 2 * i + half < B) ((uint16_t*)out)[o0 + (int64_t)(2 * i + half) * N] = f32_to_bf16(bf16_to_f32(f32_to_bf16(y[i])) + bf16_to_f32(rv[i]));
  }
}

int g_tune_gemm_tiles = -1;      // 0: never, 1: always, -1: from the shape

// Where this kernel is the faster one.  Its time goes by the workgroups per CU, rounded up (three run at a time); that of gemm_mfma.hip by tiles per CU,
// finer by four (by two with SwiGLU).  us at K = 1024 / 2048 / 6144, gemm_mfma.hip -> here, by workgroups per CU with every tile in use:
//   one (1024 x 1024 rows): 11.3 -> 12.1, 16.9 -> 19.6, 40.5 -> 51.8; two (2048): 17.4 -> 16.0, 28.2 -> 27.4, 71.0 -> 72.3 (K = 3072 43.2 -> 43.0, 4096 53.8 -> 54.1);
//   three (3072): 24.9 -> 21.4, 41.1 -> 36.0, 107 -> 95.7; four (4096): 30.8 -> 26.7, 52.1 -> 46.3, 135 -> 127; six (6144): 44.2 -> 36.5, 73.1 -> 64.2, 201 -> 178;
// in microseconds at K = 2048, 3.0 per tile and CU + 5 there against 9.3 per workgroup + 8.5 here: tiles left over from an odd
// number of either side (12288 at 160 rows: 8 tiles, 3 workgroups a CU: 29.4 -> 34.6) must leave 4 tiles > 13 workgroups + 4.
// (Long rows on two workgroups, and on seven with 24 tiles (5952 at 1056 rows, K = 2048 / 4096 / 6144: 83.6 -> 82.3, 146 -> 148, 210 -> 215), are 1 to 3 % slower
// here by themselves.  In prompts, whose chunks overlap on two streams, it goes either way: with two workgroups left to gemm_mfma.hip above K = 4096, 2999 tokens in
// the forms for throughput take 5.54 ms instead of 5.48, 2048 tokens in the default ones 24.9 instead of 25.2.)
// SwiGLU, pairs of tiles: two (1024): 18.6 -> 16.9, 29.4 -> 28.5, 71.8 -> 73.3 (K = 4096 51.1 -> 51.1); three (1536): 33.0 -> 22.8, 48.8 -> 37.6, 116 -> 99.0; four (2048): 36.3 -> 28.9, 60.6 -> 48.6, 161 -> 128;
// seven (3584): 58.1 -> 44.1, 97.5 -> 77.6, 256 -> 209; three pairs on two workgroups 18.5 -> 17.3, 28.6 -> 28.0, 60.4 -> 71.3 (left to gemm_mfma.hip),
// four on three (6144 at 160 rows) 20.2 -> 22.4, 31.0 -> 36.9, 74.5 -> 93.5, seven on four (3584 at 512) 34.8 -> 29.3, 54.9 -> 48.0, 139 -> 127.
bool gemm_tiles_pay(int tiles, int batch, int nb, bool swiglu) {
  if (nb > 65536) return false;                                      // offsets inside a workgroup's 64 rows are 32-bit
  if (g_tune_gemm_tiles >= 0) return g_tune_gemm_tiles != 0;
  const int64_t cus = num_cus(), bt = (batch + 31) / 32;
  const int64_t per_cu = (tiles * bt + cus - 1) / cus, wgs = ((swiglu ? tiles : (tiles + 1) / 2) * ((bt + 1) / 2) + cus - 1) / cus;
  if (swiglu) return wgs >= 2 && per_cu >= 2 * wgs - (wgs >= 3);
  return wgs >= 2 && 4 * per_cu > 13 * wgs + 4;
}

static unsigned tiles_grid(int64_t groups, int mtiles) { return (unsigned)(8 * ((groups * ((mtiles + 1) / 2) + 7) / 8)); }

// The callers have checked the arguments (gemm_mfma.hip).
int launch_gemm_tiles(const void* xq, int nb, int batch, int n, const void* const* W, void* const* out, const void* const* res, const int* N, const int* epi) {
  TileArgs A{};
  A.xq = (const uint8_t*)xq; A.nb = nb; A.B = batch;
  int tiles = 0;
  for (int i = 0; i < n; i++) {
    A.g[i].W = (const uint8_t*)W[i]; A.g[i].out = out[i]; A.g[i].res = (const uint16_t*)res[i]; A.g[i].N = N[i]; A.g[i].epi = epi[i];
    A.tile_first[i] = tiles;
    tiles += (N[i] + 31) / 32;
  }
  for (int i = n; i < 4; i++) A.tile_first[i] = tiles;
  A.tiles = tiles; A.mtiles = (batch + 31) / 32;
  hipLaunchKernelGGL((gemm_q4k_q8_1_tiles_kernel<false>), dim3(tiles_grid((tiles + 1) / 2, A.mtiles)), dim3(256), 0, stream(), A);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

int launch_gemm_swiglu_tiles(const void* xq, int nb, int batch, const void* Wg, const void* Wu, int N, void* act, void* act_q8) {
  TileArgs A{};
  A.xq = (const uint8_t*)xq; A.nb = nb; A.B = batch;
  A.g[0].W = (const uint8_t*)Wg; A.g[0].out = act; A.g[0].N = N;
  A.g[1].W = (const uint8_t*)Wu; A.g[1].N = N;
  A.out_q8 = (uint8_t*)act_q8;
  A.tiles = N / 32; A.mtiles = (batch + 31) / 32;
  hipLaunchKernelGGL((gemm_q4k_q8_1_tiles_kernel<true>), dim3(tiles_grid(A.tiles, A.mtiles)), dim3(256), 0, stream(), A);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

}  // namespace bk
