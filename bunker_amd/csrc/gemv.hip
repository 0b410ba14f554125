// Q4_K dequant-GEMV kernels for gfx950: y[N] = W[N,K] . x[K], W in 144-byte
// super-blocks, streamed once from HBM with 128-bit loads.
//
// Lane mapping (all kernels here).  A wavefront walks whole weight rows.  The
// 128 nibble bytes of a super-block are 8 chunks of 16 bytes; "slot"
// s = 64*round + lane covers chunk c = s & 7 of block s >> 3, so one wave-wide
// 16-byte load fetches the nibbles of 8 consecutive blocks (1 KiB contiguous
// but for the 16-byte headers, which a second, 8-way broadcast load fetches).
// Chunk c holds, for l in [16*(c&1), 16*(c&1)+16), the low nibbles of
// sub-block 2*(c>>1) and the high nibbles of sub-block 2*(c>>1)+1.  The slice
// of the activation a lane needs therefore depends on the lane only, not on
// the row: it is loaded once into registers and reused for every row.
//
// Arithmetic.  The sub-block dots are exact int32.  Everything after them is carried
// in double: d*d8 (two fp16 values) is exact in f32, times the 6-bit scale and the
// integer dot it is exact in double, so a row's value is a sum of exactly known terms
// with ~1e-16 relative accumulation error, rounded once to f32.  The result therefore
// does not depend on the lane mapping, the launch shape or the batch size, and equals
// a plain host loop in double to the bit (up to ~1e-8 probability per output).
#include "gemv_tile.h"

namespace bk {

// NR = number of 64-slot rounds per row (K = 2048*NR when the row fills every round);
// RPI = rows a wave handles per step (all their loads are issued before any is consumed).
template <int NR, int EPI, int RPI>
__global__ __launch_bounds__(GEMV_WAVES * 64) void gemv_q4k_q8_1_kernel(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ xq_all, void* __restrict__ y,
    const uint16_t* __restrict__ res, int N, int nb) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * GEMV_WAVES + (threadIdx.x >> 6);
  const int nwaves = gridDim.x * GEMV_WAVES;
  const int bidx = blockIdx.y;
  const uint8_t* xq = xq_all + (int64_t)bidx * nb * 8 * 36;
  const int c = lane & 7;
  const ScaleSel sel = make_scale_sel(c);
  const int64_t row_bytes = (int64_t)nb * 144;
  const int64_t ybase = (int64_t)bidx * N;
  const bool odd = c & 1;
  const int step = nwaves * RPI;
  int row0 = wave * RPI;

  int boff[NR];   // byte offset of the slot's block inside a row
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int blk = r * 8 + (lane >> 3);
    boff[r] = (blk < nb ? blk : 0) * 144;
  }
  RowTile<NR, RPI> t0;
  XQ x[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int blk = r * 8 + (lane >> 3);
    load_xq(x[r], xq, blk, c, blk < nb);
  }

  for (; row0 < N; row0 += step) {
    load_rows<NR, RPI>(t0, W, row_bytes, row0, N, boff, c);
    fold_rows<NR, EPI, RPI>(t0, x, sel, odd, lane, y, res, ybase, row0, N);
  }
}

// ---------------------------------------------------------------- rows through LDS
// Same lane mapping and arithmetic as above, but the weight bytes travel HBM -> registers ->
// LDS -> registers: a step's RPI rows are contiguous in memory (RPI * NR * 72 pieces of 16 bytes),
// so the wave fetches them with fully coalesced loads (lane l takes piece l, l + 64, ...: every
// 128-byte line is requested exactly once and no header is fetched eight times), parks them in
// its private LDS tile and reads headers and nibble chunks back in the (block, chunk) mapping.
// The loads of the next step are in flight while the current step is folded.
template <int NR, int EPI, int RPI>
__global__ __launch_bounds__(GEMV_WAVES * 64) void gemv_q4k_q8_1_lds_kernel(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ xq_all, void* __restrict__ y,
    const uint16_t* __restrict__ res, int N) {
  constexpr int PIECES = RPI * NR * 72;
  __shared__ uint4 tiles[GEMV_WAVES][PIECES];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wave = blockIdx.x * GEMV_WAVES + wv;
  const int nwaves = gridDim.x * GEMV_WAVES;
  const int bidx = blockIdx.y;
  constexpr int nb = NR * 8;
  const uint8_t* xq = xq_all + (int64_t)bidx * nb * 8 * 36;
  const int c = lane & 7, b = lane >> 3;
  const ScaleSel sel = make_scale_sel(c);
  constexpr int64_t row_bytes = (int64_t)nb * 144;
  const int64_t last_piece_off = (int64_t)N * row_bytes - 16;
  const int64_t ybase = (int64_t)bidx * N;
  const bool odd = c & 1;
  const int step = nwaves * RPI;
  int row0 = wave * RPI;
  uint4* tile = tiles[wv];

  // the activation slice first, the weight rows right behind it: loads return in issue order, and the slice
  // (cache-resident) must not queue up behind rows that come from HBM
  XQ x[NR];
#pragma unroll
  for (int r = 0; r < NR; r++) load_xq(x[r], xq, r * 8 + b, c, true);

  StageRegs<NR, RPI> g;
  stage_load<NR, RPI>(g, W, (int64_t)min(row0, N - 1) * row_bytes, last_piece_off, lane);

  while (row0 < N) {
    stage_park<NR, RPI>(g, tile, lane);
    if (row0 + step < N) stage_load<NR, RPI>(g, W, (int64_t)(row0 + step) * row_bytes, last_piece_off, lane);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    RowTile<NR, RPI> t;
#pragma unroll
    for (int i = 0; i < RPI; i++) {
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const int blk = (i * NR + r) * 72 + b * 9;       // piece index of the block header
        t.hdr[i][r] = tile[blk];
        t.q[i][r] = tile[blk + 1 + c];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();                     // every lane has read its pieces before the tile is overwritten
    fold_rows<NR, EPI, RPI>(t, x, sel, odd, lane, y, res, ybase, row0, N);
    row0 += step;
  }
}

// Rows that do not fill whole rounds (K is no multiple of 2048).  The super-blocks of a step's RPI rows are numbered through, slot group
// b of round r takes number 8 r + b, whichever row that is in: S rounds for all of them, S = ceil(RPI nb / 8), where rounds row by row
// would leave up to half of the lanes without work.  A lane's activation slices still depend on the lane alone.  nb lies between NB0
// and NB1 = 8 S / RPI, so that most rounds are known to lie in one row; in the others a lane adds its term to the row it is in.
// Bound by the instructions of a round (about 70 for 64 slots) and the waves that the registers allow, no longer by idle lanes: 1.5 to 2 times the
// rounds made K = 4608 with 67527 rows 43.9 us (4.0 TB/s), here 31.4 (5.6); K = 2560, 100000 rows 34.0 -> 26.1 (5.5 TB/s).  Without the activation row
// through LDS, with a grid of two steps a wave and all of a step's operands in registers at once (a wave a SIMD less): 38.8 and 30.2.
// Waves a SIMD that the registers allow (what a lane keeps for the slots is ten registers a round).  S = 6 with two rows takes 138: held to 128, for four
// waves, it parked a piece of the next step's weights in scratch as it arrived, and a wave waited for it before it folded the step at hand
// (5376 x 54000 39.4 us direct, 32.5 so, 29.1 with three waves).
constexpr int flat_waves(int S) { return S <= 1 ? 8 : S == 2 ? 6 : S == 3 ? 5 : S <= 5 ? 4 : 3; }
template <int S, int RPI, int EPI>
__global__ __launch_bounds__(GEMV_WAVES * 64, flat_waves(S)) void gemv_q4k_q8_1_flat_kernel(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ xq_all, void* __restrict__ y,
    const uint16_t* __restrict__ res, int N, int nb) {
  constexpr int NB1 = 8 * S / RPI, NB0 = 8 * (S - 1) / RPI + 1;
  static_assert(RPI == 2 || RPI == 4, "the sums of two or four rows share their steps");
  __shared__ uint4 tiles[GEMV_WAVES][S * 72];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wave = blockIdx.x * GEMV_WAVES + wv;
  const int bidx = blockIdx.y;
  const uint8_t* xq = xq_all + (int64_t)bidx * nb * 8 * 36;
  const int c = lane & 7, b = lane >> 3;
  const ScaleSel sel = make_scale_sel(c);
  const int64_t row_bytes = (int64_t)nb * 144, last_piece_off = (int64_t)N * row_bytes - 16, ybase = (int64_t)bidx * N;
  const bool odd = c & 1;
  const int step = gridDim.x * GEMV_WAVES * RPI, pieces = RPI * nb * 9;
  int row0 = wave * RPI;
  uint4* tile = tiles[wv];

  constexpr int LOADS = (S * 72 + 63) / 64;
  uint4 g[LOADS];
  auto load = [&](int row) __attribute__((always_inline)) {
    const uint8_t* rp = W + (int64_t)row * row_bytes;
    const int last = (int)min((int64_t)(pieces - 1), (last_piece_off - (int64_t)row * row_bytes) >> 4);      // past the step or the matrix: its last piece again
#pragma unroll
    for (int u = 0; u < LOADS; u++) g[u] = load_w16(rp + min(lane + 64 * u, last) * 16);
  };
  // the activation row goes through LDS once per workgroup, its loads ahead of those of the weights (loads return in issue order); a row is
  // at most 18 NB1 pieces of 16 bytes, 4-byte aligned
  __shared__ __align__(16) uint32_t xl[NB1 * 72];
  constexpr int XLOADS = (NB1 * 72 + 255) / 256;
  uint32_t xr[XLOADS];
#pragma unroll
  for (int u = 0; u < XLOADS; u++) xr[u] = ((const uint32_t*)xq)[min((int)threadIdx.x + 256 * u, nb * 72 - 1)];
  load(min(row0, N - 1));
#pragma unroll
  for (int u = 0; u < XLOADS; u++)
    if ((int)threadIdx.x + 256 * u < NB1 * 72) xl[threadIdx.x + 256 * u] = xr[u];
  __syncthreads();
  XQ x[S];
  int in_row[S];                 // the row of the step; past the last one: RPI
#pragma unroll
  for (int r = 0; r < S; r++) {
    const int f = 8 * r + b;
    in_row[r] = f / nb;
    load_xq(x[r], (const uint8_t*)xl, f - in_row[r] * nb, c, in_row[r] < RPI);
  }

  while (row0 < N) {
#pragma unroll
    for (int u = 0; u < LOADS; u++)
      if (64 * u + 63 < S * 72 || lane + 64 * u < S * 72) tile[lane + 64 * u] = g[u];
    if (row0 + step < N) load(row0 + step);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double acc[RPI];
#pragma unroll
    for (int i = 0; i < RPI; i++) acc[i] = 0.0;
#pragma unroll
    for (int r = 0; r < S; r++) {
      int I0, I1;
      const uint4 hdr = tile[(8 * r + b) * 9], q = tile[(8 * r + b) * 9 + 1 + c];
      const double t = slot_dot(hdr, q, x[r], sel, I0, I1, odd);
      const int first = 8 * r / NB1, last = min((8 * r + 7) / NB0, RPI);      // rows that the round can lie in
#pragma unroll
      for (int i = 0; i < RPI; i++)
        if (i >= first && i <= last) acc[i] += first == last || in_row[r] == i ? t : 0.0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();                     // every lane has read its pieces before the tile is overwritten
    double tot;
    if constexpr (RPI == 4) tot = wave_sum4_f64(acc[0], acc[1], acc[2], acc[3], lane);
    else tot = wave_sum2_f64(acc[0], acc[1], lane);
    const int row = row0 + (RPI == 4 ? 2 * (lane & 1) + ((lane >> 1) & 1) : (lane & 1));
    if (lane < RPI && row < N) store_out<EPI>(y, res, ybase + row, (float)tot);
    row0 += step;
  }
}

// Any K that is a multiple of 256: rounds are a run-time loop and the activation
// slice is re-read (from L2) in every round.
template <int EPI>
__global__ __launch_bounds__(GEMV_WAVES * 64) void gemv_q4k_q8_1_generic_kernel(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ xq_all, void* __restrict__ y,
    const uint16_t* __restrict__ res, int N, int nb) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * GEMV_WAVES + (threadIdx.x >> 6);
  const int nwaves = gridDim.x * GEMV_WAVES;
  const int bidx = blockIdx.y;
  const uint8_t* xq = xq_all + (int64_t)bidx * nb * 8 * 36;
  const int c = lane & 7;
  const ScaleSel sel = make_scale_sel(c);
  const int64_t row_bytes = (int64_t)nb * 144;
  const int rounds = (nb + 7) / 8;
  for (int row = wave; row < N; row += nwaves) {
    const uint8_t* rp = W + (int64_t)row * row_bytes;
    double acc = 0.0;
    for (int r = 0; r < rounds; r++) {
      const int blk = r * 8 + (lane >> 3);
      const bool active = blk < nb;
      XQ x;
      load_xq(x, xq, blk, c, active);
      const int bo = (active ? blk : 0) * 144;
      const uint4 hdr = *(const uint4*)(rp + bo);
      const uint4 q = *(const uint4*)(rp + bo + 16 + 16 * c);
      int I0, I1;
      acc += slot_dot(hdr, q, x, sel, I0, I1, c & 1);
    }
    const float tot = (float)wave_sum_f64(acc);
    if (lane == 0) store_out<EPI>(y, res, (int64_t)bidx * N + row, tot);
  }
}

// Exact int32 sub-block dots I[N, 8*nb]: lane pairs (c even, c odd) hold the two
// 16-element halves of sub-blocks 2g and 2g+1.
__global__ __launch_bounds__(GEMV_WAVES * 64) void q4k_q8_1_subdots_kernel(
    const uint8_t* __restrict__ W, const uint8_t* __restrict__ xq, int32_t* __restrict__ I, int N, int nb) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * GEMV_WAVES + (threadIdx.x >> 6);
  const int nwaves = gridDim.x * GEMV_WAVES;
  const int c = lane & 7;
  const ScaleSel sel = make_scale_sel(c);
  const int64_t row_bytes = (int64_t)nb * 144;
  const int rounds = (nb + 7) / 8;
  for (int row = wave; row < N; row += nwaves) {
    const uint8_t* rp = W + (int64_t)row * row_bytes;
    for (int r = 0; r < rounds; r++) {
      const int blk = r * 8 + (lane >> 3);
      const bool active = blk < nb;
      XQ x;
      load_xq(x, xq, blk, c, active);
      const int bo = (active ? blk : 0) * 144;
      const uint4 hdr = *(const uint4*)(rp + bo);
      const uint4 q = *(const uint4*)(rp + bo + 16 + 16 * c);
      int I0, I1;
      (void)slot_dot(hdr, q, x, sel, I0, I1, c & 1);
      const int s0 = I0 + dpp_i32<DPP_QUAD_XOR1>(I0);
      const int s1 = I1 + dpp_i32<DPP_QUAD_XOR1>(I1);
      if (active) I[(int64_t)row * nb * 8 + blk * 8 + c] = (c & 1) ? s1 : s0;
    }
  }
}

int g_tune_gemv_impl = 2;               // 2: rows staged through LDS when K is a multiple of 2048, else the rule of gemv_flat_rounds;
                                        // 3: the flat form wherever it exists; 0: direct loads in the (block, chunk) mapping
int g_tune_rpi = 0, g_tune_cap = 16;     // tuning hooks (bk_tune_set): rows per wave step (0: from the shape), workgroups per CU
int g_tune_steps = 0;                    // > 0: the grid that gives every wave this many row steps (the last one may be short)

// Workgroups for a launch that needs `wgs` of them at one row step per wave.  Up to the cap (16 per CU) that many; a
// longer matrix gets the grid in which every wave takes exactly two steps (the second one's rows are in flight while
// the first is folded).  Measured on the 151936 x 2048 matrix, four rows per step: one step per wave 28.9 us, two 27.4,
// three 28.7, four 29.4, eight 30.6, and 28.0-29.3 with the grid cut at the cap, where some waves take three steps and
// the rest two.
int gemv_grid_for(int wgs) {
  if (g_tune_steps > 0) return (wgs + g_tune_steps - 1) / g_tune_steps;
  const int cap = num_cus() * g_tune_cap;
  return wgs <= cap ? wgs : (wgs + 1) / 2;
}

static int gemv_grid(int N, int rows_per_wg) { return gemv_grid_for((N + rows_per_wg - 1) / rows_per_wg); }

template <int NR, int EPI>
static void launch_q8_1_rpi(dim3 block, const uint8_t* w, const uint8_t* x, void* y, const uint16_t* r, int N, int nb, int batch) {
  const int rpi = (g_tune_rpi == 1 || g_tune_rpi == 2) ? g_tune_rpi : 4;
  dim3 grid(gemv_grid(N, GEMV_WAVES * rpi), batch);
  if (rpi == 1) hipLaunchKernelGGL((gemv_q4k_q8_1_kernel<NR, EPI, 1>), grid, block, 0, stream(), w, x, y, r, N, nb);
  else if (rpi == 2) hipLaunchKernelGGL((gemv_q4k_q8_1_kernel<NR, EPI, 2>), grid, block, 0, stream(), w, x, y, r, N, nb);
  else { grid.x = gemv_grid(N, GEMV_WAVES * 4); hipLaunchKernelGGL((gemv_q4k_q8_1_kernel<NR, EPI, 4>), grid, block, 0, stream(), w, x, y, r, N, nb); }
}

template <int NR, int EPI>
static void launch_q8_1_lds(dim3 block, const uint8_t* w, const uint8_t* x, void* y, const uint16_t* r, int N, int batch) {
  // rows of 2048: two rows per wave step while the matrix is small (twice the workgroups in flight: qkv 3.95 -> 3.65 us,
  // gate+up 4.8 -> 4.7), four for a long one (lm_head: 29.8 us against 33 with two)
  const int rpi = NR == 1 ? ((g_tune_rpi == 2 || (g_tune_rpi == 0 && N <= 16384)) ? 2 : 4) : 2;
  dim3 grid(gemv_grid(N, GEMV_WAVES * rpi), batch);
  if (NR == 1 && rpi == 4) hipLaunchKernelGGL((gemv_q4k_q8_1_lds_kernel<NR, EPI, (NR == 1 ? 4 : 2)>), grid, block, 0, stream(), w, x, y, r, N);
  else hipLaunchKernelGGL((gemv_q4k_q8_1_lds_kernel<NR, EPI, 2>), grid, block, 0, stream(), w, x, y, r, N);
}

// As many workgroups as the chip holds at once, with the steps dealt out evenly.
template <int S, int RPI, int EPI>
static void launch_q8_1_flat(const uint8_t* w, const uint8_t* x, void* y, const uint16_t* r, int N, int nb, int batch) {
  const int64_t wgs = ((int64_t)N + GEMV_WAVES * RPI - 1) / (GEMV_WAVES * RPI), room = num_cus() * flat_waves(S);
  const int64_t steps = g_tune_steps > 0 ? g_tune_steps : (wgs * batch + room - 1) / room;
  hipLaunchKernelGGL((gemv_q4k_q8_1_flat_kernel<S, RPI, EPI>), dim3((unsigned)((wgs + steps - 1) / steps), batch), dim3(GEMV_WAVES * 64), 0, stream(), w, x, y, r, N, nb);
}

// Rounds a step, 10 S + RPI, of the flat form where it is the faster one, 0 where direct loads are: these start sooner (no pass through LDS), so launches of
// about one step a wave stay with them, the more rounds the flat form saves the fewer.  us by rows, direct -> flat (1024 SIMDs):
//   K =  512: 13000 5.3 -> 5.6, 26000 6.05 -> 5.3, 54000  9.8 ->  6.6, 100000 15.8 ->  9.9;  1024: 17000 5.7 -> 5.7, 26000 6.7 -> 6.45, 54000 10.4 -> 9.1, 100000 16.3 -> 12.6;
//   K = 1536: 33000 8.7 -> 8.9, 54000 11.5 -> 11.3, 100000 18.6 -> 16.9 (1792 saves no round and stays);  2304: 8000 6.5 -> 6.5, 13000 8.5 -> 7.9, 33000 14.6 -> 11.4, 100000 32.7 -> 25.1;
//   K = 3072: 8000 6.9 -> 6.9, 10000 7.7 -> 7.9, 13000 9.1 -> 8.4, 54000 22.3 -> 18.7;  3584: 8000 7.3 -> 7.4, 10000 8.0 -> 8.7, 13000 9.8 -> 9.2, 86820 38.1 -> 31.4;
//   K = 3840: 17000 11.7 -> 12.6, 26000 15.2 -> 16.2, 33000 17.9 -> 16.7, 81032 36.6 -> 31.3;  4608: 4000 7.3 -> 6.1, 8000 8.7 -> 8.7, 13000 12.1 -> 10.9, 67527 43.9 -> 31.4;
//   K = 5120: 13000 12.6 -> 11.1, 60774 40.2 -> 30.3;  5888: 1500 7.0 -> 4.95, 4000 8.25 -> 6.9, 8000 9.45 -> 8.9, 13000 13.35 -> 12.8, 54000 41.3 -> 31.0.
static int gemv_flat_rounds(int nb, int N, int batch) {
  if (nb % 8 == 0 || nb == 7 || nb > 23) return 0;
  const int rpi = nb < 16 ? 4 : 2, S = (rpi * nb + 7) / 8;
  const int64_t wgs = ((int64_t)N + GEMV_WAVES * rpi - 1) / (GEMV_WAVES * rpi) * batch, cus = num_cus();
  bool pays = true;
  if (S == 1) pays = wgs > 5 * cus;
  else if (S == 2) pays = wgs > 6 * cus;
  else if (S == 3) pays = wgs > 15 * cus;
  else if (S == 6 && rpi == 4) pays = wgs <= 2 * cus || wgs > flat_waves(S) * cus;
  else if (S == 7) pays = wgs > 3 * cus;
  else if (S == 8) pays = wgs > 7 * cus;
  return pays || g_tune_gemv_impl == 3 ? 10 * S + rpi : 0;
}

template <int EPI>
static void launch_q8_1_variant(const void* W, const void* xq, void* y, const void* res, int N, int nb, int batch) {
  const int rounds = (nb + 7) / 8;
  dim3 block(GEMV_WAVES * 64);
  dim3 grid(1, batch);
  const uint8_t* w = (const uint8_t*)W; const uint8_t* x = (const uint8_t*)xq; const uint16_t* r = (const uint16_t*)res;
  switch (g_tune_gemv_impl == 0 ? 0 : gemv_flat_rounds(nb, N, batch)) {
    case 14: return launch_q8_1_flat<1, 4, EPI>(w, x, y, r, N, nb, batch);
    case 24: return launch_q8_1_flat<2, 4, EPI>(w, x, y, r, N, nb, batch);
    case 34: return launch_q8_1_flat<3, 4, EPI>(w, x, y, r, N, nb, batch);
    case 54: return launch_q8_1_flat<5, 4, EPI>(w, x, y, r, N, nb, batch);
    case 64: return launch_q8_1_flat<6, 4, EPI>(w, x, y, r, N, nb, batch);
    case 74: return launch_q8_1_flat<7, 4, EPI>(w, x, y, r, N, nb, batch);
    case 84: return launch_q8_1_flat<8, 4, EPI>(w, x, y, r, N, nb, batch);
    case 52: return launch_q8_1_flat<5, 2, EPI>(w, x, y, r, N, nb, batch);
    case 62: return launch_q8_1_flat<6, 2, EPI>(w, x, y, r, N, nb, batch);
  }
  switch (rounds) {
    case 1: if (g_tune_gemv_impl != 0 && nb == 8) launch_q8_1_lds<1, EPI>(block, w, x, y, r, N, batch); else launch_q8_1_rpi<1, EPI>(block, w, x, y, r, N, nb, batch);
      break;
    case 2: if (g_tune_gemv_impl != 0 && nb == 16) launch_q8_1_lds<2, EPI>(block, w, x, y, r, N, batch); else launch_q8_1_rpi<2, EPI>(block, w, x, y, r, N, nb, batch);
      break;
    case 3: if (g_tune_gemv_impl != 0 && nb == 24) launch_q8_1_lds<3, EPI>(block, w, x, y, r, N, batch); else launch_q8_1_rpi<3, EPI>(block, w, x, y, r, N, nb, batch);
      break;
    default:
      grid.x = gemv_grid(N, GEMV_WAVES);
      hipLaunchKernelGGL((gemv_q4k_q8_1_generic_kernel<EPI>), grid, block, 0, stream(), w, x, y, r, N, nb);
  }
}

int launch_gemv_q4k_q8_1(const void* W, const void* xq, void* y, int N, int K, int batch, int out_dtype,
                         const void* residual) {
  BK_REQUIRE(W && xq && y, "gemv_q4k_q8_1: null pointer");
  BK_REQUIRE(N > 0 && K > 0 && K % 256 == 0, "gemv_q4k_q8_1: K=%d must be a positive multiple of 256 (N=%d)", K, N);
  BK_REQUIRE(batch > 0 && batch <= 65535, "gemv_q4k_q8_1: bad batch=%d", batch);
  BK_REQUIRE(out_dtype == DT_F32 || out_dtype == DT_BF16, "gemv_q4k_q8_1: out_dtype must be 0 (f32) or 1 (bf16)");
  BK_REQUIRE(!(residual && out_dtype != DT_BF16), "gemv_q4k_q8_1: a residual needs bf16 output");
  BK_REQUIRE(((uintptr_t)W & 15) == 0 && ((uintptr_t)xq & 3) == 0, "gemv_q4k_q8_1: W must be 16-byte and xq 4-byte aligned");
  const int nb = K / 256;
  if (out_dtype == DT_F32) launch_q8_1_variant<EPI_F32>(W, xq, y, nullptr, N, nb, batch);
  else if (!residual) launch_q8_1_variant<EPI_BF16>(W, xq, y, nullptr, N, nb, batch);
  else launch_q8_1_variant<EPI_BF16_ADD>(W, xq, y, residual, N, nb, batch);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

int launch_q4k_q8_1_subdots(const void* W, const void* xq, int32_t* I, int N, int K) {
  BK_REQUIRE(W && xq && I, "q4k_q8_1_subdots: null pointer");
  BK_REQUIRE(N > 0 && K > 0 && K % 256 == 0, "q4k_q8_1_subdots: K=%d must be a positive multiple of 256", K);
  BK_REQUIRE(((uintptr_t)W & 15) == 0 && ((uintptr_t)xq & 3) == 0, "q4k_q8_1_subdots: misaligned pointer");
  hipLaunchKernelGGL(q4k_q8_1_subdots_kernel, dim3(gemv_grid(N, GEMV_WAVES)), dim3(GEMV_WAVES * 64), 0, stream(),
                     (const uint8_t*)W, (const uint8_t*)xq, I, N, K / 256);
  BK_LAUNCH_CHECK();
  return BK_OK;
}

// ---------------------------------------------------------------- f32 activations
// Dequantise-and-dot with x in f32: per slot, 16 low-nibble and 16 high-nibble
// weights against 32 activation values held in registers.
//   y += d*sc0*sum(nib_lo*x_lo) - dmin*m0*sum(x_lo) + d*sc1*sum(nib_hi*x_hi) - dmin*m1*sum(x_hi)
struct XF {
  float lo[16], hi[16];
  float sum_c;   // sum of the 32 activations of sub-block c (for the lane's share of the mins)
};

// Four bytes' low nibbles (SHIFT 0) or high ones (SHIFT 4) against four activations.  LIFTED: the activations are 2^24 times what they are.  A nibble alone in
// 16 bits is a subnormal half of 2^-24 times its value, which the mixed FMA reads as it is, in either half of a register: the products are the same numbers
// as those of a converted nibble and the activation itself, down to the smallest.
typedef __attribute__((ext_vector_type(2))) _Float16 half2_t;
template <int SHIFT, bool LIFTED>
__device__ __forceinline__ float nibdot4(uint32_t q, const float* x, float acc) {
  if constexpr (LIFTED) {
    const half2_t n02 = __builtin_bit_cast(half2_t, (q >> SHIFT) & 0x000f000fu), n13 = __builtin_bit_cast(half2_t, (q >> (SHIFT + 8)) & 0x000f000fu);
    acc = fmaf((float)n02[0], x[0], acc);
    acc = fmaf((float)n13[0], x[1], acc);
    acc = fmaf((float)n02[1], x[2], acc);
    acc = fmaf((float)n13[1], x[3], acc);
  } else {
    const uint32_t n4 = (q >> SHIFT) & 0x0f0f0f0fu;
    acc = fmaf((float)(n4 & 0xffu), x[0], acc);
    acc = fmaf((float)((n4 >> 8) & 0xffu), x[1], acc);
    acc = fmaf((float)((n4 >> 16) & 0xffu), x[2], acc);
    acc = fmaf((float)(n4 >> 24), x[3], acc);
  }
  return acc;
}

// Activations may be lifted where all are below XF_LIFT_BELOW (32 lifted ones still add up to less than 2^127).  Where all are below XF_TINY they are taken
// times XF_TINY_LIFT as well and the result is brought back, so that a row is rounded once below the normal range and not at every step.
constexpr float XF_LIFT = 0x1p24f, XF_LIFT_BELOW = 0x1p98f, XF_TINY = 0x1p-63f, XF_TINY_LIFT = 0x1p64f;

// The lane's 32 activations of super-block blk (taken from at(i), float4 i of the row; LIFTED: as lifted ones).  Lanes c and c ^ 1 hold the two halves of
// sub-blocks 2g and 2g+1, so the sum of sub-block c is the lane's own half plus its neighbour's.  Every lane of the wave takes part in the exchange.
template <bool LIFTED, typename AT>
__device__ __forceinline__ void load_xf(XF& x, AT at, int blk, int c, bool active) {
  const int g = c >> 1, half = c & 1;
  const int p0 = (active ? blk : 0) * 64 + 16 * g + 4 * half;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float4 a = at(p0 + i), b = at(p0 + 8 + i);
    x.lo[4 * i] = a.x; x.lo[4 * i + 1] = a.y; x.lo[4 * i + 2] = a.z; x.lo[4 * i + 3] = a.w;
    x.hi[4 * i] = b.x; x.hi[4 * i + 1] = b.y; x.hi[4 * i + 2] = b.z; x.hi[4 * i + 3] = b.w;
  }
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (!active) { x.lo[i] = 0.0f; x.hi[i] = 0.0f; }
    s0 += x.lo[i];
    s1 += x.hi[i];
  }
  s0 += dpp_f32<DPP_QUAD_XOR1>(s0);
  s1 += dpp_f32<DPP_QUAD_XOR1>(s1);
  x.sum_c = half ? s1 : s0;
  if (LIFTED) x.sum_c *= 1.0f / XF_LIFT;      // (exact: what is subnormal then has few enough bits)
}

template <bool LIFTED>
__device__ __forceinline__ float slot_dot_f32(const uint4& hdr, const uint4& q, const XF& x, const ScaleSel& sel) {
  const float d = half_to_f32((uint16_t)(hdr.x & 0xffffu));
  const float dmin = half_to_f32((uint16_t)(hdr.x >> 16));
  uint32_t sc, m;
  lane_scale_min(sel, hdr.y, hdr.z, hdr.w, sc, m);
  const float fsc = d * (float)sc;
  const float fm = (dmin * (float)m) * x.sum_c;
  float a = 0.0f, b = 0.0f;
  a = nibdot4<0, LIFTED>(q.x, &x.lo[0], a);
  b = nibdot4<4, LIFTED>(q.x, &x.hi[0], b);
  a = nibdot4<0, LIFTED>(q.y, &x.lo[4], a);
  b = nibdot4<4, LIFTED>(q.y, &x.hi[4], b);
  a = nibdot4<0, LIFTED>(q.z, &x.lo[8], a);
  b = nibdot4<4, LIFTED>(q.z, &x.hi[8], b);
  a = nibdot4<0, LIFTED>(q.w, &x.lo[12], a);
  b = nibdot4<4, LIFTED>(q.w, &x.hi[12], b);
  const float f0 = dpp_f32<DPP_PAIR_EVEN>(fsc);
  const float f1 = dpp_f32<DPP_PAIR_ODD>(fsc);
  return (f0 * a + f1 * b) - fm;
}

// One row of any length and any activations, by one wave: rounds are a run-time loop, the activation slice is re-read (from L2) in every round, so that
// lifting it (32 multiplications for one use) costs more than converting the nibbles (16 instructions): 4096 x 8192 11.4 -> 11.15 us, 2048 x 12288 9.75 -> 9.35.
__device__ __forceinline__ void row_dot_f32(const uint8_t* W, const float* xf, float* y, int row, int nb, int lane, const ScaleSel& sel) {
  const uint8_t* rp = W + (int64_t)row * nb * 144;
  const int c = lane & 7, rounds = (nb + 7) / 8;
  float acc = 0.0f;
  for (int r = 0; r < rounds; r++) {
    const int blk = r * 8 + (lane >> 3);
    XF x;
    load_xf<false>(x, [&](int i) { return ((const float4*)xf)[i]; }, blk, c, blk < nb);
    const int bo = (blk < nb ? blk : 0) * 144;
    uint4 hdr = *(const uint4*)(rp + bo);
    const uint4 q = *(const uint4*)(rp + bo + 16 + 16 * c);
    if (blk >= nb) hdr.x = 0;                             // past the row: d = dmin = 0
    float top = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) top = fmaxf(fmaxf(top, fabsf(x.lo[i])), fabsf(x.hi[i]));
    float down = 1.0f;
    if (__builtin_expect(!__any(top >= XF_TINY), 0)) {
#pragma unroll
      for (int i = 0; i < 16; i++) { x.lo[i] *= XF_TINY_LIFT; x.hi[i] *= XF_TINY_LIFT; }
      x.sum_c *= XF_TINY_LIFT;
      down = 1.0f / XF_TINY_LIFT;
    }
    acc += slot_dot_f32<false>(hdr, q, x, sel) * down;
  }
  const float tot = wave_sum(acc);
  if (lane == 0) y[row] = tot;
}

// Rows of up to 8 * NR super-blocks: the LDS staging of gemv_q4k_q8_1_lds_kernel (RPI contiguous rows per wave step,
// every 128-byte line requested once, the next step's rows in flight during the arithmetic), for any nb: the lanes past
// the row fold a clamped block, its scales and the activations replaced by zeros.  What bounds it is latency (launch, one memory round trip, x to the
// lanes, fold) up to a few thousand rows, then vector issue.  The workgroup reads x once and hands it to its four waves through LDS: read by every
// wave in 16-byte pieces 64 bytes apart, x was 33 MB through the caches for a 9.4 MB matrix, and the weights were only asked for behind it.  With that and
// the mixed FMAs (fifteen instructions for eight weights where conversions made it nineteen), us back to back on cold weights: 1024 x 1024 2.75 -> 2.6,
// 4096 x 4096 6.1 -> 5.15 (5.46 -> 4.31 on weights in the memory-side cache), 2048 x 6144 5.85 -> 4.6, 12288 x 2048 6.85 -> 5.7, 40000 x 1024 13.4 -> 10.6,
// 151936 x 2048 43.3 -> 37-41, 50000 x 6144 51.7 -> 41 (4.2 TB/s).  Activations are lifted (nibdot4) on their way into LDS; a vector with one that
// cannot be goes row by row behind the loop (in front of it, the loop's operands took 172 registers instead of 138).
template <int NR, int RPI>
__global__ __launch_bounds__(GEMV_WAVES * 64) void gemv_q4k_f32_lds_kernel(
    const uint8_t* __restrict__ W, const float* __restrict__ xf, float* __restrict__ y, int N, int nb, int nwg) {
  constexpr int LOADS = StageRegs<NR, RPI>::LOADS, TILE = StageRegs<NR, RPI>::PIECES, XLOADS = NR * 8 * 64 / (GEMV_WAVES * 64);
  __shared__ uint4 lds[GEMV_WAVES * TILE + NR * 8 * 64];
  __shared__ int4 range;           // per wave, of its share of x: 0 every activation tiny, 1 not, 3 one that cannot be lifted
  uint4* const xlds = lds + GEMV_WAVES * TILE;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int c = lane & 7, b = lane >> 3;
  const ScaleSel sel = make_scale_sel(c);
  const int row_pieces = nb * 9, tile_pieces = RPI * row_pieces;
  const int64_t last_piece = (int64_t)N * row_pieces - 1;
  const int step = nwg * GEMV_WAVES * RPI;
  int row0 = (blockIdx.x * GEMV_WAVES + wv) * RPI;
  uint4* tile = lds + wv * TILE;

  XF x[NR];
  uint32_t in_row[NR];            // all ones, or zero past the row: a lane there has d = dmin = 0 and adds nothing, whatever its block holds
#pragma unroll
  for (int r = 0; r < NR; r++) in_row[r] = r * 8 + b < nb ? ~0u : 0u;
  // x first (all workgroups but the first ones find it in a cache), the first rows right behind it: one memory round trip for both.  Past the
  // row the load's range check returns zeros.
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)xf, 0, nb * 1024, 0x00027000);
  uint4 xp[XLOADS];
#pragma unroll
  for (int u = 0; u < XLOADS; u++)
    xp[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(xres, (int)(threadIdx.x + GEMV_WAVES * 64 * u) * 16, 0, 0));
  StageRegs<NR, RPI> g;
  auto request = [&](int r0) {
    const int64_t base = (int64_t)r0 * row_pieces;
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
      // every lane loads in every round (past the tile: its last piece, past the matrix: the matrix's last piece)
      const int64_t piece = base + min(lane + 64 * u, tile_pieces - 1);
      g.v[u] = load_w16(W + (piece < last_piece ? piece : last_piece) * 16);
    }
  };
  request(min(row0, N - 1));
  __builtin_amdgcn_sched_barrier(0);
  // piece p lies at p ^ ((p >> 4) & 3): the eight lanes of a super-block read from eight different banks
  auto at_piece = [](int p) { return p ^ ((p >> 4) & 3); };
  float top = 0.0f;
#pragma unroll
  for (int u = 0; u < XLOADS; u++) {
    const float4 v = __builtin_bit_cast(float4, xp[u]);
    top = fmaxf(fmaxf(top, fabsf(v.x)), fabsf(v.y));
    top = fmaxf(fmaxf(top, fabsf(v.z)), fabsf(v.w));
    xlds[at_piece(threadIdx.x + GEMV_WAVES * 64 * u)] =
        __builtin_bit_cast(uint4, make_float4(v.x * XF_LIFT, v.y * XF_LIFT, v.z * XF_LIFT, v.w * XF_LIFT));
  }
  ((int*)&range)[wv] = __any(top >= XF_LIFT_BELOW) ? 3 : __any(top >= XF_TINY);
  __syncthreads();
  const int4 f = range;
#pragma unroll
  for (int r = 0; r < NR; r++) load_xf<true>(x[r], [&](int i) { return __builtin_bit_cast(float4, xlds[at_piece(i)]); }, r * 8 + b, c, true);
  const int kind = __builtin_amdgcn_readfirstlane(f.x | f.y | f.z | f.w);
  const int end = kind == 3 ? 0 : N;
  float down = 1.0f;
  if (__builtin_expect(kind == 0, 0)) {
#pragma unroll
    for (int r = 0; r < NR; r++) {
#pragma unroll
      for (int i = 0; i < 16; i++) { x[r].lo[i] *= XF_TINY_LIFT; x[r].hi[i] *= XF_TINY_LIFT; }
      x[r].sum_c *= XF_TINY_LIFT;
    }
    down = 1.0f / XF_TINY_LIFT;
  }
  while (row0 < end) {
#pragma unroll
    for (int u = 0; u < LOADS; u++)
      if (lane + 64 * u < tile_pieces) tile[lane + 64 * u] = g.v[u];
    if (row0 + step < N) request(row0 + step);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float acc[RPI];
#pragma unroll
    for (int i = 0; i < RPI; i++) {
      acc[i] = 0.0f;
#pragma unroll
      for (int r = 0; r < NR; r++) {
        const int blk = i * row_pieces + min(r * 8 + b, nb - 1) * 9;       // piece index of the block header
        uint4 hdr = tile[blk];
        hdr.x &= in_row[r];
        acc[i] += slot_dot_f32<true>(hdr, tile[blk + 1 + c], x[r], sel);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();                     // every lane has read its pieces before the tile is overwritten
#pragma unroll
    for (int i = 0; i < RPI; i++) {
      const float tot = wave_sum(acc[i]);
      if (lane == 0 && row0 + i < N) y[row0 + i] = tot * down;
    }
    row0 += step;
  }
  if (__builtin_expect(kind == 3, 0)) {
    int l = lane;
    asm("" : "+v"(l));      // (seen through, what this path derives from it stays in registers across the loop above)
    const ScaleSel sl = make_scale_sel(l & 7);
    for (; row0 < N; row0 += step)
      for (int i = 0; i < RPI && row0 + i < N; i++) row_dot_f32(W, xf, y, row0 + i, nb, l, sl);
  }
}

// Longer rows.
__global__ __launch_bounds__(GEMV_WAVES * 64) void gemv_q4k_f32_generic_kernel(
    const uint8_t* __restrict__ W, const float* __restrict__ xf, float* __restrict__ y, int N, int nb) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * GEMV_WAVES + (threadIdx.x >> 6);
  const int nwaves = gridDim.x * GEMV_WAVES;
  const ScaleSel sel = make_scale_sel(lane & 7);
  for (int row = wave; row < N; row += nwaves) row_dot_f32(W, xf, y, row, nb, lane, sel);
}

template <int NR, int RPI>
static void launch_f32_lds(const uint8_t* w, const float* x, float* y, int N, int nb) {
  const int wgs = gemv_grid(N, GEMV_WAVES * RPI);
  hipLaunchKernelGGL((gemv_q4k_f32_lds_kernel<NR, RPI>), dim3(wgs), dim3(GEMV_WAVES * 64), 0, stream(), w, x, y, N, nb, wgs);
}

int launch_gemv_q4k_f32(const void* W, const float* x, float* y, int N, int K) {
  BK_REQUIRE(W && x && y, "gemv_q4k_f32: null pointer");
  BK_REQUIRE(N > 0 && K > 0 && K % 256 == 0, "gemv_q4k_f32: K=%d must be a positive multiple of 256 (N=%d)", K, N);
  BK_REQUIRE(((uintptr_t)W & 15) == 0 && ((uintptr_t)x & 15) == 0, "gemv_q4k_f32: W and x must be 16-byte aligned");
  const int nb = K / 256, rounds = (nb + 7) / 8;
  const uint8_t* w = (const uint8_t*)W;
  // Two rows per wave step.  One where two would leave CUs without a workgroup and the rows are short (1024 x 1024 2.55 us
  // against 3.13; rows of 6144 lost with one, 2048 of them 5.8 us against 5.3).  Four did not help a long matrix
  // (151936 x 2048: 41.1 us with two, 41.2 with four).
  switch (rounds) {
    case 1: if (N <= GEMV_WAVES * 2 * num_cus()) launch_f32_lds<1, 1>(w, x, y, N, nb); else launch_f32_lds<1, 2>(w, x, y, N, nb); break;
    case 2: launch_f32_lds<2, 2>(w, x, y, N, nb); break;
    case 3: launch_f32_lds<3, 2>(w, x, y, N, nb); break;
    default:
      hipLaunchKernelGGL(gemv_q4k_f32_generic_kernel, dim3(gemv_grid(N, GEMV_WAVES)), dim3(GEMV_WAVES * 64), 0, stream(), w, x, y, N, nb);
  }
  BK_LAUNCH_CHECK();
  return BK_OK;
}

}  // namespace bk
