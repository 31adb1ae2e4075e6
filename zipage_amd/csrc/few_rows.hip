// y = x W^T for few rows of x, 16-bit: what a decode step asks of its weights.
#include "mfma.h"
#include <algorithm>
#include <climits>
#include <type_traits>

namespace {

constexpr int kCUs = 256;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
template <typename T> __device__ __forceinline__ f32x4 product(const u32x4& w, const u32x4& x, const f32x4& c);
template <> __device__ __forceinline__ f32x4 product<BF16>(const u32x4& w, const u32x4& x, const f32x4& c) { return mfma_bf16(w, x, c); }
template <> __device__ __forceinline__ f32x4 product<F16>(const u32x4& w, const u32x4& x, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), c, 0, 0, 0);
}

template <typename T> __device__ __forceinline__ uint32_t pack(float lo, float hi);
template <> __device__ __forceinline__ uint32_t pack<BF16>(float lo, float hi) { return pack_bf16(lo, hi); }
template <> __device__ __forceinline__ uint32_t pack<F16>(float lo, float hi) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, f16x2{(_Float16)lo, (_Float16)hi});
}

struct FewArgs {
  const uint16_t* x;   // rows of x_st elements
  const uint16_t* w;   // (M, K)
  uint16_t* out;       // rows of o_st elements
  int n, K, M;
  int64_t x_st, o_st;
};

// 16 * TT rows of x (TILES: tiles of them side by side, which share W in the L2; otherwise these are all, and the division that finds
// a tile, 0.1 to 0.4 us, is saved) and 16 * MT of W per workgroup, four waves that share the contraction.  Both pass through LDS in
// stages of 128 elements of every row, a step of 32 for each wave: loads of whole cache lines, for the L1 takes four to five cycles for
// every line touched, whole or in part.  A row's sixteen pieces lie in the order of (piece ^ row).  Bound by the weights'
// stream: what counts is bytes in flight, so the ring takes what LDS there is, for two workgroups where the tiles are small.
// Weights from memory, us (the library): 16 rows, 1024 -> 4096 4.4 (7.6), 2048 -> 1024 5.5 (11.0), 3072 -> 1024 6.7 (12.0), 4096
// -> 4096 9.6 (15.8), 4096 -> 24 576 45 (46), 12 288 -> 4096 22.5 (22.7); 32 rows, 1024 -> 4096 5.0 (11.4), 4096 -> 4096 10.9
// (13.4); 48 rows, 1024 -> 4096 6.6 (11.4), 3072 -> 1024 11.2 (11.7); errors the same.  The caller's rule has where it is slower.
template <int TT, int MT> struct FewTile {
  static constexpr int kLoads = TT + MT, kBytes = kLoads * 4096;       // of a wave; of a stage
  static constexpr int kRing = kLoads <= 2 ? 9 : kLoads == 3 ? 6 : kLoads == 4 ? 9 : kLoads == 5 ? 7 : kLoads == 6 ? 6 : 5;
};
template <typename T, int TT, int MT, bool TILES>
__global__ __launch_bounds__(256, 2) void few_rows_kernel(FewArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef FewTile<TT, MT> Tile;
  constexpr int L = Tile::kLoads, R = Tile::kRing;
  static_assert((R - 2) * L < 64, "loads that a wait can count");
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row_tiles = TILES ? (a.n + 16 * TT - 1) / (16 * TT) : 1;
  const int n0 = TILES ? (int)(blockIdx.x % row_tiles) * 16 * TT : 0, rows = TILES ? min(16 * TT, a.n - n0) : a.n;
  const int m0 = (int)(blockIdx.x / row_tiles) * 16 * MT, steps = a.K / 32, stages = (steps + 3) / 4;
  const int x_row = (int)a.x_st * 2;                     // bytes
  const u32x4 xr = rows_from(a.x + n0 * a.x_st, (uint32_t)(rows - 1) * x_row + a.K * 2);
  const u32x4 wr = rows_from(a.w + (int64_t)m0 * a.K, (uint32_t)min(16 * MT, a.M - m0) * a.K * 2);
  int from[L];                                           // of four rows a load; what is not there lies past the end
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int at = wave * L + i, row = at * 4 + g, r = at < 4 * MT ? row : row - 16 * MT;
    const bool there = at < 4 * MT ? m0 + r < a.M : r < rows;
    from[i] = (there ? r * (at < 4 * MT ? a.K * 2 : x_row) : INT_MIN) + (l16 ^ (row & 15)) * 16;
  }
  auto issue = [&](int s) {                              // past the last stage zeros come, so that the count stays
    char* const to = lds_raw + (s % R * Tile::kBytes + wave * L * 1024);
    const bool whole = s * 4 + 4 <= steps;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      int at = from[i] + s * 256;
      if (!whole) at = s * 256 + (l16 ^ ((wave * L + i) * 4 + g & 15)) * 16 < a.K * 2 ? at : INT_MIN;
      load_to_lds(wave * L + i < 4 * MT ? wr : xr, to + i * 1024, at, 0);
    }
  };
#pragma unroll 1
  for (int s = 0; s < R - 1; ++s) issue(s);
  f32x4 acc[TT][MT] = {};
  const int read_at = l16 * 256 + ((wave * 4 + g) ^ l16) * 16;
#pragma unroll 1
  for (int s = 0; s < stages; ++s) {
    // this stage is there, and the one before has been read
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((R - 2) * L) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(s + R - 1);
    if (s * 4 + wave >= steps) continue;
    const char* const at = lds_raw + s % R * Tile::kBytes + read_at;
    u32x4 wf[MT], xf[TT];
#pragma unroll
    for (int j = 0; j < MT; ++j) wf[j] = *(const u32x4*)(at + j * 4096);
#pragma unroll
    for (int t = 0; t < TT; ++t) xf[t] = *(const u32x4*)(at + (MT + t) * 4096);
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[t][j] = product<T>(wf[j], xf[t], acc[t][j]);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");    // no load is left on its way to LDS
  __syncthreads();
  // tile i of the TT * MT goes to wave i % 4, which adds up the others' shares in the order of the waves
  f32x4* const red = (f32x4*)lds_raw;
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int j = 0; j < MT; ++j) red[((t * MT + j) * 4 + wave) * 64 + lane] = acc[t][j];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (TT * MT + 3) / 4; ++i) {
    const int id = i * 4 + wave, t = id / MT, j = id - t * MT;
    if (id >= TT * MT) break;
    f32x4 y = red[id * 256 + lane];
#pragma unroll
    for (int k = 1; k < 4; ++k) y += red[id * 256 + k * 64 + lane];
    const int n = n0 + t * 16 + l16, m = m0 + j * 16 + g * 4;
    if (n >= a.n || m >= a.M) continue;
    *(uint2*)(a.out + n * a.o_st + m) = uint2{pack<T>(y[0], y[1]), pack<T>(y[2], y[3])};
  }
}

template <typename T, int TT, int MT, bool TILES = false> int launch_few(const FewArgs& a, hipStream_t st) {
  constexpr int ring = FewTile<TT, MT>::kRing * FewTile<TT, MT>::kBytes, sums = TT * MT * 4096, smem = ring > sums ? ring : sums;
  if (smem > 64 * 1024 && hipFuncSetAttribute((const void*)few_rows_kernel<T, TT, MT, TILES>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              smem) != hipSuccess) {
    zp_set_error("few_rows_linear: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((few_rows_kernel<T, TT, MT, TILES>), dim3((unsigned)((a.M + 16 * MT - 1) / (16 * MT) * ((a.n + 16 * TT - 1) / (16 * TT)))), dim3(256), smem, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
// Rows of W per workgroup: 16 where that makes at most a workgroup per CU, else 32, since each workgroup reads all of x (16
// rows of x, us with 16, 32 and 64 rows of W: 1024 -> 4096 4.4, 4.8, 6.8; 4096 -> 4096 9.7, 11.0, 16.0; 1024 -> 6144 6.2, 5.2,
// 7.1; 4096 -> 24 576 46.3, 45.2, 52.9).  64 where more rows of x leave one workgroup's ring on a CU and that makes one round of
// what were two, with contractions short enough to be bound by the beginning of a workgroup (24 rows, us with 32 and 64 rows of
// W: 128 -> 12 288 6.2, 4.4; 512 -> 9216 8.4, 6.3; 1024 -> 12 288 11.6, 9.0; 1536 -> 14 336 15.0, 12.6).
template <typename T, int TT> int launch_few(const FewArgs& a, hipStream_t st) {
  if (a.M <= 4096) return launch_few<T, TT, 1>(a, st);
  if constexpr (TT == 2)
    if (a.M > 8192 && a.K < 2048) return launch_few<T, 2, 4>(a, st);
  return launch_few<T, TT, 2>(a, st);
}
template <typename T> int launch_few(const FewArgs& a, hipStream_t st) {
  if (a.n <= 16) return launch_few<T, 1>(a, st);
  return a.n <= 32 ? launch_few<T, 2>(a, st) : launch_few<T, 4>(a, st);
}
// More than 64 rows: the smallest tiles that make at most a workgroup per CU.  Weights from memory, us (the library): 128 rows,
// 1024 -> 4096 7.8 (12.3), 2048 -> 1024 6.5 (8.5), 1024 -> 6144 9.8 (12.6), 512 -> 2048 5.2 (7.9), 4096 -> 4096 18.2 (23.6); 256 rows, 1024
// -> 4096 10.1 (11.9), 512 -> 3072 7.4 (9.0), 1024 -> 768 6.0 (8.1), 128 -> 4096 5.5 (5.5).
template <typename T> int launch_row_tiles(const FewArgs& a, hipStream_t st) {
  const auto groups = [&](int rows, int outs) { return (int64_t)((a.n + rows - 1) / rows) * ((a.M + outs - 1) / outs); };
  if (groups(32, 16) <= kCUs) return launch_few<T, 2, 1, true>(a, st);
  if (groups(32, 32) <= kCUs) return launch_few<T, 2, 2, true>(a, st);
  if (groups(64, 32) <= kCUs) return launch_few<T, 4, 2, true>(a, st);
  return launch_few<T, 4, 4, true>(a, st);
}


// 16 * TT rows of x and 16 * MT of W per workgroup over one of `parts` shares of the contraction, whose fp32 sums lie in planes that
// split_sum_kernel adds up: 65 to 256 rows are few output tiles, which leave CUs idle.  Stages of 64 elements pass through LDS in two
// rings, of x and of W, which four waves fill each; a row's eight pieces lie in the order of (piece ^ row).  Bound by the lines'
// way from L2 to LDS, 22 to 26 bytes a clock and CU, and the planes' way to memory and back.  Weights from memory, us (the
// library): 12 288 -> 4096, 64 rows 25.5 (36.3), 128 31.1 (66.0), 192 37 (89), 256 41 (53); 4096 -> 6144, 17.2 (17.6), 21.1 (25.0), 25.0
// (33.3), 28 (39.5); 64 rows, 4096 -> 151 936 227 (262).  Errors against 64 bits are the library's.
struct SplitArgs : FewArgs {
  float* planes;       // parts > 1: (parts, n, M)
  int parts;           // of the contraction
  int row_tiles, col_tiles;
};
template <int TT, int MT> struct SplitTile {
  static constexpr int kWavesX = TT >= 8 ? 4 : 2, kWavesW = 8 / kWavesX, kX = TT / kWavesX, kW = MT / kWavesW;
  static constexpr int kLoadsX = TT / 2, kLoadsW = MT / 2;               // of a wave, a stage
  static constexpr int kRoom = TT * MT <= 32 ? 80 : 160;                 // KB
  static constexpr int kRingX = TT >= 12 || kRoom < TT * 16 ? 3 : 4;
  static constexpr int kRingW = (kRoom - kRingX * TT * 2) / (MT * 2) < 12 ? (kRoom - kRingX * TT * 2) / (MT * 2) : 12;
  static constexpr int kBytes = kRingX * TT * 2048 + kRingW * MT * 2048;
  static_assert(TT % kWavesX == 0 && MT % kWavesW == 0 && TT % 2 == 0 && MT % 2 == 0 && kRingX >= 3 && kRingW >= 3, "shares of waves");
  static_assert((kRingX - 2) * kLoadsX < 64 && (kRingW - 2) * kLoadsW < 64, "loads that a wait can count");
};
template <typename T, int TT, int MT>
__global__ __launch_bounds__(512, (SplitTile<TT, MT>::kRoom == 80 ? 4 : 2)) void split_rows_kernel(SplitArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef SplitTile<TT, MT> Tile;
  constexpr int NX = Tile::kX, NW = Tile::kW, RX = Tile::kRingX, RW = Tile::kRingW;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // an XCD takes a contiguous share of (part, column tile, row tile)
  const int total = a.parts * a.col_tiles * a.row_tiles, share = (total + 7) / 8;
  const int lin = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || lin >= total) return;
  const int part = lin / (a.col_tiles * a.row_tiles), tile = lin - part * a.col_tiles * a.row_tiles;
  const int m0 = tile / a.row_tiles * 16 * MT, n0 = tile % a.row_tiles * 16 * TT;
  const int steps = a.K / 32, all = (steps + 1) / 2;                     // stages of 64 elements
  const int s0 = (int)((int64_t)all * part / a.parts), s1 = (int)((int64_t)all * (part + 1) / a.parts);
  const int len = s1 - s0, turn = (int)(blockIdx.x >> 3) % 32 * len / 32;
  const int wx = wave / Tile::kWavesW, ww = wave % Tile::kWavesW, lane_at = l16 * 128 + (g ^ (l16 & 7)) * 16;
  char* const lds_w = lds_raw + RX * TT * 2048;
  f32x4 acc[NX][NW] = {};
  // the first four waves ask for the rows of x, the others for those of W
  auto run = [&](auto which) {
    constexpr bool kX = which.value;
    constexpr int L = kX ? Tile::kLoadsX : Tile::kLoadsW, R = kX ? RX : RW, kStage = (kX ? TT : MT) * 2048;
    const int row = kX ? (int)a.x_st * 2 : a.K * 2, there = kX ? min(16 * TT, a.n - n0) : min(16 * MT, a.M - m0);
    const u32x4 rows = rows_from(kX ? a.x + n0 * a.x_st : a.w + (int64_t)m0 * a.K, (uint32_t)(there - 1) * row + a.K * 2);
    const int piece = ((lane & 7) ^ (lane >> 3)) * 16;
    char* const to = (kX ? lds_raw : lds_w) + (wave & 3) * L * 1024;
    int from[L];                                         // of eight rows a load; what is not there lies past the end
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int r = ((wave & 3) * L + i) * 8 + (lane >> 3);
      from[i] = (r < there ? r * row : INT_MIN) + piece;
    }
    // load j of stage i; past the last stage zeros come, so that the count stays
    auto issue = [&](int i, int j) {
      const int s = s0 + (i + turn < len ? i + turn : i + turn - len);
      const bool inside = i < len && s * 128 + piece < a.K * 2;
      load_to_lds(rows, to + i % R * kStage + j * 1024, inside ? from[j] + s * 128 : INT_MIN, 0);
    };
#pragma unroll 1
    for (int i = 0; i < R - 1; ++i)
#pragma unroll
      for (int j = 0; j < L; ++j) issue(i, j);
#pragma unroll 1
    for (int i = 0; i < len; ++i) {
      // this stage is there, and the one before has been read
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((R - 2) * L) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const char* const xs = lds_raw + i % RX * (TT * 2048), * const ws = lds_w + i % RW * (MT * 2048);
      u32x4 wf[2][NW], xf[2][NX];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int j = 0; j < NW; ++j) wf[half][j] = *(const u32x4*)(ws + (ww * NW + j) * 2048 + (lane_at ^ half * 64));
#pragma unroll
        for (int t = 0; t < NX; ++t) xf[half][t] = *(const u32x4*)(xs + (wx * NX + t) * 2048 + (lane_at ^ half * 64));
      }
      // the next stage's loads one by one between the products: in a row they hold a wave up
      int asked = 0;
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int t = 0; t < NX; ++t)
#pragma unroll
          for (int j = 0; j < NW; ++j) {
            acc[t][j] = product<T>(wf[half][j], xf[half][t], acc[t][j]);
            const int done = (half * NX + t) * NW + j + 1;
            if (done * L / (2 * NX * NW) > asked) {
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (; asked < done * L / (2 * NX * NW); ++asked) issue(i + R - 1, asked);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
    }
  };
  if (wave < 4) run(std::integral_constant<bool, true>());
  else run(std::integral_constant<bool, false>());
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // no load is left on its way to LDS
  float* const plane = a.planes + (int64_t)part * a.n * a.M;
#pragma unroll
  for (int t = 0; t < NX; ++t) {
    const int n = n0 + (wx * NX + t) * 16 + l16;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const int m = m0 + (ww * NW + j) * 16 + g * 4;
      if (n >= a.n || m >= a.M) continue;
      if (a.parts > 1) *(f32x4*)(plane + (int64_t)n * a.M + m) = acc[t][j];
      else *(uint2*)(a.out + n * a.o_st + m) = uint2{pack<T>(acc[t][j][0], acc[t][j][1]), pack<T>(acc[t][j][2], acc[t][j][3])};
    }
  }
}

// out = the planes, added up in their order
template <typename T>
__global__ __launch_bounds__(256) void split_sum_kernel(SplitArgs a) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, all = (int64_t)a.n * a.M;
  if (i >= all) return;
  f32x4 y = *(const f32x4*)(a.planes + i);
#pragma unroll 4
  for (int p = 1; p < a.parts; ++p) y += *(const f32x4*)(a.planes + p * all + i);
  const int64_t row = i / a.M;
  *(uint2*)(a.out + row * a.o_st + (i - row * a.M)) = uint2{pack<T>(y[0], y[1]), pack<T>(y[2], y[3])};
}

struct SplitPlan { int tt, mt, parts; };
// The tiles and parts of the least estimate, us: stages at 26 bytes a clock and CU, W at 5.5 TB/s, planes at 5 TB/s both ways, and what a
// workgroup's beginning and end and another launch take.  Within 7 % of the fastest of all that there are at 17 sizes of
// 64 to 256 rows, 12 of them the fastest.
SplitPlan split_plan(int n, int K, int M) {
  const int tt = n <= 32 ? 2 : n <= 64 ? 4 : n <= 128 ? 8 : n <= 192 ? 12 : 16, stages = (K + 63) / 64;
  SplitPlan best = {tt, 8, 1};
  double least = 1e30;
  for (int mt = 8; mt >= 4; mt -= 2) {
    if (mt != 8 && (tt == 2 || tt == 4 && mt == 6 || tt == 12 && mt == 4)) continue;
    const int64_t tiles = (int64_t)((n + 16 * tt - 1) / (16 * tt)) * ((M + 16 * mt - 1) / (16 * mt));
    for (int parts = 1; parts <= 16 && parts <= stages / 2 && (parts == 1 || tiles * parts <= kCUs); ++parts) {
      const double work = (double)((tiles * parts + kCUs - 1) / kCUs) * ((stages + parts - 1) / parts) * (tt + mt) * (2048 / 26.0 / 2000);
      const double read = (double)K * M * (2 / 5.5e6), sums = parts > 1 ? 2 + (double)parts * n * M * (8 / 5e6) : 0;
      const double all = std::max(work, read) + sums;
      if (all < least) least = all, best = {tt, mt, parts};
    }
  }
  return best;
}
template <typename T, int TT, int MT> int launch_split(SplitArgs a, hipStream_t st) {
  a.row_tiles = (a.n + 16 * TT - 1) / (16 * TT);
  a.col_tiles = (a.M + 16 * MT - 1) / (16 * MT);
  constexpr int smem = SplitTile<TT, MT>::kBytes;
  if (hipFuncSetAttribute((const void*)split_rows_kernel<T, TT, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) {
    zp_set_error("split_rows_linear: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  const int64_t total = (int64_t)a.parts * a.col_tiles * a.row_tiles;
  hipLaunchKernelGGL((split_rows_kernel<T, TT, MT>), dim3((unsigned)((total + 7) / 8 * 8)), dim3(512), smem, st, a);
  if (a.parts > 1 && a.out)
    hipLaunchKernelGGL((split_sum_kernel<T>), dim3((unsigned)(((int64_t)a.n * a.M + 1023) / 1024)), dim3(256), 0, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
template <typename T> int launch_split(const SplitPlan& p, const SplitArgs& a, hipStream_t st) {
#define ZP_SPLIT(TT, MT) if (p.tt == TT && p.mt == MT) return launch_split<T, TT, MT>(a, st)
  ZP_SPLIT(2, 8); ZP_SPLIT(4, 4); ZP_SPLIT(4, 8); ZP_SPLIT(8, 4); ZP_SPLIT(8, 6); ZP_SPLIT(8, 8); ZP_SPLIT(12, 6); ZP_SPLIT(12, 8);
  ZP_SPLIT(16, 4); ZP_SPLIT(16, 6); ZP_SPLIT(16, 8);
#undef ZP_SPLIT
  zp_set_error("split_rows_linear: no tiles of %d x %d", p.tt, p.mt);
  return ZP_EUNSUPPORTED;
}

}  // namespace

static int few_linear(const char* name, int most, const void* x, const void* w, void* out, int32_t n, int32_t K, int32_t M, int64_t x_stride,
                      int64_t out_stride, int32_t dtype, hipStream_t st) {
  ZP_REQUIRE(n >= 0 && K > 0 && M > 0 && x_stride >= K && out_stride >= M, "%s: bad dims", name);
  if ((dtype != ZP_BF16 && dtype != ZP_F16) || n > most || K % 32 || M % 4 || x_stride % 8 || out_stride % 4 ||
      x_stride > (1 << 23) || K > (1 << 23)) {
    zp_set_error("%s: 16-bit, %d rows (at most %d) of %d elements (a multiple of 32), %d outputs (a multiple of 4) unsupported",
                 name, n, most, K, M);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(x && w && out && aligned16(x) && aligned16(w) && ((uintptr_t)out & 7) == 0, "%s: null or unaligned pointer", name);
  const FewArgs a = {(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)out, n, K, M, x_stride, out_stride};
  if (n <= 64) return dtype == ZP_BF16 ? launch_few<BF16>(a, st) : launch_few<F16>(a, st);
  return dtype == ZP_BF16 ? launch_row_tiles<BF16>(a, st) : launch_row_tiles<F16>(a, st);
}
extern "C" int zp_few_rows_linear(const void* x, const void* w, void* out, int32_t n, int32_t K, int32_t M, int64_t x_stride,
                                  int64_t out_stride, int32_t dtype, void* stream) {
  return few_linear("few_rows_linear", 64, x, w, out, n, K, M, x_stride, out_stride, dtype, (hipStream_t)stream);
}
extern "C" int zp_row_tiles_linear(const void* x, const void* w, void* out, int32_t n, int32_t K, int32_t M, int64_t x_stride,
                                   int64_t out_stride, int32_t dtype, void* stream) {
  return few_linear("row_tiles_linear", 256, x, w, out, n, K, M, x_stride, out_stride, dtype, (hipStream_t)stream);
}
// 0: nothing but the result is written.
extern "C" int64_t zp_split_rows_workspace(int32_t n, int32_t K, int32_t M) {
  if (n <= 0 || n > 256 || K <= 0 || M <= 0) return 0;
  const int parts = split_plan(n, K, M).parts;
  return parts > 1 ? (int64_t)parts * n * M * 4 : 0;
}
extern "C" int zp_split_rows_linear(const void* x, const void* w, void* out, int32_t n, int32_t K, int32_t M, int64_t x_stride,
                                    int64_t out_stride, int32_t dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  ZP_REQUIRE(n >= 0 && K > 0 && M > 0 && x_stride >= K && out_stride >= M, "split_rows_linear: bad dims");
  if ((dtype != ZP_BF16 && dtype != ZP_F16) || n > 256 || K % 32 || M % 4 || x_stride % 8 || out_stride % 4 || x_stride > (1 << 22)) {
    zp_set_error("split_rows_linear: 16-bit, %d rows (at most 256) of %d elements (a multiple of 32), %d outputs (a multiple of 4) "
                 "unsupported", n, K, M);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  const SplitPlan p = split_plan(n, K, M);
  ZP_REQUIRE(x && w && (out || p.parts > 1) && aligned16(x) && aligned16(w) && ((uintptr_t)out & 7) == 0,
             "split_rows_linear: null or unaligned pointer");
  ZP_REQUIRE(p.parts == 1 || (workspace && aligned16(workspace) && workspace_bytes >= (int64_t)p.parts * n * M * 4),
             "split_rows_linear: workspace of %lld bytes", (long long)workspace_bytes);
  SplitArgs a;
  (FewArgs&)a = {(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)out, n, K, M, x_stride, out_stride};
  a.planes = (float*)workspace;
  a.parts = p.parts;
  return dtype == ZP_BF16 ? launch_split<BF16>(p, a, (hipStream_t)stream) : launch_split<F16>(p, a, (hipStream_t)stream);
}
