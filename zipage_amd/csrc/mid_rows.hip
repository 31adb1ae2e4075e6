// y = x W^T for up to some hundred rows of x, 16-bit: what a decode step of a full batch asks of its weights.
#include "mfma.h"
#include <climits>
#include <type_traits>

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
template <typename T> __device__ __forceinline__ f32x4 product(const u32x4& w, const u32x4& x, const f32x4& c);
template <> __device__ __forceinline__ f32x4 product<BF16>(const u32x4& w, const u32x4& x, const f32x4& c) { return mfma_bf16(w, x, c); }
template <> __device__ __forceinline__ f32x4 product<F16>(const u32x4& w, const u32x4& x, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), c, 0, 0, 0);
}
template <typename T> __device__ __forceinline__ uint32_t pack(float lo, float hi);
template <> __device__ __forceinline__ uint32_t pack<BF16>(float lo, float hi) { return pack_bf16(lo, hi); }
template <> __device__ __forceinline__ uint32_t pack<F16>(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, f16x2{(_Float16)lo, (_Float16)hi});
}

struct MidArgs {
  const uint16_t* x;   // rows of x_st elements
  const uint16_t* w;   // (M, K)
  uint16_t* out;       // rows of o_st elements
  float* planes;       // parts > 1: (parts, n, M)
  int n, K, M;
  int64_t x_st, o_st;
  int parts;           // of the contraction
  int row_tiles, col_tiles;
};

template <int TT, int MT> struct MidTile {
  static constexpr int kWavesX = TT >= 8 ? 4 : 2, kWavesW = 8 / kWavesX, kX = TT / kWavesX, kW = MT / kWavesW;
  static constexpr int kLoadsX = TT / 2, kLoadsW = MT / 2;               // of a wave, a stage
  static constexpr int kRoom = TT * MT <= 32 ? 80 : 160;                 // KB
  static constexpr int kRingX = TT >= 12 || kRoom < TT * 16 ? 3 : 4;
  static constexpr int kRingW = (kRoom - kRingX * TT * 2) / (MT * 2) < 12 ? (kRoom - kRingX * TT * 2) / (MT * 2) : 12;
  static constexpr int kBytes = kRingX * TT * 2048 + kRingW * MT * 2048;
  static_assert(TT % kWavesX == 0 && MT % kWavesW == 0 && TT % 2 == 0 && MT % 2 == 0 && kRingX >= 3 && kRingW >= 3, "");
};
template <typename T, int TT, int MT>
__global__ __launch_bounds__(512, (MidTile<TT, MT>::kRoom == 80 ? 4 : 2)) void mid_rows_kernel(MidArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef MidTile<TT, MT> Tile;
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
    auto issue = [&](int s) {                            // past the last stage zeros come, so that the count stays
      const bool inside = s < s1 && s * 128 + piece < a.K * 2;
#pragma unroll
      for (int i = 0; i < L; ++i) load_to_lds(rows, to + (s - s0) % R * kStage + i * 1024, inside ? from[i] + s * 128 : INT_MIN, 0);
    };
#pragma unroll 1
    for (int s = 0; s < R - 1; ++s) issue(s0 + s);
#pragma unroll 1
    for (int s = s0; s < s1; ++s) {
      // this stage is there, and the one before has been read
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((R - 2) * L) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      issue(s + R - 1);
      const char* const xs = lds_raw + (s - s0) % RX * (TT * 2048), * const ws = lds_w + (s - s0) % RW * (MT * 2048);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4 wf[NW], xf[NX];
#pragma unroll
        for (int j = 0; j < NW; ++j) wf[j] = *(const u32x4*)(ws + (ww * NW + j) * 2048 + (lane_at ^ half * 64));
#pragma unroll
        for (int t = 0; t < NX; ++t) xf[t] = *(const u32x4*)(xs + (wx * NX + t) * 2048 + (lane_at ^ half * 64));
#pragma unroll
        for (int t = 0; t < NX; ++t)
#pragma unroll
          for (int j = 0; j < NW; ++j) acc[t][j] = product<T>(wf[j], xf[t], acc[t][j]);
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
__global__ __launch_bounds__(256) void mid_sum_kernel(MidArgs a) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, all = (int64_t)a.n * a.M;
  if (i >= all) return;
  f32x4 y = *(const f32x4*)(a.planes + i);
#pragma unroll 4
  for (int p = 1; p < a.parts; ++p) y += *(const f32x4*)(a.planes + p * all + i);
  const int64_t row = i / a.M;
  *(uint2*)(a.out + row * a.o_st + (i - row * a.M)) = uint2{pack<T>(y[0], y[1]), pack<T>(y[2], y[3])};
}

template <typename T, int TT, int MT> int launch_mid(MidArgs a, hipStream_t st) {
  a.row_tiles = (a.n + 16 * TT - 1) / (16 * TT);
  a.col_tiles = (a.M + 16 * MT - 1) / (16 * MT);
  constexpr int smem = MidTile<TT, MT>::kBytes;
  if (hipFuncSetAttribute((const void*)mid_rows_kernel<T, TT, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) {
    zp_set_error("mid_rows_linear: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  const int64_t total = (int64_t)a.parts * a.col_tiles * a.row_tiles;
  hipLaunchKernelGGL((mid_rows_kernel<T, TT, MT>), dim3((unsigned)((total + 7) / 8 * 8)), dim3(512), smem, st, a);
  if (a.parts > 1)
    hipLaunchKernelGGL((mid_sum_kernel<T>), dim3((unsigned)(((int64_t)a.n * a.M + 1023) / 1024)), dim3(256), 0, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

}  // namespace

extern "C" int zp_mid_rows_linear(const void* x, const void* w, void* out, int32_t n, int32_t K, int32_t M, int64_t x_stride,
                                  int64_t out_stride, int32_t dtype, int tt, int mt, int parts, void* workspace, void* stream) {
  MidArgs a = {(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)out, (float*)workspace, n, K, M, x_stride, out_stride, parts, 0, 0};
  hipStream_t st = (hipStream_t)stream;
#define GO(A, B) if (tt == A && mt == B) return launch_mid<BF16, A, B>(a, st)
  GO(2, 4); GO(2, 8); GO(4, 4); GO(4, 8); GO(6, 4); GO(6, 8); GO(8, 4); GO(8, 6); GO(8, 8); GO(12, 4); GO(12, 6); GO(12, 8); GO(16, 4); GO(16, 6); GO(16, 8);
  return ZP_EUNSUPPORTED;
}
