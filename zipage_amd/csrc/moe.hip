// Mixture of experts, without a host decision anywhere: every launch shape follows from the number of
// tokens, so a step can be captured into a graph.
//
//   small_linear     products with few outputs whose result stays in fp32 (router logits)
//   moe_select       softmax or sigmoids, the best groups of experts, the best experts of those
//   moe_plan         assignments in the order of their experts, and the list of row tiles
//   moe_gate_up      both input products of an expert for a row tile, its activation and the weight
//   moe_down         the output product; each assignment's row goes to the plane of its slot
//
// An assignment is (token n, slot j), written n * (top + 1) + j; slot `top` is the shared expert's,
// which every token uses with weight 1 and which counts as expert E.  Without a shared expert slots
// are 0 .. top - 1.
//
// Expert weights are kept in the order the matrix cores read them: [out / 16][in / step][lane][16
// bytes], where lane (g, r) holds row r and elements g * 16 bytes .. of a step of 64 bytes per row; a
// wave's operand is then one contiguous KB.  W is the row operand: a lane ends with four consecutive
// outputs of one token.
#include "mfma.h"
#include <type_traits>

namespace {

template <typename T> struct Mma;
template <> struct Mma<BF16> {
  static constexpr int kStep = 32;
  __device__ static __forceinline__ f32x4 go(const u32x4& w, const u32x4& x, const f32x4& c) { return mfma_bf16(w, x, c); }
  __device__ static __forceinline__ void st4(void* p, int64_t i, const float* v) {
    uint2 o;
    o.x = pack_bf16(v[0], v[1]);
    o.y = pack_bf16(v[2], v[3]);
    *(uint2*)((uint16_t*)p + i) = o;
  }
};
template <> struct Mma<F32> {
  static constexpr int kStep = 16;
  __device__ static __forceinline__ f32x4 go(const u32x4& w, const u32x4& x, f32x4 c) {
    const f32x4 a = __builtin_bit_cast(f32x4, w), b = __builtin_bit_cast(f32x4, x);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
  }
  __device__ static __forceinline__ void st4(void* p, int64_t i, const float* v) {
    *(f32x4*)((float*)p + i) = f32x4{v[0], v[1], v[2], v[3]};
  }
};
template <typename T> constexpr int kPiece = 16 / T::bytes;   // elements a lane holds per step

// ------------------------------------------------------------------ few outputs, fp32
struct SmallArgs {
  const void* x;    // token rows of x_st elements
  const void* w;    // (M, K)
  float* out;       // (n, M)
  int n, K, M;
  int64_t x_st;
};

// 16 tokens x 16 * MT outputs per workgroup, its NW waves share the contraction.
template <typename T, int MT, int NW>
__global__ __launch_bounds__(64 * NW) void small_linear_kernel(SmallArgs a) {
  __shared__ float red[NW - 1][MT * 64 * 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
  const int steps = a.K / Mma<T>::kStep;
  const char* x = (const char*)a.x + ((int64_t)min(n0 + l16, a.n - 1) * a.x_st + g * kPiece<T>) * T::bytes;
  const char* w[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    w[t] = (const char*)a.w + ((int64_t)min(m0 + t * 16 + l16, a.M - 1) * a.K + g * kPiece<T>) * T::bytes;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int ks = wave; ks < steps; ks += NW) {
    const u32x4 xf = *(const u32x4*)(x + (int64_t)ks * 64);
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = Mma<T>::go(*(const u32x4*)(w[t] + (int64_t)ks * 64), xf, acc[t]);
  }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < MT; ++t) *(f32x4*)(red[wave - 1] + (t * 64 + lane) * 4) = acc[t];
  }
  __syncthreads();
  if (wave > 0) return;
  const int n = n0 + l16;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int k = 0; k < NW - 1; ++k) acc[t] += *(const f32x4*)(red[k] + (t * 64 + lane) * 4);
    const int m = m0 + t * 16 + g * 4;
    if (n < a.n && m < a.M) *(f32x4*)(a.out + (int64_t)n * a.M + m) = acc[t];
  }
}

// Many rows, bf16: 16 * TT tokens x 16 * MT outputs, operands through LDS.  A row read as it is multiplied gives 64 bytes of
// a line to a load, and the L1 takes four to five cycles for every line touched (16 384 tokens, 32 outputs of 4096: 69 us,
// now 31; 128 outputs 148, now 65).  A stage is 128 elements of every row, a step for each of the four waves: the same share
// of the contraction that each has above, so that sums are the same to the last bit.  A row's sixteen pieces lie in the
// order of (piece ^ row).
template <int TT, int MT> struct SmallTile {
  static constexpr int kRing = MT > 2 ? 3 : 4, kBytes = (TT + MT) * 4096, kLoads = TT + MT;   // of a stage; of a wave
};
template <int TT, int MT>
__global__ __launch_bounds__(256, 2) void small_tile_kernel(SmallArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef SmallTile<TT, MT> Tile;
  constexpr int L = Tile::kLoads, R = Tile::kRing;
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * TT, m0 = blockIdx.y * 16 * MT, steps = a.K / 32, stages = (steps + 3) / 4;
  const int x_row = (int)a.x_st * 2;                     // bytes
  const u32x4 xr = rows_from((const uint16_t*)a.x + n0 * a.x_st, (uint32_t)(min(16 * TT, a.n - n0) - 1) * x_row + a.K * 2);
  const u32x4 wr = rows_from((const uint16_t*)a.w + (int64_t)m0 * a.K, (uint32_t)min(16 * MT, a.M - m0) * a.K * 2);
  int from[L];                                           // of four rows a load; what is not there lies past the end
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int at = wave * L + i, row = at * 4 + g, r = at < 4 * MT ? row : row - 16 * MT;
    const bool there = at < 4 * MT ? m0 + r < a.M : n0 + r < a.n;
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
#pragma unroll
  for (int s = 0; s < R - 1; ++s) issue(s);
  f32x4 acc[TT][MT] = {};
  const int read_at = l16 * 256 + ((wave * 4 + g) ^ l16) * 16;
#pragma unroll 1
  for (int s = 0; s < stages; ++s) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (R - 2) * L);    // this stage is there, and the one before has been read
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
      for (int j = 0; j < MT; ++j) acc[t][j] = mfma_bf16(wf[j], xf[t], acc[t][j]);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0);                         // no load is left on its way to LDS
  __syncthreads();
  f32x4* const red = (f32x4*)lds_raw;
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) red[((wave - 1) * TT * MT + t * MT + j) * 64 + lane] = acc[t][j];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int j = 0; j < MT; ++j) {
#pragma unroll
      for (int k = 0; k < 3; ++k) acc[t][j] += red[(k * TT * MT + t * MT + j) * 64 + lane];
      const int n = n0 + t * 16 + l16, m = m0 + j * 16 + g * 4;
      if (n < a.n && m < a.M) *(f32x4*)(a.out + (int64_t)n * a.M + m) = acc[t][j];
    }
}

// ------------------------------------------------------------------ selection
constexpr int kMaxExperts = 1024;

struct SelectArgs {
  const float* z;     // (n, z_st) router logits
  int32_t* ids;       // (n, top)
  float* weights;     // (n, top)
  int32_t* counts;    // (E + 1,), cleared here
  int n, E, top, groups, keep, score, z_st;
};

__device__ __forceinline__ int lowest_holder(float best, const float* v, int per) {
  // smallest index lane + 64 j whose value is `best`
  for (int j = 0; j < per; ++j) {
    const uint64_t b = __ballot(v[j] == best);
    if (b) return j * 64 + __builtin_ctzll(b);
  }
  return 0;
}

// A wave per token.  PER values per lane: expert (or group) lane + 64 j.
template <int PER>
__global__ __launch_bounds__(256) void moe_select_kernel(SelectArgs a) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == 0)
    for (int e = threadIdx.x; e <= a.E; e += 256) a.counts[e] = 0;
  const int n = blockIdx.x * 4 + wave;
  float* const zl = lds + wave * a.E;
  float z[PER];
  float mx = -INFINITY;
  if (n < a.n) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = lane + 64 * j;
      z[j] = e < a.E ? a.z[(int64_t)n * a.z_st + e] : -INFINITY;
      if (e < a.E) zl[e] = z[j];
      mx = fmaxf(mx, z[j]);
    }
  }
  __syncthreads();
  if (n >= a.n) return;
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) sum += expf(z[j] - mx);
  const float inv = 1.f / wave_sum(sum);
  const int gs = a.E / a.groups;
  if (a.keep < a.groups) {
    float gm[PER];
    uint32_t kept = 0;                          // bit j: group lane + 64 j
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int gr = lane + 64 * j;
      gm[j] = -INFINITY;
      if (gr < a.groups)
        for (int i = 0; i < gs; ++i) gm[j] = fmaxf(gm[j], zl[gr * gs + i]);
    }
    for (int k = 0; k < a.keep; ++k) {
      float b = -INFINITY;
#pragma unroll
      for (int j = 0; j < PER; ++j) b = fmaxf(b, gm[j]);
      b = wave_max(b);
      const int gr = lowest_holder(b, gm, PER);
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (gr == lane + 64 * j) { gm[j] = -INFINITY; kept |= 1u << j; }
    }
    // experts of the other groups leave: group g's bit is in lane g % 64
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = min(lane + 64 * j, a.E - 1), gr = e / gs;
      const uint32_t bits = (uint32_t)__shfl((int)kept, gr & 63);
      if (!((bits >> (gr >> 6)) & 1u)) z[j] = -INFINITY;
    }
  }
  for (int k = 0; k < a.top; ++k) {
    float b = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; ++j) b = fmaxf(b, z[j]);
    b = wave_max(b);
    const int e = lowest_holder(b, z, PER);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (e == lane + 64 * j) z[j] = -INFINITY;
    if (lane == 0) {
      a.ids[(int64_t)n * a.top + k] = e;
      a.weights[(int64_t)n * a.top + k] = a.score == ZP_SCORE_SIGMOID ? 1.f / (1.f + expf(-b)) : expf(b - mx) * inv;
    }
  }
}

// ------------------------------------------------------------------ plan
struct PlanArgs {
  const int32_t* ids;     // (n, top)
  int32_t* counts;        // (E + 1,) zero before the first plan launch (large plans)
  int32_t* base;          // (blocks, E) large plans
  int32_t* offsets;       // (E + 2,)
  int32_t* sorted;        // (n * slots,) assignments by expert
  int32_t* tiles;         // (max_tiles, 4): expert, first position in `sorted`, rows, 0
  int32_t* ntiles;
  int n, E, top, shared, rows, max_tiles;   // rows: most rows per tile
};
constexpr int kPlanThreads = 1024;
constexpr int kPlanBlock = 4096;    // assignments per workgroup of a large plan

// Exclusive prefix sum of one value per thread over the workgroup.
__device__ __forceinline__ int block_prefix(int v, int* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int inc = wave_prefix_sum_incl(v);
  __syncthreads();
  if (lane == 63) red[wave] = inc;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < wave; ++w) before += red[w];
  return before + inc - v;
}

// Offsets and tiles from the counts in LDS (E of them); the shared expert's rows follow the others'.
__device__ __forceinline__ void offsets_and_tiles(const PlanArgs& a, const int* counts, int* offsets, int* red) {
  const int e = threadIdx.x;
  int c = e < a.E ? counts[e] : (e == a.E && a.shared ? a.n : 0);
  int at = block_prefix(c, red);
  at = min(at, a.n * (a.top + a.shared));             // counters that were not cleared stay in bounds
  c = min(c, a.n * (a.top + a.shared) - at);
  // no more tiles than full ones make, of as many rows each as the expert has for them
  const int full = (c + a.rows - 1) / a.rows, per = a.rows != 128 || full < 2 ? a.rows : ((c + full - 1) / full + 15) & ~15;
  const int t = (c + per - 1) / per;
  const int first = block_prefix(t, red);
  if (e <= a.E) {
    offsets[e] = at;
    for (int i = 0; i < t; ++i)
      if (first + i < a.max_tiles)
        *(int4*)(a.tiles + (int64_t)(first + i) * 4) = make_int4(e, at + i * per, min(per, c - i * per), 0);
    if (e == a.E) *a.ntiles = min(first + t, a.max_tiles);
  }
  __syncthreads();
}

__global__ __launch_bounds__(kPlanThreads) void moe_plan_kernel(PlanArgs a) {
  __shared__ int counts[kMaxExperts], offsets[kMaxExperts + 1], red[kPlanThreads / 64];
  const int tid = threadIdx.x, total = a.n * a.top, slots = a.top + a.shared;
  counts[tid] = 0;
  __syncthreads();
  for (int i = tid; i < total; i += kPlanThreads) atomicAdd(&counts[min(max(a.ids[i], 0), a.E - 1)], 1);
  __syncthreads();
  offsets_and_tiles(a, counts, offsets, red);
  for (int i = tid; i < total; i += kPlanThreads) {
    const int e = min(max(a.ids[i], 0), a.E - 1);
    const int n = i / a.top;
    a.sorted[min(atomicAdd(&offsets[e], 1), total - 1)] = n * slots + i - n * a.top;
  }
  if (a.shared)
    for (int n = tid; n < a.n; n += kPlanThreads) a.sorted[total + n] = n * slots + a.top;
}

// Large plans in three launches: each workgroup's counts claim a place behind the counts of others;
// offsets and tiles; placement.
__global__ __launch_bounds__(kPlanThreads) void moe_count_kernel(PlanArgs a) {
  __shared__ int counts[kMaxExperts];
  const int tid = threadIdx.x, total = a.n * a.top, i0 = blockIdx.x * kPlanBlock;
  counts[tid] = 0;
  __syncthreads();
  for (int i = i0 + tid; i < min(i0 + kPlanBlock, total); i += kPlanThreads)
    atomicAdd(&counts[min(max(a.ids[i], 0), a.E - 1)], 1);
  __syncthreads();
  if (tid < a.E) a.base[(int64_t)blockIdx.x * a.E + tid] = atomicAdd(&a.counts[tid], counts[tid]);
}
__global__ __launch_bounds__(kPlanThreads) void moe_offsets_kernel(PlanArgs a) {
  __shared__ int counts[kMaxExperts], offsets[kMaxExperts + 1], red[kPlanThreads / 64];
  const int tid = threadIdx.x;
  counts[tid] = tid < a.E ? a.counts[tid] : 0;
  __syncthreads();
  offsets_and_tiles(a, counts, offsets, red);
  for (int e = tid; e <= a.E; e += kPlanThreads) a.offsets[e] = offsets[e];
}
__global__ __launch_bounds__(kPlanThreads) void moe_place_kernel(PlanArgs a) {
  __shared__ int at[kMaxExperts];
  const int tid = threadIdx.x, total = a.n * a.top, i0 = blockIdx.x * kPlanBlock, slots = a.top + a.shared;
  if (tid < a.E) at[tid] = a.offsets[tid] + a.base[(int64_t)blockIdx.x * a.E + tid];
  __syncthreads();
  for (int i = i0 + tid; i < min(i0 + kPlanBlock, total); i += kPlanThreads) {
    const int n = i / a.top;
    a.sorted[min(atomicAdd(&at[min(max(a.ids[i], 0), a.E - 1)], 1), total - 1)] = n * slots + i - n * a.top;
  }
  if (a.shared)
    for (int n = blockIdx.x * kPlanThreads + tid; n < a.n; n += gridDim.x * kPlanThreads)
      a.sorted[total + n] = n * slots + a.top;
}

// ------------------------------------------------------------------ expert products
struct ExpertArgs {
  const void* x;          // gate_up: (n, K) tokens; down: (n * slots, K) rows by position in `sorted`
  const void* w;          // routed experts, back to back
  const void* w_shared;
  void* out;              // gate_up: (n * slots, o_st); down: planes (slots, n, o_st)
  const int32_t* sorted;
  const int32_t* tiles;
  const int32_t* ntiles;
  const float* weights;   // (n, top)
  int n, E, top, slots, max_tiles;
  int K, K_shared;        // contraction, routed and shared
  int M, M_shared;        // outputs (gate_up: of the gate alone)
  int64_t x_st, o_st, w_expert;   // w_expert: elements between experts
  int act;
  float limit, limit_shared;
  int split;              // parts in which expert_tiles_kernel takes a tile
};

// ZP_GATE_CLAMPED: w g sigmoid(1.702 g) (u + 1), g = min(gate, limit), u = clamp(up, -limit, limit)
// ZP_GATE_SILU: g sigmoid(g) u of the weighted products
template <typename T, int ACT> __device__ __forceinline__ float gated(float w, float gate, float up, float limit) {
  if (ACT == ZP_GATE_SILU) {
    const float g = w * gate;
    return g * sigmoid_of<T>(g) * (w * up);
  }
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  return w * (g * sigmoid_of<T>(1.702f * g) * (u + 1.f));
}
template <typename T> __device__ __forceinline__ float gated(int act, float w, float gate, float up, float limit) {
  return act == ZP_GATE_SILU ? gated<T, ZP_GATE_SILU>(w, gate, up, limit) : gated<T, ZP_GATE_CLAMPED>(w, gate, up, limit);
}

// Few rows per expert: the weights are streamed straight into registers.  A workgroup owns 16 * kRowsW rows of W
// (gate_up: tiles of the gate and those of `up` that belong to them) and up to 16 * MT tokens; its four waves share
// the steps of the contraction and meet in LDS.  What the weights' stream loses is what else passes the caches: 16
// rows of tokens per kRowsW tiles of W, and twice as much where two waves take the two halves of a token's cache line.
// One token tile (hardly any expert has a second): a wave takes pairs of steps, whole lines of x.  The workgroup has 128
// rows of W from six tokens per expert on (with fewer there is less of x to read again: 42 tokens of 3 of 32 experts, 3 x
// 4096 x 3072 each, 397 us, 399 with 128 rows; 53: 424, 429), and where 40 tiles and 1280 workgroups are asked for: with few
// experts, or two rounds of workgroups (two per CU), the last one, twice as long, costs more.  With 64 rows and with 128,
// whole layers of 6, 7 and 8 tokens per expert, 3 of 32 with a shared expert: 4096 wide 495 and 475 us, 449 and 450, 474 and
// 480; 4 of 32 without one 395 and 388, 393 and 390, 387 and 386.  Single products above the line, of 32 and 64 experts, are
// 3 % slower to 6 % faster (on average 1.5 % faster); below it, 8 experts of 3 x 3072 x 8192, the first, 124 and 132; 16 of
// 3 x 1536 x 4096, 66 and 69; 32 of 3 x 2048 x 1536 +3 to -4 %, the last -13 to +1 %.
// More token tiles keep 64 rows and single steps (256 tokens: 675 us; 687 with pairs, 876 with 128 rows).
constexpr int kNarrowW = 4, kWideW = 8;                // 16-row tiles of W
constexpr int kWideGrid = 1280, kWideTiles = 40, kWideRows = 6;    // workgroups, token tiles and average rows from which on
                                                                   // 128 rows of W are better
// TOGETHER: an XCD takes a contiguous share of the launch, see launch_experts
template <typename T, int MT, bool UP, int kRowsW, bool TOGETHER>
__global__ __launch_bounds__(256) void expert_rows_kernel(ExpertArgs a) {
  __shared__ __align__(16) float part[4][kRowsW * MT * 256];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t at = TOGETHER ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int tile = at % a.max_tiles, cb = at / a.max_tiles;
  if (tile >= *a.ntiles) return;
  const int4 t = *(const int4*)(a.tiles + (int64_t)tile * 4);
  const bool shared = t.x == a.E;
  const int wtiles = (shared ? a.M_shared : a.M) / 16 * (UP ? 2 : 1), K = shared ? a.K_shared : a.K;
  const int w0 = cb * kRowsW;
  if (w0 >= wtiles) return;
  const int steps = K / Mma<T>::kStep;
  const char* const w = (const char*)(shared ? a.w_shared : a.w) + (shared ? 0 : t.x * a.w_expert) * T::bytes + lane * 16;
  const char* wp[kRowsW];
#pragma unroll
  for (int i = 0; i < kRowsW; ++i) wp[i] = w + (int64_t)min(w0 + i, wtiles - 1) * steps * 1024;
  const char* x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int pos = t.y + min(i * 16 + l16, t.z - 1);
    const int64_t row = UP ? a.sorted[pos] / a.slots : pos;
    x[i] = (const char*)a.x + (row * a.x_st + g * kPiece<T>) * T::bytes;
  }
  f32x4 acc[kRowsW][MT];
#pragma unroll
  for (int k = 0; k < kRowsW; ++k)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[k][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int ks) {
    u32x4 wf[kRowsW], xf[MT];
#pragma unroll
    for (int k = 0; k < kRowsW; ++k) {
      const u32x4* const p = (const u32x4*)(wp[k] + (int64_t)ks * 1024);
      if constexpr (MT == 1) wf[k] = __builtin_nontemporal_load(p);       // hardly any expert has a second tile
      else wf[k] = *p;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) xf[i] = *(const u32x4*)(x[i] + (int64_t)ks * 64);
#pragma unroll
    for (int k = 0; k < kRowsW; ++k)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[k][i] = Mma<T>::go(wf[k], xf[i], acc[k][i]);
  };
  if constexpr (MT == 1) {
#pragma unroll kNarrowW * 2 / kRowsW
    for (int ks = wave * 2; ks + 1 < steps; ks += 8) {
      step(ks);
      step(ks + 1);
    }
    if ((steps & 1) && (steps >> 1) % 4 == wave) step(steps - 1);
  } else {
#pragma unroll 4
    for (int ks = wave; ks < steps; ks += 4) step(ks);
  }
#pragma unroll
  for (int k = 0; k < kRowsW; ++k)
#pragma unroll
    for (int i = 0; i < MT; ++i) *(f32x4*)(part[wave] + ((k * MT + i) * 64 + lane) * 4) = acc[k][i];
  __syncthreads();
  auto total = [&](int k, int i) {
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < 4; ++v) r += *(const f32x4*)(part[v] + ((k * MT + i) * 64 + lane) * 4);
    return r;
  };
  for (int u = wave; u < (UP ? kRowsW / 2 : kRowsW) * MT; u += 4) {
    const int i = u % MT, k = u / MT * (UP ? 2 : 1), wt = w0 + k;
    if (wt >= wtiles || i * 16 + l16 >= t.z) continue;
    const int pos = t.y + i * 16 + l16, as = a.sorted[pos], n = as / a.slots, slot = as - n * a.slots;
    const f32x4 first = total(k, i);
    float r[4];
    if constexpr (UP) {
      const f32x4 second = total(k + 1, i);
      const float wgt = slot < a.top ? a.weights[(int64_t)n * a.top + slot] : 1.f;
      const float lim = shared ? a.limit_shared : a.limit;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = gated<T>(a.act, wgt, first[e], second[e], lim);
      Mma<T>::st4(a.out, (int64_t)pos * a.o_st + wt * 8 + g * 4, r);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = first[e];
      Mma<T>::st4(a.out, ((int64_t)slot * a.n + n) * a.o_st + wt * 16 + g * 4, r);
    }
  }
}

// Many rows per expert: 128 or 256 tokens x 256 rows of W per workgroup, 32 of the contraction at a time.  A wave owns
// 64 rows of W and all tokens.  W is kept in the order in which the matrix cores read it, so a wave's share goes from
// memory straight into its registers; only tokens, which all four waves read, pass through LDS, by loads of their own;
// one barrier per stage.  (With W through LDS too, reads and writes of LDS took longer than the products.)
//   128 tokens: two workgroups per CU hide each other's set-up and results.  Stages are asked for two (W) and four to five
//   (tokens) ahead.
//   256 tokens: half the reads of W per product, one wave per SIMD, four and six to seven stages ahead.  From averages of
//   more than 512 rows per expert on, and only over long contractions, since nothing hides a workgroup's beginning and end.
// The L1 takes four to five cycles for every line that a load touches, whole or in part, and a stage's loads as long as its
// products if each touches whole lines: so tokens come for two stages at a time, 128 bytes of a row (64 for one stage were
// half as much again in lines).  16 384 tokens over 33 experts of 3 x 4096 x 3072 (both products, 4.95 TFLOP; the layer):
// 5.66 ms with everything through LDS, 5.24 with 256 tokens and half lines, now 4.40 (128 tokens: 4.64); of
// 3 x 2048 x 1536: 1.51 at first, 1.27 with 128 tokens, 1.31 with 256; of 3 x 1024 x 768: 488, 429 and 509 us.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
constexpr int kBlockW = 16, kWaveW = kBlockW / 4;      // 16-row tiles of W
constexpr int kBigRows = 256, kBigContraction = 2560;

__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t r, char* to, int lane_at, int at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)to, 16, lane_at, at, 0, 0);
}
__device__ __forceinline__ u32x4 load_16(__amdgpu_buffer_rsrc_t r, int lane_at, int at) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at, 0));
}
// acc += W x with the sum kept where it is, in the accumulation registers: with one wave per SIMD the compiler would
// hold the sums in both register files and move them between every two products.  It neither reorders nor copies them
// here (they are only touched by these products until `settled`), so the waits that it would put between a product and
// another use of its result are not needed before that.
__device__ __forceinline__ void mfma_in_place(f32x4& acc, const u32x4& w, const u32x4& x) {
#ifdef __HIP_DEVICE_COMPILE__                            // the constraint means another register on the host
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
#endif
}
__device__ __forceinline__ void settled(f32x4& acc) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+a"(acc));
#endif
}

// HALVES of HT 16-token tiles, of which the first NT are worked on: products and LDS reads of tiles that an expert has no rows for
// are left out, and the plan gives an expert's tiles of up to 128 as many rows each (262 rows: 96, 96 and 70 instead of 128,
// 128 and 6).  Whole layers, 3 of 32 experts and a shared one of 3 x 4096 x 3072, us: 2800 tokens 1265 -> 1090, 1900 799 -> 765,
// 1500 814 -> 757, 3300 1237 -> 1203, 5000 1556 -> 1549; 3 x 1024 x 768, 1700 tokens 78 -> 73.  Of 256 rows: tiles are full but an
// expert's last one, and only the second product has them in parts (16 384 tokens 1412 -> 1385; the first one, whose weights
// take registers, 2710 -> 2760).  Dividing the launch among XCDs by such costs instead of tiles lost up to 16 %.
template <bool UP, int HALVES, int HT, int NT>
__device__ __forceinline__ void expert_tile(const ExpertArgs& a, char* lds_raw, const int4& t, int cb) {
  constexpr int kTiles = HT * HALVES, kOwn = kTiles / 4, kPairBytes = kTiles * 2048;
  constexpr int kLeadW = HALVES == 2 ? 4 : 2, kLeadX = HALVES == 2 ? 3 : 2, kPairs = kLeadX + 1;      // stages, pairs ahead
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
  constexpr int N0 = NT < HT ? NT : HT, N1 = NT - N0;      // of the halves
  const bool shared = t.x == a.E;
  const int wtiles = (shared ? a.M_shared : a.M) / 16 * (UP ? 2 : 1), K = shared ? a.K_shared : a.K;
  const int w0 = cb * kBlockW;
  if (w0 >= wtiles) return;
  const int steps = K / 32;
  const char* wbase = (const char*)(shared ? a.w_shared : a.w) + (shared ? 0 : t.x * a.w_expert) * 2;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)(wbase + (int64_t)w0 * steps * 1024), 0,
                                                                      min(kBlockW, wtiles - w0) * steps * 1024, 0x00020000);
  // gate_up gathers tokens from all of x, down reads consecutive rows
  const char* const xbase = (const char*)a.x + (UP ? 0 : t.y * a.x_st * 2);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)xbase, 0, (int)((UP ? a.n : t.z) * a.x_st * 2), 0x00020000);
  int xoff[2 * kOwn], woff[kWaveW];                      // this wave's loads of a pair of stages; of a stage
  // a row's eight pieces of a pair lie in the order of (piece ^ row): rows of an operand don't meet in a bank
#pragma unroll
  for (int i = 0; i < 2 * kOwn; ++i) {
    const int at = wave * kOwn * 16 + i * 8 + (lane >> 3), r = min(at, t.z - 1);
    xoff[i] = (int)((UP ? a.sorted[t.y + r] / a.slots : r) * a.x_st * 2) + ((lane & 7) ^ (lane >> 3)) * 16;
    if (at >= (t.z + 15 & ~15)) xoff[i] = -(1 << 28);      // past the end: nothing is read
  }
#pragma unroll
  for (int i = 0; i < kWaveW; ++i) woff[i] = min(wave * kWaveW + i, wtiles - w0 - 1) * steps * 1024;
  // where this lane's results go, and their weights: asked for now, used behind the products
  int place[NT];
  float wgt[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) place[j] = a.sorted[t.y + min(j * 16 + l16, t.z - 1)];
  if constexpr (UP) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = place[j] / a.slots, slot = place[j] - n * a.slots;
      wgt[j] = slot < a.top ? a.weights[(int64_t)n * a.top + slot] : 1.f;
    }
  }
  // Past the end the last stage is asked for again, so that the number of loads in flight is the same in every pass of the
  // loop.  Stages behind it ask for nothing, and wait for all.
  const int pairs = (steps + 1) / 2, second = ((lane & 7) ^ (lane >> 3)) & 4 ? 64 : 0;
  auto token_rows = [&](int pair, int i) {
    const int back = (steps & 1) && pair >= pairs - 1 ? second : 0;      // a last stage alone: nothing behind the row's end
    load_to_lds(rx, lds_raw + (pair % kPairs) * kPairBytes + (wave * 2 * kOwn + i) * 1024, xoff[i] - back, min(pair, pairs - 1) * 128);
  };
  auto tokens = [&](int pair, int half) {
#pragma unroll
    for (int i = 0; i < kOwn; ++i) token_rows(pair, half * kOwn + i);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto weights = [&](int i, int ks) { return load_16(rw, lane * 16, woff[i] + min(ks, steps - 1) * 1024); };
  f32x4 acc[HALVES][kWaveW][HT];
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int i = 0; i < kWaveW; ++i)
#pragma unroll
      for (int j = 0; j < HT; ++j) acc[h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 wr[kLeadW][kWaveW], xf[HALVES][HT];
  auto fill = [&](int ks, u32x4 (&w)[kWaveW]) {
#pragma unroll
    for (int i = 0; i < kWaveW; ++i) w[i] = weights(i, ks);
    __builtin_amdgcn_sched_barrier(0);
  };
  const int lane_at = l16 * 128 + (g ^ (l16 & 7)) * 16;
  auto read_tile = [&](int ks, int h, int j) {
    xf[h][j] = *(const u32x4*)(lds_raw + (ks / 2 % kPairs) * kPairBytes + (h * HT + j) * 2048 + (lane_at ^ (ks & 1) * 64));
  };
  auto read = [&](int ks, int h) {
#pragma unroll
    for (int j = 0; j < N0; ++j) read_tile(ks, h, j);
    __builtin_amdgcn_sched_barrier(0);
  };
  static_assert(HALVES == 1 || (kOwn == 4 && HT == 2 * kWaveW), "the waits count a wave's loads");
  // A pair of stages is in LDS when all but the loads asked for after it have landed.  256 tokens: the pair behind an odd
  // stage is first read in it, three stages' loads behind; 128: in its own first stage, two stages' and a half.  Behind the
  // loop there are fewer (weights that no stage would use are not loaded, whatever is written here).
  typedef std::integral_constant<bool, true> yes;
  typedef std::integral_constant<bool, false> no;
  auto landed = [&](int odd, auto loop) {
    if constexpr (!loop.value) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if constexpr (HALVES == 2) { if (odd) asm volatile("s_waitcnt vmcnt(24)" ::: "memory"); }
    else if (!odd) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();                        // everyone's
  };
#pragma unroll
  for (int s = 0; s < kLeadX; ++s) {
    tokens(s, 0);
    tokens(s, 1);
    if constexpr (HALVES == 2) {
      if (2 * s < kLeadW) { fill(2 * s, wr[2 * s]); fill(2 * s + 1, wr[2 * s + 1]); }
    } else {
      fill(s, wr[s]);
    }
  }
  if constexpr (HALVES == 2) {
    asm volatile("s_waitcnt vmcnt(32)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read(0, 0);
  } else {
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  }
  auto stage = [&](int ks, int odd, u32x4 (&w)[kWaveW], auto loop) {      // odd: ks % 2
    constexpr bool kAsk = loop.value;
    const int next = ks / 2 + kLeadX;                    // its tokens come over the pair before this one
    if constexpr (HALVES == 2) {
      // One wave per SIMD: whatever it issues between two products is time without products.  So reads and requests
      // are spread over the products, a half ahead of their use.
#pragma unroll
      for (int i = 0; i < kWaveW; ++i)
#pragma unroll
        for (int j = 0; j < N0; ++j) {
          mfma_in_place(acc[0][i][j], w[i], xf[0][j]);
          if (j == HT / 2 - 1 && 2 * i < N1) read_tile(ks, 1, 2 * i);
          if (j == HT - 1 && 2 * i < N1) read_tile(ks, 1, 2 * i + 1);
          if (j == HT / 2 - 1 || j == HT - 1) __builtin_amdgcn_sched_barrier(0);
        }
      landed(odd, loop);
#pragma unroll
      for (int i = 0; i < kWaveW; ++i) {
#pragma unroll
        for (int j = 0; j < (N1 ? N1 : 1); ++j) {
          if constexpr (N1 > 0) mfma_in_place(acc[1][i][j], w[i], xf[1][j]);
          if (kAsk && j == (N1 ? 1 : 0)) token_rows(next, odd * kOwn + i);
          if (j == (N1 ? 3 : 0)) read_tile(ks + 1, 0, 2 * i);
          if (j == (N1 > 4 ? 5 : N1 ? 3 : 0)) read_tile(ks + 1, 0, 2 * i + 1);
          if (j & 1) __builtin_amdgcn_sched_barrier(0);
        }
        if (kAsk) w[i] = weights(i, ks + kLeadW);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      landed(odd, loop);
      if (kAsk) tokens(next, odd);
      read(ks, 0);
#pragma unroll
      for (int i = 0; i < kWaveW; ++i) {
#pragma unroll
        for (int j = 0; j < N0; ++j) acc[0][i][j] = mfma_bf16(w[i], xf[0][j], acc[0][i][j]);
        if (kAsk) w[i] = weights(i, ks + kLeadW);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int ks = 0;
#pragma unroll 1
  for (; ks + kLeadW <= steps; ks += kLeadW) {
#pragma unroll
    for (int s = 0; s < kLeadW; ++s) stage(ks + s, s & 1, wr[s], yes{});
  }
#pragma unroll
  for (int s = 0; s + 1 < kLeadW; ++s)
    if (ks + s < steps) stage(ks + s, s & 1, wr[s], no{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // loads into LDS end before the workgroup does
  if constexpr (HALVES == 2) {                           // the last products' results are in their registers
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int i = 0; i < kWaveW; ++i)
#pragma unroll
        for (int j = 0; j < HT; ++j) settled(acc[h][i][j]);
  }
  // Two result tiles side by side hold 4 outputs per lane each; lanes of neighbouring groups swap halves, so that
  // each ends with 8 consecutive outputs of one of them: group g has tile (g & 1), outputs 8 (g >> 1) on.
  auto store8 = [&](const float* lo, const float* hi, int64_t at, int tile, int tiles, bool row) {
    const auto a0 = __builtin_amdgcn_permlane16_swap(pack_bf16(lo[0], lo[1]), pack_bf16(hi[0], hi[1]), false, false);
    const auto a1 = __builtin_amdgcn_permlane16_swap(pack_bf16(lo[2], lo[3]), pack_bf16(hi[2], hi[3]), false, false);
    if (row && tile + (g & 1) < tiles)
      *(u32x4*)((uint16_t*)a.out + at + (tile + (g & 1)) * 16 + (g >> 1) * 8) = u32x4{a0[0], a1[0], a0[1], a1[1]};
  };
  const int out_tiles = UP ? wtiles / 2 : wtiles, own = w0 + wave * kWaveW;
  // which activation is asked once, not for every result: with no other wave on its SIMD a wave has only results side by side to
  // hide their chains behind (16 384 tokens, 33 experts of 3 x 4096 x 3072, the first product 2690 -> 2590 us)
  auto activated = [&](auto act) {
    const float lim = shared ? a.limit_shared : a.limit;
#pragma unroll
    for (int jj = 0; jj < NT; ++jj) {
      const int j = jj % HT, h = jj / HT, r = jj * 16 + l16;
      float v[2][4];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) v[u][k] = gated<BF16, act.value>(wgt[jj], acc[h][2 * u][j][k], acc[h][2 * u + 1][j][k], lim);
      store8(v[0], v[1], (int64_t)(t.y + r) * a.o_st, own / 2, out_tiles, r < t.z);       // every lane takes part in the swaps
    }
  };
  if constexpr (UP) {
    if (a.act == ZP_GATE_SILU) activated(std::integral_constant<int, ZP_GATE_SILU>());
    else activated(std::integral_constant<int, ZP_GATE_CLAMPED>());
    return;
  }
#pragma unroll
  for (int jj = 0; jj < NT; ++jj) {
    const int j = jj % HT, h = jj / HT;
    const bool row = jj * 16 + l16 < t.z;
    const int n = place[jj] / a.slots, slot = place[jj] - n * a.slots;
#pragma unroll
    for (int i = 0; i < kWaveW; i += 2) {
      const float lo[4] = {acc[h][i][j][0], acc[h][i][j][1], acc[h][i][j][2], acc[h][i][j][3]};
      const float hi[4] = {acc[h][i + 1][j][0], acc[h][i + 1][j][1], acc[h][i + 1][j][2], acc[h][i + 1][j][3]};
      store8(lo, hi, ((int64_t)slot * a.n + n) * a.o_st, own + i, out_tiles, row);
    }
  }
}

template <bool UP, int HALVES, int HT>
__global__ __launch_bounds__(256, HALVES == 2 ? 1 : 2) void expert_tiles_kernel(ExpertArgs a) {
  constexpr int kTiles = HT * HALVES, kGroup = 8;
  extern __shared__ __align__(16) char lds_raw[];
  // An XCD takes a contiguous share of the (tile, column block) pairs, eight tiles at a time, column block by column
  // block, so that what is in flight on it shares rows of x and of W in its L2.  Shares are of pairs, not of tiles: 33 tiles in
  // shares of five left the last XCD and half of another without work (8 experts and a shared one of 3 x 4096 x 14336, 180
  // tokens 792 -> 644 us; 3200 tokens of 3 of 32 of 3 x 4096 x 3072 1194 -> 1153).
  const int nt = *a.ntiles * a.split;
  const int Mx = max(a.M, a.M_shared) * (UP ? 2 : 1), cols = (Mx + 16 * kBlockW - 1) / (16 * kBlockW);
  const int pairs = nt * cols, share = (pairs + 7) / 8, i_xcd = blockIdx.x >> 3, lin = (blockIdx.x & 7) * share + i_xcd;
  if (i_xcd >= share || lin >= pairs) return;
  const int tg = lin / (kGroup * cols), rem = lin - tg * kGroup * cols, in_group = min(kGroup, nt - tg * kGroup);
  const int tile = tg * kGroup + rem % in_group, cb = rem / in_group;
  int4 t = *(const int4*)(a.tiles + (int64_t)(tile / a.split) * 4);
  // a part of a larger tile
  const int per = a.split > 1 ? ((t.z + a.split - 1) / a.split + 15) & ~15 : kTiles * 16;
  t.y += tile % a.split * per;
  t.z = min(t.z - tile % a.split * per, per);
  if (t.z <= 0) return;
  constexpr int kPart = kTiles / 4;
  if constexpr (HALVES == 2 && UP) {
    expert_tile<UP, HALVES, HT, kTiles>(a, lds_raw, t, cb);
  } else {
    if (t.z > 48 * kPart) expert_tile<UP, HALVES, HT, 4 * kPart>(a, lds_raw, t, cb);
    else if (t.z > 32 * kPart) expert_tile<UP, HALVES, HT, 3 * kPart>(a, lds_raw, t, cb);
    else if (HALVES == 2 || t.z > 16 * kPart) expert_tile<UP, HALVES, HT, 2 * kPart>(a, lds_raw, t, cb);
    else if constexpr (HALVES == 1) expert_tile<UP, HALVES, HT, kPart>(a, lds_raw, t, cb);
  }
}

// staged: tokens through LDS, tiles of 64 (see tile_rows), 128 and 256 rows
template <bool UP> int launch_experts(const ExpertArgs& a, int rows, bool staged, int dtype, hipStream_t st) {
  if (staged) {
    const int Mx = (a.M > a.M_shared ? a.M : a.M_shared) * (UP ? 2 : 1);
    const bool big = rows == kBigRows && a.K >= kBigContraction;
    ExpertArgs b = a;
    b.split = big || rows < 128 ? 1 : rows / 128;
    const int64_t grid = (int64_t)((b.max_tiles * b.split + 7) / 8) * 8 * ((Mx + 16 * kBlockW - 1) / (16 * kBlockW));
    const void* const fn = big ? (const void*)expert_tiles_kernel<UP, 2, 8> : (const void*)expert_tiles_kernel<UP, 1, 8>;
    const int smem = big ? 4 * 32 * 1024 : 3 * 16 * 1024;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) {
      zp_set_error("moe: cannot reserve %d bytes of LDS", smem);
      return ZP_EHIP;
    }
    if (big) hipLaunchKernelGGL((expert_tiles_kernel<UP, 2, 8>), dim3((unsigned)grid), dim3(256), smem, st, b);
    else hipLaunchKernelGGL((expert_tiles_kernel<UP, 1, 8>), dim3((unsigned)grid), dim3(256), smem, st, b);
    ZP_LAUNCH_CHECK();
    return ZP_OK;
  }
  const int Mw = (a.M > a.M_shared ? a.M : a.M_shared) * (UP ? 2 : 1);
  const auto grid_of = [&](int tiles_w) { return (int64_t)a.max_tiles * ((Mw + 16 * tiles_w - 1) / (16 * tiles_w)); };
  const bool wide = rows == 16 && dtype == ZP_BF16 && a.max_tiles >= kWideTiles && grid_of(kWideW) >= kWideGrid &&
                    (int64_t)a.n * a.top >= (int64_t)kWideRows * a.E;
  const int64_t grid = (grid_of(wide ? kWideW : kNarrowW) + 7) / 8 * 8;      // shares of eight XCDs; behind the last tile of W nothing is done
  if (grid >= (1ll << 31)) {
    zp_set_error("moe: too many tiles");
    return ZP_EUNSUPPORTED;
  }
  // The shared expert's tiles read the same weights: on one XCD, one after the other, they find them in its L2 (64 tokens of 3 of
  // 32 experts and a shared one of 3 x 4096 x 3072: 475 -> 425 us, 53: 432 -> 416, 32: 441 -> 417; 24, with two such tiles, 383
  // and 386; tiles of 32, 100 tokens 536 -> 529, 170 563 -> 552; fp32, 64 tokens 994 -> 811, 128 1391 -> 1107, tiles of 64, 200 1944 -> 1813,
  // 4000 12 510 -> 12 170).  Without one, weights that the last-level cache holds gain too (3 x 1024 x 768, 4 of 32, 17 tokens 43.9 -> 41.5; fp32
  // 61 -> 52); those from memory come as fast or faster spread over all (3 x 4096 x 3072, 17 tokens 347, 360 in shares; 64: 383, 390).  The
  // line lies low: launches of 256 MB are 10 to 15 % faster in shares, of 384 to 640 MB 6 % faster to 3 % slower, of 768 to 1280 MB 1 % faster to 2 %
  // slower.  Tiles of 64 in bf16, of many tokens over hundreds of experts, stay spread: 16 500 tokens of 1 of 512 and a shared one, 3 x 1024 x 768
  // 858 us, 883 in shares, 3 x 768 x 320 without one 285 and 306 (but 3 x 512 x 256 185 and 168).
  // A share of fewer than eight column blocks would be a part of one, and some XCD's tiles ones that are not there (up to 256 columns, 48 experts, 91
  // tokens, 64 x 4096 10.8 us, 15.7 in shares; fp32, 135 tokens, 256 x 2048 33 and 45).  The two orders are kernels of their own: what the choice
  // cost small launches was more than it gave them (2 of 3 x 256 x 2048, 48 tokens, down 12.8 us, 14.5).
  const bool together = (dtype == ZP_F32 || rows <= 32) && Mw > 7 * 16 * kNarrowW &&
               (a.slots > a.top || (int64_t)a.E * a.w_expert * (dtype == ZP_BF16 ? 2 : 4) < 320ll << 20);
#define ZP_EXPERTS(T, MT, KW)                                                                                               \
  do {                                                                                                                      \
    if (together) hipLaunchKernelGGL((expert_rows_kernel<T, MT, UP, KW, true>), dim3((unsigned)grid), dim3(256), 0, st, a); \
    else hipLaunchKernelGGL((expert_rows_kernel<T, MT, UP, KW, false>), dim3((unsigned)grid), dim3(256), 0, st, a);         \
  } while (0)
#define ZP_EXPERT_ROWS(T)                            \
  do {                                               \
    if (rows == 16) ZP_EXPERTS(T, 1, kNarrowW);      \
    else if (rows == 32) ZP_EXPERTS(T, 2, kNarrowW); \
    else ZP_EXPERTS(T, 4, kNarrowW);                 \
  } while (0)
  if (wide) ZP_EXPERTS(BF16, 1, kWideW);
  else if (dtype == ZP_BF16) ZP_EXPERT_ROWS(BF16);
  else ZP_EXPERT_ROWS(F32);
#undef ZP_EXPERT_ROWS
#undef ZP_EXPERTS
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

// Rows per tile: enough for the average expert.  bf16 tiles of 64 go through LDS as those of 128 do, where that makes workgroups for half of
// the CUs: read by every wave for itself, 64 rows take more lines of the L1 than the weights that they meet.  Staged and direct, us of whole
// layers: 3 of 32 experts and a shared one of 3 x 4096 x 3072, 200 tokens 480 and 533, 256 482 and 650, 480 493 and 683; of 3 x 1024 x 768, 200 40 and
// 54, 480 45 and 61; 8 of 128 of 3 x 2048 x 768, 320 tokens 226 and 251; 2 of 8 and a shared one of 3 x 4096 x 14 336, 180 tokens 623 and 1133.
// Of 1710 random products (1 to 256 experts, contractions of 32 to 14 336) those of 128 workgroups and more took 0.75 times as long staged, 23 in a
// thousand of them more than 2 % longer, 13 % at most (just above a round of 256); of those below, more than half were slower, up to 1.7 times
// (4 experts and a shared one of 3 x 4096 x 256, 96 tokens, the layer 48 and 33).  Tiles of 128 from 17 rows on do as well where they are staged, but
// leave the direct form with parts that mostly are not there (up to 15 % of small layers).  With up to 16 rows, tiles of 32 lose up to 4 % without
// a shared expert (100 tokens of 4 of 32, 437 and 453).  The staged form addresses x in 31 bits; rows too far apart are read where they lie.
constexpr int kStagedGroups = 128;
int tile_rows(int n, int E, int top, int dtype) {
  const int64_t avg = ((int64_t)n * top + E - 1) / E;
  if (dtype == ZP_BF16 && avg > 512) return kBigRows;
  if (dtype == ZP_BF16 && avg > 48) return 128;
  return avg <= 8 ? 16 : (avg <= 16 ? 32 : 64);       // a second tile reads an expert's weights again
}
int tile_bound(int n, int E, int top, int shared, int rows) {
  const int64_t a = (int64_t)n * top;
  const int64_t used = a < E ? a : E;
  return (int)(a / rows + used + (shared ? (n + rows - 1) / rows : 0));
}

}  // namespace

extern "C" int zp_small_linear(const void* x, const void* w, float* out, int32_t n, int32_t K, int32_t M,
                               int64_t x_stride, int32_t dtype, void* stream) {
  ZP_REQUIRE(n >= 0 && K > 0 && M > 0 && x_stride >= K, "small_linear: bad dims");
  ZP_MODEL_DTYPE("small_linear");
  if (K % 32 != 0 || M % 4 != 0 || x_stride % 8 != 0) {
    zp_set_error("small_linear: K %d, M %d unsupported (multiples of 32 and 4)", K, M);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(x && w && out && aligned16(x) && aligned16(w) && aligned16(out), "small_linear: null or unaligned pointer");
  SmallArgs a = {x, w, out, n, K, M, x_stride};
  hipStream_t st = (hipStream_t)stream;
  const unsigned gx = (unsigned)((n + 15) / 16);
  const bool wide = gx >= 256 && M > 16;
  const dim3 grid(gx, (unsigned)(wide ? (M + 63) / 64 : (M + 15) / 16));
  // through LDS where there are stages enough to pass the time with (us of both, this one second: K 128, 4081 rows of 64
  // outputs 4.1 and 4.9, 16 384 of 256 14.3 and 15.2; K 160, 5.4 and 6.3; K 256, 4081 rows of 36 outputs 4.5 and 5.1, 8192
  // 5.2 and 5.1, 16 384 6.9 and 5.9; K 512, 4081 of 36 5.5 and 5.8, of 128 8.0 and 6.1), and offsets are within 31 bits
  if (wide && dtype == ZP_BF16 && K >= 256 && (int64_t)n * K >= 2200000 && 32 * x_stride * 2 < 1ll << 31 &&
      (int64_t)64 * K * 2 < 1ll << 31) {
    const dim3 tiles((unsigned)((n + 31) / 32), (unsigned)(M <= 32 ? 1 : (M + 63) / 64));
    const int smem = M <= 32 ? SmallTile<2, 2>::kRing * SmallTile<2, 2>::kBytes : SmallTile<2, 4>::kRing * SmallTile<2, 4>::kBytes;
    const void* const fn = M <= 32 ? (const void*)small_tile_kernel<2, 2> : (const void*)small_tile_kernel<2, 4>;
    if (smem > 64 * 1024 && hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) {
      zp_set_error("small_linear: cannot reserve %d bytes of LDS", smem);
      return ZP_EHIP;
    }
    if (M <= 32) hipLaunchKernelGGL((small_tile_kernel<2, 2>), tiles, dim3(256), smem, st, a);
    else hipLaunchKernelGGL((small_tile_kernel<2, 4>), tiles, dim3(256), smem, st, a);
    ZP_LAUNCH_CHECK();
    return ZP_OK;
  }
#define ZP_SMALL(T)                                                                              \
  do {                                                                                           \
    if (wide) hipLaunchKernelGGL((small_linear_kernel<T, 4, 4>), grid, dim3(256), 0, st, a);     \
    else hipLaunchKernelGGL((small_linear_kernel<T, 1, 16>), grid, dim3(1024), 0, st, a);        \
  } while (0)
  if (dtype == ZP_BF16) ZP_SMALL(BF16); else ZP_SMALL(F32);
#undef ZP_SMALL
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

extern "C" int zp_moe_select(const float* logits, int32_t* ids, float* weights, int32_t* counts, int32_t n,
                             int32_t E, int32_t top, int32_t groups, int32_t keep, int32_t score,
                             int32_t logits_stride, void* stream) {
  ZP_REQUIRE(n >= 0 && E > 0 && top > 0 && groups > 0 && E % groups == 0 && keep > 0 && keep <= groups &&
                 top <= E / groups * keep && logits_stride >= E &&
                 (score == ZP_SCORE_SOFTMAX || score == ZP_SCORE_SIGMOID), "moe_select: bad dims");
  if (E > kMaxExperts - 1) {
    zp_set_error("moe_select: %d experts (at most %d)", E, kMaxExperts - 1);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(logits && ids && weights && counts, "moe_select: null pointer");
  SelectArgs a = {logits, ids, weights, counts, n, E, top, groups, keep, score, logits_stride};
  const dim3 grid((unsigned)((n + 3) / 4));
  const size_t smem = sizeof(float) * 4 * E;
  hipStream_t st = (hipStream_t)stream;
  if (E <= 64) hipLaunchKernelGGL((moe_select_kernel<1>), grid, dim3(256), smem, st, a);
  else if (E <= 256) hipLaunchKernelGGL((moe_select_kernel<4>), grid, dim3(256), smem, st, a);
  else hipLaunchKernelGGL((moe_select_kernel<16>), grid, dim3(256), smem, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

extern "C" int64_t zp_moe_tile_rows(int32_t n, int32_t E, int32_t top, int32_t dtype) {
  return n <= 0 || E <= 0 || top <= 0 ? -1 : tile_rows(n, E, top, dtype);
}
extern "C" int64_t zp_moe_max_tiles(int32_t n, int32_t E, int32_t top, int32_t shared, int32_t rows) {
  return n <= 0 || E <= 0 || top <= 0 || rows <= 0 ? -1 : tile_bound(n, E, top, shared, rows);
}
extern "C" int64_t zp_moe_plan_workspace(int32_t n, int32_t E, int32_t top) {
  if (n <= 0 || E <= 0 || top <= 0) return -1;
  return ((int64_t)(((int64_t)n * top + kPlanBlock - 1) / kPlanBlock) * E + E + 2) * 4;
}

extern "C" int zp_moe_plan(const int32_t* ids, int32_t* counts, int32_t* sorted, int32_t* tiles, int32_t* ntiles,
                           int32_t n, int32_t E, int32_t top, int32_t shared, int32_t rows, int32_t max_tiles,
                           void* workspace, int64_t workspace_bytes, void* stream) {
  ZP_REQUIRE(n > 0 && E > 0 && E < kMaxExperts && top > 0 && rows > 0 && (shared == 0 || shared == 1) &&
                 max_tiles >= tile_bound(n, E, top, shared, rows), "moe_plan: bad dims");
  ZP_REQUIRE(ids && counts && sorted && tiles && ntiles && aligned16(tiles), "moe_plan: null or unaligned pointer");
  ZP_REQUIRE((int64_t)n * (top + shared) < (1ll << 31), "moe_plan: too many tokens");
  PlanArgs a = {ids, counts, nullptr, nullptr, sorted, tiles, ntiles, n, E, top, shared, rows, max_tiles};
  hipStream_t st = (hipStream_t)stream;
  if ((int64_t)n * top <= 2 * kPlanBlock) {
    hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(kPlanThreads), 0, st, a);
    ZP_LAUNCH_CHECK();
    return ZP_OK;
  }
  ZP_REQUIRE(workspace && workspace_bytes >= zp_moe_plan_workspace(n, E, top), "moe_plan: workspace too small");
  a.offsets = (int32_t*)workspace;
  a.base = a.offsets + E + 2;
  const unsigned blocks = (unsigned)(((int64_t)n * top + kPlanBlock - 1) / kPlanBlock);
  hipLaunchKernelGGL(moe_count_kernel, dim3(blocks), dim3(kPlanThreads), 0, st, a);
  hipLaunchKernelGGL(moe_offsets_kernel, dim3(1), dim3(kPlanThreads), 0, st, a);
  hipLaunchKernelGGL(moe_place_kernel, dim3(blocks), dim3(kPlanThreads), 0, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

static int experts(bool up, const void* x, const void* w, const void* w_shared, void* out, const int32_t* sorted,
                   const int32_t* tiles, const int32_t* ntiles, const float* weights, int32_t n, int32_t E,
                   int32_t top, int32_t shared, int32_t rows, int32_t max_tiles, int32_t K, int32_t K_shared,
                   int32_t M, int32_t M_shared, int64_t x_stride, int64_t out_stride, int32_t act,
                   float limit, float limit_shared, int32_t dtype, void* stream) {
  ZP_REQUIRE((act == ZP_GATE_CLAMPED || act == ZP_GATE_SILU) && n >= 0 && E > 0 && top > 0 && max_tiles > 0 && K > 0 && M > 0 && (!shared || (K_shared > 0 && M_shared > 0)),
             "moe experts: bad dims");
  ZP_MODEL_DTYPE("moe experts");
  if (K % 32 || K_shared % 32 || M % 16 || M_shared % 16 || x_stride % 8 || out_stride % 8 ||
      (rows != 16 && rows != 32 && rows != 64 && ((rows != 128 && rows != kBigRows) || dtype != ZP_BF16))) {
    zp_set_error("moe experts: sizes %d x %d, shared %d x %d, %d rows per tile unsupported", M, K, M_shared, K_shared, rows);
    return ZP_EUNSUPPORTED;
  }
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(x && w && (!shared || w_shared) && out && sorted && tiles && ntiles && (!up || weights), "moe experts: null pointer");
  ZP_REQUIRE(aligned16(x) && aligned16(w) && aligned16(w_shared) && aligned16(out) && aligned16(tiles) &&
                 x_stride >= (K > K_shared ? K : K_shared) && out_stride >= (M > M_shared ? M : M_shared),
             "moe experts: unaligned or overlapping rows");
  bool staged = rows >= 64 && dtype == ZP_BF16;
  if (staged) {                   // 31-bit byte offsets into x and into a block of W
    const int64_t xr = up ? n : rows, kx = K > K_shared ? K : K_shared;
    staged = xr * x_stride * 2 < (1ll << 31) && kx * 512 < (1ll << 31);
    if (rows == 64) {
      const int64_t of_w = std::max(M, shared ? M_shared : 0) * (up ? 2ll : 1ll), with = E + (shared ? (n + 63) / 64 : 0);
      staged = staged && with * of_w >= kStagedGroups * 16 * kBlockW;
    } else if (!staged) {
      zp_set_error("moe experts: %lld rows of %lld elements in one step", (long long)xr, (long long)x_stride);
      return ZP_EUNSUPPORTED;
    }
  }
  ExpertArgs a = {x, w, w_shared, out, sorted, tiles, ntiles, weights, n, E, top, top + shared, max_tiles, K, K_shared,
                  M, shared ? M_shared : 0, x_stride, out_stride, (int64_t)M * K * (up ? 2 : 1), act, limit, limit_shared, 1};
  return up ? launch_experts<true>(a, rows, staged, dtype, (hipStream_t)stream)
            : launch_experts<false>(a, rows, staged, dtype, (hipStream_t)stream);
}

extern "C" int zp_moe_gate_up(const void* x, const void* w, const void* w_shared, void* out, const int32_t* sorted,
                              const int32_t* tiles, const int32_t* ntiles, const float* weights, int32_t n,
                              int32_t E, int32_t top, int32_t shared, int32_t rows, int32_t max_tiles, int32_t K,
                              int32_t M, int32_t M_shared, int64_t x_stride, int64_t out_stride, int32_t act,
                              float limit, float limit_shared, int32_t dtype, void* stream) {
  return experts(true, x, w, w_shared, out, sorted, tiles, ntiles, weights, n, E, top, shared, rows, max_tiles, K, K,
                 M, M_shared, x_stride, out_stride, act, limit, limit_shared, dtype, stream);
}
extern "C" int zp_moe_down(const void* x, const void* w, const void* w_shared, void* out, const int32_t* sorted,
                           const int32_t* tiles, const int32_t* ntiles, int32_t n, int32_t E, int32_t top,
                           int32_t shared, int32_t rows, int32_t max_tiles, int32_t K, int32_t K_shared, int32_t M,
                           int64_t x_stride, int64_t out_stride, int32_t dtype, void* stream) {
  return experts(false, x, w, w_shared, out, sorted, tiles, ntiles, nullptr, n, E, top, shared, rows, max_tiles, K,
                 K_shared, M, M, x_stride, out_stride, ZP_GATE_CLAMPED, 0.f, 0.f, dtype, stream);
}
