// Attention of runs of prompt tokens, and the gather of the cached rows they look back on.
#include "mfma.h"
#include "launch_order.h"

namespace {

// ------------------------------------------------------------------ gather of cached rows
__global__ __launch_bounds__(256) void gather_rows_kernel(const char* src, const int32_t* rows, char* out,
                                                          int64_t total, int pieces, int64_t num_rows) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= total) return;
  const int64_t r = id / pieces, pc = id - r * pieces;
  int64_t s = rows[r];
  if (s < 0 || s >= num_rows) s = 0;
  ((u32x4*)out)[id] = ((const u32x4*)src)[s * pieces + pc];
}

// ------------------------------------------------------------------ runs of prompt tokens
struct TilesArgs {
  const uint16_t* q;      // token rows of q_st elements, head h at h * maps * (D + P)
  const uint16_t* k;      // key rows of kv_st elements, head h at h * maps * D
  const uint16_t* v;      // value rows of v_st elements, head h at h * V
  const uint16_t* ks;     // rows of s_st elements: the last P of every head's key; null: P = 0
  uint16_t* out;          // token rows of o_st elements, head h at h * V
  const int32_t* tiles;   // (T, 4): first query row, queries, first key row of the run, position
                          // of the first query counted from that key
  const float* sinks;     // (H,) logits that only join the denominator, or null
  int T, H, HK, D, P, V;  // HK key / value heads; query head h uses head h / (H / HK)
  int window, chunk;      // at most one is set, see first_seen
  int64_t q_rows, k_rows, q_st, kv_st, v_st, s_st, o_st;
  float scale, out_scale;
  float cap;              // > 0: soft cap of the scores
  // two maps: rms(o1 - balance * o2) * out_scale * sigmoid(gate), the mean over vdim
  float balance, eps;
  int vdim;
  const uint16_t* gate;   // token rows of g_st elements, head h at h * V; or null
  int64_t g_st;
  const float2* turns;    // one map: (q_rows, V / 2) cos and sin, results turn back by them; or null
  const zp_f32x4* q_turns;   // TURN: (q_half / 2) planes of (q_rows, 2) cos and sin by which queries turn; otherwise null
  int64_t q_plane;           // rows from a plane to the next
  int q_half;
  bool rising;            // a run's tiles come in the order of their keys; otherwise those with many keys first
  int few_tiles;          // tiles of keys up to which a workgroup takes the form that stages no tile ahead
};

constexpr int kTileQ = 128;   // queries per workgroup
constexpr int kTileK = 64;    // keys per LDS tile

// A workgroup owns up to 128 queries of one head; key and value tiles pass through LDS once for all of
// them (double-buffered, the next tile's loads in flight during the products), a wave owns 16 * kQT
// queries at a time and skips the steps of 32 or 64 keys none of them sees.
//
// Bound by the vector units and by the latencies of a step's chain (products, maximum, exponentials, products) with two
// waves per SIMD: matrix cores are busy a third of the time.  So the values are transposed by the LDS reads
// themselves, operands are read a group ahead of their products, a step takes 64 keys where its scores fit the registers,
// the maximum crosses lanes only when it has moved, and sums of weights are a product with ones.  8 prompts of 2048
// tokens, 32 heads of 128 with 8 of keys and values: 531 -> 435 us without limit, 347 -> 296 in chunks of 1024.
// First key position a query sees: the last `window` up to and including its own, or those of its own
// block of `chunk` positions (key 0 of the run starts a block), or all.
__device__ __forceinline__ int first_seen(int pos, int window, int chunk) {
  if (window > 0) return max(0, pos - window + 1);
  return chunk > 0 ? pos / chunk * chunk : 0;
}

// Two maps: one workgroup of eight waves per CU; else two of four waves, which share its 160 KB.
constexpr int tile_waves(int maps) { return maps == 2 ? 8 : 4; }

template <int DKS, int VCB, int MAPS> struct TileStage {
  // row strides: rows of keys 16 bytes apart in the banks, those of values, which are read 32 bytes wide, 32
  static constexpr int kK = MAPS * DKS * 32 + 8, kV = VCB * 128 + 16;
  static constexpr int kElems = kTileK * (kK + kV);
  static constexpr int kWaves = tile_waves(MAPS);
  static constexpr int kBuffers = MAPS == 2 || 8 * kElems <= 160 * 1024 ? 2 : 1;
  static constexpr int kBytes = kBuffers * kElems * 2;
};

// A lane holds 4 columns of each of two column tiles; groups of sixteen lanes swap halves with their neighbours, so that each
// ends with 8 columns of one tile: those from (c + (g & 1)) * 16 + (g >> 1) * 8 on for tiles c and c + 1.
__device__ __forceinline__ void eight_columns(const f32x4& even, const f32x4& odd, float by, float (&r)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto both = __builtin_amdgcn_permlane16_swap(__float_as_uint(even[i] * by), __float_as_uint(odd[i] * by), false, false);
    r[i] = __uint_as_float(both[0]);
    r[4 + i] = __uint_as_float(both[1]);
  }
}

// Queries as projected turn on their way in, elements j < HALF * STEP of a head with those HALF * STEP further, as the store of
// rotary positions turns and rounds them.  A lane has STEP / 2 elements in a row of every STEP; `turns`: its first two angles, whose
// planes put a wave's queries side by side (64 bytes of a query's own row to a lane touch a line with every load).  The store
// leaves out what it would read and write of q: 16 384 tokens, 32 heads over 8 of 128, window of 1024, it takes 46 us instead
// of 83, the attention 298 instead of 276, for the angles that every head reads.
template <int HALF, int STEP, int N> __device__ __forceinline__ void turn_queries(u32x4 (&q)[N], const zp_f32x4* turns, int64_t plane) {
  zp_f32x4 cs[HALF][4];
#pragma unroll
  for (int k = 0; k < HALF; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) cs[k][i] = turns[(k * STEP / 2 + i) * plane];
#pragma unroll
  for (int k = 0; k < HALF; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = q[k][i], hi = q[k + HALF][i];
      float u[2] = {__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u)};
      float v[2] = {__uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u)};
      turn_pair(u[0], v[0], cs[k][i][0], cs[k][i][1]);
      turn_pair(u[1], v[1], cs[k][i][2], cs[k][i][3]);
      q[k][i] = pack_bf16(u[0], u[1]);
      q[k + HALF][i] = pack_bf16(v[0], v[1]);
    }
}

enum { kNoCap, kCap, kBoundedCap };   // of the scores, see SoftCap
// Keys per step: 64 scores for each query where the registers hold them (8 prompts as above: 519 -> 463 us; keys of 192
// with a shared part spill: 1811 -> 1831) and many keys come here (heads of at most 128 have a kernel of their own).
constexpr int long_step(int DKS, int VCB, int MAPS, bool SHARED, int CAP) {
  return MAPS == 1 && VCB == 1 && CAP == kNoCap && (SHARED ? DKS <= 4 : DKS == 6) ? 64 : 32;
}

// Column tile t of a wave: 16 queries, map t % MAPS of the head (differential attention has two, over the same
// values; elsewhere there is one).  SHARED: the last P elements of every head's key are the row of a.ks.
// FINE: softmax weights enter the value product as two bf16 planes (17 bits), elsewhere as one.
// TURN: queries come as projected (see turn_queries); a form of its own, for the branch alone costs the flow 2.5 % where nothing turns
// (16 prompts of 256 to 768 tokens, 32 heads of 128 over 8, 95.5 us without it, 97.7 with it).
template <int DKS, int VCB, int kQT, int MAPS, bool SHARED, int CAP, bool FINE, int kStep, bool TURN>
__device__ __forceinline__ void run_tile(const TilesArgs& a, char* lds_raw, int h, int tile) {
  typedef TileStage<DKS, VCB, MAPS> Stage;
  constexpr bool kTurns = MAPS == 1 && !SHARED && CAP == kNoCap;
  constexpr bool kPinned = DKS <= 4 && (VCB == 1 || MAPS == 1);   // reads ahead: wider heads would spill
  constexpr int kT = kQT * MAPS, kWaves = Stage::kWaves, kThreads = 64 * kWaves, kPass = 16 * kQT * kWaves;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
  const int q0 = a.tiles[tile * 4], nq = min(a.tiles[tile * 4 + 1], kTileQ);
  const int kb = a.tiles[tile * 4 + 2], rel = a.tiles[tile * 4 + 3];
  // host-made descriptors: rows outside the buffers are not touched
  if (q0 < 0 || kb < 0 || rel < 0 || (int64_t)q0 + nq > a.q_rows || (int64_t)kb + rel + nq > a.k_rows) return;
  const int DT = a.D + (SHARED ? a.P : 0);
  const SoftCap cap(a.scale, a.cap);
  // without a cap the scale joins the subtraction of the maximum, for which it has to be positive: a negative one turns
  // the queries round, zero takes them away
  const uint32_t flip = CAP == kNoCap && a.scale < 0.f ? 0x80008000u : 0u, kept = CAP == kNoCap && cap.factor == 0.f ? 0u : ~0u;
  const float factor = cap.factor == 0.f ? 1.f : fabsf(cap.factor);
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  const int hk = h / (a.H / a.HK);
  const uint16_t* kbase = a.k + (int64_t)kb * a.kv_st + hk * MAPS * a.D;
  const uint16_t* vbase = a.v + (int64_t)kb * a.v_st + hk * a.V;
  const uint16_t* sbase = SHARED ? a.ks + (int64_t)kb * a.s_st : nullptr;

  for (int wg0 = 0; wg0 < nq; wg0 += kPass) {                 // uniform in the workgroup
    const int w0 = wg0 + wave * 16 * kQT;
    const int last = rel + min(wg0 + kPass, nq) - 1;          // last key any query of the pass sees
    const int first = first_seen(rel + wg0, a.window, a.chunk);
    const int hi = w0 < nq ? rel + min(w0 + 16 * kQT, nq) - 1 : -1;      // the same for the wave
    const int lo = first_seen(rel + w0, a.window, a.chunk);
    const int lo_last = first_seen(rel + w0 + 16 * kQT - 1, a.window, a.chunk);

    u32x4 qf[kT][DKS];
    int qpos[kQT], qlow[kQT];                                 // keys qlow .. qpos are seen
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const int qi = min(w0 + t / MAPS * 16 + l16, nq - 1);
      qpos[t / MAPS] = rel + qi;
      qlow[t / MAPS] = first_seen(rel + qi, a.window, a.chunk);
      const uint16_t* q = a.q + (int64_t)(q0 + qi) * a.q_st + (h * MAPS + t % MAPS) * DT;
#pragma unroll
      for (int ks = 0; ks < DKS; ++ks) {
        // past the head's end: the key columns there hold other elements, against zeros here
        const int c = ks * 32 + g * 8;
        qf[t][ks] = (*(const u32x4*)(q + (c < DT ? c : 0)) & kept) ^ flip;
        if (c >= DT) qf[t][ks] = u32x4{0u, 0u, 0u, 0u};
      }
      if constexpr (TURN) {                                   // the sign above goes through a turn unchanged
        static_assert(kTurns && DKS <= 4 && VCB == 1, "heads of at most 128");
        const zp_f32x4* const turns = a.q_turns + g * 4 * a.q_plane + q0 + qi;
        if constexpr (DKS == 4) {
          if (a.q_half == 64) turn_queries<2, 32>(qf[t], turns, a.q_plane);
          else turn_queries<1, 32>(qf[t], turns, a.q_plane);
        } else {
          turn_queries<1, 32>(qf[t], turns, a.q_plane);
        }
      }
    }
    f32x4 o[kT][VCB * 8];
    float m[kT], l[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      m[t] = CAP == kBoundedCap ? 0.f : -INFINITY;
      l[t] = 0.f;
#pragma unroll
      for (int i = 0; i < VCB * 8; ++i) o[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    constexpr int kKP = 4 * MAPS * DKS, kVP = 16 * VCB;        // pieces of a key row, DKS * 4 per map, and of a value row
    constexpr int kKN = kTileK * kKP / kThreads, kVN = kTileK * kVP / kThreads;
    u32x4 rk[kKN], rv[kVN];                                    // this thread's pieces of a tile
    auto fetch = [&](int k0) {                                 // offsets from the tile's first row: 32 bits
      const uint16_t *kt = kbase + k0 * a.kv_st, *vt = vbase + k0 * a.v_st, *st = SHARED ? sbase + k0 * a.s_st : nullptr;
      const uint32_t kv_st = (uint32_t)a.kv_st, v_st = (uint32_t)a.v_st, s_st = (uint32_t)a.s_st;
#pragma unroll
      for (int j = 0; j < kKN; ++j) {
        const int id = tid + kThreads * j, pc = id % kKP, map = pc / (4 * DKS), c = (pc % (4 * DKS)) * 8;
        const uint32_t r = min(id / kKP, last - k0);
        if (SHARED) {
          const bool own = c < a.D;
          rk[j] = *(const u32x4*)((own ? kt : st) + (own ? r * kv_st + c : r * s_st + (c < DT ? c - a.D : 0)));
        } else {
          rk[j] = *(const u32x4*)(kt + (r * kv_st + map * a.D + (c < a.D ? c : 0)));
        }
      }
#pragma unroll
      for (int j = 0; j < kVN; ++j) {
        const int id = tid + kThreads * j, c = (id % kVP) * 8;
        const uint32_t r = min(id / kVP, last - k0);
        rv[j] = *(const u32x4*)(vt + (r * v_st + (c < a.V ? c : 0)));
      }
    };
    fetch(first);
    if (Stage::kBuffers == 2) __syncthreads();                 // a pass before this one still reads its tiles
    int buf = 0;
    for (int t0 = first; t0 <= last; t0 += kTileK, buf ^= 1) {
      if (Stage::kBuffers == 1) __syncthreads();               // the tile before this one is used up
      uint16_t* const ldsk = (uint16_t*)lds_raw + (Stage::kBuffers == 2 ? buf * Stage::kElems : 0);
      uint16_t* const ldsv = ldsk + kTileK * Stage::kK;
#pragma unroll
      for (int j = 0; j < kKN; ++j) {
        const int id = tid + kThreads * j;
        *(u32x4*)(ldsk + id / kKP * Stage::kK + (id % kKP) * 8) = rk[j];
      }
#pragma unroll
      for (int j = 0; j < kVN; ++j) {
        const int id = tid + kThreads * j;
        *(u32x4*)(ldsv + id / kVP * Stage::kV + (id % kVP) * 8) = rv[j];
      }
      __syncthreads();
      if (t0 + kTileK <= last) fetch(t0 + kTileK);
#pragma unroll 1
      for (int sub = 0; sub < kTileK; sub += kStep) {
        const int k0 = t0 + sub;
        if (k0 > hi || k0 + kStep - 1 < lo) continue;          // uniform in the wave
        // operands leave LDS a group ahead of the products that use them; the barriers keep the compiler from moving each
        // read to its use, where its latency would show (463 -> 421 us).  This wave's products go before the other's
        // exponentials (441 -> 435)
        float p[kT][kStep / 4];
        u32x4 kf[2][DKS * MAPS];
        const uint16_t* const ks0 = ldsk + (sub + l16) * Stage::kK + g * 8;
        auto read_keys = [&](int tt) {
#pragma unroll
          for (int i = 0; i < DKS * MAPS; ++i) kf[tt & 1][i] = *(const u32x4*)(ks0 + tt * 16 * Stage::kK + i * 32);
        };
        __builtin_amdgcn_s_setprio(1);
        if constexpr (kPinned) read_keys(0);
#pragma unroll
        for (int tt = 0; tt < kStep / 16; ++tt) {
          if (!kPinned) read_keys(tt);
          else if (tt + 1 < kStep / 16) read_keys(tt + 1);
          if constexpr (kPinned) __builtin_amdgcn_sched_barrier(0);
          f32x4 s[kT];
#pragma unroll
          for (int t = 0; t < kT; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < DKS; ++ks)
#pragma unroll
            for (int t = 0; t < kT; ++t) s[t] = mfma_bf16(kf[tt & 1][t % MAPS * DKS + ks], qf[t][ks], s[t]);
#pragma unroll
          for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) p[t][tt * 4 + i] = s[t][i];
          if constexpr (kPinned) __builtin_amdgcn_sched_barrier(0);
        }
        // value columns of 16, transposed on their way out of LDS: lane l16 gets column l16 of eight keys
        const uint16_t* const vs = ldsv + (sub + 4 * g + (l16 >> 2)) * Stage::kV + (l16 & 3) * 4;
        constexpr int kGroups = kStep / 32 * VCB * 2;          // of four such columns and 32 keys
        u32x4 vf[2][4];
        auto read_values = [&](int n) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint16_t* const at = vs + n / (VCB * 2) * 32 * Stage::kV + (n % (VCB * 2) * 4 + i) * 16;
            const uint2 lo = read_transposed(at), hi = read_transposed(at + 16 * Stage::kV);
            vf[n & 1][i] = u32x4{lo.x, lo.y, hi.x, hi.y};
          }
        };
        __builtin_amdgcn_s_setprio(0);
        if constexpr (kPinned) read_values(0);
        if constexpr (kPinned) __builtin_amdgcn_sched_barrier(0);
        if (CAP != kNoCap) {
#pragma unroll
          for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int i = 0; i < kStep / 4; ++i) p[t][i] = cap.capped(p[t][i]);
        }
        if (k0 + kStep - 1 > rel + w0 || k0 < lo_last) {         // some query of the wave does not see all these keys
#pragma unroll
          for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int i = 0; i < kStep / 4; ++i) {
              const int key = k0 + (i >> 2) * 16 + 4 * g + (i & 3);
              if (key > qpos[t / MAPS] || key < qlow[t / MAPS]) p[t][i] = -INFINITY;
            }
        }
        if (CAP != kBoundedCap) {
#pragma unroll
          for (int t = 0; t < kT; ++t) {
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < kStep / 4; ++i) mx = fmaxf(mx, p[t][i]);
            if (CAP == kNoCap) mx *= factor;
            if (__any(mx > m[t])) {                             // in any lane: hardly ever after the first keys
              mx = fmaxf(m[t], mx);
              mx = fmaxf(mx, lane_xor16(mx));
              mx = fmaxf(mx, lane_xor32(mx));
              const float f = mx == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[t] - mx);
              m[t] = mx;
              l[t] *= f;
#pragma unroll
              for (int i = 0; i < VCB * 8; ++i) o[t][i] *= f;
            }
          }
        }
        u32x4 pf[kT][kStep / 32], pl[FINE ? kT : 1][kStep / 32];
#pragma unroll
        for (int t = 0; t < kT; ++t) {
          const float ms = m[t] == -INFINITY ? 0.f : m[t];      // a query whose window starts later
#pragma unroll
          for (int i = 0; i < kStep / 4; ++i)
            p[t][i] = __builtin_amdgcn_exp2f(CAP == kNoCap        ? fmaf(p[t][i], factor, -ms)
                                             : CAP == kBoundedCap ? p[t][i]
                                                                  : p[t][i] - ms);
#pragma unroll
          for (int d = 0; d < kStep / 8; ++d) {
            const uint32_t w = pack_bf16(p[t][2 * d], p[t][2 * d + 1]);
            pf[t][d / 4][d % 4] = w;
            if constexpr (FINE)
              pl[t][d / 4][d % 4] =
                  pack_bf16(p[t][2 * d] - __uint_as_float(w << 16), p[t][2 * d + 1] - __uint_as_float(w & 0xffff0000u));
          }
          // the sum of the weights as the values meet them: what rounding does to a weight that outweighs the others cancels
          f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int d = 0; d < kStep / 32; ++d) {
            sum = mfma_bf16(ones, pf[t][d], sum);
            if constexpr (FINE) sum = mfma_bf16(ones, pl[t][d], sum);
          }
          l[t] += sum[0];
        }
#pragma unroll
        for (int n = 0; n < kGroups; ++n) {
          if (!kPinned) read_values(n);
          else if (n + 1 < kGroups) read_values(n + 1);
          if constexpr (kPinned) __builtin_amdgcn_sched_barrier(0);
          const int half = n / (VCB * 2), c0 = n % (VCB * 2) * 4;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < kT; ++t) {
              o[t][c0 + i] = mfma_bf16(vf[n & 1][i], pf[t][half], o[t][c0 + i]);
              if constexpr (FINE) o[t][c0 + i] = mfma_bf16(vf[n & 1][i], pl[t][half], o[t][c0 + i]);
            }
          if constexpr (kPinned) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      float inv[MAPS];
#pragma unroll
      for (int map = 0; map < MAPS; ++map) {
        float lt = l[qt * MAPS + map];
        if (MAPS == 1 && a.sinks) lt += __builtin_amdgcn_exp2f(a.sinks[h] * 1.44269504088896f - m[qt]);
        inv[map] = lt > 0.f ? 1.f / lt : 0.f;
      }
      if constexpr (MAPS == 1) {
        inv[0] *= a.out_scale;
      } else {                                                 // o1 <- rms(o1 / l1 - balance * o2 / l2) * out_scale
        const float second = a.balance * inv[1];
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < VCB * 8; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float r = o[qt * 2][j][i] * inv[0] - o[qt * 2 + 1][j][i] * second;
            o[qt * 2][j][i] = r;
            if (j * 16 + 4 * g + i < a.V) ss += r * r;
          }
        ss += lane_xor16(ss);
        ss += lane_xor32(ss);
        inv[0] = a.out_scale / sqrtf(ss / (float)a.vdim + a.eps);
      }
      const int qi = w0 + qt * 16 + l16;
      const bool row = qi < nq;                                // every lane takes part in the swaps
      uint16_t* out = a.out + (int64_t)(q0 + qi) * a.o_st + h * a.V;
      const float2* turns = a.turns;
      asm volatile("" : "+s"(turns));                          // nothing of the way back is computed before the loop
      const uint16_t* gate = MAPS == 2 && a.gate ? a.gate + (int64_t)(q0 + qi) * a.g_st + h * a.V : nullptr;
#pragma unroll
      for (int c = 0; c < VCB * 8; c += 2) {
        float r[8];
        eight_columns(o[qt * MAPS][c], o[qt * MAPS][c + 1], inv[0], r);
        const int col = (c + (g & 1)) * 16 + (g >> 1) * 8;
        if (!row || col >= a.V) continue;
        if (kTurns && turns) turn_back8(r, turns + ((int64_t)(q0 + qi) * a.V + col) / 2);
        if (MAPS == 2 && gate) {
          float z[8];
          Vec8<BF16>::ld(gate, col, z);
#pragma unroll
          for (int i = 0; i < 8; ++i) r[i] *= sigmoid_of<BF16>(z[i]);
        }
        Vec8<BF16>::st(out, col, r);
      }
    }
  }
}

template <int DKS, int VCB, int kQT, int MAPS, bool SHARED, int CAP, bool FINE, int kStep, bool TURN>
__global__ __launch_bounds__(64 * tile_waves(MAPS), 2) void run_tiles_kernel(TilesArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  run_tile<DKS, VCB, kQT, MAPS, SHARED, CAP, FINE, kStep, TURN>(a, lds_raw, blockIdx.x % a.H, blockIdx.x / a.H);   // one head's tiles share an L2 when H % 8 == 0
}

// ------------------------------------------------------------------ heads of at most 128, one map, no cap
// Here the products of a tile's keys run while the exponentials of the tile before take their turn, which needs the scores
// of two tiles in registers.  A 32 x 32 product takes 8 of its 32 cycles at the vector issue, a 16 x 16 one 8 of 16: with the
// wide ones there is room for the exponentials, and for 128 value columns (16 x 16, those of a head of 128 did not pay).
// Rows go from memory into LDS without passing through registers, one load at a time between the products: eight in a row
// held a wave for 870 cycles a tile.  Queries and the first keys are asked for together.
// Of the cycles of a launch that turns its queries (window of 1024 below, 629 000 at 2.0 to 2.3 GHz) the vector units issue in 44 % and
// the matrix cores are busy in 35 %; its waves, two per SIMD, wait in 35 % of theirs, and a tenth of the time a CU has one workgroup
// or none.  Heads of 128, 32 over 8 of keys and values, 8 prompts of
// 2048 tokens: window of 1024 309 -> 278 us, all keys 371 -> 327; one prompt 52 -> 44, of 300 tokens 12.7 -> 10.6; heads of
// 64: 198 -> 181, 240 -> 216, 33 -> 29, 9.0 -> 8.2; causal with weights of 17 bits 452 -> 448, one prompt of 300 14.7 -> 12.5.
// Tried: eight waves of two heads that share their rows, in turns at the matrix cores and the vector units (322 us: a wave
// alone issues a vector instruction every six cycles) or side by side (347: they meet at the same unit); whole rows next
// to one another in LDS (281).
//
// Rows of CH 16-byte pieces (8 or 16) as loads leave them in LDS, 1 KB at a time with GAP bytes between: four rows after
// one another interleave their pieces by four, so that a lane's pieces and the column tiles are immediate offsets.  With
// eight rows per load the pieces of the second four lie FLIP apart.  What reads them falls into different banks: sixteen
// rows of one piece (keys), four rows of four (values, transposed).
template <int CH, int FLIP, int GAP> struct Staged {
  static constexpr int kRows = 64 / CH;                        // per load
  static constexpr int kLoad = 1024 + GAP, kBytes = kTileK / kRows * kLoad;
  __device__ static __forceinline__ int row(int lane) { return CH == 16 ? lane >> 2 & 3 : (lane >> 5) * 4 + (lane >> 2 & 3); }
  __device__ static __forceinline__ int piece(int lane) {
    return CH == 16 ? (lane >> 4) * 4 + (lane & 3) : (lane >> 4 & 1) * 4 + ((lane & 3) ^ FLIP * (lane >> 5));
  }
  // where pieces p of 0 .. 3 of row r begin; those from 4 on are 256 bytes further for every four
  __device__ static __forceinline__ int at(int r, int p) {
    if (CH == 16) return (r >> 2) * kLoad + (r & 3) * 64 + p * 16;
    return (r >> 3) * kLoad + (r >> 2 & 1) * 512 + (r & 3) * 64 + (p ^ FLIP * (r >> 2 & 1)) * 16;
  }
};
template <int KS, int VB> struct FlowStage {                   // 16 KS elements of a key, 32 VB of a value
  typedef Staged<2 * KS, 1, KS == 8 ? 16 : 32> K;
  typedef Staged<4 * VB, 2, 0> V;
  static constexpr int kBytes = 2 * (K::kBytes + V::kBytes);
};

// A wave's results on their way out: lane l32 of either half has a query's columns 8 (i / 4) + 4 half + i % 4 of each 32.
template <int VB>
__device__ __forceinline__ void flow_out(const TilesArgs& a, int h, int64_t row, bool there, f32x16 (&o)[VB], float m, float l) {
  const int half = (threadIdx.x & 63) >> 5;
  if (a.sinks) l += __builtin_amdgcn_exp2f(a.sinks[h] * 1.44269504088896f - m);
  const float inv = l > 0.f ? a.out_scale / l : 0.f;
  uint16_t* const out = a.out + row * a.o_st + h * a.V;
#pragma unroll
  for (int c = 0; c < VB; ++c)
#pragma unroll
    for (int i = 0; i < 16; i += 8) {                          // halves swap four columns: each ends with eight neighbours
      float r[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[c][i + e] * inv), __float_as_uint(o[c][i + 4 + e] * inv),
                                                           false, false);
        r[e] = __uint_as_float(both[0]);
        r[4 + e] = __uint_as_float(both[1]);
      }
      const int col = c * 32 + (i + half * 4) * 2;
      if (!there || col >= a.V) continue;                    // every lane took part in the swaps
      if (a.turns) turn_back8(r, a.turns + (row * a.V + col) / 2);
      Vec8<BF16>::st(out, col, r);
    }
}

// FINE and TURN as above.  A wave's 32 queries are the columns of 32 x 32 products: lane l32 of either half holds one query's scores
// for keys 8 (i / 4) + 4 half + i % 4 of a tile of 32, which are its operand elements of the products with values.
template <int KS, int VB, bool FINE, bool TURN>
__global__ __launch_bounds__(256, 2) void run_flow_kernel(TilesArgs a) {
  extern __shared__ __align__(16) char lds_raw[];
  typedef typename FlowStage<KS, VB>::K KL;
  typedef typename FlowStage<KS, VB>::V VL;
  constexpr int kQK = 2 * KS, kPV = 2 * VB;                    // products of a tile's keys, of half its values
  const int lane = threadIdx.x & 63, l16 = lane & 15, l32 = lane & 31, g = lane >> 4, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const FlowPlace place(a.T, a.HK, a.rising, blockIdx.x, blockIdx.z);
  const int h = place.hk * (int)gridDim.y + blockIdx.y, tile = place.tile;
  if (tile >= a.T) return;                                     // a part that has fewer
  const int q0 = a.tiles[tile * 4], nq = min(a.tiles[tile * 4 + 1], kTileQ);
  const int kb = a.tiles[tile * 4 + 2], rel = a.tiles[tile * 4 + 3];
  // host-made descriptors: rows outside the buffers are not touched
  if (q0 < 0 || nq <= 0 || kb < 0 || rel < 0 || (int64_t)q0 + nq > a.q_rows || (int64_t)kb + rel + nq > a.k_rows) return;
  // the scale joins the subtraction of the maximum, for which it has to be positive: a negative one turns the queries
  // round, zero takes them away
  const float by = a.scale * 1.44269504088896f, factor = by == 0.f ? 1.f : fabsf(by);
  const uint32_t flip = by < 0.f ? 0x80008000u : 0u, kept = by == 0.f ? 0u : ~0u;
  const int hk = place.hk;
  const uint16_t* const kbase = a.k + (int64_t)kb * a.kv_st + hk * a.D;
  const uint16_t* const vbase = a.v + (int64_t)kb * a.v_st + hk * a.V;

  const int w0 = wave * 32;                                    // this wave's first query
  const int first = first_seen(rel, a.window, a.chunk), last = rel + nq - 1;    // keys that any query sees
  const int lo = first_seen(rel + w0, a.window, a.chunk), lo_last = first_seen(rel + w0 + 31, a.window, a.chunk);
  const int tiles = (last - first) / kTileK + 1;
  if constexpr (VB == 4)
    if (tiles <= a.few_tiles) return run_tile<KS / 2, 1, 2, 1, false, kNoCap, FINE, 32, TURN>(a, lds_raw, h, tile);
  // tiles that queries of the wave see; none: they begin behind the last one
  const int seen0 = w0 < nq ? (lo - first) / kTileK : tiles + 1;
  const int seen1 = w0 < nq ? (rel + min(w0 + 32, nq) - 1 - first) / kTileK : tiles + 1;

  // ---- a tile's rows from memory into LDS; in place of rows past the last one come zeros, which nothing sees
  char* const kl = lds_raw;
  char* const vl = lds_raw + 2 * KL::kBytes;
  // what follows from the lane is worked out anew: kept, it would not leave the products enough registers
  auto lane_again = [&] {
    int i = lane;
    asm volatile("" : "+v"(i));
    return i;
  };
  auto lane_at = [&](auto layout, int64_t stride, int cols) {
    typedef decltype(layout) L;
    const int i = lane_again();
    return L::row(i) * (int)stride * 2 + (L::piece(i) * 8 < cols ? L::piece(i) * 16 : 0);
  };
  const int klane = lane_at(KL{}, a.kv_st, a.D), vlane = lane_at(VL{}, a.v_st, a.V);
  // rows k0 + wave * kRows on of a tile, as far as they are there
  auto rows_of = [&](auto layout, const uint16_t* rows, int64_t stride, int cols, int k0) {
    const int from = k0 + wave * decltype(layout)::kRows, left = last - from;
    const uint32_t bytes = left >= kTileK ? 0x7fffffffu : left < 0 ? 0u : (uint32_t)(left * (int)stride + cols) * 2;
    return rows_from(rows + (int64_t)from * stride, bytes);
  };
  constexpr int kKeyLoads = kTileK / KL::kRows / 4, kValueLoads = kTileK / VL::kRows / 4;      // of a wave
  u32x4 krows, vrows;
  auto rows_of_keys = [&](int j) { krows = rows_of(KL{}, kbase, a.kv_st, a.D, first + min(j, tiles) * kTileK); };
  auto rows_of_values = [&](int j) { vrows = rows_of(VL{}, vbase, a.v_st, a.V, first + min(j, tiles) * kTileK); };
  auto stage_keys = [&](int j, int n) {
    load_to_lds(krows, kl + (j & 1) * KL::kBytes + (wave + n * 4) * KL::kLoad, klane + n * 8 * KL::kRows * (int)a.kv_st, 0);
  };
  auto stage_values = [&](int j, int n) {
    load_to_lds(vrows, vl + (j & 1) * VL::kBytes + (wave + n * 4) * VL::kLoad, vlane + n * 8 * VL::kRows * (int)a.v_st, 0);
  };
  rows_of_keys(0);
#pragma unroll
  for (int n = 0; n < kKeyLoads; ++n) stage_keys(0, n);

  u32x4 qf[KS];
  {
    const int qi = min(w0 + l32, nq - 1);
    const uint16_t* q = a.q + (int64_t)(q0 + qi) * a.q_st + h * a.D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      // past the head's end: the key columns there hold other elements, against zeros here
      const int c = ks * 16 + half * 8;
      qf[ks] = *(const u32x4*)(q + (c < a.D ? c : 0));
      if (c >= a.D) qf[ks] = u32x4{0u, 0u, 0u, 0u};
    }
    if constexpr (TURN) {
      const zp_f32x4* const turns = a.q_turns + half * 4 * a.q_plane + q0 + qi;
      if constexpr (KS == 8) {
        if (a.q_half == 64) turn_queries<4, 16>(qf, turns, a.q_plane);
        else turn_queries<2, 16>(qf, turns, a.q_plane);
      } else {
        turn_queries<2, 16>(qf, turns, a.q_plane);
      }
    }
    if (by <= 0.f)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = (qf[ks] & kept) ^ flip;
  }
  f32x16 o[VB];
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int c = 0; c < VB; ++c) o[c] = f32x16{};

  // ---- one tile: its weights and what its values add, and meanwhile the scores of the next one
  const int kread = KL::at(l32, half);
  // values leave LDS transposed, lane l32 with a column of four keys
  const int vread = VL::at(4 * half + (l16 >> 2), 2 * (g & 1) + ((l16 & 3) >> 1)) + (l16 & 1) * 8;
  // Sums of weights are 16 x 16 products, which take the same registers as sixteen queries of four groups of keys: ones
  // where a group of rows and a group of keys belong to the same half of the queries.
  const uint32_t one = ((l16 >> 2) & 1) == (g & 1) ? 0x3f803f80u : 0u;
  const u32x4 ones = {one, one, one, one};
  float mx = -INFINITY;                                        // largest score of the tile whose turn is next
  auto step = [&](int j, auto here_, auto next_, f32x16 (&p)[2], f32x16 (&s)[2]) {
    constexpr bool HERE = here_.value, NEXT = next_.value;
    const char* const kt = kl + ((j + 1) & 1) * KL::kBytes + kread;
    const char* const vt = vl + (j & 1) * VL::kBytes + vread;
    // operands leave LDS kAhead ahead of their product
    constexpr int kAhead = VB == 4 ? 3 : 4, kRing = kAhead + 1;
    u32x4 kf[kRing], vf[kRing];
    // n: step n / 2, 32 keys n % 2
    auto read_keys = [&](int n) {
      if (n < kQK) kf[n % kRing] = *(const u32x4*)(kt + (n & 1) * (32 / KL::kRows) * KL::kLoad + (n >> 2) * 256 + (n >> 1 & 1) * 32);
    };
    // n: 16 keys n / VB, column tile n % VB
    auto read_values = [&](int n) {
      if (n >= 4 * VB) return;
      const char* const at = vt + n % VB * 256 + n / VB * (16 / VL::kRows) * VL::kLoad;
      const uint2 x = read_transposed((const uint16_t*)at);
      const uint2 y = read_transposed((const uint16_t*)(at + 8 / VL::kRows * VL::kLoad));
      vf[n % kRing] = u32x4{x.x, x.y, y.x, y.y};
    };
    u32x4 pf[4], pl[4];
    auto key_product = [&](int n) {
      read_keys(n + kAhead);
      if (n < 2) s[n] = f32x16{};
      s[n & 1] = mfma32_bf16(kf[n % kRing], qf[n >> 1], s[n & 1]);
    };
    auto value_product = [&](int n) {
      read_values(n + kAhead);
      o[n % VB] = mfma32_bf16(vf[n % kRing], pf[n / VB], o[n % VB]);
      if constexpr (FINE) o[n % VB] = mfma32_bf16(vf[n % kRing], pl[n / VB], o[n % VB]);
    };
    float ms = 0.f;
    // weights of pair d of the 32 keys t
    auto weights = [&](int t, int d) {
      const float x = __builtin_amdgcn_exp2f(fmaf(p[t][2 * d], factor, -ms));
      const float y = __builtin_amdgcn_exp2f(fmaf(p[t][2 * d + 1], factor, -ms));
      uint32_t w = pack_bf16(x, y);
      asm volatile("" : "+v"(w));                              // made here, not at its use
      pf[2 * t + d / 4][d % 4] = w;
      if constexpr (FINE) pl[2 * t + d / 4][d % 4] = pack_bf16(x - __uint_as_float(w << 16), y - __uint_as_float(w & 0xffff0000u));
    };
    if constexpr (NEXT)
#pragma unroll
      for (int i = 0; i < kAhead; ++i) read_keys(i);
    if constexpr (HERE) {
      const int k0 = first + j * kTileK;
      if (k0 + kTileK - 1 > rel + w0 || k0 < lo_last) {        // some query of the wave does not see all these keys
        const int i0 = lane_again(), pos = rel + min(w0 + (i0 & 31), nq - 1);
        const int low = first_seen(pos, a.window, a.chunk);
        const int from = low - k0 - 4 * (i0 >> 5), span = pos - low;     // keys low .. pos are seen
        mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            if ((unsigned)(t * 32 + (i >> 2) * 8 + (i & 3) - from) > (unsigned)span) p[t][i] = -INFINITY;
            mx = fmaxf(mx, p[t][i]);
          }
      }
      mx *= factor;
      if (__any(mx > m)) {                                     // in any lane: seldom after the first keys
        mx = fmaxf(m, mx);
        mx = fmaxf(mx, lane_xor32(mx));
        const float f = mx == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mx);
        m = mx;
        l *= f;
#pragma unroll
        for (int c = 0; c < VB; ++c) o[c] *= f;
      }
      ms = m == -INFINITY ? 0.f : m;                           // a query whose window starts later
    }
    rows_of_keys(j + 2);
    rows_of_values(j + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // what the next step needs, over what was used before the last barrier; one by one, as loads block in a row
      if (i < kKeyLoads) stage_keys(j + 2, i);
      else if (i - kKeyLoads < kValueLoads) stage_values(j + 1, i - kKeyLoads);
      if constexpr (NEXT)
#pragma unroll
        for (int e = i * kQK / 8; e < (i + 1) * kQK / 8; ++e) key_product(e);
      if constexpr (HERE) weights(0, i);
      __builtin_amdgcn_sched_barrier(0);
    }
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    auto sums = [&](int t) {
#pragma unroll
      for (int i = 2 * t; i < 2 * t + 2; ++i) {
        sum = mfma_bf16(ones, pf[i], sum);
        if constexpr (FINE) sum = mfma_bf16(ones, pl[i], sum);
      }
    };
    if constexpr (HERE) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i) read_values(i);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int e = i * kPV / 8; e < (i + 1) * kPV / 8; ++e) value_product(e);
        if (i == 0) sums(0);
        weights(1, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      sums(1);
    }
    if constexpr (NEXT) mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (HERE)
#pragma unroll
        for (int e = i * kPV / 8; e < (i + 1) * kPV / 8; ++e) value_product(kPV + e);
      if constexpr (NEXT)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[i >> 2][(i & 3) * 4 + e]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (HERE) l += sum[0];
  };

  typedef std::integral_constant<bool, true> yes;
  typedef std::integral_constant<bool, false> no;
  auto meet = [] {                                             // this wave's rows are there and its reads done, then everyone's
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Every wave takes the tiles from -1 on one by one, stages its share of what the next one needs and meets the others once
  // for each; which of them it works on is its own matter.
  int j = -1;
  f32x16 p0[2], p1[2];
  auto tile_of = [&](auto here, auto next, f32x16 (&p)[2], f32x16 (&after)[2]) {
    step(j, here, next, p, after);
    meet();
    ++j;
  };
  meet();
#pragma unroll 1
  while (j < tiles && j != seen0 - 1) tile_of(no{}, no{}, p0, p1);
  if (j < tiles) {
    tile_of(no{}, yes{}, p1, p0);
#pragma unroll 1
    while (j + 2 <= seen1) {
      tile_of(yes{}, yes{}, p0, p1);
      tile_of(yes{}, yes{}, p1, p0);
    }
    if (j < seen1) {
      tile_of(yes{}, yes{}, p0, p1);
      tile_of(yes{}, no{}, p1, p0);
    } else {
      tile_of(yes{}, no{}, p0, p1);
    }
#pragma unroll 1
    while (j < tiles) tile_of(no{}, no{}, p0, p1);
  }

  const int qi = w0 + l32;
  flow_out(a, h, q0 + qi, qi < nq, o, m, l);
}

inline dim3 flow_grid(const TilesArgs& a) { return dim3(8, a.H / a.HK, (unsigned)FlowPlace::depth(a.T, a.HK)); }
// Values of more than 64, few keys: the flow has one tile on its way, sets up for one behind it and counts keys by 64, which pays from
// three tiles on, and in small launches, where a workgroup's own time counts, from two or one.  Heads over 8 of 128, us in the
// flow alone and with short tiles in the other form: 32 heads, 256 prompts of 64 tokens 139 and 110, 128 of 128 106 and 91,
// 64 of 256 117 and 113, 512 of 32 206 and 162; 16 heads, 128 of 128 54 and 49; 2 tiles, 512 workgroups (16 of 128 tokens, 32
// heads) 16.9 and 18.6; one tile, 512 workgroups 11.1 and 10.6, 256 8.8 and 8.9, one prompt of 64 8.1 and 8.4.
inline int few_tiles(const TilesArgs& a) {
  const int64_t groups = (int64_t)a.T * a.H;
  return groups >= 1024 ? 2 : groups >= 512 ? 1 : 0;
}
template <int KS, int VB, bool FINE, bool TURN> int launch_flow(const TilesArgs& args, hipStream_t st) {
  constexpr int flow = FlowStage<KS, VB>::kBytes, steps = VB == 4 ? TileStage<KS / 2, 1, 1>::kBytes : 0, smem = flow > steps ? flow : steps;
  if (smem > 64 * 1024 && hipFuncSetAttribute((const void*)run_flow_kernel<KS, VB, FINE, TURN>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                              smem) != hipSuccess) {
    zp_set_error("run_attention: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  TilesArgs a = args;
  a.few_tiles = few_tiles(a);
  hipLaunchKernelGGL((run_flow_kernel<KS, VB, FINE, TURN>), flow_grid(a), dim3(256), smem, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
// Steps of 32 keys where tiles have no more on average: a prompt of 16 tokens, 32 heads of 128 5.2 us (5.7 in the flow), of
// 64 6.2 (6.1).  Not among many keys, where one long run may decide (31 prompts of 16 tokens and one of 512 23.1, 20.3 with 64).
inline bool few_keys(const TilesArgs& a) { return a.k_rows <= 256 && a.k_rows <= 32 * (int64_t)a.T; }
// Offsets within a tile are 32 bits, the launch is three-dimensional.
inline bool flow_takes(const TilesArgs& a) {
  const dim3 grid = flow_grid(a);
  return a.D <= 128 && a.V <= 128 && (a.V <= 64 || !few_keys(a)) && a.kv_st < 1 << 24 && a.v_st < 1 << 24 && grid.y < 65536 &&
         grid.z < 65536;
}
template <bool FINE, bool TURN> int launch_flow(const TilesArgs& a, hipStream_t st) {
  if (a.V <= 64) return a.D <= 64 ? launch_flow<4, 2, FINE, TURN>(a, st) : launch_flow<8, 2, FINE, TURN>(a, st);
  return a.D <= 64 ? launch_flow<4, 4, FINE, TURN>(a, st) : launch_flow<8, 4, FINE, TURN>(a, st);
}

template <int DKS, int VCB, int kQT, int MAPS, bool SHARED, int CAP, bool FINE, int kStep, bool TURN>
int launch_steps(const TilesArgs& a, hipStream_t st) {
  constexpr int smem = TileStage<DKS, VCB, MAPS>::kBytes;
  if (smem > 64 * 1024 &&
      hipFuncSetAttribute((const void*)run_tiles_kernel<DKS, VCB, kQT, MAPS, SHARED, CAP, FINE, kStep, TURN>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) {
    zp_set_error("run_attention: cannot reserve %d bytes of LDS", smem);
    return ZP_EHIP;
  }
  hipLaunchKernelGGL((run_tiles_kernel<DKS, VCB, kQT, MAPS, SHARED, CAP, FINE, kStep, TURN>), dim3((unsigned)a.T * a.H),
                     dim3(64 * TileStage<DKS, VCB, MAPS>::kWaves), smem, st, a);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}
template <int DKS, int VCB, int kQT, int MAPS, bool SHARED, int CAP, bool FINE = false, bool TURN = false>
int launch_run_tiles(const TilesArgs& a, hipStream_t st) {
  constexpr int kLong = long_step(DKS, VCB, MAPS, SHARED, CAP);
  if (few_keys(a)) return launch_steps<DKS, VCB, kQT, MAPS, SHARED, CAP, FINE, 32, TURN>(a, st);
  return launch_steps<DKS, VCB, kQT, MAPS, SHARED, CAP, FINE, kLong, TURN>(a, st);
}

template <bool SHARED, int CAP> int launch_one_map(const TilesArgs& a, hipStream_t st) {
  const int dk = (a.D + a.P + 31) / 32;
  if constexpr (!SHARED && CAP == kNoCap) {
    if (flow_takes(a)) return a.q_turns ? launch_flow<false, true>(a, st) : launch_flow<false, false>(a, st);
    if (a.q_turns)                                             // heads of at most 128
      return dk <= 2 ? launch_run_tiles<2, 1, 2, 1, false, kNoCap, false, true>(a, st) : launch_run_tiles<4, 1, 2, 1, false, kNoCap, false, true>(a, st);
  }
  if (a.V <= 128) {
    if (dk <= 2) return launch_run_tiles<2, 1, 2, 1, SHARED, CAP>(a, st);
    if (dk <= 4) return launch_run_tiles<4, 1, 2, 1, SHARED, CAP>(a, st);
    if (dk <= 6) return launch_run_tiles<6, 1, 2, 1, SHARED, CAP>(a, st);
    return launch_run_tiles<8, 1, 2, 1, SHARED, CAP>(a, st);
  }
  if (dk <= 4) return launch_run_tiles<4, 2, 1, 1, SHARED, CAP>(a, st);
  return launch_run_tiles<8, 2, 1, 1, SHARED, CAP>(a, st);
}
template <int CAP> int launch_two_maps(const TilesArgs& a, hipStream_t st) {
  const int dk = (a.D + 31) / 32;
  if (a.V <= 128) {
    if (dk <= 2) return launch_run_tiles<2, 1, 1, 2, false, CAP>(a, st);
    return launch_run_tiles<4, 1, 1, 2, false, CAP>(a, st);
  }
  return launch_run_tiles<4, 2, 1, 2, false, CAP>(a, st);
}
template <int CAP> int launch_forms(const TilesArgs& a, bool two, hipStream_t st) {
  return two ? launch_two_maps<CAP>(a, st) : launch_one_map<false, CAP>(a, st);
}

}  // namespace

extern "C" int zp_gather_rows(const void* src, const int32_t* rows, void* out, int32_t n,
                              int32_t row_bytes, int64_t num_rows, void* stream) {
  ZP_REQUIRE(n >= 0 && row_bytes > 0 && row_bytes % 16 == 0 && num_rows > 0, "gather_rows: bad dims");
  if (n == 0) return ZP_OK;
  ZP_REQUIRE(src && rows && out && aligned16(src) && aligned16(out), "gather_rows: null or unaligned pointer");
  const int pieces = row_bytes / 16;
  const int64_t total = (int64_t)n * pieces;
  hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (const char*)src, rows, (char*)out, total, pieces, num_rows);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

extern "C" int zp_run_attention(const void* q, const void* k, const void* v, const void* k_shared, void* out,
                                const int32_t* tiles, const float* sinks, const zp_attention_form* form, int32_t T,
                                int32_t H, int32_t HK, int32_t D, int32_t P, int32_t V, int32_t window,
                                int32_t chunk, int64_t q_rows, int64_t k_rows, int64_t q_stride,
                                int64_t kv_stride, int64_t shared_stride, int64_t out_stride, float scale,
                                float out_scale, int32_t dtype, void* stream) {
  const zp_attention_form plain = {0.f, 1, 0.f, 0.f, 0, nullptr, 0, nullptr, nullptr, 0, 0}, f = form ? *form : plain;
  const bool two = f.maps == 2;
  ZP_REQUIRE(T >= 0 && H > 0 && HK > 0 && H % HK == 0 && D > 0 && P >= 0 && V > 0 && window >= 0 && chunk >= 0 &&
                 !(window && chunk) && (f.maps == 1 || two) && f.softcap >= 0.f && (P > 0) == (k_shared != nullptr),
             "run_attention: bad dims");
  if (dtype != ZP_BF16 || D % 8 != 0 || P % 8 != 0 || D + P > (two ? 128 : 256) || V % 8 != 0 || V > 256) {
    zp_set_error("run_attention: bfloat16, D %d + %d (multiples of 8, <= 256, of two maps <= 128), V %d (multiple of 8, <= 256)",
                 D, P, V);
    return ZP_EUNSUPPORTED;
  }
  if (T == 0) return ZP_OK;
  ZP_REQUIRE(q && k && v && out && tiles, "run_attention: null pointer");
  ZP_REQUIRE(!P || f.softcap == 0.f, "run_attention: shared keys go without a soft cap");
  ZP_REQUIRE(!f.turns || (!P && f.softcap == 0.f && aligned16(f.turns)), "run_attention: turns go without shared keys and soft cap");
  ZP_REQUIRE(!f.q_turns || (!two && !P && f.softcap == 0.f && (f.q_half == 32 || f.q_half == 64) && 2 * f.q_half <= D && D <= 128 && V <= 128 && f.q_plane >= q_rows &&
                            aligned16(f.q_turns)),
             "run_attention: queries turn by 32 or 64 pairs, with one map of at most 128, without shared keys and soft cap");
  ZP_REQUIRE(!two || (!sinks && !P && !f.turns && f.vdim > 0 && f.vdim <= V && (!f.gate || f.gate_stride >= (int64_t)H * V)),
             "run_attention: two maps go without sinks, shared keys and turns, with a mean over the values");
  ZP_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out) && aligned16(k_shared) && aligned16(f.gate) &&
                 f.gate_stride % 8 == 0 && q_stride % 8 == 0 && kv_stride % 8 == 0 && shared_stride % 8 == 0 &&
                 out_stride % 8 == 0 && q_stride >= (int64_t)H * f.maps * (D + P) && out_stride >= (int64_t)H * V &&
                 (!P || shared_stride >= P) && (int64_t)T * H < (1ll << 31) &&
                 kv_stride < (1ll << 26) && shared_stride < (1ll << 26),
             "run_attention: unaligned rows or too many tiles");
  TilesArgs a = {(const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (const uint16_t*)k_shared, (uint16_t*)out,
                 tiles, sinks, T, H, HK, D, P, V, window, chunk, q_rows, k_rows, q_stride, kv_stride, kv_stride, shared_stride,
                 out_stride, scale, out_scale, f.softcap, f.balance, f.eps, f.vdim, (const uint16_t*)f.gate, f.gate_stride,
                 (const float2*)f.turns, (const zp_f32x4*)f.q_turns, f.q_plane, f.q_half, true};
  hipStream_t st = (hipStream_t)stream;
  if (P) return launch_one_map<true, kNoCap>(a, st);
  if (!(f.softcap > 0.f)) return launch_forms<kNoCap>(a, two, st);
  return soft_cap_bounded(f.softcap) ? launch_forms<kBoundedCap>(a, two, st) : launch_forms<kCap>(a, two, st);
}

// 8 prompts of 2048 tokens, 32 heads of 128 with 8 of keys and values: 448 us (torch's scaled_dot_product_attention, causal,
// 747); a prompt of 64 tokens 13 (25); prompts of different lengths, which that takes one by one with masks, in one launch.
extern "C" int zp_causal_attention(const void* q, const void* k, const void* v, void* out, const int32_t* tiles, int32_t T,
                                   int32_t H, int32_t HK, int32_t D, int64_t q_rows, int64_t k_rows, int64_t q_stride,
                                   int64_t k_stride, int64_t v_stride, int64_t out_stride, float scale, int32_t dtype,
                                   void* stream) {
  ZP_REQUIRE(T >= 0 && H > 0 && HK > 0 && H % HK == 0 && D > 0, "causal_attention: bad dims");
  if (dtype != ZP_BF16 || D % 8 != 0 || D > 128) {
    zp_set_error("causal_attention: bfloat16, D %d (multiple of 8, <= 128)", D);
    return ZP_EUNSUPPORTED;
  }
  if (T == 0) return ZP_OK;
  ZP_REQUIRE(q && k && v && out && tiles, "causal_attention: null pointer");
  ZP_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out) && q_stride % 8 == 0 && k_stride % 8 == 0 &&
                 v_stride % 8 == 0 && out_stride % 8 == 0 && q_stride >= (int64_t)H * D && out_stride >= (int64_t)H * D &&
                 k_stride >= (int64_t)HK * D && v_stride >= (int64_t)HK * D && (int64_t)T * H < (1ll << 31) &&
                 k_stride < (1ll << 26) && v_stride < (1ll << 26),
             "causal_attention: unaligned rows or too many tiles");
  TilesArgs a = {(const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, nullptr, (uint16_t*)out, tiles, nullptr, T, H, HK,
                 D, 0, D, 0, 0, q_rows, k_rows, q_stride, k_stride, v_stride, 0, out_stride, scale, 1.f, 0.f, 0.f, 0.f, D,
                 nullptr, 0, nullptr, nullptr, 0, 0, false};
  if (flow_takes(a)) return launch_flow<true, false>(a, (hipStream_t)stream);
  return launch_run_tiles<4, 1, 2, 1, false, kNoCap, true>(a, (hipStream_t)stream);
}
