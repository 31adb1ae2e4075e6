// The recurrent mixers over long runs of tokens: 16 tokens at a time on the bf16 matrix cores, fp32 operands in three
// planes, the state of a head in registers.
//
// A wave owns 16 * NC columns of the state.  S lies in the result layout of the 16x16 products (lane (g, l16) holds rows 16 kt
// + 4 g + r of column l16 in element r), which is also the layout of a right operand if the contraction is numbered
// accordingly: of 32, lane group g has rows 4 g .. 4 g + 3 of one tile and those of the next.  So S, and the rows u derived
// from it, enter the next product from the registers they were computed in; left operands give a lane the same elements
// of its row.
#pragma once
#include "scan.h"
#include "mfma.h"

namespace {

constexpr int kBlock = 16;

template <int KT, int NC> __device__ __forceinline__ void load_state(f32x4 (&S)[KT][NC], const float* state, int dv, int col0, bool fresh) {
  const int l16 = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int nc = 0; nc < NC; ++nc)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[kt][nc][r] = fresh ? 0.f : state[(int64_t)(16 * kt + 4 * g + r) * dv + col0 + nc * 16 + l16];
}
template <int KT, int NC> __device__ __forceinline__ void store_state(const f32x4 (&S)[KT][NC], float* state, int dv, int col0) {
  const int l16 = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int nc = 0; nc < NC; ++nc)
#pragma unroll
      for (int r = 0; r < 4; ++r) state[(int64_t)(16 * kt + 4 * g + r) * dv + col0 + nc * 16 + l16] = S[kt][nc][r];
}

// An fp32 operand in three bf16 planes: each is what those before it leave, rounded to eight bits and a sign.  Together they
// are its 24 bits: the second is at most 2^-8 of x, the third 2^-17.  Six products (the first plane with all, the second
// with the first two, the third with the first) miss up to 2^-24 of the product of two operands' leading bits, as much as
// an fp32 product is rounded by; eight (all but the third with the third) up to 2^-34.
struct Planes {
  uint2 hi, mid, lo;
  __device__ __forceinline__ Planes(const f32x4& x) {
    f32x4 r = x;
    hi = rounded(r);
    r = rest(r, hi);
    mid = rounded(r);
    lo = rounded(rest(r, mid));
  }
  __device__ static __forceinline__ uint2 rounded(const f32x4& x) { return uint2{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])}; }
  // x minus its rounded values, exactly: the dot product of a pair of them with (-1, 0) or (0, -1) is added to x, which saves
  // taking the pair apart.  The factors are kept from the compiler, which would make an immediate of -1 that stands for
  // another pair.
  __device__ static __forceinline__ f32x4 rest(const f32x4& x, const uint2& p) {
    uint32_t first = 0x0000bf80u, second = 0xbf800000u;
#ifdef __HIP_DEVICE_COMPILE__
    asm("" : "+s"(first));
    asm("" : "+s"(second));
#endif
    return f32x4{plus_dot(p.x, first, x[0]), plus_dot(p.x, second, x[1]), plus_dot(p.y, first, x[2]), plus_dot(p.y, second, x[3])};
  }
  __device__ static __forceinline__ float plus_dot(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(zp_bf16x2, a), __builtin_bit_cast(zp_bf16x2, b), c, false);
  }
};
// A right operand of 16 of the contraction for left ones that lie as [64 lanes][hi 4, mid 4], [64][lo 4]: the bf16 matrix
// cores take 32, so planes go in pairs, eight products in four.
constexpr int kPairFloats = 384;               // of such a left operand
struct PlanePairs {
  u32x4 hh, mm, ll, hm;
  __device__ __forceinline__ PlanePairs(const f32x4& x) {
    const Planes p(x);
    hh = u32x4{p.hi.x, p.hi.y, p.hi.x, p.hi.y};
    mm = u32x4{p.mid.x, p.mid.y, p.mid.x, p.mid.y};
    ll = u32x4{p.lo.x, p.lo.y, p.lo.x, p.lo.y};
    hm = u32x4{p.hi.x, p.hi.y, p.mid.x, p.mid.y};
  }
  __device__ __forceinline__ PlanePairs(const u32x4 (&p)[4]) : hh(p[0]), mm(p[1]), ll(p[2]), hm(p[3]) {}
  __device__ __forceinline__ void add(const u32x4& left, const uint2& lo, f32x4& c) const {
    c = mfma_bf16(left, ll, c);
    c = mfma_bf16(u32x4{lo.x, lo.y, lo.x, lo.y}, hm, c);
    c = mfma_bf16(left, mm, c);
    c = mfma_bf16(left, hh, c);
  }
  // two at a time: each waits for the one before
  __device__ __forceinline__ void add(const u32x4 (&left)[2], const uint2 (&lo)[2], f32x4& c, f32x4& d) const {
    c = mfma_bf16(left[0], ll, c);
    d = mfma_bf16(left[1], ll, d);
    c = mfma_bf16(u32x4{lo[0].x, lo[0].y, lo[0].x, lo[0].y}, hm, c);
    d = mfma_bf16(u32x4{lo[1].x, lo[1].y, lo[1].x, lo[1].y}, hm, d);
    c = mfma_bf16(left[0], mm, c);
    d = mfma_bf16(left[1], mm, d);
    c = mfma_bf16(left[0], hh, c);
    d = mfma_bf16(left[1], hh, d);
  }
};
// x is computed before what follows, whoever uses it.
__device__ __forceinline__ void settle(u32x4& x) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+v"(x));
#endif
}
// A stretch with N products ends here: what else it holds is spread over them.
template <int N, int PER> __device__ __forceinline__ void spread_over_products() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // a product
    __builtin_amdgcn_sched_group_barrier(0x002, PER, 0);    // vector instructions
  }
  __builtin_amdgcn_sched_barrier(0);
}

// Sum of squares of each of the block's 16 tokens over the wave's columns; lane l16 == 0 of group g leaves
// tokens 4 g .. 4 g + 3 in `red` (16 floats per wave).
template <int NC> __device__ __forceinline__ void block_squares(const f32x4 (&o)[NC], float* red, int wave) {
  const int l16 = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  f32x4 ss = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int nc = 0; nc < NC; ++nc) ss += o[nc] * o[nc];
#pragma unroll
  for (int r = 0; r < 4; ++r) ss[r] = row16_sum(ss[r]);
  if (l16 == 0) *(f32x4*)(red + wave * kBlock + 4 * g) = ss;
}
// Each lane of a group of sixteen reads one wave's share.
template <int NW> __device__ __forceinline__ f32x4 block_squares_total(const float* red) {
  const int l16 = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  f32x4 ss = *(const f32x4*)(red + min(l16, NW - 1) * kBlock + 4 * g);
#pragma unroll
  for (int r = 0; r < 4; ++r) ss[r] = row16_sum(l16 < NW ? ss[r] : 0.f);
  return ss;
}

// Forms for 16-bit models on the hardware's exponential, logarithm, reciprocal and reciprocal square root,
// each within a unit or two of the last of 24 bits.
__device__ __forceinline__ float fast_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
__device__ __forceinline__ float fast_softplus(float x) {
  const float y = __expf(-fabsf(x));
  // log(1 + y) as it stands loses a small y's digits
  const float l = y < 0.03125f ? y * (1.f - y * (0.5f - y * (1.f / 3.f - y * 0.25f))) : __logf(1.f + y);
  return fmaxf(x, 0.f) + l;
}

// Element (row 4 g + r, column col) of 16 token rows of bf16, for r = 0 .. 3; rows behind the last read as zero
// and are not written.
struct BlockRows {
  __amdgpu_buffer_rsrc_t rs;
  __device__ __forceinline__ BlockRows(const void* base, int64_t row, int cnt, int64_t stride)
      : rs(__builtin_amdgcn_make_buffer_rsrc((void*)((char*)base + row * stride * 2), 0, (int)(cnt * stride * 2), 0x00020000)) {}
  // as it is in memory: converting it is left to its use, so that nothing waits for the load before
  __device__ __forceinline__ uint16_t ld(int offset, int col) const {
    return __builtin_amdgcn_raw_buffer_load_b16(rs, offset, col * 2, 0);
  }
  __device__ __forceinline__ void st(int offset, int col, float v) const {
    __builtin_amdgcn_raw_buffer_store_b16(float_to_bf16_bits(v), rs, offset, col * 2, 0);
  }
};

// Columns of a 4 x 16 block of 16-bit values in LDS: lane i of a group of sixteen names row i / 4, values 4 (i % 4)
// on, and receives column i.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 read_columns(const char* p) {
  const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  return f32x4{bf16_bits_to_float((uint16_t)v[0]), bf16_bits_to_float((uint16_t)v[1]), bf16_bits_to_float((uint16_t)v[2]),
               bf16_bits_to_float((uint16_t)v[3])};
}

// Loads straight into LDS; wait_and_meet() waits for them.
struct StageLoads {
  u32x4 rs;
  __device__ __forceinline__ StageLoads(const void* base, int64_t bytes) : rs(rows_from(base, (uint32_t)bytes)) {}
  __device__ __forceinline__ void ld(void* lds, int offset, int uniform) const { load_to_lds(rs, lds, offset, uniform); }
};
__device__ __forceinline__ void wait_and_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0);               // as a builtin: the compiler then knows that nothing is outstanding
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Blocks of segment i start at slot (row - row0) / 16 + i: enough room, whatever the counts are.
__device__ __forceinline__ int64_t block_slot(int row0, const Segment& sg, int seg, int b) {
  return (sg.row - row0) / kBlock + seg + b;
}

// ------------------------------------------------------------------ runs in pieces
// A head walks its blocks one after the other, 2.4 us each, and a few heads leave most CUs idle.  The state behind a piece of a
// run is (what the piece keeps) * (the state before it) + what the piece adds to none, so few heads walk their runs in pieces
// side by side:
//
//   sums     what each piece but the last adds and keeps: nothing waits for a state
//   states   the states between pieces, from the first to the last
//   blocks   as without pieces, each from its state on
//
// Workgroups fill a CU, so pieces are as short as 256 of them (and kLeastPiece blocks) and the chain of states between them
// allow.  Where the sums and the two launches cost more than what is saved, runs stay whole (PieceCost): a block of the sums takes
// 0.3 of one with rows (0.8 for the delta rule), the launches 19 us (17 for the delta rule), states of the delta rule 4.3 us a piece,
// reckoned as 5.7 (matrix memory, 8 heads, a prompt of 155 tokens: whole 41.8 us, in pieces 42.8; linear attention, 32 heads, 200
// tokens: 53, 46).  Whole scans, before pieces and now: linear attention, 32 heads of 128, 4 prompts of 500 to 2048 tokens 374 and 287 us; 16
// heads, 8 prompts of 2048, retention 429 and 332, matrix memory 369 and 285; retention, a prompt of 700 126 and 45; delta rule, 32 heads, a
// prompt of 2048 477 and 217, two of about 1250 384 and 238.
constexpr int kPieceGroups = 256, kPieceStates = 384, kLeastPiece = 4;
struct Pieces {
  int blocks = 0, most = 1;      // of a piece, 0: runs are whole; pieces of the longest run at most
  float* states = nullptr;
};
inline bool few_heads(int64_t segments, int64_t heads) { return segments * heads * 2 <= kPieceGroups; }
// The sums take `groups` workgroups per piece and, in tenths of a block, `sum` per block; the rest `fixed` and `state` per piece.
struct PieceCost { int groups, sum, fixed, state; };
inline int64_t piece_slots(int64_t rows, int64_t segments, int64_t blocks) { return rows / (kBlock * blocks) + segments; }
// States that runs in so many rows can ask for, whatever the longest: none where the longest that fits stays whole.
inline int64_t most_states(int64_t rows, int64_t segments, int64_t heads, const PieceCost& cost) {
  if (!few_heads(segments, heads) || (rows + kBlock - 1) / kBlock * 10 <= kLeastPiece * (10 + cost.sum) + cost.fixed) return 0;
  const int64_t states = piece_slots(rows, segments, kLeastPiece) * heads;
  return states < kPieceStates ? states : kPieceStates;
}
// Runs stay whole, too, where `room` states are not enough.  `step`: blocks that are walked together.
inline Pieces pieces_of(int64_t rows, int64_t segments, int64_t heads, int64_t longest, const PieceCost& cost, int step, int64_t room) {
  Pieces p;
  const int64_t all = (longest + kBlock - 1) / kBlock;
  if (!few_heads(segments, heads)) return p;
  int64_t best = all * 10;
  for (int64_t m = kLeastPiece; m < all && m * (10 + cost.sum) + cost.fixed < best; m += step) {      // longer ones only take longer
    const int64_t most = (all + m - 1) / m, slots = piece_slots(rows, segments, m), pieces = segments * most < slots ? segments * most : slots;
    const int64_t took = m * (10 + cost.sum) + cost.fixed + most * cost.state;
    if (pieces * heads > kPieceGroups || (pieces - segments) * heads * cost.groups > kPieceGroups || slots * heads > kPieceStates ||
        slots * heads > room || took >= best) continue;
    best = took;
    p.blocks = (int)m, p.most = (int)most;
  }
  return p;
}
// Piece c of a run: the segment that it is, whether it is the last; of segments that have fewer none is left.  Its place among
// the states, a run's pieces one after the other: enough room, as with the blocks.
struct Piece {
  Segment sg;
  bool last;
  int64_t slot;
  __device__ __forceinline__ Piece(const Pieces& p, int row0, const Segment& whole, int seg, int c) : sg(whole), last(true), slot(0) {
    if (p.blocks == 0) return;
    const int tokens = p.blocks * kBlock, from = c * tokens;
    sg.row += from;
    sg.count = min(whole.count - from, tokens);
    last = from + tokens >= whole.count;
    slot = (whole.row - row0) / tokens + seg + c;
  }
};
// States between pieces lie as the waves that own 16 columns hold them: [columns / 16][rows / 16][64 lanes][4].
template <int KT> __device__ __forceinline__ void load_piece_state(f32x4 (&S)[KT][1], const float* state, int wave) {
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) S[kt][0] = *(const f32x4*)(state + ((wave * KT + kt) * 64 + (threadIdx.x & 63)) * 4);
}

}  // namespace
