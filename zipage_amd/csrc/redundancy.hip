// Key-redundancy scores: cosine-similarity Gram matrix of cached keys, per page
// ("lightning") or over the whole sequence ("raw"), with the reference's claim rule:
// the diagonal is zeroed and, for every column, the LAST row whose similarity exceeds the
// threshold is zeroed too; the row sums are the redundancy logits.
//
// The Gram matrix is symmetric, so "last row over the threshold in column j" equals "last
// column over the threshold in row j" (the key's claim); the claimed entries are subtracted
// afterwards from the rows they were taken from:
//     r_i = sum_j S_ij  -  sum_{j : c*(j) = i} S_ji .
//
// Kernels in this file:
//   gram_kernel        fp32 caches, both variants, any page size and table length:
//                      v_mfma_f32_32x32x2_f32 on keys divided by their norm in fp32, full matrix,
//                      a wave owns 32 rows for all columns.
//   gram_page_f32_kernel  fp32 caches, lightning, pages of at most 256 keys: a workgroup walks its share of
//                      the pages of a row; the normalised page resident in LDS as two fp16 planes per
//                      element (fp32-grade products on the 16-bit matrix instructions), one
//                      barrier, both operands read from that copy, every pair of key blocks once.
//   gram_raw_sym_f32_kernel  fp32 caches, raw, pages of at most 256 keys and tables of at most 16
//                      pages: every unordered pair of pages once, column tiles staged as the same
//                      two planes.
//   gram_split_kernel  16-bit caches, lightning with pages above 256 keys: normalised keys
//                      split into two bf16 planes, three MFMAs per k-step, full matrix.
//   gram_page_kernel   16-bit caches, lightning: a workgroup walks the pages of one (layer,
//                      sequence, kv head) row; stored keys loaded straight into LDS and put on
//                      the matrix cores, 1/norm factors on the accumulators, every pair of key
//                      blocks once, the summed key as a product over the keys, the next page
//                      requested while a page's row sums are finished.
//   raw_prep_kernel, gram_raw_wide_kernel / gram_raw_kernel, raw_claim_value_kernel, raw_chain_kernel
//                      16-bit caches, raw: the same over the pages of a sequence, the row sums
//                      accumulated in the cache dtype chunk by chunk as the reference does.
//   red_softmax_kernel claim corrections of the raw variant and the softmax of both.
#include "common.h"
#include <type_traits>
#include <math.h>

namespace {

// Sum over the PIECES (16 or 32) consecutive lanes that hold one key row.
template <int PIECES> __device__ __forceinline__ float pieces_sum(float v) {
  static_assert(PIECES == 16 || PIECES == 32, "a key row spans 16 or 32 lanes");
  v = row16_sum(v);
  if (PIECES == 32) v += lane_xor16(v);
  return v;
}
// The valid pages of one block-table row in table order, listed in LDS by the first wave of the
// workgroup (64 entries per step: one load per lane, a ballot ranks the valid ones), instead of a
// serial walk by one thread with a global load per entry.  vpage[n] / vidx[n]: page id / table
// index of the n-th valid page; vord[j]: rank of table entry j or -1; *n_out: their number; *me_out:
// the rank of entry `jp` (0 when it is not valid).  Null pointers are skipped; the caller meets at
// a barrier before reading.
__device__ __forceinline__ void list_valid_pages(const int32_t* __restrict__ row, int NB, int num_pages,
                                                 int jp, int* vpage, int* vidx, int* vord, int* n_out,
                                                 int* me_out) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  int n = 0;
  if (lane == 0 && me_out) *me_out = 0;
  for (int j0 = 0; j0 < NB; j0 += 64) {
    const int j = j0 + lane;
    const int c = j < NB ? row[j] : -1;
    const int pid = page_is_pad(c) ? -1 : page_id(c);
    const bool ok = pid >= 0 && pid < num_pages;
    const unsigned long long m = __builtin_amdgcn_ballot_w64(ok);
    const int pos = n + __builtin_popcountll(m & lanemask_lt());
    if (ok) {
      if (vpage) vpage[pos] = pid;
      if (vidx) vidx[pos] = j;
      if (me_out && j == jp) *me_out = pos;
    }
    if (vord && j < NB) vord[j] = ok ? pos : -1;
    n += __builtin_popcountll(m);
  }
  if (lane == 0) *n_out = n;
}

// Over the 32 lanes of a wave half: the entry with the largest column index (and its value).
__device__ __forceinline__ void last_claim_reduce(int& c, float& v) {
#define ZP_CLAIM_STEP(OC, OV)              \
  do {                                     \
    const int oc_ = (OC);                  \
    const float ov_ = (OV);                \
    if (oc_ > c) { c = oc_; v = ov_; }     \
  } while (0)
  ZP_CLAIM_STEP(dpp_row_ror<8>(c), dpp_row_ror<8>(v));
  ZP_CLAIM_STEP(dpp_row_ror<4>(c), dpp_row_ror<4>(v));
  ZP_CLAIM_STEP(dpp_row_ror<2>(c), dpp_row_ror<2>(v));
  ZP_CLAIM_STEP(dpp_row_ror<1>(c), dpp_row_ror<1>(v));
  ZP_CLAIM_STEP(lane_xor16(c), lane_xor16(v));
#undef ZP_CLAIM_STEP
}

// Reductions of sixteen values each over the 32 lanes of a wave half.  Every step takes the other half of the lanes' share of two values
// and leaves each lane one of them, so the sixteen take fifteen such steps instead of eighty, and one store instead of sixteen.
// What is left in x[0] of lane i, and of i + 16, is value r (returned).  Lanes 8, 4, 2, 1 and 16 apart are joined, in this order, as
// row16_sum and half_sum do.
template <int APART, typename V> __device__ __forceinline__ V lane_xor_row(V v) {
  const int x = __builtin_bit_cast(int, v);
  int o;
  if constexpr (APART == 8) o = __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false);        // row_ror:8
  else if constexpr (APART == 4)                                                                  // half_mirror of quad_perm [3,2,1,0]
    o = __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, x, 0x1B, 0xf, 0xf, false), 0x141, 0xf, 0xf, false);
  else if constexpr (APART == 2) o = __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, false);    // quad_perm [2,3,0,1]
  else o = __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, false);                              // quad_perm [1,0,3,2]
  return __builtin_bit_cast(V, o);
}
template <int APART, int N, typename V, typename Join> __device__ __forceinline__ void halve_values(V* x, int lane, Join join) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const V lo = join(x[2 * i], lane_xor_row<APART>(x[2 * i])), hi = join(x[2 * i + 1], lane_xor_row<APART>(x[2 * i + 1]));
    x[i] = lane & APART ? hi : lo;
  }
}
template <typename V, typename Join> __device__ __forceinline__ int sixteen_half_reduce(V (&x)[16], int lane, Join join) {
  halve_values<8, 8>(x, lane, join);
  halve_values<4, 4>(x, lane, join);
  halve_values<2, 2>(x, lane, join);
  halve_values<1, 1>(x, lane, join);
  x[0] = join(x[0], lane_xor16(x[0]));
  return (lane & 1 ? 8 : 0) | (lane & 2 ? 4 : 0) | (lane & 4 ? 2 : 0) | (lane & 8 ? 1 : 0);
}
__device__ __forceinline__ int sixteen_half_max(int (&x)[16], int lane) {
  return sixteen_half_reduce(x, lane, [](int a, int b) { return max(a, b); });
}
__device__ __forceinline__ int sixteen_half_sum(float (&x)[16], int lane) {
  return sixteen_half_reduce(x, lane, [](float a, float b) { return a + b; });
}
// The entries with the largest column index, and their values.
template <int APART, int N> __device__ __forceinline__ void halve_claims(int* c, float* v, int lane) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    int cc[2];
    float vv[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int oc = lane_xor_row<APART>(c[2 * i + k]);
      const float ov = lane_xor_row<APART>(v[2 * i + k]);
      cc[k] = max(c[2 * i + k], oc);
      vv[k] = oc > c[2 * i + k] ? ov : v[2 * i + k];
    }
    c[i] = lane & APART ? cc[1] : cc[0];
    v[i] = lane & APART ? vv[1] : vv[0];
  }
}
__device__ __forceinline__ void sixteen_last_claims(int (&c)[16], float (&v)[16], int lane) {
  halve_claims<8, 8>(c, v, lane);
  halve_claims<4, 4>(c, v, lane);
  halve_claims<2, 2>(c, v, lane);
  halve_claims<1, 1>(c, v, lane);
  const int oc = lane_xor16(c[0]);
  const float ov = lane_xor16(v[0]);
  if (oc > c[0]) { c[0] = oc; v[0] = ov; }
}

// A similarity as 2^-32 fixed point (two's complement in an unsigned 64-bit word) and back: sums of
// such words are exact and independent of the order of the additions.
__device__ __forceinline__ unsigned long long to_fixed32(float v) {
  return (unsigned long long)(long long)(v * 4294967296.f);
}
__device__ __forceinline__ float from_fixed32(unsigned long long w) {
  return (float)(long long)w * (1.f / 4294967296.f);
}

constexpr int kThreads = 256;
constexpr int kWaves = 4;
constexpr int kDmax = 128;
constexpr int TN = 64;                  // keys per column tile
constexpr int ROWF = kDmax + 4;         // floats per LDS row: 16-byte aligned rows whose 16-byte reads by
                                        // eight consecutive rows fall into eight different bank groups
constexpr int KS = kDmax / 2;           // MFMA k-steps (2 per instruction)
constexpr int kChunk = 16;              // columns the reference's all-pairs kernel takes per step
                                        // (BLOCK_N, raw_redudancy_score.py:176)

typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Unpack;
template <> struct Unpack<F32> {
  static constexpr int N = 4;
  __device__ static __forceinline__ void run(const vec16& v, float* o) {
    o[0] = __uint_as_float(v.x); o[1] = __uint_as_float(v.y);
    o[2] = __uint_as_float(v.z); o[3] = __uint_as_float(v.w);
  }
};
template <> struct Unpack<BF16> {
  static constexpr int N = 8;
  __device__ static __forceinline__ void run(const vec16& v, float* o) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = __uint_as_float(w[i] << 16);
      o[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};
template <> struct Unpack<F16> {
  static constexpr int N = 8;
  __device__ static __forceinline__ void run(const vec16& v, float* o) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = f16_bits_to_float((uint16_t)(w[i] & 0xffffu));
      o[2 * i + 1] = f16_bits_to_float((uint16_t)(w[i] >> 16));
    }
  }
};

struct GramArgs {
  const char* k;
  const int32_t* table;
  void* r_out;     // lightning: (rows, NB*BS) row sums in the cache dtype
  float* ws_sum;   // raw: fp32 plain row sums
  int32_t* ws_col; // raw: last column over the threshold (logical index, -1 none)
  float* ws_val;   // raw: its value
  float* ws_chunk; // raw, 16-bit caches: [row][T / 16][kDmax] sums of the normalised keys per chunk
  int B, NB, BS, Hkv, D, num_pages;
  int64_t k_sl, k_sp;
  float threshold, eps;
  int parts;       // the page kernels: workgroups per row; each walks every parts-th entry of its block table.  All pairs, 16 bit: per page
};

template <typename T, bool RAW, int NW>
__global__ __launch_bounds__(NW * 64) void gram_kernel(GramArgs p) {
  constexpr int kThreads = NW * 64, kWaves = NW;    // shadow the file-wide 4-wave constants
  constexpr int NE = Unpack<T>::N;                  // elements per 16-byte piece
  constexpr int PIECES = kDmax / NE;                // pieces per full key row
  constexpr int ROWS_PER_IT = kThreads / PIECES;
  constexpr int STAGE_IT = TN / ROWS_PER_IT;
  constexpr int NSUB = TN / 32;

  extern __shared__ __align__(16) char smem[];
  float* kbuf0 = (float*)smem;
  float* kbuf1 = kbuf0 + TN * ROWF;
  unsigned long long* l_corr = (unsigned long long*)(kbuf1 + TN * ROWF);   // lightning: [BS] claimed from a row
  float* l_sum = (float*)(l_corr + (RAW ? 0 : p.BS));                     //            [BS] row sums
  float* l_val = l_sum + (RAW ? 0 : p.BS);          //            [BS] claimed values
  int* l_col = (int*)(l_val + (RAW ? 0 : p.BS));    //            [BS] claimed columns
  int* vpage = l_col + (RAW ? 0 : p.BS);            // [NB] valid page ids (raw)
  int* vidx = vpage + p.NB;                         // [NB] their table index

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int jp = blockIdx.x % p.NB;                 // row page (table index)
  const int h = (blockIdx.x / p.NB) % p.Hkv;
  const int b = (blockIdx.x / (p.NB * p.Hkv)) % p.B;
  const int l = blockIdx.x / (p.NB * p.Hkv * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t orow = (((int64_t)l * p.B + b) * p.Hkv + h);
  const float epsr = Elem<T>::rnd(p.eps);

  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) {  // pad page: logits -inf (lightning); raw marks it in the epilogue
    if (!RAW)
      for (int s = tid; s < p.BS; s += kThreads)
        Elem<T>::st(p.r_out, orow * Tn + (int64_t)jp * p.BS + s, -INFINITY);
    return;
  }

  __shared__ int ncols_s;
  if (RAW) {
    list_valid_pages(p.table + (int64_t)b * p.NB, p.NB, p.num_pages, jp, vpage, vidx, nullptr, &ncols_s, nullptr);
  } else if (tid == 0) {
    vpage[0] = rpid; vidx[0] = jp; ncols_s = 1;
  }
  for (int i = tid; i < 2 * TN * ROWF; i += kThreads) kbuf0[i] = 0.f;
  __syncthreads();
  const int tiles_per_page = p.BS / TN;
  const int ntiles = ncols_s * tiles_per_page;
  const int dpieces = p.D / NE;
  const int64_t k_row = (int64_t)p.Hkv * p.D * T::bytes;
  const char* kbase = p.k + (l * p.k_sl) * T::bytes + (int64_t)h * p.D * T::bytes;

  const int st_piece = tid % PIECES, st_row0 = tid / PIECES;
  vec16 pre[STAGE_IT];
  auto issue_loads = [&](int tile) {
    const int vp = tile / tiles_per_page, toff = (tile - vp * tiles_per_page) * TN;
    const char* src = kbase + (int64_t)vpage[vp] * p.k_sp * T::bytes + (int64_t)toff * k_row;
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i) {
      const int row = st_row0 + i * ROWS_PER_IT;
      pre[i] = vec16{0u, 0u, 0u, 0u};
      if (st_piece < dpieces) pre[i] = *(const vec16*)(src + (int64_t)row * k_row + st_piece * 16);
    }
  };
  // normalise (k / max(rnd(|k|), rnd(eps)) in fp32) on the way into LDS
  auto commit_loads = [&](float* buf) {
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i) {
      const int row = st_row0 + i * ROWS_PER_IT;
      float e[NE];
      Unpack<T>::run(pre[i], e);
      float ss = 0.f;
#pragma unroll
      for (int q = 0; q < NE; ++q) ss += e[q] * e[q];
      ss = pieces_sum<PIECES>(ss);
      // one reciprocal per key and a multiplication per element (the hardware square root and
      // reciprocal are each within 1 ulp; a division per element would dominate the staging)
      const float rn = __builtin_amdgcn_rcpf(fmaxf(Elem<T>::rnd(__builtin_amdgcn_sqrtf(ss)), epsr));
      if (st_piece < dpieces) {
        float* d = buf + row * ROWF + st_piece * NE;
#pragma unroll
        for (int q = 0; q < NE; q += 2) *(float2*)(d + q) = make_float2(e[q] * rn, e[q + 1] * rn);
      }
    }
  };

  const int row_blocks = p.BS / 32;
  const int NR = (row_blocks + kWaves - 1) / kWaves;
  for (int rr = 0; rr < NR; ++rr) {
    const int rb = rr * kWaves + wave;
    const bool active = rb < row_blocks;
    // ---- A fragments: this lane's key row, normalised.  The order of the contraction index is
    // free as long as both operands agree: k-step 4j + i of wave half `half` takes element
    // 8j + 4 half + i, so a lane's B operands for four steps are one 16-byte LDS read.
    float afrag[KS];
    {
      const int slot = (active ? rb : 0) * 32 + col;
      const char* src = kbase + (int64_t)rpid * p.k_sp * T::bytes + (int64_t)slot * k_row;
      float ss = 0.f;
#pragma unroll
      for (int pc = 0; pc < PIECES; ++pc) {
        float e[NE];
        vec16 v = vec16{0u, 0u, 0u, 0u};
        if (pc < dpieces) v = *(const vec16*)(src + pc * 16);
        Unpack<T>::run(v, e);
#pragma unroll
        for (int q = 0; q < NE; ++q) ss += e[q] * e[q];
        if constexpr (NE == 4) {
          // piece pc holds elements 4 pc .. 4 pc + 3 = (j, half) = (pc / 2, pc % 2)
          if ((pc & 1) == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) afrag[(pc >> 1) * 4 + q] = e[q];
          } else if (half) {
#pragma unroll
            for (int q = 0; q < 4; ++q) afrag[(pc >> 1) * 4 + q] = e[q];
          }
        } else {
#pragma unroll
          for (int q = 0; q < NE / 2; ++q) afrag[pc * (NE / 2) + q] = half ? e[2 * q + 1] : e[2 * q];
        }
      }
      const float rn = __builtin_amdgcn_rcpf(fmaxf(Elem<T>::rnd(__builtin_amdgcn_sqrtf(ss)), epsr));
#pragma unroll
      for (int s = 0; s < KS; ++s) afrag[s] = active ? afrag[s] * rn : 0.f;
    }
    float rsum[16], cval[16];
    int ccol[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) { rsum[r] = 0.f; cval[r] = 0.f; ccol[r] = -1; }

    if (ntiles > 0) { issue_loads(0); commit_loads(kbuf0); }
    __syncthreads();
    for (int tile = 0; tile < ntiles; ++tile) {
      float* cur = (tile & 1) ? kbuf1 : kbuf0;
      float* nxt = (tile & 1) ? kbuf0 : kbuf1;
      if (tile + 1 < ntiles) issue_loads(tile + 1);
      const int vp = tile / tiles_per_page, toff = (tile - vp * tiles_per_page) * TN;
      const int jc = vidx[vp];
      if (active) {
#pragma unroll
        for (int st = 0; st < NSUB; ++st) {
          f32x16_t acc;
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] = 0.f;
          if constexpr (NE == 4) {
            const float4* b4 = (const float4*)(cur + (st * 32 + col) * ROWF + 4 * half);
#pragma unroll
            for (int j4 = 0; j4 < KS / 4; ++j4) {
              const float4 bv = b4[2 * j4];
              acc = __builtin_amdgcn_mfma_f32_32x32x2f32(afrag[4 * j4 + 0], bv.x, acc, 0, 0, 0);
              acc = __builtin_amdgcn_mfma_f32_32x32x2f32(afrag[4 * j4 + 1], bv.y, acc, 0, 0, 0);
              acc = __builtin_amdgcn_mfma_f32_32x32x2f32(afrag[4 * j4 + 2], bv.z, acc, 0, 0, 0);
              acc = __builtin_amdgcn_mfma_f32_32x32x2f32(afrag[4 * j4 + 3], bv.w, acc, 0, 0, 0);
            }
          } else {
            const float* brow = cur + (st * 32 + col) * ROWF + half;
#pragma unroll
            for (int s = 0; s < KS; ++s)
              acc = __builtin_amdgcn_mfma_f32_32x32x2f32(afrag[s], brow[2 * s], acc, 0, 0, 0);
          }
          const int cslot = toff + st * 32 + col;
          const int cidx = jc * p.BS + cslot;  // logical column index of this lane
          const bool same_page = jc == jp;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
            float s = acc[r];
            if (same_page && rslot == cslot) s = 0.f;
            rsum[r] += s;
            if (s > p.threshold) { ccol[r] = cidx; cval[r] = s; }
          }
        }
      }
      if (tile + 1 < ntiles) commit_loads(nxt);
      __syncthreads();
    }
    // ---- combine over the 32 lanes of each half (they share rows)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float s = rsum[r];
      int c = ccol[r];
      float v = cval[r];
      s = half_sum(s);
      last_claim_reduce(c, v);
      if (active && col == 0) {
        const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
        if (RAW) {
          const int64_t oi = orow * Tn + (int64_t)jp * p.BS + rslot;
          p.ws_sum[oi] = s;
          p.ws_col[oi] = c;
          p.ws_val[oi] = v;
        } else {
          l_sum[rslot] = s;
          l_col[rslot] = c - jp * p.BS;  // column slot inside the page (or negative)
          l_val[rslot] = v;
        }
      }
    }
  }
  if (!RAW) {
    // every key hands the value of its claimed entry to the row it was taken from; several keys
    // may claim from one row, so the values are added as 2^-32 fixed point: exact to 2^-33 per
    // term and independent of the order (a scan of all keys per row cost ~10 % of the kernel)
    for (int i = tid; i < p.BS; i += kThreads) l_corr[i] = 0ull;
    __syncthreads();
    for (int j = tid; j < p.BS; j += kThreads) {
      const int c = l_col[j];
      if (c >= 0 && c < p.BS) atomicAdd(&l_corr[c], to_fixed32(l_val[j]));
    }
    __syncthreads();
    for (int i = tid; i < p.BS; i += kThreads)
      Elem<T>::st(p.r_out, orow * Tn + (int64_t)jp * p.BS + i, l_sum[i] - from_fixed32(l_corr[i]));
  }
}

// ------------------------------------------------------------------ fp32 products on the fp16 matrix cores
// A normalised key element x (|x| <= 1) is scaled by 2^12 and written as two fp16 numbers,
// h1 = fp16(x') and h2 = fp16(x' - h1), both rounded to nearest: x' - h1 is exact in fp32 (13
// bits), so |x' - h1 - h2| <= 2^-24 |x'|, what rounding a real number to fp32 loses; the scale
// keeps h2 out of fp16's subnormal range for every element that matters (|x| >= 2^-14) and the
// largest scaled element (4096) far below fp16's maximum.  The products h1.g1, h1.g2, h2.g1 are
// exact in the fp32 accumulator, h2.g2 (<= 2^-24 |x||y|) is left out, and the 2^24 of the two
// scales comes off the result exactly.  Three v_mfma_f32_32x32x16_f16 (8 passes each, 16 k) replace eight
// v_mfma_f32_32x32x2_f32 (16 passes each): 3/16 of the matrix-core time at fp32-grade accuracy, and the
// two planes take the LDS bytes of the fp32 element they replace.
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
constexpr float kPlaneScale = 4096.f;                 // 2^12 per operand
constexpr float kPlaneUnscale = 1.f / (4096.f * 4096.f);
constexpr int KSH = kDmax / 16;                       // k-steps of the 16-bit instructions over a key row
constexpr int kPlaneBytes = kDmax * 2;                // one plane of one LDS row; the row keeps ROWF * 4 bytes
__device__ __forceinline__ void split_planes(const float4 e, f16x4_t& h1, f16x4_t& h2) {
  const f32x2_t a = {e.x, e.y}, b = {e.z, e.w};
  const f16x2_t a1 = __builtin_convertvector(a, f16x2_t), b1 = __builtin_convertvector(b, f16x2_t);
  const f32x2_t ar = {e.x - (float)a1[0], e.y - (float)a1[1]}, br = {e.z - (float)b1[0], e.w - (float)b1[1]};
  const f16x2_t a2 = __builtin_convertvector(ar, f16x2_t), b2 = __builtin_convertvector(br, f16x2_t);
  h1 = f16x4_t{a1[0], a1[1], b1[0], b1[1]};
  h2 = f16x4_t{a2[0], a2[1], b2[0], b2[1]};
}
__device__ __forceinline__ f32x16_t mma_planes(const f16x8_t a1, const f16x8_t a2, const f16x8_t b1,
                                               const f16x8_t b2, f32x16_t acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2, b1, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b2, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, b1, acc, 0, 0, 0);
  return acc;
}
// largest of a lane's sixteen tile entries (claims are rare: one maximum per lane and a ballot
// decide whether a tile has any entry over the threshold)
__device__ __forceinline__ float tile_lane_max(const f32x16_t& acc) {
  float m[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    m[q] = __builtin_fmaxf(__builtin_fmaxf(acc[4 * q], acc[4 * q + 1]), __builtin_fmaxf(acc[4 * q + 2], acc[4 * q + 3]));
  return __builtin_fmaxf(__builtin_fmaxf(m[0], m[1]), __builtin_fmaxf(m[2], m[3]));
}

// ------------------------------------------------------------------ fp32 caches, raw, every pair of pages once
// One workgroup per (layer, sequence, head, valid page a), pages of at most 256 keys.  The
// similarity matrix of a sequence is symmetric, so page a multiplies its rows only with the pages
// (a + d) mod n, d = 0 .. n/2 (the pairs at distance n/2 go to the lower half of the pages when n
// is even).  A tile off the diagonal page serves both of its sides: the rows get their partial
// row sums and their claim (last column over the threshold) as in gram_kernel; the columns get
// the tile's column sums -- slot [d][key], written by exactly one workgroup and added in a fixed
// order by the softmax kernel -- and the last ROW over the threshold as their claim.  Claims meet
// in one 64-bit word per key, (index + 1) << 32 | value bits, through atomicMax: the largest
// index wins whatever the order of the workgroups.
constexpr int kSymWaves = 8;
constexpr int kSymMaxDist = 8;      // column-sum slots per key the workspace holds: tables of <= 16 pages

__global__ void fill_u64_kernel(unsigned long long* dst, int64_t n, unsigned long long v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = v;
}

__global__ __launch_bounds__(kSymWaves * 64) void gram_raw_sym_f32_kernel(GramArgs p) {
  typedef F32 T;
  constexpr int kThreads = kSymWaves * 64;
  constexpr int PIECES = kDmax / 4;                 // 16-byte pieces per key row
  constexpr int ROWS_PER_IT = kThreads / PIECES;    // 16
  constexpr int STAGE_IT = TN / ROWS_PER_IT;        // 4
  constexpr int NSUB = TN / 32;

  extern __shared__ __align__(16) char smem[];
  float* kbuf0 = (float*)smem;
  float* kbuf1 = kbuf0 + TN * ROWF;
  float* l_cpart = kbuf1 + TN * ROWF;               // [2][kSymWaves][TN] column sums per wave and tile
  int* vpage = (int*)(l_cpart + 2 * kSymWaves * TN);
  int* vidx = vpage + p.NB;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int jp = blockIdx.x % p.NB;
  const int h = (blockIdx.x / p.NB) % p.Hkv;
  const int b = (blockIdx.x / (p.NB * p.Hkv)) % p.B;
  const int l = blockIdx.x / (p.NB * p.Hkv * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t obase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;
  unsigned long long* ws_claim = (unsigned long long*)p.ws_col;   // (rows, Tn) words of 64 bits
  const int64_t n_keys = (int64_t)gridDim.x * p.BS;               // == L * B * Hkv * Tn

  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) return;

  __shared__ int nvalid_s, mine_s;
  list_valid_pages(p.table + (int64_t)b * p.NB, p.NB, p.num_pages, jp, vpage, vidx, nullptr, &nvalid_s, &mine_s);
  for (int i = tid; i < 2 * TN * ROWF; i += kThreads) kbuf0[i] = 0.f;
  __syncthreads();
  const int n = nvalid_s, ai = mine_s;
  const int nd = n / 2 + (((n & 1) || ai < n / 2) ? 1 : 0);     // distances 0 .. nd-1
  const int tiles_per_page = p.BS / TN;
  const int ntiles = nd * tiles_per_page;
  // tile / tiles_per_page without a division per tile (at most a few hundred tiles, a handful per page)
  const int tpp_rcp = (65536 + tiles_per_page - 1) / tiles_per_page;
  const int dpieces = p.D / 4;
  const int64_t k_row = (int64_t)p.Hkv * p.D * 4;
  const char* kbase = p.k + (l * p.k_sl) * 4 + (int64_t)h * p.D * 4;

  const int st_piece = tid % PIECES, st_row0 = tid / PIECES;
  vec16 pre[STAGE_IT];
  auto col_page = [&](int d) { return ai + d < n ? ai + d : ai + d - n; };
  auto issue_loads = [&](int tile) {
    const int d = (tile * tpp_rcp) >> 16, toff = (tile - d * tiles_per_page) * TN;
    const char* src = kbase + (int64_t)vpage[col_page(d)] * p.k_sp * 4 + (int64_t)toff * k_row;
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i) {
      const int row = st_row0 + i * ROWS_PER_IT;
      pre[i] = vec16{0u, 0u, 0u, 0u};
      if (st_piece < dpieces) pre[i] = *(const vec16*)(src + (int64_t)row * k_row + st_piece * 16);
    }
  };
  auto commit_loads = [&](float* buf) {
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i) {
      const int row = st_row0 + i * ROWS_PER_IT;
      float e[4];
      Unpack<T>::run(pre[i], e);
      float ss = (e[0] * e[0] + e[1] * e[1]) + (e[2] * e[2] + e[3] * e[3]);
      ss = pieces_sum<PIECES>(ss);
      const float rn = __builtin_amdgcn_rcpf(fmaxf(__builtin_amdgcn_sqrtf(ss), p.eps)) * kPlaneScale;
      if (st_piece < dpieces) {
        f16x4_t h1, h2;
        split_planes(make_float4(e[0] * rn, e[1] * rn, e[2] * rn, e[3] * rn), h1, h2);
        char* dst = (char*)(buf + row * ROWF) + st_piece * 8;
        *(f16x4_t*)dst = h1;
        *(f16x4_t*)(dst + kPlaneBytes) = h2;
      }
    }
  };

  const int row_blocks = p.BS / 32;
  const int rb = wave;
  const bool active = rb < row_blocks;
  // A fragments: this lane's key row of page a, normalised and split; k-step s of wave half
  // `half` takes elements 16 s + 8 half .. + 7 (pieces 4 s + 2 half and the next one), the same
  // order as the B operand's 16-byte LDS reads
  f16x8_t a1[KSH], a2[KSH];
  {
    const int slot = (active ? rb : 0) * 32 + col;
    const char* src = kbase + (int64_t)rpid * p.k_sp * 4 + (int64_t)slot * k_row;
    float4 mine[2 * KSH];
    float ss = 0.f;
#pragma unroll
    for (int pc = 0; pc < PIECES; ++pc) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (pc < dpieces) v = *(const float4*)(src + pc * 16);
      ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
      if (((pc >> 1) & 1) == 0) mine[(pc >> 2) * 2 + (pc & 1)] = v;
      else if (half) mine[(pc >> 2) * 2 + (pc & 1)] = v;
    }
    const float rn = active ? __builtin_amdgcn_rcpf(fmaxf(__builtin_amdgcn_sqrtf(ss), p.eps)) * kPlaneScale : 0.f;
#pragma unroll
    for (int s = 0; s < KSH; ++s) {
      f16x4_t l1, l2, u1, u2;
      const float4 lo = mine[2 * s], up = mine[2 * s + 1];
      split_planes(make_float4(lo.x * rn, lo.y * rn, lo.z * rn, lo.w * rn), l1, l2);
      split_planes(make_float4(up.x * rn, up.y * rn, up.z * rn, up.w * rn), u1, u2);
      a1[s] = f16x8_t{l1[0], l1[1], l1[2], l1[3], u1[0], u1[1], u1[2], u1[3]};
      a2[s] = f16x8_t{l2[0], l2[1], l2[2], l2[3], u2[0], u2[1], u2[2], u2[3]};
    }
  }
  float rsum[16], cval[16];
  int ccol[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) { rsum[r] = 0.f; cval[r] = 0.f; ccol[r] = -1; }
  const float thr_s = p.threshold * (kPlaneScale * kPlaneScale);
  bool wave_claims = false;       // any tile of this wave with an entry over the threshold (uniform)

  // the column sums of tile t are complete after the barrier that ends it: the waves' shares are
  // added in wave order and stored while tile t+1 is being multiplied
  auto finish_columns = [&](int tile) {
    const int d = (tile * tpp_rcp) >> 16, toff = (tile - d * tiles_per_page) * TN;
    if (d == 0 || tid >= TN) return;
    const float* pt = l_cpart + (tile & 1) * kSymWaves * TN;
    float v = pt[tid];
#pragma unroll
    for (int w2 = 1; w2 < kSymWaves; ++w2) v += pt[w2 * TN + tid];
    const int jc = vidx[col_page(d)];
    p.ws_chunk[(int64_t)(d - 1) * n_keys + obase + (int64_t)jc * p.BS + toff + tid] = v * kPlaneUnscale;
  };

  if (ntiles > 0) { issue_loads(0); commit_loads(kbuf0); }
  __syncthreads();
  for (int tile = 0; tile < ntiles; ++tile) {
    float* cur = (tile & 1) ? kbuf1 : kbuf0;
    float* nxt = (tile & 1) ? kbuf0 : kbuf1;
    if (tile + 1 < ntiles) issue_loads(tile + 1);
    const int d = (tile * tpp_rcp) >> 16, toff = (tile - d * tiles_per_page) * TN;
    const int jc = vidx[col_page(d)];
    float* cpart = l_cpart + ((tile & 1) * kSymWaves + wave) * TN;
#pragma unroll
    for (int st = 0; st < NSUB; ++st) {
      float csum = 0.f, rv = 0.f;
      int rlast = -1;
      if (active) {
        f32x16_t acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
        const char* br = (const char*)(cur + (st * 32 + col) * ROWF) + 16 * half;
#pragma unroll
        for (int s = 0; s < KSH; ++s)
          acc = mma_planes(a1[s], a2[s], *(const f16x8_t*)(br + 32 * s),
                           *(const f16x8_t*)(br + kPlaneBytes + 32 * s), acc);
        // sums, claim values and the threshold stay in the planes' scale (a power of two: the
        // same bits come out when it is taken off at the end)
        const int cslot = toff + st * 32 + col;
        const int cidx = jc * p.BS + cslot;   // logical index of this lane's column key
        if (d == 0) {     // the page against itself: a key is not its own neighbour
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3) == cslot) acc[r] = 0.f;
        }
        const bool any_over = __builtin_amdgcn_ballot_w64(tile_lane_max(acc) > thr_s) != 0ull;
        wave_claims |= any_over;
        if (!any_over) {
#pragma unroll
          for (int r = 0; r < 16; ++r) { rsum[r] += acc[r]; csum += acc[r]; }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
            const float sv = acc[r];
            rsum[r] += sv;
            csum += sv;
            const bool over = sv > thr_s;
            if (over && cidx > ccol[r]) { ccol[r] = cidx; cval[r] = sv; }
            if (over) { rlast = rslot; rv = sv; }   // rslot grows with r inside a lane
          }
          if (d != 0) {
            const int orl = lane_xor32(rlast);
            const float orv = lane_xor32(rv);
            if (orl > rlast) { rlast = orl; rv = orv; }
            if (half == 0 && rlast >= 0)   // the column key's claim candidate among page a's rows
              atomicMax(&ws_claim[obase + cidx], ((unsigned long long)(unsigned)(jp * p.BS + rlast + 1) << 32) |
                                                     __float_as_uint(rv * kPlaneUnscale));
          }
        }
      }
      if (d != 0) {
        csum += lane_xor32(csum);
        if (half == 0) cpart[st * 32 + col] = csum;
      }
    }
    if (tile + 1 < ntiles) commit_loads(nxt);
    __syncthreads();
    finish_columns(tile);
  }
  // ---- row side: sums and claims over the 32 lanes of each half
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float sv = half_sum(rsum[r]);
    int c = ccol[r];
    float v = cval[r];
    if (wave_claims) last_claim_reduce(c, v);
    if (active && col == 0) {
      const int64_t oi = obase + (int64_t)jp * p.BS + rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
      p.ws_sum[oi] = sv * kPlaneUnscale;
      if (c >= 0)
        atomicMax(&ws_claim[oi], ((unsigned long long)(unsigned)(c + 1) << 32) | __float_as_uint(v * kPlaneUnscale));
    }
  }
}

// ------------------------------------------------------------------ fp32 caches, lightning, whole page in LDS
// Pages of at most 256 keys; a workgroup walks its share of the pages of a (layer, sequence, head) row:
// a page is loaded once with coalesced 16-byte loads into registers (requested under the tiles of
// the page before), normalised on the way into LDS (132 KB), and after ONE barrier every wave
// multiplies its 32 rows (A operand read from the same LDS copy) with its share of the column
// blocks (every unordered pair of blocks once): no tile pipeline, no strided row loads.
constexpr int kPage32Rows = 256;
constexpr int kPage32Threads = 512;
__global__ __launch_bounds__(kPage32Threads) void gram_page_f32_kernel(GramArgs p) {
  typedef F32 T;
  constexpr int PIECES = kDmax / 4;                            // 16-byte pieces per key row (32)
  constexpr int ROWS_PER_IT = kPage32Threads / PIECES;         // 16
  constexpr int ITERS = kPage32Rows / ROWS_PER_IT;             // 16
  extern __shared__ __align__(16) char smem[];
  float* kpl = (float*)smem;                                   // [256][ROWF] normalised keys
  unsigned long long* l_corr = (unsigned long long*)(kpl + kPage32Rows * ROWF);
  unsigned long long* l_claim = l_corr + kPage32Rows;       // (claimed index + 1) << 32 | value bits
  float* l_sum = (float*)(l_claim + kPage32Rows);
  float* l_csum = l_sum + kPage32Rows;                        // [4][256] column sums per distance
  int* l_code = (int*)(l_csum + 4 * kPage32Rows);             // [NB] the block table row

  const int tid0 = threadIdx.x;
  // a workgroup walks the pages of one (layer, sequence, kv head) row: the next page's keys are
  // requested into registers under the tiles of this one (a page fills the LDS a CU has, so
  // nothing else could overlap its load)
  const int h = blockIdx.x % p.Hkv;
  const int part = (blockIdx.x / p.Hkv) % p.parts;
  const int b = (blockIdx.x / (p.Hkv * p.parts)) % p.B;
  const int l = blockIdx.x / (p.Hkv * p.parts * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t rowbase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;
  const int dpieces = p.D / 4;
  const int64_t k_row = (int64_t)p.Hkv * p.D * 4;
  const char* layer = p.k + l * p.k_sl * 4 + (int64_t)h * p.D * 4;

  for (int j = tid0; j < p.NB; j += kPage32Threads) l_code[j] = p.table[(int64_t)b * p.NB + j];
  __syncthreads();
  auto page_of = [&](int j) {     // page id of table entry j, or -1 (uniform)
    const int code = __builtin_amdgcn_readfirstlane(l_code[j]);
    const int pid = page_is_pad(code) ? -1 : page_id(code);
    return pid < p.num_pages ? pid : -1;
  };
  auto next_valid = [&](int j) {        // of this workgroup's entries
    while (j < p.NB && page_of(j) < 0) j += p.parts;
    return j;
  };
  for (int j = part; j < p.NB; j += p.parts) {      // entries without a page score -inf
    if (page_of(j) >= 0) continue;
    for (int s = tid0; s < p.BS; s += kPage32Threads) Elem<T>::st(p.r_out, rowbase + (int64_t)j * p.BS + s, -INFINITY);
  }
  float4 raw[ITERS];
  auto request = [&](int j, int piece, int prow0) {
    const char* page = layer + (int64_t)page_of(j) * p.k_sp * 4;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int row = it * ROWS_PER_IT + prow0;
      raw[it] = *(const float4*)(page + (int64_t)(row < p.BS ? row : 0) * k_row +
                                 (piece < dpieces ? piece : 0) * 16);
    }
  };
  int jp = next_valid(part);
  if (jp < p.NB) request(jp, tid0 % PIECES, tid0 / PIECES);
#pragma unroll 1
  while (jp < p.NB) {
  // The thread id is made opaque once per page: what is derived from it (LDS addresses, row
  // indices) is then computed where a page uses it, not before the loop and held in registers
  // through all of it, where the prefetched page needs them.
  int tid = tid0;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int piece = tid % PIECES, prow0 = tid / PIECES;
  const int64_t obase = rowbase + (int64_t)jp * p.BS;
  // ---- stage: norms and the normalised copy of the page requested a page ago
  {
    const int row0 = prow0;
    if (tid < kPage32Rows) { l_corr[tid] = 0ull; l_claim[tid] = 0ull; }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int row = it * ROWS_PER_IT + row0;
      if (!(row < p.BS && piece < dpieces)) raw[it] = make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 e = raw[it];
      float ss = (e.x * e.x + e.y * e.y) + (e.z * e.z + e.w * e.w);
      ss = pieces_sum<PIECES>(ss);
      const float rn = __builtin_amdgcn_rcpf(fmaxf(__builtin_amdgcn_sqrtf(ss), p.eps)) * kPlaneScale;
      f16x4_t h1, h2;
      split_planes(make_float4(e.x * rn, e.y * rn, e.z * rn, e.w * rn), h1, h2);
      char* dst = (char*)(kpl + row * ROWF) + piece * 8;
      *(f16x4_t*)dst = h1;
      *(f16x4_t*)(dst + kPlaneBytes) = h2;
    }
  }
  __syncthreads();
  const int nj = next_valid(jp + p.parts);
  if (nj < p.NB) request(nj, piece, prow0);

  // ---- Gram tiles, every unordered pair of 32-key blocks once: wave a multiplies its block with
  // the blocks (a + d) mod n, d = 0 .. n/2 (the last distance only for the lower half of the
  // waves when n is even).  A tile off the diagonal block serves both of its sides: the rows get
  // their partial row sums and claims as before, the columns get the tile's column sums
  // (slot [d][key], written by exactly one wave, added in a fixed order at the end) and the last
  // ROW over the threshold as their claim.  Claims travel as (index, value) pairs through one
  // 64-bit atomicMax per key, so the result does not depend on the order of the waves.
  const int nrb = p.BS / 32;
  if (wave < nrb) {
    const int rb = wave;
    // lane (col, half) holds elements 16 s + 8 half .. + 7 of key rb * 32 + col for k-step s
    f16x8_t a1[KSH], a2[KSH];
    {
      const char* ar = (const char*)(kpl + (rb * 32 + col) * ROWF) + 16 * half;
#pragma unroll
      for (int s = 0; s < KSH; ++s) {
        a1[s] = *(const f16x8_t*)(ar + 32 * s);
        a2[s] = *(const f16x8_t*)(ar + kPlaneBytes + 32 * s);
      }
    }
    float rsum[16], cval[16];
    int ccol[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) { rsum[r] = 0.f; cval[r] = 0.f; ccol[r] = -1; }
    const int nd = nrb / 2 + (((nrb & 1) || rb < nrb / 2) ? 1 : 0);   // distances 0 .. nd-1
    const float thr_s = p.threshold * (kPlaneScale * kPlaneScale);
    bool wave_claims = false;     // any tile of this wave with an entry over the threshold (uniform)
#pragma unroll 1
    for (int d = 0; d < nd; ++d) {
      const int cb = rb + d < nrb ? rb + d : rb + d - nrb;
      f32x16_t acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      const char* br = (const char*)(kpl + (cb * 32 + col) * ROWF) + 16 * half;
#pragma unroll
      for (int s = 0; s < KSH; ++s)
        acc = mma_planes(a1[s], a2[s], *(const f16x8_t*)(br + 32 * s),
                         *(const f16x8_t*)(br + kPlaneBytes + 32 * s), acc);
      // sums, claim values and the threshold stay in the planes' scale (a power of two: the same
      // bits come out when it is taken off at the end)
      const int cslot = cb * 32 + col;
      if (d == 0) {     // the block against itself: a key is not its own neighbour
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3) == cslot) acc[r] = 0.f;
      }
      const bool any_over = __builtin_amdgcn_ballot_w64(tile_lane_max(acc) > thr_s) != 0ull;
      wave_claims |= any_over;
      float csum = 0.f, rv = 0.f;     // column side: sum over this lane's rows, last row over the threshold
      int rlast = -1;
      if (!any_over) {
#pragma unroll
        for (int r = 0; r < 16; ++r) { rsum[r] += acc[r]; csum += acc[r]; }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
          const float sv = acc[r];
          rsum[r] += sv;
          csum += sv;
          const bool over = sv > thr_s;
          // columns come in ascending order until they wrap
          if (over && (cb >= rb || cslot > ccol[r])) { ccol[r] = cslot; cval[r] = sv; }
          if (over) { rlast = rslot; rv = sv; }     // rslot grows with r inside a lane
        }
      }
      if (d != 0) {
        csum += lane_xor32(csum);
        if (half == 0) l_csum[(d - 1) * kPage32Rows + cslot] = csum * kPlaneUnscale;
        if (any_over) {
          const int orl = lane_xor32(rlast);
          const float orv = lane_xor32(rv);
          if (orl > rlast) { rlast = orl; rv = orv; }
          if (half == 0 && rlast >= 0)
            atomicMax(&l_claim[cslot], ((unsigned long long)(unsigned)(rlast + 1) << 32) |
                                           __float_as_uint(rv * kPlaneUnscale));
        }
      }
    }
    // 128 sequences of 9 pages, a value after the other 565 us without claims and 620 with one at every key, now 513 and 545
    const int r = sixteen_half_sum(rsum, lane);
    if (wave_claims) sixteen_last_claims(ccol, cval, lane);
    if ((lane & 16) == 0) {
      const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
      l_sum[rslot] = rsum[0] * kPlaneUnscale;
      if (wave_claims && ccol[0] >= 0)
        atomicMax(&l_claim[rslot], ((unsigned long long)(unsigned)(ccol[0] + 1) << 32) |
                                       __float_as_uint(cval[0] * kPlaneUnscale));
    }
  }
  __syncthreads();
  for (int j = tid; j < p.BS; j += kPage32Threads) {
    const unsigned long long cl = l_claim[j];
    const int c = (int)(cl >> 32) - 1;
    if (c >= 0 && c < p.BS) atomicAdd(&l_corr[c], to_fixed32(__uint_as_float((unsigned)cl)));
  }
  __syncthreads();
  const int ndist = nrb / 2;     // column-side slots in use: distances 1 .. nrb/2
  for (int i = tid; i < p.BS; i += kPage32Threads) {
    float sv = l_sum[i];
    const int blk = i >> 5;
    for (int d = 1; d <= ndist; ++d) {
      // the wave that wrote slot [d][i] is block (blk - d) mod n; with n even the last distance
      // is only run by the lower half of the waves
      const int a = blk - d >= 0 ? blk - d : blk - d + nrb;
      const bool ran = d < nrb / 2 + (((nrb & 1) || a < nrb / 2) ? 1 : 0);
      if (ran) sv += l_csum[(d - 1) * kPage32Rows + i];
    }
    Elem<T>::st(p.r_out, obase + i, sv - from_fixed32(l_corr[i]));
  }
  __syncthreads();   // the page and the per-key slots in LDS are free for the next page
  jp = nj;
  }
}

// ------------------------------------------------------------------ 16-bit caches: split-bf16 Gram
// Same algorithm with the contraction on the bf16 matrix cores.  The fp32 normalised key
// x = k / n is split into hi = bf16(x) and lo = bf16(x - hi); S = hi.hi + hi.lo + lo.hi drops
// only the lo.lo term (relative 2^-18), i.e. fp32-grade dot products at a third of the bf16
// MFMA rate instead of the 16x slower fp32 MFMA.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
constexpr int ROWH = kDmax * 2 + 16;  // bytes per LDS row of one bf16 plane (16 B pad)

__device__ __forceinline__ void split8(const float* x, bf16x8_t& hi, bf16x8_t& lo) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const __bf16 h = (__bf16)x[q];
    hi[q] = h;
    lo[q] = (__bf16)(x[q] - (float)h);
  }
}

// NW waves per workgroup: every wave owns one 32-row block of the row page per round, so with 8
// waves a 256-token page needs a single pass over the column tiles (they are normalised and split
// once instead of twice).
template <typename T, bool RAW, int NW>
__global__ __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) void gram_split_kernel(GramArgs p) {
  constexpr int kThreads = NW * 64, kWaves = NW;   // shadow the file-wide 4-wave constants
  static_assert(T::bytes == 2, "split path is for 16-bit caches");
  constexpr int PIECES = kDmax / 8;                 // 16-byte pieces per full key row
  constexpr int ROWS_PER_IT = kThreads / PIECES;    // 16
  constexpr int STAGE_IT = TN / ROWS_PER_IT;        // 4
  constexpr int NSUB = TN / 32;
  constexpr int KSB = kDmax / 16;                   // bf16 MFMA k-steps
  constexpr int PLANE = TN * ROWH;                  // bytes of one plane of one buffer

  extern __shared__ __align__(16) char smem[];
  char* buf0 = smem;                                // [hi plane][lo plane]
  char* buf1 = smem + 2 * PLANE;
  unsigned long long* l_corr = (unsigned long long*)(smem + 4 * PLANE);   // [BS] claimed from a row
  float* l_sum = (float*)(l_corr + (RAW ? 0 : p.BS));
  float* l_val = l_sum + (RAW ? 0 : p.BS);
  int* l_col = (int*)(l_val + (RAW ? 0 : p.BS));
  int* vpage = l_col + (RAW ? 0 : p.BS);
  int* vidx = vpage + p.NB;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int jp = blockIdx.x % p.NB;
  const int h = (blockIdx.x / p.NB) % p.Hkv;
  const int b = (blockIdx.x / (p.NB * p.Hkv)) % p.B;
  const int l = blockIdx.x / (p.NB * p.Hkv * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t orow = (((int64_t)l * p.B + b) * p.Hkv + h);
  const float epsr = Elem<T>::rnd(p.eps);

  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) {
    if (!RAW)
      for (int s = tid; s < p.BS; s += kThreads)
        Elem<T>::st(p.r_out, orow * Tn + (int64_t)jp * p.BS + s, -INFINITY);
    return;
  }
  __shared__ int ncols_s;
  if (RAW) {
    list_valid_pages(p.table + (int64_t)b * p.NB, p.NB, p.num_pages, jp, vpage, vidx, nullptr, &ncols_s, nullptr);
  } else if (tid == 0) {
    vpage[0] = rpid; vidx[0] = jp; ncols_s = 1;
  }
  for (int i = tid; i < 4 * PLANE / 4; i += kThreads) ((uint32_t*)smem)[i] = 0u;
  __syncthreads();
  const int tiles_per_page = p.BS / TN;
  const int ntiles = ncols_s * tiles_per_page;
  const int dpieces = p.D / 8;
  const int64_t k_row = (int64_t)p.Hkv * p.D * 2;
  const char* kbase = p.k + (l * p.k_sl) * 2 + (int64_t)h * p.D * 2;

  const int st_piece = tid % PIECES, st_row0 = tid / PIECES;
  vec16 pre[STAGE_IT];
  auto issue_loads = [&](int tile) {
    const int vp = tile / tiles_per_page, toff = (tile - vp * tiles_per_page) * TN;
    const char* src = kbase + (int64_t)vpage[vp] * p.k_sp * 2 + (int64_t)toff * k_row;
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i) {
      const int row = st_row0 + i * ROWS_PER_IT;
      const int pc = st_piece < dpieces ? st_piece : 0;  // clamp: unconditional load
      pre[i] = *(const vec16*)(src + (int64_t)row * k_row + pc * 16);
    }
  };
  auto commit_loads = [&](char* buf) {
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i) {
      const int row = st_row0 + i * ROWS_PER_IT;
      float e[8];
      Unpack<T>::run(pre[i], e);
      float ss = 0.f;
      if (st_piece < dpieces) {
#pragma unroll
        for (int q = 0; q < 8; ++q) ss += e[q] * e[q];
      }
      ss = pieces_sum<PIECES>(ss);
      const float n = fmaxf(Elem<T>::rnd(sqrtf(ss)), epsr);
      if (st_piece < dpieces) {
#pragma unroll
        for (int q = 0; q < 8; ++q) e[q] = e[q] / n;
        bf16x8_t hi, lo;
        split8(e, hi, lo);
        *(bf16x8_t*)(buf + row * ROWH + st_piece * 16) = hi;
        *(bf16x8_t*)(buf + PLANE + row * ROWH + st_piece * 16) = lo;
      }
    }
  };

  const int row_blocks = p.BS / 32;
  const int NR = (row_blocks + kWaves - 1) / kWaves;
  for (int rr = 0; rr < NR; ++rr) {
    const int rb = rr * kWaves + wave;
    const bool active = rb < row_blocks;
    // ---- A fragments: this lane's key row; lane (row, half) holds k = 16 s + 8 half + i
    bf16x8_t ahi[KSB], alo[KSB];
    {
      const int slot = (active ? rb : 0) * 32 + col;
      const char* src = kbase + (int64_t)rpid * p.k_sp * 2 + (int64_t)slot * k_row;
      float x[KSB][8];
      float ss = 0.f;
#pragma unroll
      for (int s = 0; s < KSB; ++s) {
        const int pc = 2 * s + half;
        vec16 v = vec16{0u, 0u, 0u, 0u};
        if (pc < dpieces) v = *(const vec16*)(src + pc * 16);
        Unpack<T>::run(v, x[s]);
#pragma unroll
        for (int q = 0; q < 8; ++q) ss += x[s][q] * x[s][q];
      }
      ss += lane_xor32(ss);  // the other half of the row
      const float n = fmaxf(Elem<T>::rnd(sqrtf(ss)), epsr);
#pragma unroll
      for (int s = 0; s < KSB; ++s) {
#pragma unroll
        for (int q = 0; q < 8; ++q) x[s][q] = active ? x[s][q] / n : 0.f;
        split8(x[s], ahi[s], alo[s]);
      }
    }
    float rsum[16], cval[16];
    int ccol[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) { rsum[r] = 0.f; cval[r] = 0.f; ccol[r] = -1; }

    if (ntiles > 0) { issue_loads(0); commit_loads(buf0); }
    __syncthreads();
    for (int tile = 0; tile < ntiles; ++tile) {
      char* cur = (tile & 1) ? buf1 : buf0;
      char* nxt = (tile & 1) ? buf0 : buf1;
      if (tile + 1 < ntiles) issue_loads(tile + 1);
      const int vp = tile / tiles_per_page, toff = (tile - vp * tiles_per_page) * TN;
      const int jc = vidx[vp];
      if (active) {
#pragma unroll 1
        for (int st = 0; st < NSUB; ++st) {
          f32x16_t acc;
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] = 0.f;
          const char* brow = cur + (st * 32 + col) * ROWH + half * 16;
#pragma unroll
          for (int s0 = 0; s0 < KSB; s0 += 4) {
            bf16x8_t bh[4], bl[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              bh[s] = *(const bf16x8_t*)(brow + (s0 + s) * 32);
              bl[s] = *(const bf16x8_t*)(brow + PLANE + (s0 + s) * 32);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahi[s0 + s], bh[s], acc, 0, 0, 0);
              acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahi[s0 + s], bl[s], acc, 0, 0, 0);
              acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(alo[s0 + s], bh[s], acc, 0, 0, 0);
            }
          }
          const int cslot = toff + st * 32 + col;
          const int cidx = jc * p.BS + cslot;
          const bool same_page = jc == jp;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
            float s = acc[r];
            if (same_page && rslot == cslot) s = 0.f;
            rsum[r] += s;
            if (s > p.threshold) { ccol[r] = cidx; cval[r] = s; }
          }
        }
      }
      if (tile + 1 < ntiles) commit_loads(nxt);
      __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float s = rsum[r];
      int c = ccol[r];
      float v = cval[r];
      s = half_sum(s);
      last_claim_reduce(c, v);
      if (active && col == 0) {
        const int rslot = rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
        if (RAW) {
          const int64_t oi = orow * Tn + (int64_t)jp * p.BS + rslot;
          p.ws_sum[oi] = s;
          p.ws_col[oi] = c;
          p.ws_val[oi] = v;
        } else {
          l_sum[rslot] = s;
          l_col[rslot] = c - jp * p.BS;
          l_val[rslot] = v;
        }
      }
    }
  }
  if (!RAW) {
    // claim values go to the rows they were taken from as 2^-32 fixed-point atomics
    // (order-independent), not through a scan of all claims per row
    for (int i = tid; i < p.BS; i += kThreads) l_corr[i] = 0ull;
    __syncthreads();
    for (int j = tid; j < p.BS; j += kThreads) {
      const int c = l_col[j];
      if (c >= 0 && c < p.BS) atomicAdd(&l_corr[c], to_fixed32(l_val[j]));
    }
    __syncthreads();
    for (int i = tid; i < p.BS; i += kThreads)
      Elem<T>::st(p.r_out, orow * Tn + (int64_t)jp * p.BS + i, l_sum[i] - from_fixed32(l_corr[i]));
  }
}

// ------------------------------------------------------------------ lightning, whole page in LDS
// Per-page variant for 16-bit caches and pages of up to 256 keys: the page is normalised and
// split once into LDS (hi and lo planes, 2 x 68 KB).  The Gram matrix is symmetric, so every
// unordered pair of 32-key blocks is multiplied once: wave a takes the blocks (a, a+d mod n)
// for d = 0..n/2 (the pairs at distance n/2 go to the lower half of the waves), which is 5 or 4
// tiles per wave for a 256-key page instead of 8.  A tile only feeds the claim rule (its
// entries over the threshold update the last-column-over-threshold of the keys on BOTH of its
// sides); the row sums do not need the matrix at all:
//     sum_{j != i} e_i.e_j = e_i . (sum_j e_j - e_i)
// is one fp32 dot product per key against the page's summed key, done while the raw keys are
// still in registers.  The values of the (at most one per key) claimed entries are recomputed
// afterwards from the two planes.
constexpr int kPageThreads = 512;
constexpr int kPageWaves = kPageThreads / 64;
constexpr int kPageRows = 256;

// Two floats to packed bf16 (round to nearest even) in one v_cvt_pk_bf16_f32.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
}
// hi = bf16(x), lo = bf16(x - hi) for eight values, packed pairwise.
__device__ __forceinline__ void split8_pk(const float* x, u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t h = pk_bf16(x[2 * i], x[2 * i + 1]);
    hi[i] = h;
    lo[i] = pk_bf16(x[2 * i] - __uint_as_float(h << 16), x[2 * i + 1] - __uint_as_float(h & 0xffff0000u));
  }
}


// Largest value over the 32 lanes of a wave half.
__device__ __forceinline__ int half_max_i(int v) {
  v = max(v, dpp_row_ror<8>(v));
  v = max(v, dpp_row_ror<4>(v));
  v = max(v, dpp_row_ror<2>(v));
  v = max(v, dpp_row_ror<1>(v));
  return max(v, lane_xor16(v));
}

// The 16-bit MFMA of the cache dtype: products of cache elements are exact in fp32.
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
template <typename T> struct Mfma16;
template <> struct Mfma16<BF16> {
  typedef bf16x8_t V;
  __device__ static __forceinline__ f32x16_t run(V a, V b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma16<F16> {
  typedef f16x8_t V;
  __device__ static __forceinline__ f32x16_t run(V a, V b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// A float as three 16-bit pieces of the cache dtype (hi + mid + lo carries its fp32 mantissa).
template <typename T> struct Split3;
template <> struct Split3<BF16> {
  __device__ static __forceinline__ void run(float v, uint16_t* o) {
    const float h = bf16_round(v), m = bf16_round(v - h), l = bf16_round(v - h - m);
    o[0] = (uint16_t)(__float_as_uint(h) >> 16);
    o[1] = (uint16_t)(__float_as_uint(m) >> 16);
    o[2] = (uint16_t)(__float_as_uint(l) >> 16);
  }
  // two floats, their pieces side by side
  __device__ static __forceinline__ void two(float x, float y, uint32_t* o) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const zp_f32x2 v = {x, y};
      o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, zp_bf16x2));
      x -= __uint_as_float(o[i] << 16);
      y -= __uint_as_float(o[i] & 0xffff0000u);
    }
  }
};
template <> struct Split3<F16> {
  __device__ static __forceinline__ void run(float v, uint16_t* o) {
    o[0] = float_to_f16_bits(v);
    const float r1 = v - f16_bits_to_float(o[0]);
    o[1] = float_to_f16_bits(r1);
    o[2] = float_to_f16_bits(r1 - f16_bits_to_float(o[1]));
  }
  __device__ static __forceinline__ void two(float x, float y, uint32_t* o) {
    uint16_t a[3], b[3];
    run(x, a);
    run(y, b);
#pragma unroll
    for (int i = 0; i < 3; ++i) o[i] = (uint32_t)a[i] | ((uint32_t)b[i] << 16);
  }
};

// The cosine matrix factors as S_ij = rn_i rn_j (k_i . k_j) with rn = 1 / norm: the raw 16-bit
// keys go to the matrix cores as they are (one MFMA per k-step, exact products, fp32 sums) and
// the two scale factors are applied to the accumulators.  Sixteen waves share a compute unit's
// four vector units, and vector instruction issue is the first thing they run out of, so
// everything that can be is kept off the vector ALUs:
//   * the page goes from global memory straight into LDS (no staging registers, no LDS stores);
//     a load instruction moves four key rows, which sit 1040 bytes apart in groups of four so that
//     the matrix cores' fragment reads spread over the banks: piece g (16 bytes) of row r of a
//     group at (g / 4) * 256 + r * 64 + (g % 4) * 16;
//   * wave a loads row block a, so it can take the block's norms from the diagonal of its own
//     Gram tile (which the claim rule needs anyway) before any barrier;
//   * the summed normalised key  sum_j rn_j k_j  is a matrix product too, contracted over the
//     keys: A = rn as three 16-bit pieces (rows 0..2), B = the keys read through the transposing
//     LDS load (`ds_read_b64_tr_b16`: lane i of sixteen receives column i of a 4 x 16 block).
// One plane of raw keys in LDS (65 KB), so two workgroups share a compute unit.  A workgroup
// walks the pages of one row: once the tiles of a page are done nothing reads its keys in LDS
// any more, so the next page is requested then and lands while the row sums are finished.
constexpr int kPgGrp = 1040;                          // bytes from one group of four key rows to the next
constexpr int kPgBytes = (kPageRows / 4) * kPgGrp;    // the page in LDS
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));
typedef void __attribute__((address_space(3))) * lds_ptr_t;

#ifdef ZP_PAGE_STAMP
// Measurement build: thread 0 of every workgroup records the core-clock counter at the phase
// boundaries and the constant-rate counter at both ends.
constexpr int kPageStampMax = 1 << 16;
__device__ long long zp_page_stamp_buf[kPageStampMax * 12];
extern "C" int zp_debug_page_stamps(long long* dst, int n_groups) {
  return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(zp_page_stamp_buf), (size_t)n_groups * 12 * 8);
}
#define ZP_PSTAMP() do { if (tid == 0 && nst < 10) st_[nst++] = clock64(); } while (0)
#else
#define ZP_PSTAMP() do { } while (0)
#endif

// 1 / norm as 16-bit pieces for the matrix cores.  bf16 has fp32's exponent range: three pieces
// carry all 24 mantissa bits.  fp16 does not: the pieces are taken of rn * 2^-x with x chosen per
// block of 32 keys so that the block's largest value sits at the top of fp16's range, which leaves
// 39 bits below it; the accumulator is rescaled where the block changes.
template <typename T> struct RnScale;
template <> struct RnScale<BF16> { static constexpr bool per_block = false; };
template <> struct RnScale<F16> { static constexpr bool per_block = true; };

template <typename T>
__global__ __launch_bounds__(kPageThreads, 4) void gram_page_kernel(GramArgs p) {
  static_assert(T::bytes == 2, "16-bit caches only");
  typedef typename Mfma16<T>::V frag_t;
  constexpr int PIECES = kDmax / 8;
  constexpr int KSB = kDmax / 16;

  extern __shared__ __align__(16) char smem[];
  char* k_pl = smem;                                   // raw keys
  char* s_pl = smem + kPgBytes;                        // [4][kDmax] 16-bit: summed key as hi, mid, lo; zeros
  char* rn_pl = s_pl + 4 * kDmax * 2;                  // [4][kPageRows] 16-bit: 1 / norm as hi, mid, lo; zeros
  // claimed from a row / row sums: two copies, taken in turn by the pages of the walk, because a
  // page's last phase reads them while the next page's first phase writes them
  unsigned long long* l_corr2 = (unsigned long long*)(rn_pl + 4 * kPageRows * 2);
  float* l_sum2 = (float*)(l_corr2 + 2 * kPageRows);
  float* l_rn = l_sum2 + 2 * kPageRows;                // 1 / norm
  int* l_col = (int*)(l_rn + kPageRows);
  int* l_bexp = l_col + kPageRows;                     // [kPageWaves] scale exponent of a block's rn pieces
  int* l_any2 = l_bexp + kPageWaves;                   // [2] whether a key of the page has a claim
  int* l_code = l_any2 + 2;                            // [NB] the block table row

  const int tid = threadIdx.x;
#ifdef ZP_PAGE_STAMP
  long long st_[10];
  int nst = 0;
#endif
  // a workgroup walks its share of the pages of one (layer, sequence, kv head) row
  const int h = blockIdx.x % p.Hkv;
  const int part = (blockIdx.x / p.Hkv) % p.parts;
  const int b = (blockIdx.x / (p.Hkv * p.parts)) % p.B;
  const int l = blockIdx.x / (p.Hkv * p.parts * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t rowbase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;
  const float epsr = Elem<T>::rnd(p.eps);
  const int dpieces = p.D / 8;
  const int k_row = p.Hkv * p.D * 2;
  const char* layer = p.k + l * p.k_sl * 2 + (int64_t)h * p.D * 2;
  const int nrb = p.BS / 32;

  for (int j = tid; j < p.NB; j += kPageThreads) l_code[j] = p.table[(int64_t)b * p.NB + j];
  if (tid < kDmax / 2) ((uint32_t*)(s_pl + 3 * kDmax * 2))[tid] = 0u;
  else if (tid < kDmax / 2 + kPageRows / 2) ((uint32_t*)(rn_pl + 3 * kPageRows * 2))[tid - kDmax / 2] = 0u;
  if (dpieces < PIECES) {   // the tail of every key row must read as zero
    for (int i = tid; i < kPgBytes / 4; i += kPageThreads) ((uint32_t*)k_pl)[i] = 0u;
  }
  __syncthreads();
  // page id of table entry j, or -1 (wave-uniform)
  auto page_of = [&](int j) {
    const int code = __builtin_amdgcn_readfirstlane(l_code[j]);
    const int pid = page_is_pad(code) ? -1 : page_id(code);
    return pid < p.num_pages ? pid : -1;
  };
  auto next_valid = [&](int j) {        // of this workgroup's entries
    while (j < p.NB && page_of(j) < 0) j += p.parts;
    return j;
  };
  for (int j = part; j < p.NB; j += p.parts) {      // entries without a page score -inf
    if (page_of(j) >= 0) continue;
    for (int s = tid; s < p.BS; s += kPageThreads) Elem<T>::st(p.r_out, rowbase + (int64_t)j * p.BS + s, -INFINITY);
  }
  // ---- a page into LDS: wave w requests row block w, eight instructions of four rows
  auto request = [&](int j, int w, int ln) {
    if (w >= nrb) return;
    const int st_g = (ln >> 4) * 4 + (ln & 3), st_r = (ln >> 2) & 3;
    const char* page = layer + (int64_t)page_of(j) * p.k_sp * 2;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(page + (int64_t)w * 32 * k_row), 0, 32 * k_row, 0x00020000);
    const int voff = st_r * k_row + st_g * 16;
    if (st_g < dpieces) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(k_pl + (w * 8 + i) * kPgGrp), 16, voff,
                                                 i * 4 * k_row, 0, 0);
    }
  };

  int jp = next_valid(part);
  if (jp < p.NB) request(jp, __builtin_amdgcn_readfirstlane(tid >> 6), tid & 63);
  int par = 0;
#pragma unroll 1
  while (jp < p.NB) {
    // Lane and wave numbers are made opaque once per page: what is derived from them (LDS
    // addresses, row indices) is then computed where a page uses it instead of once before the
    // loop and held in registers through all of it, which the tiles have none to spare for.
    int lane = tid & 63;
    asm volatile("" : "+v"(lane));
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    asm volatile("" : "+s"(wave));
    const int half = lane >> 5, col = lane & 31;
    const int a = wave;
    // fragment of k-step s of this lane's row: base + (s / 2) * 256 + (s % 2) * 32
    const int rd_off = (col >> 2) * kPgGrp + (col & 3) * 64 + half * 16;
#ifdef ZP_PAGE_STAMP
    nst = 0;
    const long long wall0 = wall_clock64();
#endif
    ZP_PSTAMP();
    unsigned long long* l_corr = l_corr2 + par * kPageRows;
    float* l_sum = l_sum2 + par * kPageRows;
    const char* page = layer + (int64_t)page_of(jp) * p.k_sp * 2;
    const int64_t obase = rowbase + (int64_t)jp * p.BS;
    const int tix = wave * 64 + lane;
    if (tix < kPageRows) { l_col[tix] = -1; l_corr[tix] = 0ull; }
    if (tix == 0) l_any2[par] = 0;
    ZP_PSTAMP();   // 1

    // ---- norms from the diagonal of the Gram matrix: wave a multiplies its own block (a, a) as
    // soon as its own rows have landed; the 32 lanes that hold a diagonal entry turn it into 1 / norm
    frag_t ak[KSB];
    f32x16_t diag;
#pragma unroll
    for (int r = 0; r < 16; ++r) diag[r] = 0.f;
    if (wave < nrb) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const char* arow = k_pl + a * 8 * kPgGrp + rd_off;
#pragma unroll
      for (int s = 0; s < KSB; ++s) ak[s] = *(const frag_t*)(arow + (s >> 1) * 256 + (s & 1) * 32);
#pragma unroll
      for (int s = 0; s < KSB; ++s) diag = Mfma16<T>::run(ak[s], ak[s], diag);
      // lane (col, half) owns rows (r/4)*8 + half*4 + r%4 of column col: entry (col, col) is its
      // register (col/8)*4 + col%4 when (col%8)/4 == half
      const int my_r = (col >> 3) * 4 + (col & 3);
      float ss = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) ss = r == my_r ? diag[r] : ss;
      const bool mine = ((col & 7) >> 2) == half;
      // the quotient only scales fp32 sums: the 1-ulp reciprocal is exact enough
      const float rn = __builtin_amdgcn_rcpf(fmaxf(Elem<T>::rnd(sqrtf(ss)), epsr));
      float f = rn;
      if constexpr (RnScale<T>::per_block) {
        int e = mine ? (int)((__float_as_uint(rn) >> 23) & 0xffu) : 0;   // biased exponent
        e = half_max_i(e);
        e = max(e, lane_xor32(e));
        const int x = e - 127 - 14;          // rn = f * 2^x, the block's largest f in [2^14, 2^15)
        f = ldexpf(rn, -x);
        if (lane == 0) l_bexp[a] = x;
      }
      if (mine) {
        l_rn[a * 32 + col] = rn;
        l_sum[a * 32 + col] = ss * rn * rn;      // |e_i|^2, taken off the row sum below
        uint16_t o[3];
        Split3<T>::run(f, o);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) *(uint16_t*)(rn_pl + pl * kPageRows * 2 + (a * 32 + col) * 2) = o[pl];
      }
    }
    ZP_PSTAMP();   // 2: norms of wave 0's block
    __syncthreads();
    ZP_PSTAMP();   // 3: page and norms complete

    // ---- summed normalised key S = sum_j rn_j k_j on the matrix cores, by the upper four waves
    // (which have one tile fewer below): wave 7 - t takes the head dims 32 t .. 32 t + 31 and walks
    // the keys sixteen at a time.  A: rows 0..2 = the pieces of rn (lanes col >= 3 read zeros);
    // B: the keys transposed.  The three rows of the result are added smallest first and stored as
    // three 16-bit planes, so that the matrix cores can multiply the keys with S as well.
    if (wave >= kPageWaves - 4) {
      // these four waves carry the key sum on top of their tiles and are what the barrier behind
      // the tiles waits for: they issue ahead of the other waves of the compute unit until then
      __builtin_amdgcn_s_setprio(2);
      const int dt = kPageWaves - 1 - wave;
      f32x16_t acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      const char* asrc = rn_pl + (col < 3 ? col : 3) * kPageRows * 2 + half * 16;
      // transposing read: lane i of a group of sixteen supplies the address of key row i / 4, four
      // dims at (i % 4) * 4 of the group's sixteen dims; groups: (half, dims 16 (g & 1) ..)
      const int i16 = lane & 15, g4 = lane >> 4;
      const char* bsrc = k_pl + (g4 >> 1) * 2 * kPgGrp + dt * 256 + (i16 >> 2) * 64 +
                         ((g4 & 1) * 2 + ((i16 & 3) >> 1)) * 16 + (i16 & 1) * 8;
      // a block of 32 keys is two k-steps; the operands of the next block are requested before the
      // products of this one, so the chain of dependent products does not also wait for LDS
      int xcur = 0;
      frag_t af[2][2];
      s16x4_t bl[2][2], bh[2][2];
      auto fetch = [&](int blk, auto buf) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int ks = 2 * blk + u;
          af[buf.value][u] = *(const frag_t*)(asrc + ks * 32);
          bl[buf.value][u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (s16x4_t __attribute__((address_space(3)))*)(bsrc + ks * 4 * kPgGrp));
          bh[buf.value][u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (s16x4_t __attribute__((address_space(3)))*)(bsrc + (ks * 4 + 1) * kPgGrp));
        }
      };
      auto products = [&](int blk, auto buf) {
        if constexpr (RnScale<T>::per_block) {
          const int xb = l_bexp[blk];
          if (blk > 0) {
#pragma unroll
            for (int r = 0; r < 3; ++r) acc[r] = ldexpf(acc[r], xcur - xb);
          }
          xcur = xb;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const s16x8_t bb = __builtin_shufflevector(bl[buf.value][u], bh[buf.value][u], 0, 1, 2, 3, 4, 5, 6, 7);
          acc = Mfma16<T>::run(af[buf.value][u], __builtin_bit_cast(frag_t, bb), acc);
        }
      };
      typedef std::integral_constant<int, 0> B0;
      typedef std::integral_constant<int, 1> B1;
      fetch(0, B0{});
#pragma unroll 1
      for (int blk = 0; blk < nrb; blk += 2) {
        if (blk + 1 < nrb) fetch(blk + 1, B1{});
        products(blk, B0{});
        if (blk + 1 < nrb) {
          if (blk + 2 < nrb) fetch(blk + 2, B0{});
          products(blk + 1, B1{});
        }
      }
      if (half == 0) {
        float sv = (acc[2] + acc[1]) + acc[0];
        if constexpr (RnScale<T>::per_block) sv = ldexpf(sv, xcur);
        uint16_t o[3];
        Split3<T>::run(sv, o);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) *(uint16_t*)(s_pl + pl * kDmax * 2 + (dt * 32 + col) * 2) = o[pl];
      }
    }
    ZP_PSTAMP();   // 4: (wave 0 has nothing to do for the key sum)

    // ---- Gram tiles: wave a owns row block a and the column blocks (a + d) mod n
    float rn_row[16];
    if (wave < nrb) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {   // the lane's rows come in runs of four
        const float4 v = *(const float4*)(l_rn + a * 32 + q * 8 + half * 4);
        rn_row[4 * q] = v.x; rn_row[4 * q + 1] = v.y; rn_row[4 * q + 2] = v.z; rn_row[4 * q + 3] = v.w;
      }
      // a tile whose largest entry stays below this cannot hold a claim (slack for the rounding of
      // the two ways the scale factors are multiplied in)
      const float thr_lo = p.threshold - fabsf(p.threshold) * 1e-5f - 1e-30f;
      float rn_max = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) rn_max = fmaxf(rn_max, rn_row[r]);
      int dcol[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) dcol[r] = -1;
      const int nd = nrb / 2 + ((nrb & 1) || a < nrb / 2 ? 1 : 0);   // distances 0 .. nd-1
      // what a tile feeds: the last column over the threshold of the keys on both of its sides
      bool dense = false;             // the last tile had claims: the next is likely to, and nothing asks first
      auto scan = [&](const f32x16_t& acc, int cb, bool off_diagonal) {
        const int cslot = cb * 32 + col;
        const float rn_col = l_rn[cslot];
        // most tiles hold no entry over the threshold, and one maximum decides.  With a positive
        // threshold only positive products matter, and those are at most the largest product
        // times the largest row factor: that bound needs no multiplication per entry.
        if (thr_lo > 0.f && !dense) {
          float amax = 0.f;
#pragma unroll
          for (int r = 0; r < 16; ++r) amax = fmaxf(amax, acc[r]);
          if (!__any(amax * rn_max * rn_col > thr_lo)) return;
        }
        if (!dense) {
          float big = -INFINITY;
#pragma unroll
          for (int r = 0; r < 16; ++r) big = fmaxf(big, acc[r] * rn_row[r]);
          if (!__any(big * rn_col > thr_lo)) return;
        }
        // row side: key (a, r) sees column cslot; column side (off the diagonal block, where both
        // (i, j) and (j, i) are computed): key cslot sees the rows of block a, whose index grows
        // with r inside a lane, so the last hit is the largest
        int rlast = -1;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool over = acc[r] * (rn_row[r] * rn_col) > p.threshold;
          dcol[r] = max(dcol[r], over ? cslot : -1);
          rlast = over ? r : rlast;
        }
        dense = __any(rlast >= 0);
        if (off_diagonal && dense) {
          int ci = rlast < 0 ? -1 : a * 32 + (rlast >> 2) * 8 + half * 4 + (rlast & 3);
          ci = max(ci, lane_xor32(ci));
          if (half == 0 && ci >= 0) atomicMax(&l_col[cslot], ci);
        }
      };
      {
        // the diagonal block was multiplied for the norms; a key against itself counts as 0
        f32x16_t acc;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[r] = (r >> 2) * 8 + half * 4 + (r & 3) == col ? 0.f : diag[r];
        scan(acc, a, false);
      }
#pragma unroll 1
      for (int d = 1; d < nd; ++d) {
        const int cb = a + d < nrb ? a + d : a + d - nrb;
        const char* brow = k_pl + cb * 8 * kPgGrp + rd_off;
        f32x16_t acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
        frag_t bk[KSB];
#pragma unroll
        for (int s = 0; s < KSB; ++s) bk[s] = *(const frag_t*)(brow + (s >> 1) * 256 + (s & 1) * 32);
#pragma unroll
        for (int s = 0; s < KSB; ++s) acc = Mfma16<T>::run(ak[s], bk[s], acc);
        scan(acc, cb, true);
      }
      // most waves see no entry over the threshold: then the reduction over the lanes is skipped
      bool mine = false;
#pragma unroll
      for (int r = 0; r < 16; ++r) mine |= dcol[r] >= 0;
      if (__any(mine)) {
        const int r = sixteen_half_max(dcol, lane);
        if (lane == 0) l_any2[par] = 1;
        if ((lane & 16) == 0 && dcol[0] >= 0) atomicMax(&l_col[a * 32 + (r >> 2) * 8 + half * 4 + (r & 3)], dcol[0]);
      }
    }
    ZP_PSTAMP();   // 5: tiles of wave 0
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
    ZP_PSTAMP();   // 6: tiles of all waves, key sum planes

    // ---- value of every key's claimed entry, subtracted from the row it was taken from.  Several
    // keys may claim from one row: the values are added as 2^-32 fixed point with integer atomics,
    // which is exact for a cosine above 2^-8 and does not depend on the order of the additions.
    // Two lanes per key: theirs are the pieces of its row that the tiles were multiplied with, and those of the row it claims
    // from, which is still in LDS, so a wave is done with its 32 keys at once; the sixteen pieces' sums are added as a
    // tree, pieces eight apart first.  With both rows from the cache, four keys at a time: 64 rows of 9 pages whose keys nearly all
    // have a claim 163 us, now 114; without claims 75 either way.
    if (__builtin_amdgcn_readfirstlane(l_any2[par]) != 0) {
      const int key = wave * 32 + col;
      const int cl = wave < nrb ? l_col[key] : -1;
      // cl == key: with a negative threshold the zeroed diagonal entry itself can be the claim; its
      // value is 0, nothing to hand back
      const bool claimed = cl >= 0 && cl != key;
      if (__any(claimed)) {
        const int c = claimed ? cl : key;
        const char* crow = k_pl + (c >> 2) * kPgGrp + (c & 3) * 64 + half * 16;
        float t[KSB];
#pragma unroll
        for (int s = 0; s < KSB; ++s) {
          float ej[8], ec[8];
          Unpack<T>::run(__builtin_bit_cast(vec16, ak[s]), ej);
          Unpack<T>::run(*(const vec16*)(crow + (s >> 1) * 256 + (s & 1) * 32), ec);
          t[s] = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) t[s] = fmaf(ej[e], ec[e], t[s]);
        }
        static_assert(KSB == 8, "sixteen pieces");
        float v = ((t[0] + t[4]) + (t[2] + t[6])) + ((t[1] + t[5]) + (t[3] + t[7]));
        v += lane_xor32(v);
        if (claimed && half == 0) atomicAdd(&l_corr[c], to_fixed32(v * (l_rn[key] * l_rn[c])));
      }
      __syncthreads();
    }
    // ---- nothing below reads the page in LDS: the next page of the row is requested now and
    // lands while this one finishes
    const int nj = next_valid(jp + p.parts);
    if (nj < p.NB) request(nj, wave, lane);

    // ---- row sums without the matrix: sum_{j != i} e_i.e_j = rn_i (k_i . S) - |e_i|^2, the products
    // k_i . S as one more tile whose columns 0..2 are the planes of S (the other lanes read zeros)
    if (wave < nrb) {
      f32x16_t acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      const char* srow = s_pl + (col < 3 ? col : 3) * kDmax * 2 + half * 16;
#pragma unroll
      for (int s = 0; s < KSB; ++s) acc = Mfma16<T>::run(ak[s], *(const frag_t*)(srow + s * 32), acc);
      float t[16];
#pragma unroll
      for (int r = 0; r < 16; ++r)   // lane col 0 adds the lo, mid and hi products (lanes col 2, 1, 0), smallest first
        t[r] = (dpp_row_shl<2>(acc[r]) + dpp_row_shl<1>(acc[r])) + acc[r];
      if (col == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float4* dst = (float4*)(l_sum + a * 32 + q * 8 + half * 4);
          float4 v = *dst;
          v.x = t[4 * q] * rn_row[4 * q] - v.x;
          v.y = t[4 * q + 1] * rn_row[4 * q + 1] - v.y;
          v.z = t[4 * q + 2] * rn_row[4 * q + 2] - v.z;
          v.w = t[4 * q + 3] * rn_row[4 * q + 3] - v.w;
          *dst = v;
        }
      }
    }
    ZP_PSTAMP();   // 7: row sums and claim values of wave 0
    __syncthreads();
    ZP_PSTAMP();   // 8
    if (tix < p.BS) Elem<T>::st(p.r_out, obase + tix, l_sum[tix] - from_fixed32(l_corr[tix]));
#ifdef ZP_PAGE_STAMP
    ZP_PSTAMP();   // 9
    if (tid == 0 && blockIdx.x * p.NB + jp < kPageStampMax) {
      long long* dst = zp_page_stamp_buf + ((int64_t)blockIdx.x * p.NB + jp) * 12;
      for (int i = 0; i < 10; ++i) dst[i] = i < nst ? st_[i] : 0;
      dst[10] = wall0;
      dst[11] = wall_clock64() - wall0;
    }
#endif
    jp = nj;
    par ^= 1;
  }
}
#undef ZP_PSTAMP

// ------------------------------------------------------------------ raw, 16-bit caches
// All-pairs variant over the whole sequence.  Four launches; the claims use the symmetric scheme
// of the page kernel above, with pages in the role of its 32-key blocks:
//   1. raw_prep_kernel: 1 / norm of every key, the sum of the normalised keys of every 16-key
//      chunk; claims start at "none".
//   2. gram_raw_kernel: one workgroup per valid page a; it multiplies page a with the pages
//      (a + d) mod n, d = 0..n/2, so every unordered pair of pages is done once, and records for
//      the keys on both sides the last (logical) column over the threshold with integer
//      atomic maxima (order-independent, so the result is deterministic).
//   3. raw_claim_value_kernel: the fp32 value of every key's claimed entry.
//   4. raw_chain_kernel: the row sums, accumulated chunk by chunk in the cache dtype as the
//      reference does, with the diagonal and the claimed entries taken out of their chunks.
// The softmax kernel then normalises the rows.

// One workgroup per valid page: 1 / norm of every key, claims reset to "none", and the sum of the
// normalised keys of every 16-key chunk of the page (fp32), which is all the row sums need:
//   sum_{j in chunk} e_i . e_j = e_i . (sum_{j in chunk} e_j).
// The reference walks the columns in chunks of 16 (BLOCK_N, raw_redudancy_score.py:176) and
// rounds after each chunk, so the chunk is the unit whose sum has to be exact.
template <typename T>
__global__ __launch_bounds__(kThreads) void raw_prep_kernel(GramArgs p) {
  static_assert(T::bytes == 2, "16-bit caches only");
  constexpr int PIECES = kDmax / 8, GROUPS = kThreads / PIECES;   // 16 groups of 16 lanes
  const int tid = threadIdx.x;
  const int piece = tid % PIECES, g = tid / PIECES;
  const int jp = blockIdx.x % p.NB;
  const int h = (blockIdx.x / p.NB) % p.Hkv;
  const int b = (blockIdx.x / (p.NB * p.Hkv)) % p.B;
  const int l = blockIdx.x / (p.NB * p.Hkv * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t obase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn + (int64_t)jp * p.BS;
  const float epsr = Elem<T>::rnd(p.eps);
  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) return;
  const bool pok = piece < p.D / 8;
  const int64_t k_row = (int64_t)p.Hkv * p.D * 2;
  const char* kbase = p.k + (l * p.k_sl + (int64_t)rpid * p.k_sp) * 2 + (int64_t)h * p.D * 2 +
                      (pok ? piece : 0) * 16;
  const int cpp = p.BS / kChunk;                       // chunks per page
  float* csum = p.ws_chunk + (obase / kChunk) * kDmax;  // [chunk][kDmax] of this page
  for (int c = g; c < cpp; c += GROUPS) {
    u32x4 raw[kChunk];
#pragma unroll
    for (int u = 0; u < kChunk; ++u)
      raw[u] = *(const u32x4*)(kbase + (int64_t)(c * kChunk + u) * k_row);
    float cs[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) cs[q] = 0.f;
#pragma unroll
    for (int u = 0; u < kChunk; ++u) {
      if (!pok) raw[u] = u32x4{0u, 0u, 0u, 0u};
      float e[8];
      Unpack<T>::run(vec16{raw[u].x, raw[u].y, raw[u].z, raw[u].w}, e);
      float ss = 0.f;
#pragma unroll
      for (int q = 0; q < 8; ++q) ss = fmaf(e[q], e[q], ss);
      ss = pieces_sum<PIECES>(ss);
      const float rn = __builtin_amdgcn_rcpf(fmaxf(Elem<T>::rnd(sqrtf(ss)), epsr));
#pragma unroll
      for (int q = 0; q < 8; ++q) cs[q] = fmaf(e[q], rn, cs[q]);
      if (piece == 0) {
        const int64_t oi = obase + c * kChunk + u;
        p.ws_sum[oi] = rn;      // kept for the row-sum kernel
        p.ws_val[oi] = rn;      // read by the Gram kernel, replaced by the claim values after it
        p.ws_col[oi] = -1;
      }
    }
    float* dst = csum + (int64_t)c * kDmax + piece * 8;
    *(float4*)dst = make_float4(cs[0], cs[1], cs[2], cs[3]);
    *(float4*)(dst + 4) = make_float4(cs[4], cs[5], cs[6], cs[7]);
  }
}

// Four waves per SIMD, i.e. two workgroups per compute unit (their LDS fits twice): one's barrier
// and LDS waits hide behind the other's tiles.  The register cap spills a few addresses outside
// the tile loop; measured 10-15 % faster than one workgroup per unit.
template <typename T, int TNc>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4)))
void gram_raw_kernel(GramArgs p) {
  static_assert(T::bytes == 2, "16-bit caches only");
  typedef typename Mfma16<T>::V frag_t;
  constexpr int kThreads = 512, kWaves = 8;
  constexpr int PIECES = kDmax / 8;
  constexpr int ROWS_PER_IT = kThreads / PIECES;    // 32
  constexpr int STAGE_IT = TNc / ROWS_PER_IT;
  constexpr int NSUB = TNc / 32;
  constexpr int KSB = kDmax / 16;
  constexpr int PLANE = TNc * ROWH;

  extern __shared__ __align__(16) char smem[];
  char* buf0 = smem;                                // raw keys of a column tile
  char* buf1 = smem + PLANE;
  float* l_rn = (float*)(smem + 2 * PLANE);         // [2][TNc] 1 / norm of the tile's keys
  int* l_cside = (int*)(l_rn + 2 * TNc);            // [2][TNc] column-side claims of a tile
  float* l_rnrow = (float*)(l_cside + 2 * TNc);     // [BS] 1 / norm of the row page's keys
  int* vpage = (int*)(l_rnrow + p.BS);
  int* vidx = vpage + p.NB;
  __shared__ int nvalid_s, mine_s;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int jp = blockIdx.x % p.NB;
  const int h = (blockIdx.x / p.NB) % p.Hkv;
  const int b = (blockIdx.x / (p.NB * p.Hkv)) % p.B;
  const int l = blockIdx.x / (p.NB * p.Hkv * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t obase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;

  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) return;
  list_valid_pages(p.table + (int64_t)b * p.NB, p.NB, p.num_pages, jp, vpage, vidx, nullptr, &nvalid_s, &mine_s);
  // head dims below 128 leave the upper pieces of every LDS row at zero
  for (int i = tid; i < 2 * PLANE / 4; i += kThreads) ((uint32_t*)smem)[i] = 0u;
  if (tid < 2 * TNc) l_cside[tid] = -1;
  for (int i = tid; i < p.BS; i += kThreads) l_rnrow[i] = p.ws_val[obase + (int64_t)jp * p.BS + i];
  __syncthreads();
  const int nv = nvalid_s, ia = mine_s;
  const int nd = nv / 2 + (((nv & 1) || ia < nv / 2) ? 1 : 0);   // page distances 0 .. nd-1
  const int tiles_per_page = p.BS / TNc;
  const int ntiles = nd * tiles_per_page;
  const int dpieces = p.D / 8;
  const int64_t k_row = (int64_t)p.Hkv * p.D * 2;
  const char* kbase = p.k + (l * p.k_sl) * 2 + (int64_t)h * p.D * 2;
  const float* rn_all = p.ws_val + obase;           // written by raw_prep_kernel

  const int st_piece = tid % PIECES, st_row0 = tid / PIECES;
  const bool st_ok = st_piece < dpieces;
  u32x4 pre[STAGE_IT];
  float pre_rn = 0.f;
  auto tile_page = [&](int tile, int& d, int& toff) {
    d = tile / tiles_per_page;
    toff = (tile - d * tiles_per_page) * TNc;
    const int ic = ia + d;
    return ic < nv ? ic : ic - nv;
  };
  auto issue_loads = [&](int tile) {
    int d, toff;
    const int ic = tile_page(tile, d, toff);
    const char* src = kbase + (int64_t)vpage[ic] * p.k_sp * 2 + (int64_t)toff * k_row +
                      (st_ok ? st_piece : 0) * 16;
#pragma unroll
    for (int i = 0; i < STAGE_IT; ++i)
      pre[i] = *(const u32x4*)(src + (int64_t)(st_row0 + i * ROWS_PER_IT) * k_row);
    if (tid < TNc) pre_rn = rn_all[vidx[ic] * p.BS + toff + tid];
  };
  auto commit_loads = [&](char* buf, int tile) {
    if (st_ok) {
#pragma unroll
      for (int i = 0; i < STAGE_IT; ++i)
        *(u32x4*)(buf + (st_row0 + i * ROWS_PER_IT) * ROWH + st_piece * 16) = pre[i];
    }
    if (tid < TNc) l_rn[(tile & 1) * TNc + tid] = pre_rn;
  };
  // Hands the column-side claims of a finished tile to the keys of its page and clears the slot.
  auto flush_cside = [&](int tile) {
    if (tid < TNc) {
      int d, toff;
      const int ic = tile_page(tile, d, toff);
      int* slot = l_cside + (tile & 1) * TNc + tid;
      const int v = *slot;
      if (v >= 0) {
        atomicMax(p.ws_col + obase + (int64_t)vidx[ic] * p.BS + toff + tid, v);
        *slot = -1;
      }
    }
  };
  const float thr_lo = p.threshold - fabsf(p.threshold) * 1e-5f - 1e-30f;

  const int row_blocks = p.BS / 32;
  const int NR = (row_blocks + kWaves - 1) / kWaves;
  for (int rr = 0; rr < NR; ++rr) {
    const int rb = rr * kWaves + wave;
    const bool active = rb < row_blocks;
    // ---- A fragments: this lane's key row as stored; lane (row, half) holds k = 16 s + 8 half + i
    frag_t ak[KSB];
    const float* rsrc = l_rnrow + (active ? rb : 0) * 32 + half * 4;   // this lane's 16 rows: 1 / norm
    {
      const int slot = (active ? rb : 0) * 32 + col;
      const char* src = kbase + (int64_t)rpid * p.k_sp * 2 + (int64_t)slot * k_row;
#pragma unroll
      for (int s = 0; s < KSB; ++s) {
        const int pc = 2 * s + half;
        u32x4 v = u32x4{0u, 0u, 0u, 0u};
        if (pc < dpieces) v = *(const u32x4*)(src + pc * 16);
        ak[s] = __builtin_bit_cast(frag_t, v);
      }
    }
    int dcol[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) dcol[r] = -1;

    if (ntiles > 0) { issue_loads(0); commit_loads(buf0, 0); }
    __syncthreads();
    for (int tile = 0; tile < ntiles; ++tile) {
      char* cur = (tile & 1) ? buf1 : buf0;
      char* nxt = (tile & 1) ? buf0 : buf1;
      if (tile + 1 < ntiles) issue_loads(tile + 1);
      if (tile > 0) flush_cside(tile - 1);   // its slot is next written two tiles from now
      int d, toff;
      const int ic = tile_page(tile, d, toff);
      const int jc = vidx[ic];
      if (active) {
#pragma unroll 1
        for (int st = 0; st < NSUB; ++st) {
          f32x16_t acc;
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] = 0.f;
          const char* brow = cur + (st * 32 + col) * ROWH + half * 16;
          const float rn_col = l_rn[(tile & 1) * TNc + st * 32 + col];
#pragma unroll
          for (int s0 = 0; s0 < KSB; s0 += 4) {
            frag_t bk[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) bk[s] = *(const frag_t*)(brow + (s0 + s) * 32);
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = Mfma16<T>::run(ak[s0 + s], bk[s], acc);
          }
          float rn_row[16];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4 v = *(const float4*)(rsrc + g * 8);
            rn_row[4 * g] = v.x; rn_row[4 * g + 1] = v.y; rn_row[4 * g + 2] = v.z; rn_row[4 * g + 3] = v.w;
          }
          const int cslot = toff + st * 32 + col;
          const int cidx = jc * p.BS + cslot;
          if (d == 0) {
            // the page against itself: a key against itself counts as 0
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3) == cslot) acc[r] = 0.f;
          }
          // most tiles hold no entry over the threshold: one maximum decides
          float big = -INFINITY;
#pragma unroll
          for (int r = 0; r < 16; ++r) big = fmaxf(big, acc[r] * rn_row[r]);
          if (!__any(big * rn_col > thr_lo)) continue;
          // row side: key (rb, r) sees column cidx; column side (other pages only: inside a
          // page both (i, j) and (j, i) are computed): key cidx sees the rows of this block,
          // whose index grows with r inside a lane
          int rlast = -1;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool over = acc[r] * (rn_row[r] * rn_col) > p.threshold;
            dcol[r] = max(dcol[r], over ? cidx : -1);
            rlast = over ? r : rlast;
          }
          if (d != 0 && __any(rlast >= 0)) {
            int ci = rlast < 0 ? -1
                               : jp * p.BS + rb * 32 + (rlast >> 2) * 8 + half * 4 + (rlast & 3);
            ci = max(ci, lane_xor32(ci));
            if (half == 0 && ci >= 0) atomicMax(&l_cside[(tile & 1) * TNc + st * 32 + col], ci);
          }
        }
      }
      if (tile + 1 < ntiles) commit_loads(nxt, tile + 1);
      __syncthreads();
    }
    if (ntiles > 0) flush_cside(ntiles - 1);
    bool any_mine = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) any_mine |= dcol[r] >= 0;
    if (__any(any_mine)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = half_max_i(dcol[r]);
        if (active && col == 0 && c >= 0)
          atomicMax(p.ws_col + obase + (int64_t)jp * p.BS + rb * 32 + (r >> 2) * 8 + half * 4 + (r & 3), c);
      }
    }
    __syncthreads();   // the claim slots are clear again before the next round writes them
  }
}

// Pages of a row, whose keys and chunk sums each of them reads, on one XCD, one after the other.
__device__ __forceinline__ unsigned row_of_page(unsigned id, unsigned pages, unsigned NB, int& jp) {
  const unsigned rows = pages / NB;
  if (rows % 8 != 0) { jp = id % NB; return id / NB; }
  jp = (id >> 3) % NB;
  return (id >> 3) / NB * 8 + (id & 7);
}

// The same for pages that are whole 128-key tiles, built like the page kernel of the lightning
// variant: four waves, each with TWO row blocks of the row page in registers (64 rows), so a B
// fragment read from LDS feeds two products; the column tiles go from global memory straight into
// LDS (wave w requests rows 32 w .. 32 w + 31 of a tile, the layout of `gram_page_kernel`), two
// buffers, one barrier per tile, the request for tile t + 1 beside the products of tile t, a load at a
// time.  Two workgroups per compute unit (two waves per SIMD, 256 registers each).  PARTS: a workgroup has some of
// a page's tiles (see tile_parts); where it has all, first and last tile are known, which is 2 to 3 % of the kernel.
// Of 7200 cycles a tile (two workgroups on a CU) its products take 2048; the rest is the other workgroup's products, the look at
// the largest ones, and 1800 of waits, barriers and claims.  48 sequences of 2049 to 2560 tokens, 8 heads: 395 -> 343 us, 378 -> 328
// without claims; 23 of two layers whose keys are copies of one another 361 -> 337; 2 sequences 23.4 -> 21.0.  A page's own rows
// come in whole lines with its first tiles and the claims of a block and its transpose are worked out once; requests one by one,
// fragments of the next columns before the look at these, no division per tile: request and claims 10 900 -> 5200 cycles a page,
// products 63 800 -> 51 500.  Rows on one XCD halve what L2 misses, at no change in time.  Tried: the products of two column blocks
// in turns, with the maxima of one beside the other's (registers for the row factors go, 357 and 337); claims by ballots and LDS
// atomics (680 against 507 where half of the keys have copies).
constexpr int kRawTile = 128;
constexpr int kRawTileBytes = (kRawTile / 4) * kPgGrp;
template <typename T, bool PARTS>
__global__ __launch_bounds__(256, 2) void gram_raw_wide_kernel(GramArgs p) {
  static_assert(T::bytes == 2, "16-bit caches only");
  typedef typename Mfma16<T>::V frag_t;
  constexpr int kThreads = 256, kWaves = 4, TNc = kRawTile;
  constexpr int PIECES = kDmax / 8;
  constexpr int NSUB = TNc / 32;
  constexpr int KSB = kDmax / 16;

  extern __shared__ __align__(16) char smem[];
  char* buf0 = smem;                                // raw keys of a column tile
  char* buf1 = smem + kRawTileBytes;
  float* l_rn = (float*)(smem + 2 * kRawTileBytes); // [2][TNc] 1 / norm of the tile's keys
  int* l_cside = (int*)(l_rn + 2 * TNc);            // [2][TNc] column-side claims of a tile
  float* l_rnrow = (float*)(l_cside + 2 * TNc);     // [BS] 1 / norm of the row page's keys
  int* vpage = (int*)(l_rnrow + p.BS);
  int* vidx = vpage + p.NB;
  __shared__ int nvalid_s, mine_s;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, col = lane & 31;
  const unsigned pages = PARTS ? gridDim.x / p.parts : gridDim.x;
  const int part = PARTS ? blockIdx.x / pages : 0;
  int jp;
  const unsigned row = row_of_page(PARTS ? blockIdx.x % pages : blockIdx.x, pages, p.NB, jp);
  const int h = row % p.Hkv;
  const int b = row / p.Hkv % p.B;
  const int l = row / p.Hkv / p.B;
  const int Tn = p.NB * p.BS;
  const int64_t obase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;

  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) return;
  const int dpieces = p.D / 8;
  const int k_row = p.Hkv * p.D * 2;
  const char* kbase = p.k + (l * p.k_sl) * 2 + (int64_t)h * p.D * 2;
  // rows of a page -> LDS, a wave 32 of a tile: eight instructions of four rows; past the end of a head's rows come zeros
  const int st_g = (lane >> 4) * 4 + (lane & 3), st_r = (lane >> 2) & 3;
  const int st_voff = st_g < dpieces ? st_r * k_row + st_g * 16 : 0x40000000;
  auto rows_of = [&](int pid, int toff) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(kbase + (int64_t)pid * p.k_sp * 2 + (int64_t)(toff + wave * 32) * k_row), 0, 32 * k_row, 0x00020000);
  };
  auto stage = [&](const __amdgpu_buffer_rsrc_t& rs, char* buf, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(buf + (wave * 8 + i) * kPgGrp), 16, st_voff, i * 4 * k_row, 0, 0);
  };
  auto stage_all = [&](const __amdgpu_buffer_rsrc_t& rs, char* buf) {
#pragma unroll
    for (int i = 0; i < 8; ++i) stage(rs, buf, i);
  };
  // A page of at most two tiles is its own first ones: its rows are asked for before anything else.
  const int tiles_per_page = p.BS / TNc;
  const bool own = part == 0 && tiles_per_page <= 2;
  if (own) {
    stage_all(rows_of(rpid, 0), buf0);
    if (tiles_per_page == 2) stage_all(rows_of(rpid, TNc), buf1);
  }
  list_valid_pages(p.table + (int64_t)b * p.NB, p.NB, p.num_pages, jp, vpage, vidx, nullptr, &nvalid_s, &mine_s);
  if (tid < 2 * TNc) l_cside[tid] = -1;
  for (int i = tid; i < p.BS; i += kThreads) l_rnrow[i] = p.ws_val[obase + (int64_t)jp * p.BS + i];
  __syncthreads();
  const int nv = nvalid_s, ia = mine_s;
  const int nd = nv / 2 + (((nv & 1) || ia < nv / 2) ? 1 : 0);   // page distances 0 .. nd-1
  const int from = PARTS ? nd * tiles_per_page * part / p.parts : 0;                       // its tiles
  const int to = PARTS ? nd * tiles_per_page * (part + 1) / p.parts : nd * tiles_per_page;
  const float* rn_all = p.ws_val + obase;           // written by raw_prep_kernel
  float pre_rn = 0.f;                               // of the next tile's key `tid`
  // Hands the column-side claims of a finished tile to the keys of its page and clears the slot.
  auto flush_cside = [&](int tile, int64_t at) {
    if (tid < TNc) {
      int* slot = l_cside + (tile & 1) * TNc + tid;
      const int v = *slot;
      if (v >= 0) {
        atomicMax(p.ws_col + at + tid, v);
        *slot = -1;
      }
    }
  };
  const float thr_lo = p.threshold - fabsf(p.threshold) * 1e-5f - 1e-30f;
  const bool bounded = p.threshold > 0.f;           // the largest product of a tile bounds its entries
  // fragment of k-step s of this lane's row of a 32-row block: base + (s / 2) * 256 + (s % 2) * 32
  const int rd_off = (col >> 2) * kPgGrp + (col & 3) * 64 + half * 16;

  const int row_blocks = p.BS / 32;
  const int NR = (row_blocks + 2 * kWaves - 1) / (2 * kWaves);
  for (int rr = 0; rr < NR; ++rr) {
    const int rb0 = (rr * kWaves + wave) * 2;          // this wave's two row blocks: rb0, rb0 + 1
    const bool act = rb0 < row_blocks;
    int d = from / tiles_per_page, toff = (from - d * tiles_per_page) * TNc, ic = ia + d < nv ? ia + d : ia + d - nv;
    int64_t before_at = 0;                             // the keys of the tile before
    int there = own && rr == 0 ? tiles_per_page : from;          // tiles that were asked for
    if (there == from && from < to) {
      stage_all(rows_of(__builtin_amdgcn_readfirstlane(vpage[ic]), toff), from & 1 ? buf1 : buf0);
      if (tid < TNc) pre_rn = rn_all[vidx[ic] * p.BS + toff + tid];
      ++there;
    }
    // ---- A fragments: this lane's two key rows as stored; lane (row, half) holds k = 16 s + 8 half + i.  Rows in LDS were asked
    // for in whole lines
    frag_t ak[2][KSB];
    if (own) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int s = 0; s < KSB; ++s)
          ak[g][s] = *(const frag_t*)(smem + (act ? rb0 + g : 0) * 8 * kPgGrp + rd_off + (s >> 1) * 256 + (s & 1) * 32);
    } else {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const char* src = kbase + (int64_t)rpid * p.k_sp * 2 + (int64_t)((act ? rb0 + g : 0) * 32 + col) * k_row;
#pragma unroll
        for (int s = 0; s < KSB; ++s) {
          const int pc = 2 * s + half;
          u32x4 v = u32x4{0u, 0u, 0u, 0u};
          if (pc < dpieces) v = *(const u32x4*)(src + pc * 16);
          ak[g][s] = __builtin_bit_cast(frag_t, v);
        }
      }
    }
    float rn_row[2][16], rn_most[2];                   // of the rows whose products this lane has
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      rn_most[g] = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 v = *(const float4*)(l_rnrow + (act ? rb0 + g : 0) * 32 + half * 4 + q * 8);
        rn_row[g][4 * q] = v.x, rn_row[g][4 * q + 1] = v.y, rn_row[g][4 * q + 2] = v.z, rn_row[g][4 * q + 3] = v.w;
        rn_most[g] = fmaxf(rn_most[g], fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
      }
    }

    int dcol[2][16];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int r = 0; r < 16; ++r) dcol[g][r] = -1;
    for (int tile = from; tile < to; ++tile) {
      char* const cur = (tile & 1) ? buf1 : buf0;
      char* const nxt = (tile & 1) ? buf0 : buf1;
      const int jc = vidx[ic];
      int toff1 = toff + TNc, d1 = d, ic1 = ic;        // the next one
      if (toff1 == p.BS) toff1 = 0, ++d1, ic1 = ic + 1 < nv ? ic + 1 : 0;
      const int next_pid = __builtin_amdgcn_readfirstlane(vpage[ic1]), next_idx = vidx[ic1];
      // this wave's share of the tile (and its A fragments, the first time) has landed; after the
      // barrier so has everybody's, and everybody is done with the tile before
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (tid < TNc) l_rn[(tile & 1) * TNc + tid] = d == 0 ? l_rnrow[toff + tid] : pre_rn;
      __syncthreads();
      const bool ask = there < to && there == tile + 1;
      const __amdgpu_buffer_rsrc_t next = rows_of(next_pid, toff1);
      if (ask) {
        if (tid < TNc) pre_rn = rn_all[next_idx * p.BS + toff1 + tid];
        ++there;
      }
      if (tile > from) flush_cside(tile - 1, before_at);   // its slot is next written two tiles from now
      before_at = obase + (int64_t)jc * p.BS + toff;
      const int tile_d = d, tile_off = toff;
      d = d1, toff = toff1, ic = ic1;
      // blocks of columns that lie below both row blocks' diagonals have been seen
      const int first = !act ? NSUB : tile_d == 0 ? min(max(rb0 - (tile_off >> 5), 0), NSUB) : 0;
      const bool beside = ask && first == 0;           // loads one by one beside the products: eight in a row hold a wave
      if (ask && !beside) stage_all(next, nxt);
      if (first == NSUB) continue;
      // What a tile of 32 x 32 products feeds: the last column over the threshold of its rows and the last row over the
      // threshold of its columns.  Inside a page blocks below the diagonal are the transposes of those above it.
      auto claims = [&](f32x16_t& acc, int g, int st, float rn_col) {
        const int rb = rb0 + g, cb = (tile_off >> 5) + st;
        if (tile_d == 0 && cb <= rb) {
          if (cb < rb) return;
          // the page against itself: a key against itself counts as 0
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if ((r >> 2) * 8 + half * 4 + (r & 3) == col) acc[r] = 0.f;
        }
        const int cidx = jc * p.BS + tile_off + st * 32 + col;
        int rlast = -1;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool over = acc[r] * (rn_row[g][r] * rn_col) > p.threshold;
          dcol[g][r] = max(dcol[g][r], over ? cidx : -1);
          rlast = over ? r : rlast;
        }
        if ((tile_d != 0 || cb != rb) && __any(rlast >= 0)) {
          int ci = rlast < 0 ? -1 : jp * p.BS + rb * 32 + (rlast >> 2) * 8 + half * 4 + (rlast & 3);
          ci = max(ci, lane_xor32(ci));
          if (half == 0 && ci >= 0) atomicMax(&l_cside[(tile & 1) * TNc + st * 32 + col], ci);
        }
      };
      // Two row blocks against 32 columns at a time.  Fragments leave LDS kAhead ahead of their products, those of the next
      // columns too.  Most tiles hold no entry over the threshold: their largest product, as integers, which order what is
      // positive, and the largest row factor decide.  From zero on: 48 sequences whose pages point away from one another, all products
      // of most lanes negative, 604 us with all bits set for none, which is no number and lets everything through, now 540 (random keys 470).
      constexpr int kAhead = 3, kRing = 4;
      static_assert(KSB % kRing == 0, "places of the ring are constants");
      frag_t bk[kRing];
      const char* brow = cur + first * 8 * kPgGrp + rd_off;
      auto fragment = [&](int s) { bk[s % kRing] = *(const frag_t*)(brow + (s >> 1) * 256 + (s & 1) * 32); };
#pragma unroll
      for (int s = 0; s < kAhead; ++s) fragment(s);
#pragma unroll 1
      for (int st = first; st < NSUB; ++st) {
        const float rn_col = l_rn[(tile & 1) * TNc + st * 32 + col];
        f32x16_t acc[2];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[g][r] = 0.f;
#pragma unroll
        for (int s = 0; s < KSB; ++s) {
          if (s + kAhead == KSB && st + 1 < NSUB) brow += 8 * kPgGrp;      // behind the last columns they come again
          fragment((s + kAhead) % KSB);
#pragma unroll
          for (int g = 0; g < 2; ++g) acc[g] = Mfma16<T>::run(ak[g][s], bk[s % kRing], acc[g]);
          if (beside && (s == 2 || s == 5)) stage(next, nxt, 2 * st + (s == 5));
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          int big = 0;
#pragma unroll
          for (int r = 0; r < 16; ++r) big = max(big, __float_as_int(acc[g][r]));
          if (!bounded || __any(!(__int_as_float(big) * rn_most[g] * rn_col <= thr_lo))) claims(acc[g], g, st, rn_col);
        }
      }
    }
    __syncthreads();   // everybody is done with the last tile
    if (from < to) flush_cside(to - 1, before_at);
    bool any_mine = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) any_mine |= dcol[0][r] >= 0 || dcol[1][r] >= 0;
    if (__any(any_mine)) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = half_max_i(dcol[g][r]);
          const int64_t at = obase + (int64_t)jp * p.BS + (rb0 + g) * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
          if (act && col == 0 && c >= 0) atomicMax(p.ws_col + at, c);
        }
    }
    __syncthreads();   // the claim slots are clear again before the next round writes them
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void raw_claim_value_kernel(GramArgs p) {
  static_assert(T::bytes == 2, "16-bit caches only");
  constexpr int PIECES = kDmax / 8, GROUPS = kThreads / PIECES;
  const int tid = threadIdx.x;
  const int piece = tid % PIECES, g = tid / PIECES;
  const unsigned pages = gridDim.x / p.parts, page = blockIdx.x % pages, part = blockIdx.x / pages;
  const int jp = page % p.NB;
  const int h = (page / p.NB) % p.Hkv;
  const int b = (page / (p.NB * p.Hkv)) % p.B;
  const int l = page / (p.NB * p.Hkv * p.B);
  const int Tn = p.NB * p.BS;
  const int64_t obase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;
  const float epsr = Elem<T>::rnd(p.eps);
  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) return;
  const bool pok = piece < p.D / 8;
  const int64_t k_row = (int64_t)p.Hkv * p.D * 2;
  const char* kbase = p.k + (l * p.k_sl) * 2 + (int64_t)h * p.D * 2 + (pok ? piece : 0) * 16;
  // The claims of all keys are asked for at once; one after the other, each waits for memory, and where there are none that is all there
  // is to do (2880 pages without claims 12.3 us, now 6.6; with claims of half of the keys 60 and 59).
  __shared__ int l_claim[kThreads];
  for (int s0 = 0; s0 < p.BS; s0 += kThreads) {
    const int n = min(kThreads, p.BS - s0), mine = tid < n ? p.ws_col[obase + (int64_t)jp * p.BS + s0 + tid] : -1;
    if (s0 > 0) __syncthreads();
    l_claim[tid] = mine;
    if (!__syncthreads_or(mine >= 0)) continue;
    for (int i = part * GROUPS + g; i < n; i += GROUPS * p.parts) {
      const int slot = s0 + i, c = l_claim[i];
      const int64_t oi = obase + (int64_t)jp * p.BS + slot;
      if (c < 0 || c >= Tn) continue;     // uniform over the 16 lanes of a key
      if (c == jp * p.BS + slot) {        // negative threshold: the zeroed diagonal entry was claimed
        if (piece == 0) p.ws_val[oi] = 0.f;
        continue;
      }
      const int cp = c / p.BS, cs = c - cp * p.BS;
      const int ccode = p.table[(int64_t)b * p.NB + cp];
      const int cpid = page_is_pad(ccode) ? -1 : page_id(ccode);
      if (cpid < 0 || cpid >= p.num_pages) continue;
      u32x4 ra = *(const u32x4*)(kbase + (int64_t)rpid * p.k_sp * 2 + (int64_t)slot * k_row);
      u32x4 rc = *(const u32x4*)(kbase + (int64_t)cpid * p.k_sp * 2 + (int64_t)cs * k_row);
      if (!pok) { ra = u32x4{0u, 0u, 0u, 0u}; rc = ra; }
      float ea[8], ec[8];
      Unpack<T>::run(vec16{ra.x, ra.y, ra.z, ra.w}, ea);
      Unpack<T>::run(vec16{rc.x, rc.y, rc.z, rc.w}, ec);
      float sa = 0.f, sc = 0.f, t = 0.f;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        sa = fmaf(ea[q], ea[q], sa);
        sc = fmaf(ec[q], ec[q], sc);
        t = fmaf(ea[q], ec[q], t);
      }
      sa = pieces_sum<PIECES>(sa);
      sc = pieces_sum<PIECES>(sc);
      t = pieces_sum<PIECES>(t);
      const float rna = __builtin_amdgcn_rcpf(fmaxf(Elem<T>::rnd(sqrtf(sa)), epsr));
      const float rnc = __builtin_amdgcn_rcpf(fmaxf(Elem<T>::rnd(sqrtf(sc)), epsr));
      if (piece == 0) p.ws_val[oi] = t * rna * rnc;
    }
  }
}

// ------------------------------------------------------------------ raw, 16-bit: row sums
// The reference accumulates a key's row sum in the CACHE dtype: per column page one partial sum,
// rounded after each 16-column chunk (raw_redudancy_score.py:146-155: load, add the chunk's fp32
// sum, store in the cache dtype), then the partial sums of the pages are added in fp32 and rounded
// once (:218, torch.sum).  This kernel restates that chain exactly.
//   chunk sum   c(i, chunk) = rn_i (k_i . s_chunk) - [i in chunk] S_ii - sum_{j in chunk, claimed by i} S_ij
// with s_chunk the sum of the chunk's normalised keys from raw_prep_kernel.  The dot products of
// a page's 256 keys with 32 chunks at a time run on the matrix cores: the keys as stored (exact
// 16-bit products), s_chunk split into three 16-bit planes (together its full fp32 mantissa).
// One workgroup per valid page.  A wave has 64 keys as the columns of two products, so a fragment of the planes read from LDS
// feeds both (with 32, LDS was as busy as the matrix cores), and one exchange between its halves leaves every lane with one
// key's 32 chunk sums in order: the chain runs in registers, on all lanes.  What it replaces went through LDS, half of the
// threads walked the chain of a tile behind a barrier, and the claims of a row went through a list.  48 sequences of 2049 to 2560
// tokens, 8 heads: 274 -> 183 us; 2 of them 26.5 -> 17.7.  Bound by what a page does one after the other: of 42 000 cycles (two
// workgroups on a CU) the table, the keys and the first planes take 16 000, the products 12 000 (7100 of them the matrix
// cores'), splitting and corrections 9000.
// chunk sums are below 16 + 1 in magnitude: 2^-26 fixed point fits 32 bits, and integer atomics
// make the sum of several claims independent of their order
// Chunks that raw_chain_kernel takes at a time; words of a key's corrections, 16 bytes of neighbours in different banks; bytes of
// LDS: a round's 256 keys, and then planes and corrections.
constexpr int kChainTile = 32, kChainLd = kChainTile + 4;
constexpr int kChainBytes = 256 / 4 * kPgGrp;
// Tokens and pages of a row that 16-bit caches take.  A limit of the interface: the claims of a row once lay in the LDS, now a row's pages and
// chunks do, a twentieth of it here, and longer rows are not tested.
constexpr int kMostRawTokens = 13120;
static_assert(3 * kChainTile * ROWH + 256 * kChainLd * 4 <= kChainBytes, "planes and corrections fit where the keys were");
__device__ __forceinline__ int to_fixed26(float v) { return (int)(v * 67108864.f); }
__device__ __forceinline__ float from_fixed26(int w) { return (float)w * (1.f / 67108864.f); }

#ifdef ZP_PAGE_STAMP
__device__ long long zp_chain_stamp_buf[(1 << 16) * 12];
extern "C" int zp_debug_chain_stamps(long long* dst, int n_groups) {
  return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(zp_chain_stamp_buf), (size_t)n_groups * 12 * 8);
}
#define ZP_CSTAMP(i) do { if (tid == 0) { const long long c_ = clock64(); acc_[i] += c_ - last_; last_ = c_; } } while (0)
#else
#define ZP_CSTAMP(i) do { } while (0)
#endif

template <typename T>
__global__ __launch_bounds__(256, 2) void raw_chain_kernel(GramArgs p) {
  static_assert(T::bytes == 2, "16-bit caches only");
  typedef typename Mfma16<T>::V frag_t;
  constexpr int kT = 256, KSB = kDmax / 16, CT = kChainTile;     // CT chunks per tile
  constexpr int KEYS = kT;                                          // keys per round
  extern __shared__ __align__(16) char smem[];
  char* planes = smem;                                   // [3][CT] rows of ROWH bytes
  int* cl = (int*)(smem + 3 * CT * ROWH);                // [KEYS][kChainLd] corrections
  int* vidx = (int*)(smem + kChainBytes);                // [NB] logical page of the n-th valid page
  int* chunk_of = vidx + p.NB;                           // [NB * BS / 16] logical chunk of the n-th one of the valid pages
  __shared__ int nvalid_s, mine_s, corrected[2];         // corrected: whether a tile has any

  const int tid = threadIdx.x, lane = tid & 63;
  const int half = lane >> 5, col = lane & 31;
#ifdef ZP_PAGE_STAMP
  long long acc_[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  long long last_ = clock64();
  const long long wall0 = wall_clock64();
#endif
  int jp;
  const unsigned row = row_of_page(blockIdx.x, gridDim.x, p.NB, jp);
  const int h = row % p.Hkv;
  const int b = row / p.Hkv % p.B;
  const int l = row / p.Hkv / p.B;
  const int Tn = p.NB * p.BS;
  const int64_t obase = (((int64_t)l * p.B + b) * p.Hkv + h) * Tn;

  const int code = p.table[(int64_t)b * p.NB + jp];
  int rpid = page_is_pad(code) ? -1 : page_id(code);
  if (rpid >= p.num_pages) rpid = -1;
  if (rpid < 0) {
    for (int s = tid; s < p.BS; s += kT) Elem<T>::st(p.r_out, obase + (int64_t)jp * p.BS + s, -INFINITY);
    return;
  }
  const int cpp = p.BS / kChunk;
  const int dpieces = p.D / 8;
  const int k_row = p.Hkv * p.D * 2;
  const char* kpage = p.k + (l * p.k_sl + (int64_t)rpid * p.k_sp) * 2 + (int64_t)h * p.D * 2;
  const float* chunk_all = p.ws_chunk + (obase / kChunk) * kDmax;
  // ---- the wave's 64 keys in whole lines into LDS, where planes and corrections will lie: rows of 256 bytes asked for as
  // operands touch each line four times, which takes three times as long
  const int st_g = (lane >> 4) * 4 + (lane & 3), st_r = (lane >> 2) & 3;
  char* const keys = smem + (tid >> 6) * 16 * kPgGrp;
  auto stage_keys = [&](int first) {
    const int left = p.BS - first;
    if (left <= 0 || st_g >= dpieces) return;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(kpage + (int64_t)first * k_row), 0, min(left, 64) * k_row, 0x00020000);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(keys + i * kPgGrp), 16, st_r * k_row + st_g * 16, i * 4 * k_row, 0, 0);
  };
  const int wave64 = __builtin_amdgcn_readfirstlane(tid & ~63);
  stage_keys(wave64);
  list_valid_pages(p.table + (int64_t)b * p.NB, p.NB, p.num_pages, jp, nullptr, vidx, nullptr, &nvalid_s, &mine_s);
  __syncthreads();
  const int nchunks = nvalid_s * cpp;
  const int ntiles = (nchunks + CT - 1) / CT;
  const int my_ord = mine_s;
  for (int i = tid; i < nchunks; i += kT) chunk_of[i] = vidx[i / cpp] * cpp + i % cpp;
  __syncthreads();

  const int rounds = (p.BS + KEYS - 1) / KEYS;
  for (int rr = 0; rr < rounds; ++rr) {
    const int key0 = rr * KEYS, row0 = jp * p.BS + key0;   // first slot of this round
    const int slot = key0 + tid;                           // the key whose chain this lane walks
    const bool live = slot < p.BS;
    // What a tile needs is requested one tile ahead: its chunk sums (CT x kDmax floats), which are split into the three planes
    // once the tile before is done with them, and the claims of its CT * kChunk keys, whose values are corrections where
    // they were taken from this round's keys.
    constexpr int kSums = CT * (kDmax / 4) / kT, kClaims = CT * kChunk / kT;
    float4 pv[kSums];
    int from[kClaims];
    float value[kClaims];
    auto request = [&](int tile) {
#pragma unroll
      for (int u = 0; u < kSums; ++u) {
        const int i = tid + u * kT;
        const int vc = tile * CT + i / (kDmax / 4), q4 = i % (kDmax / 4);
        pv[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (vc < nchunks) pv[u] = *(const float4*)(chunk_all + (int64_t)chunk_of[vc] * kDmax + q4 * 4);
      }
#pragma unroll
      for (int u = 0; u < kClaims; ++u) {
        const int i = tid + u * kT, vc = tile * CT + i / kChunk;
        from[u] = -1;
        if (vc < nchunks) {
          const int64_t t = obase + (int64_t)chunk_of[vc] * kChunk + i % kChunk;
          from[u] = p.ws_col[t] - row0;
          value[u] = p.ws_val[t];
        }
      }
    };
    // the next tile's planes, the corrections of its entries
    auto store = [&](int tile, int own_chunk, float diag) {
#pragma unroll
      for (int u = 0; u < kSums; ++u) {
        const int i = tid + u * kT;
        const int m = i / (kDmax / 4), q4 = i % (kDmax / 4);
        uint32_t lo[3], hi[3];
        Split3<T>::two(pv[u].x, pv[u].y, lo);
        Split3<T>::two(pv[u].z, pv[u].w, hi);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) *(uint2*)(planes + (pl * CT + m) * ROWH + q4 * 8) = make_uint2(lo[pl], hi[pl]);
      }
      bool any = false;
#pragma unroll
      for (int u = 0; u < kClaims; ++u)
        if (from[u] >= 0 && from[u] < KEYS && key0 + from[u] < p.BS) {
          atomicAdd(&cl[from[u] * kChainLd + (tid + u * kT) / kChunk], to_fixed26(value[u]));
          any = true;
        }
      const int own = own_chunk - tile * CT;
      if (live && own >= 0 && own < CT) {
        atomicAdd(&cl[tid * kChainLd + own], to_fixed26(diag));
        any = true;
      }
      if (any) corrected[tile & 1] = 1;
    };
    request(0);
    const float rn = live ? p.ws_sum[obase + row0 + tid] : 0.f;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's keys are in LDS
    ZP_CSTAMP(0);   // table lookup, page list, first requests
    // ---- B fragments: keys as stored; lane (col, half) holds k = 16 s + 8 half + i of keys col and col + 32 of the wave's 64
    frag_t bk[2][KSB];
    float ssq[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const bool there = key0 + wave64 + g * 32 + col < p.BS;
      const char* src = keys + (g * 8 + (col >> 2)) * kPgGrp + (col & 3) * 64 + half * 16;
      ssq[g] = 0.f;
#pragma unroll
      for (int s = 0; s < KSB; ++s) {
        u32x4 v = *(const u32x4*)(src + (s >> 1) * 256 + (s & 1) * 32);
        if (!there || 2 * s + half >= dpieces) v = u32x4{0u, 0u, 0u, 0u};
        bk[g][s] = __builtin_bit_cast(frag_t, v);
        float e[8];
        Unpack<T>::run(vec16{v.x, v.y, v.z, v.w}, e);
#pragma unroll
        for (int q = 0; q < 8; ++q) ssq[g] = fmaf(e[q], e[q], ssq[g]);
      }
      ssq[g] += lane_xor32(ssq[g]);
    }
    const float diag = (half ? ssq[1] : ssq[0]) * rn * rn;    // S_ii, the entry the reference zeroes
    const int own_chunk = my_ord * cpp + slot / kChunk;
    float part = 0.f, total = 0.f;                    // chain state of this lane's key
    __syncthreads();                                  // everyone has its keys
    for (int i = tid; i < KEYS * kChainLd / 4; i += kT) ((int4*)cl)[i] = make_int4(0, 0, 0, 0);
    if (tid == 0) corrected[0] = 0;
    __syncthreads();
    store(0, own_chunk, diag);
    if (ntiles > 1) request(1);
    ZP_CSTAMP(1);   // first planes
    int cm = 0;                              // where the next chunk lies inside its page
    for (int tile = 0; tile < ntiles; ++tile) {
      __syncthreads();                       // the tile's planes and corrections are in LDS
      const bool some = corrected[tile & 1] != 0;
      if (tid == 0) corrected[(tile + 1) & 1] = 0;
      ZP_CSTAMP(2);   // barrier
      // ---- chunk sums of the tile: A = planes (rows = chunks), B = keys
      f32x16_t acc[2];
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[g][r] = 0.f;
      // fragments leave LDS kAhead ahead of their products, the smallest plane first
      constexpr int kAhead = 4, kFrags = 3 * KSB;
      frag_t a[kAhead + 1];
      auto fragment = [&](int n) { a[n % (kAhead + 1)] = *(const frag_t*)(planes + ((2 - n / KSB) * CT + col) * ROWH + half * 16 + n % KSB * 32); };
#pragma unroll
      for (int n = 0; n < kAhead; ++n) fragment(n);
#pragma unroll
      for (int n = 0; n < kFrags; ++n) {
        if (n + kAhead < kFrags) fragment(n + kAhead);
        acc[0] = Mfma16<T>::run(a[n % (kAhead + 1)], bk[0][n % KSB], acc[0]);
        acc[1] = Mfma16<T>::run(a[n % (kAhead + 1)], bk[1][n % KSB], acc[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // lane (col, half) has chunks 8 (r / 4) + 4 half + r % 4 of keys col and col + 32; now all of them of one key
      float v[CT];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0][r]), __float_as_uint(acc[1][r]), false, false);
        const int m = (r >> 2) * 8 + (r & 3);
        v[m] = __uint_as_float(both[0]) * rn;
        v[m + 4] = __uint_as_float(both[1]) * rn;
      }
      if (some) {
#pragma unroll
        for (int m = 0; m < CT; m += 4) {
          int4* const at = (int4*)(cl + tid * kChainLd + m);
          const int4 c = *at;
          v[m] -= from_fixed26(c.x);
          v[m + 1] -= from_fixed26(c.y);
          v[m + 2] -= from_fixed26(c.z);
          v[m + 3] -= from_fixed26(c.w);
          *at = make_int4(0, 0, 0, 0);
        }
      }
      ZP_CSTAMP(3);   // products
      __syncthreads();                       // everyone is done with the planes and this lane's corrections are clear
      ZP_CSTAMP(4);   // barrier
      if (tile + 1 < ntiles) {
        store(tile + 1, own_chunk, diag);
        if (tile + 2 < ntiles) request(tile + 2);
      }
      ZP_CSTAMP(5);   // next planes stored
      // ---- the reference's chain: one cache-dtype partial sum per column page.  Behind the last chunk there are zeros.
      auto page_ends = [&](int chunks) {
        if (cm == 0) { total += part; part = 0.f; }
        cm += chunks;
        if (cm >= cpp) cm = 0;
      };
      if (cpp % 8 == 0) {
#pragma unroll
        for (int m = 0; m < CT; ++m) {
          if (m % 8 == 0) page_ends(8);
          part = Elem<T>::rnd(part + v[m]);
        }
      } else {
#pragma unroll
        for (int m = 0; m < CT; ++m) {
          page_ends(1);
          part = Elem<T>::rnd(part + v[m]);
        }
      }
      ZP_CSTAMP(6);   // chain
    }
    if (live) Elem<T>::st(p.r_out, obase + row0 + tid, total + part);
    if (rr + 1 < rounds) {
      __syncthreads();                       // everyone is done with the planes
      stage_keys(key0 + KEYS + wave64);
    }
  }
#ifdef ZP_PAGE_STAMP
  if (tid == 0 && blockIdx.x < (1 << 16)) {
    long long* dst = zp_chain_stamp_buf + (int64_t)blockIdx.x * 12;
    for (int i = 0; i < 8; ++i) dst[i] = acc_[i];
    dst[10] = wall0;
    dst[11] = wall_clock64() - wall0;
  }
#endif
}
#undef ZP_CSTAMP

// ------------------------------------------------------------------ softmax epilogue
// One workgroup per (layer, sequence, head) row of T logits:
//   raw only: r_i = rowsum_i - sum_{j: c*(j)=i} v_j, pad pages -inf
//   x = rnd(r / divisor); x = rnd(x - max); out = rnd(exp(x) / sum)
__device__ __forceinline__ float block_reduce(float v, float* lds, bool is_max) {
  if (is_max) v = wave_max(v); else v = wave_sum(v);
  __syncthreads();
  if (lane_id() == 0) lds[wave_id()] = v;
  __syncthreads();
  float m = lds[0];
#pragma unroll
  for (int i = 1; i < kWaves; ++i) m = is_max ? fmaxf(m, lds[i]) : m + lds[i];
  return m;
}

template <typename T, bool RAW>
__global__ __launch_bounds__(kThreads) void red_softmax_kernel(
    void* __restrict__ red, void* __restrict__ logits, const int32_t* __restrict__ table,
    const float* __restrict__ ws_sum, const int32_t* __restrict__ ws_col,
    const float* __restrict__ ws_val, int B, int NB, int BS, int Hkv, int num_pages,
    float tscale /* raw: temperature; lightning: temperature*BS */,
    int rows_ready /* raw: the row sums are already in `red` (16-bit caches) */,
    const float* __restrict__ ws_csum = nullptr /* raw, fp32, every pair of pages once: column-side
        sums [distance - 1][row][Tn]; ws_col then holds 64-bit (index + 1, value) claims */,
    int64_t n_keys = 0) {
  extern __shared__ __align__(16) char smem[];
  __shared__ float red_lds[kWaves];
  const int Tn = NB * BS;
  // raw: [Tn] 64-bit sums of the values claimed from each row, then the [Tn] floats of the row
  unsigned long long* corr = (unsigned long long*)smem;
  const bool from_ws = RAW && !rows_ready;
  float* x = (float*)(smem + (from_ws ? (size_t)Tn * 8 : 0));
  const int64_t row = blockIdx.x;
  const int b = (int)((row / Hkv) % B);
  const int64_t base = row * Tn;
  const int32_t* trow = table + (int64_t)b * NB;
  int nvalid = 0;
  unsigned long long there = 0;       // which of the first 64 pages are
  for (int j0 = 0; j0 < NB; j0 += 64) {
    const int c = j0 + lane_id() < NB ? trow[j0 + lane_id()] : -1;
    const int pid = page_is_pad(c) ? -1 : page_id(c);
    const unsigned long long valid = __ballot(pid >= 0 && pid < num_pages);
    if (j0 == 0) there = valid;
    nvalid += __popcll(valid);
  }
  auto page_there = [&](int j) -> bool {
    if (j < 64) return there >> j & 1;
    const int c = trow[j], pid = page_is_pad(c) ? -1 : page_id(c);
    return pid >= 0 && pid < num_pages;
  };
  // a row's loads side by side: one after the other, each waits for memory (64 bf16 sequences of 8 rows 8.3 us, now 6.3; one fp32 one with
  // the sums of the raw variant's pairs of pages 24.5, now 13.9; 40 42 and 20)
  constexpr int kAhead = 12;
  const float divisor = RAW ? tscale * (float)(nvalid * BS) : tscale;
  const unsigned long long* claims = (const unsigned long long*)ws_col;
  if (from_ws) {
    // every key hands the value of its claimed entry to the row it was taken from: 2^-32 fixed
    // point with integer atomics, exact and independent of the order
    for (int t = threadIdx.x; t < Tn; t += kThreads) corr[t] = 0ull;
    __syncthreads();
    for (int t0 = threadIdx.x; t0 < Tn; t0 += kAhead * kThreads) {
      int cc[kAhead];
      float v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int64_t at = base + min(t0 + u * kThreads, Tn - 1);
        if (ws_csum) {
          const unsigned long long cl = claims[at];
          cc[u] = (int)(cl >> 32) - 1;
          v[u] = __uint_as_float((unsigned)cl);
        } else {
          cc[u] = ws_col[at];
          v[u] = ws_val[at];
        }
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int t = t0 + u * kThreads;
        if (t < Tn && cc[u] >= 0 && cc[u] < Tn && page_there(t / BS)) atomicAdd(&corr[cc[u]], to_fixed32(v[u]));
      }
    }
    __syncthreads();
  }
  float mloc = -INFINITY;
  if (!from_ws) {
    for (int t0 = threadIdx.x; t0 < Tn; t0 += kAhead * kThreads) {
      float r[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) r[u] = Elem<T>::ld(red, base + min(t0 + u * kThreads, Tn - 1));
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int t = t0 + u * kThreads;
        if (t >= Tn) break;
        if (logits) Elem<T>::st(logits, base + t, r[u]);
        const float xv = Elem<T>::rnd(r[u] / divisor);
        x[t] = xv;
        mloc = fmaxf(mloc, xv);
      }
    }
  }
  for (int t0 = threadIdx.x; from_ws && t0 < Tn; t0 += kAhead * kThreads) {
    float sv[kAhead];
    int rank[kAhead];                 // of a key's page among those that are there
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int t = min(t0 + u * kThreads, Tn - 1);
      sv[u] = ws_sum[base + t];
      rank[u] = ws_csum ? __popcll(there & ((1ull << t / BS) - 1)) : 0;      // pairs of pages: tables of at most 16
    }
    // the column-side sums of a key's page: distance d was written by the valid page d places before it (cyclically), if that
    // page ran the distance
    for (int d = 1; ws_csum && d <= nvalid / 2; ++d) {
      float x[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) x[u] = ws_csum[(int64_t)(d - 1) * n_keys + base + min(t0 + u * kThreads, Tn - 1)];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int a = rank[u] - d >= 0 ? rank[u] - d : rank[u] - d + nvalid;
        const bool ran = d < nvalid / 2 + (((nvalid & 1) || a < nvalid / 2) ? 1 : 0);
        if (ran) sv[u] += x[u];
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int t = t0 + u * kThreads;
      if (t >= Tn) break;
      const float r = page_there(t / BS) ? Elem<T>::rnd(sv[u] - from_fixed32(corr[t])) : -INFINITY;
      if (logits) Elem<T>::st(logits, base + t, r);
      const float xv = Elem<T>::rnd(r / divisor);
      x[t] = xv;
      mloc = fmaxf(mloc, xv);
    }
  }
  const float m = block_reduce(mloc, red_lds, true);
  float sloc = 0.f;
  for (int t = threadIdx.x; t < Tn; t += kThreads) {
    const float e = expf(Elem<T>::rnd(x[t] - m));
    x[t] = e;
    sloc += e;
  }
  const float ssum = block_reduce(sloc, red_lds, false);
  for (int t = threadIdx.x; t < Tn; t += kThreads) Elem<T>::st(red, base + t, x[t] / ssum);
}

int check_common(const char* name, const void* k_cache, const int32_t* table, void* red_out,
                 int L, int B, int NB, int BS, int Hkv, int D, int dtype, int64_t k_sl,
                 int64_t k_sp) {
  ZP_REQUIRE(k_cache && table && red_out, "%s: null pointer", name);
  ZP_REQUIRE(L >= 0 && B >= 0 && NB > 0 && BS > 0 && Hkv > 0 && D > 0, "%s: bad dims", name);
  ZP_REQUIRE(dtype >= ZP_BF16 && dtype <= ZP_F32, "%s: unknown dtype tag %d", name, dtype);
  const int es = zp_dtype_bytes(dtype);
  if (!(D <= kDmax && (D * es) % 16 == 0)) {
    zp_set_error("%s: head_dim %d unsupported (need <= %d and a multiple of %d)", name, D, kDmax,
                 16 / es);
    return ZP_EUNSUPPORTED;
  }
  if (BS % TN != 0) {
    zp_set_error("%s: page size %d is not a multiple of %d", name, BS, TN);
    return ZP_EUNSUPPORTED;
  }
  ZP_REQUIRE(((uintptr_t)k_cache % 16) == 0 && (k_sl * es) % 16 == 0 && (k_sp * es) % 16 == 0,
             "%s: key cache must be 16-byte aligned", name);
  return ZP_OK;
}

// fp32 all-pairs: can every unordered pair of pages be multiplied once (pages of at most 256
// keys in whole 64-key tiles, column-sum slots for every distance in the workspace)?
inline bool raw_f32_symmetric(int NB, int BS) {
  return BS <= 256 && BS % TN == 0 && NB / 2 <= kSymMaxDist;
}

// Workgroups of the page kernels, `per_cu` of which a CU holds, walk whole rows where these fill the CUs in rounds that are at
// least 90 % full: a page then lands while the one before is finished (512 16-bit rows of 9 pages: 86 us, 93 with a page
// each; 1024 fp32 rows: 435, 486).  Otherwise a page each, so that few rows or a thin last round leave no CU idle (8 rows of
// 10 pages: 49 us by rows, 13, fp32 108, 18; 768 16-bit rows of 9: 149, 140; 320 fp32 rows: 237, 172; all but the 435 and 486
// with the softmax).
GramArgs page_walks(GramArgs a, int L, int per_cu) {
  const int64_t rows = (int64_t)L * a.B * a.Hkv, slots = 256 * per_cu;
  const bool walk = (rows + slots - 1) / slots * slots * 9 <= rows * 10 || rows * a.NB > (1 << 22);
  a.parts = walk ? 1 : a.NB;
  return a;
}

// All pairs, 16 bit: the column tiles of a page are divided among workgroups where that ends the launch earlier, in rounds of two
// workgroups per CU whose beginning takes as long as two tiles; claims are integer maxima whatever the order.  Pages of 1, 2, 3, 4
// and 8 sequences of 8 heads, us whole and in parts: 54.6 and 22.6 (5), 56.5 and 33.8 (3), 58.0 and 41.9 (2), 79.2 and 64.5
// (3), 118.8 and 104.9 (2); of 6, 12, 24 and 40 best whole (74.5 and 80.0 with 2; 143 and 145; 267 and 275; 412 and 440).
GramArgs tile_parts(GramArgs a, int64_t pages) {
  const int tiles = (a.NB / 2 + 1) * (a.BS / kRawTile);
  int64_t least = INT64_MAX;
  for (int n = 1; n <= 5 && n <= tiles && pages * n <= INT32_MAX; ++n) {
    const int64_t cost = (pages * n + 511) / 512 * (2 * n + tiles) * (60 / n);
    if (cost < least) least = cost, a.parts = n;
  }
  return a;
}
// The keys of a page, whose claims are looked up one after the other, go to several workgroups where all of them run at once, six on a
// CU: more take longer to launch than the claims of most pages (us with 1, 2, 4 and 8 workgroups, without claims and with claims of
// half of the keys: 72 pages of 256 4.5, 4.5, 4.6, 4.4 and 12.7, 7.8, 5.7, 5.0; 288 4.6, 4.6, 4.9, 5.5 and 16.6, 11.2, 9.4, 10.2; 576 4.7,
// 4.6, 5.5, 8.8 and 21.0, 15.2, 14.8, 15.9; 1728 4.6, 7.2, 12.4, 23 and 36.8, 35.9, 33.6, 39.4).
GramArgs claim_parts(GramArgs a, int64_t pages) {
  for (a.parts = 8; a.parts > 1 && pages * a.parts > 1536; a.parts /= 2) {}
  return a;
}

template <typename T, bool RAW>
int launch_gram(const GramArgs& a, int L, hipStream_t st) {
  dim3 grid((unsigned)((int64_t)L * a.B * a.Hkv * a.NB));
  const size_t tail = (RAW ? 0 : (size_t)a.BS * 20) + sizeof(int) * 2 * a.NB;
  if constexpr (T::bytes == 2 && !RAW) {
    // the block table row sits in LDS
    const size_t smem = (size_t)kPgBytes + 4 * kDmax * 2 + 4 * kPageRows * 2 +
                        (size_t)kPageRows * (2 * 8 + 2 * 4 + 4 + 4) + sizeof(int) * (kPageWaves + 2 + a.NB);
    if (a.BS <= kPageRows && a.BS % 32 == 0 && smem <= 80 * 1024 + 8) {
      const GramArgs w = page_walks(a, L, 2);
      grid = dim3((unsigned)((int64_t)L * a.B * a.Hkv * w.parts));
      if (hipFuncSetAttribute((const void*)gram_page_kernel<T>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
        zp_set_error("redundancy: cannot reserve %zu bytes of LDS", smem);
        return ZP_EHIP;
      }
      hipLaunchKernelGGL((gram_page_kernel<T>), grid, dim3(kPageThreads), smem, st, w);
      ZP_LAUNCH_CHECK();
      return ZP_OK;
    }
  }
  if constexpr (T::bytes == 4 && !RAW) {
    if (a.BS <= kPage32Rows && a.BS % 32 == 0 && a.NB <= 1024) {
      const GramArgs w = page_walks(a, L, 1);
      grid = dim3((unsigned)((int64_t)L * a.B * a.Hkv * w.parts));
      const size_t smem = (size_t)kPage32Rows * ROWF * 4 + (size_t)kPage32Rows * (8 + 8 + 4 + 4 * 4) +
                          sizeof(int) * a.NB;
      if (hipFuncSetAttribute((const void*)gram_page_f32_kernel,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
        zp_set_error("redundancy: cannot reserve %zu bytes of LDS", smem);
        return ZP_EHIP;
      }
      hipLaunchKernelGGL(gram_page_f32_kernel, grid, dim3(kPage32Threads), smem, st, w);
      ZP_LAUNCH_CHECK();
      return ZP_OK;
    }
  }
  if constexpr (T::bytes == 4 && RAW) {
    if (raw_f32_symmetric(a.NB, a.BS)) {
      const int64_t n = (int64_t)L * a.B * a.Hkv * a.NB * a.BS;
      const size_t smem = sizeof(float) * (2 * TN * ROWF + 2 * kSymWaves * TN) + sizeof(int) * 2 * a.NB;
      if (hipFuncSetAttribute((const void*)gram_raw_sym_f32_kernel,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
        zp_set_error("redundancy: cannot reserve %zu bytes of LDS", smem);
        return ZP_EHIP;
      }
      hipLaunchKernelGGL(fill_u64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                         (unsigned long long*)a.ws_col, n, 0ull);
      hipLaunchKernelGGL(gram_raw_sym_f32_kernel, grid, dim3(kSymWaves * 64), smem, st, a);
      ZP_LAUNCH_CHECK();
      return ZP_OK;
    }
  }
  if constexpr (T::bytes == 2 && RAW) {
    // column tiles of 128 keys when the page size allows: half as many workgroup barriers
    const int tn = a.BS % 128 == 0 ? 128 : TN;
    const size_t smem1 = 2 * (size_t)tn * ROWH + sizeof(int) * 4 * tn + sizeof(float) * a.BS +
                         sizeof(int) * 2 * a.NB;
    const void* fn = tn == 128 ? (const void*)gram_raw_kernel<T, 128> : (const void*)gram_raw_kernel<T, TN>;
    // whole 128-key tiles: the four-wave kernel with two row blocks per wave
    const size_t smemw = 2 * (size_t)kRawTileBytes + sizeof(int) * 4 * kRawTile + sizeof(float) * a.BS +
                         sizeof(int) * 2 * a.NB;
    const bool wide = tn == 128 && smemw <= 80 * 1024;
    const size_t smem2 = kChainBytes + sizeof(int) * (a.NB + a.NB * a.BS / kChunk);
    if ((int64_t)a.NB * (a.BS + 1) > kMostRawTokens) {
      zp_set_error("redundancy: a row of %d pages of %d tokens (16-bit caches: at most %d tokens and pages)", a.NB, a.BS, kMostRawTokens);
      return ZP_EUNSUPPORTED;
    }
    const GramArgs cut = tile_parts(a, grid.x), claims = claim_parts(a, grid.x);
    const void* const wide_fn = cut.parts > 1 ? (const void*)gram_raw_wide_kernel<T, true> : (const void*)gram_raw_wide_kernel<T, false>;
    if (hipFuncSetAttribute(wide ? wide_fn : fn,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)(wide ? smemw : smem1)) != hipSuccess ||
        hipFuncSetAttribute((const void*)raw_chain_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)smem2) != hipSuccess) {
      zp_set_error("redundancy: cannot reserve %zu / %zu bytes of LDS", smem1, smem2);
      return ZP_EHIP;
    }
    hipLaunchKernelGGL((raw_prep_kernel<T>), grid, dim3(kThreads), 0, st, a);
    if (wide && cut.parts > 1) hipLaunchKernelGGL((gram_raw_wide_kernel<T, true>), dim3(grid.x * cut.parts), dim3(256), smemw, st, cut);
    else if (wide) hipLaunchKernelGGL((gram_raw_wide_kernel<T, false>), grid, dim3(256), smemw, st, cut);
    else if (tn == 128) hipLaunchKernelGGL((gram_raw_kernel<T, 128>), grid, dim3(512), smem1, st, a);
    else hipLaunchKernelGGL((gram_raw_kernel<T, TN>), grid, dim3(512), smem1, st, a);
    hipLaunchKernelGGL((raw_claim_value_kernel<T>), dim3(grid.x * claims.parts), dim3(kThreads), 0, st, claims);
    hipLaunchKernelGGL((raw_chain_kernel<T>), grid, dim3(256), smem2, st, a);
    ZP_LAUNCH_CHECK();
    return ZP_OK;
  }
  if constexpr (T::bytes == 2 && !RAW) {
    const size_t smem = 4 * (size_t)TN * ROWH + tail;
    const bool wide = a.BS / 32 > kWaves;   // more row blocks than 4 waves: use 8 and halve the passes
    const void* fn = wide ? (const void*)gram_split_kernel<T, RAW, 8> : (const void*)gram_split_kernel<T, RAW, 4>;
    if (smem > 64 * 1024 &&
        hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
      zp_set_error("redundancy: cannot reserve %zu bytes of LDS", smem);
      return ZP_EHIP;
    }
    if (wide) hipLaunchKernelGGL((gram_split_kernel<T, RAW, 8>), grid, dim3(512), smem, st, a);
    else hipLaunchKernelGGL((gram_split_kernel<T, RAW, 4>), grid, dim3(kThreads), smem, st, a);
  } else {
    const size_t smem = sizeof(float) * 2 * TN * ROWF + tail;
    // more row blocks than 4 waves: 8 waves take the page's rows in one pass, so every column
    // tile is staged (and normalised) once instead of twice
    const bool wide = a.BS / 32 > kWaves;
    const void* fn = wide ? (const void*)gram_kernel<T, RAW, 8> : (const void*)gram_kernel<T, RAW, 4>;
    if (smem > 64 * 1024 &&
        hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
      zp_set_error("redundancy: cannot reserve %zu bytes of LDS", smem);
      return ZP_EHIP;
    }
    if (wide) hipLaunchKernelGGL((gram_kernel<T, RAW, 8>), grid, dim3(512), smem, st, a);
    else hipLaunchKernelGGL((gram_kernel<T, RAW, 4>), grid, dim3(kThreads), smem, st, a);
  }
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

template <typename T, bool RAW>
int launch_softmax(void* red, void* logits, const int32_t* table, const float* ws_sum,
                   const int32_t* ws_col, const float* ws_val, int L, int B, int NB, int BS,
                   int Hkv, int num_pages, double temperature, hipStream_t st, int rows_ready = 0,
                   const float* ws_csum = nullptr) {
  const size_t smem = (size_t)NB * BS * ((RAW && !rows_ready) ? 12 : 4);
  if (smem > 150 * 1024) {
    zp_set_error("redundancy: a row of %d tokens exceeds LDS", NB * BS);
    return ZP_EUNSUPPORTED;
  }
  if (smem > 64 * 1024 &&
      hipFuncSetAttribute((const void*)red_softmax_kernel<T, RAW>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) {
    zp_set_error("redundancy: cannot reserve %zu bytes of LDS", smem);
    return ZP_EHIP;
  }
  dim3 grid((unsigned)((int64_t)L * B * Hkv));
  hipLaunchKernelGGL((red_softmax_kernel<T, RAW>), grid, dim3(kThreads), smem, st, red, logits,
                     table, ws_sum, ws_col, ws_val, B, NB, BS, Hkv, num_pages,
                     RAW ? (float)temperature : (float)(temperature * (double)BS), rows_ready,
                     ws_csum, (int64_t)L * B * Hkv * NB * BS);
  ZP_LAUNCH_CHECK();
  return ZP_OK;
}

}  // namespace

extern "C" int zp_redundancy_lightning(const void* k_cache, const int32_t* block_table,
                                       void* red_out, void* logits_out, int32_t L, int32_t B,
                                       int32_t NB, int32_t BS, int32_t Hkv, int32_t D,
                                       int32_t num_pages, int64_t k_sl, int64_t k_sp,
                                       float threshold, double temperature, int32_t dtype,
                                       void* stream) {
  int rc = check_common("redundancy_lightning", k_cache, block_table, red_out, L, B, NB, BS, Hkv,
                        D, dtype, k_sl, k_sp);
  if (rc != ZP_OK) return rc;
  if (L == 0 || B == 0) return ZP_OK;
  GramArgs a;
  a.k = (const char*)k_cache; a.table = block_table; a.r_out = red_out;
  a.ws_sum = nullptr; a.ws_col = nullptr; a.ws_val = nullptr; a.ws_chunk = nullptr;
  a.B = B; a.NB = NB; a.BS = BS; a.Hkv = Hkv; a.D = D; a.num_pages = num_pages;
  a.k_sl = k_sl; a.k_sp = k_sp; a.threshold = threshold; a.eps = 1e-6f;
  hipStream_t st = (hipStream_t)stream;
  ZP_DISPATCH_DTYPE(dtype, {
    rc = launch_gram<T, false>(a, L, st);
    if (rc != ZP_OK) return rc;
    rc = launch_softmax<T, false>(red_out, logits_out, block_table, nullptr, nullptr, nullptr, L,
                                  B, NB, BS, Hkv, num_pages, temperature, st);
  });
  return rc;
}

extern "C" int64_t zp_redundancy_raw_workspace(int32_t L, int32_t B, int32_t NB, int32_t BS,
                                               int32_t Hkv) {
  // three fp32 / int32 words per key, and for 16-bit caches kDmax floats per chunk of 16 keys
  return (int64_t)L * B * Hkv * NB * BS * (12 + 4 * kDmax / kChunk);
}

extern "C" int zp_redundancy_raw(const void* k_cache, const int32_t* block_table, void* red_out,
                                 void* logits_out, int32_t L, int32_t B, int32_t NB, int32_t BS,
                                 int32_t Hkv, int32_t D, int32_t num_pages, int64_t k_sl,
                                 int64_t k_sp, float threshold, double temperature, int32_t dtype,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = check_common("redundancy_raw", k_cache, block_table, red_out, L, B, NB, BS, Hkv, D,
                        dtype, k_sl, k_sp);
  if (rc != ZP_OK) return rc;
  if (L == 0 || B == 0) return ZP_OK;
  const int64_t n = (int64_t)L * B * Hkv * NB * BS;
  const int64_t need = zp_redundancy_raw_workspace(L, B, NB, BS, Hkv);
  ZP_REQUIRE(workspace && workspace_bytes >= need,
             "redundancy_raw: workspace of %lld bytes required", (long long)need);
  ZP_REQUIRE(((uintptr_t)workspace % 16) == 0, "redundancy_raw: workspace must be 16-byte aligned");
  GramArgs a;
  a.k = (const char*)k_cache; a.table = block_table;
  a.r_out = red_out;   // 16-bit caches: the row sums go here before the softmax
  a.ws_sum = (float*)workspace; a.ws_col = (int32_t*)workspace + n; a.ws_val = (float*)workspace + 2 * n;
  a.ws_chunk = (float*)workspace + 3 * n;
  a.B = B; a.NB = NB; a.BS = BS; a.Hkv = Hkv; a.D = D; a.num_pages = num_pages;
  a.k_sl = k_sl; a.k_sp = k_sp; a.threshold = threshold; a.eps = 1e-6f;
  hipStream_t st = (hipStream_t)stream;
  ZP_DISPATCH_DTYPE(dtype, {
    rc = launch_gram<T, true>(a, L, st);
    if (rc != ZP_OK) return rc;
    rc = launch_softmax<T, true>(red_out, logits_out, block_table, a.ws_sum, a.ws_col, a.ws_val, L,
                                 B, NB, BS, Hkv, num_pages, temperature, st, T::bytes == 2,
                                 (T::bytes == 4 && raw_f32_symmetric(NB, BS)) ? a.ws_chunk : nullptr);
  });
  return rc;
}
