// limb.hip — quantized GEMMs over f32 activations on the int8 matrix cores
// (gfx950), for many rows.
//
//   k_lg_prep     rows (f32 or bf16) -> 31-bit block floating point, one
//                 exponent per row, as four int8 limbs in the MFMA order,
//                 with the row's group sums; with the routing blocks of a
//                 grouped call in the same launch.
//   k_lg          y = rows . dequant(W)^T on v_mfma_i32_16x16x64_i8: gate
//                 and up with SwiGLU, or one matrix; grouped (work items of
//                 <= 16 entries of one expert) or dense (16-row tiles).
//   k_lg_combine  out[t] = sum over t's entries in ascending expert order
//                 of fma(down[entry], w[entry], out).
//
// The arithmetic: a row is written as x_j = m_j 2^-f with |m_j| <= 2^30 and
// m = d0 + 2^8 d1 + 2^16 d2 + 2^24 d3 (signed bytes), so a value keeps its
// 24 mantissa bits down to 2^-6 of the row's largest and is off by at most
// 2^-30 of that below: less than f32 rounds the sums by, unless the largest
// meets a weight of zero. Codes enter as bytes; the sums of a group,
// S_L = sum_j q_j d_Lj, are exact int32 (|S_L| <= 128 * 15 * 128), and
//     t = (S0 + 2^8 S1) + 2^16 (S2 + 2^8 S3),  acc = fma(s, t, acc)
// rounds where an f32 sum of the group would, but not within it. The bias
// term sum_g b_g sum_{j in g} x_j runs on v_mfma_f32_16x16x4_f32 over the
// group sums (scaled by 2^f), and the result is acc 2^-f. A row with an
// infinity or NaN gets NaN group sums, so all its outputs are NaN. Groups of 32
// take v_mfma_i32_16x16x32_i8, one group per operand (masking the other
// groups' codes to zero in 64-input operands took twice the matrix work, 32
// mask instructions per tile and step, and registers beyond what there are:
// 16 rows 2048 -> 152064 115 us against 93).
#include "common.h"
#include "kernels.h"

namespace smoe {

typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kLgM = 16;    // rows per work item (one MFMA tile)
constexpr uint32_t kLgKC = 128;  // inputs per step: one 32-code chunk per lane

__host__ __device__ constexpr uint32_t lg_kp(uint32_t K) { return (K + kLgKC - 1) / kLgKC * kLgKC; }
// Group sums per row, padded to a multiple of 16 bytes.
__host__ __device__ constexpr uint32_t lg_gp(uint32_t K, uint32_t G) { return (lg_kp(K) / G + 3) / 4 * 4; }

// ---------------------------------------------------------------------------
// Rows -> limbs.
//
// Limb memory: row r, step j (128 inputs), half h, limb L, lane block kb:
// 16 bytes at r * KP * 4 + ((j * 2 + h) * 4 + L) * 64 + kb * 16. The 16
// inputs of (j, h, kb) are those the lanes kb of k_lg hold as B operand h:
// for groups of 64, 128 j + 64 h + {0, 32, 16, 48}[kb] (the halves of two
// lanes' chunks, exchanged by a permlane swap, so that an operand lies in
// one group); of 32, eight of each of two groups, 128 j + 64 h + 8 kb and 32
// on (the four lanes' chunks transposed by their words); else 128 j + 32 kb +
// 16 h. Byte order: code words unpack to even codes, then odd codes, of eight.
// ---------------------------------------------------------------------------
template <bool BF16>
__device__ __forceinline__ void lg_load8(const void* x, uint64_t i, float (&f)[8]) {
  if constexpr (BF16) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(x) + i);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[2 * j] = __uint_as_float(w[j] << 16);
      f[2 * j + 1] = __uint_as_float(w[j] & 0xFFFF0000u);
    }
  } else {
    const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(x) + i);
    const f32x4 a = p[0], b = p[1];
    f[0] = a.x, f[1] = a.y, f[2] = a.z, f[3] = a.w, f[4] = b.x, f[5] = b.y, f[6] = b.z, f[7] = b.w;
  }
}

// Row r by one wave: two passes over the row (the second from the caches).
template <int G, bool BF16>
__device__ __forceinline__ void lg_prep_row(const void* x, uint32_t r, uint32_t K, uint8_t* limbs, float* xsum,
                                            int32_t* xexp, uint32_t lane) {
  const uint32_t KP = lg_kp(K), gp = lg_gp(K, G);
  const uint64_t row = (uint64_t)r * K;
  float amax = 0.f, fin = 0.f;  // fin: 0 while every value is finite, else NaN
  for (uint32_t i = lane * 8; i < K; i += 512) {
    float f[8];
    lg_load8<BF16>(x, row + i, f);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      amax = fmaxf(amax, fabsf(f[j]));
      fin = __builtin_fmaf(f[j], 0.f, fin);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    amax = fmaxf(amax, __shfl_xor(amax, o, kWave));
    fin += __shfl_xor(fin, o, kWave);
  }
  const bool finite = fin == 0.f;
  // |x| < 2^E with E the frexp exponent of amax: |m| < 2^30.
  const int fx = finite && amax > 0.f ? 30 - __builtin_amdgcn_frexp_expf(amax) : 0;
  if (lane == 0) xexp[r] = fx;
  float* const xs = xsum + (uint64_t)r * gp;
  uint8_t* const lr = limbs + (uint64_t)r * KP * 4;
  for (uint32_t u = lane; u < KP / 16; u += kWave) {  // (j, h, kb) = u / 8, u / 4 % 2, u % 4
    const uint32_t j = u >> 3, h = (u >> 2) & 1, kb = u & 3;
    // The unit's first and second eight inputs. K is a multiple of 32, so each
    // eight lies in the row or past it.
    const uint32_t pos = G == 64   ? 128 * j + 64 * h + 32 * (kb & 1) + 16 * (kb >> 1)
                         : G == 32 ? 128 * j + 64 * h + 8 * kb
                                   : 128 * j + 32 * kb + 16 * h;
    float f[16];
#pragma unroll
    for (uint32_t e = 0; e < 2; ++e) {
      const uint32_t at = pos + e * (G == 32 ? 32 : 8);
      float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (at < K) lg_load8<BF16>(x, row + at, a);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[8 * e + i] = a[i];
    }
    int32_t d[4][16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int32_t m = finite ? (int32_t)__builtin_rintf(__builtin_ldexpf(f[i], fx)) : 0;
      const int32_t d0 = (int32_t)((uint32_t)m << 24) >> 24, m1 = (m - d0) >> 8;
      const int32_t d1 = (int32_t)((uint32_t)m1 << 24) >> 24, m2 = (m1 - d1) >> 8;
      const int32_t d2 = (int32_t)((uint32_t)m2 << 24) >> 24;
      d[0][i] = d0, d[1][i] = d1, d[2][i] = d2, d[3][i] = (m2 - d2) >> 8;
    }
    // Pairwise sums of the two eights.
    float s[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float* const v = f + 8 * e;
      s[e] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
#pragma unroll
    for (int L = 0; L < 4; ++L) {
      u32x4 v;
      v.x = pack_bytes(d[L][0], d[L][2], d[L][4], d[L][6]);
      v.y = pack_bytes(d[L][1], d[L][3], d[L][5], d[L][7]);
      v.z = pack_bytes(d[L][8], d[L][10], d[L][12], d[L][14]);
      v.w = pack_bytes(d[L][9], d[L][11], d[L][13], d[L][15]);
      *reinterpret_cast<u32x4*>(lr + (((uint64_t)j * 2 + h) * 4 + L) * 64 + kb * 16) = v;
    }
    // Group sums: over kb, and over h too with groups of 128. KP / 16 is a
    // multiple of 8, so the lanes of a group are active together.
    if constexpr (G != 32) s[0] += s[1];
#pragma unroll
    for (int e = 0; e < (G == 32 ? 2 : 1); ++e) {
      s[e] += __shfl_xor(s[e], 1, kWave);
      s[e] += __shfl_xor(s[e], 2, kWave);
      if (G == 128) s[e] += __shfl_xor(s[e], 4, kWave);
      const bool first = G == 128 ? (u & 7) == 0 : kb == 0;
      const uint32_t g = G == 32 ? 4 * j + 2 * h + e : G == 64 ? 2 * j + h : j;
      if (first) xs[g] = finite ? __builtin_ldexpf(s[e], fx) : __builtin_nanf("");
    }
  }
}

// ---------------------------------------------------------------------------
// Routing of a grouped call: entry i = (token, slot) gets its position in
// (expert, token) order by counting the entries before it, each of the N
// ids read from LDS: N^2 compares spread over N / 8 blocks, any number of
// experts, no atomics, and nothing that has to be cleared first.
// Items: expert e with its entries at [p, p + c) takes ceil(c / 16) slots
// from p / 16 + min(e, p) on (each hit expert has at least one entry, so
// the ranges of successive hit experts never overlap); its last entry marks
// the slots up to the next hit expert's as empty.
// ---------------------------------------------------------------------------
struct LgRoute {
  const int32_t* idx;  // [n, k]
  const float* w;
  uint32_t n, k, E, n_slots;
  uint2* items;        // [n_slots] expert, start | count << 16
  uint32_t* item_tok;  // [n_slots, 16] token of each item row (unset past the count)
  uint2* tok_pw;       // [n, k] (position, weight bits), ascending expert
  uint32_t* err;
};

__host__ __device__ constexpr uint32_t lg_slot(uint32_t e, uint32_t p) { return p / kLgM + (e < p ? e : p); }
static uint32_t lg_slots(uint32_t N, uint32_t E) { return N / kLgM + (E < N ? E : N) + 1; }

constexpr uint32_t kLgRouteE = 8, kLgRouteT = 256 / kLgRouteE;  // entries per block, threads per entry

template <typename F>
__device__ __forceinline__ uint32_t route_reduce(uint32_t v, F f) {
#pragma unroll
  for (int o = kLgRouteT / 2; o > 0; o >>= 1) v = f(v, (uint32_t)__shfl_xor((int)v, o, kWave));
  return v;
}

__device__ __forceinline__ void lg_route_block(const LgRoute& a, uint32_t block, uint32_t* ids) {
  const uint32_t N = a.n * a.k, tid = threadIdx.x, sl = tid % kLgRouteT;
  const uint32_t b0 = block * kLgRouteE, i0 = b0 + tid / kLgRouteT;
  const bool live = i0 < N;
  const uint32_t i = live ? i0 : N - 1;
  bool bad = false;
  for (uint32_t j = tid; j < (N + 3) / 4 * 4; j += 256) {
    const int32_t id = j < N ? a.idx[j] : -1;
    const bool ok = id >= 0 && (uint32_t)id < a.E;
    bad |= j < N && !ok;
    ids[j] = j < N ? (ok ? (uint32_t)id : 0u) : 0xFFFFFFFFu;
  }
  const float wt = a.w[i];
  __syncthreads();
  const uint32_t e = ids[i], e1 = e + 1, t = i / a.k;
  uint32_t less = 0, eq = 0, gap = 0xFFFFFFFFu;
  // Entries [lo, hi) of this thread's share, in fours (lo a multiple of 4).
  auto count = [&](uint32_t lo, uint32_t hi) {
    for (uint32_t j = lo + sl * 4; j < hi; j += kLgRouteT * 4) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(ids + j);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        less += v[c] < e ? 1u : 0u;
        eq += v[c] == e ? 1u : 0u;
        gap = min(gap, v[c] - e1);  // the next larger id (ids below e1 wrap to huge)
      }
    }
  };
  count(0, b0);
  uint32_t before = eq;  // equal ids ahead of the block, then those within it
  if (sl < kLgRouteE && b0 + sl < i) before += ids[b0 + sl] == e ? 1u : 0u;
  count(b0, N);
  auto add = [](uint32_t x, uint32_t y) { return x + y; };
  less = route_reduce(less, add);
  eq = route_reduce(eq, add);
  before = route_reduce(before, add);
  gap = route_reduce(gap, [](uint32_t x, uint32_t y) { return min(x, y); });
  // The entry's place among its token's, and repeated ids.
  uint32_t ord = 0;
  if (sl < a.k) {
    const uint32_t s0 = i - t * a.k, o = ids[t * a.k + sl];
    ord = (o < e || (o == e && sl < s0)) ? 1u : 0u;
    bad |= o == e && sl != s0;
  }
  ord = route_reduce(ord, add);
  if (bad) *a.err = 2u;
  if (!live) return;
  const uint32_t pos = less + before, item = lg_slot(e, less) + before / kLgM;
  if (sl == 0) {
    a.item_tok[item * kLgM + before % kLgM] = t;
    a.tok_pw[t * a.k + ord] = make_uint2(pos, __float_as_uint(wt));
    if (before % kLgM == 0) a.items[item] = make_uint2(e, pos | (min(kLgM, eq - before) << 16));
  }
  if (before == eq - 1) {
    const uint32_t end = less + eq, e2 = e1 + gap;
    const uint32_t hi = end < N ? lg_slot(e2, end) : a.n_slots;
    for (uint32_t s = item + 1 + sl; s < hi; s += kLgRouteT) a.items[s] = make_uint2(0u, 0u);
  }
}

// Blocks 0 .. nb_route - 1 route; the others prepare four rows each.
template <int G, bool BF16>
__global__ __launch_bounds__(256) void k_lg_prep(LgRoute rt, uint32_t nb_route, const void* __restrict__ x,
                                                 uint32_t rows, uint32_t K, uint8_t* __restrict__ limbs,
                                                 float* __restrict__ xsum, int32_t* __restrict__ xexp) {
  extern __shared__ __attribute__((aligned(16))) uint32_t ids[];
  if (blockIdx.x < nb_route) {
    lg_route_block(rt, blockIdx.x, ids);
    return;
  }
  const uint32_t r = (blockIdx.x - nb_route) * 4 + (threadIdx.x >> 6);
  if (r < rows) lg_prep_row<G, BF16>(x, r, K, limbs, xsum, xexp, threadIdx.x & 63);
}

// ---------------------------------------------------------------------------
// The GEMM. A block is four waves: KS of them split K (step st to wave st
// mod KS, so that the waves' loads of a row lie side by side), 4 / KS split
// the columns. A wave holds NT column tiles of 16 (gate/up: NT / 2 gate and
// as many up tiles) over the item's 16 rows; lane (c, kb) = (l % 16, l / 16)
// loads the 32-code chunk kb of a step from weight row c of each tile and
// the limbs of row c, one step ahead, straight into registers (no block
// barrier in the loop). The scales and biases of the block's columns, one
// contiguous range each, are copied to LDS as they are.
//
// What bounds it: the fold of the limb sums (24 VALU instructions per tile
// and group of 64, 33 with the unpacking, against 4 MFMAs) and, with two
// waves per SIMD, what a unit spends before its first step. 512 tokens,
// 2560 x 640, 512 experts, top-10 (654 items of 16 rows), traced: gate/up 326 us
// (305 at least), down 170 (161); counters: VALU busy 57 % and 51 %, matrix
// cores 23 % and 22 %; HBM reads run at 2.5 TB/s.
// Steps, gate/up us: operand-order loads (64 cache accesses per load instead
// of 16) 455; memory-order loads and a lane permute 367; the next group's
// MFMAs ahead of a fold, one set of weight registers re-filled tile by tile
// 359; bias first and two sums per output 350; the scales' loads together 335.
// ---------------------------------------------------------------------------
struct LgArgs {
  const uint8_t* base;  // expert e at base + e * stride
  uint64_t stride;
  uint64_t w[2], s[2], b[2];  // gate / up (or one matrix in [0]) from the expert's base
  uint32_t cols, K;     // weight rows of each matrix, inputs
  const uint8_t* limbs;
  const float* xsum;
  const int32_t* xexp;
  const uint2* items;        // null: dense, item i = rows 16 i ..
  const uint32_t* item_tok;  // limb row of each item row, or null: the entry itself
  uint32_t n_items, n_rows, ncb;
  float* out;           // [entries, cols]
};

__device__ __forceinline__ i32x4 mfma_i8(u32x4 a, u32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

// Over 32 inputs: eight of each lane.
__device__ __forceinline__ i32x4 mfma_i8_32(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)a1 << 32) | a0), (long)(((uint64_t)b1 << 32) | b0), c, 0, 0, 0);
}

// The 4 x 4 words (lane block of 16, register) transposed.
__device__ __forceinline__ void transpose4(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
  const auto ac = __builtin_amdgcn_permlane32_swap(a, c, false, false);
  const auto bd = __builtin_amdgcn_permlane32_swap(b, d, false, false);
  const auto ab = __builtin_amdgcn_permlane16_swap(ac[0], bd[0], false, false);
  const auto cd = __builtin_amdgcn_permlane16_swap(ac[1], bd[1], false, false);
  a = ab[0], b = ab[1], c = cd[0], d = cd[1];
}

// LDS bytes of the scales (or biases) of `rows` weight rows: 16-byte pieces.
__host__ __device__ constexpr uint32_t lg_scale_lds(uint32_t rows, uint32_t gpr) { return (rows * gpr * 2 + 15) / 16 * 16; }

template <int BITS, int G, bool GU, int KS, int NT>
__global__ __launch_bounds__(256, 2) void k_lg(LgArgs a) {
  constexpr int CB = chunk_bytes<BITS>();
  constexpr int NS = 4 / KS;                    // column shares
  constexpr int NM = GU ? 2 : 1, TM = NT / NM;  // matrices, tiles of each per wave
  constexpr int COLW = TM * 16, COLB = NS * COLW;  // columns per wave, per block
  constexpr uint32_t GS = kLgKC / G;            // groups per step
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t c16 = lane & 15, kb = lane >> 4;
  // XCD x = blockIdx % 8 takes a contiguous range of the units (item
  // slowest), so an item's column blocks share their rows, and an expert's
  // items its weights, in one L2.
  const uint32_t total = a.n_items * a.ncb, per = (total + 7) / 8;
  const uint32_t u = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || u >= total) return;
  const uint32_t item = u / a.ncb, cb = u % a.ncb;
  uint32_t e = 0, start = item * kLgM, cnt, tok = 0;
  if (a.items) {
    if (a.item_tok) tok = a.item_tok[item * kLgM + c16];
    const uint2 it = a.items[item];
    e = __builtin_amdgcn_readfirstlane(it.x);
    start = __builtin_amdgcn_readfirstlane(it.y & 0xFFFFu);
    cnt = __builtin_amdgcn_readfirstlane(it.y >> 16);
    if (cnt == 0) return;
  } else {
    cnt = min(kLgM, a.n_rows - start);
  }
  const uint32_t K = a.K, cols = a.cols, KP = lg_kp(K), nst = KP / kLgKC, cpr = K / kChunk;
  const uint32_t gpr = K / G, gp = lg_gp(K, G);
  const uint32_t ROWB = cpr * CB;
  const uint8_t* const blob = a.base + (uint64_t)e * a.stride;
  const uint32_t ks = wave % KS, ns = wave / KS;
  const uint32_t colb = cb * COLB;                       // the block's first column
  const uint32_t rowsb = min((uint32_t)COLB, cols - colb);  // its weight rows per matrix
  const uint32_t row0 = min(ns * COLW, rowsb - 1);       // the wave's first of them (clamped)

  // Limb row of this lane's A row (rows past the count repeat the last).
  const uint32_t rl = min(c16, cnt - 1);
  const uint32_t arow = a.item_tok ? (uint32_t)__shfl((int)tok, (int)rl, kWave) : start + rl;
  // Loads are made in memory order, four lanes per row's 64 (48) bytes (lane
  // order 4 row + part: one cache access per four lanes, where the operand
  // order would take one per lane), and a lane permute brings each row's
  // parts to the operand's lanes (c, kb).
  const uint32_t lr = lane >> 2, lp = lane & 3;
  const int psrc = (int)((c16 * 4 + kb) * 4);
  const uint32_t lrow = a.item_tok ? (uint32_t)__shfl((int)tok, (int)min(lr, cnt - 1), kWave) : start + min(lr, cnt - 1);
  const uint8_t* const ap = a.limbs + (uint64_t)lrow * KP * 4 + lp * 16;
  const float* const xs = a.xsum + (uint64_t)arow * gp;
  const int32_t fexp = a.xexp[arow];

  uint32_t roff[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) roff[t] = min(row0 + t * 16u + lr, rowsb - 1) * ROWB;
  const uint8_t* wp[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) wp[m] = blob + a.w[m] + (uint64_t)colb * ROWB;

  // Scales then biases of the block's rows, per matrix: LDS [m][s, b][row][gpr].
  const uint32_t seg = lg_scale_lds(COLB, gpr), bytes = rowsb * gpr * 2;
  const uint8_t* sb[2 * NM];
  uintptr_t al = 0;
#pragma unroll
  for (int m = 0; m < 2 * NM; ++m) {
    sb[m] = blob + (m & 1 ? a.b[m / 2] : a.s[m / 2]) + (uint64_t)colb * gpr * 2;
    al |= (uintptr_t)sb[m];
  }
  // 16-byte pieces of all of them as one list, SU loads per thread in flight
  // (one at a time, each waited for by its LDS write, took 5.4 us of a
  // unit's 22 at 2560 x 640); then what is left of each by two bytes.
  const uint32_t whole = al % 16 == 0 ? bytes / 16 : 0u;
  constexpr uint32_t SU = NT >= 8 ? 6 : 2;
  for (uint32_t p0 = tid; p0 < whole * 2 * NM; p0 += 256 * SU) {
    u32x4 v[SU];
    uint32_t dst[SU];
#pragma unroll
    for (uint32_t j = 0; j < SU; ++j) {
      uint32_t i = min(p0 + 256 * j, whole * 2 * NM - 1), m = 0;
      const uint8_t* src = sb[0];
#pragma unroll
      for (int k = 1; k < 2 * NM; ++k)
        if (i >= whole) i -= whole, m = k, src = sb[k];
      v[j] = *reinterpret_cast<const u32x4*>(src + i * 16);
      dst[j] = m * seg + i * 16;
    }
#pragma unroll
    for (uint32_t j = 0; j < SU; ++j) *reinterpret_cast<u32x4*>(lds + dst[j]) = v[j];
  }
#pragma unroll
  for (int m = 0; m < 2 * NM; ++m)
    for (uint32_t i = whole * 16 + tid * 2; i < bytes; i += 512)
      *reinterpret_cast<uint16_t*>(lds + m * seg + i) = *reinterpret_cast<const uint16_t*>(sb[m] + i);

  // Group sums of the bias term, four of this wave's groups per MFMA: lane
  // block kb of batch q takes the (4 q + kb)-th; zero past the last.
  auto bias_group = [&](uint32_t q) { return (ks + (4 * q + kb) / GS * KS) * GS + (4 * q + kb) % GS; };
  constexpr uint32_t QB = 4;  // batches per round of loads
  auto load_sums = [&](uint32_t q, float(&v)[QB]) {
#pragma unroll
    for (uint32_t j = 0; j < QB; ++j) {
      const uint32_t g = bias_group(q + j);
      const float sum = xs[min(g, nst * GS - 1)];
      v[j] = g < nst * GS ? sum : 0.f;
    }
  };
  Raw<BITS> w[NT];
  auto issue_w = [&](uint32_t off, int t) { w[t] = load_raw<BITS, false>(wp[t / TM] + lane_off(roff[t % TM] + off)); };
  auto w_off = [&](uint32_t st) { return min(st * 4 + lp, cpr - 1) * CB; };
  u32x4 rw[2][4], x[2][4];  // the step's rows as loaded, and in operand order
  auto issue_x = [&](uint32_t st) {
    const uint8_t* p = ap + (uint64_t)st * 512;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int L = 0; L < 4; ++L) rw[h][L] = *reinterpret_cast<const u32x4*>(p + (h * 4 + L) * 64);
  };

  float xv[QB];
  load_sums(0, xv);
  const uint32_t last = ks < nst ? (nst - 1 - ks) / KS * KS + ks : 0u;  // this wave's last step
  if (ks < nst) {
    issue_x(ks);
    const uint32_t off = w_off(ks);
#pragma unroll
    for (int t = 0; t < NT; ++t) issue_w(off, t);
  }
  // The copies above are in LDS once their writes have completed; the loads
  // of the first step stay in flight across the barrier.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // Two sums per output where a step has several groups (even and odd
  // groups): half the additions of one at the size of the whole sum.
  f32x4 tot[NT], odd[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) tot[t] = odd[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t srow[TM];  // LDS element of the lane's rows
#pragma unroll
  for (int t = 0; t < TM; ++t) srow[t] = min(row0 + t * 16u + c16, rowsb - 1) * gpr;
  auto scale = [&](int t, int arr, uint32_t g) {
    const uint16_t* const p = reinterpret_cast<const uint16_t*>(lds + (2 * (t / TM) + arr) * seg);
    return bf16f(p[srow[t % TM] + min(g, gpr - 1)]);
  };
  // The bias term first, while the sums are small: in the loop each step's
  // would round at the size of the whole sum.
  for (uint32_t q = 0; q * 4 < (nst - min(ks, nst) + KS - 1) / KS * GS; q += QB) {
    if (q) load_sums(q, xv);
#pragma unroll
    for (uint32_t j = 0; j < QB; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        tot[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j], scale(t, 1, bias_group(q + j)), tot[t], 0, 0, 0);
  }
  auto perm = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(psrc, (int)v); };
  // A tile's codes as the two B operands of a step.
  auto operands = [&](const Raw<BITS>& raw, u32x4 (&b)[2]) {
    Raw<BITS> w;
#pragma unroll
    for (int i = 0; i < BITS; ++i) w.d[i] = perm(raw.d[i]);
    if constexpr (G == 64 && BITS == 4) {
      // Chunk halves of lanes kb and kb + 2 exchanged: operand h lies in
      // group h.
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(w.d[i], w.d[i + 2], false, false);
        w.d[i] = r[0];
        w.d[i + 2] = r[1];
      }
    }
    // Word i of the four lanes' chunks (one group each) to lane block i, as
    // register (group).
    if constexpr (G == 32 && BITS == 4) transpose4(w.d[0], w.d[1], w.d[2], w.d[3]);
    uint32_t q[8];
    unpack_bytes(w, q);
    if constexpr (G == 64 && BITS == 3) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(q[i], q[i + 4], false, false);
        q[i] = r[0];
        q[i + 4] = r[1];
      }
    }
    if constexpr (G == 32 && BITS == 3) {
      transpose4(q[0], q[2], q[4], q[6]);
      transpose4(q[1], q[3], q[5], q[7]);
    }
    b[0] = u32x4{q[0], q[1], q[2], q[3]};
    b[1] = u32x4{q[4], q[5], q[6], q[7]};
  };
  // The limb sums of group g (of the step's GS) of a tile.
  auto sums = [&](const u32x4 (&b)[2], uint32_t g, i32x4 (&S)[4]) {
    const i32x4 z = {0, 0, 0, 0};
    if constexpr (G == 64) {
#pragma unroll
      for (int L = 0; L < 4; ++L) S[L] = mfma_i8(x[g][L], b[g], z);
    } else if constexpr (G == 32) {
      const uint32_t h = g / 2, o = g % 2 * 2;
#pragma unroll
      for (int L = 0; L < 4; ++L) S[L] = mfma_i8_32(x[h][L][o], x[h][L][o + 1], b[h][o], b[h][o + 1], z);
    } else {
#pragma unroll
      for (int L = 0; L < 4; ++L) S[L] = mfma_i8(x[0][L], b[0], z);
#pragma unroll
      for (int L = 0; L < 4; ++L) S[L] = mfma_i8(x[1][L], b[1], S[L]);
    }
  };
  auto fold = [&](const i32x4 (&S)[4], float s, f32x4& acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int32_t lo = S[0][i] + (int32_t)((uint32_t)S[1][i] << 8);
      const int32_t hi = S[2][i] + (int32_t)((uint32_t)S[3][i] << 8);
      acc[i] = __builtin_fmaf(s, __builtin_fmaf((float)hi, 65536.f, (float)lo), acc[i]);
    }
  };
  for (uint32_t st = ks; st < nst; st += KS) {
    // The next step's loads go out as the registers they land in are read,
    // the rows' here, a tile's when it becomes an operand (past the last
    // step: the last again), and are in flight while the step is computed.
    const uint32_t ahead = min(st + KS, last), off = w_off(ahead);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int L = 0; L < 4; ++L)
        x[h][L] = u32x4{perm(rw[h][L].x), perm(rw[h][L].y), perm(rw[h][L].z), perm(rw[h][L].w)};
    issue_x(ahead);
    // (tile, group) pairs, group fastest: the next pair's limb sums are on
    // the matrix cores while a pair's are folded.
    constexpr int NU = NT * (int)GS;
    u32x4 b[2][2];
    i32x4 S[2][4];
    operands(w[0], b[0]);
    issue_w(off, 0);
    sums(b[0], 0, S[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int t = i / (int)GS, tn = (i + 1) / (int)GS;
      if (i % (int)GS == 0 && t + 1 < NT) {
        operands(w[t + 1], b[(t + 1) & 1]);
        issue_w(off, t + 1);
      }
      if (i + 1 < NU) sums(b[tn & 1], (i + 1) % GS, S[(i + 1) & 1]);
      fold(S[i & 1], scale(t, 0, st * GS + i % GS), i % (int)GS % 2 ? odd[t] : tot[t]);
      __builtin_amdgcn_sched_barrier(0);  // keeps the later tiles' operands out of the registers
    }
  }

  if constexpr (GS > 1) {
#pragma unroll
    for (int t = 0; t < NT; ++t) tot[t] += odd[t];
  }

  // K shares added through LDS (over the scales), tiles spread over the
  // waves; with KS = 1 each wave finishes its own.
  int32_t f[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = -__shfl(fexp, (int)(4 * kb + i), kWave);
  auto finish = [&](f32x4 v0, f32x4 v1, uint32_t col) {
    if (col >= cols) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t r = 4 * kb + i;
      if (r >= cnt) continue;
      const float y0 = __builtin_ldexpf(v0[i], f[i]);
      a.out[(uint64_t)(start + r) * cols + col] = GU ? silu_mul(y0, __builtin_ldexpf(v1[i], f[i])) : y0;
    }
  };
  if constexpr (KS == 1) {
#pragma unroll
    for (int t = 0; t < TM; ++t) finish(tot[t], tot[GU ? TM + t : t], colb + ns * COLW + t * 16 + c16);
  } else {
    __syncthreads();
    f32x4* const red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int t = 0; t < NT; ++t) red[(wave * NT + t) * 64 + lane] = tot[t];
    __syncthreads();
    auto sum = [&](uint32_t share, uint32_t t) {
      const f32x4* const p = red + ((share * KS) * NT + t) * 64 + lane;
      if constexpr (KS == 4)
        return (p[0] + p[NT * 64]) + (p[2 * NT * 64] + p[3 * NT * 64]);
      else
        return p[0] + p[NT * 64];
    };
    for (uint32_t i = wave; i < NS * TM; i += 4) {
      const uint32_t share = i / TM, t = i % TM;
      const f32x4 v0 = sum(share, t);
      finish(v0, GU ? sum(share, TM + t) : v0, colb + share * COLW + t * 16 + c16);
    }
  }
}

// out[t] = sum of t's entries in ascending expert order (moe_cpu.rs:330-337).
template <uint32_t MAXK>
__global__ __launch_bounds__(256) void k_lg_combine(const uint2* __restrict__ tok_pw, uint32_t k, uint32_t H,
                                                    const float* __restrict__ down, float* __restrict__ out) {
  const uint32_t t = blockIdx.x;
  uint32_t pos[MAXK];
  float w[MAXK];
#pragma unroll
  for (uint32_t r = 0; r < MAXK; ++r) {
    const uint2 pw = tok_pw[t * k + (r < k ? r : k - 1)];
    pos[r] = pw.x;
    w[r] = __uint_as_float(pw.y);
  }
  for (uint32_t h = threadIdx.x * 4; h < H; h += 1024) {
    f32x4 d[MAXK];
#pragma unroll
    for (uint32_t r = 0; r < MAXK; ++r) d[r] = *reinterpret_cast<const f32x4*>(down + (uint64_t)pos[r] * H + h);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (uint32_t r = 0; r < MAXK; ++r)
      if (r < k)
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = __builtin_fmaf(d[r][c], w[r], o[c]);
    *reinterpret_cast<f32x4*>(out + (uint64_t)t * H + h) = o;
  }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
static uint64_t al256(uint64_t n) { return (n + 255) & ~255ull; }

// Limbs, group sums and exponents of `rows` rows of K inputs.
struct LgRows {
  uint8_t* limbs;
  float* xsum;
  int32_t* xexp;
};
static uint64_t lg_rows_bytes(uint64_t rows, uint32_t K, uint32_t G, uint8_t* base, LgRows* r) {
  const uint64_t lb = al256(rows * lg_kp(K) * 4), sb = al256(rows * lg_gp(K, G) * 4);
  if (r) {
    r->limbs = base;
    r->xsum = reinterpret_cast<float*>(base + lb);
    r->xexp = reinterpret_cast<int32_t*>(base + lb + sb);
  }
  return lb + sb + al256(rows * 4);
}

static hipError_t lg_prep(const LgRoute* rt, const void* x, bool bf16, uint32_t rows, uint32_t K, uint32_t G,
                          const LgRows& r, hipStream_t st) {
  const LgRoute none{};
  const uint32_t N = rt ? rt->n * rt->k : 0, nb = (N + kLgRouteE - 1) / kLgRouteE;
  const uint32_t lds = (N + 3) / 4 * 16;
  const dim3 grid(nb + (rows + 3) / 4);
  auto go = [&](auto fn) {
    hipLaunchKernelGGL(fn, grid, dim3(256), lds, st, rt ? *rt : none, nb, x, rows, K, r.limbs, r.xsum, r.xexp);
    return hipGetLastError();
  };
  if (bf16) return G == 32 ? go(k_lg_prep<32, true>) : G == 64 ? go(k_lg_prep<64, true>) : go(k_lg_prep<128, true>);
  return G == 32 ? go(k_lg_prep<32, false>) : G == 64 ? go(k_lg_prep<64, false>) : go(k_lg_prep<128, false>);
}

template <int BITS, int G, bool GU, int KS, int NT>
static hipError_t lg_inst(LgArgs a, hipStream_t st) {
  constexpr uint32_t NS = 4 / KS, CW = NS * (GU ? NT / 2 : NT) * 16;
  a.ncb = (a.cols + CW - 1) / CW;
  const uint32_t scales = (GU ? 4 : 2) * lg_scale_lds(CW, a.K / G), red = KS > 1 ? 4 * NT * 64 * 16 : 0;
  const uint32_t lds = scales > red ? scales : red;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> raised{0};
    const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(&k_lg<BITS, G, GU, KS, NT>), 160 * 1024, raised);
    if (e != hipSuccess) return e;
  }
  const uint32_t per = (a.n_items * a.ncb + 7) / 8;
  hipLaunchKernelGGL((k_lg<BITS, G, GU, KS, NT>), dim3(8 * per), dim3(256), lds, st, a);
  return hipGetLastError();
}

constexpr uint32_t kLgRound = 512;  // blocks resident at once: two on each CU

template <int BITS, int G, bool GU>
static hipError_t lg_shape(const LgArgs& a, hipStream_t st) {
  // Narrow waves (2, then 4 tiles) while their blocks fit the chip at once:
  // a small call is the latency of its steps, and a step of 8 tiles takes
  // 2.5 us (16 rows, 2048 -> 4096: 10.8 us with 2 tiles, 13.1 with 4, 17.8
  // with 8; 128 rows 20.9, 18.4, 20.1; 256 rows 32.5, 27.0, 26.2). K is
  // split over the block's waves as well, but for calls of more blocks with
  // less than two steps per wave, whose waves split the columns (2560 x 640
  // down, 512 tokens: 178 us against 270).
  auto blocks = [&](uint32_t nt) { return a.n_items * ((a.cols * (GU ? 2 : 1) + nt * 16 - 1) / (nt * 16)); };
  if (blocks(2) <= kLgRound) return lg_inst<BITS, G, GU, 4, 2>(a, st);
  if (blocks(4) <= kLgRound) return lg_inst<BITS, G, GU, 4, 4>(a, st);
  if (a.K >= 1024 || blocks(8) <= kLgRound) return lg_inst<BITS, G, GU, 4, 8>(a, st);
  return lg_inst<BITS, G, GU, 1, 8>(a, st);
}

template <bool GU>
static hipError_t lg_gemm(const LgArgs& a, uint32_t bits, uint32_t G, hipStream_t st) {
  if (bits == 4)
    return G == 32 ? lg_shape<4, 32, GU>(a, st) : G == 64 ? lg_shape<4, 64, GU>(a, st) : lg_shape<4, 128, GU>(a, st);
  return G == 32 ? lg_shape<3, 32, GU>(a, st) : G == 64 ? lg_shape<3, 64, GU>(a, st) : lg_shape<3, 128, GU>(a, st);
}

// Dense: y[n, out_dim] = x[n, in_dim] . dequant(W)^T.
uint64_t limb_qmm_workspace(uint32_t in_dim, uint32_t group, uint32_t n_tokens) {
  return lg_rows_bytes(n_tokens, in_dim, group, nullptr, nullptr);
}

// Whether the limb GEMM is the faster one where k_pf_mm has tiles too (at
// most 8192 inputs). k_pf_mm walks units of 32 rows x 256 columns, the busiest
// block `units` of them one after another, each with its whole K as latency;
// the limb GEMM runs rounds of 512 blocks of 16 rows x 128 columns. Measured over
// 8700 random calls (2 to 1024 rows, 256 to 150000 columns, 256 to 8192 inputs,
// all groups and bits): where a block has several units, a round of limb blocks
// per unit is no slower (time against k_pf_mm's 0.5 to 1.09). With one unit it
// is the faster up to 128 blocks (0.25 to 1.0); up to 256 from 512 inputs on
// (0.42 to 1.0; 256 inputs, 4 bits 0.9 to 1.15); a whole round (to 512) where a
// unit costs enough: groups of 64 and 128 from 2048 inputs on (0.66 to 1.09) or,
// 3 bits, 1024 (0.7 to 0.97), groups of 32 only with 3 bits from 2048 on (0.83
// to 1.07; 4 bits 0.93 to 1.2); past a round never (1.0 to 2.2). Asking only for
// 128 rows or one round took one call in twelve over its start, by up to 2.2
// times (82 rows 2048 -> 16896, group 32: 80 us against 38).
bool limb_qmm_faster(uint32_t out_dim, uint32_t in_dim, uint32_t group, uint32_t bits, uint32_t n, uint32_t units) {
  const uint64_t blocks = (uint64_t)((n + kLgM - 1) / kLgM) * ((out_dim + 127) / 128);
  if (in_dim > 8192 || (n > 128 && blocks > (in_dim < 1024 ? kLgRound / 2 : kLgRound))) return false;
  if (units > 1) return blocks <= (uint64_t)kLgRound * units;
  const bool large = group > 32, three = bits == 3;
  if (blocks <= kLgRound / 4) return true;
  if (blocks <= kLgRound / 2) return in_dim >= 512 || (three && large);
  return blocks <= kLgRound && (large || three) && in_dim >= (large && three ? 1024u : 2048u);
}

// Whether two rows of a shape without tiles are faster on k_qmv, one after the
// other (three or more never were: 1.05 to 3.8 times the limb GEMM's time).
// Time of two k_qmv calls against it, group 32: up to 4096 columns 0.73 to 0.97
// where k_qmv's lanes are mostly full (1056 to 4096 inputs, from 5664 on), 1.09
// to 1.3 up to 1024 inputs, 1.1 for 4128 to 5600; from 4096 to 16384 columns 1.0
// to 2.6; wider, up to 2048 inputs, 0.83 to 0.97 (1056 on, or 160 on past 32768
// columns: 0.82 to 0.98), else 0.9 to 1.7. Groups of 64 and 128: 0.9 to 0.98 at
// 1056 to 2048 inputs and up to 4096 columns, 0.97 to 3 elsewhere.
bool qmm_two_rows_faster(uint32_t out_dim, uint32_t in_dim, uint32_t group) {
  if (out_dim <= 4096) return in_dim > 1024 && (in_dim <= 2048 || (group == 32 && (in_dim <= 4096 || in_dim > 5632)));
  return group == 32 && out_dim > 16384 && in_dim <= 2048 && in_dim > (out_dim > 32768 ? 128u : 1024u);
}

hipError_t launch_limb_qmm(const QView& w, const float* x, float* y, uint32_t out_dim, uint32_t in_dim, uint32_t n,
                           uint8_t* ws, hipStream_t st) {
  LgRows r;
  lg_rows_bytes(n, in_dim, w.group, ws, &r);
  const hipError_t e = lg_prep(nullptr, x, false, n, in_dim, w.group, r, st);
  if (e != hipSuccess) return e;
  LgArgs a{};
  a.base = w.codes;
  a.s[0] = (uint64_t)((const uint8_t*)w.scales - w.codes);
  a.b[0] = (uint64_t)((const uint8_t*)w.biases - w.codes);
  a.cols = out_dim;
  a.K = in_dim;
  a.limbs = r.limbs;
  a.xsum = r.xsum;
  a.xexp = r.xexp;
  a.n_items = (n + kLgM - 1) / kLgM;
  a.n_rows = n;
  a.out = y;
  return lg_gemm<false>(a, w.bits, w.group, st);
}

struct LgPrefill {
  LgRows x, act;
  uint2* items;
  uint32_t* item_tok;
  uint2* tok_pw;
  float *actf, *down;
};
static uint64_t lg_prefill_layout(uint32_t H, uint32_t I, uint32_t G, uint32_t n, uint32_t E, uint32_t k,
                                  uint8_t* base, LgPrefill* p) {
  const uint64_t N = (uint64_t)n * k;
  uint64_t off = 0;
  auto take = [&](uint64_t bytes) {
    uint8_t* const q = base ? base + off : nullptr;
    off += al256(bytes);
    return q;
  };
  LgPrefill l{};
  l.items = reinterpret_cast<uint2*>(take((uint64_t)lg_slots((uint32_t)N, E) * 8));
  l.item_tok = reinterpret_cast<uint32_t*>(take((uint64_t)lg_slots((uint32_t)N, E) * kLgM * 4));
  l.tok_pw = reinterpret_cast<uint2*>(take(N * 8));
  l.actf = reinterpret_cast<float*>(take(N * I * 4));
  l.down = reinterpret_cast<float*>(take(N * H * 4));
  off += lg_rows_bytes(n, H, G, base ? base + off : nullptr, base ? &l.x : nullptr);
  off += lg_rows_bytes(N, I, G, base ? base + off : nullptr, base ? &l.act : nullptr);
  if (p) *p = l;
  return off;
}

uint64_t limb_prefill_workspace(uint32_t hidden, uint32_t inter, uint32_t group, uint32_t n_tokens,
                                uint32_t n_experts, uint32_t k) {
  return lg_prefill_layout(hidden, inter, group, n_tokens, n_experts, k, nullptr, nullptr);
}

hipError_t launch_limb_prefill(const BlobGeom& g, const uint8_t* experts, uint64_t stride, uint32_t E,
                               const int32_t* idx, const float* w, const void* x, bool x_bf16, uint32_t n, uint32_t k,
                               float* out, uint8_t* ws, uint32_t* err, hipStream_t st) {
  LgPrefill p;
  lg_prefill_layout(g.hidden, g.inter, g.group, n, E, k, ws, &p);
  const uint32_t N = n * k;
  const LgRoute rt{idx, w, n, k, E, lg_slots(N, E), p.items, p.item_tok, p.tok_pw, err};
  hipError_t e = lg_prep(&rt, x, x_bf16, n, g.hidden, g.group, p.x, st);
  if (e != hipSuccess) return e;
  LgArgs a{};
  a.base = experts;
  a.stride = stride;
  for (int m = 0; m < 2; ++m) a.w[m] = g.w[m], a.s[m] = g.s[m], a.b[m] = g.b[m];
  a.cols = g.inter;
  a.K = g.hidden;
  a.limbs = p.x.limbs;
  a.xsum = p.x.xsum;
  a.xexp = p.x.xexp;
  a.item_tok = p.item_tok;
  a.items = p.items;
  a.n_items = rt.n_slots;
  a.out = p.actf;
  e = lg_gemm<true>(a, g.bits, g.group, st);
  if (e != hipSuccess) return e;
  e = lg_prep(nullptr, p.actf, false, N, g.inter, g.group, p.act, st);
  if (e != hipSuccess) return e;
  a.w[0] = g.w[2], a.s[0] = g.s[2], a.b[0] = g.b[2];
  a.cols = g.hidden;
  a.K = g.inter;
  a.limbs = p.act.limbs;
  a.xsum = p.act.xsum;
  a.xexp = p.act.xexp;
  a.item_tok = nullptr;
  a.out = p.down;
  e = lg_gemm<false>(a, g.bits, g.group, st);
  if (e != hipSuccess) return e;
  if (k <= 8)
    hipLaunchKernelGGL(k_lg_combine<8>, dim3(n), dim3(256), 0, st, p.tok_pw, k, g.hidden, p.down, out);
  else
    hipLaunchKernelGGL(k_lg_combine<16>, dim3(n), dim3(256), 0, st, p.tok_pw, k, g.hidden, p.down, out);
  return hipGetLastError();
}

}  // namespace smoe
