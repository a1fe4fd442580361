// phase.hip — the expert FFN of one token as two kernels (gfx950), any width.
//
//   k_ph_gateup   gate + up + SwiGLU of every slot in the table (routed slots
//                 and the shared expert).
//   k_ph_route    the same with the routing in the launch.
//   k_ph_down     down rows of every slot, combined in slot order with the
//                 shared term and the residual.
//
// Both keep their activations (the hidden vector, the slots' SwiGLU outputs)
// in LDS as 31-bit block floating point, one exponent per 32 values, in four
// int8 limbs, written once per block while the weights are in flight: a
// code then costs one byte unpack and four v_dot4c_i32_i8 per four inputs,
// the sums of a chunk's limbs are exact and a chunk is rounded once, to f32. A
// value is off by at most 2^-31 of its chunk's power of two (2^-30 of the
// largest of its 32), and keeps its 24 bits down to 2^-6 of that.
// Traced per launch, 2560 x 640 (512 experts, top-10, shared expert): 13.4 us
// with the routing in the launch + 12.4; 2048 x 512 top-8: 5.1 + 6.6.
// Converting codes to floats for FMAs, with every wave loading the activations
// again, took 11.4 + 21.6 (and a routing launch of 11) and 6.4 + 8.7. What is
// left is a launch, the table's and the rows' round trips and the dots after
// them, at an eighth (2048 x 512) to half (7168 x 2048) of the HBM rate.
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "topk.h"

namespace smoe {

constexpr int kL4Words = 36;  // LDS dwords per chunk: 32 of limbs, scale, sum, pad (conflict-free 16-byte reads)

struct Limbs4 {
  uint32_t w[4][8];
  float scale, xs;
};

// A chunk's values as limbs, four lanes per chunk (lane q of the quad holds
// values 8 q .. 8 q + 7): x_j = m_j 2^-f, |m_j| <= 2^30, bytes in the order of
// unpack_bytes. f <= 149: 2^-f is a float, and at 149 every m_j is exact. A
// chunk with an infinity: its finite values 0, the infinities +-2^30 at a scale
// of infinity, so that a product is infinite or NaN as an f32 one is (a NaN
// comes from the sum xs). live: store.
__device__ __forceinline__ void store_limbs4_quad(uint32_t* dst, const float (&x)[8], int q, bool live) {
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(x[j]));
  amax = fmaxf(amax, dpp_f<0xB1>(amax, 0.f));
  amax = fmaxf(amax, dpp_f<0x4E>(amax, 0.f));
  const bool inf = amax == INFINITY;
  const int f = inf ? -200 : amax > 0.f ? min(30 - __builtin_amdgcn_frexp_expf(amax), 149) : 0;
  int32_t d[4][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = __builtin_amdgcn_fmed3f(__builtin_ldexpf(x[j], f), -0x1p30f, 0x1p30f);
    const int32_t m = (int32_t)__builtin_rintf(v);
    const int32_t d0 = (int32_t)((uint32_t)m << 24) >> 24, m1 = (m - d0) >> 8;
    const int32_t d1 = (int32_t)((uint32_t)m1 << 24) >> 24, m2 = (m1 - d1) >> 8;
    const int32_t d2 = (int32_t)((uint32_t)m2 << 24) >> 24;
    d[0][j] = d0, d[1][j] = d1, d[2][j] = d2, d[3][j] = (m2 - d2) >> 8;
  }
  float xs = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  xs += dpp_f<0xB1>(xs, 0.f);
  xs += dpp_f<0x4E>(xs, 0.f);
  if (!live) return;
#pragma unroll
  for (int L = 0; L < 4; ++L)
    *reinterpret_cast<uint2*>(dst + 8 * L + 2 * q) = make_uint2(
        pack_bytes(d[L][0], d[L][2], d[L][4], d[L][6]), pack_bytes(d[L][1], d[L][3], d[L][5], d[L][7]));
  if (q == 0) *reinterpret_cast<uint2*>(dst + 32) = make_uint2(__float_as_uint(inf ? INFINITY : __builtin_ldexpf(1.0f, -f)), __float_as_uint(xs));
}

__device__ __forceinline__ void load_limbs4(const uint32_t* p, Limbs4& o) {
  const u32x4* p4 = reinterpret_cast<const u32x4*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const u32x4 v = p4[i];
#pragma unroll
    for (int c = 0; c < 4; ++c) o.w[i / 2][(i % 2) * 4 + c] = v[c];
  }
  const uint2 t = *reinterpret_cast<const uint2*>(p + 32);
  o.scale = __uint_as_float(t.x);
  o.xs = __uint_as_float(t.y);
}

// s * sum_j q_j x_j + b * sum_j x_j of one chunk.
template <int BITS>
__device__ __forceinline__ float chunk_dot4(const Raw<BITS>& raw, const Limbs4& x, float s, float b) {
  uint32_t q[8];
  unpack_bytes(raw, q);
  int32_t S[4] = {0, 0, 0, 0};
#pragma unroll
  for (int w = 0; w < 8; ++w)
#pragma unroll
    for (int L = 0; L < 4; ++L) S[L] = __builtin_amdgcn_sdot4((int)q[w], (int)x.w[L][w], S[L], false);
  // |S_L| <= 32 * 15 * 128: the pairs are exact in 32 bits and as floats.
  const int32_t lo = S[0] + (int32_t)((uint32_t)S[1] << 8), hi = S[2] + (int32_t)((uint32_t)S[3] << 8);
  return __builtin_fmaf(s, __builtin_fmaf((float)hi, 65536.f, (float)lo) * x.scale, b * x.xs);
}

// The blob of slot s and the table's scalars, from the device table or the
// kernel argument (selects: a lane-indexed argument would go through
// scratch).
__device__ __forceinline__ const uint8_t* slot_blob(const FfnTable* dev, const FfnTable& val, uint32_t s) {
  if (dev) return dev->blob[s];
  const uint8_t* p = val.blob[0];
#pragma unroll
  for (uint32_t i = 1; i < (uint32_t)kMaxSlots; ++i) p = s == i ? val.blob[i] : p;
  return p;
}

// ---------------------------------------------------------------------------
// Gate/up. A wave takes 64 / LR * P rows (gate and up) of one slot: LR lanes
// per row, lane l the chunks l, l + LR, ..., IB of them per round (the last
// round's past the row re-read its last chunk against zero limbs). 16 lanes per
// row, in rounds as long as the row where it has up to 80 chunks, leave at most
// 15 of its chunk places empty, where whole-wave rows of 80 chunks left 48 of
// 128; few long rows take 64 (gateup_shape).
// ---------------------------------------------------------------------------
// x as limbs: a quad of threads per chunk; chunks past the row are zero. All
// of a thread's values are loaded at once, ahead of the weights (up to four
// chunks: rows are at most 256 long and a block has kPhW waves). One round trip
// after another, behind the weights' loads, took 8 slots of 2048 x 512 (gate/up
// and down) 11.8 us against 11.0, of 7168 x 2048 77.0 against 74.7.
constexpr uint32_t kPhW = 4;  // waves per gate/up block
constexpr uint32_t kPhXR = 4;
constexpr uint32_t kPhNQ = kPhW * kWave / 4;  // chunks per round
static_assert(kPhXR * kPhNQ * kChunk >= 8192, "the widest row");

template <int RC>  // the row is padded to a multiple of RC chunks
struct StageX {
  f32x4 v[kPhXR][2];
  static __device__ __forceinline__ uint32_t padded(uint32_t cpr) { return (cpr + RC - 1) / RC * RC; }
  __device__ __forceinline__ void load(const float* x, uint32_t cpr) {
    const uint32_t qd = threadIdx.x >> 2, q = threadIdx.x & 3;
#pragma unroll
    for (uint32_t i = 0; i < kPhXR; ++i) {
      if (i * kPhNQ >= padded(cpr)) break;
      const f32x4* const p = reinterpret_cast<const f32x4*>(x + (size_t)min(qd + i * kPhNQ, cpr - 1) * kChunk + q * 8);
      v[i][0] = p[0];
      v[i][1] = p[1];
    }
  }
  __device__ __forceinline__ void store(uint32_t cpr, uint32_t* limbs) const {
    const uint32_t qd = threadIdx.x >> 2, q = threadIdx.x & 3, n = padded(cpr);
#pragma unroll
    for (uint32_t i = 0; i < kPhXR; ++i) {
      if (i * kPhNQ >= n) break;
      const uint32_t ch = qd + i * kPhNQ;
      const float z[8] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w, v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
      float f[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = ch < cpr ? z[j] : 0.f;
      store_limbs4_quad(limbs + (size_t)min(ch, n - 1) * kL4Words, f, (int)q, ch < n);
    }
  }
};

// STAGE: the limbs are still to be loaded, and written after the weights' loads.
template <int BITS, int P, int IB, int LR, bool STAGE>
__device__ __forceinline__ void ph_gateup_rows(const uint8_t* blob_, const BlobGeom& g, uint32_t row0, uint32_t lane,
                                               const float* x, uint32_t* limbs, float* act) {
  constexpr int CB = chunk_bytes<BITS>();
  const gbytes blob = as_global(blob_);
  const uint32_t cpr = g.hidden / kChunk, gpr = g.hidden >> __builtin_ctz(g.group);
  const uint32_t cps = __builtin_ctz(g.group / kChunk);
  const uint32_t lc = lane % LR, lrow = lane / LR;
  uint32_t row[P];
#pragma unroll
  for (int p = 0; p < P; ++p) row[p] = min(row0 + p * (64 / LR) + lrow, g.inter - 1);
  Raw<BITS> raw[IB][P][2];
  uint32_t sv[IB][P][2], bv[IB][P][2];
  auto load = [&](uint32_t c0) {
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      const uint32_t c = min(c0 + i * LR + lc, cpr - 1);
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          raw[i][p][m] = load_raw_g<BITS>(blob + g.w[m] + (uint64_t)row[p] * (cpr * CB) + c * CB);
          const uint64_t gi = ((uint64_t)row[p] * gpr + (c >> cps)) * 2;
          sv[i][p][m] = gld<false, uint16_t>(blob + g.s[m] + gi);
          bv[i][p][m] = gld<false, uint16_t>(blob + g.b[m] + gi);
        }
    }
  };
  StageX<IB * LR> xs;
  if constexpr (STAGE) xs.load(x, cpr);
  __builtin_amdgcn_sched_barrier(0);
  load(0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (STAGE) xs.store(cpr, limbs);
  // The block's limbs are written; the weights stay in flight.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  float sum[P][2];
#pragma unroll
  for (int p = 0; p < P; ++p) sum[p][0] = sum[p][1] = 0.f;
  for (uint32_t c0 = 0;;) {
#pragma unroll
    for (int i = 0; i < IB; ++i) {
      Limbs4 xl;
      load_limbs4(limbs + (size_t)(c0 + i * LR + lc) * kL4Words, xl);
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int m = 0; m < 2; ++m)
          sum[p][m] += chunk_dot4<BITS>(raw[i][p][m], xl, __uint_as_float(sv[i][p][m] << 16), __uint_as_float(bv[i][p][m] << 16));
      // One chunk's limbs in registers at a time: its dots end here, and the
      // next chunk's reads stay behind them (a scheduling barrier alone left the
      // dots behind the last read: up to 458 registers, one wave per SIMD).
#pragma unroll
      for (int p = 0; p < P; ++p) asm volatile("" : "+v"(sum[p][0]), "+v"(sum[p][1]) : : "memory");
    }
    c0 += LR * IB;
    if (c0 >= cpr) break;
    load(c0);
  }
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const float gs = LR == 16 ? row_sum16_all(sum[p][0]) : group_sum<LR>(sum[p][0]);
    const float us = LR == 16 ? row_sum16_all(sum[p][1]) : group_sum<LR>(sum[p][1]);
    const uint32_t r = row0 + p * (64 / LR) + lrow;
    if (lc == 0 && r < g.inter) act[r] = silu_mul(gs, us);
  }
}

template <int BITS, int P, int IB, int LR, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_ph_gateup(BlobGeom routed, BlobGeom shared, const FfnTable* __restrict__ tab_dev,
                                                        FfnTable tab_val, uint32_t tiles, const float* __restrict__ x,
                                                        float* __restrict__ act) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t slot = blockIdx.x / tiles, row0 = (blockIdx.x % tiles * WPB + wave) * (64 / LR * P);
  const uint32_t k = tab_dev ? tab_dev->k : tab_val.k;
  const uint8_t* const blob = slot_blob(tab_dev, tab_val, slot);
  float* const out = act + (size_t)slot * routed.inter;
  if (slot < k)
    ph_gateup_rows<BITS, P, IB, LR, true>(blob, routed, row0, lane, x, lds, out);
  else
    ph_gateup_rows<4, P, IB, LR, true>(blob, shared, row0, lane, x, lds, out);
}

// ---------------------------------------------------------------------------
// Routing and gate/up in one launch. Every routed wave takes its slot's expert
// itself, the slot-th member of the top-k set in ascending index order
// (topk_slot_logits: softmax is monotone, so the set is that of the logits
// where the margin is clear; else the reference's probabilities and scan).
// The last block finds the reference's slot order and weights, as k_topk
// does, while the others stream their rows: at 512 experts, top-10, its 11 us
// were a launch of their own between the router and the experts (39 -> 32 us
// per layer at 2560 x 640). It writes the table in the order the
// act rows have, and the place of each of the reference's slots in it.
// Grid y: tokens, so that a layer of several is one launch (2560 x 640, 8
// layers, two / four tokens: 503 / 996 us one after another, 320 / 520 so).
// ---------------------------------------------------------------------------
// softmax_ref reads prob in 16-byte pieces, in every element of an array of
// these (one per wave).
template <int PL>
struct RouteLds {
  alignas(16) float prob[64 * PL];
  float val[kMaxK];
  int32_t id[kMaxK], set[kMaxK];
  int32_t is_set;
};

template <int PL>
__device__ void ph_route_table(const float* __restrict__ logits, uint32_t E, uint32_t k, int normalize,
                               const RouteOut& out, uint32_t wave, int lane, RouteLds<PL>& s) {
  float v[PL], l[PL];
#pragma unroll
  for (int e = 0; e < PL; ++e) {
    const uint32_t jt = e * 64 + lane, jl = lane * PL + e;
    v[e] = jt < E ? logits[jt] : -INFINITY;
    l[e] = jl < E ? logits[jl] : -INFINITY;
  }
  // The set on a wave of its own beside the scan (the other waves only meet
  // the barriers: those of softmax_ref, and one after the scan).
  if (wave != 0) {
    if (wave == 1) {
      const bool set = topk_set_logits<PL>(l, E, k, lane, s.set);
      if (lane == 0) s.is_set = set;
    }
    for (int i = 0; i < kSoftmaxBarriers + 1; ++i) __syncthreads();
    return;
  }
  softmax_ref<PL, true>(v, E, lane, s.prob, load_exp_tab(lane));
  exact_topk_t<PL>(v, k, lane, s.id, s.val);
  __syncthreads();
  const int32_t id = lane < (int)k ? s.id[lane] : 0;
  const float sv = lane < (int)k ? s.val[lane] : 0.f;
  // normalize_weights, moe_router.rs:130-141: sequential sum in slot order.
  float w = sv;
  if (normalize) {
    float sum = 0.f;
    for (uint32_t i = 0; i < k; ++i) sum += readlane_f(sv, (int)i);
    if (sum > 0.f) w = sv * (1.0f / sum);
  }
  const bool is_set = s.is_set;
  uint32_t at = is_set ? 0u : (uint32_t)lane;  // place among the ascending indices
  if (is_set)
    for (uint32_t i = 0; i < k; ++i) at += s.set[i] < id ? 1u : 0u;
  if (lane >= (int)k) return;
  if (out.idx) out.idx[lane] = id;
  if (out.weight) out.weight[lane] = w;
  out.table->blob[at] = out.experts + (uint64_t)id * out.stride;
  out.table->weight[at] = w;
  out.table->order[lane] = (uint8_t)at;
  if (lane == 0) {
    out.table->k = k;
    out.table->has_shared = out.shared_blob != nullptr;
    if (out.shared_blob) {
      out.table->blob[k] = out.shared_blob;
      out.table->weight[k] = 1.0f;
      out.table->shared_gate = out.gate_scores ? out.gate_scores[0] : __builtin_nanf("");
    }
  }
}

template <int BITS, int PL, int P, int IB, int LR, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_ph_route(BlobGeom routed, BlobGeom shared, const float* __restrict__ logits,
                                                       uint32_t E, uint32_t k, int normalize, RouteOut ro, uint32_t tiles,
                                                       const float* __restrict__ x, float* __restrict__ act,
                                                       uint32_t lstride, uint32_t astride) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  __shared__ RouteLds<PL> rl[WPB];
  static_assert(alignof(RouteLds<PL>) == 16 && sizeof(RouteLds<PL>) % 16 == 0, "rl[wave].prob is read by 16 bytes");
  const uint32_t t = blockIdx.y;
  logits += (size_t)t * lstride;
  x += (size_t)t * routed.hidden;
  act += (size_t)t * astride;
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t slot = blockIdx.x / tiles, row0 = (blockIdx.x % tiles * WPB + wave) * (64 / LR * P);
  // Every wave of a block goes the same way (they read the same logits), so
  // the barriers inside are met by all of them.
  if (blockIdx.x == gridDim.x - 1) {
    ro.table += t;
    if (ro.idx) ro.idx += (size_t)t * k;
    if (ro.weight) ro.weight += (size_t)t * k;
    if (ro.gate_scores) ro.gate_scores += t;
    ph_route_table<PL>(logits, E, k, normalize, ro, wave, (int)lane, rl[0]);
    return;
  }
  float* const out = act + (size_t)slot * routed.inter;
  if (slot == k) {
    ph_gateup_rows<4, P, IB, LR, true>(ro.shared_blob, shared, row0, lane, x, lds, out);
    return;
  }
  const uint32_t cpr = routed.hidden / kChunk;
  StageX<IB * LR> xs;
  xs.load(x, cpr);
  float l[PL];
#pragma unroll
  for (int e = 0; e < PL / 4; ++e) {
    const f32x4 q = *reinterpret_cast<const f32x4*>(logits + lane * PL + 4 * e);
#pragma unroll
    for (int c = 0; c < 4; ++c) l[4 * e + c] = lane * PL + 4 * e + c < E ? q[c] : -INFINITY;
  }
  xs.store(cpr, lds);
  int32_t id;
  if (!topk_slot_logits<PL>(l, E, k, slot, (int)lane, id)) {
    float v[PL];
#pragma unroll
    for (int e = 0; e < PL; ++e) v[e] = e * 64 + lane < E ? logits[e * 64 + lane] : -INFINITY;
    softmax_ref<PL, true>(v, E, (int)lane, rl[wave].prob, load_exp_tab((int)lane));
    exact_topk_t<PL>(v, k, (int)lane, rl[wave].id, nullptr);
    __syncthreads();
    id = __builtin_amdgcn_readfirstlane(rl[wave].id[slot]);
  }
  ph_gateup_rows<BITS, P, IB, LR, false>(ro.experts + (uint64_t)id * ro.stride, routed, row0, lane, x, lds, out);
}

// ---------------------------------------------------------------------------
// Down + combine. One block per NR hidden rows (8; 4 in blocks of more
// than 8 waves, whose lanes have half the registers, and where 8 would leave
// CUs without a block); a lane owns one (slot,
// chunk) of the flat list of k * inter / 32 and reads it for all the rows, so only
// the last wave has empty lanes; one more wave takes the shared expert's
// chunks (4-bit). The products go to LDS, a thread per (row, slot) adds a
// slot's chunks, and a thread per row combines the slots in the reference's
// order: moe = fma(out_s, w_s, moe) (deferred.rs:458-466), then the shared
// term and the residual.
// ---------------------------------------------------------------------------
template <int BITS, bool NT, uint32_t NR>
struct DownRows {
  Raw<BITS> raw[NR];
  uint32_t s[NR], b[NR];
  __device__ __forceinline__ void load(const uint8_t* blob_, const BlobGeom& g, uint32_t row0, uint32_t c) {
    const gbytes blob = as_global(blob_);
    const uint32_t cpr = g.inter / kChunk, gpr = g.inter >> __builtin_ctz(g.group);
    const uint32_t cg = c >> __builtin_ctz(g.group / kChunk);
#pragma unroll
    for (uint32_t r = 0; r < NR; ++r) {
      const uint32_t row = min(row0 + r, g.hidden - 1);
      raw[r] = load_raw_g<BITS, NT>(blob + g.w[2] + (uint64_t)row * (cpr * chunk_bytes<BITS>()) + c * chunk_bytes<BITS>());
      const uint64_t gi = ((uint64_t)row * gpr + cg) * 2;
      s[r] = gld<false, uint16_t>(blob + g.s[2] + gi);
      b[r] = gld<false, uint16_t>(blob + g.b[2] + gi);
    }
  }
  __device__ __forceinline__ void dot(const uint32_t* limbs, float* part, uint32_t ld) const {
    Limbs4 xl;
    load_limbs4(limbs, xl);
#pragma unroll
    for (uint32_t r = 0; r < NR; ++r)
      part[r * ld] = chunk_dot4<BITS>(raw[r], xl, __uint_as_float(s[r] << 16), __uint_as_float(b[r] << 16));
  }
};

// LDS of k_ph_down: limbs of every chunk, then the products [NR][ld].
__host__ __device__ constexpr uint32_t ph_down_ld(uint32_t chunks) { return chunks | 1u; }
__host__ __device__ constexpr uint32_t ph_down_lds(uint32_t chunks, uint32_t nr) {
  return chunks * kL4Words * 4 + nr * ph_down_ld(chunks) * 4;
}

template <int BITS, uint32_t NR, int TB>
__global__ __launch_bounds__(TB) void k_ph_down(BlobGeom routed, BlobGeom shared, const FfnTable* __restrict__ tab_dev,
                                                  FfnTable tab_val, uint32_t k, uint32_t has_shared,
                                                  const float* __restrict__ act, const float* h_mid,
                                                  const float* __restrict__ shared_out, float* hidden_out,
                                                  int ordered, uint32_t astride) {
  extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
  if (tab_dev) {  // grid y: tokens
    tab_dev += blockIdx.y;
    act += (size_t)blockIdx.y * astride;
    h_mid += (size_t)blockIdx.y * routed.hidden;
    hidden_out += (size_t)blockIdx.y * routed.hidden;
  }
  __shared__ uint8_t sord[kMaxK];
  __shared__ float so[NR][kMaxSlots + 1];
  __shared__ float sw[kMaxSlots];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t I = routed.inter, H = routed.hidden, cpr = I / kChunk;
  const uint32_t items = k * cpr, chunks = (k + has_shared) * cpr, ld = ph_down_ld(chunks);
  const uint32_t rwaves = (blockDim.x >> 6) - has_shared;
  const uint32_t row0 = blockIdx.x * NR;
  const bool is_routed = wave < rwaves;
  const uint32_t item = is_routed ? min(wave * 64 + lane, items - 1) : items + min(lane, cpr - 1);
  const uint32_t slot = item / cpr, c = item - slot * cpr;
  const uint8_t* const blob = slot_blob(tab_dev, tab_val, slot);
  // What the combine needs, ahead of the weights.
  float hm = 0.f, sh_in = 0.f, gate = 0.f, wk = 0.f;
  if (tid < NR) {
    const uint32_t r = min(row0 + tid, H - 1);
    hm = h_mid[r];
    gate = tab_dev ? tab_dev->shared_gate : tab_val.shared_gate;
    if (!has_shared && shared_out) sh_in = shared_out[r];
  }
  if (tab_dev) {
    if (tid < k) wk = tab_dev->weight[tid];
    if (tid < k) sord[tid] = ordered ? tab_dev->order[tid] : (uint8_t)tid;
  } else {
    if (tid < k) sord[tid] = (uint8_t)tid;
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)kMaxK; ++i) wk = tid == i ? tab_val.weight[i] : wk;
  }
  // Activations: a quad of threads per chunk, at most four rounds (64 lanes
  // per wave hold 16 quads, and there is a lane per chunk).
  const uint32_t nq = blockDim.x >> 2, qd = tid >> 2, q = tid & 3;
  f32x4 st[4][2];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const f32x4* const p = reinterpret_cast<const f32x4*>(act + (size_t)min(qd + i * nq, chunks - 1) * kChunk + q * 8);
    st[i][0] = p[0];
    st[i][1] = p[1];
  }
  uint32_t* const limbs = lds;
  float* const part = reinterpret_cast<float*>(lds + (size_t)chunks * kL4Words);
  auto stage = [&]() {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      if (i * nq >= chunks) break;
      const uint32_t ch = qd + i * nq;
      const float v[8] = {st[i][0].x, st[i][0].y, st[i][0].z, st[i][0].w, st[i][1].x, st[i][1].y, st[i][1].z, st[i][1].w};
      store_limbs4_quad(limbs + (size_t)min(ch, chunks - 1) * kL4Words, v, (int)q, ch < chunks);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (is_routed) {
    DownRows<BITS, true, NR> d;
    d.load(blob, routed, row0, c);
    __builtin_amdgcn_sched_barrier(0);
    stage();
    if (wave * 64 + lane < items) d.dot(limbs + (size_t)item * kL4Words, part + item, ld);
  } else {
    DownRows<4, false, NR> d;
    d.load(blob, shared, row0, c);
    __builtin_amdgcn_sched_barrier(0);
    stage();
    if (lane < cpr) d.dot(limbs + (size_t)item * kL4Words, part + item, ld);
  }
  if (tid < k) sw[tid] = wk;
  __syncthreads();
  // Thread (row, slot): the slot's chunks in four interleaved sums.
  for (uint32_t i = tid; i < NR * (k + has_shared); i += blockDim.x) {
    const uint32_t r = i % NR, s = i / NR;
    const float* const p = part + r * ld + s * cpr;
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    uint32_t j = 0;
    for (; j + 4 <= cpr; j += 4)
#pragma unroll
      for (uint32_t v = 0; v < 4; ++v) a[v] += p[j + v];
    for (; j < cpr; ++j) a[j & 3] += p[j];
    so[r][s] = (a[0] + a[1]) + (a[2] + a[3]);
  }
  __syncthreads();
  if (tid < NR && row0 + tid < H) {
    float moe = 0.f;
    for (uint32_t i = 0; i < k; ++i) {
      const uint32_t s = sord[i];
      moe = __builtin_fmaf(so[tid][s], sw[s], moe);
    }
    float sum = moe;
    if (has_shared || shared_out) {
      const float sh = has_shared ? so[tid][k] : sh_in;
      sum = __builtin_isnan(gate) ? moe + sh : __builtin_fmaf(sh, sigmoidf_ref(gate), moe);
    }
    hidden_out[row0 + tid] = hm + sum;
  }
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------
// Calls fn with the instance's (P, IB, LR) as integral constants. The sums of
// a row depend on LR alone, which the number of tokens does not enter.
template <typename F>
static hipError_t gateup_shape(const BlobGeom& routed, uint32_t n_slots, uint32_t n_tokens, F fn) {  // n_slots: of a token
  const std::integral_constant<int, 16> l16;
  const uint32_t n = (routed.hidden / kChunk + 15) / 16;
  // Rows of more chunks than one round of 16 lanes takes, and few of them: a
  // whole wave per row, which 1 slot of 7168 x 64 (gate/up and down) takes 12.6
  // us with, 15.2 with 16 lanes; 16 of 7168 x 128 18.1 and 20.0, 16 of 7168 x
  // 192 22.7 and 22.0.
  if (n > 5 && n_slots * routed.inter <= 2048) {
    const std::integral_constant<int, 64> l64;
    const std::integral_constant<int, 2> p;
    return n <= 8 ? fn(p, std::integral_constant<int, 2>{}, l64) : fn(p, std::integral_constant<int, 4>{}, l64);
  }
  // 4 rows per wave while that makes no more than 1024 waves (one per SIMD),
  // else 8, whose limbs serve two rows each: 8 slots of 2048 x 512 (gate/up
  // and down) 10.8 us against 11.8, 8 of 2048 x 1024 15.9 against 14.3, 10 of
  // 2560 x 640 18.8 against 17.3, 8 of 7168 x 2048 74.0 against 72.2 (all four
  // with the row's values staged one round trip after another; as it is the
  // faster side takes 10.9, 14.5, 17.4 and 64.3). Four waves share a block's
  // limbs (one: 12.2, two: 11.3 at 2048 x 512).
  // Rounds of as many chunks per lane as the row has up to three (1024: rounds
  // of 4 left half of the places empty, 8 slots of 1024 x 1536 19.7 us against
  // 15.3), of 5 where they divide the row into fewer places
  // than rounds of 4 (2560: one of 5, not two of 4).
  const bool five = (n + 4) / 5 * 5 < (n + 3) / 4 * 4;
  auto rows = [&](auto p) {
    if (n == 1) return fn(p, std::integral_constant<int, 1>{}, l16);
    if (n == 2) return fn(p, std::integral_constant<int, 2>{}, l16);
    if (n == 3) return fn(p, std::integral_constant<int, 3>{}, l16);
    return five ? fn(p, std::integral_constant<int, 5>{}, l16) : fn(p, std::integral_constant<int, 4>{}, l16);
  };
  return n_slots * n_tokens * routed.inter <= 4096 ? rows(std::integral_constant<int, 1>{}) : rows(std::integral_constant<int, 2>{});
}
// Blocks per slot, and the bytes of a row's limbs in LDS.
static uint32_t ph_tiles(uint32_t inter, uint32_t rows) { return (inter + rows * kPhW - 1) / (rows * kPhW); }
static uint32_t ph_x_lds(uint32_t hidden, uint32_t rc) {
  return (hidden / kChunk + rc - 1) / rc * rc * kL4Words * 4;
}

template <int BITS>
static hipError_t gateup_bits(const BlobGeom& routed, const BlobGeom& shared, const FfnTable* tab_dev,
                              const FfnTable& tab_val, uint32_t n_slots, const float* x, float* act, hipStream_t st) {
  return gateup_shape(routed, n_slots, 1, [&](auto p, auto ib, auto lr) {
    constexpr int P = decltype(p)::value, IB = decltype(ib)::value, LR = decltype(lr)::value;
    const uint32_t tiles = ph_tiles(routed.inter, 64 / LR * P);
    hipLaunchKernelGGL((k_ph_gateup<BITS, P, IB, LR, kPhW>), dim3(tiles * n_slots), dim3(64 * kPhW),
                       ph_x_lds(routed.hidden, IB * LR), st, routed, shared, tab_dev, tab_val, tiles, x, act);
    return hipGetLastError();
  });
}

// Hidden 4096 has gate/up waves of its own (decode.hip); the selection reads
// eight logits per lane at most.
bool ph_route_supported(uint32_t hidden, uint32_t n_experts) { return hidden != 4096 && n_experts <= 512; }

template <int BITS, int PL>
static hipError_t route_bits(const BlobGeom& routed, const BlobGeom& shared, const float* logits, uint32_t E,
                             uint32_t k, bool normalize, const RouteOut& out, uint32_t n_slots, const float* x,
                             float* act, hipStream_t st, uint32_t n_tokens, uint32_t lstride, uint32_t astride) {
  return gateup_shape(routed, n_slots, n_tokens, [&](auto p, auto ib, auto lr) {
    constexpr int P = decltype(p)::value, IB = decltype(ib)::value, LR = decltype(lr)::value;
    const uint32_t tiles = ph_tiles(routed.inter, 64 / LR * P);
    hipLaunchKernelGGL((k_ph_route<BITS, PL, P, IB, LR, kPhW>), dim3(tiles * n_slots + 1, n_tokens), dim3(64 * kPhW),
                       ph_x_lds(routed.hidden, IB * LR), st, routed, shared, logits, E, k, (int)normalize, out, tiles, x,
                       act, lstride, astride);
    return hipGetLastError();
  });
}

hipError_t launch_ph_route(const BlobGeom& routed, const BlobGeom& shared, const float* logits, uint32_t E,
                           uint32_t k, bool normalize, const RouteOut& out, uint32_t n_slots, const float* x,
                           float* act, hipStream_t st, uint32_t n_tokens, uint32_t lstride, uint32_t astride) {
  auto go = [&](auto fn) {
    return fn(routed, shared, logits, E, k, normalize, out, n_slots, x, act, st, n_tokens, lstride, astride);
  };
  if (routed.bits == 4) return E <= 256 ? go(route_bits<4, 4>) : go(route_bits<4, 8>);
  return E <= 256 ? go(route_bits<3, 4>) : go(route_bits<3, 8>);
}

hipError_t launch_ph_gateup(const BlobGeom& routed, const BlobGeom& shared, const FfnTable* tab_dev,
                            const FfnTable& tab_val, uint32_t n_slots, const float* x, float* act, hipStream_t st) {
  return routed.bits == 4 ? gateup_bits<4>(routed, shared, tab_dev, tab_val, n_slots, x, act, st)
                          : gateup_bits<3>(routed, shared, tab_dev, tab_val, n_slots, x, act, st);
}

// Waves of a k_ph_down block: a lane per (slot, chunk), and the shared wave.
static uint32_t ph_down_waves(uint32_t inter, uint32_t k, bool has_shared) {
  return (k * (inter / kChunk) + 63) / 64 + has_shared;
}
constexpr uint32_t kPdLds = 156 * 1024;
bool ph_down_supported(uint32_t inter, uint32_t k, bool has_shared) {
  return ph_down_waves(inter, k, has_shared) <= 16 && ph_down_lds((k + has_shared) * (inter / kChunk), 4) <= kPdLds;
}

template <int BITS, uint32_t NR, int TB>
static hipError_t down_inst(const BlobGeom& routed, const BlobGeom& shared, const FfnTable* tab_dev,
                            const FfnTable& tab_val, uint32_t k, uint32_t has_shared, const float* act,
                            const float* h_mid, const float* shared_out, float* hidden_out, bool ordered,
                            hipStream_t st, uint32_t n_tokens, uint32_t astride) {
  const uint32_t lds = ph_down_lds((k + has_shared) * (routed.inter / kChunk), NR);
  if (lds > 60 * 1024) {
    static std::atomic<uint64_t> raised{0};
    const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(&k_ph_down<BITS, NR, TB>), kPdLds, raised);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_ph_down<BITS, NR, TB>), dim3((routed.hidden + NR - 1) / NR, n_tokens),
                     dim3(64 * ph_down_waves(routed.inter, k, has_shared)), lds, st, routed, shared, tab_dev, tab_val, k,
                     has_shared, act, h_mid, shared_out, hidden_out, (int)ordered, astride);
  return hipGetLastError();
}

template <int BITS>
static hipError_t down_bits(const BlobGeom& routed, const BlobGeom& shared, const FfnTable* tab_dev,
                            const FfnTable& tab_val, uint32_t k, uint32_t has_shared, const float* act,
                            const float* h_mid, const float* shared_out, float* hidden_out, bool ordered,
                            hipStream_t st, uint32_t n_tokens, uint32_t astride) {
  // Eight rows per block where that still makes a block per CU, else four (8
  // slots of 1024 x 1536, gate/up and down: 15.1 us with eight, 13.8 with four;
  // of 512 x 2048 13.8 and 12.3).
  if (ph_down_waves(routed.inter, k, has_shared) > 8)
    return down_inst<BITS, 4, 1024>(routed, shared, tab_dev, tab_val, k, has_shared, act, h_mid, shared_out, hidden_out, ordered, st, n_tokens, astride);
  if ((routed.hidden + 7) / 8 * n_tokens < 256)
    return down_inst<BITS, 4, 512>(routed, shared, tab_dev, tab_val, k, has_shared, act, h_mid, shared_out, hidden_out, ordered, st, n_tokens, astride);
  return down_inst<BITS, 8, 512>(routed, shared, tab_dev, tab_val, k, has_shared, act, h_mid, shared_out, hidden_out, ordered, st, n_tokens, astride);
}

hipError_t launch_ph_down(const BlobGeom& routed, const BlobGeom& shared, const FfnTable* tab_dev,
                          const FfnTable& tab_val, uint32_t n_slots, const float* act, const float* h_mid,
                          const float* shared_out, float* hidden_out, hipStream_t st, bool ordered,
                          uint32_t n_tokens, uint32_t astride) {
  const uint32_t k = tab_val.k, has_shared = n_slots > k ? 1u : 0u;
  return routed.bits == 4 ? down_bits<4>(routed, shared, tab_dev, tab_val, k, has_shared, act, h_mid, shared_out, hidden_out, ordered, st, n_tokens, astride)
                          : down_bits<3>(routed, shared, tab_dev, tab_val, k, has_shared, act, h_mid, shared_out, hidden_out, ordered, st, n_tokens, astride);
}

}  // namespace smoe
