// router.hip — noaux_tc routing (DeepSeek-V3 / Cogito-V2) from precomputed
// gate logits, one wave per token.
//
//   k_noaux_topk  sigmoid scores, correction bias, group scores (sum of the
//                 top two biased scores of each group), the reference's
//                 running-minimum top-k over the group scores, the group
//                 mask, the same top-k over the masked biased scores, and
//                 the renormalised, scaled un-biased weights, in the
//                 reference's slot order and summation order
//                 (crates/streammoe/src/riir/moe/moe_router.rs:211-330).
//
// Lane l holds experts l, l + 64, ... Groups of a power-of-two size up to
// 64 take their top two with a lane butterfly (the scan's result: the two
// largest values with multiplicity); other sizes are scanned in lane g for
// group g over an LDS copy strided by group_size + 1 (so the lanes' reads
// fall in different banks), with the reference's compares. Both top-k
// passes use exact_topk_t, the reference's scan order and tie rules.
#include "common.h"
#include "kernels.h"
#include "topk.h"

namespace smoe {

// (largest, second largest) pairs merged with the pair the DPP control
// brings in (lanes outside ROW_MASK merge with (-inf, -inf): unchanged).
template <int CTRL, int ROW_MASK = 0xF, int P>
__device__ __forceinline__ void top2_merge(float (&a1)[P], float (&a2)[P]) {
#pragma unroll
  for (int e = 0; e < P; ++e) {
    const float c1 = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(-INFINITY), __float_as_int(a1[e]),
                                                                CTRL, ROW_MASK, 0xF, false));
    const float c2 = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(-INFINITY), __float_as_int(a2[e]),
                                                                CTRL, ROW_MASK, 0xF, false));
    const float t2 = fmaxf(fminf(a1[e], c1), fmaxf(a2[e], c2));
    a1[e] = fmaxf(a1[e], c1);
    a2[e] = t2;
  }
}

template <int P>
__global__ __launch_bounds__(64) void k_noaux_topk(const float* logits,
                                                   const float* __restrict__ bias, uint32_t n,
                                                   uint32_t n_group, uint32_t topk_group, uint32_t k,
                                                   float scale, float* scores_out, RouteOut out) {
  __shared__ float s_sig[64 * P];        // un-biased sigmoid scores
  __shared__ float s_bsd[64 * P + 64];   // biased scores, element j at j + j / group_size (scan layout)
  __shared__ float s_gsc[64];            // group scores
  __shared__ int32_t s_idx[kMaxK];
  __shared__ float s_val[kMaxK];
  const uint32_t t = blockIdx.x;
  const int lane = threadIdx.x;
  const uint32_t gs = n / n_group;
  // Power-of-two groups of at most 64 elements lie inside one 64-element
  // chunk: their top two come from a lane butterfly; other sizes are
  // scanned from LDS.
  const bool lanes_path = gs <= 64 && (gs & (gs - 1)) == 0;
  const float* lg = logits + (size_t)t * n;

  // 1-2. s = 1 / (1 + exp(-logit)); biased = s + correction_bias. Lane l
  // holds elements l, l + 64, ... (coalesced loads).
  float b[P];
#pragma unroll
  for (int e = 0; e < P; ++e) {
    const uint32_t j = e * 64 + lane;
    b[e] = -INFINITY;
    if (j < n) {
      const float s = 1.0f / (1.0f + expf(-lg[j]));
      b[e] = s + bias[j];
      s_sig[j] = s;
      if (!lanes_path) s_bsd[j + j / gs] = b[e];
      if (scores_out) scores_out[(size_t)t * n + j] = s;
    }
  }

  // 3. Group score = top1 + top2 of the group's biased scores, as the
  // reference's linear scan (v > top1: shift; else v > top2) leaves them:
  // the two largest values with multiplicity, NaN never taken (here: -inf,
  // which no compare takes either).
  if (lanes_path) {
    // DPP merges of (largest, second) pairs over disjoint lane sets: quad
    // swaps (lane ^ 1, lane ^ 2), the 8-lane half-row mirror, the row
    // mirror (every lane of a group of <= 16 then holds its result), then
    // row 1 (3) takes row 0 (2) and row 3 rows 0-1: for 32 and 64 the
    // result is in the group's last lane.
    float a1[P], a2[P];
#pragma unroll
    for (int e = 0; e < P; ++e) {
      a1[e] = b[e] == b[e] ? b[e] : -INFINITY;
      a2[e] = -INFINITY;
    }
    if (gs >= 2) top2_merge<0xB1>(a1, a2);
    if (gs >= 4) top2_merge<0x4E>(a1, a2);
    if (gs >= 8) top2_merge<0x141>(a1, a2);
    if (gs >= 16) top2_merge<0x140>(a1, a2);
    if (gs >= 32) top2_merge<0x142, 0xA>(a1, a2);
    if (gs >= 64) top2_merge<0x143, 0xC>(a1, a2);
#pragma unroll
    for (int e = 0; e < P; ++e) {
      const uint32_t j = e * 64 + lane;
      if (j < n && j % gs == gs - 1) s_gsc[j / gs] = a1[e] + a2[e];
    }
  } else {
    __syncthreads();
    if ((uint32_t)lane < n_group) {
      const float* p = s_bsd + (size_t)lane * (gs + 1);
      float top1 = -INFINITY, top2 = -INFINITY;
      uint32_t i = 0;
      for (; i + 8 <= gs; i += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[i + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const bool gt1 = v[u] > top1, gt2 = v[u] > top2;
          top2 = gt1 ? top1 : (gt2 ? v[u] : top2);
          top1 = gt1 ? v[u] : top1;
        }
      }
      for (; i < gs; ++i) {
        const float v = p[i];
        const bool gt1 = v > top1, gt2 = v > top2;
        top2 = gt1 ? top1 : (gt2 ? v : top2);
        top1 = gt1 ? v : top1;
      }
      s_gsc[lane] = top1 + top2;
    }
  }
  __syncthreads();

  // 4. topk() of the group scores; lanes past n_group hold -inf, which
  // never beats a slot.
  float gsc[1] = {(uint32_t)lane < n_group ? s_gsc[lane] : -INFINITY};
  const int32_t kept = exact_topk_t<1>(gsc, topk_group, lane, nullptr, nullptr);

  // 5. Mask the groups that were not kept (a start slot that was never
  // replaced keeps group 0, as the reference's index set does): the OR of
  // the kept groups' bits over the queue lanes.
  const uint64_t bit = kept >= 0 ? 1ull << kept : 0ull;
  const uint32_t klo = wave_or_last((uint32_t)bit), khi = wave_or_last((uint32_t)(bit >> 32));
  const uint64_t keep = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)khi, 63) << 32) |
                        (uint32_t)__builtin_amdgcn_readlane((int)klo, 63);
#pragma unroll
  for (int e = 0; e < P; ++e) {
    const uint32_t j = e * 64 + lane;
    if (j >= n || !((keep >> (j / gs)) & 1ull)) b[e] = -INFINITY;
  }

  // 6. topk() of the masked biased scores.
  exact_topk_t<P>(b, k, lane, s_idx, s_val);
  __syncthreads();

  // 7. Gather the un-biased scores (lane s: slot s), sum them in slot
  // order, w *= 1 / sum when sum > 0, then w *= routed_scaling_factor.
  const int32_t id = lane < (int)k ? s_idx[lane] : 0;
  float w = s_sig[id];
  float sum = 0.f;
  for (uint32_t s = 0; s < k; ++s) sum += readlane_f(w, (int)s);
  if (lane < (int)k) {
    if (sum > 0.f) {
      const float inv = 1.0f / sum;
      w *= inv;
    }
    w *= scale;
    if (out.idx) out.idx[(size_t)t * k + lane] = id;
    if (out.weight) out.weight[(size_t)t * k + lane] = w;
    if (out.table && t == 0) {
      out.table->blob[lane] = out.experts + (uint64_t)id * out.stride;
      out.table->weight[lane] = w;
    }
  }
  if (out.table && t == 0 && lane == 0) {
    out.table->k = k;
    out.table->has_shared = out.shared_blob != nullptr;
    if (out.shared_blob) {
      out.table->blob[k] = out.shared_blob;
      out.table->weight[k] = 1.0f;
      out.table->shared_gate = out.gate_scores ? out.gate_scores[0] : __builtin_nanf("");
    }
  }
}

hipError_t launch_noaux_topk(const float* logits, const float* bias, uint32_t n_tokens, uint32_t n,
                             uint32_t n_group, uint32_t topk_group, uint32_t k, float scale,
                             float* scores_out, const RouteOut& out, hipStream_t st) {
  if (n == 0 || n > kNoauxMaxExperts || n_group == 0 || n_group > kNoauxMaxGroups || n % n_group ||
      topk_group == 0 || topk_group > n_group || k == 0 || k > n || k > (uint32_t)kMaxK)
    return hipErrorInvalidValue;
  const uint32_t p = (n + 63) / 64;
  const dim3 grid(n_tokens), block(64);
  if (p <= 1)
    hipLaunchKernelGGL(k_noaux_topk<1>, grid, block, 0, st, logits, bias, n, n_group, topk_group, k, scale,
                       scores_out, out);
  else if (p <= 2)
    hipLaunchKernelGGL(k_noaux_topk<2>, grid, block, 0, st, logits, bias, n, n_group, topk_group, k, scale,
                       scores_out, out);
  else if (p <= 4)
    hipLaunchKernelGGL(k_noaux_topk<4>, grid, block, 0, st, logits, bias, n, n_group, topk_group, k, scale,
                       scores_out, out);
  else if (p <= 8)
    hipLaunchKernelGGL(k_noaux_topk<8>, grid, block, 0, st, logits, bias, n, n_group, topk_group, k, scale,
                       scores_out, out);
  else
    hipLaunchKernelGGL(k_noaux_topk<16>, grid, block, 0, st, logits, bias, n, n_group, topk_group, k, scale,
                       scores_out, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Router logits of many tokens: logits[t, e] = W[e] . x[t] in f32 on
// v_mfma_f32_16x16x4_f32. A block of eight waves holds 16 tokens x 32 experts;
// the waves split the inputs, 32 at a time, each copying its own piece of
// the 16 x rows and 32 router rows to LDS (LDS DMA in memory order, four lanes
// per row's 64 bytes) one piece ahead and reading it back in operand order,
// so the loop has no block barrier. 16-byte part p of row r is stored at part
// p ^ (r / 4 % 4): the 16 rows of an operand read fall on all banks.
//
// Rounding: an accumulator runs over 8 inputs (two MFMAs) and the sums are
// then added pairwise (a binary tree over a wave's inputs, then over the
// waves), as the one-row kernel's lanes are, not along one chain of `hidden`
// additions.
//
// 512 tokens, 256 experts, hidden 2048: 94 us with a block per (token, expert
// row), each reading both rows again (2 GB through L2); 12.4 us
// here, the limit of its chain of eight pieces per wave (the matrix cores are
// busy 3.5 us of it).
// ---------------------------------------------------------------------------
constexpr uint32_t kRlT = 16, kRlE = 32, kRlW = 8;           // tokens, experts, waves per block
constexpr uint32_t kRlK = 32;                                // inputs per piece
constexpr uint32_t kRlRows = kRlT + kRlE;                    // rows of a piece
constexpr uint32_t kRlPiece = kRlRows * kRlK * 4;            // bytes
constexpr uint32_t kRlRing = 2;                              // pieces in LDS per wave
constexpr uint32_t kRlLds = kRlW * kRlRing * kRlPiece;
static_assert(kRlLds <= 160 * 1024, "LDS per CU");
static_assert(kRlLds >= kRlW * 2 * 64 * 16, "the waves' sums fit over the pieces");

__global__ __launch_bounds__(64 * kRlW) void k_router_mm(const float* __restrict__ W, const float* __restrict__ x,
                                                         uint32_t n, uint32_t E, uint32_t H,
                                                         float* __restrict__ logits) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t c16 = lane & 15, kb = lane >> 4;
  const uint32_t ne = (E + kRlE - 1) / kRlE;
  const uint32_t t0 = blockIdx.x / ne * kRlT, e0 = blockIdx.x % ne * kRlE;
  uint8_t* const mine = lds + wave * kRlRing * kRlPiece;
  // Lane l copies part l % 4 of row l / 4 of each group of 16 rows; rows past
  // the end repeat the last (their sums are dropped).
  const uint32_t lr = lane >> 2, part = ((lane & 3) ^ (lr >> 2)) * 16;
  const uint8_t* src[3];
  src[0] = reinterpret_cast<const uint8_t*>(x + (size_t)min(t0 + lr, n - 1) * H) + part;
  src[1] = reinterpret_cast<const uint8_t*>(W + (size_t)min(e0 + lr, E - 1) * H) + part;
  src[2] = reinterpret_cast<const uint8_t*>(W + (size_t)min(e0 + 16 + lr, E - 1) * H) + part;
  // Piece i of this wave: inputs [32 (wave + 8 i), + 32), as two 16-input
  // columns of 64 bytes per row.
  constexpr uint32_t NC = kRlK / 16;
  const uint32_t np = (H / kRlK + kRlW - 1 - wave) / kRlW;
  auto copy = [&](uint32_t i) {
    const uint32_t k0 = (wave + kRlW * i) * (kRlK * 4);
    uint8_t* const dst = mine + i % kRlRing * kRlPiece;
#pragma unroll
    for (uint32_t g = 0; g < 3; ++g)
#pragma unroll
      for (uint32_t c = 0; c < NC; ++c) dma16(src[g] + k0 + c * 64, dst + (g * NC + c) * 1024);
  };
  f32x4 sum[2][8];  // pairwise tree of each tile: level v holds 2^v pieces' sums
  uint32_t have = 0;
  if (np) copy(0);
  const uint32_t rd = c16 * 64 + ((kb ^ (c16 >> 2)) * 16);  // operand part of lane (row, kb)
  for (uint32_t i = 0; i < np; ++i) {
    // The reads of the piece before are done, its buffer takes the next
    // piece's copies; then this piece has landed when this wave's copies of
    // it have (the next piece's six stay in flight; a third buffer 13.0 us).
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (i + 1 < np) {
      copy(i + 1);
      asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const uint8_t* const p = mine + i % kRlRing * kRlPiece + rd;
    static_assert(3 * NC == 6, "copies per piece");
    f32x4 leaf[2][2 * NC];
#pragma unroll
    for (uint32_t c = 0; c < NC; ++c) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(p + c * 1024);
#pragma unroll
      for (uint32_t t = 0; t < 2; ++t) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(p + ((t + 1) * NC + c) * 1024);
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
        leaf[t][2 * c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, z, 0, 0, 0);
        leaf[t][2 * c + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, z, 0, 0, 0);
        leaf[t][2 * c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, leaf[t][2 * c], 0, 0, 0);
        leaf[t][2 * c + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, leaf[t][2 * c + 1], 0, 0, 0);
      }
    }
    f32x4 s[2];
#pragma unroll
    for (uint32_t t = 0; t < 2; ++t) s[t] = (leaf[t][0] + leaf[t][1]) + (leaf[t][2] + leaf[t][3]);
    // Binary counter: carry the sum up past the levels that are full.
    bool done = false;
#pragma unroll
    for (uint32_t v = 0; v < 8; ++v) {
      if (done) continue;
      if (have >> v & 1) {
        s[0] += sum[0][v];
        s[1] += sum[1][v];
      } else {
        sum[0][v] = s[0];
        sum[1][v] = s[1];
        done = true;
      }
    }
    ++have;
  }
  f32x4 tot[2] = {};
#pragma unroll
  for (uint32_t v = 0; v < 8; ++v)
    if (have >> v & 1) {
      tot[0] += sum[0][v];
      tot[1] += sum[1][v];
    }
  // The waves' sums, pairwise.
  __syncthreads();
  f32x4* const red = reinterpret_cast<f32x4*>(lds);
  red[(wave * 2 + 0) * 64 + lane] = tot[0];
  red[(wave * 2 + 1) * 64 + lane] = tot[1];
  __syncthreads();
  if (wave < 2) {
    const f32x4* const p = red + wave * 64 + lane;
    const f32x4 v = ((p[0] + p[128]) + (p[256] + p[384])) + ((p[512] + p[640]) + (p[768] + p[896]));
    const uint32_t e = e0 + wave * 16 + c16;
    if (e < E)
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t t = t0 + kb * 4 + i;
        if (t < n) logits[(size_t)t * E + e] = v[i];
      }
  }
}

// Whether a call runs on k_router_mm: whole pieces, no more of them per wave
// than the tree has room for, and enough logits: a wave's chain of pieces costs
// 7 us more than one row's block at hidden 2048 (23 at 7168), the one-row
// kernel 0.27 us per million products, so the line is at about 2^14 logits
// whatever the hidden size.
bool router_mm_supported(uint32_t n_tokens, uint32_t n_experts, uint32_t hidden) {
  return (uint64_t)n_tokens * n_experts >= (1u << 14) && hidden % kRlK == 0 && hidden <= 32768;
}

hipError_t launch_router_mm(const float* W, const float* x, uint32_t n_tokens, uint32_t n_experts, uint32_t hidden,
                            float* logits, hipStream_t st) {
  static std::atomic<uint64_t> raised{0};
  const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(&k_router_mm), kRlLds, raised);
  if (e != hipSuccess) return e;
  const uint32_t blocks = (n_tokens + kRlT - 1) / kRlT * ((n_experts + kRlE - 1) / kRlE);
  hipLaunchKernelGGL(k_router_mm, dim3(blocks), dim3(64 * kRlW), kRlLds, st, W, x, n_tokens, n_experts, hidden, logits);
  return hipGetLastError();
}

}  // namespace smoe
