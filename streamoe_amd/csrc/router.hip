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
// Rounding: the sums are those of k_router_logits bit for bit, so a token's
// logits, and the pick between nearly tied experts, do not depend on how many
// tokens share the call. Its thread t of 256 chains FMAs over the inputs 1024 i +
// 4 t + {0, 1, 2, 3}, which is one MFMA per i (the instruction adds its four
// products one FMA after another); the 256 leaves are then added as a binary
// tree. Wave w takes the leaves' groups of eight 2 w, 2 w + 1 and 16 above
// them, i innermost: neighbours meet in its registers, and rows that are not
// whole turns of 1024 still split evenly (hidden 512 or 2560).
//
// 512 tokens, 256 experts, hidden 2048: 94 us with a block per (token, expert
// row), each reading both rows again (2 GB through L2); 12.1 us
// here, the limit of its chain of eight pieces per wave (the matrix cores are
// busy 3.5 us of it).
// ---------------------------------------------------------------------------
constexpr uint32_t kRlT = 16, kRlE = 32, kRlW = 8;           // tokens, experts, waves per block
constexpr uint32_t kRlK = 32;                                // inputs per piece: eight leaves
constexpr uint32_t kRlTurn = 1024;                           // inputs from one FMA group of a leaf to the next
constexpr uint32_t kRlQ = kRlTurn / kRlK / kRlW;             // leaf groups per wave
constexpr uint32_t kRlRows = kRlT + kRlE;                    // rows of a piece
constexpr uint32_t kRlPiece = kRlRows * kRlK * 4;            // bytes
constexpr uint32_t kRlRing = 2;                              // pieces in LDS per wave
constexpr uint32_t kRlLds = kRlW * kRlRing * kRlPiece;
static_assert(kRlLds <= 160 * 1024, "LDS per CU");
static_assert(kRlQ == 4 && kRlT * kRlE == 64 * kRlW, "pairs of groups; a thread per logit");
static_assert(kRlLds >= kRlW * 2 * 2 * 64 * 16, "the pairs' sums fit over the pieces");

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
  // Piece (q, i): inputs [1024 i + at(q), + 32), as two 16-input columns of 64
  // bytes per row. Group q has `turns(q)` of them.
  constexpr uint32_t NC = kRlK / 16;
  auto at = [&](uint32_t q) { return (2 * wave + (q & 1) + 2 * kRlW * (q >> 1)) * kRlK; };
  auto turns = [&](uint32_t q) { return at(q) < H ? (H - at(q) + kRlTurn - 1) / kRlTurn : 0u; };
  uint32_t issued = 0;  // pieces copied so far
  auto copy = [&](uint32_t q, uint32_t i) {
    const uint32_t k0 = (i * kRlTurn + at(q)) * 4;
    uint8_t* const dst = mine + issued++ % kRlRing * kRlPiece;
#pragma unroll
    for (uint32_t g = 0; g < 3; ++g)
#pragma unroll
      for (uint32_t c = 0; c < NC; ++c) dma16(src[g] + k0 + c * 64, dst + (g * NC + c) * 1024);
  };
  // Lane (row, kb)'s input 4 m + kb of a column.
  uint32_t rd[4];
#pragma unroll
  for (uint32_t m = 0; m < 4; ++m) rd[m] = c16 * 64 + ((m ^ (c16 >> 2)) * 16) + kb * 4;
  f32x4 sum[kRlQ][2];
  uint32_t done = 0;
  if (turns(0)) copy(0, 0);
#pragma unroll
  for (uint32_t q = 0; q < kRlQ; ++q) {
    f32x4 leaf[2][4 * NC];
#pragma unroll
    for (uint32_t m = 0; m < 4 * NC; ++m) leaf[0][m] = leaf[1][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const uint32_t ni = turns(q);
    for (uint32_t i = 0; i < ni; ++i) {
      // The reads of the piece before are done, its buffer takes the next
      // piece's copies; then this piece has landed when this wave's copies of
      // it have (the next piece's six stay in flight; a third buffer 13.0 us).
      // Later groups have no more turns than this one.
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      const bool here = i + 1 < ni, next = q + 1 < kRlQ && turns(q + 1) > 0;
      if (here || next) {
        copy(here ? q : q + 1, here ? i + 1 : 0);
        asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      static_assert(3 * NC == 6, "copies per piece");
      const uint8_t* const p = mine + done++ % kRlRing * kRlPiece;
      auto word = [&](uint32_t g, uint32_t c, uint32_t m) {
        return *reinterpret_cast<const float*>(p + rd[m] + (g * NC + c) * 1024);
      };
#pragma unroll
      for (uint32_t c = 0; c < NC; ++c)
#pragma unroll
        for (uint32_t m = 0; m < 4; ++m) {
          const float a = word(0, c, m);
#pragma unroll
          for (uint32_t t = 0; t < 2; ++t)
            leaf[t][4 * c + m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, word(t + 1, c, m), leaf[t][4 * c + m], 0, 0, 0);
        }
    }
#pragma unroll
    for (uint32_t t = 0; t < 2; ++t)
      sum[q][t] = ((leaf[t][0] + leaf[t][1]) + (leaf[t][2] + leaf[t][3])) + ((leaf[t][4] + leaf[t][5]) + (leaf[t][6] + leaf[t][7]));
  }
  // The tree over the 16 pairs of groups, pairs w and w + 8 from wave w: thread
  // (tile, word) adds that word of each pair's 256 and stores its logit.
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
    for (uint32_t t = 0; t < 2; ++t)
      reinterpret_cast<f32x4*>(lds)[((wave + kRlW * j) * 2 + t) * 64 + lane] = sum[2 * j][t] + sum[2 * j + 1][t];
  __syncthreads();
  const float* const red = reinterpret_cast<const float*>(lds) + threadIdx.x;
  float v[16];
#pragma unroll
  for (uint32_t j = 0; j < 16; ++j) v[j] = red[j * 512];
#pragma unroll
  for (uint32_t d = 1; d < 16; d *= 2)
#pragma unroll
    for (uint32_t j = 0; j < 16; j += 2 * d) v[j] += v[j + d];
  const uint32_t t = t0 + (wave & 3) * 4 + (lane & 3), e = e0 + (wave >> 2) * 16 + (lane >> 2);
  if (t < n && e < E) logits[(size_t)t * E + e] = v[0];
}

// Whether a call runs on k_router_mm: whole pieces, and enough logits: a
// wave's chain of pieces costs 7 us more than one row's block at hidden 2048
// (21 at 7168), the one-row kernel 0.27 us per million products, so the line is
// at about 2^14 logits whatever the hidden size.
bool router_mm_supported(uint32_t n_tokens, uint32_t n_experts, uint32_t hidden) {
  return (uint64_t)n_tokens * n_experts >= (1u << 14) && hidden % kRlK == 0;
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
