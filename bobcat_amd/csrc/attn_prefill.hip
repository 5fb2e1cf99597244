// Prefill attention on MFMA: causal GQA softmax(q·k/√d)·v for a batch of
// queries against the f16 KV cache (Metal::attention with n_queries > 1 and
// its attention_flash kernel, crates/bobcat-metal/src/backend.rs:2150-2320,
// attention.metal:289-480).
//
// A workgroup of four waves serves one KV head; a wave owns 32 consecutive
// queries of one query head.  With a group of G query heads per KV head the
// waves are G heads x 4/G query tiles (three heads leave one wave idle), so
// they share every key block.  K and V of a block of 32 keys go to LDS once,
// double buffered, the next block's loads in flight behind the current
// block's MFMAs: reading K from the cache by each wave cost 32 cache lines
// per load in four waves, more address cycles than the MFMAs take.
//
// Per block a wave computes S^T = K·Q^T (keys × queries) with
// v_mfma_f32_32x32x16_f16, so each lane holds 16 scores of one query: the
// online softmax needs one cross-lane move (lane l and l^32 share a query),
// and the lane's scores of keys 16j + 4·(l/32) + {0..3, 8..11} are, as
// probabilities, the B operand of k-step j of O^T += V^T·P^T; V is laid out
// in LDS by quads of keys so that the A operand has the same keys.  The
// queries and the probabilities are split into f16 high and low parts (~22
// bits) and both are multiplied; K and V are the cache's f16 values, so the
// products are exact and accumulate in f32.  Scores stay unscaled; the
// softmax runs in powers of two, p = 2^(s·c − m), c = scale·log2(e).
//
// 512 queries over 8,192 keys, 32 x 8 heads of 64: 97 us with four key splits
// and 9 us to combine them (340 TFLOP/s of the 4·hd operations a visible key
// takes, the matrix cores doing twice that); 414 us before, unsplit.  What
// bounds it now is issue slots: ~16 MFMAs and ~200 other instructions per
// wave and block, most of them the softmax and the splitting of p.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device.h"
#include "kernels.h"
#include "runtime.h"

namespace bch {

typedef _Float16 ph4_t __attribute__((ext_vector_type(4)));
typedef _Float16 ph8_t __attribute__((ext_vector_type(8)));
typedef _Float16 ph2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float pf2_t __attribute__((ext_vector_type(2)));
typedef float pf16_t __attribute__((ext_vector_type(16)));

constexpr int kPrefQ = 32;        // queries per wave
constexpr int kPrefKeys = 32;     // keys per block

// The output gate of gated attention (Qwen3.5, qwen35.rs:422-424): with
// `gate` set, output element d of (query z, head h) is multiplied by
// sigmoid(gate[z·query_stride + h·head_stride + d]).
struct AttnGate {
  const float *gate;
  uint32_t head_stride, query_stride;
  __device__ float at(uint32_t z, uint32_t head, uint32_t d) const {
    return gate ? 1.0f / (1.0f + expf(-gate[(uint64_t)z * query_stride + (uint64_t)head * head_stride + d])) : 1.f;
  }
};

// Query tiles per workgroup for a group of G query heads.
__host__ __device__ constexpr uint32_t attn_prefill_tiles(uint32_t group) { return group == 1 ? 4 : group == 2 ? 2 : 1; }

template <int HD>
__global__ __launch_bounds__(256, HD == 64 ? 3 : HD == 128 ? 2 : 1) void k_attn_prefill(const float *__restrict__ q, const _Float16 *__restrict__ kc,
                                                      const _Float16 *__restrict__ vc, float *__restrict__ out,
                                                      uint32_t n_heads, uint32_t n_kv, uint32_t first_pos,
                                                      uint32_t n_queries, uint32_t q_stride, uint32_t out_stride,
                                                      float scale, float *__restrict__ partials, AttnGate gate) {
  constexpr int KS = HD / 16;      // k-steps of the score product
  constexpr int OB = HD / 32;      // 32-row blocks of the output
  constexpr int CH = HD / 8;       // 16-byte chunks of a cache row
  constexpr int NP = HD / 64;      // pieces of K and of V per thread and block
  // K: chunk c of key k at slot 32c + (k ^ c%8); V: keys 4i .. 4i+3 of
  // element d at quad i·HD + d.
  __shared__ __align__(16) _Float16 k_s[2][kPrefKeys * HD], v_s[2][kPrefKeys * HD];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const uint32_t kv = blockIdx.y, group = n_heads / n_kv, tiles = attn_prefill_tiles(group);
  const uint32_t wg_q0 = blockIdx.x * tiles * kPrefQ;
  const bool active = (uint32_t)wave < group * tiles && wg_q0 + wave / group * kPrefQ < n_queries;
  const uint32_t head = kv * group + (active ? wave % group : 0);
  const uint32_t q0 = wg_q0 + (active ? wave / group : 0) * kPrefQ;
  const uint32_t col = lane % 32, half_id = lane / 32;
  const uint32_t z = min(q0 + col, n_queries - 1);  // this lane's query (past the end: a copy, never stored)
  const uint32_t qpos = first_pos + q0 + col;
  const uint32_t kend = first_pos + min(q0 + kPrefQ, n_queries);                      // keys of the wave's last query
  const uint32_t wg_kend = first_pos + min(wg_q0 + tiles * kPrefQ, n_queries);        // and of the workgroup's
  const uint64_t row_elems = (uint64_t)n_kv * HD;                                     // cache elements per position
  // Key split blockIdx.z of gridDim.z: a contiguous run of whole 32-key
  // blocks of the workgroup's keys (possibly none, or none visible to a
  // query: that split's partial then has max -inf and sum 0, and weighs
  // nothing in the combine).
  const uint32_t n_blocks = (wg_kend + kPrefKeys - 1) / kPrefKeys, n_split = gridDim.z, split = blockIdx.z;
  const uint32_t b_lo = (uint32_t)((uint64_t)split * n_blocks / n_split);
  const uint32_t b_hi = (uint32_t)((uint64_t)(split + 1) * n_blocks / n_split);

  // The block's cache rows through a descriptor of the block: rows past the
  // end read zeros (their scores are masked), and an address is one constant
  // per thread.  The whole address is in the vector offset: that is what is
  // compared with the descriptor's size (a scalar offset is not).
  const uint32_t row_bytes = n_kv * HD * 2;
  u32x4_t kr[NP];
  uint32_t vr[NP][4];
  auto load = [&](uint32_t blk) __attribute__((always_inline)) {
    const uint32_t kb = blk * kPrefKeys, bytes = min((uint32_t)kPrefKeys, wg_kend - kb) * row_bytes - kv * HD * 2;
    const uint64_t at = kb * row_elems + (uint64_t)kv * HD;
    const __amdgpu_buffer_rsrc_t kd = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(kc) + at, 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vd = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(vc) + at, 0, bytes, 0x00020000);
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const uint32_t c = tid + 256 * p;
      kr[p] = __builtin_amdgcn_raw_buffer_load_b128(kd, c / CH * row_bytes + (c % CH) * 16, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const uint32_t c = tid + 256 * p, dp = c % (HD / 2), kq = c / (HD / 2);
#pragma unroll
      for (int i = 0; i < 4; i++)
        vr[p][i] = __builtin_amdgcn_raw_buffer_load_b32(vd, (4 * kq + i) * row_bytes + 4 * dp, 0, 0);
    }
  };
  auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const uint32_t c = tid + 256 * p, key = c / CH, chunk = c % CH;
      *reinterpret_cast<u32x4_t *>(&k_s[buf][(chunk * 32 + (key ^ (chunk & 7))) * 8]) = kr[p];
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const uint32_t c = tid + 256 * p, dp = c % (HD / 2), kq = c / (HD / 2);
      // (k0, k1) and (k2, k3) of elements 2dp (low halves) and 2dp + 1.
      const u32x4_t w = {__builtin_amdgcn_perm(vr[p][1], vr[p][0], 0x05040100u),
                       __builtin_amdgcn_perm(vr[p][3], vr[p][2], 0x05040100u),
                       __builtin_amdgcn_perm(vr[p][1], vr[p][0], 0x07060302u),
                       __builtin_amdgcn_perm(vr[p][3], vr[p][2], 0x07060302u)};
      *reinterpret_cast<u32x4_t *>(&v_s[buf][(kq * HD + 2 * dp) * 4]) = w;
    }
  };
  if (b_lo < b_hi) load(b_lo);

  // The query's k-step fragments as the B operand: Q[z][16·s + 8·half .. +8].
  ph8_t qh[KS], ql[KS];
  {
    const float *qr = q + (uint64_t)z * q_stride + (uint64_t)head * HD + 8 * half_id;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const float4 a = *reinterpret_cast<const float4 *>(qr + 16 * s);
      const float4 b = *reinterpret_cast<const float4 *>(qr + 16 * s + 4);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int j = 0; j < 8; j++) {
        qh[s][j] = (_Float16)v[j];
        ql[s][j] = (_Float16)(v[j] - (float)qh[s][j]);
      }
    }
  }
  pf16_t o[OB];
#pragma unroll
  for (int b = 0; b < OB; b++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[b][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;  // the maximum in units of log2
  const float c2 = scale * 1.44269504088896340736f;

  auto block = [&](uint32_t kb, int buf) __attribute__((always_inline)) {
    // S^T = K·Q^T: lane supplies K[kb + col][16·s + 8·half .. +8].
    pf16_t sc;
#pragma unroll
    for (int i = 0; i < 16; i++) sc[i] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const uint32_t chunk = 2 * s + half_id;
      const ph8_t ka = *reinterpret_cast<const ph8_t *>(&k_s[buf][(chunk * 32 + (col ^ (chunk & 7))) * 8]);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qh[s], sc, 0, 0, 0);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, ql[s], sc, 0, 0, 0);
    }
    // sc[r] is the score of key kb + 8·(r/4) + 4·half + r%4 for this lane's
    // query; only blocks that reach past the wave's first query have a key
    // to mask.
    if (kb + kPrefKeys - 1 > first_pos + q0) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const uint32_t key = kb + 8 * (r / 4) + 4 * half_id + (r % 4);
        if (key > qpos || key >= kend) sc[r] = -INFINITY;
      }
    }
    float mx = sc[0];
#pragma unroll
    for (int r = 1; r < 16; r++) mx = fmaxf(mx, sc[r]);
    // (The two lanes of a query, 32 apart: the swap leaves both values in each.)
    const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    mx = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1])) * c2;
    // -inf while no key of this split has been visible to the query (a
    // causal split can start after it): the block then adds exact zeros.
    if (__builtin_amdgcn_ballot_w64(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= corr;
#pragma unroll
      for (int b = 0; b < OB; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[b][i] *= corr;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    float psum = 0.f;
    ph8_t ph[2], pl[2];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[r], c2, -m_use));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[r + 1], c2, -m_use));
      psum += p0 + p1;
      const pf2_t pv = {p0, p1};
      const ph2_t hi = __builtin_convertvector(pv, ph2_t);
      const pf2_t rest = {p0 - (float)hi[0], p1 - (float)hi[1]};
      const ph2_t lo = __builtin_convertvector(rest, ph2_t);
      ph[r / 8][r % 8] = hi[0], ph[r / 8][r % 8 + 1] = hi[1];
      pl[r / 8][r % 8] = lo[0], pl[r / 8][r % 8 + 1] = lo[1];
    }
    l_run += psum;
    // O^T += V^T·P^T over 2 k-steps of 16 keys: lane supplies V^T[32b + col]
    // of keys 16j + 4·half + {0..3, 8..11} and the probabilities of the same.
    // Keys past the wave's last query may be those of the workgroup's later
    // queries: their values are left out, as they may not be finite.
    auto add = [&](auto past) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 2; j++) {
#pragma unroll
        for (int b = 0; b < OB; b++) {
          const uint32_t d = 32 * b + col;
          const ph4_t v0 = *reinterpret_cast<const ph4_t *>(&v_s[buf][((4 * j + half_id) * HD + d) * 4]);
          const ph4_t v1 = *reinterpret_cast<const ph4_t *>(&v_s[buf][((4 * j + 2 + half_id) * HD + d) * 4]);
          ph8_t a = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
          if constexpr (past) {
#pragma unroll
            for (int i = 0; i < 8; i++)
              if (kb + 16 * j + 4 * half_id + (i & 4) * 2 + (i & 3) >= kend) a[i] = (_Float16)0.f;
          }
          o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ph[j], o[b], 0, 0, 0);
          o[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pl[j], o[b], 0, 0, 0);
        }
      }
    };
    if (kb + kPrefKeys > kend)
      add(std::true_type{});
    else
      add(std::false_type{});
  };
  if (b_lo < b_hi) {
    stage(0);
    load(min(b_lo + 1, b_hi - 1));
    lds_barrier();
    for (uint32_t b = b_lo; b < b_hi; b++) {
      const int buf = (int)((b - b_lo) & 1);
      // Buffer buf ^ 1 was read before the last barrier.
      if (b + 1 < b_hi) {
        stage(buf ^ 1);
        load(min(b + 2, b_hi - 1));
      }
      if (active && b * kPrefKeys < kend) block(b * kPrefKeys, buf);
      lds_barrier();
    }
  }
  if (!active) return;
  const float l_all = l_run + __shfl_xor(l_run, 32, 64);
  if (q0 + col >= n_queries) return;
  float inv = 1.f / l_all;
  float *orow = out + (uint64_t)(q0 + col) * out_stride + (uint64_t)head * HD;
  if (n_split > 1) {
    // Unnormalised partial (max in log2, sum, output) of this split,
    // combined by k_attn_prefill_combine.
    float *pp = partials + (((uint64_t)(q0 + col) * n_heads + head) * n_split + split) * (HD + 2);
    if (half_id == 0) {
      pp[0] = m_run;
      pp[1] = l_all;
    }
    orow = pp + 2;
    inv = 1.f;
  }
#pragma unroll
  for (int b = 0; b < OB; b++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const uint32_t d = 32 * b + 8 * g + 4 * half_id;
      if (n_split > 1) {
#pragma unroll
        for (int i = 0; i < 4; i++) orow[d + i] = o[b][4 * g + i];
      } else {
        *reinterpret_cast<float4 *>(orow + d) =
            float4{o[b][4 * g] * inv * gate.at(q0 + col, head, d), o[b][4 * g + 1] * inv * gate.at(q0 + col, head, d + 1),
                   o[b][4 * g + 2] * inv * gate.at(q0 + col, head, d + 2),
                   o[b][4 * g + 3] * inv * gate.at(q0 + col, head, d + 3)};
      }
    }
}

// Output of each (query, head) from its key splits' partials: one workgroup
// of HD threads per (query, head).
template <int HD>
__global__ __launch_bounds__(HD) void k_attn_prefill_combine(const float *__restrict__ partials, float *__restrict__ out,
                                                              uint32_t n_heads, uint32_t n_split, uint32_t out_stride,
                                                              AttnGate gate) {
  const uint32_t slot = blockIdx.x, z = slot / n_heads, head = slot % n_heads, d = threadIdx.x;
  const float *pp = partials + (uint64_t)slot * n_split * (HD + 2);
  float M = -INFINITY;
  for (uint32_t sp = 0; sp < n_split; sp++) M = fmaxf(M, pp[sp * (HD + 2)]);
  float L = 0.f, O = 0.f;
  for (uint32_t sp = 0; sp < n_split; sp++) {
    const float w = __builtin_amdgcn_exp2f(pp[sp * (HD + 2)] - M);
    L = fmaf(pp[sp * (HD + 2) + 1], w, L);
    O = fmaf(pp[sp * (HD + 2) + 2 + d], w, O);
  }
  out[(uint64_t)z * out_stride + (uint64_t)head * HD + d] = O / L * gate.at(z, head, d);
}

bool attn_prefill_mfma_supported(uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, bool kv_half) {
  return kv_half && n_kv && n_heads % n_kv == 0 && n_heads / n_kv <= 4 &&
         (head_dim == 64 || head_dim == 128 || head_dim == 256);
}

uint64_t attn_prefill_partial_floats(uint32_t n_queries, uint32_t n_heads, uint32_t head_dim, uint32_t splits) {
  return (uint64_t)n_queries * n_heads * splits * (head_dim + 2);
}

uint32_t attn_prefill_splits(uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, uint32_t first_pos,
                             uint32_t n_queries, uint64_t partial_floats) {
  if (!n_queries || !n_heads) return 1;
  // Enough workgroups for two per CU (three, which heads of 64 have registers
  // for, made their kernel 4% faster and its combine as much slower), at least kMinSplitBlocks 32-key blocks
  // per split of the batch's middle tile, and no more partials than the
  // scratch holds.
  constexpr uint32_t kTargetGroups = 512, kMinSplitBlocks = 2, kMaxSplits = 16;
  // A workgroup holds at most 128 rows (queries x heads), and several splits
  // make fewer than 2·kTargetGroups workgroups.
  static_assert(kAttnPartialFloats >= (2ull * kTargetGroups - 2) * 128 * (256 + 2), "the op's partials");
  const uint32_t per_wg = kPrefQ * attn_prefill_tiles(n_heads / n_kv);
  const uint32_t tiles = (n_queries + per_wg - 1) / per_wg;
  uint32_t want = (kTargetGroups + tiles * n_kv - 1) / (tiles * n_kv);
  const uint32_t mid_blocks = (first_pos + (n_queries + 1) / 2 + kPrefKeys - 1) / kPrefKeys;
  want = std::min(want, mid_blocks / kMinSplitBlocks);
  want = std::min<uint32_t>(want, kMaxSplits);
  const uint64_t per_split = (uint64_t)n_queries * n_heads * (head_dim + 2);
  want = (uint32_t)std::min<uint64_t>(want, partial_floats / per_split);
  return std::max<uint32_t>(want, 1);
}

void run_attn_prefill_mfma(hipStream_t s, const float *q, const void *k_cache, const void *v_cache, float *out,
                           uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, uint32_t first_pos,
                           uint32_t n_queries, uint32_t q_stride, uint32_t out_stride, float scale, float *partials,
                           uint64_t partial_floats, const float *gate, uint32_t gate_head_stride,
                           uint32_t gate_query_stride) {
  if (!n_queries || !n_heads) return;
  const uint32_t n_split =
      partials ? attn_prefill_splits(n_heads, n_kv, head_dim, first_pos, n_queries, partial_floats) : 1;
  const uint32_t per_wg = kPrefQ * attn_prefill_tiles(n_heads / n_kv);
  const dim3 grid((n_queries + per_wg - 1) / per_wg, n_kv, n_split);
  const _Float16 *kc = static_cast<const _Float16 *>(k_cache);
  const _Float16 *vc = static_cast<const _Float16 *>(v_cache);
  const AttnGate g{gate, gate_head_stride, gate_query_stride};
  auto go = [&](auto hd) {
    constexpr int HD = decltype(hd)::value;
    k_attn_prefill<HD><<<grid, 256, 0, s>>>(q, kc, vc, out, n_heads, n_kv, first_pos, n_queries, q_stride,
                                            out_stride, scale, partials, g);
    if (n_split > 1)
      k_attn_prefill_combine<HD><<<n_queries * n_heads, HD, 0, s>>>(partials, out, n_heads, n_split, out_stride, g);
  };
  if (head_dim == 64)
    go(std::integral_constant<int, 64>{});
  else if (head_dim == 128)
    go(std::integral_constant<int, 128>{});
  else
    go(std::integral_constant<int, 256>{});
}

}  // namespace bch

using namespace bch;

extern "C" int bch_attention_prefill(bch_ctx *ctx, bch_view q, bch_view k_cache, bch_view v_cache, bch_view out,
                                     uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim, uint32_t first_pos,
                                     uint32_t n_queries, uint32_t n_ctx) {
  const uint64_t last_pos = (uint64_t)first_pos + n_queries;
  if (!attn_prefill_mfma_supported(n_heads, n_kv_heads, head_dim, true) || last_pos > n_ctx)
    return fail(BCH_ERR_ATTENTION_LIMITS,
                "attention_prefill: f16 caches, heads of 64, 128 or 256, at most 4 query heads per KV head and positions "
                "inside the context, got %u and %u heads of %u at positions up to %llu of %u",
                n_heads, n_kv_heads, head_dim, (unsigned long long)last_pos, n_ctx);
  const uint64_t query_bytes = (uint64_t)n_queries * n_heads * head_dim * 4;
  const uint64_t cache_bytes = last_pos * n_kv_heads * head_dim * 2;
  const float *qp;
  const void *kp, *vp;
  float *op;
  BCH_TRY(view_ptr(ctx, "attention_prefill", q, query_bytes, &qp));
  BCH_TRY(view_ptr(ctx, "attention_prefill", k_cache, cache_bytes, &kp));
  BCH_TRY(view_ptr(ctx, "attention_prefill", v_cache, cache_bytes, &vp));
  BCH_TRY(view_ptr(ctx, "attention_prefill", out, query_bytes, &op));
  if (reinterpret_cast<uintptr_t>(kp) % 16 || reinterpret_cast<uintptr_t>(vp) % 16 ||
      reinterpret_cast<uintptr_t>(qp) % 16 || reinterpret_cast<uintptr_t>(op) % 16)
    return fail(BCH_ERR_ARGUMENT, "attention_prefill: operands must be 16-byte aligned");
  // Key splits with their partials in memory that the context has held since
  // it was opened (unsplit without it): a call allocates and waits for nothing.
  return launch(ctx, {"attention_prefill", 0, 0, 0}, [&](hipStream_t s) {
    run_attn_prefill_mfma(s, qp, kp, vp, op, n_heads, n_kv_heads, head_dim, first_pos, n_queries,
                          n_heads * head_dim, n_heads * head_dim, 1.0f / sqrtf((float)head_dim), ctx->attn_partials,
                          ctx->attn_partials ? kAttnPartialFloats : 0, nullptr, 0, 0);
  });
}
