// Gated DeltaNet kernels and the output gate of Qwen3.5's attention: the
// MI355X counterparts of gdn_conv / gdn_gates / gdn_recurrence /
// gdn_gated_norm / attention_gate (crates/bobcat-metal/src/gdn.metal) and of
// the CPU Model::delta_net (crates/bobcat/src/qwen35.rs:430-516).
//
// The recurrence gives every column of a value head's state its own wave:
// a column evolves on its own given the token's key, query, value entry and
// gates (remembered_c = Σ_r S[r][c]·k[r], S[r][c] += k[r]·β(v_c − remembered_c),
// out_c = Σ_r S[r][c]·q[r]), so the k_dim rows of a column live in the
// registers of one wave (k_dim/64 per lane) for a whole prefill batch and the
// two dot products per token are wave reductions.  16 heads of 128 columns
// make 2048 waves.  The workgroup stages 32 tokens at a time in LDS (the
// normalised query and key, its columns' values, the gates), so the
// sequential token loop reads LDS instead of waiting on memory per token.
#include <cmath>
#include <type_traits>

#include "device.h"
#include "kernels.h"
#include "runtime.h"

namespace bch {

constexpr int kGdnCols = 4;  // columns (waves) per workgroup

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
// transformers' softplus returns its input above 20 (qwen35.rs:775-778).
__device__ __forceinline__ float softplus_f(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

constexpr int kGdnChunk = 32;  // tokens staged in LDS at a time

template <int RPL>
__global__ __launch_bounds__(kGdnCols * 64) void k_gdn_recurrence(GdnArgs a) {
  constexpr int KD = RPL * 64;  // k_dim
  // A chunk of tokens staged by the workgroup: the l2-normalised query
  // (times q_scale) and key of this head, the four columns' values, and
  // the gates.  The token loop then waits on LDS, not on memory.
  __shared__ float qs[kGdnChunk][KD], ks[kGdnChunk][KD], vs[kGdnChunk][kGdnCols], bs[kGdnChunk], ds[kGdnChunk];
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t col0 = blockIdx.x * kGdnCols, col = col0 + wave, head = blockIdx.y;
  const uint32_t key_head = head % a.n_k, key_dim = a.n_k * a.k_dim, conv_dim = 2 * key_dim + a.n_v * a.v_dim;
  const uint32_t r0 = lane * RPL;
  float *S = a.state + (uint64_t)head * a.k_dim * a.v_dim;
  float rows[RPL];
#pragma unroll
  for (int i = 0; i < RPL; i++) rows[i] = S[(uint64_t)(r0 + i) * a.v_dim + col];
  for (uint32_t t0 = 0; t0 < a.n_tokens; t0 += kGdnChunk) {
    const uint32_t n = min((uint32_t)kGdnChunk, a.n_tokens - t0);
    __syncthreads();  // the previous chunk is consumed
    // Wave w stages tokens w, w + 4, ...: l2_normalize of the query and the
    // key (qwen35.rs:464-470), each lane holding rows r0 .. r0+RPL-1.
    for (uint32_t j = wave; j < n; j += kGdnCols) {
      const float *tok = a.y + (uint64_t)(t0 + j) * conv_dim;
      float q[RPL], k[RPL], sq = 0.f, sk = 0.f;
#pragma unroll
      for (int i = 0; i < RPL; i++) {
        q[i] = tok[key_head * a.k_dim + r0 + i];
        k[i] = tok[key_dim + key_head * a.k_dim + r0 + i];
      }
#pragma unroll
      for (int i = 0; i < RPL; i++) {
        sq = fmaf(q[i], q[i], sq);
        sk = fmaf(k[i], k[i], sk);
      }
      sq = wave_sum(sq);
      sk = wave_sum(sk);
      const float fq = a.q_scale / sqrtf(sq + 1e-6f), fk = 1.0f / sqrtf(sk + 1e-6f);
#pragma unroll
      for (int i = 0; i < RPL; i++) {
        qs[j][r0 + i] = q[i] * fq;
        ks[j][r0 + i] = k[i] * fk;
      }
      if (lane < kGdnCols) vs[j][lane] = tok[2 * key_dim + head * a.v_dim + col0 + lane];
      if (lane == 0) {
        const uint64_t gs = a.gate_stride ? a.gate_stride : a.n_v;
        const float b = a.beta[(uint64_t)(t0 + j) * gs + head];
        const float d = a.alpha[(uint64_t)(t0 + j) * gs + head];
        bs[j] = a.raw_gates ? sigmoid_f(b) : b;
        ds[j] = a.raw_gates ? expf(a.a[head] * softplus_f(d + a.dt_bias[head])) : d;
      }
    }
    __syncthreads();
    for (uint32_t j = 0; j < n; j++) {
      const float decay = ds[j], beta = bs[j];
      float rem = 0.f;
#pragma unroll
      for (int i = 0; i < RPL; i++) {
        rows[i] *= decay;
        rem = fmaf(rows[i], ks[j][r0 + i], rem);
      }
      rem = wave_sum(rem);
      const float delta = (vs[j][wave] - rem) * beta;
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < RPL; i++) {
        rows[i] = fmaf(ks[j][r0 + i], delta, rows[i]);
        o = fmaf(rows[i], qs[j][r0 + i], o);
      }
      o = wave_sum(o);
      if (lane == 0) a.out[(uint64_t)(t0 + j) * a.n_v * a.v_dim + head * a.v_dim + col] = o;
    }
  }
#pragma unroll
  for (int i = 0; i < RPL; i++) S[(uint64_t)(r0 + i) * a.v_dim + col] = rows[i];
}

// One token (decode): a workgroup per value head, CB blocks of 64 columns;
// in block cb lane c owns column 64·cb + c of the head's state and wave w of
// the block rows [w·KD/4, (w+1)·KD/4), so each row of a block is one
// coalesced 256-byte access; the two dot products over the rows are per-lane
// sums, then a sum over the block's four waves in LDS (in wave order).  (The
// wave-per-column form above spreads a column over 64 lanes, which touches a
// cache line per row and per column.)  With norm_w the head's output gets
// the gated norm of k_gdn_gated_norm in the same workgroup.
template <int KD, int CB>
__global__ __launch_bounds__(256 * CB) void k_gdn_step(GdnArgs a) {
  constexpr int RW = KD / 4;  // rows per wave
  __shared__ float qn[KD], kn[KD], part[CB][4][64];
  __shared__ float gate_s[2], ss_s[CB];
  const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t cb = wave / 4, wq = wave % 4;
  const uint32_t head = blockIdx.y, col = cb * 64 + lane;
  const uint32_t key_head = head % a.n_k, key_dim = a.n_k * a.k_dim;
  const float *tok = a.y;
  float *S = a.state + (uint64_t)head * KD * a.v_dim + col;
  // The token's small inputs first, then the state rows: memory returns in
  // issue order, so the norms below wait for the small loads alone and run
  // while the state streams in.  The loads are unconditional (every wave
  // reads a query or key row; waves past 1 discard theirs), so the waits
  // count exactly.
  const float *src = tok + (wave == 1 ? key_dim : 0u) + key_head * KD;
  float e[KD / 64];
#pragma unroll
  for (int i = 0; i < KD / 64; i++) e[i] = src[lane * (KD / 64) + i];
  const float v = tok[2 * key_dim + head * a.v_dim + col];
  const float gz = a.norm_w ? a.gate_z[(uint64_t)head * a.v_dim + col] : 0.f;
  const float nw = a.norm_w ? a.norm_w[col] : 0.f;
  // The head's gate inputs (uniform: scalar loads).
  const float gb = a.beta[head], gd = a.alpha[head];
  const float ga = a.raw_gates ? a.a[head] : 0.f, gdt = a.raw_gates ? a.dt_bias[head] : 0.f;
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  float rows[RW];
#pragma unroll
  for (int i = 0; i < RW; i++) rows[i] = S[(uint64_t)(wq * RW + i) * a.v_dim];
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // Waves 0 and 1 normalise the query and the key (qwen35.rs:464-470).
  if (wave < 2) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < KD / 64; i++) ss = fmaf(e[i], e[i], ss);
    ss = wave_sum(ss);
    const float f = wave == 0 ? a.q_scale / sqrtf(ss + 1e-6f) : 1.0f / sqrtf(ss + 1e-6f);
#pragma unroll
    for (int i = 0; i < KD / 64; i++) (wave == 0 ? qn : kn)[lane * (KD / 64) + i] = e[i] * f;
  } else if (wave == 2 && lane == 0) {
    gate_s[0] = a.raw_gates ? sigmoid_f(gb) : gb;
    gate_s[1] = a.raw_gates ? expf(ga * softplus_f(gd + gdt)) : gd;
  }
  __syncthreads();
  const float beta = gate_s[0], decay = gate_s[1];
  float rem = 0.f;
#pragma unroll
  for (int i = 0; i < RW; i++) {
    rows[i] *= decay;
    rem = fmaf(rows[i], kn[wq * RW + i], rem);
  }
  part[cb][wq][lane] = rem;
  __syncthreads();
  rem = (part[cb][0][lane] + part[cb][1][lane]) + (part[cb][2][lane] + part[cb][3][lane]);
  const float delta = (v - rem) * beta;
  float o = 0.f;
#pragma unroll
  for (int i = 0; i < RW; i++) {
    rows[i] = fmaf(kn[wq * RW + i], delta, rows[i]);
    o = fmaf(rows[i], qn[wq * RW + i], o);
    S[(uint64_t)(wq * RW + i) * a.v_dim] = rows[i];
  }
  __syncthreads();
  part[cb][wq][lane] = o;
  __syncthreads();
  o = (part[cb][0][lane] + part[cb][1][lane]) + (part[cb][2][lane] + part[cb][3][lane]);
  float *orow = a.out + (uint64_t)head * a.v_dim;
  if (!a.norm_w) {
    if (wq == 0) orow[col] = o;
    return;
  }
  // The gated norm of the head: RMS over its v_dim outputs (block sums in
  // block order), then w ⊙ (o·scale) ⊙ silu(z).
  if (wq == 0) {
    const float ss = wave_sum(o * o);
    if (lane == 0) ss_s[cb] = ss;
  }
  __syncthreads();
  if (wq != 0) return;
  float ss = 0.f;
#pragma unroll
  for (int b = 0; b < CB; b++) ss += ss_s[b];
  const float scale = rsqrtf(ss / (float)a.v_dim + a.norm_eps);
  orow[col] = nw * (o * scale) * (gz / (1.0f + expf(-gz)));
}

bool gdn_step_supported(const GdnArgs &a) {
  return a.n_tokens == 1 && a.v_dim % kGdnCols == 0 && a.v_dim % 64 == 0 && a.v_dim <= 256 &&
         (a.k_dim == 64 || a.k_dim == 128);
}

bool run_gdn_recurrence(hipStream_t s, const GdnArgs &a) {
  if (a.v_dim % kGdnCols || a.n_tokens == 0) return false;
  if (gdn_step_supported(a)) {
    const uint32_t cb = a.v_dim / 64;
    const dim3 grid(1, a.n_v);
#define BCH_STEP(KD, CB) k_gdn_step<KD, CB><<<grid, 256 * CB, 0, s>>>(a)
    if (a.k_dim == 64) {
      if (cb == 1) BCH_STEP(64, 1); else if (cb == 2) BCH_STEP(64, 2); else if (cb == 3) BCH_STEP(64, 3); else BCH_STEP(64, 4);
    } else {
      if (cb == 1) BCH_STEP(128, 1); else if (cb == 2) BCH_STEP(128, 2); else if (cb == 3) BCH_STEP(128, 3); else BCH_STEP(128, 4);
    }
#undef BCH_STEP
    return true;
  }
  const dim3 grid(a.v_dim / kGdnCols, a.n_v);
  if (a.k_dim == 64)
    k_gdn_recurrence<1><<<grid, kGdnCols * 64, 0, s>>>(a);
  else if (a.k_dim == 128)
    k_gdn_recurrence<2><<<grid, kGdnCols * 64, 0, s>>>(a);
  else
    return false;
  return true;
}

// --- chunked prefill ------------------------------------------------------
//
// The gated delta rule over a chunk of C tokens from the state S0 at its
// start, with gamma_t the product of the decays up to token t (from the
// chunk's start), reads (the WY/UT form of the delta rule):
//   A[t][s] = beta_t (gamma_t / gamma_s) k_t.k_s          s < t
//   (I + A) D = diag(beta) (V - diag(gamma) K S0)         D = the chunk's deltas
//   D = U - W S0,  U = (I + A)^-1 diag(beta) V,  W = (I + A)^-1 diag(beta gamma) K
//   O = diag(gamma) Q S0 + P D,  P[t][s] = (gamma_t / gamma_s) q_t.k_s   s <= t
//   S_C = gamma_C S0 + Kt^T D,   Kt[s] = (gamma_C / gamma_s) k_s
// which unrolls the per-token recurrence of qwen35.rs:475-511 exactly (in
// exact arithmetic).  k_gdn_chunk_prep computes W, U, P, diag(gamma) Q, Kt
// and gamma_C for every (chunk, head) at once: U and W by forward
// substitution over blocks of 16 tokens; the decays as differences of a
// float64 running sum of log-decays.  k_gdn_chunk_scan then carries the
// state through the chunks: each column of S evolves on its own, so a
// workgroup owns NC columns of one head and walks the chunks in order.

constexpr int kGdnC = 64;  // tokens per chunk

// The chunk matrices are stored as the scan's v_mfma_f32_16x16x4_f32 reads
// them: 16 rows x 16 columns at a time, 256 floats, lane l's four (row
// l%16, columns 4s + l/16 of k-steps s = 0..3) together.  Offset of element
// (i, k) of a matrix of 16·kb columns.
__device__ __forceinline__ uint32_t gdn_frag(uint32_t i, uint32_t k, uint32_t kb) {
  return ((i / 16 * kb + k / 16) * 64 + i % 16 + 16 * (k % 4)) * 4 + k / 4 % 4;
}

__host__ __device__ constexpr uint64_t gdn_chunk_floats(uint32_t kd, uint32_t vd) {
  return 64ull * (3ull * kd + vd) + 64ull * 64ull + 64ull;
}

typedef float gdn4_t __attribute__((ext_vector_type(4)));

// Whether no lane of the wave holds an infinity or a NaN.
__device__ __forceinline__ bool wave_finite(gdn4_t v) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; i++) bad |= (__float_as_uint(v[i]) & 0x7f800000u) == 0x7f800000u;
  return __ballot(bad) == 0;
}

// One workgroup of 8 waves per (chunk, head).  K K^T and Q K^T, the blocks
// of 16 tokens below the diagonal of the solve and the diagonal blocks'
// inverses (taken by substitution, 16 x 16) times the right-hand sides all
// run on f32 MFMAs: element i of an accumulator is row 4·(lane/16) + i, which
// a B operand reads at k-step i when the A operand takes its columns in that
// order, so a solved block feeds the next blocks from registers.  512 tokens,
// 16 heads of 128 x 128: 22 us; with one thread per column of [W | U]
// and FMA products it took 55, most of it LDS reads.
template <int KD>
__global__ __launch_bounds__(512) void k_gdn_chunk_prep(GdnArgs a, float *__restrict__ scratch, uint32_t n_chunks) {
  constexpr int C = kGdnC, KP = KD + 4, R = KD / 64, B = C / 16, KB = KD / 16, TP = 20;
  __shared__ __align__(16) float qs[C][KP], ks[C][KP];
  __shared__ __align__(16) float am[C][C + 4];    // -A, the blocks on and below the diagonal
  __shared__ __align__(16) float inv[B][16][TP];  // (I + A)^-1 of each diagonal block
  __shared__ float bs[C], wgam[C], gq[C], gk[C];
  __shared__ double lg[C];
  const uint32_t tid = threadIdx.x, lane = tid % 64, n = lane % 16, quad = lane / 16;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const uint32_t chunk = blockIdx.x, head = blockIdx.y;
  const uint32_t vd = a.v_dim;
  const uint32_t t0 = chunk * C, L = min((uint32_t)C, a.n_tokens - t0);
  const uint32_t key_head = head % a.n_k, key_dim = a.n_k * KD, conv_dim = 2 * key_dim + a.n_v * vd;
  float *base = scratch + ((uint64_t)head * n_chunks + chunk) * gdn_chunk_floats(KD, vd);
  float *Wg = base, *Ug = Wg + C * KD, *Qg = Ug + (uint64_t)C * vd, *Kt = Qg + C * KD, *Pg = Kt + C * KD;
  float *gC = Pg + C * C;
  // The l2-normalised query (times q_scale) and key of each token
  // (qwen35.rs:464-470); rows past the chunk's end are zero.  Wave w takes
  // tokens w, w+8, ..., all of their loads issued before any is used; the
  // value columns of the wave's first U tile are requested behind them.
  constexpr int TW = C / 8;  // tokens per wave
  float q[TW][R], k[TW][R];
#pragma unroll
  for (int jj = 0; jj < TW; jj++) {
    const uint32_t j = wave + 8 * jj;
    const float *tok = a.y + (uint64_t)(t0 + min(j, L - 1)) * conv_dim;
#pragma unroll
    for (int i = 0; i < R; i++) {
      q[jj][i] = j < L ? tok[key_head * KD + lane * R + i] : 0.f;
      k[jj][i] = j < L ? tok[key_dim + key_head * KD + lane * R + i] : 0.f;
    }
  }
  // Column 16·tile + n of V, rows 16b + 4·quad + i.
  gdn4_t v[B];
  auto load_v = [&](uint32_t tile) __attribute__((always_inline)) {
    const float *col = a.y + (uint64_t)t0 * conv_dim + 2 * key_dim + head * vd + min(16 * tile + n, vd - 1);
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t t = 16 * b + 4 * quad + i;
        const float x = col[(uint64_t)min(t, L - 1) * conv_dim];
        v[b][i] = t < L ? x : 0.f;
      }
  };
  load_v(wave);
#pragma unroll
  for (int jj = 0; jj < TW; jj++) {
    const uint32_t j = wave + 8 * jj;
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < R; i++) {
      sq = fmaf(q[jj][i], q[jj][i], sq);
      sk = fmaf(k[jj][i], k[jj][i], sk);
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    const float fq = a.q_scale / sqrtf(sq + 1e-6f), fk = 1.0f / sqrtf(sk + 1e-6f);
#pragma unroll
    for (int i = 0; i < R; i++) {
      qs[j][lane * R + i] = q[jj][i] * fq;
      ks[j][lane * R + i] = k[jj][i] * fk;
    }
  }
  // Gates: beta, and the running sum of the log-decays in float64.
  if (wave == 0) {
    float b = 0.f, l = 0.f;
    if (lane < L) {
      const uint64_t gs = a.gate_stride ? a.gate_stride : a.n_v;
      const float rb = a.beta[(uint64_t)(t0 + lane) * gs + head];
      const float rd = a.alpha[(uint64_t)(t0 + lane) * gs + head];
      b = a.raw_gates ? sigmoid_f(rb) : rb;
      l = a.raw_gates ? a.a[head] * softplus_f(rd + a.dt_bias[head]) : logf(rd);
    }
    double s = l;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double o = __shfl_up(s, off, 64);
      if (lane >= (uint32_t)off) s += o;
    }
    const double lC = __shfl(s, (int)L - 1, 64);
    bs[lane] = b;
    lg[lane] = s;
    wgam[lane] = lane < L ? b * expf((float)s) : 0.f;
    gq[lane] = lane < L ? expf((float)s) : 0.f;
    gk[lane] = lane < L ? expf((float)(lC - s)) : 0.f;
    if (lane == 0) gC[0] = expf((float)lC);
  }
  __syncthreads();
  // Waves 0-3: A's row block `wave`; waves 4-7: P's, the longest beside the
  // shortest of A on a SIMD.  Blocks above the diagonal are zero.
  {
    const bool is_a = wave < 4;
    const uint32_t rb = is_a ? wave : 7 - wave;
    const float *rows = is_a ? &ks[16 * rb + n][0] : &qs[16 * rb + n][0];
    gdn4_t acc[B];
#pragma unroll
    for (int b = 0; b < B; b++) acc[b] = gdn4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
      const gdn4_t rv = *reinterpret_cast<const gdn4_t *>(rows + 16 * kb + 4 * quad);
#pragma unroll
      for (int b = 0; b < B; b++) {
        if ((uint32_t)b > rb) continue;  // (uniform over the wave)
        const gdn4_t cv = *reinterpret_cast<const gdn4_t *>(&ks[16 * b + n][16 * kb + 4 * quad]);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[i], cv[i], acc[b], 0, 0, 0);
      }
    }
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t t = 16 * rb + 4 * quad + i, u = 16 * b + n;
        const float dec = (u <= t && t < L) ? expf((float)(lg[t] - lg[u])) : 0.f;
        // (Selected, not multiplied, to zero: a later token may not be finite.)
        if (is_a)
          am[t][u] = u < t ? -(bs[t] * dec * acc[b][i]) : 0.f;
        else
          Pg[gdn_frag(t, u, B)] = u <= t ? dec * acc[b][i] : 0.f;
      }
  }
  // diag(gamma) Q and Kt, by the four floats of a lane of the scan.
  for (uint32_t e = tid; e < (uint32_t)(C * KD / 4); e += 512) {
    const uint32_t l = e % 64, blk = e / 64, row = l % 16;
    const uint32_t t = 16 * (blk / KB) + row, r = 16 * (blk % KB) + l / 16;
    const uint32_t r2 = 16 * (blk / B) + row, t2 = 16 * (blk % B) + l / 16;
    gdn4_t qv, kv;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      qv[s] = gq[t] * qs[t][r + 4 * s];
      kv[s] = gk[t2 + 4 * s] * ks[t2 + 4 * s][r2];
    }
    *reinterpret_cast<gdn4_t *>(Qg + 4ull * e) = qv;
    *reinterpret_cast<gdn4_t *>(Kt + 4ull * e) = kv;
  }
  __syncthreads();
  // The inverse of diagonal block `wave`, a column per lane of 16.
  if (wave < B) {
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; t++) {
      x[t] = n == (uint32_t)t ? 1.f : 0.f;
      float row[16];
#pragma unroll
      for (int u4 = 0; u4 < (t + 3) / 4; u4++)
        *reinterpret_cast<gdn4_t *>(&row[4 * u4]) =
            *reinterpret_cast<const gdn4_t *>(&am[16 * wave + t][16 * wave + 4 * u4]);
#pragma unroll
      for (int u = 0; u < t; u++) x[t] = fmaf(row[u], x[u], x[t]);
    }
    if (quad == 0) {
#pragma unroll
      for (int t = 0; t < 16; t++) inv[wave][t][n] = x[t];
    }
  }
  __syncthreads();
  // X_b = inv_b (rhs_b - sum_{j<b} A_bj X_j), 16 columns of [W | U] at a time.
  // A block that is not finite is substituted row by row: the inverse's
  // zeros would carry its infinities and NaNs back to earlier tokens.
  auto solve = [&](gdn4_t (&x)[B]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < B; b++) {
#pragma unroll
      for (int j = 0; j < b; j++) {
        const gdn4_t av = *reinterpret_cast<const gdn4_t *>(&am[16 * b + n][16 * j + 4 * quad]);
#pragma unroll
        for (int i = 0; i < 4; i++) x[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], x[j][i], x[b], 0, 0, 0);
      }
      if (!wave_finite(x[b])) {
#pragma unroll 1
        for (uint32_t uq = 0; uq < 4; uq++)
#pragma unroll
          for (uint32_t ui = 0; ui < 4; ui++) {
            const float xu = __shfl(x[b][ui], (int)(16 * uq + n), 64);
#pragma unroll
            for (uint32_t i = 0; i < 4; i++)
              if (4 * quad + i > 4 * uq + ui)
                x[b][i] = fmaf(am[16 * b + 4 * quad + i][16 * b + 4 * uq + ui], xu, x[b][i]);
          }
        continue;
      }
      const gdn4_t iv = *reinterpret_cast<const gdn4_t *>(&inv[b][n][4 * quad]);
      gdn4_t y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; i++) y = __builtin_amdgcn_mfma_f32_16x16x4f32(iv[i], x[b][i], y, 0, 0, 0);
      x[b] = y;
    }
  };
  for (uint32_t tile = wave; tile < (uint32_t)KB; tile += 8) {
    gdn4_t x[B];
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t t = 16 * b + 4 * quad + i;
        x[b][i] = wgam[t] * ks[t][16 * tile + n];
      }
    solve(x);
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
      for (int i = 0; i < 4; i++)  // (the scan adds -W S0)
        Wg[gdn_frag(16 * b + 4 * quad + i, 16 * tile + n, KB)] = -x[b][i];
  }
  for (uint32_t tile = wave; 16 * tile < vd; tile += 8) {
    if (tile != wave) load_v(tile);
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) v[b][i] *= bs[16 * b + 4 * quad + i];
    solve(v);
    if (16 * tile + n < vd) {  // (a last tile of 8 columns)
#pragma unroll
      for (int b = 0; b < B; b++)
#pragma unroll
        for (int i = 0; i < 4; i++) Ug[(uint64_t)(16 * b + 4 * quad + i) * vd + 16 * tile + n] = v[b][i];
    }
  }
}

// The scan: a workgroup owns 16 columns of a head's state and walks the
// chunks; wave w computes tokens 16w .. 16w+15 of D and O and KD/4 rows of
// the state, all on f32 MFMAs (16x16x4, the same FMAs as a dot product's).
// The chunk's matrices come from memory straight into operand registers, each
// requested for the next chunk as soon as it is spent; only S and D pass
// through LDS, stored as the B operand reads them.  What bounds it is the
// chain of chunks, 112 MFMAs of 32 cycles per wave and chunk (heads of 128):
// 512 tokens, 16 heads of 128 x 128: 29 us (the FMA form with the matrices
// staged in LDS took 99).

template <int KD>
__global__ __launch_bounds__(256) void k_gdn_chunk_scan(GdnArgs a, const float *__restrict__ scratch,
                                                        uint32_t n_chunks) {
  constexpr int C = kGdnC, NC = 16, KB = KD / 16, CB = C / 16, MT = KD / 64;
  __shared__ __align__(16) float s_s[KD * NC], d_s[C * NC];
  const uint32_t tid = threadIdx.x, lane = tid % 64, vd = a.v_dim;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
  // Blocks are numbered so that the column blocks of one head run on one
  // XCD (workgroup i goes to XCD i % 8) and share its L2.
  const uint32_t n_cb = (vd + NC - 1) / NC, total = n_cb * a.n_v;
  uint32_t v = blockIdx.x;
  if (total % 8 == 0) v = (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8;
  const uint32_t head = v / n_cb, col = (v % n_cb) * NC + lane % 16, quad = lane / 16;
  const bool in = col < vd;  // (a last block of 8 columns)
  const uint32_t colc = min(col, vd - 1);
  float *S = a.state + (uint64_t)head * KD * vd + colc;
  // This lane's state: rows 16(MT·wave + m) + 4·quad + i of column col.
  gdn4_t st[MT];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int i = 0; i < 4; i++) st[m][i] = in ? S[(uint64_t)(16 * (MT * wave + m) + 4 * quad + i) * vd] : 0.f;
  // Element (k, col) of a B operand in LDS, for k = 16·b + 4·quad + i.
  auto b_at = [&](uint32_t b, int i) { return (b * 64 + lane % 16 + 16 * i) * 4 + quad; };
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int i = 0; i < 4; i++) s_s[b_at(MT * wave + m, i)] = st[m][i];

  const uint64_t per_chunk = gdn_chunk_floats(KD, vd);
  const float *base0 = scratch + (uint64_t)head * n_chunks * per_chunk;
  gdn4_t wf[KB], qf[KB], pf[CB], kf[MT][CB], u;
  float gC;
  auto part = [&](uint32_t c, uint64_t at, uint32_t blk) {
    return *reinterpret_cast<const gdn4_t *>(base0 + c * per_chunk + at + (blk * 64 + lane) * 4);
  };
  const uint64_t u_at = C * KD, q_at = u_at + (uint64_t)C * vd, k_at = q_at + C * KD, p_at = k_at + C * KD;
  auto load_wq = [&](uint32_t c) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < KB; b++) wf[b] = part(c, 0, wave * KB + b);
#pragma unroll
    for (int i = 0; i < 4; i++) u[i] = base0[c * per_chunk + u_at + (uint64_t)(16 * wave + 4 * quad + i) * vd + colc];
#pragma unroll
    for (int b = 0; b < KB; b++) qf[b] = part(c, q_at, wave * KB + b);
  };
  auto load_pk = [&](uint32_t c) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < CB; b++) pf[b] = part(c, p_at, wave * CB + b);
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int b = 0; b < CB; b++) kf[m][b] = part(c, k_at, (MT * wave + m) * CB + b);
    gC = base0[c * per_chunk + p_at + C * C];
  };
  load_wq(0);
  load_pk(0);
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();
  for (uint32_t c = 0; c < n_chunks; c++) {
    const uint32_t t0 = c * C, L = min((uint32_t)C, a.n_tokens - t0), next = min(c + 1, n_chunks - 1);
    // D = U - W S0 and O = diag(gamma) Q S0.
    gdn4_t d = u, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < KB; b++) {
      const gdn4_t sv = *reinterpret_cast<const gdn4_t *>(&s_s[(b * 64 + lane) * 4]);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        d = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][s], sv[s], d, 0, 0, 0);
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[b][s], sv[s], o, 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) d_s[b_at(wave, i)] = d[i];
    __builtin_amdgcn_sched_barrier(0);
    load_wq(next);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();  // D is whole; S0 is spent
    // O += P D, S_C = gamma_C S0 + Kt^T D.  P is zero above its diagonal, and
    // a later token's infinities and NaNs may not meet those zeros: the wave
    // leaves out the blocks past its own, and takes its own by selected FMAs
    // if its deltas are not finite.
    const bool finite = wave_finite(d);
    const uint32_t p_blocks = wave + (finite ? 1 : 0);
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int i = 0; i < 4; i++) st[m][i] *= gC;
#pragma unroll
    for (int b = 0; b < CB; b++) {
      const gdn4_t dv = *reinterpret_cast<const gdn4_t *>(&d_s[(b * 64 + lane) * 4]);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        if ((uint32_t)b < p_blocks) o = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[b][s], dv[s], o, 0, 0, 0);
#pragma unroll
        for (int m = 0; m < MT; m++) st[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[m][b][s], dv[s], st[m], 0, 0, 0);
      }
    }
    if (!finite) {
#pragma unroll 1
      for (uint32_t t = 0; t < 16; t++) {
        const float dv = d_s[(wave * 64 + lane % 16 + 16 * (t % 4)) * 4 + t / 4];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
          const float pv = base0[c * per_chunk + p_at + gdn_frag(16 * wave + 4 * quad + i, 16 * wave + t, CB)];
          o[i] = t <= 4 * quad + i ? fmaf(pv, dv, o[i]) : o[i];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_pk(next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int i = 0; i < 4; i++) s_s[b_at(MT * wave + m, i)] = st[m][i];
    float *orow = a.out + (uint64_t)(t0 + 16 * wave + 4 * quad) * a.n_v * vd + head * vd + colc;
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (in && 16 * wave + 4 * quad + i < L) orow[(uint64_t)i * a.n_v * vd] = o[i];
    lds_barrier();  // S_C is whole; D is spent
  }
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (in) S[(uint64_t)(16 * (MT * wave + m) + 4 * quad + i) * vd] = st[m][i];
}

constexpr int kGdnScanCols = 8;  // value columns come in multiples of this

bool gdn_chunked_supported(const GdnArgs &a) {
  return (a.k_dim == 64 || a.k_dim == 128) && a.v_dim % kGdnScanCols == 0 && a.v_dim <= 256 && a.n_tokens > 0;
}

uint64_t gdn_chunk_scratch_floats(uint32_t n_v, uint32_t k_dim, uint32_t v_dim, uint32_t n_tokens) {
  const uint64_t chunks = (n_tokens + kGdnC - 1) / kGdnC;
  return (uint64_t)n_v * chunks * gdn_chunk_floats(k_dim, v_dim);
}

bool run_gdn_chunked(hipStream_t s, const GdnArgs &a, float *scratch) {
  if (!gdn_chunked_supported(a)) return false;
  const uint32_t n_chunks = (a.n_tokens + kGdnC - 1) / kGdnC;
  const dim3 prep(n_chunks, a.n_v);
  const uint32_t scan = a.n_v * ((a.v_dim + 15) / 16);
  if (a.k_dim == 64) {
    k_gdn_chunk_prep<64><<<prep, 512, 0, s>>>(a, scratch, n_chunks);
    k_gdn_chunk_scan<64><<<scan, 256, 0, s>>>(a, scratch, n_chunks);
  } else {
    k_gdn_chunk_prep<128><<<prep, 512, 0, s>>>(a, scratch, n_chunks);
    k_gdn_chunk_scan<128><<<scan, 256, 0, s>>>(a, scratch, n_chunks);
  }
  return true;
}

// The causal convolution with SiLU of gdn_conv / the DeltaNet step
// (qwen35.rs:448-462): a thread takes one channel of kGdnConvTokens tokens,
// each input loaded once for all the outputs it enters (bound by memory: 512
// x 6,144 in 8 us, 19 with one output per thread).  Input t - past + i comes
// from the batch or, before it, from `hist`.  The newest term is added
// first, then the window oldest first, as the reference adds them.  A second
// launch then leaves the latest k-1 inputs in `hist` (after every read of
// the old history).
constexpr int kGdnConvTokens = 8;

template <int KS>
__global__ __launch_bounds__(256) void k_gdn_conv(const float *__restrict__ x, const float *__restrict__ taps,
                                                  const float *__restrict__ hist, float *__restrict__ y,
                                                  uint32_t channels, uint32_t n_tokens, uint32_t x_stride) {
  constexpr int TC = kGdnConvTokens, PAST = KS - 1;
  const uint32_t c = blockIdx.y * 256 + threadIdx.x, t0 = blockIdx.x * TC;
  if (c >= channels) return;
  float tp[KS], w[TC + PAST];
#pragma unroll
  for (int i = 0; i < TC + PAST; i++) {
    const int src = (int)t0 - PAST + i;
    if (src >= 0)
      w[i] = x[(uint64_t)min((uint32_t)src, n_tokens - 1) * x_stride + c];
    else
      w[i] = hist[(uint64_t)c * PAST + (PAST + src)];  // (first token block only)
  }
#pragma unroll
  for (int k = 0; k < KS; k++) tp[k] = taps[(uint64_t)c * KS + k];
#pragma unroll
  for (int j = 0; j < TC; j++) {
    float sum = tp[PAST] * w[j + PAST];
#pragma unroll
    for (int k = 0; k < PAST; k++) sum += tp[k] * w[j + k];
    if (t0 + j < n_tokens) y[(uint64_t)(t0 + j) * channels + c] = sum / (1.0f + expf(-sum));
  }
}

__global__ void k_gdn_conv_history(const float *__restrict__ x, float *__restrict__ hist, uint32_t channels,
                                   uint32_t ksize, uint32_t n_tokens, uint32_t x_stride) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const uint32_t past = ksize - 1;
  float window[kGdnMaxKernel - 1];
  for (uint32_t j = 0; j < past; j++) {
    const int src = (int)n_tokens - (int)past + (int)j;
    window[j] = src >= 0 ? x[(uint64_t)src * x_stride + c] : hist[(uint64_t)c * past + (past + src)];
  }
  for (uint32_t j = 0; j < past; j++) hist[(uint64_t)c * past + j] = window[j];
}

void run_gdn_conv(hipStream_t s, const float *x, const float *taps, float *hist, float *y, uint32_t channels,
                  uint32_t ksize, uint32_t n_tokens, uint32_t x_stride) {
  const uint64_t n = (uint64_t)n_tokens * channels;
  if (!n) return;
  const uint32_t xs = x_stride ? x_stride : channels;
  const dim3 grid((n_tokens + kGdnConvTokens - 1) / kGdnConvTokens, (channels + 255) / 256);
  auto go = [&](auto k) {
    k_gdn_conv<decltype(k)::value><<<grid, 256, 0, s>>>(x, taps, hist, y, channels, n_tokens, xs);
  };
  switch (ksize) {
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    case 6: go(std::integral_constant<int, 6>{}); break;
    case 7: go(std::integral_constant<int, 7>{}); break;
    default: go(std::integral_constant<int, 8>{}); break;
  }
  k_gdn_conv_history<<<(channels + 255) / 256, 256, 0, s>>>(x, hist, channels, ksize, n_tokens, xs);
}

// gdn_gates (gdn.metal:125-149): beta <- sigmoid(beta), alpha <- the decay
// exp(a·softplus(alpha + dt_bias)), per value head of each token.
__global__ void k_gdn_gates(float *beta, float *alpha, const float *a, const float *dt_bias, uint32_t n_v,
                            uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t h = i % n_v;
  beta[i] = sigmoid_f(beta[i]);
  alpha[i] = expf(a[h] * softplus_f(alpha[i] + dt_bias[h]));
}

void run_gdn_gates(hipStream_t s, float *beta, float *alpha, const float *a, const float *dt_bias, uint32_t n_v,
                   uint32_t n) {
  k_gdn_gates<<<(n + 255) / 256, 256, 0, s>>>(beta, alpha, a, dt_bias, n_v, n);
}

// The gated output norm (qwen35.rs:505-511): one wave per row of v_dim.
__global__ __launch_bounds__(64) void k_gdn_gated_norm(float *x, const float *__restrict__ w,
                                                       const float *__restrict__ z, uint32_t v_dim, float eps,
                                                       uint32_t n_v, uint32_t z_stride) {
  float *row = x + (uint64_t)blockIdx.x * v_dim;
  const float *g = z_stride ? z + (uint64_t)(blockIdx.x / n_v) * z_stride + (uint64_t)(blockIdx.x % n_v) * v_dim
                            : z + (uint64_t)blockIdx.x * v_dim;
  float ss = 0.f;
  for (uint32_t i = threadIdx.x; i < v_dim; i += 64) ss = fmaf(row[i], row[i], ss);
  ss = wave_sum(ss);
  const float scale = (float)(1.0 / sqrt((double)ss / (double)v_dim + (double)eps));
  for (uint32_t i = threadIdx.x; i < v_dim; i += 64) {
    const float gi = g[i];
    row[i] = w[i] * (row[i] * scale) * (gi / (1.0f + expf(-gi)));
  }
}

void run_gdn_gated_norm(hipStream_t s, float *x, const float *w, const float *z, uint32_t v_dim, uint32_t n_rows,
                        float eps, uint32_t n_v, uint32_t z_stride) {
  k_gdn_gated_norm<<<n_rows, 64, 0, s>>>(x, w, z, v_dim, eps, std::max(1u, n_v), z_stride);
}

// attention_gate (gdn.metal:306-322): each query head's output times the
// sigmoid of its gate, which follows its queries in the projection.
__global__ void k_attention_gate(float *attn, const float *q_gate, uint32_t head_dim, uint32_t q_dim, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t t = i / q_dim;
  const uint32_t e = (uint32_t)(i % q_dim), h = e / head_dim, d = e % head_dim;
  attn[i] *= sigmoid_f(q_gate[t * 2 * q_dim + (uint64_t)(2 * h + 1) * head_dim + d]);
}

void run_attention_gate(hipStream_t s, float *attn, const float *q_gate, uint32_t head_dim, uint32_t q_dim,
                        uint32_t n_tokens) {
  const uint64_t n = (uint64_t)n_tokens * q_dim;
  k_attention_gate<<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(attn, q_gate, head_dim, q_dim, n);
}

}  // namespace bch

// ---------------------------------------------------------------------
// C ABI (Metal::gdn_conv / gdn_gates / gdn_recurrence / gdn_gated_norm /
// attention_gate, crates/bobcat-metal/src/backend.rs).
// ---------------------------------------------------------------------

using namespace bch;

extern "C" int bch_gdn_conv(bch_ctx *ctx, bch_view x, bch_view taps, bch_view history, bch_view y, uint32_t channels,
                            uint32_t kernel_size, uint32_t n_tokens) {
  if (kernel_size < 2 || kernel_size > kGdnMaxKernel)
    return fail(BCH_ERR_DELTANET_LIMITS, "gdn_conv: 2 to %u taps, got %u", kGdnMaxKernel, kernel_size);
  const float *xp, *tp;
  float *hp, *yp;
  BCH_TRY(view_ptr(ctx, "gdn_conv", x, (uint64_t)n_tokens * channels * 4, &xp));
  BCH_TRY(view_ptr(ctx, "gdn_conv", taps, (uint64_t)channels * kernel_size * 4, &tp));
  BCH_TRY(view_ptr(ctx, "gdn_conv", history, (uint64_t)channels * (kernel_size - 1) * 4, &hp));
  BCH_TRY(view_ptr(ctx, "gdn_conv", y, (uint64_t)n_tokens * channels * 4, &yp));
  return launch(ctx, {"gdn_conv", channels, kernel_size, 0},
                [&](hipStream_t s) { run_gdn_conv(s, xp, tp, hp, yp, channels, kernel_size, n_tokens); });
}

extern "C" int bch_gdn_gates(bch_ctx *ctx, bch_view beta, bch_view alpha, bch_view a, bch_view dt_bias,
                             uint32_t n_v_heads, uint32_t n) {
  if (n_v_heads == 0) return fail(BCH_ERR_ARGUMENT, "gdn_gates: no heads");
  float *bp, *ap;
  const float *a_p, *dp;
  BCH_TRY(view_ptr(ctx, "gdn_gates", beta, (uint64_t)n * 4, &bp));
  BCH_TRY(view_ptr(ctx, "gdn_gates", alpha, (uint64_t)n * 4, &ap));
  BCH_TRY(view_ptr(ctx, "gdn_gates", a, (uint64_t)n_v_heads * 4, &a_p));
  BCH_TRY(view_ptr(ctx, "gdn_gates", dt_bias, (uint64_t)n_v_heads * 4, &dp));
  return launch(ctx, {"gdn_gates", n, n_v_heads, 0}, [&](hipStream_t s) { run_gdn_gates(s, bp, ap, a_p, dp, n_v_heads, n); });
}

extern "C" int bch_gdn_recurrence(bch_ctx *ctx, bch_view y, bch_view beta, bch_view decay, bch_view state,
                                  bch_view out, const bch_delta_shape *shape, uint32_t n_tokens, float q_scale) {
  if (!shape) return fail(BCH_ERR_ARGUMENT, "gdn_recurrence: no shape");
  const uint32_t nk = shape->n_k_heads, nv = shape->n_v_heads, dk = shape->k_dim, dv = shape->v_dim;
  if (nk == 0 || nv % nk || (dk != 64 && dk != 128) || dv == 0 || dv % kGdnCols)
    return fail(BCH_ERR_DELTANET_LIMITS,
                "gdn_recurrence: key heads of 64 or 128, value heads a multiple of %d and of the key heads "
                "(got %u/%u heads of %u/%u)", kGdnCols, nk, nv, dk, dv);
  GdnArgs a{};
  const uint64_t conv_dim = 2ull * nk * dk + (uint64_t)nv * dv;
  BCH_TRY(view_ptr(ctx, "gdn_recurrence", y, (uint64_t)n_tokens * conv_dim * 4, &a.y));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence", beta, (uint64_t)n_tokens * nv * 4, &a.beta));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence", decay, (uint64_t)n_tokens * nv * 4, &a.alpha));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence", state, (uint64_t)nv * dk * dv * 4, &a.state));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence", out, (uint64_t)n_tokens * nv * dv * 4, &a.out));
  a.n_k = nk;
  a.n_v = nv;
  a.k_dim = dk;
  a.v_dim = dv;
  a.n_tokens = n_tokens;
  a.q_scale = q_scale;
  a.raw_gates = false;
  if (n_tokens == 0) return BCH_OK;
  return launch(ctx, {"gdn_recurrence", nv, dv, (uint64_t)nv * dk * dv * 8},
                [&](hipStream_t s) { run_gdn_recurrence(s, a); });
}

extern "C" uint64_t bch_gdn_chunk_scratch_floats(const bch_delta_shape *shape, uint32_t n_tokens) {
  if (!shape) return 0;
  return gdn_chunk_scratch_floats(shape->n_v_heads, shape->k_dim, shape->v_dim, n_tokens);
}

extern "C" int bch_gdn_recurrence_chunked(bch_ctx *ctx, bch_view y, bch_view beta, bch_view decay, bch_view state,
                                          bch_view out, const bch_delta_shape *shape, uint32_t n_tokens,
                                          float q_scale, bch_view scratch) {
  if (!shape) return fail(BCH_ERR_ARGUMENT, "gdn_recurrence_chunked: no shape");
  const uint32_t nk = shape->n_k_heads, nv = shape->n_v_heads, dk = shape->k_dim, dv = shape->v_dim;
  if (nk == 0 || nv % nk || (dk != 64 && dk != 128) || dv == 0 || dv % kGdnScanCols || dv > 256)
    return fail(BCH_ERR_DELTANET_LIMITS,
                "gdn_recurrence_chunked: key heads of 64 or 128, value heads of at most 256 and a multiple of %d, "
                "value heads a multiple of the key heads (got %u/%u heads of %u/%u)",
                kGdnScanCols, nk, nv, dk, dv);
  GdnArgs a{};
  const uint64_t conv_dim = 2ull * nk * dk + (uint64_t)nv * dv;
  BCH_TRY(view_ptr(ctx, "gdn_recurrence_chunked", y, (uint64_t)n_tokens * conv_dim * 4, &a.y));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence_chunked", beta, (uint64_t)n_tokens * nv * 4, &a.beta));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence_chunked", decay, (uint64_t)n_tokens * nv * 4, &a.alpha));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence_chunked", state, (uint64_t)nv * dk * dv * 4, &a.state));
  BCH_TRY(view_ptr(ctx, "gdn_recurrence_chunked", out, (uint64_t)n_tokens * nv * dv * 4, &a.out));
  float *sp;
  BCH_TRY(view_ptr(ctx, "gdn_recurrence_chunked", scratch, gdn_chunk_scratch_floats(nv, dk, dv, n_tokens) * 4, &sp));
  if (reinterpret_cast<uintptr_t>(sp) % 16) return fail(BCH_ERR_ARGUMENT, "gdn_recurrence_chunked: scratch not 16-byte aligned");
  a.n_k = nk;
  a.n_v = nv;
  a.k_dim = dk;
  a.v_dim = dv;
  a.n_tokens = n_tokens;
  a.q_scale = q_scale;
  a.raw_gates = false;
  if (n_tokens == 0) return BCH_OK;
  return launch(ctx, {"gdn_recurrence_chunked", nv, dv, (uint64_t)nv * dk * dv * 8},
                [&](hipStream_t s) { run_gdn_chunked(s, a, sp); });
}

extern "C" int bch_gdn_gated_norm(bch_ctx *ctx, bch_view x, bch_view weight, bch_view z, uint32_t v_dim, uint32_t n_rows,
                                  float eps) {
  float *xp;
  const float *wp, *zp;
  BCH_TRY(view_ptr(ctx, "gdn_gated_norm", x, (uint64_t)n_rows * v_dim * 4, &xp));
  BCH_TRY(view_ptr(ctx, "gdn_gated_norm", weight, (uint64_t)v_dim * 4, &wp));
  BCH_TRY(view_ptr(ctx, "gdn_gated_norm", z, (uint64_t)n_rows * v_dim * 4, &zp));
  return launch(ctx, {"gdn_gated_norm", n_rows, v_dim, 0},
                [&](hipStream_t s) { run_gdn_gated_norm(s, xp, wp, zp, v_dim, n_rows, eps); });
}

extern "C" int bch_attention_gate(bch_ctx *ctx, bch_view attn, bch_view q_gate, uint32_t head_dim, uint32_t q_dim,
                                  uint32_t n_tokens) {
  if (head_dim == 0 || q_dim % head_dim) return fail(BCH_ERR_GATE_SHAPE, "attention_gate: %u is not whole heads of %u", q_dim, head_dim);
  float *ap;
  const float *gp;
  BCH_TRY(view_ptr(ctx, "attention_gate", attn, (uint64_t)n_tokens * q_dim * 4, &ap));
  BCH_TRY(view_ptr(ctx, "attention_gate", q_gate, (uint64_t)n_tokens * 2 * q_dim * 4, &gp));
  return launch(ctx, {"attention_gate", n_tokens, q_dim, 0},
                [&](hipStream_t s) { run_attention_gate(s, ap, gp, head_dim, q_dim, n_tokens); });
}
