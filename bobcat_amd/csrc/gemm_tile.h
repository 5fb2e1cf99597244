// The prefill GEMM tile: D[token][row] = Σ_k X[token][k]·W[row][k] on MFMA,
// the quantised weights converted to fp16 in LDS on the way (matmul.hip
// chooses the tile and launches it).
//
// A workgroup of four waves, one per SIMD, computes 32·MB weight rows x
// 32·NB·(4/WR) tokens; a wave owns NB blocks of 32 tokens against MB/WR of
// the row blocks (v_mfma_f32_32x32x16_f16, the inputs as the M operand, so D
// has rows along the lanes and stores of 32 rows are contiguous).
//
// What bounds it: issue slots.  A wave issues an instruction every ~5 cycles
// and a 32x32x16 MFMA occupies the matrix core for 33.6: with six other
// instructions beside it an MFMA takes 39.6 cycles, with eight 60 (measured in
// registers alone), and there is no second wave on the SIMD to hide more.
// Hence:
//  * The inputs are stored fragment-major (frag_offset): each wave load is
//    1 KB of consecutive bytes straight into MFMA operand registers.  Rows
//    of tokens (32 cache lines per load) kept the L1 address path busy for
//    longer than the MFMAs.
//  * Weights are converted with 1.6 instructions each: the quant bits of two
//    weights, masked, are a pair of subnormal fp16 integers, and
//    v_fma_mix{lo,hi}_f16 scales, subtracts and rounds in one.  Scales are
//    unpacked once per 256 columns.
//  * Loads, conversions and LDS accesses are spread between the MFMAs one by
//    one, held there by scheduling fences: the compiler's own order (and its
//    group scheduling) left runs of a hundred instructions without an MFMA.
//  * Every load has two to four stages to arrive and the LDS fragments of
//    the next k-step are read one k-step ahead, across the barrier too.
// 10752 x 2048 at 512 tokens: 34.3 us (657 TFLOP/s) against 50.4 for the
// kernel this replaces (LDS rows, row-major inputs, a barrier that drained the
// loads of every stage); 6144 x 2048: 21; 2048 x 10752 in four splits: 29.5
// against 40.4 in eight.  A call with its input conversion and the sum of its
// splits, before and after: 10752 x 2048 54.8 and 38.5 us, 6144 x 2048 35.4
// and 25, 2048 x 2048 24.7 and 19.6, 2048 x 10752 55.2 and 43.
#pragma once
#include <type_traits>
#include <utility>

#include "../../include/bobcat_hip.h"
#include "formats.h"
#include "frag.h"
#include "kernels.h"

namespace bch {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
// (Clang vector types rather than uint4: copies of uint4 become memcpy
// calls that kept these registers in scratch memory.)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }

template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
    (f(std::integral_constant<int, I>{}), ...);
  }(std::make_integer_sequence<int, N>{});
}

constexpr int kGk = 64;  // columns per stage

// N bytes (a multiple of 4) at a byte address of any alignment.
template <int N>
struct __attribute__((packed, aligned(1))) AnyBytes {
  uint32_t w[N / 4];
};
template <int N>
__device__ __forceinline__ void load_any(const uint8_t *p, uint32_t *out) {
  const AnyBytes<N> v = *reinterpret_cast<const AnyBytes<N> *>(p);
#pragma unroll
  for (int i = 0; i < N / 4; i++) out[i] = v.w[i];
}
// The same at an address aligned to N (at most 16).
template <int N>
__device__ __forceinline__ void load_aligned(const uint8_t *p, uint32_t *out) {
  load_any<N>(static_cast<const uint8_t *>(__builtin_assume_aligned(p, N < 16 ? N : 16)), out);
}
__device__ __forceinline__ uint32_t load_u16(const uint8_t *p) { return *reinterpret_cast<const uint16_t *>(p); }

// (v & m) | k in one instruction (the compiler forms two for such constants).
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t m, uint32_t k) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(m), "v"(k));
  return r;
}
// v shifted left by N (right by −N).
template <int N>
__device__ __forceinline__ uint32_t shl(uint32_t v) {
  if constexpr (N >= 0)
    return v << N;
  else
    return v >> -N;
}

// One thread's weights of one row: PQ = 8 or 16 consecutive columns of each
// 32-column half of a 64-column stage (columns PQ·c .. and 32 + PQ·c ..).
//   load_header(row, sb)  once per 256 columns (super-block sb)
//   load<S>(row, sb, st)  raw weights of stage S of super-block sb (stage st
//                         of the row), kept in slot S
//   unpack(c), scales<S>(c)  once per super-block and per stage
//   ints<S, HI, D>(), mix<S, HI, D>()  weights 4D .. 4D+3 of a half
// A weight is fp16(a·q − b) with a, b in f32, as dequant_elem and a rounding
// give it, bit for bit.  q arrives as a subnormal fp16: its bits alone, at
// bit P of the half, are q·2^(P−24), exact in v_fma_mix (which widens it to
// f32), and a carries the inverse power of two.
constexpr float kUp24 = 16777216.f, kUp20 = 1048576.f;  // for integers at bits 0 and 4
struct GemmWBase {
  float a_lo, c_lo, a_hi, c_hi;  // c = −b
  half2_t e, o;
  half8_t w;
  template <int S, int HI, int D>
  __device__ __forceinline__ void mix() {
    constexpr int at = 4 * (D & 1);
    const float a = HI ? a_hi : a_lo, c = HI ? c_hi : c_lo;
    w[at] = (_Float16)fmaf((float)e[0], a, c);
    w[at + 1] = (_Float16)fmaf((float)o[0], a, c);
    w[at + 2] = (_Float16)fmaf((float)e[1], a, c);
    w[at + 3] = (_Float16)fmaf((float)o[1], a, c);
  }
  // The integers of elements 0, 2 and of 1, 3.
  __device__ __forceinline__ void pair(uint32_t ev, uint32_t od) {
    e = __builtin_bit_cast(half2_t, ev);
    o = __builtin_bit_cast(half2_t, od);
  }
};

template <uint32_t FMT, int PQ>
struct GemmW;

// Q4_K and Q5_K scales: every 6-bit scale and minimum of a super-block as a byte.
struct KScales {
  uint32_t sc[4];
  float d, dmin;
  __device__ __forceinline__ void unpack(u32x4 h) {
    sc[0] = h.y & 0x3f3f3f3fu;
    sc[1] = h.z & 0x3f3f3f3fu;
    sc[2] = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
    sc[3] = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
    d = half_bits_to_float(h.x & 0xffffu);
    dmin = half_bits_to_float(h.x >> 16);
  }
  // Blocks 2S and 2S + 1, whose quants lie at bits 0 and 4.
  template <int S>
  __device__ __forceinline__ void stage(GemmWBase &g) const {
    const uint32_t s = sc[S < 2 ? 0 : 2], m = sc[S < 2 ? 1 : 3];
    g.a_lo = d * kUp24 * (S % 2 ? ubyte2(s) : ubyte0(s));
    g.c_lo = -(dmin * (S % 2 ? ubyte2(m) : ubyte0(m)));
    g.a_hi = d * kUp20 * (S % 2 ? ubyte3(s) : ubyte1(s));
    g.c_hi = -(dmin * (S % 2 ? ubyte3(m) : ubyte1(m)));
  }
};

template <int PQ>
struct GemmW<12, PQ> : GemmWBase {  // Q4_K
  u32x4 h;
  uint32_t q[4][PQ / 4];
  KScales k;
  __device__ __forceinline__ void load_header(const uint8_t *row, uint32_t sb, int) {
    h = *reinterpret_cast<const u32x4 *>(row + (uint64_t)sb * 144);
  }
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t sb, uint32_t, int c) {
    load_aligned<PQ>(row + (uint64_t)sb * 144 + 16 + 32 * S + PQ * c, q[S]);
  }
  __device__ __forceinline__ void unpack(int) { k.unpack(h); }
  template <int S>
  __device__ __forceinline__ void scales(int) {
    k.stage<S>(*this);
  }
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {
    constexpr uint32_t m = HI ? 0x00f000f0u : 0x000f000fu;
    pair(q[S][D] & m, (q[S][D] >> 8) & m);
  }
};

template <int PQ>
struct GemmW<13, PQ> : GemmWBase {  // Q5_K: the fifth bits (qh) belong to the whole super-block
  u32x4 h;
  uint32_t qh[PQ / 4], qh_next[PQ / 4], q[4][PQ / 4];
  KScales k;
  __device__ __forceinline__ void load_header(const uint8_t *row, uint32_t sb, int c) {
    const uint8_t *b = row + (uint64_t)sb * 176;
    h = *reinterpret_cast<const u32x4 *>(b);
    load_aligned<PQ>(b + 16 + PQ * c, qh_next);
  }
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t sb, uint32_t, int c) {
    load_aligned<PQ>(row + (uint64_t)sb * 176 + 48 + 32 * S + PQ * c, q[S]);
  }
  __device__ __forceinline__ void unpack(int) {
    k.unpack(h);
#pragma unroll
    for (int i = 0; i < PQ / 4; i++) qh[i] = qh_next[i];
  }
  template <int S>
  __device__ __forceinline__ void scales(int) {
    k.stage<S>(*this);
  }
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {
    constexpr int B = 2 * S + HI;  // the bit of a qh byte, to bit 4 or 8
    constexpr uint32_t m = HI ? 0x00f000f0u : 0x000f000fu, mt = HI ? 0x01000100u : 0x00100010u;
    const uint32_t v = q[S][D], t = qh[D];
    pair(and_or(shl<(HI ? 8 : 4) - B>(t), mt, v & m), and_or(shl<(HI ? 0 : -4) - B>(t), mt, (v >> 8) & m));
  }
};

template <int PQ>
struct GemmW<14, PQ> : GemmWBase {  // Q6_K: blocks of 210 bytes, at 2-byte addresses
  uint32_t sc[4], sc_next[4], d16, d16_next;
  uint32_t lo[4][PQ / 4], hi[4][PQ / 4], top[4][PQ / 4];
  __device__ __forceinline__ void load_header(const uint8_t *row, uint32_t sb, int) {
    const uint8_t *b = row + (uint64_t)sb * 210;
    load_any<16>(b + 192, sc_next);
    d16_next = load_u16(b + 208);
  }
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t sb, uint32_t, int c) {
    const uint8_t *b = row + (uint64_t)sb * 210 + PQ * c;
    load_any<PQ>(b + 64 * (S / 2), lo[S]);
    load_any<PQ>(b + 64 * (S / 2) + 32, hi[S]);
    load_any<PQ>(b + 128 + 32 * (S / 2), top[S]);
  }
  __device__ __forceinline__ void unpack(int) {
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = sc_next[i];
    d16 = d16_next;
  }
  // Stage S: quarters 2·(S%2) and 2·(S%2) + 1 of half S/2; their scales are
  // bytes 0, 1 and 2, 3 of dword S, one per 16 columns.
  template <int S>
  __device__ __forceinline__ void scales(int c) {
    const float d = half_bits_to_float(d16);
    const uint32_t s = sc[S] >> (8 * (PQ * c / 16));
    const float lo_s = d * (float)(int8_t)(s & 0xffu), hi_s = d * (float)(int8_t)((s >> 16) & 0xffu);
    constexpr float up = S % 2 ? kUp20 : kUp24;  // the nibbles stay where they lie
    a_lo = up * lo_s, c_lo = -32.f * lo_s;
    a_hi = up * hi_s, c_hi = -32.f * hi_s;
  }
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {
    constexpr int K2 = 2 * (2 * (S % 2) + HI);  // the quarter's bits in a top byte
    constexpr int P = S % 2 ? 4 : 0;
    constexpr uint32_t m = 0x000f000fu << P, mt = 0x00300030u << P;
    const uint32_t v = HI ? hi[S][D] : lo[S][D], t = top[S][D];
    pair(and_or(shl<P + 4 - K2>(t), mt, v & m), and_or(shl<P - 4 - K2>(t), mt, (v >> 8) & m));
  }
};

template <int PQ>
struct GemmW<8, PQ> : GemmWBase {  // Q8_0: two blocks of 34 bytes a stage
  uint32_t q[4][2][PQ / 4], d[4][2];
  __device__ __forceinline__ void load_header(const uint8_t *, uint32_t, int) {}
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t, uint32_t st, int c) {
    const uint8_t *b = row + (uint64_t)st * 68;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      d[S][h] = load_u16(b + 34 * h);
      load_any<PQ>(b + 34 * h + 2 + PQ * c, q[S][h]);
    }
  }
  __device__ __forceinline__ void unpack(int) {}
  template <int S>
  __device__ __forceinline__ void scales(int) {
    const float lo_s = half_bits_to_float(d[S][0]), hi_s = half_bits_to_float(d[S][1]);
    a_lo = kUp24 * lo_s, c_lo = -128.f * lo_s;  // the bytes with their sign bit flipped
    a_hi = kUp24 * hi_s, c_hi = -128.f * hi_s;
  }
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {
    const uint32_t v = q[S][HI][D] ^ 0x80808080u;
    pair(v & 0x00ff00ffu, (v >> 8) & 0x00ff00ffu);
  }
};

template <int PQ>
struct GemmW<2, PQ> : GemmWBase {  // Q4_0: two blocks of 18 bytes a stage, high nibbles the upper 16
  uint32_t q[4][2][PQ / 4], d[4][2];
  int sh;
  __device__ __forceinline__ void load_header(const uint8_t *, uint32_t, int) {}
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t, uint32_t st, int c) {
    const uint8_t *b = row + (uint64_t)st * 36;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      d[S][h] = load_u16(b + 18 * h);
      load_any<PQ>(b + 18 * h + 2 + PQ * c % 16, q[S][h]);
    }
  }
  __device__ __forceinline__ void unpack(int) {}
  template <int S>
  __device__ __forceinline__ void scales(int c) {
    sh = 4 * (PQ * c / 16);
    const float lo_s = half_bits_to_float(d[S][0]), hi_s = half_bits_to_float(d[S][1]);
    a_lo = kUp24 * lo_s, c_lo = -8.f * lo_s;
    a_hi = kUp24 * hi_s, c_hi = -8.f * hi_s;
  }
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {
    const uint32_t v = q[S][HI][D] >> sh;
    pair(v & 0x000f000fu, (v >> 8) & 0x000f000fu);
  }
};

template <int PQ>
struct GemmW<1, PQ> : GemmWBase {  // F16
  uint32_t q[4][2][PQ / 2];
  __device__ __forceinline__ void load_header(const uint8_t *, uint32_t, int) {}
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t, uint32_t st, int c) {
    const uint8_t *b = row + (uint64_t)st * 128 + 2 * PQ * c;
#pragma unroll
    for (int h = 0; h < 2; h++) load_aligned<2 * PQ>(b + 64 * h, q[S][h]);
  }
  __device__ __forceinline__ void unpack(int) {}
  template <int S>
  __device__ __forceinline__ void scales(int) {}
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {}
  template <int S, int HI, int D>
  __device__ __forceinline__ void mix() {
    constexpr int at = 4 * (D & 1);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const half2_t v = __builtin_bit_cast(half2_t, q[S][HI][2 * D + i]);
      w[at + 2 * i] = v[0], w[at + 2 * i + 1] = v[1];
    }
  }
};

template <int PQ>
struct GemmW<0, PQ> : GemmWBase {  // F32
  uint32_t q[4][2][PQ];
  __device__ __forceinline__ void load_header(const uint8_t *, uint32_t, int) {}
  template <int S>
  __device__ __forceinline__ void load(const uint8_t *row, uint32_t, uint32_t st, int c) {
    const uint8_t *b = row + (uint64_t)st * 256 + 4 * PQ * c;
#pragma unroll
    for (int h = 0; h < 2; h++) load_aligned<4 * PQ>(b + 128 * h, q[S][h]);
  }
  __device__ __forceinline__ void unpack(int) {}
  template <int S>
  __device__ __forceinline__ void scales(int) {}
  template <int S, int HI, int D>
  __device__ __forceinline__ void ints() {}
  template <int S, int HI, int D>
  __device__ __forceinline__ void mix() {
    constexpr int at = 4 * (D & 1);
#pragma unroll
    for (int i = 0; i < 4; i++) w[at + i] = (_Float16)__uint_as_float(q[S][HI][4 * D + i]);
  }
};

// Expert groups of a grouped launch (Metal::matmul_experts): the entries of
// expert e are positions offsets[e] .. offsets[e+1] of `entries`, each entry
// v = token·n_used + slot; the inputs are those of the positions in order,
// and position p writes output row entries[p].
struct ExpertGroups {
  const uint32_t *offsets, *entries;
  uint32_t n_experts;
};

// The inputs of k_split_hi (matmul.hip): fragment-major fp16 of each token
// times a power of two, and what undoes it.
struct HiInputs {
  const _Float16 *h;
  const float *unscale;
};

// Y (store) or partials: D[token][row] of the launch.  Splits > 1 (of whole
// 256-column super-blocks) write partial products to P[split]
// (k_gemm_reduce applies the store).  STORE 3 is the SwiGLU pair
// (Metal::matmul_experts's paired tile, matmul.metal:249-395): the tile's
// first half of rows are rows of W (gate projections), the other half the
// same rows of W2 (up projections), and Y receives silu(gate)·up, so the
// gate products never go through memory.
//
// STORE 0 overwrites (also the partials of split columns), 1 accumulates,
// 2 is y = silu(y)·D.
//
// GROUPED: the expert-grouped launch (matmul.metal:462-504).  W (and W2)
// stack n_experts matrices; blockIdx.x is the row tile, blockIdx.y numbers
// the token tiles of all experts one after the other (the grid is an upper
// bound); n_tokens counts the positions.  Its inputs' blocks are whole (32
// positions, the buffer rounded up).
template <uint32_t FMT, int STORE, int MB, int NB, int WR, bool GROUPED>
__global__ __launch_bounds__(256, 1) void k_gemm(const uint8_t *__restrict__ W, const uint8_t *__restrict__ W2,
                                                 uint64_t row_bytes, HiInputs X, float *__restrict__ Y,
                                                 float *__restrict__ P, uint32_t n_rows, uint32_t n_cols,
                                                 uint32_t n_tokens, uint32_t splits, ExpertGroups groups) {
  static_assert(!GROUPED || STORE == 0 || STORE == 3, "grouped launches overwrite");
  constexpr bool PAIR = STORE == 3;
  static_assert((MB == 2 || MB == 4) && MB % (PAIR ? 2 * WR : WR) == 0, "row blocks");
  constexpr int RB = 32 * MB, OR = PAIR ? RB / 2 : RB, NT = 256, WT = 4 / WR, BT = 32 * NB * WT;
  constexpr int MW = MB / WR;    // row blocks of a wave
  constexpr int TPR = NT / RB;   // threads per weight row: 2 or 4
  constexpr int PQ = 32 / TPR;   // columns per thread of each 32-column half: 16 or 8
  constexpr int CH = PQ / 8;     // 16-byte chunks of those
  __shared__ __align__(16) _Float16 A[4][RB * kGk];
  __shared__ float us_s[BT];                    // the tile's token scales
  __shared__ uint32_t ent_s[GROUPED ? BT : 1];  // grouped: the tile's entries
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, h = lane / 32;
  const int wr = wave % WR, wt = wave / WR;
  uint32_t rt, sp = 0, tok0, tok_end = n_tokens;  // tokens [tok0, tok_end) of this tile's group
  if constexpr (GROUPED) {
    // Find this tile's expert: the offsets go to LDS, one thread walks them.
    __shared__ uint32_t off_s[kMoeMaxExperts + 1];
    __shared__ uint32_t pick[3];
    for (uint32_t e = tid; e <= groups.n_experts; e += NT) off_s[e] = groups.offsets[e];
    __syncthreads();
    if (tid == 0) {
      uint32_t t = blockIdx.y, e = 0;
      for (; e < groups.n_experts; e++) {
        const uint32_t tiles = (off_s[e + 1] - off_s[e] + BT - 1) / BT;
        if (t < tiles) break;
        t -= tiles;
      }
      pick[0] = e;
      pick[1] = e < groups.n_experts ? off_s[e] + t * BT : 0;
      pick[2] = e < groups.n_experts ? off_s[e + 1] : 0;
    }
    __syncthreads();
    if (pick[0] >= groups.n_experts) return;  // past the last tile (uniform)
    W += (uint64_t)pick[0] * n_rows * row_bytes;
    if (PAIR) W2 += (uint64_t)pick[0] * n_rows * row_bytes;
    tok0 = __builtin_amdgcn_readfirstlane(pick[1]);
    tok_end = __builtin_amdgcn_readfirstlane(pick[2]);
    rt = blockIdx.x;
    if (tid < BT) ent_s[tid] = groups.entries[min(tok0 + tid, tok_end - 1)];
  } else {
    const uint32_t n_rt = (n_rows + OR - 1) / OR, n_tt = (n_tokens + BT - 1) / BT;
    const uint32_t total = n_rt * n_tt * splits;
    // XCD-aware order: workgroup L runs on XCD L % 8, so logical tile
    // (L % 8)·⌈total/8⌉ + L/8 hands each XCD a contiguous run, split-major
    // then token-tile-major: the row tiles sharing a token tile's inputs
    // share that XCD's L2.
    const uint32_t per = (total + 7) / 8, logical = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (logical >= total) return;
    rt = logical % n_rt;
    sp = logical / (n_rt * n_tt);
    tok0 = ((logical / n_rt) % n_tt) * BT;
  }
  const uint32_t row0 = rt * OR;
  const uint32_t x_cols = (n_cols + 7) / 8 * 8;  // of the fragment blocks
  const uint32_t n_stages = n_cols / kGk, n_sb = (n_stages + 3) / 4;
  const uint32_t sb0 = sp * n_sb / splits, sb1 = (sp + 1) * n_sb / splits;  // never empty: splits <= n_sb

  // Converting role: weight row ar, part ac.  (Rows past the end are
  // clamped; their outputs are never stored.)
  const int ar = tid / TPR, ac = tid % TPR;
  const uint8_t *wrow = PAIR && ar >= OR ? W2 + (uint64_t)min(row0 + ar - OR, n_rows - 1) * row_bytes
                                         : W + (uint64_t)min(row0 + ar, n_rows - 1) * row_bytes;
  // MFMA role: token blocks NB·wt + j of the tile, read through a descriptor
  // of the lane's block(s).  TAIL: formats whose rows need not be whole
  // super-blocks; the descriptor ends with the columns, and the stages past
  // them read zeros (load_x).
  constexpr bool TAIL = !GROUPED && (FMT == BCH_F32 || FMT == BCH_F16 || FMT == BCH_Q8_0 || FMT == BCH_Q4_0);
  __amdgpu_buffer_rsrc_t xr[NB];
  uint32_t xv[NB], xs[NB];
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const uint32_t p0 = tok0 + 32 * (NB * wt + j);
    if constexpr (GROUPED) {
      // Positions need not start a block: the lanes span two.
      const uint32_t b0 = __builtin_amdgcn_readfirstlane(min(p0, tok_end - 1) / 32);
      const uint32_t p = min(p0 + lane % 32, tok_end - 1);
      xr[j] = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(X.h) + (uint64_t)b0 * 32 * x_cols, 0,
                                                128 * x_cols, 0x00020000);
      xv[j] = (p / 32 - b0) * 64 * x_cols + (32 * h + p % 32) * 16;
      xs[j] = 1024;
    } else {
      const uint32_t b = __builtin_amdgcn_readfirstlane(min(p0, n_tokens - 1) / 32);
      const uint32_t R = min(32u, n_tokens - 32 * b);
      xr[j] = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(X.h) + (uint64_t)b * 32 * x_cols, 0,
                                                R * n_stages * (2 * kGk), 0x00020000);
      xv[j] = (h * R + min((uint32_t)lane % 32, R - 1)) * 16;
      xs[j] = 32 * R;
    }
  }
  if (tid < BT) us_s[tid] = X.unscale[min(tok0 + tid, tok_end - 1)];
  typedef GemmW<FMT, PQ> GW;
  GW w;
  // LDS: the weights of columns 16s + 8hh .. of row r are 16 bytes at slot
  // (s·MB + r/32)·64 + (r%32 + 32·hh), so a wave's fragment read is 1 KB of
  // consecutive bytes; the slots are swizzled so that the two or four
  // threads of a row write to different banks.
  auto swz = [](int s, int hh) { return 4 * (s & 1) + 2 * hh; };
  auto put = [&](int half, int p, _Float16 *buf, half8_t v) __attribute__((always_inline)) {
    const int j = 4 * half + CH * ac + p, s = j / 2, hh = j % 2;
    *reinterpret_cast<half8_t *>(buf + ((s * MB + ar / 32) * 64 + ((ar % 32 + 32 * hh) ^ swz(s, hh))) * 8) = v;
  };
  // The conversion of a stage in small operations that can sit between
  // MFMAs: the scales, then two per four weights.
  constexpr int UNITS = 2 * (PQ / 4), OPS = 1 + 2 * UNITS;
  auto dq_op = [&](auto idx, auto stage, _Float16 *buf) __attribute__((always_inline)) {
    constexpr int U = decltype(idx)::value, S = decltype(stage)::value;
    if constexpr (U == 0) {
      if constexpr (S == 0) w.unpack(ac);
      w.template scales<S>(ac);
    } else {
      constexpr int V = (U - 1) / 2, HI = V / (PQ / 4), D = V % (PQ / 4);
      if constexpr (U % 2 == 1) {
        w.template ints<S, HI, D>();
      } else {
        w.template mix<S, HI, D>();
        if constexpr (D % 2 == 1) put(HI, D / 2, buf, w.w);
      }
    }
  };
  const int rd0 = lane ^ swz(0, h), rd1 = lane ^ swz(1, h);
  // (The wave's row block i is block wr + WR·i of the tile, so a wave holds
  // the gate and the up block of the same rows.)
  auto frag = [&](const _Float16 *buf, int s, int i) __attribute__((always_inline)) {
    return *reinterpret_cast<const half8_t *>(buf + ((s * MB + wr + WR * i) * 64 + ((s & 1) ? rd1 : rd0)) * 8);
  };

  float16_t acc[MW][NB];
#pragma unroll
  for (int i = 0; i < MW; i++)
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;

  // Pipeline: stage t (64 columns) runs its MFMAs from LDS buffer t % 4 while
  // the weights of stage t + 2 are converted into buffer (t + 2) % 4; then
  // the raw weights of stage t + 6 are requested, and as each k-step's inputs
  // are spent, those of stage t + 2.  One barrier a stage.  Requests past the
  // end re-read the last stage (the inputs) or super-block; nothing uses them.
  u32x4 x[2][4][NB];
  half8_t wf[2][MW];
  const uint32_t last_stage = 4 * sb1 - 1, last_sb = sb1 - 1;
  auto load_x = [&](uint32_t stage, int slot, auto sj) __attribute__((always_inline)) {
    constexpr int s = decltype(sj)::value / NB, j = decltype(sj)::value % NB;
    const uint32_t step = (4 * stage + s) * xs[j];
    if constexpr (TAIL)  // (only the vector offset is sure to be checked against the descriptor's size)
      x[slot][s][j] = __builtin_amdgcn_raw_buffer_load_b128(xr[j], xv[j] + step, 0, 0);
    else  // always inside the columns
      x[slot][s][j] = __builtin_amdgcn_raw_buffer_load_b128(xr[j], xv[j], step, 0);
  };
  auto load_w = [&](auto stage, uint32_t sb) __attribute__((always_inline)) {
    constexpr int S = decltype(stage)::value;
    w.template load<S>(wrow, sb, min(4 * sb + S, n_stages - 1), ac);
  };
  w.load_header(wrow, sb0, ac);
  static_for<4>([&](auto S) __attribute__((always_inline)) { load_w(S, sb0); });
  __builtin_amdgcn_sched_barrier(0);
  static_for<4 * NB>([&](auto sj) __attribute__((always_inline)) { load_x(4 * sb0, 0, sj); });
  __builtin_amdgcn_sched_barrier(0);
  static_for<4 * NB>([&](auto sj) __attribute__((always_inline)) { load_x(4 * sb0 + 1, 1, sj); });
  __builtin_amdgcn_sched_barrier(0);
  static_for<2>([&](auto S) __attribute__((always_inline)) {
    static_for<OPS>([&](auto i) __attribute__((always_inline)) { dq_op(i, S, A[decltype(S)::value]); });
  });
  w.load_header(wrow, min(sb0 + 1, last_sb), ac);
  static_for<2>([&](auto S) __attribute__((always_inline)) { load_w(S, min(sb0 + 1, last_sb)); });
  lds_barrier();
#pragma unroll
  for (int i = 0; i < MW; i++) wf[0][i] = frag(A[0], 0, i);

  auto run = [&](auto mine) __attribute__((always_inline)) {
    constexpr bool LIVE = decltype(mine)::value;
    uint32_t sb = sb0;
    do {
      static_for<4>([&](auto stage) __attribute__((always_inline)) {
        constexpr int S = decltype(stage)::value, SD = (S + 2) % 4;  // SD: the stage being converted
        constexpr int MF = 4 * MW * NB;                              // MFMAs
        const uint32_t sx = min(4 * sb + S + 2, last_stage);
        static_for<MF>([&](auto mi) __attribute__((always_inline)) {
          constexpr int m = decltype(mi)::value, s = m / (MW * NB), i = (m / NB) % MW, j = m % NB;
          if constexpr (LIVE) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, x[S % 2][s][j]),
                                                               wf[s & 1][i], acc[i][j], 0, 0, 0);
            if constexpr (j == 0) wf[(s + 1) & 1][i] = s < 3 ? frag(A[S], s + 1, i) : frag(A[(S + 1) % 4], 0, i);
            if constexpr (i == MW - 1) load_x(sx, S % 2, std::integral_constant<int, s * NB + j>{});
          }
          static_for<OPS>([&](auto oi) __attribute__((always_inline)) {
            if constexpr (decltype(oi)::value * (MF - 2) / OPS == m) dq_op(oi, std::integral_constant<int, SD>{}, A[SD]);
          });
          if constexpr (m == MF - 1) {
            if constexpr (SD == 0) w.load_header(wrow, min(sb + 2, last_sb), ac);
            load_w(std::integral_constant<int, SD>{}, min(sb + (S < 2 ? 1 : 2), last_sb));
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        lds_barrier();
      });
    } while (++sb < sb1);
  };
  // Grouped: a wave whose tokens all lie past its expert's entries only
  // converts its share of the weights (in a loop of its own, with the same
  // barriers: a branch at every MFMA broke up the order above).
  if (!GROUPED || __builtin_amdgcn_readfirstlane(tok0 + 32 * NB * wt < tok_end ? 1 : 0) != 0)
    run(std::true_type{});
  else
    run(std::false_type{});

  // acc[i][j][e]: token 32·(NB·wt + j) + 8(e/4) + 4h + e%4 of the tile, row
  // 32·(wr + WR·i) + lane%32.  The epilogue's loads (prior outputs, with
  // clamped addresses) are unconditional so that they issue together; only
  // the stores test bounds.
  constexpr int OW = PAIR ? MW / 2 : MW;
  float *dst = splits > 1 ? P + (uint64_t)sp * n_tokens * n_rows : Y;
  // (Opaque here, so that the epilogue's addresses are not computed before
  // the loop and carried through it: that took 40 registers and a third of
  // the loop's speed.)
  uint32_t rows = n_rows, trow0 = row0, ttok0 = tok0;
  asm volatile("" : "+s"(rows), "+s"(trow0), "+s"(ttok0));
#pragma unroll
  for (int i = 0; i < OW; i++) {
    const uint32_t row = trow0 + 32 * (wr + WR * i) + lane % 32;
    const uint32_t rowc = min(row, rows - 1);
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int tw = 32 * (NB * wt + j);  // first token of the block in the tile
      const uint32_t tb = ttok0 + tw;
      float v[16], prior[16];
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int tl = tw + 8 * (e / 4) + 4 * h + e % 4;
        v[e] = acc[i][j][e] * us_s[tl];
        if constexpr (PAIR)
          prior[e] = acc[(i + OW) % MW][j][e] * us_s[tl];  // the up product
        else if constexpr (STORE != 0)
          prior[e] = Y[(uint64_t)min(ttok0 + tl, n_tokens - 1) * rows + rowc];
      }
      // Output row of tile token tl: the token itself, or (grouped) its entry.
      auto y_row = [&](int tl) -> uint64_t {
        if constexpr (GROUPED)
          return ent_s[tl];
        else
          return ttok0 + tl;
      };
#pragma unroll
      for (int e = 0; e < 16; e++) {
        if constexpr (PAIR)
          v[e] = silu_f(v[e]) * prior[e];
        else if constexpr (STORE == 1)
          v[e] += prior[e];
        else if constexpr (STORE == 2)
          v[e] *= silu_f(prior[e]);
      }
      if (row >= rows) continue;
      if (tb + 32 <= tok_end) {
#pragma unroll
        for (int e = 0; e < 16; e++) dst[y_row(tw + 8 * (e / 4) + 4 * h + e % 4) * rows + row] = v[e];
      } else {
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int tl = tw + 8 * (e / 4) + 4 * h + e % 4;
          if (ttok0 + tl < tok_end) dst[y_row(tl) * rows + row] = v[e];
        }
      }
    }
  }
}

}  // namespace bch
