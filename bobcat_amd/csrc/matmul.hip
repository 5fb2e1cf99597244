// Prefill GEMM: Y[t] (store) W·X[t] for a batch of tokens, on MFMA.
//
// Counterpart of Metal::matmul, Metal::matmul_experts and Metal::expand +
// matmul_f16 (crates/bobcat-metal/src/backend.rs:2470-2549,
// matmul.metal:249-504, quant.metal:276-306).  The reference expands Q4_K
// matrices to fp16 before a full 512-token batch; here each workgroup
// dequantises its weight tile straight into LDS instead, so the expanded
// matrix never touches HBM.  One kernel, k_gemm (gemm_tile.h), serves dense
// and expert-grouped launches; accumulation is fp32.
//
// The inputs are rounded to fp16 once per batch by the kernels here: each
// token scaled by the power of two that puts its largest magnitude in
// [2^13, 2^14) (half precision cannot overflow) — 11 significant bits, finer
// than bf16 — the scale undone in the epilogue, in the fragment-major layout
// the tile's loads want.
//
// Split K.  With few tiles (outputs of a 2048-wide residual stream) the
// column range is split over up to kMaxSplitK workgroups; each writes its
// partial product to scratch and k_gemm_reduce adds them in a fixed order
// and applies the store, so the result does not depend on timing.
#include <mutex>
#include "gemm_tile.h"
#include "runtime.h"

namespace bch {

constexpr int kBK = 256;      // columns a row must be a multiple of (one Q4_K super-block)
constexpr uint32_t kMaxSplitK = 8;

// Bytes of the fp16 inputs of `rows` rows, and where their scales follow.
static uint64_t frag_halves(uint32_t rows, uint32_t n_cols) { return (uint64_t)rows * ((n_cols + 7) / 8 * 8); }

// Eight consecutive floats, and their part of a row's maximum and fp16 form.
struct Eight {
  float4 a, b;
  __device__ __forceinline__ float amax() const {
    return fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                 fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w))));
  }
  __device__ __forceinline__ half8_t half(float s) const {
    half8_t o;
    o[0] = (_Float16)(a.x * s), o[1] = (_Float16)(a.y * s), o[2] = (_Float16)(a.z * s), o[3] = (_Float16)(a.w * s);
    o[4] = (_Float16)(b.x * s), o[5] = (_Float16)(b.y * s), o[6] = (_Float16)(b.z * s), o[7] = (_Float16)(b.w * s);
    return o;
  }
};

// A row's fp16 fragments from its values value(i) (floats 8i .. 8i+7, of n8
// eights), times the power of two that puts the largest in [2^13, 2^14); the
// scale's inverse goes to *unscale.  256 threads; PER > 0: each keeps its PER
// eights (i = tid + 256·k) in registers, PER = 0: value() is called twice.
// also(i, v) sees every eight once.
template <int PER, class Value, class Also>
__device__ __forceinline__ void split_row(uint32_t n8, FragRow row, float *unscale, Value value, Also also) {
  const uint32_t tid = threadIdx.x;
  Eight v[PER > 0 ? PER : 1];
  float mx = 0.f;
  if constexpr (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; k++) v[k] = value(min(tid + 256 * k, n8 - 1));
#pragma unroll
    for (int k = 0; k < PER; k++) mx = fmaxf(mx, v[k].amax());
  } else {
    for (uint32_t i = tid; i < n8; i += 256) mx = fmaxf(mx, value(i).amax());
  }
  __shared__ float red[4];
  mx = block_max<256>(mx, red);
  int ex = 0;
  if (mx > 0.f) frexpf(mx, &ex);  // mx < 2^ex
  const int k2 = max(-100, min(100, 14 - ex));
  const float scale = ldexpf(1.0f, k2);
  if (tid == 0) *unscale = ldexpf(1.0f, -k2);
  auto put = [&](uint32_t i, const Eight &e) {
    *reinterpret_cast<half8_t *>(row.base + (uint64_t)i * row.stride) = e.half(scale);
    also(i, e);
  };
  if constexpr (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; k++)
      if (tid + 256 * k < n8) put(tid + 256 * k, v[k]);
  } else {
    for (uint32_t i = tid; i < n8; i += 256) put(i, value(i));
  }
}

// Row t of X to fp16 fragments (split_row), one workgroup per row.  With
// `entries`, row p of H is row entries[p] / x_div of X, at most last_row
// (the positions of an expert-grouped launch).  Bound by the reads and the
// scattered 16-byte writes: 512 x 10752 in 8.9 us (~6 when the inputs were
// plain rows; the GEMM's loads gain more than that).
template <int PER>
__global__ __launch_bounds__(256) void k_split_hi(const float *__restrict__ X, uint32_t n_cols, uint32_t frag_rows,
                                                 const uint32_t *__restrict__ entries, uint32_t x_div, uint32_t last_row,
                                                 _Float16 *__restrict__ H, float *__restrict__ unscale) {
  const uint32_t t = frag_row_of(blockIdx.x, gridDim.x);
  const uint32_t src = entries ? min(entries[t] / x_div, last_row) : t;
  const float4 *x4 = reinterpret_cast<const float4 *>(X + (uint64_t)src * n_cols);
  const uint32_t n8 = (n_cols + 7) / 8, n4 = n_cols / 4;
  split_row<PER>(n8, FragRow::of(H, t, frag_rows, 8 * n8), unscale + t, [&](uint32_t i) {
    return Eight{x4[2 * i], 2 * i + 1 < n4 ? x4[2 * i + 1] : float4{0.f, 0.f, 0.f, 0.f}};
  }, [](uint32_t, const Eight &) {});
}

// k_split_hi of `rows` rows (their blocks laid out for frag_rows), choosing
// the register form by row length.
static void split_hi(hipStream_t s, const float *x, uint32_t rows, uint32_t frag_rows, uint32_t n_cols, _Float16 *h,
                     float *unscale, const uint32_t *entries = nullptr, uint32_t x_div = 1, uint32_t last_row = 0) {
  if (!rows) return;
  auto go = [&](auto per) {
    k_split_hi<decltype(per)::value><<<rows, 256, 0, s>>>(x, n_cols, frag_rows, entries, x_div, last_row, h, unscale);
  };
  const uint32_t per = div_ceil(div_ceil(n_cols, 8), 256);
  if (per <= 1)
    go(std::integral_constant<int, 1>{});
  else if (per <= 2)
    go(std::integral_constant<int, 2>{});
  else if (per <= 6)
    go(std::integral_constant<int, 6>{});
  else
    go(std::integral_constant<int, 0>{});
}

// k_rms_norm (ops.hip) and k_split_hi in one pass over each row: `out`
// receives exactly k_rms_norm's values (same per-thread sums, reduction and
// scale), and H/unscale the fp16 form of those values that k_split_hi would
// make, so the GEMM that follows skips its own conversion.
//
// PER > 0: each thread keeps its PER elements (i = tid + 256·k, the order
// of k_rms_norm's sums) in registers, so the row is read once; PER = 0
// loops over rows of any length, re-reading.
//
// SUM: x first receives the column-split partial products of the GEMM
// that accumulated into it (P[split][row][i], added in split order and then
// to x, exactly as k_gemm_reduce<1> would), and the sums are written back.
//
// rows_h: H gets plain rows (for the library GEMM) instead of fragments.
// H null: the norm alone.
template <int PER, int SPLITS>
__global__ __launch_bounds__(256) void k_rms_norm_split(float *__restrict__ x, const float *__restrict__ w,
                                                       float *__restrict__ out, uint32_t n, float eps,
                                                       _Float16 *__restrict__ H, float *__restrict__ unscale,
                                                       const float *__restrict__ P, uint32_t splits,
                                                       float *__restrict__ unscale_copy, bool rows_h) {
  constexpr bool SUM = SPLITS > 0;
  __shared__ float red[4];
  const uint32_t t = frag_row_of(blockIdx.x, gridDim.x), tid = threadIdx.x;
  float *xr = x + (uint64_t)t * n;
  float *orow = out + (uint64_t)t * n;
  FragRow hrow = FragRow::of(H, t, gridDim.x, (n + 7) / 8 * 8);
  if (rows_h) hrow = FragRow{H + (uint64_t)t * n, 8};
  const uint64_t pstride = (uint64_t)gridDim.x * n;
  const float *prow = P + (uint64_t)t * n;
  auto pending = [&](uint32_t i) {
    float v = prow[i];
    for (uint32_t sp = 1; sp < splits; sp++) v += prow[sp * pstride + i];
    return v;
  };
  // The partials of element i, all loaded before any is added (SPLITS > 0).
  auto partials = [&](uint32_t i, float *pv) __attribute__((always_inline)) {
#pragma unroll
    for (int sp = 0; sp < (SUM ? SPLITS : 1); sp++) pv[sp] = prow[sp * pstride + i];
  };
  float xv[PER > 0 ? PER : 1], wv[PER > 0 ? PER : 1];
  float ss = 0.f;
  if constexpr (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const uint32_t i = tid + 256 * k;
      xv[k] = i < n ? xr[i] : 0.f;
      wv[k] = i < n ? w[i] : 0.f;
    }
    if constexpr (SUM) {
      float pv[PER][SUM ? SPLITS : 1];
#pragma unroll
      for (int k = 0; k < PER; k++) partials(min(tid + 256 * k, n - 1), pv[k]);
#pragma unroll
      for (int k = 0; k < PER; k++) {
        const uint32_t i = tid + 256 * k;
        float v = pv[k][0];
#pragma unroll
        for (int sp = 1; sp < SPLITS; sp++) v += pv[k][sp];
        if (i < n) {
          xv[k] += v;
          xr[i] = xv[k];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < PER; k++)
      if (tid + 256 * k < n) ss = fmaf(xv[k], xv[k], ss);
  } else {
    if constexpr (SUM)
      for (uint32_t i = tid; i < n; i += 256) xr[i] += pending(i);  // each thread re-reads only its own elements
    for (uint32_t i = tid; i < n; i += 256) ss = fmaf(xr[i], xr[i], ss);
  }
  ss = block_sum<256>(ss, red);
  const float scale = (float)(1.0 / sqrt((double)ss / (double)n + (double)eps));
  float mx = 0.f;
  if constexpr (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const uint32_t i = tid + 256 * k;
      xv[k] = wv[k] * (xv[k] * scale);
      if (i < n) {
        orow[i] = xv[k];
        mx = fmaxf(mx, fabsf(xv[k]));
      }
    }
  } else {
    for (uint32_t i = tid; i < n; i += 256) {
      const float v = w[i] * (xr[i] * scale);
      orow[i] = v;
      mx = fmaxf(mx, fabsf(v));
    }
  }
  if (!H) return;
  mx = block_max<256>(mx, red);
  int ex = 0;
  if (mx > 0.f) frexpf(mx, &ex);  // mx < 2^ex
  const int k2 = max(-100, min(100, 14 - ex));
  const float s2 = ldexpf(1.0f, k2);
  if (tid == 0) {
    unscale[t] = ldexpf(1.0f, -k2);
    if (unscale_copy) unscale_copy[t] = ldexpf(1.0f, -k2);
  }
  if constexpr (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; k++)
      if (tid + 256 * k < n) *hrow.at(tid + 256 * k) = (_Float16)(xv[k] * s2);
  } else {
    for (uint32_t i = tid; i < n; i += 256) *hrow.at(i) = (_Float16)(orow[i] * s2);
  }
}

template <int STORE>
__global__ __launch_bounds__(256) void k_gemm_reduce(const float *__restrict__ P, uint32_t splits, uint64_t n,
                                                     float *__restrict__ Y);

void finish_pending_sum(hipStream_t s, PendingSum &p, float *y) {
  if (p.splits > 1) {
    const dim3 g((uint32_t)((p.n + 255) / 256));
    k_gemm_reduce<1><<<g, 256, 0, s>>>(p.part, p.splits, p.n, y);
  }
  p = PendingSum{};
}

void run_rms_norm_split(hipStream_t s, float *x, const float *w, float *out, uint32_t n, uint32_t rows, float eps,
                        void *scratch, PendingSum *pending, float *unscale_copy) {
  if (!rows) return;
  _Float16 *hx = static_cast<_Float16 *>(scratch);
  float *unscale = hx ? reinterpret_cast<float *>(hx + frag_halves(rows, n)) : nullptr;
  const bool rows_h = unscale_copy != nullptr;
  bool sum = pending && pending->splits > 1;
  const uint32_t ps = sum ? pending->splits : 0;
  if (sum && (pending->n != (uint64_t)rows * n || (ps != 2 && ps != 4 && ps != 8) ||
              (hx && reinterpret_cast<const uint8_t *>(pending->part) < reinterpret_cast<uint8_t *>(unscale + rows)))) {
    // Not this norm's rows, or the fp16 inputs written here would cover the
    // partials: add them first.
    finish_pending_sum(s, *pending, x);
    sum = false;
  }
  const float *P = sum ? pending->part : nullptr;
  const uint32_t splits = sum ? pending->splits : 0;
  auto go = [&](auto per) {
    constexpr int PER = decltype(per)::value;
    if (!sum)
      k_rms_norm_split<PER, 0><<<rows, 256, 0, s>>>(x, w, out, n, eps, hx, unscale, P, splits, unscale_copy, rows_h);
    else if (splits == 2)
      k_rms_norm_split<PER, 2><<<rows, 256, 0, s>>>(x, w, out, n, eps, hx, unscale, P, splits, unscale_copy, rows_h);
    else if (splits == 4)
      k_rms_norm_split<PER, 4><<<rows, 256, 0, s>>>(x, w, out, n, eps, hx, unscale, P, splits, unscale_copy, rows_h);
    else
      k_rms_norm_split<PER, 8><<<rows, 256, 0, s>>>(x, w, out, n, eps, hx, unscale, P, splits, unscale_copy, rows_h);
  };
  if (n <= 1024)
    go(std::integral_constant<int, 4>{});
  else if (n <= 2048)
    go(std::integral_constant<int, 8>{});
  else if (n <= 4096)
    go(std::integral_constant<int, 16>{});
  else
    go(std::integral_constant<int, 0>{});
  if (pending) *pending = PendingSum{};
}

// Y (store) Σ_split P[split], the splits added in order.
template <int STORE>
__global__ __launch_bounds__(256) void k_gemm_reduce(const float *__restrict__ P, uint32_t splits, uint64_t n,
                                                     float *__restrict__ Y) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v = P[i];
  for (uint32_t sp = 1; sp < splits; sp++) v += P[sp * n + i];
  if (STORE == 0)
    Y[i] = v;
  else if (STORE == 1)
    Y[i] += v;
  else
    Y[i] = silu_f(Y[i]) * v;
}

// Tile and column split of a launch: the choice with the least estimated
// time among the tiles a format has — rounds of workgroups over the CUs
// times the tile's time per 64-column stage, measured on MI355X at 512 tokens
// (64 x 128: 0.36 us, 64 x 256: 0.47, 128 x 256: 0.85 with most CUs busy,
// plus 4 us to start and store), plus the partials' way through memory
// (written and read at ~4.5 TB/s) and a launch to add them (half of its 2 us,
// whether or not the next norm does it: the choice is the same for both, so
// that both give the same bits).  What the choices give at 512 tokens, a
// call with its input conversion and the sum of its splits, in us:
//   6144 x 2048    64 x 256 (192 tiles, one round) 25; 64 x 128 26.6, 128 x 256 (96 CUs) 33
//   10752 x 2048   128 x 256 37-38.5; 64 x 256 (two rounds) 38.5, 64 x 128 38.9
//   3072 x 2048    64 x 128 18.3; 64 x 256 21, 128 x 256 31
//   2048 x 10752   64 x 256 in four splits 43; 128 x 256 in eight 45.6 or four
//                  50, 64 x 256 in eight 47, two 50 or unsplit (64 CUs) 77
//   2048 x 2048    64 x 128 in two splits 19.6 (the driver's norms add them
//                  on the way); unsplit 17.0, in four 25
struct GemmShape {
  uint32_t mb, nb, splits;  // 32·mb rows x 128·nb tokens
};

// The most splits a shape may take: what its no-allocation scratch has always
// been sized for (bch_matmul_noalloc refuses what needs more).
static uint32_t gemm_max_splits(uint32_t n_rows, uint32_t n_cols, uint32_t n_tokens, uint64_t part_floats, uint32_t cus) {
  auto tiles = [&](uint32_t br, uint32_t bt) { return (uint64_t)div_ceil(n_rows, br) * div_ceil(n_tokens, bt); };
  const uint64_t enough = (uint64_t)cus * 3 / 5;
  const uint32_t n_stages = n_cols / kGk;
  auto fits = [&](uint32_t splits) {
    return splits <= kMaxSplitK && n_stages / splits >= 8 && (uint64_t)splits * n_tokens * n_rows <= part_floats;
  };
  const bool wide = n_tokens > 128 && n_rows > 64;
  uint32_t splits = 1;
  if (wide && tiles(128, 256) >= enough) return 1;
  if (wide && n_cols >= 8192) {
    while (tiles(128, 256) * splits < cus && fits(2 * splits)) splits *= 2;
    return splits;
  }
  if (n_rows > 64 && tiles(128, 128) >= enough) return 1;
  while (tiles(64, 128) * splits * 2 <= cus && fits(2 * splits)) splits *= 2;
  return splits;
}

static GemmShape gemm_shape(uint32_t format, uint32_t n_rows, uint32_t n_cols, uint32_t n_tokens, uint64_t part_floats,
                            uint32_t cus, bool pair) {
  struct Tile {
    uint32_t mb, nb;
    float stage_us;
  };
  // (The 128-row tile is Q4_K's only; a pair's rows are half gate, half up.)
  const Tile tiles[] = {{2, 1, 0.36f}, {2, 2, 0.47f}, {4, 2, 0.85f}};
  const uint32_t n_sb = (n_cols / kGk + 3) / 4;
  const uint32_t most = pair ? 1u : gemm_max_splits(n_rows, n_cols, n_tokens, part_floats, cus);
  GemmShape best{2, 1, 1};
  float best_us = 1e30f;
  for (const Tile &t : tiles) {
    if (t.mb == 4 && format != BCH_Q4K) continue;
    const uint64_t wgs = (uint64_t)div_ceil(n_rows, (pair ? 16 : 32) * t.mb) * div_ceil(n_tokens, 128 * t.nb);
    for (uint32_t sp = 1; sp <= most && sp <= n_sb; sp *= 2) {
      const uint64_t rounds = (wgs * sp + cus - 1) / cus;
      float us = rounds * (4.f * ((n_sb + sp - 1) / sp) * t.stage_us + 4.f);
      if (sp > 1) us += 1.f + 8e-6f / 4.5f * sp * n_tokens * n_rows;
      if (us < best_us) best_us = us, best = GemmShape{t.mb, t.nb, sp};
    }
  }
  return best;
}

template <uint32_t FMT>
static void gemm_fmt(hipStream_t s, const uint8_t *W, const uint8_t *W2, uint64_t rb, const HiInputs &x, float *y,
                     float *part, uint64_t part_floats, uint32_t n_rows, uint32_t n_cols, uint32_t n_tokens,
                     uint32_t store, uint32_t cus, PendingSum *defer) {
  const GemmShape g = gemm_shape(FMT, n_rows, n_cols, n_tokens, part_floats, cus, store == 3);
  auto go = [&](auto how, auto mb, auto nb) {
    constexpr int STORE = decltype(how)::value, MB = decltype(mb)::value, NB = decltype(nb)::value;
    const uint32_t total = div_ceil(n_rows, (STORE == 3 ? 16 : 32) * MB) * div_ceil(n_tokens, 128 * NB) * g.splits;
    k_gemm<FMT, STORE, MB, NB, 1, false><<<8 * div_ceil(total, 8), 256, 0, s>>>(
        W, W2, rb, x, y, part, n_rows, n_cols, n_tokens, g.splits, ExpertGroups{});
  };
  auto tile = [&](auto how) {
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> two{};
    if constexpr (FMT == BCH_Q4K) {
      if (g.mb == 4) return go(how, std::integral_constant<int, 4>{}, two);
    }
    if (g.nb == 2)
      go(how, two, two);
    else
      go(how, two, one);
  };
  if (store == 3)
    tile(std::integral_constant<int, 3>{});
  else if (g.splits > 1 || store == 0)
    tile(std::integral_constant<int, 0>{});
  else if (store == 1)
    tile(std::integral_constant<int, 1>{});
  else
    tile(std::integral_constant<int, 2>{});
  if (g.splits <= 1) return;
  const uint64_t n = (uint64_t)n_tokens * n_rows;
  if (store == 1 && defer) {
    // The next kernel (k_rms_norm_split) adds the partials.
    *defer = PendingSum{part, g.splits, n};
    return;
  }
  const dim3 grid((uint32_t)((n + 255) / 256));
  if (store == 0)
    k_gemm_reduce<0><<<grid, 256, 0, s>>>(part, g.splits, n, y);
  else if (store == 1)
    k_gemm_reduce<1><<<grid, 256, 0, s>>>(part, g.splits, n, y);
  else
    k_gemm_reduce<2><<<grid, 256, 0, s>>>(part, g.splits, n, y);
}

// The fp16 inputs (2 bytes a column) and one f32 unscale per row of inputs.
uint64_t matmul_split_bytes(uint32_t n_rows, uint32_t n_cols) {
  return 2 * frag_halves(n_rows, n_cols) + 4ull * n_rows;
}
uint64_t matmul_expert_bytes(uint32_t positions, uint32_t n_cols) {
  return 2 * frag_halves((positions + 31) / 32 * 32, n_cols) + 4ull * positions;
}

uint64_t matmul_scratch_bytes(uint32_t n_tokens, uint32_t n_cols, uint32_t n_rows) {
  return (matmul_split_bytes(n_tokens, n_cols) + 255) / 256 * 256 + 4ull * kMaxSplitK * n_tokens * n_rows;
}

static uint32_t device_cus() {
  static uint32_t cus = 0;
  if (!cus) {
    int dev = 0;
    hipDeviceProp_t prop;
    cus = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
              ? (uint32_t)prop.multiProcessorCount
              : 256u;
  }
  return cus;
}

void run_matmul(hipStream_t s, uint32_t format, const uint8_t *W, uint32_t n_rows, uint32_t n_cols, const float *xf,
                float *y, uint32_t n_tokens, uint32_t store, void *scratch, uint64_t scratch_bytes, bool split_ready,
                const uint8_t *W2, PendingSum *defer) {
  if (defer) *defer = PendingSum{};
  if (!n_tokens) return;
  const uint64_t rb = bch_row_bytes(format, n_cols);
  // The fp16 inputs and their scales (n_tokens·(2·n_cols + 4) bytes, within
  // matmul_split_bytes), then the split-K partials.  With split_ready the
  // previous launch on this scratch converted the same inputs.
  _Float16 *hx = static_cast<_Float16 *>(scratch);
  float *unscale = reinterpret_cast<float *>(hx + frag_halves(n_tokens, n_cols));
  if (!split_ready) split_hi(s, xf, n_tokens, n_tokens, n_cols, hx, unscale);
  const HiInputs x{hx, unscale};
  const uint64_t used = (matmul_split_bytes(n_tokens, n_cols) + 255) / 256 * 256;
  float *part = reinterpret_cast<float *>(static_cast<uint8_t *>(scratch) + used);
  const uint64_t part_floats = scratch_bytes > used ? (scratch_bytes - used) / 4 : 0;
  const uint32_t cus = device_cus();
  switch (format) {
    case 12: gemm_fmt<12>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
    case 1: gemm_fmt<1>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
    case 14: gemm_fmt<14>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
    case 13: gemm_fmt<13>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
    case 8: gemm_fmt<8>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
    case 2: gemm_fmt<2>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
    default: gemm_fmt<0>(s, W, W2, rb, x, y, part, part_floats, n_rows, n_cols, n_tokens, store, cus, defer); break;
  }
}

static bool matmul_format(uint32_t f) {
  return f == 12 || f == 1 || f == 0 || f == 13 || f == 14 || f == 8 || f == 2;
}

void run_matmul_experts(hipStream_t s, uint32_t format, const uint8_t *W, const uint8_t *up, uint32_t n_rows,
                        uint32_t n_cols, uint32_t n_experts, const float *xf, bool shared_input,
                        const uint32_t *offsets, const uint32_t *entries, uint32_t n_used, float *y,
                        uint32_t n_tokens, void *split) {
  if (!n_tokens) return;
  const uint64_t rb = bch_row_bytes(format, n_cols);
  const uint32_t positions = n_used * n_tokens, padded = (positions + 31) / 32 * 32;
  _Float16 *hx = static_cast<_Float16 *>(split);
  float *unscale = reinterpret_cast<float *>(hx + frag_halves(padded, n_cols));
  // The inputs in the order of the grouped positions, so that a tile's
  // fragments are consecutive bytes (a shared token is converted once per
  // expert that takes it: 8 MB at 512 tokens, against a gather of 16-byte
  // pieces in every stage of every tile).
  split_hi(s, xf, positions, padded, n_cols, hx, unscale, entries, shared_input ? n_used : 1u,
           (shared_input ? n_tokens : positions) - 1);
  const HiInputs x{hx, unscale};
  const ExpertGroups g{offsets, entries, n_experts};
  // Tiles of 128 positions, or of 64 when the experts hold fewer: each tile
  // converts its rows' weights again, and that is what bounds it.  Pair and
  // down of 1792 x 2048, 32 experts, 4 a token: at 40 positions an expert 62
  // and 33 us with tiles of 64, 67 and 36 with 128; at 64 78 and 48, 74 and 41.
  // The two cross, with tokens spread evenly at random, at 33 positions an
  // expert of 128 experts, 46 of 64, 52 of 32 and 60 of 8.
  const bool few = positions <= 40 * n_experts;
  auto go = [&](auto fmt, auto mb, auto wr) {
    // 32·mb rows (half of them gate rows with `up`) x 128 / wr tokens.
    constexpr uint32_t F = decltype(fmt)::value;
    constexpr int MB = decltype(mb)::value, WR = decltype(wr)::value;
    const dim3 grid(div_ceil(n_rows, (up ? 16 : 32) * MB), div_ceil(positions, 128 / WR) + n_experts);
    if (up)
      k_gemm<F, 3, MB, 1, WR, true><<<grid, 256, 0, s>>>(W, up, rb, x, y, nullptr, n_rows, n_cols, positions, 1, g);
    else
      k_gemm<F, 0, MB, 1, WR, true><<<grid, 256, 0, s>>>(W, W, rb, x, y, nullptr, n_rows, n_cols, positions, 1, g);
  };
  constexpr std::integral_constant<int, 1> one{};
  constexpr std::integral_constant<int, 2> two{};
  if (format == BCH_Q4K && few)
    go(std::integral_constant<uint32_t, 12>{}, std::integral_constant<int, 4>{}, two);
  else if (format == BCH_Q4K)
    go(std::integral_constant<uint32_t, 12>{}, std::integral_constant<int, 4>{}, one);
  else if (format == BCH_F16)
    go(std::integral_constant<uint32_t, 1>{}, two, one);
  else
    go(std::integral_constant<uint32_t, 0>{}, two, one);
}

// --- bch_matmul_noalloc: the split inputs in a static device array ---------
//
// For callers that cannot allocate (code under graph capture, serving loops
// that forbid hipMalloc): the per-launch input split lives in `scratch`, a
// file-scope device array that every GPU the library runs on holds until the
// process ends.  Its device address on each GPU comes from
// hipGetSymbolAddress, once per device, when bch_open runs there; host code
// never passes the array's name itself to a kernel.  All calls on one GPU
// share the array: calls that overlap on one GPU (two streams, two threads)
// race on it.  Nothing in it needs clearing (each launch writes every byte it
// reads).

constexpr uint64_t kNoAllocScratchBytes = 16ull << 20;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices] = {};

int matmul_noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return fail(BCH_ERR_NO_DEVICE, "device %d beyond %d", device, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return BCH_OK;
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p)
    return fail(BCH_ERR_EXECUTION, "cannot find the no-allocation scratch on device %d: %s", device,
                hipGetErrorString(e));
  g_scratch_ptr[device] = p;
  return BCH_OK;
}

static void *noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[device];
}

}  // namespace bch

using namespace bch;

extern "C" uint64_t bch_matmul_noalloc_max_bytes(void) { return kNoAllocScratchBytes; }

extern "C" int bch_matmul_noalloc(bch_ctx *ctx, uint32_t format, bch_view weights, uint32_t n_rows, uint32_t n_cols,
                                  bch_view x, bch_view y, uint32_t n_tokens, uint32_t store) {
  if (!matmul_format(format))
    return fail(BCH_ERR_UNSUPPORTED_FORMAT, "format %u matrices have no matrix-matrix kernel", format);
  if (store > 2) return fail(BCH_ERR_ARGUMENT, "matmul_noalloc: unknown store mode %u", store);
  if (n_rows == 0 || n_cols == 0 || n_cols % kBK)
    return fail(BCH_ERR_ARGUMENT, "matmul_noalloc: %u x %u needs columns in multiples of %d", n_rows, n_cols, kBK);
  // The inputs plus the partials of the most column splits the shape may take
  // (bch_matmul's pick is one of them, and with this much room the launch
  // below picks the same, so the results equal bch_matmul's bit for bit).
  const uint32_t most = gemm_max_splits(n_rows, n_cols, n_tokens, (uint64_t)kMaxSplitK * n_tokens * n_rows, device_cus());
  const uint64_t need = (matmul_split_bytes(n_tokens, n_cols) + 255) / 256 * 256 +
                        (most > 1 ? 4ull * most * n_tokens * n_rows : 0);
  if (need > kNoAllocScratchBytes)
    return fail(BCH_ERR_ARGUMENT,
                "matmul_noalloc: %u tokens of %u x %u need %llu bytes of scratch, more than its %llu "
                "(use bch_matmul)",
                n_tokens, n_rows, n_cols, (unsigned long long)need, (unsigned long long)kNoAllocScratchBytes);
  const uint64_t rb = bch_row_bytes(format, n_cols);
  const uint8_t *W;
  const float *xp;
  float *yp;
  BCH_TRY(view_ptr(ctx, "matmul_noalloc", weights, rb * n_rows, &W));
  BCH_TRY(view_ptr(ctx, "matmul_noalloc", x, (uint64_t)n_tokens * n_cols * 4, &xp));
  BCH_TRY(view_ptr(ctx, "matmul_noalloc", y, (uint64_t)n_tokens * n_rows * 4, &yp));
  if (reinterpret_cast<uintptr_t>(W) % 16 || reinterpret_cast<uintptr_t>(xp) % 16)
    return fail(BCH_ERR_ARGUMENT, "matmul_noalloc: weights and inputs must be 16-byte aligned");
  void *split = noalloc_scratch(ctx->device);
  if (!split) return fail(BCH_ERR_NO_DEVICE, "matmul_noalloc: the scratch of device %d is not set up", ctx->device);
  if (!ctx->recording && !ctx->capturing) return fail(BCH_ERR_NOT_RECORDING, "no recording is open");
  // No profiling events here (creating them allocates): the launch only.
  if (n_tokens) run_matmul(ctx->stream, format, W, n_rows, n_cols, xp, yp, n_tokens, store, split, kNoAllocScratchBytes);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(BCH_ERR_EXECUTION, "matmul_noalloc launch: %s", hipGetErrorString(e));
  return BCH_OK;
}

extern "C" int bch_matmul(bch_ctx *ctx, uint32_t format, bch_view weights, uint32_t n_rows, uint32_t n_cols,
                          bch_view x, bch_view y, uint32_t n_tokens, uint32_t store) {
  if (!matmul_format(format))
    return fail(BCH_ERR_UNSUPPORTED_FORMAT, "format %u matrices have no matrix-matrix kernel", format);
  if (store > 2) return fail(BCH_ERR_ARGUMENT, "matmul: unknown store mode %u", store);
  if (n_rows == 0 || n_cols == 0 || n_cols % kBK)
    return fail(BCH_ERR_ARGUMENT, "matmul: %u x %u needs columns in multiples of %d", n_rows, n_cols, kBK);
  const uint64_t rb = bch_row_bytes(format, n_cols);
  const uint8_t *W;
  const float *xp;
  float *yp;
  BCH_TRY(view_ptr(ctx, "matmul", weights, rb * n_rows, &W));
  BCH_TRY(view_ptr(ctx, "matmul", x, (uint64_t)n_tokens * n_cols * 4, &xp));
  BCH_TRY(view_ptr(ctx, "matmul", y, (uint64_t)n_tokens * n_rows * 4, &yp));
  if (reinterpret_cast<uintptr_t>(W) % 16 || reinterpret_cast<uintptr_t>(xp) % 16)
    return fail(BCH_ERR_ARGUMENT, "matmul: weights and inputs must be 16-byte aligned");
  const char *name = format == 12 ? "matmul_q4k"
                     : format == 14 ? "matmul_q6k"
                     : format == 13 ? "matmul_q5k"
                     : format == 8  ? "matmul_q8_0"
                     : format == 2  ? "matmul_q4_0"
                     : format == 1  ? "matmul_f16"
                                    : "matmul_f32";
  void *split = nullptr;
  const uint64_t scratch_bytes = matmul_scratch_bytes(n_tokens, n_cols, n_rows);
  BCH_TRY(ctx_scratch(ctx, scratch_bytes, &split));
  return launch(ctx, {name, n_rows, n_cols, rb * n_rows}, [&](hipStream_t s) {
    if (n_tokens) run_matmul(s, format, W, n_rows, n_cols, xp, yp, n_tokens, store, split, scratch_bytes);
  });
}

namespace bch {

// ---------------------------------------------------------------------
// Expanded fp16 weights and the SwiGLU hand-off of the library GEMM pair
// ---------------------------------------------------------------------

// out[r][c] = the fp16 weight k_gemm dequantises into LDS for row r,
// column c (the same conversion code, so the same bits).  Two threads per
// 64-column stage of a row, each 16 columns of both halves.
template <uint32_t FMT>
__global__ __launch_bounds__(256) void k_expand_f16(const uint8_t *__restrict__ W, uint64_t row_bytes, uint32_t n_rows,
                                                    uint32_t n_cols, _Float16 *__restrict__ out) {
  const uint32_t n_stages = n_cols / kGk;
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint64_t)n_rows * n_stages * 2) return;
  const int c = (int)(i & 1);
  const uint64_t rs = i >> 1;
  const uint32_t row = (uint32_t)(rs / n_stages), st = (uint32_t)(rs % n_stages), sb = st / 4;
  const uint8_t *wr = W + (uint64_t)row * row_bytes;
  half8_t *dst = reinterpret_cast<half8_t *>(out + (uint64_t)row * n_cols + st * kGk + 16 * c);
  GemmW<FMT, 16> w;
  w.load_header(wr, sb, c);
  w.unpack(c);
  static_for<4>([&](auto stage) __attribute__((always_inline)) {
    constexpr int S = decltype(stage)::value;
    if (st % 4 != S) return;
    w.template load<S>(wr, sb, st, c);
    w.template scales<S>(c);
    static_for<8>([&](auto u) __attribute__((always_inline)) {
      constexpr int HI = decltype(u)::value / 4, D = decltype(u)::value % 4;
      w.template ints<S, HI, D>();
      w.template mix<S, HI, D>();
      if constexpr (D % 2 == 1) dst[4 * HI + D / 2] = w.w;
    });
  });
}

bool expand_f16_supported(uint32_t format, uint32_t n_cols) {
  return n_cols % kGk == 0 && (format == 12 || format == 1 || format == 0 || format == 13 || format == 14 ||
                               format == 8 || format == 2);
}

void run_expand_f16(hipStream_t s, uint32_t format, const uint8_t *W, uint32_t n_rows, uint32_t n_cols,
                    _Float16 *out) {
  const uint64_t rb = bch_row_bytes(format, n_cols);
  const uint64_t threads = (uint64_t)n_rows * (n_cols / kGk) * 2;
  const dim3 grid((uint32_t)div_ceil(threads, 256));
  switch (format) {
    case 12: k_expand_f16<12><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
    case 1: k_expand_f16<1><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
    case 14: k_expand_f16<14><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
    case 13: k_expand_f16<13><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
    case 8: k_expand_f16<8><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
    case 2: k_expand_f16<2><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
    default: k_expand_f16<0><<<grid, 256, 0, s>>>(W, rb, n_rows, n_cols, out); break;
  }
}

// Token t of the pair product D [n_tokens][2 n_ff] (gate rows, then up
// rows, of inputs scaled by 1/us[t]): ffn = silu(g·us)·(u·us), as k_gemm's
// paired epilogue computes it, then the fp16 inputs of the down projection
// exactly as k_split_hi makes them from ffn (H [n_tokens][n_ff], then
// unscale [n_tokens]).  F32 (optional) receives ffn itself.  PER as
// split_row.
template <int PER>
__global__ __launch_bounds__(256) void k_swiglu_split(const float *__restrict__ D, uint32_t n_ff,
                                                      const float *__restrict__ us, float *__restrict__ F32,
                                                      _Float16 *__restrict__ H, float *__restrict__ unscale) {
  const uint32_t t = frag_row_of(blockIdx.x, gridDim.x), n8 = (n_ff + 7) / 8, n4 = n_ff / 4;
  const float4 *g4 = reinterpret_cast<const float4 *>(D + (uint64_t)t * 2 * n_ff);
  const float4 *u4 = g4 + n4;
  const float s = us[t];
  auto act = [&](uint32_t i) {
    const float4 g = g4[i], u = u4[i];
    return float4{silu_f(g.x * s) * (u.x * s), silu_f(g.y * s) * (u.y * s), silu_f(g.z * s) * (u.z * s),
                  silu_f(g.w * s) * (u.w * s)};
  };
  float4 *f4 = F32 ? reinterpret_cast<float4 *>(F32 + (uint64_t)t * n_ff) : nullptr;
  split_row<PER>(n8, FragRow::of(H, t, gridDim.x, 8 * n8), unscale + t, [&](uint32_t i) {
    return Eight{act(2 * i), 2 * i + 1 < n4 ? act(2 * i + 1) : float4{0.f, 0.f, 0.f, 0.f}};
  }, [&](uint32_t i, const Eight &e) {
    if (!f4) return;
    f4[2 * i] = e.a;
    if (2 * i + 1 < n4) f4[2 * i + 1] = e.b;
  });
}

void run_swiglu_split(hipStream_t s, const float *D, uint32_t n_ff, uint32_t n_tokens, const float *us, float *f32,
                      void *scratch) {
  _Float16 *H = static_cast<_Float16 *>(scratch);
  float *unscale = reinterpret_cast<float *>(H + frag_halves(n_tokens, n_ff));
  const uint32_t per = div_ceil(div_ceil(n_ff, 8), 256);
  if (per <= 2)
    k_swiglu_split<2><<<n_tokens, 256, 0, s>>>(D, n_ff, us, f32, H, unscale);
  else if (per <= 6)
    k_swiglu_split<6><<<n_tokens, 256, 0, s>>>(D, n_ff, us, f32, H, unscale);
  else
    k_swiglu_split<0><<<n_tokens, 256, 0, s>>>(D, n_ff, us, f32, H, unscale);
}

}  // namespace bch
