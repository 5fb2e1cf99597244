// The fp16 inputs of the prefill GEMM as its tile reads them (gemm_tile.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bch {

// Fragment-major inputs: blocks of 32 tokens (the last holds the R that
// remain, so nothing is padded), in a block [k / 8][token][k % 8].  Lane
// l of a k-step of 16 columns reads 16 bytes: token l % 32, columns
// 16·step + 8·(l / 32).  Offset in halves of columns 8·k8 .. of token t.
__host__ __device__ __forceinline__ uint64_t frag_offset(uint32_t t, uint32_t k8, uint32_t n_tokens, uint32_t n_cols) {
  const uint32_t b = t / 32, R = n_tokens - 32 * b < 32 ? n_tokens - 32 * b : 32;
  return (uint64_t)b * 32 * n_cols + ((uint64_t)k8 * R + t % 32) * 8;
}

// Where a token's fp16 inputs go: columns 8i .. 8i+7 at base + i·stride.
struct FragRow {
  _Float16 *base;
  uint32_t stride;  // halves between pieces of eight columns
  __device__ __forceinline__ static FragRow of(_Float16 *h, uint32_t t, uint32_t n_tokens, uint32_t n_cols) {
    const uint32_t b = t / 32;
    return {h + frag_offset(t, 0, n_tokens, n_cols), 8 * min(32u, n_tokens - 32 * b)};
  }
  __device__ __forceinline__ _Float16 *at(uint32_t k) const { return base + (uint64_t)(k / 8) * stride + k % 8; }
};

// The row that workgroup `b` of `rows` one-row workgroups converts.  Eight
// consecutive rows share each 128-byte line of a fragment block; workgroup b
// runs on XCD b % 8, so whole runs of 64 are dealt so that such eight meet in
// one XCD's L2, which then writes whole lines.
__device__ __forceinline__ uint32_t frag_row_of(uint32_t b, uint32_t rows) {
  return b < rows / 64 * 64 ? b / 64 * 64 + b % 8 * 8 + b / 8 % 8 : b;
}

}  // namespace bch
