// Blockwise 4-bit quantization of dense weights (the storage side: `quantize_4bit` at
// _vendor/experts.py:408-426): per 64 consecutive values the largest magnitude, each value times
// its reciprocal to the nearest code (the count of code midpoints below it), two codes per byte
// with the first in the high nibble. Bit for bit the torch formulation in quant.py.
//
// Bound by HBM: one read of the dense stack, half a byte per value written. Eight lanes hold one
// block (eight values each: the block maximum is seven max and three cross-lane steps), so a
// wave's loads are contiguous and a lane's codes are one 4-byte store. The nearest code costs
// one LDS lookup and one compare per value: [-1, 1] is cut into 32 cells (`fma(x, 16, 16)`
// truncated, monotone in x), a cell holds the number of midpoints in the cells below it and the
// one midpoint inside it, which needs codes whose midpoints are no closer than a cell (NF4).
// Other codes, and blocks whose scale is not a normal number (their products can be NaN), count
// all 15 midpoints. One OLMoE layer's stacks (402 M bf16 values): 12.6 ms as torch operations
// (24 chunks of ~20 passes over 64-bit indexes), 0.23 ms here for the whole call, 4.5 TB/s (a device
// copy of 4 GiB reaches 4.7 TB/s).
#pragma once

#include "common.h"

namespace e4b {

constexpr int kQuantThreads = 256;
constexpr int kQuantUnroll = 4;   // 8-value pieces per thread, their loads in flight together
constexpr int kQuantCells = 33;   // 32 cells of [-1, 1) and the one that 1 falls in

// A 16-entry code, by value: sorted midpoints, the code of each sorted position (four bits each),
// and the code of an all-zero block.
struct QuantCode {
  float mids[15];
  uint64_t perm;
  int zero;
};

// The sorted position of x: midpoints below it (an exact midpoint goes to the lower code, a NaN
// to the last, as torch.bucketize orders them).
E4B_DEV int quant_count(const QuantCode& q, float x) {
  int c = 0;
#pragma unroll
  for (int i = 0; i < 15; ++i) c += !(q.mids[i] >= x);
  return c;
}

E4B_DEV int quant_cell(float x) { return static_cast<int>(__builtin_fmaf(x, 16.0f, 16.0f)); }

template <int DT, bool CELLS>
__global__ void __launch_bounds__(kQuantThreads) quantize4_kernel(const void* __restrict__ w, int64_t pieces,
                                                                  QuantCode q, uint32_t* __restrict__ packed,
                                                                  float* __restrict__ absmax) {
  __shared__ float2 cells[CELLS ? kQuantCells : 1];
  if constexpr (CELLS) {
    if (threadIdx.x < kQuantCells) {
      int below = 0;
      float mid = __builtin_inff();
#pragma unroll
      for (int i = 0; i < 15; ++i) {
        const int c = quant_cell(q.mids[i]);
        below += c < static_cast<int>(threadIdx.x);
        if (c == static_cast<int>(threadIdx.x)) mid = q.mids[i];
      }
      cells[threadIdx.x] = make_float2(mid, __builtin_bit_cast(float, below));
    }
    __syncthreads();
  }
  // piece = eight values; a block's eight pieces sit in eight neighbouring lanes. Every piece of
  // the grid's tail block group reads piece 0 (never stored).
  const int64_t first = int64_t(blockIdx.x) * (kQuantThreads * kQuantUnroll) + threadIdx.x;
  uint32_t raw[kQuantUnroll][DT == E4B_FP32 ? 8 : 4];
#pragma unroll
  for (int u = 0; u < kQuantUnroll; ++u) {
    const int64_t p = first + u * kQuantThreads;
    const int64_t pc = p < pieces ? p : 0;
    const uint4* src = static_cast<const uint4*>(w) + pc * (DT == E4B_FP32 ? 2 : 1);
#pragma unroll
    for (int i = 0; i < (DT == E4B_FP32 ? 2 : 1); ++i) {
      const uint4 v = src[i];
      raw[u][4 * i] = v.x; raw[u][4 * i + 1] = v.y; raw[u][4 * i + 2] = v.z; raw[u][4 * i + 3] = v.w;
    }
  }
#pragma unroll
  for (int u = 0; u < kQuantUnroll; ++u) {
    const int64_t p = first + u * kQuantThreads;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (DT == E4B_FP32) v[i] = __uint_as_float(raw[u][i]);
      else v[i] = (i & 1) ? hi_f<DT>(raw[u][i / 2]) : lo_f<DT>(raw[u][i / 2]);
    }
    // as integers the magnitudes order like the values, a NaN above infinity: it stays the maximum
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = max(m, __float_as_uint(v[i]) & 0x7fffffffu);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o)));
    const float am = __uint_as_float(m);
    const bool some = am > 0.0f;  // false for a NaN too: such a block takes the zero code
    const float inv = some ? 1.0f / am : 0.0f;
    uint32_t word = 0;
    // a normal scale and its reciprocal: every product lies within a rounding of [-1, 1]
    const bool plain = !some || (m >= 0x00800000u && m < 0x7f000000u);
    if (CELLS && __all(plain)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = v[i] * inv;
        const float2 cell = cells[some ? quant_cell(x) : 0];
        const uint32_t idx = __builtin_bit_cast(uint32_t, cell.y) + !(cell.x >= x);
        word |= idx << (8 * (i / 2) + ((i & 1) ? 0 : 4));
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int pos = quant_count(q, v[i] * inv);
        const uint32_t idx = static_cast<uint32_t>(q.perm >> (4 * pos)) & 15u;
        word |= idx << (8 * (i / 2) + ((i & 1) ? 0 : 4));
      }
    }
    if (!some) word = static_cast<uint32_t>(q.zero) * 0x11111111u;
    if (p < pieces) {
      packed[p] = word;
      if ((p & 7) == 0) absmax[p >> 3] = am;
    }
  }
}

constexpr int kQuant8Block = 256;

// Second level of double quantization: rows of n values, each less its row's offset, in blocks of 256 to
// a sorted 256-entry code whose 255 midpoints lie in device memory (`double_quant` in quant.py bit for
// bit). A row's last block is padded with zeros. Block (row, 256-value block), one value per thread: its
// code by an eight-step search of the midpoints in LDS. Small (1 / 64 of the weights), so bound by
// launches: ~25 torch operations with two device-to-host copies each became this one.
__global__ void __launch_bounds__(kQuant8Block) quantize8_kernel(const float* __restrict__ values,
                                                                 const float* __restrict__ offset, int64_t n,
                                                                 int64_t blocks, const float* __restrict__ mids,
                                                                 int zero, uint8_t* __restrict__ codes,
                                                                 float* __restrict__ absmax) {
  __shared__ float mid_s[kQuant8Block];
  __shared__ uint32_t top[kQuant8Block / kWave];
  const int64_t row = blockIdx.x / blocks, b = blockIdx.x % blocks;
  const int64_t i = b * kQuant8Block + threadIdx.x;
  mid_s[threadIdx.x] = threadIdx.x < kQuant8Block - 1 ? mids[threadIdx.x] : 0.0f;
  const float c = i < n ? values[row * n + i] - offset[row] : 0.0f;
  uint32_t m = __float_as_uint(c) & 0x7fffffffu;  // a NaN stays the maximum
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o)));
  if ((threadIdx.x & (kWave - 1)) == 0) top[threadIdx.x / kWave] = m;
  __syncthreads();
  m = max(max(top[0], top[1]), max(top[2], top[3]));
  const float am = __uint_as_float(m);
  const bool some = am > 0.0f;
  const float x = c * (some ? 1.0f / am : 0.0f);
  int pos = 0;  // midpoints below x: the search keeps mids[pos - 1] < x (a NaN passes them all)
#pragma unroll
  for (int s = kQuant8Block / 2; s > 0; s >>= 1) pos += !(mid_s[pos + s - 1] >= x) ? s : 0;
  if (i < n) codes[row * n + i] = static_cast<uint8_t>(some ? pos : zero);
  if (threadIdx.x == 0) absmax[blockIdx.x] = am;
}

}  // namespace e4b
