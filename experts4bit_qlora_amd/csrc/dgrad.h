// Input gradient of a frozen grouped projection in the fp16 matrix-core mode, for the training
// layer (e4b_train_backward):
//
//   out[m, :] = g[m, :] . deq(W[e_m]) + lscale * lt[m, :] . A[e_m]
//
// over expert-sorted rows: g [M, n] the gradient of the projection's output as scaled fp16 rows with
// their exponents (scale.h), W [E, n, k] NF4 weights times 2^shift[e] decoded through the LDS table
// of fp16 code pairs, lt = g . B the adapter's inner gradient [M, lr] and A [E, lr, k] the adapter:
// the delta is a rank-lr product in the tile's accumulators (lora_mfma.h), so no pass over the
// output rows adds it. The reduction runs over the weights' OUTPUT features, so an MFMA operand
// holds eight weight rows of one column, and packed bytes hold neighbours along the columns:
//
//   dgrad_wide_kernel    256 rows x 256 columns, eight waves of 128 x 64. Weights are decoded once per
//                        tile into LDS rows as they lie in memory (one lookup and one packed multiply
//                        per byte) and read as operands by transposing reads; gradient rows are
//                        staged as in the forward's wide kernel. One barrier per 64-deep step.
//   dgrad_narrow_kernel  32 rows x 256 columns for the experts' short tails and mid-size batches, bound
//                        by decoding the weights: nothing but the table is in LDS. A lane holds one
//                        packed word (eight columns) of eight weight rows, a coalesced load per row;
//                        v_perm pairs the decoded rows, and the eight columns of every lane are eight
//                        MFMA column blocks. The four waves take every fourth 16-deep step and their sums
//                        meet in LDS at the end: no barrier in the loop.
//
// Against dgrad_mfma_kernel (train.h: e4b_grouped_dgrad's exact bf16 weights, decoded in registers
// and transposed by v_perm before staging, the delta added by a pass of its own): both OLMoE projections
// at 2,048 tokens, rank 16, took 612 us there plus 141 us of delta passes, and take 361 us of wide
// launches here (600 and 496 TFLOP/s) with the narrow ones (76 us alone, 1.0-1.8 TB/s of weights) beside
// them on a second stream.
#pragma once

#include "gemm.h"
#include "gemm_wide.h"
#include "lora_mfma.h"

namespace e4b {

struct Dgrad16Args {
  const uint16_t* g;     // [M, w.n] scaled fp16 rows
  const int32_t* g_exp;  // [M] their exponents
  e4b_qweight w;
  e4b_routing rt;
  const float* lt;       // [M, lr] or null
  const void* la;        // [E, lr, w.k]
  int lbdt, lr;
  float lscale;
  void* out;             // [M, w.k] fp32, or bf16
  int out_f32;
};

constexpr int kDgradWideThreads = 512;
constexpr int kDgradNarrowThreads = 256;
constexpr int kDgradCols = 256;

// 4 x 16-bit transposing LDS read: the 16 lanes of a group name the 16 8-byte pieces of a 4-row x
// 16-column block (lane i: row i / 4, columns 4 (i % 4) ..) and lane i receives column i, rows 0..3.
E4B_DEV uint2 lds_read_tr(const uint16_t* p) {
  typedef short s4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4_t* lds_t;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p)));
}

// Eight 16-bit columns of the lane's row from two runs of four packed into two words each (v, and w the
// run eight columns on), the lane halves holding columns 4 (l / 32) .. of each run: after the swap
// the lower half stores the first run's eight columns, the upper half the second's.
E4B_DEV void store_runs8(uint16_t* row, int half, const uint32_t (&v)[2], const uint32_t (&w)[2]) {
  const auto a = __builtin_amdgcn_permlane32_swap(v[0], w[0], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(v[1], w[1], false, false);
  *reinterpret_cast<uint4*>(row + 8 * half) = make_uint4(a[0], b[0], a[1], b[1]);
}

// One tile. HALF: at most 128 rows (waves of 64 x 64).
template <int FMT, bool HALF>
E4B_DEV void dgrad_wide_tile(const Dgrad16Args& p, int e, int row0, int row_end, int c_tile,
                             uint16_t (&As)[2][kWideTileM * kTileK], uint16_t (&Ws)[2][kTileK * kDgradCols],
                             const float* code2_s, int* row_shift_s, const uint32_t* ptab) {
  constexpr int BM = HALF ? kWideTileM / 2 : kWideTileM;
  constexpr int MS = BM / 64, NS = 2;  // 32 x 32 blocks per wave: BM / 2 rows x 64 columns
  constexpr int AP = BM * kTileK / 8 / kDgradWideThreads;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid) / kWave;
  const int wave_m = wid & 1, wave_c = wid >> 1;
  const int half = lane >> 5, c32 = lane & 31;
  const int64_t n = p.w.n, K = p.w.k;
  const int64_t c0 = int64_t(c_tile) * kDgradCols;

  // gradient piece i of thread t: tile row 64 i + t / 8, columns 8 (t % 8) .. of the step (rows past the
  // expert's end read its last one: never stored)
  uint32_t aoff[AP];
#pragma unroll
  for (int i = 0; i < AP; ++i)
    aoff[i] = static_cast<uint32_t>((int64_t(min(row0 + 64 * i + (tid >> 3), row_end - 1)) * n) / 8 + (tid & 7));
  const int wsh = min(p.w.shift[e], kDeltaShiftMax);
  const int g_exp_row = p.g_exp[min(row0 + (tid & (BM - 1)), row_end - 1)];
  // weights: thread t decodes columns 32 (t % 8) .. + 31 of weight row t / 8 of the step (columns past k
  // read column 0: never stored)
  const int wr = tid >> 3, wc = tid & 7;
  const int64_t cc = c0 + 32 * wc < K ? c0 + 32 * wc : 0;
  const uint8_t* wptr = p.w.packed + (int64_t(e) * n + wr) * (K / 2) + cc / 2;
  const int64_t nb = n * (K / 64);
  const int64_t blk0 = int64_t(wr) * (K / 64) + cc / 64;
  const float offset = (FMT == E4B_FMT_NF4_DQ) ? p.w.offset[e] : 0.0f;

  f32x16_t acc[MS][NS];
  static_for<MS>([&](auto ms) { static_for<NS>([&](auto ns) { acc[ms][ns] = f32x16_t{}; }); });

  u32x4_t areg[AP];
  uint4 wq;
  float sa;
  uint32_t sq = 0;
  auto load_a = [&](int i, int64_t s) {
    areg[i] = (reinterpret_cast<const u32x4_t*>(p.g) + s * (kTileK / 8))[aoff[i]];
  };
  auto load_w = [&](int64_t s) {
    wq = *reinterpret_cast<const uint4*>(wptr + s * kTileK * (K / 2));
    const int64_t blk = blk0 + s * kTileK * (K / 64);
    if constexpr (FMT == E4B_FMT_NF4) {
      sa = static_cast<const float*>(p.w.absmax)[e * nb + blk];
    } else {
      sq = static_cast<const uint8_t*>(p.w.absmax)[e * nb + blk];
      sa = p.w.absmax2[e * ((nb + 255) / 256) + blk / 256];
    }
  };
  auto scale_pair = [&]() -> uint32_t {
    float scale = sa;
    if constexpr (FMT == E4B_FMT_NF4_DQ) {
      const float prod = code2_s[sq] * sa;
      scale = prod + offset;
    }
    scale = __builtin_amdgcn_ldexpf(scale, wsh);
    return cvt_pair<E4B_FP16>(scale, scale);
  };
  // Weight tile in LDS: 512-byte rows (one per weight row of the step) of eight 64-byte pieces, piece
  // c at c ^ (row & 3): the four rows of a transposing read lie in distinct banks. A thread stores its
  // piece's four 16-byte parts in the order i ^ sw, so that the sixteen lanes LDS serves together (two
  // rows x eight pieces) write sixteen distinct bank groups.
  const int sw = (((wc >> 2) << 1) | (wr & 1)) & 3;
  const int w_st = wr * kDgradCols + ((wc ^ (wr & 3)) << 5) + (sw << 3);
  auto store_a = [&](int buf, int i) {
    *reinterpret_cast<u32x4_t*>(&As[buf][lds_at_w(64 * i + (tid >> 3), 8 * (tid & 7))]) = areg[i];
  };
  uint32_t rw[4];  // the words in store order
  auto rotate = [&]() {
    const uint32_t x = (sw & 1) ? wq.y : wq.x, y = (sw & 1) ? wq.x : wq.y;
    const uint32_t z = (sw & 1) ? wq.w : wq.z, w = (sw & 1) ? wq.z : wq.w;
    rw[0] = (sw & 2) ? z : x;
    rw[1] = (sw & 2) ? w : y;
    rw[2] = (sw & 2) ? x : z;
    rw[3] = (sw & 2) ? y : w;
  };
  const uint32_t* tab = ptab + (lane & (kPairCopies - 1));
  auto store_w = [&](int buf, int i, uint32_t sc) {
    uint32_t o[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) o[b] = pk_mul_f16(tab[((rw[i] >> (8 * b)) & 0xffu) * kPairCopies], sc);
    *reinterpret_cast<uint4*>(&Ws[buf][w_st ^ (i << 3)]) = make_uint4(o[0], o[1], o[2], o[3]);
  };

  // operands of MFMA group j (16 weight rows): gradient rows as in the forward's wide kernel; weight
  // columns 64 wave_c + 32 ns + lane % 32, rows 16 j + 8 half .. + 7 by two transposing reads
  const int a_frag = (wave_m * (BM / 2) + c32) * kTileK;
  const int a_sw = (lane ^ (c32 >> 3)) & 7;
  auto frag_a = [&](int buf, int j, int ms) -> uint4 {
    const int fcol = ((2 * j + half) ^ a_sw) << 3;
    return *reinterpret_cast<const uint4*>(&As[buf][a_frag + ms * 32 * kTileK + (fcol ^ ((ms & 1) << 5))]);
  };
  const int tr_row = 8 * half + ((lane & 15) >> 2);
  int w_frag[NS];
#pragma unroll
  for (int ns = 0; ns < NS; ++ns)
    w_frag[ns] = tr_row * kDgradCols + (((2 * wave_c + ns) ^ (tr_row & 3)) << 5) + (((lane >> 4) & 1) << 4) + 4 * (lane & 3);
  auto frag_w = [&](int buf, int j, int ns) -> uint4 {
    const uint16_t* at = &Ws[buf][w_frag[ns] + j * 16 * kDgradCols];
    const uint2 lo = lds_read_tr(at), hi = lds_read_tr(at + 4 * kDgradCols);
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
  };

  const int64_t steps = n / kTileK, last = steps - 1;
#pragma unroll
  for (int i = 0; i < AP; ++i) load_a(i, 0);
  load_w(0);
  if (tid < BM) row_shift_s[tid] = exp_shift(g_exp_row);
  __syncthreads();  // code2 table, code-pair table, row shifts
  if (p.lt) {
    // the accumulators start as the tile's delta, scaled like the products; gradient buffer 1 is free until
    // step 0, one barrier further on
    uint16_t* const ts = As[1];
    for (int q0 = 0; q0 < p.lr; q0 += 16) {
      if (q0) __syncthreads();  // the last step's t is read
      lora_t_stage<BM, kDgradWideThreads>(p, ts, row0, row_end - 1, row_shift_s, q0);
      uint4 b[NS][4];
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) {
        const int64_t c = c0 + 64 * wave_c + 32 * ns + c32;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int q = q0 + 8 * half + i;
          const float x = adapter_at(p.la, p.lbdt, (int64_t(e) * p.lr + (q < p.lr ? q : 0)) * K + (c < K ? c : 0));
          v[i] = q < p.lr ? __builtin_amdgcn_ldexpf(x, wsh) : 0.0f;
        }
        delta_parts8(v, b[ns]);
      }
      __syncthreads();
      static_for<MS>([&](auto ms) {
        uint4 t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          t[i] = reinterpret_cast<const uint4*>(ts)[(2 * i + half) * BM + wave_m * (BM / 2) + 32 * int(ms) + c32];
        static_for<NS>([&](auto ns) {
          delta_products(p.lbdt, t, b[ns], [&](const uint4& tp, const uint4& bp) {
            acc[ms][ns] = mfma_32x32x16<E4B_BF16>(bp, tp, acc[ms][ns]);
          });
        });
      });
    }
  }
  {
    const uint32_t sc = scale_pair();
    rotate();
    load_w(min<int64_t>(1, last));
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      store_a(0, i);
      load_a(i, min<int64_t>(1, last));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) store_w(0, i, sc);
  }
  __syncthreads();
  // step s: the next group's operands are read while this group multiplies; step s + 1 is staged
  // ahead of the step's barrier, which lies before the last group (its MFMAs cover the next step's
  // first reads). Past the last step the loads re-read it and the staged buffer is not used.
  uint4 fa[2][MS], fw[2][NS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) fa[0][ms] = frag_a(0, 0, ms);
#pragma unroll
  for (int ns = 0; ns < NS; ++ns) fw[0][ns] = frag_w(0, 0, ns);
  for (int64_t s = 0; s < steps; ++s) {
    const int cur = static_cast<int>(s & 1);
    const uint32_t sc = scale_pair();
    rotate();
    load_w(min<int64_t>(s + 2, last));
    static_for<4>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j == 3) __syncthreads();
      const int nbuf = j < 3 ? cur : cur ^ 1;
      constexpr int nj = (j + 1) & 3;
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) fa[nj & 1][ms] = frag_a(nbuf, nj, ms);
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) fw[nj & 1][ns] = frag_w(nbuf, nj, ns);
      static_for<MS>([&](auto ms) {
        static_for<NS>([&](auto ns) {
          acc[ms][ns] = mfma_32x32x16<E4B_FP16>(fw[j & 1][int(ns)], fa[j & 1][int(ms)], acc[ms][ns]);
        });
      });
      if constexpr (j < 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if ((j == 0 && i < 2) || (j > 0 && i == j + 1)) {
            if (i < AP) {
              store_a(cur ^ 1, i);
              load_a(i, min<int64_t>(s + 2, last));
            }
            store_w(cur ^ 1, i, sc);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // lane holds row 32 ms + lane % 32 of the wave's rows, columns 8 q + 4 half + 0..3 of each 32-column
  // block (q = 0..3); the operand scales come off first (exact)
  const int lane_e = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
  const int half_e = lane_e >> 5;
  static_for<MS>([&](auto ms) {
    const int r = wave_m * (BM / 2) + 32 * int(ms) + (lane_e & 31);
    const int d = -(row_shift_s[r] + wsh);
    static_for<NS>([&](auto ns) {
      const int64_t c = c0 + 64 * wave_c + 32 * int(ns);
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = __builtin_amdgcn_ldexpf(acc[ms][ns][i], d);
      if (row0 + r < row_end && c < K) {  // K is a multiple of 64: blocks are whole
        if (p.out_f32) {
          float* const row = static_cast<float*>(p.out) + int64_t(row0 + r) * K + c + 4 * half_e;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(row + 8 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        } else {
          uint16_t* const row = static_cast<uint16_t*>(p.out) + int64_t(row0 + r) * K + c;
          uint32_t w[4][2];
#pragma unroll
          for (int q = 0; q < 8; ++q) w[q / 2][q & 1] = cvt_pair<E4B_BF16>(v[2 * q], v[2 * q + 1]);
          store_runs8(row, half_e, w[0], w[1]);
          store_runs8(row + 16, half_e, w[2], w[3]);
        }
      }
    });
    __builtin_amdgcn_sched_barrier(0);
  });
}

template <int FMT>
__global__ void __launch_bounds__(kDgradWideThreads) dgrad_wide_kernel(Dgrad16Args p) {
  static_assert(FMT != E4B_FMT_MXFP4, "NF4 weights");
  __shared__ __attribute__((aligned(16))) uint16_t As[2][kWideTileM * kTileK];
  __shared__ __attribute__((aligned(16))) uint16_t Ws[2][kTileK * kDgradCols];
  __shared__ float code2_s[(FMT == E4B_FMT_NF4_DQ) ? 256 : 1];
  __shared__ int row_shift_s[kWideTileM];
  __shared__ uint32_t ptab[256 * kPairCopies];
  const int c_tiles = static_cast<int>((p.w.k + kDgradCols - 1) / kDgradCols);
  const TileItem item = tile_item(p.rt, c_tiles);
  if (!item.ok) return;
  const int end = p.rt.offsets[item.e + 1];
  {
    // pass j fills entries 32 j + t / 16, copy t % 16
    const float lo = p.w.code[(threadIdx.x / kPairCopies) & 15];
    const int odd = threadIdx.x / kPairCopies >= 16;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      ptab[j * kDgradWideThreads + threadIdx.x] = cvt_pair<E4B_FP16>(p.w.code[2 * j + odd], lo);
    if constexpr (FMT == E4B_FMT_NF4_DQ) {
      if (threadIdx.x < 256) code2_s[threadIdx.x] = p.w.code2[threadIdx.x];
    }
  }
  if (end - item.row0 <= kWideTileM / 2)
    dgrad_wide_tile<FMT, true>(p, item.e, item.row0, min(item.row0 + kWideTileM / 2, end), item.n_tile, As, Ws, code2_s,
                               row_shift_s, ptab);
  else
    dgrad_wide_tile<FMT, false>(p, item.e, item.row0, min(item.row0 + kWideTileM, end), item.n_tile, As, Ws, code2_s,
                                row_shift_s, ptab);
}

template <int FMT>
__global__ void __launch_bounds__(kDgradNarrowThreads) __attribute__((amdgpu_waves_per_eu(2)))
dgrad_narrow_kernel(Dgrad16Args p) {
  static_assert(FMT != E4B_FMT_MXFP4, "NF4 weights");
  constexpr int kCopies = 64;
  constexpr int NB = 8;  // MFMA column blocks: block b holds columns 8 c + b
  __shared__ __attribute__((aligned(256))) uint32_t ptab[256 * kCopies];
  __shared__ float code2_s[(FMT == E4B_FMT_NF4_DQ) ? 256 : 1];
  const int c_tiles = static_cast<int>((p.w.k + kDgradCols - 1) / kDgradCols);
  const TileItem item = tile_item(p.rt, c_tiles);
  if (!item.ok) return;
  const int e = item.e, row0 = item.row0;
  const int row_end = min(row0 + kTileMSmall, p.rt.offsets[e + 1]);
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid) / kWave;
  const int half = lane >> 5, c32 = lane & 31;
  const int64_t n = p.w.n, K = p.w.k;
  const int64_t c0 = int64_t(item.n_tile) * kDgradCols;
  // the lane's eight columns (columns past k read column 0: never stored) and its gradient row
  const int64_t cl = c0 + 8 * c32 < K ? c0 + 8 * c32 : 0;
  const int grow = min(row0 + c32, row_end - 1);
  const int wsh = min(p.w.shift[e], kDeltaShiftMax);
  const int rsh = exp_shift(p.g_exp[grow]);
  const float offset = (FMT == E4B_FMT_NF4_DQ) ? p.w.offset[e] : 0.0f;
  {
    // wave w fills entries w + 4 i (high nibble i / 4, low nibble w + 4 (i % 4)), a copy per lane
    float lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) lo[i] = p.w.code[wid + 4 * i];
#pragma unroll
    for (int i = 0; i < 64; ++i)
      ptab[(wid + 4 * i) * kCopies + lane] = cvt_pair<E4B_FP16>(p.w.code[i >> 2], lo[i & 3]);
    if constexpr (FMT == E4B_FMT_NF4_DQ) code2_s[tid] = p.w.code2[tid];
  }
  // uniform bases plus 32-bit lane offsets (one expert's weights and scales stay below 4 GB)
  const int64_t nb = n * (K / 64), nb2 = (nb + 255) / 256;
  const uint8_t* const wbase = p.w.packed + int64_t(e) * n * (K / 2);
  const uint32_t w_off = static_cast<uint32_t>(8 * half * (K / 2) + cl / 2);
  const uint16_t* const gbase = p.g + int64_t(row0) * n;
  const uint32_t g_off = static_cast<uint32_t>((grow - row0) * n + 8 * half);

  // step t (16 weight rows): the lane's words of rows 16 t + 8 half + i, its gradient piece, and ONE block
  // scale: eight neighbouring lanes hold the 64 columns of one block, and lane i of them loads and
  // decodes row i's scale for all (every lane loading its eight rows' scales kept the load pipeline
  // busy: 25 load instructions per step instead of 11, 322 -> 263 us for both projections of the
  // Qwen3 step at 509 tokens, with the loads kept in order below)
  uint32_t wq[2][8];
  float sa[2];
  uint32_t sq[2];
  uint4 gv[2];
  const uint32_t s_off = static_cast<uint32_t>((8 * half + (lane & 7)) * (K / 64) + cl / 64);
  auto load = [&](auto set_c, int64_t t) {
    constexpr int set = decltype(set_c)::value;
    gv[set] = *reinterpret_cast<const uint4*>(gbase + 16 * t + g_off);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      wq[set][i] = *reinterpret_cast<const uint32_t*>(wbase + (16 * t + i) * (K / 2) + w_off);
    if constexpr (FMT == E4B_FMT_NF4) {
      sa[set] = (static_cast<const float*>(p.w.absmax) + int64_t(e) * nb + 16 * t * (K / 64))[s_off];
    } else {
      sq[set] = (static_cast<const uint8_t*>(p.w.absmax) + int64_t(e) * nb + 16 * t * (K / 64))[s_off];
      sa[set] = (p.w.absmax2 + int64_t(e) * nb2)[(static_cast<uint32_t>(16 * t * (K / 64)) + s_off) / 256];
    }
  };
  f32x16_t acc[NB];
  static_for<NB>([&](auto b) { acc[b] = f32x16_t{}; });
  const uint32_t copy_off = lane * 4;
  auto step = [&](auto set_c) {
    constexpr int set = decltype(set_c)::value;
    uint32_t sc[8];
    {
      float scale = sa[set];
      if constexpr (FMT == E4B_FMT_NF4_DQ) {
        const float prod = code2_s[sq[set]] * sa[set];
        scale = prod + offset;
      }
      scale = __builtin_amdgcn_ldexpf(scale, wsh);
      const int own = static_cast<int>(cvt_pair<E4B_FP16>(scale, scale));
      static_for<8>([&](auto ic) {  // row_newbcast: lane i of each 16 to its lower eight, lane 8 + i to its upper
        constexpr int i = decltype(ic)::value;
        const int lower = __builtin_amdgcn_update_dpp(0, own, 0x150 + i, 0xf, 0x3, false);
        sc[i] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(lower, own, 0x158 + i, 0xf, 0xc, false));
      });
    }
    static_for<4>([&](auto bc) {  // packed byte: columns 8 c + 2 b and + 1
      constexpr int b = decltype(bc)::value;
      uint32_t v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t addr = __builtin_amdgcn_perm(wq[set][i], copy_off, 0x0c0c0000u | (uint32_t(4 + b) << 8));
        v[i] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(ptab) + addr);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = pk_mul_f16(v[i], sc[i]);
      uint32_t ev[4], od[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ev[q] = __builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], 0x05040100u);
        od[q] = __builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], 0x07060302u);
      }
      acc[2 * b] = mfma_32x32x16<E4B_FP16>(make_uint4(ev[0], ev[1], ev[2], ev[3]), gv[set], acc[2 * b]);
      acc[2 * b + 1] = mfma_32x32x16<E4B_FP16>(make_uint4(od[0], od[1], od[2], od[3]), gv[set], acc[2 * b + 1]);
    });
  };
  // n is a multiple of 64: every wave has n / 64 steps, wave w the steps w, w + 4, ...
  const int64_t steps = n / 64;
  auto at = [&](int64_t i) { return wid + 4 * min(i, steps - 1); };
  load(std::integral_constant<int, 0>{}, at(0));
  load(std::integral_constant<int, 1>{}, at(1));
  __syncthreads();  // tables
  if (p.lt) {  // the delta, scaled like the products: wave w takes the 16-rank steps w, w + 4, ...
    for (int q0 = 16 * wid; q0 < p.lr; q0 += 64) {
      uint4 t[4];
      lora_t_piece(p, grow, q0 + 8 * half, rsh, t);
      static_for<NB>([&](auto b) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int q = q0 + 8 * half + i;
          const float x = adapter_at(p.la, p.lbdt, (int64_t(e) * p.lr + (q < p.lr ? q : 0)) * K + cl + int(b));
          v[i] = q < p.lr ? __builtin_amdgcn_ldexpf(x, wsh) : 0.0f;
        }
        uint4 a[4];
        delta_parts8(v, a);
        delta_products(p.lbdt, t, a, [&](const uint4& tp, const uint4& ap) { acc[b] = mfma_32x32x16<E4B_BF16>(ap, tp, acc[b]); });
      });
    }
  }
  int64_t i = 0;
  for (; i + 2 <= steps; i += 2) {
    // the order is kept by hand: loads moved across a step make its wait one for the newest loads
    step(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    load(std::integral_constant<int, 0>{}, at(i + 2));
    __builtin_amdgcn_sched_barrier(0);
    step(std::integral_constant<int, 1>{});
    __builtin_amdgcn_sched_barrier(0);
    load(std::integral_constant<int, 1>{}, at(i + 3));
    __builtin_amdgcn_sched_barrier(0);
  }
  if (i < steps) step(std::integral_constant<int, 0>{});

  // The waves' sums: accumulators 4 w .. 4 w + 3 of every block belong to wave w, which adds the other
  // waves' in wave order. Half the blocks at a time fit the table's LDS: slot (block, source wave,
  // owner) of 4 accumulators x 64 lanes.
  f32x4_t* const red = reinterpret_cast<f32x4_t*>(ptab);  // [4 blocks][4 sources][4 owners][64]
  f32x4_t sum[NB];
  static_for<2>([&](auto h) {
    __syncthreads();  // the table's (the first half's) reads are done
    static_for<4>([&](auto b) {
      static_for<4>([&](auto o) {
        const f32x16_t& a = acc[4 * int(h) + int(b)];
        red[((int(b) * 4 + wid) * 4 + int(o)) * kWave + lane] =
            f32x4_t{a[4 * int(o)], a[4 * int(o) + 1], a[4 * int(o) + 2], a[4 * int(o) + 3]};
      });
    });
    __syncthreads();
    static_for<4>([&](auto b) {
      f32x4_t s = red[(int(b) * 16 + wid) * kWave + lane];
#pragma unroll
      for (int src = 1; src < 4; ++src) s += red[((int(b) * 4 + src) * 4 + wid) * kWave + lane];
      sum[4 * int(h) + int(b)] = s;
    });
  });
  // accumulator 4 w + i of block b: column 8 (8 w + 4 half + i) + b of row lane % 32, so a lane holds 32
  // neighbouring columns
  const int64_t c = c0 + 64 * wid + 32 * half;
  if (row0 + c32 >= row_end || c >= K) return;
  const int d = -(rsh + wsh);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float v[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) v[b] = __builtin_amdgcn_ldexpf(sum[b][q], d);
    const int64_t o = int64_t(row0 + c32) * K + c + 8 * q;
    if (p.out_f32) {
      float4* const to = reinterpret_cast<float4*>(static_cast<float*>(p.out) + o);
      to[0] = make_float4(v[0], v[1], v[2], v[3]);
      to[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.out) + o) =
          make_uint4(cvt_pair<E4B_BF16>(v[0], v[1]), cvt_pair<E4B_BF16>(v[2], v[3]), cvt_pair<E4B_BF16>(v[4], v[5]),
                     cvt_pair<E4B_BF16>(v[6], v[7]));
    }
  }
}

}  // namespace e4b
