// The LoRA delta of a grouped GEMM tile, on the matrix cores, in the tile's fp32 accumulators
// (the LORA instances of gemm_wide8_kernel, gemm_narrow_kernel and gemm_mfma_kernel):
//
//   acc[m, j] += lscale * sum_q t[m, q] * B[e, row(j), q]
//
// a rank-r product of the tile's t rows (t = x . A^T, fp32, from lora_t_mfma_kernel below) and the B
// rows of the tile's weight rows. Both operands are split into bf16 parts (t into three, B into as many
// as its dtype needs: split_parts8), exactly, and multiplied part by part on bf16 MFMAs with fp32
// accumulation: every product is exact, so the delta is an fp32 sum as the vector passes (lora.h)
// form it. At rank 16 the eight products of an fp32 adapter are about 5 % of a 256 x 256 gate_up tile's
// MFMAs; the delta costs no pass over the GEMM's output rows. Operands come straight from global
// memory, once per tile, at the tile's start (the accumulators begin as the scaled delta).
#pragma once

#include "gemm.h"
#include "lora.h"

namespace e4b {

// A value of the adapter, in its dtype.
E4B_DEV float adapter_at(const void* a, int dt, int64_t i) {
  if (dt == E4B_FP32) return static_cast<const float*>(a)[i];
  const uint16_t v = static_cast<const uint16_t*>(a)[i];
  return dt == E4B_BF16 ? to_f<E4B_BF16>(v) : to_f<E4B_FP16>(v);
}

// The leading bf16 part of v, taken off it, in the upper half of the result: truncated, so it never overflows
// and three parts hold any finite fp32 value exactly (two any fp16 one). FIRST (v may be any value): an
// infinity or NaN is its own first part and leaves zeros.
template <bool FIRST>
E4B_DEV uint32_t bf16_part(float& v) {
  if constexpr (FIRST) v = __builtin_canonicalizef(v);  // a NaN keeps a bit of its upper half
  const uint32_t b = __float_as_uint(v);
  const float rest = v - __uint_as_float(b & 0xffff0000u);
  v = !FIRST || __builtin_isfinite(v) ? rest : 0.0f;
  return b;
}

// bf16 pairs with their infinities and NaNs as zeros, for a delta's products with the other side's lower
// parts: those are zero wherever the leading part is all of the value, and an infinity times that zero
// would make the sum a NaN. (t, u and the weight gradients form a sum that comes out NaN again instead,
// value by value: cleaning their operands as they are read cost the 2,048-token training step 1.5 %.)
E4B_DEV uint32_t finite_pair(uint32_t w) {
  const uint32_t inf = ((w & 0x7f807f80u) + 0x00800080u) & 0x80008000u;  // exponents of all ones, in bits 15 and 31
  return w & ~((inf - (inf >> 15)) | inf);
}
E4B_DEV uint4 finite8(const uint4& v) {
  return make_uint4(finite_pair(v.x), finite_pair(v.y), finite_pair(v.z), finite_pair(v.w));
}

// Bf16 parts that hold an adapter value of dtype DT exactly.
template <int DT>
constexpr int kAdapterParts = DT == E4B_BF16 ? 1 : DT == E4B_FP16 ? 2 : 3;

// 8 fp32 values as NP bf16 parts, MFMA operand pieces (value 2i in the low half of word i).
template <int NP>
E4B_DEV void split_parts8(const float (&v)[8], uint4 (&part)[NP]) {
  uint32_t w[NP][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
    static_for<NP>([&](auto q) __attribute__((always_inline)) {
      if constexpr (int(q) == NP - 1) {
        w[q][i] = cvt_pair<E4B_BF16>(a, b);  // what is left fits a part: exact
      } else {
        const uint32_t pa = bf16_part<int(q) == 0>(a), pb = bf16_part<int(q) == 0>(b);
        w[q][i] = __builtin_amdgcn_perm(pb, pa, 0x07060302u);
      }
    });
  }
#pragma unroll
  for (int q = 0; q < NP; ++q) part[q] = make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]);
}

// The operand of a delta: three parts, and the leading one's finite values.
E4B_DEV void delta_parts8(const float (&v)[8], uint4 (&part)[4]) {
  uint4 p3[3];
  split_parts8<3>(v, p3);
  part[0] = p3[0]; part[1] = p3[1]; part[2] = p3[2];
  part[3] = finite8(p3[0]);
}

// The products of a delta: mul(a, b) for the parts of t and b (an adapter's, of dtype dt), all but that of the
// two last (below 2^-28 of |t||adapter|), the smaller ones first.
template <class F>
E4B_DEV void delta_products(int dt, const uint4 (&t)[4], const uint4 (&b)[4], F&& mul) {
  if (dt == E4B_FP32) {
    mul(t[1], b[2]);
    mul(t[3], b[2]);
  }
  if (dt != E4B_BF16) {
    mul(t[2], b[1]);
    mul(t[1], b[1]);
    mul(t[3], b[1]);
  }
  mul(t[2], b[3]);
  mul(t[1], b[3]);
  mul(t[0], b[0]);
}

// lscale * (2^e * t[m, q0 + i]) (0 past the rank), i = 0..7, split: the power of two goes to t, which is as
// small as e is large. With the rank a multiple of 8 the eight values are two 16-byte loads, else
// eight element loads.
template <class Args>
E4B_DEV void lora_t_piece(const Args& p, int64_t m, int q0, int e2, uint4 (&part)[4]) {
  float v[8];
  const float* t = p.lt + m * p.lr;
  if ((p.lr & 7) == 0) {
    const float4 a = *reinterpret_cast<const float4*>(t + (q0 < p.lr ? q0 : 0));
    const float4 b = *reinterpret_cast<const float4*>(t + (q0 < p.lr ? q0 : 0) + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = t[q0 + i < p.lr ? q0 + i : 0];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = q0 + i < p.lr ? __builtin_amdgcn_ldexpf(v[i], e2) * p.lscale : 0.0f;
  delta_parts8(v, part);
}

// 2^e * B[ex, row, q0 + i] (0 past the rank), i = 0..7, from the adapter dtype, split.
E4B_DEV void lora_b_piece(const GemmArgs& p, int ex, int64_t row, int q0, int e2, uint4 (&part)[4]) {
  float v[8];
  const int64_t base = (int64_t(ex) * p.w.n + row) * p.lr;
  const int64_t q0c = q0 < p.lr ? q0 : 0;
  if ((p.lr & 7) == 0 && p.lbdt == E4B_FP32) {
    const float4 a = *reinterpret_cast<const float4*>(static_cast<const float*>(p.lb) + base + q0c);
    const float4 b = *reinterpret_cast<const float4*>(static_cast<const float*>(p.lb) + base + q0c + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else if ((p.lr & 7) == 0) {
    const uint4 a = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.lb) + base + q0c);
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint16_t l = static_cast<uint16_t>(w[i]), h = static_cast<uint16_t>(w[i] >> 16);
      v[2 * i] = p.lbdt == E4B_BF16 ? to_f<E4B_BF16>(l) : to_f<E4B_FP16>(l);
      v[2 * i + 1] = p.lbdt == E4B_BF16 ? to_f<E4B_BF16>(h) : to_f<E4B_FP16>(h);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t o = base + (q0 + i < p.lr ? q0 + i : 0);
      if (p.lbdt == E4B_FP32) v[i] = static_cast<const float*>(p.lb)[o];
      else if (p.lbdt == E4B_BF16) v[i] = to_f<E4B_BF16>(static_cast<const uint16_t*>(p.lb)[o]);
      else v[i] = to_f<E4B_FP16>(static_cast<const uint16_t*>(p.lb)[o]);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = q0 + i < p.lr ? __builtin_amdgcn_ldexpf(v[i], e2) : 0.0f;
  delta_parts8(v, part);
}

// The t operands of a workgroup's BM rows and the 16 ranks from q0, split once for all its waves, in LDS (ts:
// 64 BM values): operand i of row r, ranks 8 h .. of the step, at 16-byte piece (2 i + h) BM + r. Row r is
// min(row0 + r, row_last), times 2^shift[r].
template <int BM, int NT, class Args>
E4B_DEV void lora_t_stage(const Args& p, uint16_t* ts, int64_t row0, int64_t row_last, const int* shift, int q0) {
  for (int j = threadIdx.x; j < 2 * BM; j += NT) {
    const int r = j % BM, h = j / BM;
    uint4 part[4];
    lora_t_piece(p, min(row0 + r, row_last), q0 + 8 * h, shift[r], part);
#pragma unroll
    for (int i = 0; i < 4; ++i) reinterpret_cast<uint4*>(ts)[(2 * i + h) * BM + r] = part[i];
  }
}

// The delta of the 32 x 32 accumulator blocks of eight waves that each hold all BM rows, weights first
// (v_mfma_f32_32x32x16: lane l supplies weight / tile row l % 32 and the eight ranks 8 (l / 32) .. of
// each 16-rank step), scaled like the fp16 mode's products: t rows times 2^shift (their activation row's,
// exact); B row brow, times 2^bshift (the expert's weight shift). Run on zeroed accumulators before a
// tile's main loop; the epilogue then removes the scales from the sum. ts: LDS that nothing else touches
// until the workgroup's next barrier. With every wave splitting all the rows' t itself an OLMoE layer at
// 1,531 tokens took 331 us, so 319.
template <int BM, int NT>
E4B_DEV void lora_delta_32x32(const GemmArgs& p, f32x16_t (&acc)[BM / 32], int e, int64_t row0, int64_t row_last,
                              const int* shift, int bshift, int64_t brow, uint16_t* ts, int lane) {
  const int half = lane >> 5;
  for (int q0 = 0; q0 < p.lr; q0 += 16) {
    if (q0) __syncthreads();  // the last step's t is read
    lora_t_stage<BM, NT>(p, ts, row0, row_last, shift, q0);
    uint4 b[4];
    lora_b_piece(p, e, brow, q0 + 8 * half, bshift, b);
    __syncthreads();
    static_for<BM / 32>([&](auto ms) {
      uint4 t[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) t[i] = reinterpret_cast<const uint4*>(ts)[(2 * i + half) * BM + 32 * int(ms) + (lane & 31)];
      delta_products(p.lbdt, t, b, [&](const uint4& tp, const uint4& bp) { acc[ms] = mfma_32x32x16<E4B_BF16>(bp, tp, acc[ms]); });
    });
  }
}

// 16 x 16 accumulator blocks (v_mfma_f32_16x16x32: lane l supplies row / column l % 16 and the
// eight ranks 8 (l / 16) .. of each 32-rank step); t row of block row ms: min(arow0 + 16 ms,
// arow_last); scales as above.
template <int MS, int NS, class AS>
E4B_DEV void lora_delta_16x16(const GemmArgs& p, f32x4_t (&acc)[MS][NS], int e, int64_t arow0, int64_t arow_last,
                              AS&& ashift, int bshift, const int64_t (&brow)[NS], int lane) {
  const int g8 = 8 * (lane >> 4);
  for (int q0 = 0; q0 < p.lr; q0 += 32) {
    uint4 t[MS][4];
#pragma unroll
    for (int ms = 0; ms < MS; ++ms) lora_t_piece(p, min(arow0 + 16 * ms, arow_last), q0 + g8, ashift(ms), t[ms]);
    static_for<NS>([&](auto ns) {
      uint4 b[4];
      lora_b_piece(p, e, brow[ns], q0 + g8, bshift, b);
      static_for<MS>([&](auto ms) {
        delta_products(p.lbdt, t[ms], b, [&](const uint4& tp, const uint4& bp) {
          acc[ms][ns] = mfma_16x16x32<E4B_BF16>(tp, bp, acc[ms][ns]);
        });
      });
    });
  }
}

// t[m, q] = sum_c x_m[c] * A[e, q, c] for the sorted rows m of every routing tile (one expert per
// tile), on the matrix cores: the t of the fp16-mode LoRA path (rows past the routed ones are not
// written). One workgroup per BM-row part of a tile, one wave per 16 rows, each wave all ranks of
// its rows (NSM 16-rank blocks) on v_mfma_f32_16x16x32_bf16. x rows are bf16 (exact operands); A is
// staged per 64-deep chunk in LDS as its bf16 parts (one of a bf16, two of an fp16, three of an fp32
// adapter: split_parts8), so every product is exact and t is an fp32 sum, as the VALU passes
// (lora_a_kernel) form it. The chunks are double-buffered, one barrier per chunk, with A two chunks and
// x three chunks ahead in registers: a launch has only a workgroup or two per CU, so the x loads in flight
// per wave set its rate. Both of an OLMoE layer's t at 1,531 tokens: 43 us one chunk ahead, 31 so; 38
// with an fp32 adapter's third part and the compensated totals.
constexpr int kLoraTK = 64;  // K per chunk
constexpr int kLoraTGroups = kLoraTK / 8;

// LDS element offset of the 16-byte group holding columns 8 g .. 8 g + 7 of rank row q: 128-byte
// rows with the groups XOR-swizzled by q % 8, so the fragment reads of 16 consecutive ranks at one
// group spread over all banks.
E4B_DEV int lora_t_at(int q, int g) { return q * kLoraTK + (((g ^ q) & 7) << 3); }

// The sums of t and u. One fp32 accumulator over the whole row was 1.5 times as far from 64 bits as the
// vector units' 64 partial sums; here at most eight products of 32 columns add up (each half of a chunk and
// the adapters' lower parts apart) before they go to the total, whose rounding errors are kept (two-sum):
// 0.7 times the vector units' error. (Four: 0.5 times, and 1.5 us more per launch at 258 tokens.)
template <int NSM, bool LOW>
struct RankSums {
  f32x4_t acc[LOW ? 3 : 2][NSM], total[NSM], lost[NSM];
  E4B_DEV RankSums() {
    const f32x4_t zero{0.0f, 0.0f, 0.0f, 0.0f};
    static_for<NSM>([&](auto n) __attribute__((always_inline)) {
      acc[0][n] = acc[1][n] = total[n] = lost[n] = zero;
      if constexpr (LOW) acc[2][n] = zero;
    });
  }
  E4B_DEV void fold() {
    static_for<2 * NSM>([&](auto j) __attribute__((always_inline)) {
      f32x4_t &a = acc[int(j) & 1][int(j) / 2], &t = total[int(j) / 2];
      const f32x4_t s = t + a, b = s - t;
      lost[int(j) / 2] += (t - (s - b)) + (a - b);
      t = s;
      a = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    });
  }
  E4B_DEV float value(int n, int i) const { return total[n][i] + (LOW ? lost[n][i] + acc[LOW ? 2 : 0][n][i] : lost[n][i]); }
};

template <int ADT, int BM, int NSM>
__global__ void __launch_bounds__(BM / 16 * kWave) lora_t_mfma_kernel(const uint16_t* __restrict__ x, int gather_k,
                                                                      e4b_routing rt, const void* __restrict__ A,
                                                                      int rank, int64_t in, float* __restrict__ t) {
  constexpr int NT = BM / 16 * kWave;
  constexpr int NP = kAdapterParts<ADT>;
  constexpr int NSTAGE = 16 * NSM * kLoraTGroups;  // 16-byte groups per chunk
  constexpr int SPT = (NSTAGE + NT - 1) / NT;      // staging groups per thread
  __shared__ __align__(16) uint16_t as[NP][2][16 * NSM * kLoraTK];
  const int sub = rt.tile_m / BM;
  const int tile = static_cast<int>(blockIdx.x) / sub;
  if (tile >= rt.meta[0]) return;  // uniform
  const int e = rt.tiles[2 * tile];
  const int row0 = rt.tiles[2 * tile + 1] + (static_cast<int>(blockIdx.x) % sub) * BM;
  const int rows = min(BM, rt.offsets[e + 1] - row0);
  if (rows <= 0) return;  // uniform: a part past the end of its expert's last tile
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & (kWave - 1), w = tid / kWave;
  const int l16 = lane & 15, g = lane >> 4;
  // the lane's x row (clamped to the part's rows; only real rows are stored)
  const int rr = row0 + min(16 * w + l16, rows - 1);
  const int64_t src = gather_k > 0 ? rt.sorted_flat[rr] / gather_k : rr;
  const uint16_t* xr = x + src * in;
  const int nchunks = static_cast<int>(in / kLoraTK);
  auto chunk = [&](int c) { return min(c, nchunks - 1); };  // past the last chunk it is re-read

  // staging: thread tid takes groups j = tid + NT i of the chunk's [16 NSM ranks][8 groups], as loaded until
  // they are stored (inlined always: a call left standing would put the sets in scratch memory)
  constexpr int kRaw = ADT == E4B_FP32 ? 2 : 1;
  uint4 sets[2][SPT][kRaw];
  auto load_a = [&](auto set, int c) __attribute__((always_inline)) {
    static_for<SPT>([&](auto i) __attribute__((always_inline)) {
      const int j = tid + NT * int(i);
      if (NSTAGE % NT != 0 && j >= NSTAGE) return;
      const int q = min(j / kLoraTGroups, rank - 1), gg = j % kLoraTGroups;
      const int64_t o = (int64_t(e) * rank + q) * in + int64_t(c) * kLoraTK + 8 * gg;  // 8 values: kRaw pieces
      const uint4* const src = static_cast<const uint4*>(A) + o / 8 * kRaw;
#pragma unroll
      for (int h = 0; h < kRaw; ++h) sets[decltype(set)::value][i][h] = src[h];
    });
  };
  auto store_a = [&](auto set, int buf) __attribute__((always_inline)) {
    static_for<SPT>([&](auto i) __attribute__((always_inline)) {
      const int j = tid + NT * int(i);
      if (NSTAGE % NT != 0 && j >= NSTAGE) return;
      const int q = j / kLoraTGroups, gg = j % kLoraTGroups;
      const uint4 (&raw)[kRaw] = sets[decltype(set)::value][i];
      uint4 part[NP];
      if constexpr (ADT == E4B_BF16) {  // its own only part
        part[0] = q < rank ? raw[0] : make_uint4(0, 0, 0, 0);
      } else {
        float v[8];
        load8<ADT>(raw, 0, v);
#pragma unroll
        for (int h = 0; h < 8; ++h) v[h] = q < rank ? v[h] : 0.0f;
        split_parts8<NP>(v, part);
      }
#pragma unroll
      for (int h = 0; h < NP; ++h) *reinterpret_cast<uint4*>(&as[h][buf][lora_t_at(q, gg)]) = part[h];
    });
  };
  // x fragments of a chunk: 32-deep step s takes columns 32 s + 8 g .. + 7
  auto load_x = [&](uint4 (&xf)[2], int c) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
      xf[s] = *reinterpret_cast<const uint4*>(xr + int64_t(c) * kLoraTK + 32 * s + 8 * g);
  };

  RankSums<NSM, (NP > 1)> sums;
  // chunk c from LDS buffer c % 2 and x set c % 4; meanwhile chunk c + 1's A goes from registers (set
  // (c + 1) % 2) into the other buffer, chunk c + 2's A and chunk c + 3's x are requested
  uint4 xs[4][2];
  auto step = [&](auto uc, int c) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;  // c % 4
    constexpr int cur = u & 1;
    load_a(std::integral_constant<int, cur>{}, chunk(c + 2));
    load_x(xs[(u + 3) & 3], chunk(c + 3));
    static_for<2>([&](auto s) __attribute__((always_inline)) {
      static_for<NSM>([&](auto ns) __attribute__((always_inline)) {
        const int at = lora_t_at(16 * int(ns) + l16, 4 * int(s) + g);
        static_for<NP>([&](auto h) __attribute__((always_inline)) {
          f32x4_t& to = sums.acc[int(h) == 0 ? int(s) : 2][ns];
          to = mfma_16x16x32<E4B_BF16>(xs[u][s], *reinterpret_cast<const uint4*>(&as[h][cur][at]), to);
        });
      });
    });
    store_a(std::integral_constant<int, cur ^ 1>{}, cur ^ 1);  // its last readers passed the previous barrier
    __syncthreads();
  };
  load_a(std::integral_constant<int, 0>{}, chunk(0));
#pragma unroll
  for (int i = 0; i < 3; ++i) load_x(xs[i], chunk(i));
  load_a(std::integral_constant<int, 1>{}, chunk(1));
  store_a(std::integral_constant<int, 0>{}, 0);
  __syncthreads();
  int c = 0;
  for (; c + 4 <= nchunks; c += 4) {
    static_for<4>([&](auto u) { step(u, c + int(u)); });
    if (c & 4) sums.fold();  // every second trip
  }
  static_for<3>([&](auto u) {
    if (c + int(u) < nchunks) step(u, c + int(u));
  });
  sums.fold();
  // a sum that came out NaN, once more by multiply-adds: neither the product of an infinity and a lower part
  // that is zero nor the rounding error of an infinite total is one of its terms
  auto again = [&](int r, int q) {
    const int64_t row = gather_k > 0 ? rt.sorted_flat[row0 + r] / gather_k : row0 + r;
    float v = 0.0f;
    for (int64_t c = 0; c < in; ++c)
      v = __builtin_fmaf(to_f<E4B_BF16>(x[row * in + c]), adapter_at(A, ADT, (int64_t(e) * rank + q) * in + c), v);
    return v;
  };
  // lane holds t[row 16 w + 4 g + i][rank 16 ns + l16]
#pragma unroll
  for (int ns = 0; ns < NSM; ++ns) {
    const int q = 16 * ns + l16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * w + 4 * g + i;
      if (q < rank && r < rows) {
        const float v = sums.value(ns, i);
        t[int64_t(row0 + r) * rank + q] = v == v ? v : again(r, q);
      }
    }
  }
}

}  // namespace e4b
