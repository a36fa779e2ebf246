// Row kernels of the training layer (e4b_train_forward / e4b_train_backward): what lies between its
// grouped GEMMs, one wave per row, every value read and written once. The layer ran these as torch
// elementwise operations (a dozen passes over [M, n] rows each way) and the adapters' inner products
// on the VALU.
//
//   train_act_kernel      h = act(proj) with its scaled fp16 rows for the down GEMM
//   train_act_bwd_kernel  dL/dproj from dL/dh and proj, likewise
//   combine_bwd_kernel    dL/ddown rows and the router weights' gradients from dL/dout
//   lora_u_mfma_kernel    u = g . B[e] on the matrix cores, B read in its parameter layout
#pragma once

#include "common.h"
#include "dgrad.h"
#include "lora.h"
#include "lora_mfma.h"
#include "route.h"
#include "scale.h"
#include "train.h"

namespace e4b {

constexpr int kRowThreads = 256;

E4B_DEV void unpack8(const uint4& q, float (&v)[8]) {
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = lo_f<E4B_BF16>(w[i]);
    v[2 * i + 1] = hi_f<E4B_BF16>(w[i]);
  }
}
E4B_DEV uint4 pack8(const float (&v)[8]) {
  return make_uint4(cvt_pair<E4B_BF16>(v[0], v[1]), cvt_pair<E4B_BF16>(v[2], v[3]), cvt_pair<E4B_BF16>(v[4], v[5]),
                    cvt_pair<E4B_BF16>(v[6], v[7]));
}
// a bf16 piece times 2^d as fp16 (exact for the row's shift; see bf16x2_to_f16x2)
E4B_DEV uint4 scaled16(const uint4& a, int d) {
  return make_uint4(bf16x2_to_f16x2(a.x, d), bf16x2_to_f16x2(a.y, d), bf16x2_to_f16x2(a.z, d), bf16x2_to_f16x2(a.w, d));
}

// A wave's row of `pieces` 16-byte pieces made by piece(i, first), to rows `out` (bf16) and `out16` (the same
// values as scaled fp16, exponent to *exp). RP pieces per lane stay in registers between finding the
// row's exponent and scaling; a longer row makes its remaining pieces twice. first: the piece is the
// lane's own and made for the first time.
template <int RP, class F>
E4B_DEV void make_row(int64_t pieces, F&& piece, uint4* out, uint4* out16, int32_t* exp) {
  const int lane = threadIdx.x & (kWave - 1);
  uint4 v[RP];
  uint32_t m = 0;
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const int64_t i = lane + int64_t(j) * kWave;
    v[j] = piece(i < pieces ? i : 0, i < pieces);
    m = max(m, bf16_exp_max(v[j]));
  }
  for (int64_t i = lane + int64_t(RP) * kWave; i < pieces; i += kWave) m = max(m, bf16_exp_max(piece(i, true)));
  m = wave_max_u32(m);
  if (lane == 0) *exp = static_cast<int32_t>(m >> 7);
  const int d = exp_shift(static_cast<int>(m >> 7));
#pragma unroll
  for (int j = 0; j < RP; ++j) {
    const int64_t i = lane + int64_t(j) * kWave;
    if (i < pieces) {
      out[i] = v[j];
      out16[i] = scaled16(v[j], d);
    }
  }
  for (int64_t i = lane + int64_t(RP) * kWave; i < pieces; i += kWave) {
    const uint4 a = piece(i, false);
    out[i] = a;
    out16[i] = scaled16(a, d);
  }
}

// torch.clamp's value: a NaN stays one (fminf would drop it).
E4B_DEV float clamp_to(float v, float lo, float hi) { return v < lo ? lo : (v > hi ? hi : v); }

// h[m] = bf16(act(proj[m])) for the routed rows: gated (proj rows of 2 I: gate, then up) or single.
template <bool GATED, int RP>
__global__ void __launch_bounds__(kRowThreads) train_act_kernel(const uint16_t* __restrict__ proj,
                                                                const int32_t* __restrict__ offsets, int E, int64_t I,
                                                                int epi, float limit, uint16_t* __restrict__ h,
                                                                uint16_t* __restrict__ h16, int32_t* __restrict__ h_exp) {
  const int64_t row = int64_t(blockIdx.x) * (kRowThreads / kWave) + threadIdx.x / kWave;
  if (row >= offsets[E]) return;  // whole waves; no barrier follows
  const uint4* pr = reinterpret_cast<const uint4*>(proj + row * (GATED ? 2 * I : I));
  make_row<RP>(I / 8, [&](int64_t i, bool) {
    float g[8], o[8];
    unpack8(pr[i], g);
    if constexpr (GATED) {
      float u[8];
      unpack8(pr[I / 8 + i], u);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (epi == E4B_EPI_CLAMP_SWIGLU && limit > 0.0f) {
          g[q] = g[q] > limit ? limit : g[q];
          u[q] = clamp_to(u[q], -limit, limit);
        }
        o[q] = silu_f32(g[q]) * u[q];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) o[q] = silu_f32(g[q]);
    }
    return pack8(o);
  }, reinterpret_cast<uint4*>(h + row * I), reinterpret_cast<uint4*>(h16 + row * I), h_exp + row);
}

// dproj[m] = dL/dproj from dh = dL/dh and proj. A clamp (limit > 0) passes the gradient where its
// input lies within the limits, as torch.clamp does.
template <bool GATED, int RP>
__global__ void __launch_bounds__(kRowThreads) train_act_bwd_kernel(
    const uint16_t* __restrict__ dh, const uint16_t* __restrict__ proj, const int32_t* __restrict__ offsets, int E,
    int64_t I, int epi, float limit, uint16_t* __restrict__ dproj, uint16_t* __restrict__ dproj16,
    int32_t* __restrict__ exp) {
  const int64_t row = int64_t(blockIdx.x) * (kRowThreads / kWave) + threadIdx.x / kWave;
  if (row >= offsets[E]) return;
  const int64_t half = I / 8;
  const uint4* pr = reinterpret_cast<const uint4*>(proj + row * (GATED ? 2 * I : I));
  const uint4* dr = reinterpret_cast<const uint4*>(dh + row * I);
  const bool clamp = epi == E4B_EPI_CLAMP_SWIGLU && limit > 0.0f;
  make_row<RP>(GATED ? 2 * half : half, [&](int64_t i, bool) {
    const bool up = GATED && i >= half;
    const int64_t c = up ? i - half : i;
    float g[8], d[8], o[8];
    unpack8(pr[c], g);
    unpack8(dr[c], d);
    if constexpr (GATED) {
      float u[8];
      unpack8(pr[half + c], u);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const bool gin = !clamp || g[q] <= limit, uin = !clamp || (u[q] >= -limit && u[q] <= limit);
        const float gc = clamp && g[q] > limit ? limit : g[q];
        const float uc = clamp ? clamp_to(u[q], -limit, limit) : u[q];
        const float s = sigmoid_f32(gc);
        const float dg = d[q] * uc * (s * (1.0f + gc * (1.0f - s)));
        const float du = d[q] * (gc * s);
        o[q] = up ? (uin ? du : 0.0f) : (gin ? dg : 0.0f);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float s = sigmoid_f32(g[q]);
        o[q] = d[q] * (s * (1.0f + g[q] * (1.0f - s)));
      }
    }
    return pack8(o);
  }, reinterpret_cast<uint4*>(dproj + row * (GATED ? 2 * I : I)),
     reinterpret_cast<uint4*>(dproj16 + row * (GATED ? 2 * I : I)), exp + row);
}

// The combine's backward for flat row f = token t, slot s (sorted row m = inv[f]): d[m] =
// bf16(w[f] * grad[t]) with its scaled fp16 row, and gw[f] = down[m] . grad[t] (a dropped id: no row,
// gradient 0). One wave per flat row.
template <int GDT, int RP>
__global__ void __launch_bounds__(kRowThreads) combine_bwd_kernel(const void* __restrict__ grad,
                                                                  const uint16_t* __restrict__ down,
                                                                  const int32_t* __restrict__ inv,
                                                                  const void* __restrict__ wts, int wdt, int64_t M, int k,
                                                                  int64_t H, uint16_t* __restrict__ d,
                                                                  uint16_t* __restrict__ d16, int32_t* __restrict__ exp,
                                                                  void* __restrict__ gw) {
  const int64_t f = int64_t(blockIdx.x) * (kRowThreads / kWave) + threadIdx.x / kWave;
  if (f >= M) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int m = inv[f];
  auto put = [&](float v) {
    if (!gw || lane != 0) return;
    if (wdt == E4B_FP32) static_cast<float*>(gw)[f] = v;
    else static_cast<uint16_t*>(gw)[f] = wdt == E4B_BF16 ? from_f<E4B_BF16>(v) : from_f<E4B_FP16>(v);
  };
  if (m < 0) {
    put(0.0f);
    return;
  }
  const float w = adapter_at(wts, wdt, f);
  const int64_t t = f / k;
  const uint4* dn = reinterpret_cast<const uint4*>(down + int64_t(m) * H);
  float dot = 0.0f;
  make_row<RP>(H / 8, [&](int64_t i, bool first) {
    float g[8], x[8], o[8];
    load8<GDT>(grad, t * H + 8 * i, g);
    unpack8(dn[i], x);
    float s = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      s = __builtin_fmaf(g[q], x[q], s);
      o[q] = w * g[q];
    }
    dot += first ? s : 0.0f;
    return pack8(o);
  }, reinterpret_cast<uint4*>(d + int64_t(m) * H), reinterpret_cast<uint4*>(d16 + int64_t(m) * H), exp + m);
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) dot += __shfl_xor(dot, o);
  put(dot);
}

// The adapter gradients of a call without tokens.
__global__ void __launch_bounds__(kRowThreads) zero_halves_kernel(uint16_t* __restrict__ p, int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * kRowThreads + threadIdx.x; i < n; i += int64_t(gridDim.x) * kRowThreads) p[i] = 0;
}

// u[m, q] = sum_c g_m[c] * B[e, c, q] for the sorted rows of every routing tile: lora_t_mfma_kernel with
// the adapter matrix in the other orientation (its ranks contiguous), so a 64-deep chunk is staged in
// LDS as it lies in memory ([64 c][ranks], one array per bf16 part) and its operands come from
// transposing reads instead of a transposed copy of B. VEC: whole 16-byte pieces of ranks (rank a
// multiple of 8, B aligned), a template argument because a branch around the loads makes every
// later wait a wait for all of them (both of an OLMoE step's u at 2,048 tokens: 105 -> 67 us).
template <int BDT, int BM, int NSM, bool VEC>
__global__ void __launch_bounds__(BM / 16 * kWave) lora_u_mfma_kernel(const uint16_t* __restrict__ g, e4b_routing rt,
                                                                      const void* __restrict__ B, int rank, int64_t n,
                                                                      float* __restrict__ u) {
  constexpr int NT = BM / 16 * kWave;
  constexpr int RB = 16 * NSM;
  constexpr int NP = kAdapterParts<BDT>;
  constexpr int NSTAGE = kLoraTK * RB / 8;     // 8-rank groups per chunk
  constexpr int SPT = (NSTAGE + NT - 1) / NT;  // per thread
  __shared__ __align__(16) uint16_t bs[NP][2][kLoraTK * RB];
  const int sub = rt.tile_m / BM;
  const int tile = static_cast<int>(blockIdx.x) / sub;
  if (tile >= rt.meta[0]) return;  // uniform
  const int e = rt.tiles[2 * tile];
  const int row0 = rt.tiles[2 * tile + 1] + (static_cast<int>(blockIdx.x) % sub) * BM;
  const int rows = min(BM, rt.offsets[e + 1] - row0);
  if (rows <= 0) return;  // uniform: a part past the end of its expert's last tile
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & (kWave - 1), w = tid / kWave;
  const int l16 = lane & 15, gr = lane >> 4;
  const uint16_t* xr = g + int64_t(row0 + min(16 * w + l16, rows - 1)) * n;
  const int nchunks = static_cast<int>(n / kLoraTK);
  auto chunk = [&](int c) { return min(c, nchunks - 1); };  // past the last chunk it is re-read
  float sets[2][SPT][8];
  auto load_b = [&](auto set, int c) __attribute__((always_inline)) {
    float (&sv)[SPT][8] = sets[decltype(set)::value];
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
      const int j = tid + NT * i;
      if (NSTAGE % NT != 0 && j >= NSTAGE) break;
      const int row = j / (RB / 8), q0 = 8 * (j % (RB / 8));
      const int64_t o = (int64_t(e) * n + int64_t(c) * kLoraTK + row) * rank;
      if constexpr (VEC) {
        load8<BDT>(B, o + (q0 < rank ? q0 : 0), sv[i]);
      } else {
#pragma unroll
        for (int h = 0; h < 8; ++h) sv[i][h] = adapter_at(B, BDT, o + (q0 + h < rank ? q0 + h : 0));
      }
#pragma unroll
      for (int h = 0; h < 8; ++h) sv[i][h] = q0 + h < rank ? sv[i][h] : 0.0f;
    }
  };
  auto store_b = [&](auto set, int buf) __attribute__((always_inline)) {
    const float (&sv)[SPT][8] = sets[decltype(set)::value];
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
      const int j = tid + NT * i;
      if (NSTAGE % NT != 0 && j >= NSTAGE) break;
      const int at = wgrad_at<RB>(j / (RB / 8), 8 * (j % (RB / 8)));
      uint4 part[NP];
      split_parts8<NP>(sv[i], part);
#pragma unroll
      for (int h = 0; h < NP; ++h) *reinterpret_cast<uint4*>(&bs[h][buf][at]) = part[h];
    }
  };
  auto load_x = [&](uint4 (&xf)[2], int c) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
      xf[s] = *reinterpret_cast<const uint4*>(xr + int64_t(c) * kLoraTK + 32 * s + 8 * gr);
  };
  auto operand = [&](const uint16_t* b, int s, int base) -> uint4 {
    const int row = 32 * s + 8 * gr + (l16 >> 2), col = base + 4 * (l16 & 3);
    const uint2 lo = lds_read_tr(b + wgrad_at<RB>(row, col));
    const uint2 hi = lds_read_tr(b + wgrad_at<RB>(row + 4, col));
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
  };
  RankSums<NSM, (NP > 1)> sums;
  uint4 xs[4][2];  // B two chunks and g three chunks ahead, as lora_t_mfma_kernel
  auto step = [&](auto uc, int c) __attribute__((always_inline)) {
    constexpr int v = decltype(uc)::value;  // c % 4
    constexpr int cur = v & 1;
    load_b(std::integral_constant<int, cur>{}, chunk(c + 2));
    load_x(xs[(v + 3) & 3], chunk(c + 3));
    static_for<2>([&](auto s) __attribute__((always_inline)) {
      static_for<NSM>([&](auto ns) __attribute__((always_inline)) {
        static_for<NP>([&](auto h) __attribute__((always_inline)) {
          f32x4_t& to = sums.acc[int(h) == 0 ? int(s) : 2][ns];
          to = mfma_16x16x32<E4B_BF16>(xs[v][s], operand(bs[h][cur], s, 16 * ns), to);
        });
      });
    });
    store_b(std::integral_constant<int, cur ^ 1>{}, cur ^ 1);  // its last readers passed the previous barrier
    __syncthreads();
  };
  load_b(std::integral_constant<int, 0>{}, chunk(0));
#pragma unroll
  for (int i = 0; i < 3; ++i) load_x(xs[i], chunk(i));
  load_b(std::integral_constant<int, 1>{}, chunk(1));
  store_b(std::integral_constant<int, 0>{}, 0);
  __syncthreads();
  int c = 0;
  for (; c + 4 <= nchunks; c += 4) {
    static_for<4>([&](auto q) { step(q, c + int(q)); });
    if (c & 4) sums.fold();  // every second trip
  }
  static_for<3>([&](auto q) {
    if (c + int(q) < nchunks) step(q, c + int(q));
  });
  sums.fold();
  auto again = [&](int r, int q) {  // as lora_t_mfma_kernel
    float v = 0.0f;
    for (int64_t c = 0; c < n; ++c)
      v = __builtin_fmaf(to_f<E4B_BF16>(g[int64_t(row0 + r) * n + c]), adapter_at(B, BDT, (int64_t(e) * n + c) * rank + q), v);
    return v;
  };
#pragma unroll
  for (int ns = 0; ns < NSM; ++ns) {
    const int q = 16 * ns + l16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * w + 4 * gr + i;
      if (q < rank && r < rows) {
        const float v = sums.value(ns, i);
        u[int64_t(row0 + r) * rank + q] = v == v ? v : again(r, q);
      }
    }
  }
}

}  // namespace e4b
