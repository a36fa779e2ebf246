// Prefill grouped GEMM, wide tiles with two waves per SIMD: 256 sorted rows x 256 weight rows
// per workgroup, eight waves of 256 x 32 each on 32 x 32 x 16 MFMAs. Two weight formats: in the
// fp16 matrix-core mode (F16C: bf16 activations stored as scaled fp16 rows, NF4 / double-quant
// NF4 weights decoded through an LDS code-pair table, v_mfma_f32_32x32x16_f16), and MXFP4 with
// bf16 activations (e2m1 bytes converted in registers by v_cvt_scalef32_pk_bf16_fp4, exact in
// bf16, v_mfma_f32_32x32x16_bf16; groups 0 and 1 of a step are one e8m0 block, 2 and 3 the next).
//
// Weights never pass through LDS: every lane loads packed bytes of its own MFMA column's weight
// row and decodes them into the operand registers. Lane half h (l / 32) loads K = 32 h .. + 31 of
// a 64-deep step, one 16-byte load; two v_permlane32_swap give each half the words it feeds to
// the four MFMA groups, K = 16 j + 8 h .. + 7, so K runs in its natural order. With all 256 rows
// of the tile in one wave each weight is still decoded exactly once per tile. Against staging the
// decoded weights in LDS (eight waves of 128 x 64) a step writes 32 KB and reads 64 KB less there
// and its barrier waits for no decode: launches alone, Qwen3 gate_up / down at 4,096 tokens
// 272 / 173 -> 235 / 145 us, both gpt-oss projections at 2,048 tokens 665 -> ~500 us. What is left:
// the matrix cores' own rate (a register-only loop of these MFMAs on random data is held to
// 1.6 PFLOP/s by the card's power limit, 1.4 with one fragment read per MFMA), ~12 us per tile
// before its first and after its last step, and the last round's idle CUs.
//
// Pipeline: step s computes from activation buffer s % 2 while step s + 1's activation pieces are
// stored from registers into the other buffer and those registers take the global loads of step
// s + 2; a weight set (two) takes step s + 2's bytes once step s has decoded them; one barrier
// per step. A chunk of MFMAs covers the fragment reads of the next chunk and the table lookups of
// the next MFMA group.
//
// The weights are the MFMA's first operand, so lane l holds tile row l % 32 and weight columns
// 8 * (i / 4) + 4 * (l / 32) + i % 4, i = 0..15, of each 32 x 32 block: a row's scale is one value
// per lane and block, a lane's columns come in runs of four (v_permlane32_swap makes them runs of
// eight, one 16-byte store), and a gated tile, whose waves hold 16 gate and the same 16 up columns,
// has accumulators i and i + 8 of one lane to combine. (With the activations first a lane held
// one column of 16 rows: 128 two-byte stores per lane, and the launch with two of its 32 steps took
// 76 us for the Qwen3 down projection at 4,096 tokens.)
#pragma once

#include "gemm.h"
#include "gemm_wide.h"
#include "lora_mfma.h"

namespace e4b {

constexpr int kWide8Threads = 512;

// The code-pair table: entry of byte value b for lane l at byte address 256 b + 4 (l % 32). One
// v_perm_b32 forms the address, and the 32 lanes that LDS serves together read 32 banks.
constexpr int kWide8Copies = 32;
constexpr int kWide8TabStride = 64;  // words per entry

// A tile's record and its rows' sources, loaded by the kernel in the round trip after the tile's
// (beside the code tables' loads): the expert, its first sorted row and the expert's row end, and
// in the fp16 mode, for thread t, the sources of tile rows 64 i + t / 8 (i < 4: its activation
// pieces) and t % 256 (its row shift) -- sorted_flat at each row clamped to the last one with a
// gather, the row itself without. Sources of rows past the expert's end are dropped where they
// are used.
struct Wide8Rows {
  int e, row0, end;
  int sf[5];
};

// One tile. HALF: a tile of at most 128 rows as 128 rows x 256 weight rows (waves of 128 x 32).
template <int DT, int FMT, bool F16C, bool HALF, bool LORA, bool H16>
E4B_DEV void wide8_tile(const GemmArgs& p, const Wide8Rows& tr, int n_tile, uint16_t (&As)[2][kWideTileM * kTileK],
                        const float* code2_s, int* row_shift_s, const uint32_t* ptab) {
  constexpr int CT = F16C ? E4B_FP16 : DT;
  constexpr int BM = HALF ? kWideTileM / 2 : kWideTileM, BN = kWideTileN;
  constexpr int MS = BM / 32;  // 32-row MFMA tiles per wave
  constexpr int NT = kWide8Threads;
  constexpr int AP = BM * kTileK / 8 / NT;  // 16-byte activation pieces per thread and step
  constexpr int RS = 2;                     // register sets of global loads
  const bool pair = is_gated(p.epi);
  const int cols = pair ? BN / 2 : BN;
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid) / kWave;
  const int half = lane >> 5;
  const int e = tr.e;
  const int row0 = tr.row0;
  const int row_end = min(row0 + BM, tr.end);
  const int64_t n = p.w.n;
  const int64_t k = p.w.k;
  const int64_t col0 = int64_t(n_tile) * cols;
  if (col0 >= p.n_out) return;

  // activation piece i of thread t: tile row 64 i + t / 8, columns 8 (t % 8) .. + 7 (eight lanes
  // read one row's 128 contiguous bytes); aoff[i]: that piece of step 0 in 16-byte units of p.a
  const int apart = tid & 7;
  const bool gather = p.gather_k > 0;
  auto row_src = [&](int r, int s) -> int64_t { return r < row_end ? (gather ? s / p.gather_k : s) : 0; };
  uint32_t aoff[AP];
#pragma unroll
  for (int i = 0; i < AP; ++i) {
    const int r = row0 + 64 * i + (tid >> 3);
    if constexpr (F16C) {
      aoff[i] = static_cast<uint32_t>((row_src(r, tr.sf[i]) * k) / 8 + apart);
    } else {
      // bf16 activations (MXFP4): each source loaded here behind its row test, which measured
      // ~1 % faster for the gpt-oss prefill than the sources loaded ahead by the kernel
      const int64_t src = (r < row_end) ? (gather ? p.rt.sorted_flat[r] / p.gather_k : r) : 0;
      aoff[i] = static_cast<uint32_t>((src * k) / 8 + apart);
    }
  }
  const int wsh = F16C ? (LORA ? min(p.w.shift[e], kDeltaShiftMax) : p.w.shift[e]) : 0;
  // the exponent of tile row t (t < BM), stored to row_shift_s (the epilogue's shifts) once the
  // first steps' loads are out
  const int a_exp_row = F16C ? p.a_exp[row_src(row0 + (tid & (kWideTileM - 1)), tr.sf[4])] : 0;
  // weights: wave w's MFMA column c = lane % 32 is weight row col0 + 32 w + c; for a gated epilogue
  // columns 0..15 are the gate rows of output columns col0 + 16 w + c, columns 16..31 their up
  // rows. Columns past n_out read weight row 0 and are never stored
  const int c32 = lane & 31;
  const int64_t jcol = pair ? col0 + 16 * wid + (c32 & 15) : col0 + 32 * wid + c32;  // the lane's output column
  const int64_t grow = jcol < p.n_out ? jcol + (pair && c32 >= 16 ? n / 2 : 0) : 0;
  const uint8_t* wptr = p.w.packed + (int64_t(e) * n + grow) * (k / 2) + 16 * half;
  const int64_t nb = n * (k / 64);
  const float offset = (FMT == E4B_FMT_NF4_DQ) ? p.w.offset[e] : 0.0f;

  f32x16_t acc[MS];
  static_for<MS>([&](auto ms) { acc[ms] = f32x16_t{}; });

  u32x4_t areg[AP];
  uint4 wq[RS];
  float sa[RS];
  uint32_t sq[RS];  // double quant: code index; MXFP4: the e8m0 scale of the lane's loaded values
  auto load_a = [&](int i, int64_t kb) {
    areg[i] = (reinterpret_cast<const u32x4_t*>(p.a) + kb * (kTileK / 8))[aoff[i]];
  };
  auto load_w = [&](int set, int64_t kb) {
    wq[set] = *reinterpret_cast<const uint4*>(wptr + kb * 32);
    if constexpr (FMT == E4B_FMT_MXFP4) {
      sq[set] = static_cast<const uint8_t*>(p.w.absmax)[(int64_t(e) * n + grow) * (k / 32) + 2 * kb + half];
    } else if constexpr (FMT == E4B_FMT_NF4) {
      sa[set] = static_cast<const float*>(p.w.absmax)[e * nb + grow * (k / 64) + kb];
    } else {
      const int64_t blk = grow * (k / 64) + kb;
      sq[set] = static_cast<const uint8_t*>(p.w.absmax)[e * nb + blk];
      sa[set] = p.w.absmax2[e * ((nb + 255) / 256) + blk / 256];
    }
  };
  // a step's block scale: as an fp16 pair with 2^shift applied (exact) for the table decode; for
  // the e2m1 conversion the e8m0 bytes of the step's two blocks in bits 0..7 and 8..15
  auto scale_pair = [&](int set) -> uint32_t {
    if constexpr (FMT == E4B_FMT_MXFP4) {
      const auto r = __builtin_amdgcn_permlane32_swap(sq[set], sq[set], false, false);
      return r[0] | (r[1] << 8);
    }
    float scale;
    if constexpr (FMT == E4B_FMT_NF4) {
      scale = sa[set];
    } else {
      const float prod = code2_s[sq[set]] * sa[set];
      scale = prod + offset;
    }
    scale = __builtin_amdgcn_ldexpf(scale, wsh);
    return cvt_pair<E4B_FP16>(scale, scale);
  };
  auto store_a = [&](int buf, int i) {
    *reinterpret_cast<u32x4_t*>(&As[buf][lds_at_w(64 * i + (tid >> 3), 8 * apart)]) = areg[i];
  };
  // A loaded set's words exchanged between the lane halves: a half's words of groups 0, 2, 1, 3 end
  // up in x, y, z, w (the swap gives both lanes the lower lane's pair, then the upper lane's).
  auto arrange = [&](int set) {
    const auto a = __builtin_amdgcn_permlane32_swap(wq[set].x, wq[set].y, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(wq[set].z, wq[set].w, false, false);
    wq[set] = make_uint4(a[0], a[1], b[0], b[1]);
  };
  // Word j of an arranged set (K = 16 j + 8 half .. + 7 of the step) to the MFMA operand: its four
  // bytes' code pairs (lookup), then times the scale pair (scaled); e2m1 converts in scaled.
  const uint32_t copy_off = (lane & (kWide8Copies - 1)) * 4;
  auto lookup = [&](int set, int j, uint32_t (&o)[4]) {
    const uint32_t w = j == 0 ? wq[set].x : j == 1 ? wq[set].z : j == 2 ? wq[set].y : wq[set].w;
    if constexpr (FMT == E4B_FMT_MXFP4) {
      o[0] = w;
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        // byte b of w into address bits 8..15, the lane's copy into bits 0..7
        const uint32_t addr = __builtin_amdgcn_perm(w, copy_off, 0x0c0c0000u | (uint32_t(4 + b) << 8));
        o[b] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(ptab) + addr);
      }
    }
  };
  auto scaled = [&](const uint32_t (&o)[4], uint32_t sc, int j) -> uint4 {
    uint32_t v[4];
    if constexpr (FMT == E4B_FMT_MXFP4) {
      fp4_word<CT>(o[0], e8m0_to_f32(j < 2 ? sc & 0xffu : sc >> 8), v);
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b) v[b] = pk_mul_f16(o[b], sc);
    }
    return make_uint4(v[0], v[1], v[2], v[3]);
  };

  // activation fragment of MFMA group j, row block ms: row 32 ms + lane % 32, the group of columns
  // 16 j + 8 half .. + 7; the row's swizzle term is (l & 7) ^ ((l >> 3) & 3) ^ 4 (ms & 1)
  const int a_frag = c32 * kTileK;
  const int a_sw = (lane ^ (c32 >> 3)) & 7;
  auto frag = [&](int buf, int j, int ms) -> uint4 {
    const int fcol = ((2 * j + half) ^ a_sw) << 3;
    return *reinterpret_cast<const uint4*>(&As[buf][a_frag + ms * 32 * kTileK + (fcol ^ ((ms & 1) << 5))]);
  };

  const int64_t ksteps = k / kTileK;
  const int64_t klast = ksteps - 1;
#pragma unroll
  for (int i = 0; i < AP; ++i) load_a(i, 0);
  load_w(0, 0);
  load_w(1, min<int64_t>(1, klast));
  if (F16C && tid < BM) row_shift_s[tid] = exp_shift(a_exp_row);
  __syncthreads();  // code2 table, code-pair table, row shifts
  if constexpr (LORA) {
    // the accumulators start as the tile's LoRA delta, scaled like the products (lora_mfma.h): the rows' t
    // (clamped to the expert's rows: the rest is never stored) times their activation shifts, the B row
    // of the lane's column times the expert's weight shift. Activation buffer 1 is free until step 0,
    // one barrier further on
    lora_delta_32x32<BM, NT>(p, acc, e, row0, row_end - 1, row_shift_s, wsh, grow, As[1], lane);
  }
  // step 0's activations into buffer 0; their registers take step 1
#pragma unroll
  for (int i = 0; i < AP; ++i) {
    store_a(0, i);
    load_a(i, min<int64_t>(1, klast));
  }
  uint32_t raw[4];
  arrange(0);
  lookup(0, 0, raw);
  __syncthreads();

  // step kb (weight set u = kb % 2): MFMA group j in two chunks of MS / 2 row blocks, each chunk's
  // fragments read while the chunk before it multiplies (left to the compiler, a fragment was
  // read two MFMAs ahead and every pair of MFMAs waited for LDS). Step kb + 1's activation pieces
  // are stored into the other buffer ahead of the last chunk, each piece's registers taking step
  // kb + 2 at once, and the step's one barrier lies there too, so the last chunk covers the next
  // step's first fragment reads. The weight set takes step kb + 2 once its last word is looked up.
  // (Past the last step the loads re-read the last step and the stores fill a buffer no later
  // step reads.)
  constexpr int CH = MS / 2;
  uint4 fr[2][CH];
#pragma unroll
  for (int q = 0; q < CH; ++q) fr[0][q] = frag(0, 0, q);
  uint32_t sc = scale_pair(0);
  uint4 bv = scaled(raw, sc, 0);
  auto iteration = [&](auto uc, int64_t kb) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    constexpr int nset = u ^ 1;
    const int cur = static_cast<int>(kb & 1);
    static_for<8>([&](auto cc) {
      constexpr int c = decltype(cc)::value, j = c / 2, h = c % 2;
      if constexpr (c == 7) __syncthreads();
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        if constexpr (c < 7) fr[(c + 1) & 1][q] = frag(cur, (c + 1) / 2, ((c + 1) % 2) * CH + q);
        else fr[0][q] = frag(cur ^ 1, 0, q);
      }
      if constexpr (h == 0) {  // the next group's table lookups
        if constexpr (j < 3) {
          lookup(u, j + 1, raw);
        } else {
          arrange(nset);
          lookup(nset, 0, raw);
        }
      }
      static_for<CH>([&](auto q) {
        acc[h * CH + int(q)] = mfma_32x32x16<CT>(bv, fr[c & 1][int(q)], acc[h * CH + int(q)]);
      });
      if constexpr (c == 6) sc = scale_pair(nset);
      if constexpr (h == 1) bv = scaled(raw, sc, (j + 1) & 3);
      if constexpr (h == 0 && j < AP) {
        store_a(cur ^ 1, j);
        load_a(j, min<int64_t>(kb + 2, klast));
      }
      if constexpr (c == 5) load_w(u, min<int64_t>(kb + 2, klast));  // the set's last word is looked up
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS reads
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  const int64_t kmain = ksteps - ksteps % RS;
  for (int64_t kb0 = 0; kb0 < kmain; kb0 += RS) {
    iteration(std::integral_constant<int, 0>{}, kb0);
    iteration(std::integral_constant<int, 1>{}, kb0 + 1);
  }
  if (kmain < ksteps) iteration(std::integral_constant<int, 0>{}, kmain);

  // epilogue: the operand scales come off (2^-(row shift + expert shift), exact), then the
  // gated or plain store; the lane index is formed again here (v_mbcnt) so nothing from before
  // the loop stays live across it
  const int lane_e = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
  const int half_e = lane_e >> 5;
  auto unscale = [&](auto ms) {
    if constexpr (F16C || H16) {
      const int d = H16 ? -p.out_f16_shift : -(row_shift_s[32 * int(ms) + (lane_e & 31)] + wsh);
      static_for<16>([&](auto i) { acc[ms][int(i)] = __builtin_amdgcn_ldexpf(acc[ms][int(i)], d); });
    }
  };
  const bool has_bias = p.w.bias != nullptr;
  const uint16_t* bias = static_cast<const uint16_t*>(p.w.bias);
  // Eight 16-bit columns of the lane's row from two runs of four (v and the run eight columns on, each
  // packed into two words): after the swap a lane of the lower half holds the first run's eight
  // columns, one of the upper half the second's. col: the first run's first column.
  auto store8 = [&](uint16_t* row, int64_t col, uint32_t (&v)[2], uint32_t (&w)[2]) {
    const auto a = __builtin_amdgcn_permlane32_swap(v[0], w[0], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(v[1], w[1], false, false);
    // lower half: a[0], b[0] its own first run, a[1], b[1] the upper lane's first run; upper half:
    // the lower lane's second run, then its own
    *reinterpret_cast<uint4*>(row + col + 8 * half_e) = make_uint4(a[0], b[0], a[1], b[1]);
  };
  const bool vec = (p.n_out & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;  // whole 16-byte pieces
  // a run of four neighbouring bias values (zeros without one)
  auto bias4 = [&](int64_t at, float (&b)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = has_bias ? to_f<DT>(bias[int64_t(e) * n + at + i]) : 0.0f;
  };
  if (pair) {
    // output columns col0 + 16 w + 8 q + 4 (l / 32) + 0..3 (q = 0, 1) from accumulators 4 q + 0..3
    // (gate) and 8 + 4 q + 0..3 (up)
    const int64_t j0 = col0 + 16 * wid;
    if (!p.out_f32 && vec && j0 + 16 <= p.n_out) {  // whole runs to 16-bit rows: act(gate, up, i)
      auto rows = [&](auto&& act) {
        static_for<MS>([&](auto ms) {
          unscale(ms);
          uint32_t v[2][2];
          static_for<4>([&](auto q) {  // two columns each
            const int i = 2 * int(q);
            v[i / 4][(i / 2) & 1] =
                cvt_pair<DT>(act(acc[ms][i], acc[ms][8 + i], i), act(acc[ms][i + 1], acc[ms][9 + i], i + 1));
          });
          const int rr = row0 + 32 * int(ms) + (lane_e & 31);
          if (rr < row_end) store8(static_cast<uint16_t*>(p.out) + int64_t(rr) * p.n_out, j0, v[0], v[1]);
        });
      };
      if (p.epi == E4B_EPI_SWIGLU && !has_bias) {
        rows([&](float g, float u, int) { return silu_f32(g) * u; });
        return;
      }
      float bg[2][4], bu[2][4];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        bias4(j0 + 8 * q + 4 * half_e, bg[q]);
        bias4(n / 2 + j0 + 8 * q + 4 * half_e, bu[q]);
      }
      if (p.epi == E4B_EPI_GPTOSS)
        rows([&](float g, float u, int i) {
          return gated(E4B_EPI_GPTOSS, g, u, p.alpha, p.limit, bg[i >> 2][i & 3], bu[i >> 2][i & 3]);
        });
      else
        rows([&](float g, float u, int i) {
          return gated(p.epi, g, u, p.alpha, p.limit, bg[i >> 2][i & 3], bu[i >> 2][i & 3]);
        });
      return;
    }
    static_for<MS>([&](auto ms) {
      unscale(ms);
      const int rr = row0 + 32 * int(ms) + (lane_e & 31);
      static_for<8>([&](auto i) {
        const int64_t jj = j0 + 8 * (int(i) >> 2) + 4 * half_e + (int(i) & 3);
        if (rr < row_end && jj < p.n_out) {
          const float bg = has_bias ? to_f<DT>(bias[int64_t(e) * n + jj]) : 0.0f;
          const float bu = has_bias ? to_f<DT>(bias[int64_t(e) * n + n / 2 + jj]) : 0.0f;
          store_elem<DT>(p, int64_t(rr) * p.n_out + jj,
                         gated(p.epi, acc[ms][int(i)], acc[ms][8 + int(i)], p.alpha, p.limit, bg, bu));
        }
      });
    });
    return;
  }
  // columns col0 + 32 w + 8 q + 4 (l / 32) + 0..3 (q = 0..3) from accumulators 4 q + 0..3
  const int64_t c0 = col0 + 32 * wid;
  if (vec && c0 + 32 <= p.n_out && p.epi == E4B_EPI_NONE) {  // whole runs
    if (!H16 && p.out_f32) {  // fp32 rows
      float b[4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q) bias4(c0 + 8 * q + 4 * half_e, b[q]);
      static_for<MS>([&](auto ms) {
        unscale(ms);
        const int rr = row0 + 32 * int(ms) + (lane_e & 31);
        if (rr < row_end) {
          float* const row = static_cast<float*>(p.out) + int64_t(rr) * p.n_out + c0 + 4 * half_e;
          static_for<4>([&](auto q) {
            *reinterpret_cast<float4*>(row + 8 * int(q)) =
                make_float4(acc[ms][4 * int(q)] + b[q][0], acc[ms][4 * int(q) + 1] + b[q][1],
                            acc[ms][4 * int(q) + 2] + b[q][2], acc[ms][4 * int(q) + 3] + b[q][3]);
          });
        }
      });
      return;
    }
    if (H16 || !has_bias) {  // 16-bit rows; H16 (down): fp16, the operand scales left on (the host checks the form)
      static_for<MS>([&](auto ms) {
        unscale(ms);
        const int rr = row0 + 32 * int(ms) + (lane_e & 31);
        uint32_t v[4][2];
        static_for<8>([&](auto q) {
          v[int(q) / 2][int(q) & 1] = cvt_pair<H16 ? E4B_FP16 : DT>(acc[ms][2 * int(q)], acc[ms][2 * int(q) + 1]);
        });
        if (rr < row_end) {
          uint16_t* const row = static_cast<uint16_t*>(p.out) + int64_t(rr) * p.n_out;
          store8(row, c0, v[0], v[1]);
          store8(row, c0 + 16, v[2], v[3]);
        }
      });
      return;
    }
  }
  // general path
  static_for<MS>([&](auto ms) {
    unscale(ms);
    const int rr = row0 + 32 * int(ms) + (lane_e & 31);
    static_for<16>([&](auto i) {
      const int64_t nn = c0 + 8 * (int(i) >> 2) + 4 * half_e + (int(i) & 3);
      if (rr < row_end && nn < p.n_out) {
        if constexpr (H16) {
          static_cast<uint16_t*>(p.out)[int64_t(rr) * p.n_out + nn] = from_f<E4B_FP16>(acc[ms][int(i)]);
        } else {
          const float b = has_bias ? to_f<DT>(bias[int64_t(e) * n + nn]) : 0.0f;
          store_elem<DT>(p, int64_t(rr) * p.n_out + nn, single(p.epi, acc[ms][int(i)], b));
        }
      }
    });
  });
}

// H16: the down rows as fp16 with the operand scales left on (GemmArgs::out_f16_shift).
template <int DT, int FMT, bool F16C, bool LORA = false, bool H16 = false>
__global__ void __launch_bounds__(kWide8Threads) gemm_wide8_kernel(GemmArgs p) {
  static_assert(F16C ? (DT == E4B_BF16 && FMT != E4B_FMT_MXFP4) : (DT == E4B_BF16 && FMT == E4B_FMT_MXFP4),
                "fp16 mode with NF4 weights, or bf16 activations with MXFP4 weights");
  static_assert(!LORA || F16C, "the LoRA epilogue runs in the fp16 mode");
  static_assert(!H16 || (F16C && !LORA), "fp16 down rows: the fp16 mode without LoRA");
  constexpr int BM = kWideTileM, BN = kWideTileN;
  __shared__ __attribute__((aligned(16))) uint16_t As[2][BM * kTileK];
  __shared__ float code2_s[(FMT == E4B_FMT_NF4_DQ) ? 256 : 1];
  __shared__ __attribute__((aligned(16))) int row_shift_s[F16C ? BM : 4];
  __shared__ __attribute__((aligned(256))) uint32_t ptab[F16C ? 256 * kWide8TabStride : 1];
  const int cols = is_gated(p.epi) ? BN / 2 : BN;
  const int n_tiles = static_cast<int>((p.n_out + cols - 1) / cols);
  const TileItem item = tile_item(p.rt, n_tiles);
  if (!item.ok) return;
  const int n_tile = item.n_tile;
  Wide8Rows tr;
#pragma unroll
  for (int i = 0; i < 5; ++i) tr.sf[i] = 0;
  tr.e = item.e;
  tr.row0 = item.row0;
  tr.end = p.rt.offsets[item.e + 1];
  {
    const int mlast = static_cast<int>(p.M) - 1;
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < (F16C ? 5 : 0); ++i) {  // the fp16 mode (MXFP4 loads its sources in the tile)
      const int r = min(item.row0 + (i < 4 ? 64 * i + (tid >> 3) : (tid & (kWideTileM - 1))), mlast);
      const int v = p.rt.sorted_flat[r];
      tr.sf[i] = p.gather_k > 0 ? v : r;
    }
  }
  if constexpr (F16C) {
    // the table of code pairs: pass j fills entries 16 j .. 16 j + 15, thread t copy t % 32 of entry
    // 16 j + t / 32 (high nibble j, low nibble t / 32)
    static_assert(kWide8Threads == 16 * kWide8Copies, "table fill");
    const float lo = p.w.code[threadIdx.x / kWide8Copies];
    uint32_t* const fill = ptab + (threadIdx.x / kWide8Copies) * kWide8TabStride + threadIdx.x % kWide8Copies;
#pragma unroll
    for (int j = 0; j < 16; ++j) fill[16 * j * kWide8TabStride] = cvt_pair<E4B_FP16>(p.w.code[j], lo);
    if constexpr (FMT == E4B_FMT_NF4_DQ) {
      if (threadIdx.x < 256) code2_s[threadIdx.x] = p.w.code2[threadIdx.x];
    }
  }
  const int rows = tr.end - tr.row0;  // the tile's rows, capped at BM below
  if (rows <= BM / 2) wide8_tile<DT, FMT, F16C, true, LORA, H16>(p, tr, n_tile, As, code2_s, row_shift_s, ptab);
  else wide8_tile<DT, FMT, F16C, false, LORA, H16>(p, tr, n_tile, As, code2_s, row_shift_s, ptab);
}

}  // namespace e4b
