// Prefill grouped GEMM on 4-bit weights (int4 W4A16 and MXFP4): the nibbles
// stay 4-bit until they are in registers, so an expert's weights are read once
// per M-tile at a quarter of their bf16 size.
//
// One ring stage = 128 reduction elements: BM x 256 bytes of bf16 activations
// and 256 x 64 bytes of nibbles, with their scales (int4: also zeros and row
// sums).
//
// MXFP4: v_cvt_scalef32_pk_bf16_fp4 gives e2m1 x 2^e exactly in bf16, and the
// MFMAs go straight into the accumulators.  What bounds it (Mixtral M=33 GEMM1,
// 146 us at first): the scale bytes fetched per stage, a line per lane (110 us
// without them; now 16 bytes per row and four stages, 122), then the
// conversions (12 us).
//
// int4: the bf16 number with bits 0x4300 | q is 128 + q (exact), so a stage's
// MFMAs give t = sum((128 + q) x) per weight row and
// slot, and the group is folded in fp32 as
//   acc += scale * (t - (128 + zero) * xs),   xs = sum(x) over the group:
// the streaming kernels' arithmetic (no 16-bit rounding of the dequantized
// weight).  Extracting two nibbles per register gives elements 0 4 1 5 2 6 3 7
// of 8, so the activations come in that order: x through rows_for_int4_kernel
// (which also sums the groups), the intermediate straight from GEMM1's
// epilogue (whose 128 activation columns are one group).
// What bounds int4: the vector unit and the matrix cores in turn.  A wave's
// stage is 64 MFMAs (1024 cycles) and about 320 vector instructions (nibbles
// 112, scales 48, fold 128) of 4 cycles each, and the two waves of a SIMD hardly
// overlap one's MFMAs with the other's vector work.  Mixtral M=500 GEMM1 390
// us; without the fold's multiplications 330, without the unpacking as well
// 307, without the DMA too 267.  The streaming kernels, which read the weights
// again for every 32 slots: 434-498 us (call 720 -> 600 us, M=800 1152 -> 754).
#include <algorithm>
#include <type_traits>

#include "prefill.hpp"

namespace fmoe {
namespace prefill {

template <int BM_, int WAVES_M_, int WAVES_N_, int NBUF_, bool MX_, Mode MODE_>
struct W4Cfg {
  static constexpr int BM = BM_, BN = 256, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, NBUF = NBUF_;
  static constexpr bool MX = MX_;
  static constexpr Mode MODE = MODE_;
  static constexpr int NW = WAVES_M * WAVES_N, NT = NW * 64;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, MI = WM / 16, NI = WN / 16;
  // units of a stage: 4 per 16 activation rows (2 x 128 bytes per row, 8 rows
  // each), 1 per 16 weight rows
  static constexpr int A_UNITS = BM / 16 * 4, B_UNITS = BN / 16, UNITS = A_UNITS + B_UNITS;
  static constexpr int UPW = (UNITS + NW - 1) / NW;
  static constexpr int STAGE = UNITS * kUnit;
  // small loads of a stage, one wave each (the last waves).  int4: scales of
  // 128 weight rows (2), zeros (1), row sums of 64 slots; MXFP4: the four
  // scale bytes of 64 weight rows (4)
  static constexpr int AUX = MX ? BN / 64 : 3 + (BM + 63) / 64;
  // MXFP4 scale slots hold 16 bytes (four stages) per weight row
  static constexpr int AUX_LDS = MX ? 2 * BN * 16 : NBUF * (BN * 2 + BN / 2 + BM * 4);
  static_assert(!MX || NBUF <= 4, "two scale slots cover the ring");
  static_assert(UNITS % NW == 0, "every wave issues UPW units");
  static_assert(AUX <= NW, "one small load per wave");
  static_assert((MODE == Mode::kGemm1Silu ? NI / 2 : NI) % 2 == 0, "weight blocks in pairs");
  static_assert(NBUF * STAGE + AUX_LDS <= 160 * 1024, "LDS budget");
};

// x rows in the nibble order, and their group sums: one thread per 8 elements,
// 16 threads per 128-element group.
__global__ __launch_bounds__(256) void rows_for_int4_kernel(const uint16_t* __restrict__ x, int64_t n_vec,
                                                            uint16_t* __restrict__ xp, float* __restrict__ xs) {
  const int64_t v = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const bool live = v < n_vec;
  const i32x4_t raw = *reinterpret_cast<const i32x4_t*>(x + (live ? v : 0) * 8);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = static_cast<uint32_t>(raw[i]);
    s += __uint_as_float(w << 16) + __uint_as_float(w & 0xffff0000u);
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, kWave);
  if (!live) return;
  // elements (0, 4), (1, 5), (2, 6), (3, 7)
  const uint32_t a = raw[0], b = raw[1], c = raw[2], d = raw[3];
  *reinterpret_cast<uint4*>(xp + v * 8) = make_uint4((a & 0xffffu) | (c << 16), (a >> 16) | (c & 0xffff0000u),
                                                     (b & 0xffffu) | (d << 16), (b >> 16) | (d & 0xffff0000u));
  if (threadIdx.x % 16 == 0) xs[v / 16] = s;
}

template <class C, int ACT>
__global__ __launch_bounds__(C::NT) void gemm_w4_kernel(GemmParams p) {
  constexpr int BM = C::BM, BN = C::BN, WM = C::WM, WN = C::WN, MI = C::MI, NI = C::NI, NW = C::NW, NBUF = C::NBUF;
  constexpr Mode MODE = C::MODE;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NBUF][C::STAGE];
  // int4: fp16 scales, u4 zeros, row sums; MXFP4: scale bytes per weight row
  __shared__ __attribute__((aligned(256))) uint16_t sc_lds[NBUF][C::MX ? 1 : BN];
  __shared__ __attribute__((aligned(256))) uint32_t zr_lds[NBUF][C::MX ? 1 : BN / 8];
  __shared__ __attribute__((aligned(256))) float xs_lds[NBUF][C::MX ? 1 : BM];
  __shared__ __attribute__((aligned(256))) uint32_t mx_lds[C::MX ? 2 * BN * 4 : 1];

  const int tid = threadIdx.x, lane = tid % kWave, g = lane >> 4, r16 = lane & 15;
  const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wid / C::WAVES_N, wn = wid % C::WAVES_N;

  const int groups = static_cast<int>(p.Kred / 128);
  Work w;
  if (!locate<BM, MODE>(p, groups, lane, w)) return;
  const int e = w.e, nt = w.nt, row_beg = w.row_beg, row_end = w.row_end;
  const bool wave_live = C::WAVES_M == 1 || __builtin_amdgcn_readfirstlane(row_end - row_beg > wm * WM);
  const int per_k = (groups + w.n_splits - 1) / w.n_splits;
  const int k0 = min(groups, w.split * per_k);
  const int nk = min(groups, k0 + per_k) - k0;

  auto a_src_row = [&](int r) -> int64_t {
    int s = row_beg + r;
    if (s >= row_end) s = row_beg;  // padding row: any valid row, result discarded
    return MODE == Mode::kGemm1Silu ? p.topk_indx[s] / p.top_k : s;
  };
  // Weight row of tile column tc (0..255).  A tile past the last weight row
  // (Nout is a multiple of 128) repeats the 128 rows before it.
  auto w_row = [&](int tc) -> int64_t {
    if (MODE == Mode::kGemm1Silu) {
      const int s = tc / WN, within = tc % WN;
      const int64_t j = static_cast<int64_t>(nt) * (BN / 2) + s * (WN / 2) + within % (WN / 2);
      return gemm1_row(ACT, p.N_act, j, within < WN / 2 ? 0 : 1);
    }
    const int64_t row = static_cast<int64_t>(nt) * BN + tc;
    return row < p.Nout ? row : row - 128;
  };
  // ---- DMA sources: unit u = NW i + wid, activation units first
  const uint8_t* Be = p.B + static_cast<int64_t>(e) * p.Nout * (p.Kred / 2);
  const uint8_t* src[C::UPW];
  int step_bytes[C::UPW];  // from one stage to the next
#pragma unroll
  for (int i = 0; i < C::UPW; ++i) {
    const int u = NW * i + wid;
    if (u < C::A_UNITS) {
      // block u / 4, row half u % 2, 128-byte half (u / 2) % 2 of the group
      const int row = u / 4 * 16 + (u & 1) * 8 + (lane >> 3);
      src[i] = p.A + a_src_row(row) * (2 * p.Kred) + static_cast<int64_t>(k0) * 256 + (u >> 1 & 1) * 128 +
               ((lane & 7) ^ (lane >> 3)) * 16;
      step_bytes[i] = 256;
    } else if (p.b_tiled) {
      // lane 16 g + r: bytes 16 g .. of row r, as the tiled block stores them
      const int64_t row = w_row(tile_row<true>(u - C::A_UNITS, r16));
      src[i] = Be + ((row >> 4) * groups + k0) * 1024 + (16 * g + (row & 15)) * 16;
      step_bytes[i] = 1024;
    } else {
      // row-major: 4 lanes read a row's 64 bytes, chunks swizzled by row
      const int r = lane >> 2;
      const int64_t row = w_row(tile_row<true>(u - C::A_UNITS, r));
      src[i] = Be + (row * groups + k0) * 64 + ((lane & 3) ^ (r >> 1 & 3)) * 16;
      step_bytes[i] = 64;
    }
  }
  // the wave's small load, if it has one
  const int aux = NW - 1 - wid;
  const uint8_t* aux_src = nullptr;
  int64_t aux_step = 0;
  uint8_t* aux_dst = nullptr;
  int aux_slot = 0;
  bool aux_lane = aux < C::AUX;
  if constexpr (C::MX) {
    if (aux < C::AUX) {  // scale bytes of LDS weight rows 64 aux + lane
      const int row = 64 * aux + lane;
      aux_src = p.b_mxscale + (static_cast<int64_t>(e) * p.Nout + w_row(tile_row<true>(row / 16, row % 16))) * (4 * groups);
    }
  } else if (aux < 2) {  // scales of tile columns 128 aux + 2 lane, + 1
    const int tc = 128 * aux + 2 * lane;
    aux_src = reinterpret_cast<const uint8_t*>(p.b_gscale + (static_cast<int64_t>(e) * groups + k0) * p.Nout + w_row(tc));
    aux_step = 2 * p.Nout;
    aux_dst = reinterpret_cast<uint8_t*>(&sc_lds[0][128 * aux]);
    aux_slot = BN * 2;
  } else if (aux == 2) {  // zeros of tile columns 8 lane .. + 7
    const int tc = 8 * min(lane, BN / 8 - 1);
    aux_src = p.b_zero + ((static_cast<int64_t>(e) * groups + k0) * p.Nout + w_row(tc)) / 2;
    aux_step = p.Nout / 2;
    aux_dst = reinterpret_cast<uint8_t*>(&zr_lds[0][0]);
    aux_slot = BN / 2;
    aux_lane = lane < BN / 8;
  } else if (aux < C::AUX) {  // row sums of slots 64 (aux - 3) + lane
    const int r = 64 * (aux - 3) + lane;
    aux_src = reinterpret_cast<const uint8_t*>(p.a_scale + a_src_row(min(r, BM - 1)) * groups + k0);
    aux_step = 4;
    aux_dst = reinterpret_cast<uint8_t*>(&xs_lds[0][64 * (aux - 3)]);
    aux_slot = BM * 4;
    aux_lane = r < BM;
  }
  // MXFP4 scales: a load per row and stage touches a line per lane, so where
  // a row's scale bytes divide into 16-byte pieces they come for four stages
  // at once (Mixtral M=33 GEMM1 146 -> 110 us without the per-stage loads)
  const bool mx_quads = groups % 4 == 0;
  // loads per stage that every wait may count on (the scale loads of four
  // stages come on top: a wait that sees one waits for that one too)
  const int per = C::UPW + (aux < C::AUX && !(C::MX && mx_quads) ? 1 : 0);
  auto issue_unit = [&](int kt, int i) {
    dma16(src[i] + static_cast<int64_t>(kt) * step_bytes[i], lds[kt % NBUF] + (NW * i + wid) * kUnit);
  };
  auto issue_aux = [&](int kt) {
    if constexpr (C::MX) {
      if (aux >= C::AUX) return;
      const int k = k0 + kt;
      if (!mx_quads)
        dma4(reinterpret_cast<const float*>(aux_src + 4 * k), reinterpret_cast<float*>(&mx_lds[(kt % NBUF) * BN + 64 * aux]));
      else if (kt == 0 || k % 4 == 0)
        dma16(aux_src + 16 * (k / 4), reinterpret_cast<uint8_t*>(&mx_lds[(k / 4 % 2) * (4 * BN) + 256 * aux]));
      return;
    }
    if (aux < C::AUX)
      if (aux_lane)
        dma4(reinterpret_cast<const float*>(aux_src + kt * aux_step),
             reinterpret_cast<float*>(aux_dst + (kt % NBUF) * aux_slot));
  };
  auto issue = [&](int kt) {
#pragma unroll
    for (int i = 0; i < C::UPW; ++i) issue_unit(kt, i);
    issue_aux(kt);
  };
  auto wait_full = [&](auto newer) {
    constexpr int N = decltype(newer)::value;
    wait_loads<N * (C::UPW + 1)>(N * per);
    barrier_nofence();
  };
  auto wait_stage = [&](int newer) {
    wait_loads<(NBUF - 1) * (C::UPW + 1)>(newer * per);
    barrier_nofence();
  };
  using Ring2 = std::integral_constant<int, NBUF - 2>;
  using T = std::true_type;
  using F = std::false_type;

  f32x4_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // MFMA step s (0..3) of a group takes elements 32 g + 8 s .. + 7 from lane
  // group g in both operands: 16-byte chunk 4 g + s of the row's 256 bytes,
  // dword s of the lane's 16 bytes of nibbles.
  int fo[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) fo[s] = (g >> 1) * 2048 + frag_off(lane, 4 * (g & 1) + s);
  const int bo = p.b_tiled ? 16 * lane : 16 * (4 * r16 + (g ^ (r16 >> 1 & 3)));
  bf16x8_t fa[2][MI];
  i32x4_t bq[NI];
  uint32_t mx[NI];  // MXFP4: the scale bytes of the lane's row of each block
  auto read_a = [&](int slot, int s, int q) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      fa[q][i] = __builtin_bit_cast(bf16x8_t, lds16(lds[slot] + (wm * MI + i) * 4 * kUnit + fo[s]));
  };
  auto read_b = [&](int kt) {
    const int slot = kt % NBUF;
#pragma unroll
    for (int j = 0; j < NI; ++j) bq[j] = lds16(lds[slot] + (C::A_UNITS + wn * NI + j) * kUnit + bo);
    if constexpr (C::MX) {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int row = (wn * NI + j) * 16 + r16, k = k0 + kt;
        mx[j] = mx_lds[mx_quads ? (k / 4 % 2) * (4 * BN) + 4 * row + k % 4 : slot * BN + row];
      }
    }
  };
  // the two constants in registers, so that and + or are one v_and_or_b32
  uint32_t nib_mask, nib_one, nib_f32;
  asm volatile("v_mov_b32 %0, 0x000f000f" : "=v"(nib_mask));
  asm volatile("v_mov_b32 %0, 0x43004300" : "=v"(nib_one));
  asm volatile("v_mov_b32 %0, 0x43000000" : "=v"(nib_f32));
  auto unpack = [&](int j, int s) {
    const uint32_t v = static_cast<uint32_t>(bq[j][s]);
    i32x4_t o;
#pragma unroll
    for (int h = 0; h < 4; ++h) o[h] = static_cast<int>(((v >> (4 * h)) & nib_mask) | nib_one);
    return __builtin_bit_cast(bf16x8_t, o);
  };

#pragma unroll
  for (int s = 0; s < NBUF; ++s)
    if (s < nk) issue(s);
  wait_stage(min(NBUF - 1, nk - 1));
  if (!wave_live) {
    int kt = 0;
    for (; kt + NBUF < nk; ++kt) {
      wait_full(Ring2{});
      issue(kt + NBUF);
    }
    for (; kt + 1 < nk; ++kt) wait_stage(min(NBUF - 2, nk - 2 - kt));
  } else if (nk > 0) {
    read_a(0, 0, 0);
    read_b(0);
    // One stage: the fragments of step s + 1 are read during step s; before
    // the last step the slot's reads are over, and one wait and one barrier
    // publish the next stage and free the slot (as gemm_prefill_kernel).
    // MXFP4: e2m1 -> bf16 with the block's scale folded in (exact), straight
    // into the accumulators
    auto stage_mx = [&](int kt, auto more, auto dma) {
      constexpr bool MORE = decltype(more)::value, DMA = decltype(dma)::value;
      const int slot = kt % NBUF, next = (kt + 1) % NBUF;
      float sc[NI];  // the lane's 32 elements of the group are scale block g
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const uint32_t ex = __builtin_amdgcn_ubfe(mx[j], 8 * g, 8);
        sc[j] = ex == 0 ? 0x1p-127f : (ex == 255 ? __builtin_nanf("") : __uint_as_float(ex << 23));
      }
      auto cvt = [&](int j, int s) {
        const uint32_t v = static_cast<uint32_t>(bq[j][s]);
        i32x4_t o;
        o[0] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc[j], 0));
        o[1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc[j], 1));
        o[2] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc[j], 2));
        o[3] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc[j], 3));
        return __builtin_bit_cast(bf16x8_t, o);
      };
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        read_a(slot, s + 1, (s + 1) & 1);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const bf16x8_t fb = cvt(j, s);
#pragma unroll
          for (int i = 0; i < MI; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb, fa[s & 1][i], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      bf16x8_t fb[NI];
#pragma unroll
      for (int j = 0; j < NI; ++j) fb[j] = cvt(j, 3);
      if constexpr (MORE) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads have left the slot
        if constexpr (DMA)
          wait_full(Ring2{});
        else
          wait_stage(min(NBUF - 2, nk - 2 - kt));
        read_a(next, 0, 0);
        read_b(kt + 1);
      }
      if constexpr (DMA) issue_aux(kt + NBUF);
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (DMA) {
#pragma unroll
          for (int u = 0; u < C::UPW; ++u)
            if (u * NI / C::UPW == j) issue_unit(kt + NBUF, u);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[1][i], acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto stage_int4 = [&](int kt, auto more, auto dma) {
      constexpr bool MORE = decltype(more)::value, DMA = decltype(dma)::value;
      const int slot = kt % NBUF, next = (kt + 1) % NBUF;
      f32x4_t t[MI][NI];
      i32x4_t sc[NI / 2];  // 8 fp16 scales of a block pair's 8 columns
      uint32_t zr[NI / 2];
      float xs[MI];
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        read_a(slot, s + 1, (s + 1) & 1);
        if (s == 2) {
#pragma unroll
          for (int h = 0; h < NI / 2; ++h) {
            const int tc = wn * WN + h * 32 + g * 8;
            sc[h] = *reinterpret_cast<const i32x4_t*>(&sc_lds[slot][tc]);
            zr[h] = zr_lds[slot][tc / 8];
          }
#pragma unroll
          for (int i = 0; i < MI; ++i) xs[i] = xs_lds[slot][wm * WM + i * 16 + r16];
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const bf16x8_t fb = unpack(j, s);
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const f32x4_t c = s == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : t[i][j];
            t[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb, fa[s & 1][i], c, 0, 0, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      bf16x8_t fb[NI];
#pragma unroll
      for (int j = 0; j < NI; ++j) fb[j] = unpack(j, 3);
      if constexpr (MORE) {
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the reads have left the slot
        if constexpr (DMA)
          wait_full(Ring2{});
        else
          wait_stage(min(NBUF - 2, nk - 2 - kt));
        read_a(next, 0, 0);
        read_b(kt + 1);
      }
      if constexpr (DMA) issue_aux(kt + NBUF);
      // the last step's products of block column j, then the fold of column j - 1
#pragma unroll
      for (int j = 0; j <= NI; ++j) {
        __builtin_amdgcn_sched_barrier(0);
        if (j < NI) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
            t[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[1][i], t[i][j], 0, 0, 0);
        }
        if constexpr (DMA) {
#pragma unroll
          for (int u = 0; u < C::UPW; ++u)
            if (u * NI / C::UPW == j) issue_unit(kt + NBUF, u);
        }
        if (j == 0) continue;
        float sv[4], zv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = ((j - 1) & 1) * 4 + r;
          const uint32_t hw = static_cast<uint32_t>(sc[(j - 1) / 2][c / 2]);
          sv[r] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(c & 1 ? hw >> 16 : hw)));
          asm("" : "+v"(sv[r]));  // one conversion, then plain fp32 FMAs
          // 128 + zero, from the nibble as the weights are
          zv[r] = __uint_as_float(__builtin_amdgcn_ubfe(zr[(j - 1) / 2], 4 * c, 4) << 16 | nib_f32);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][j - 1][r] = __builtin_fmaf(sv[r], __builtin_fmaf(-zv[r], xs[i], t[i][j - 1][r]), acc[i][j - 1][r]);
      }
    };
    auto stage = [&](int kt, auto more, auto dma) {
      if constexpr (C::MX)
        stage_mx(kt, more, dma);
      else
        stage_int4(kt, more, dma);
    };
    int kt = 0;
    for (; kt + NBUF < nk; ++kt) stage(kt, T{}, T{});
    for (; kt + 1 < nk; ++kt) stage(kt, T{}, F{});
    stage(kt, F{}, F{});
  }

  // ---- epilogue: the lane holds slot row lane % 16 of each 16-row block i and
  // columns 8 g .. + 7 of each pair of weight blocks.  Routing weights first
  // (no load may sit between the stores: their counter is shared).
  float gv[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int s = row_beg + wm * WM + i * 16 + r16;
    gv[i] = (p.gamma && s < row_end) ? p.gate_scal[s] : 1.0f;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) asm volatile("" ::"v"(gv[i]));
  if constexpr (MODE == Mode::kGemm1Silu && C::MX) {
    uint16_t* act = static_cast<uint16_t*>(p.out);
    const int64_t c0 = static_cast<int64_t>(nt) * (BN / 2) + wn * (WN / 2);
    float gb[NI / 2][4], ub[NI / 2][4];
#pragma unroll
    for (int j = 0; j < NI / 2; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        gemm1_bias<ACT>(p, e, c0 + tile_col<true>(j, lane) + c, gb[j][c], ub[j][c]);
        asm volatile("" ::"v"(gb[j][c]), "v"(ub[j][c]));
      }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int s = row_beg + wm * WM + i * 16 + r16;
      if (s >= row_end) continue;
#pragma unroll
      for (int j = 0; j < NI / 2; j += 2) {
        uint4 o;
        uint32_t* ow = reinterpret_cast<uint32_t*>(&o);
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          float a[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int jj = j + h / 2, c = 2 * (h % 2) + u;
            a[u] = gemm1_act<ACT>(p, acc[i][jj][c], acc[i][jj + NI / 2][c], gb[jj][c], ub[jj][c], gv[i]);
          }
          ow[h] = pack_bf16x2(a[0], a[1]);
        }
        *reinterpret_cast<uint4*>(act + static_cast<int64_t>(s) * p.N_act + c0 + tile_col<true>(j, lane)) = o;
      }
    }
  } else if constexpr (MODE == Mode::kGemm1Silu) {
    // bf16 activations in the nibble order, and their group sums (of the
    // rounded values): lane, the row's 4 lanes, then the waves through LDS
    __syncthreads();
    float* part = reinterpret_cast<float*>(&lds[0][0]);  // [BM][WAVES_N]
    uint16_t* act = static_cast<uint16_t*>(p.out);
    const int64_t c0 = static_cast<int64_t>(nt) * (BN / 2) + wn * (WN / 2);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int s = row_beg + wm * WM + i * 16 + r16;
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < NI / 2; j += 2) {
        float a[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
          a[c] = gemm1_act<ACT>(p, acc[i][j + c / 4][c % 4], acc[i][j + c / 4 + NI / 2][c % 4], 0.f, 0.f, gv[i]);
        uint4 o;
        uint32_t* ow = reinterpret_cast<uint32_t*>(&o);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t v = pack_bf16x2(a[c], a[c + 4]);
          ow[c] = v;
          sum += __uint_as_float(v << 16) + __uint_as_float(v & 0xffff0000u);
        }
        if (s < row_end)
          *reinterpret_cast<uint4*>(act + static_cast<int64_t>(s) * p.N_act + c0 + tile_col<true>(j, lane)) = o;
      }
      sum += __shfl_xor(sum, 16, kWave);
      sum += __shfl_xor(sum, 32, kWave);
      if (lane < 16) part[(wm * WM + i * 16 + r16) * C::WAVES_N + wn] = sum;
    }
    __syncthreads();
    if (tid < BM && row_beg + tid < row_end) {
      float sum = 0.f;
#pragma unroll
      for (int q = 0; q < C::WAVES_N; ++q) sum += part[tid * C::WAVES_N + q];
      p.act_qs[static_cast<int64_t>(row_beg + tid) * (p.N_act / 128) + nt] = sum;
    }
  } else {
    const int64_t c0 = static_cast<int64_t>(nt) * BN + wn * WN;
    float bv[NI][4] = {};
    if (p.bias && w.split == 0) {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int64_t col = c0 + tile_col<true>(j, lane);
        if (col < p.Nout)
#pragma unroll
          for (int c = 0; c < 4; ++c) bv[j][c] = p.bias[static_cast<int64_t>(e) * p.Nout + col + c];
      }
    }
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) asm volatile("" ::"v"(bv[j][c]));
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = wm * WM + i * 16 + r16, s = row_beg + row;
      if (s >= row_end) continue;
      float* y = w.tail >= 0 ? p.tail_part + static_cast<int64_t>(w.tail) * (BM * BN) + row * BN -
                                   static_cast<int64_t>(nt) * BN
                             : static_cast<float*>(p.out) + w.split * p.out_split_stride +
                                   static_cast<int64_t>(s) * p.Nout;
#pragma unroll
      for (int j = 0; j < NI; j += 2) {
        const int64_t col = c0 + tile_col<true>(j, lane);
        if (col >= p.Nout) continue;
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = (acc[i][j + c / 4][c % 4] + bv[j + c / 4][c % 4]) * gv[i];
        *reinterpret_cast<float4*>(y + col) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(y + col + 4) = make_float4(v[4], v[5], v[6], v[7]);
      }
    }
  }
}

}  // namespace prefill

// 128-row tiles, 2x4 waves, 3-deep ring of 48 KiB stages.
int launch_w4(Mode mode, const GemmParams& p, hipStream_t s) {
  using namespace prefill;
  using C1 = W4Cfg<128, 2, 4, 3, false, Mode::kGemm1Silu>;
  using C2 = W4Cfg<128, 2, 4, 3, false, Mode::kGemm2>;
  const int groups = static_cast<int>(p.Kred / 128);
  if (mode == Mode::kGemm2) return launch_tiles<C2>(p, s, groups, gemm_w4_kernel<C2, kActSilu>);
  return launch_tiles<C1>(p, s, groups, p.act == kActGelu ? gemm_w4_kernel<C1, kActGelu> : gemm_w4_kernel<C1, kActSilu>);
}

// MXFP4: 128 rows as int4; 64 and 32 rows with 2- and 3-deep rings, two
// workgroups per CU (72 and 80 KiB of LDS).  Mixtral, 32 rows, 2x4 / 1x4 waves:
// M=33 200 / 209 us a call; a 4-deep ring (one workgroup per CU) 224; 64 rows,
// 2-deep / 4-deep: M=100 230 / 287.
int launch_mx(Mode mode, int bm, const GemmParams& p, hipStream_t s) {
  using namespace prefill;
  const int groups = static_cast<int>(p.Kred / 128);
#define G1(BM, WMS, WNS, NB, ACT) gemm_w4_kernel<W4Cfg<BM, WMS, WNS, NB, true, Mode::kGemm1Silu>, ACT>
#define L(BM, WMS, WNS, NB)                                                                                  \
  (mode == Mode::kGemm2                                                                                      \
       ? launch_tiles<W4Cfg<BM, WMS, WNS, NB, true, Mode::kGemm2>>(                                          \
             p, s, groups, gemm_w4_kernel<W4Cfg<BM, WMS, WNS, NB, true, Mode::kGemm2>, kActSilu>)            \
       : launch_tiles<W4Cfg<BM, WMS, WNS, NB, true, Mode::kGemm1Silu>>(                                      \
             p, s, groups, p.act == kActSwiglu ? G1(BM, WMS, WNS, NB, kActSwiglu)                            \
                                               : (p.act == kActGelu ? G1(BM, WMS, WNS, NB, kActGelu)         \
                                                                    : G1(BM, WMS, WNS, NB, kActSilu))))
  if (bm == 128) return L(128, 2, 4, 3);
  if (bm == 64) return L(64, 2, 4, 2);
  if (bm == 32) return L(32, 2, 4, 3);
#undef L
#undef G1
  return fmoe_host::fail(FMOE_ERR_UNSUPPORTED, "mxfp4 prefill: block_m=%d is not supported", bm);
}

size_t w4_tail_bytes(int64_t max_tiles, int64_t Nout) {
  using C = prefill::W4Cfg<128, 2, 4, 3, false, Mode::kGemm2>;
  return static_cast<size_t>(prefill::tail_pairs_for<C>(prefill::gemm_w4_kernel<C, kActSilu>, max_tiles, Nout)) *
         C::BM * C::BN * 4;
}

// x [M, K] -> the nibble order and group sums of the int4 prefill kernels
int rows_for_int4(const void* x, int64_t M, int64_t K, void* xp, float* xs, hipStream_t s) {
  const int64_t n_vec = M * K / 8;
  prefill::rows_for_int4_kernel<<<dim3(static_cast<unsigned>((n_vec + 255) / 256)), dim3(256), 0, s>>>(
      static_cast<const uint16_t*>(x), n_vec, static_cast<uint16_t*>(xp), xs);
  return fmoe_host::check_launch("rows_for_int4");
}

}  // namespace fmoe
