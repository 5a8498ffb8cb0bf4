// Prefill grouped GEMM: one expert per M-tile; MFMA tiles fed from a ring of
// LDS stages filled by direct-to-LDS DMA.
//
// Workgroup = 4 or 8 waves laid out WAVES_M x WAVES_N; tile BM x BN; SB = 128
// bytes of the reduction dim per row per stage (bf16: two
// v_mfma_f32_16x16x32_bf16 steps; fp8: one 128-wide scale block, one
// v_mfma_f32_16x16x128_f8f6f4 with its result scaled by a_scale[row] *
// w_scale[block] into the fp32 accumulator).
//
// Measured on MI355X, which is what the structure follows:
//  * DMA: global_load_lds_dwordx4 delivers ~2x the bytes per clock when
//    consecutive lanes read one row's contiguous bytes (8 lanes x 16 B)
//    than when every lane reads a different row.  LDS: a ds_read_b128
//    fragment read runs at full rate only if each 8 consecutive lanes hit 8
//    distinct 16-byte columns of a 128-byte window.  A stage is therefore a
//    set of 1 KiB units in row-major, XOR-swizzled layouts (see frag_off):
//    one unit is one wave-instruction of DMA, written without staging
//    registers or ds_write, and every fragment read is conflict-free.
//  * With the DMA running, operand delivery (not LDS or MFMA issue) bounds
//    the kernel, so the tile is as large as LDS allows (256 x 256 for bf16:
//    128 flop per byte moved) and two or three stages are kept in flight.
// Lane group g = L/16 sees reduction bytes 16g..16g+15 of each 64-byte half in
// both operands, so the MFMA dot products are exact permutations of the
// textbook ones.
//
// The DMA is issued from inline asm (M0 = LDS destination): the compiler then
// does not treat the LDS ring as written by an outstanding vector-memory op
// (it would insert vmcnt(0) before every fragment read).  Completion is
// ordered explicitly: per-wave vmcnt wait for the stage, then s_barrier
// without a fence (later stages keep streaming across it).
//
// GEMM1 (gate/up + SiLU): each wave's BN/WAVES_N weight rows are half gate rows
// and the matching up rows, so gate block j and up block j sit in the same
// lanes; silu(gate) * up is formed in registers and only the bf16 activation
// is written.  GEMM2: rows scaled by the routing weight; each slot row is
// stored as bf16 (one split), as fp32 split-K planes (stage-level calls), or,
// for the tail tiles of the fused path's tail split, as fp32 parts that
// tail_fold_kernel adds; the top-k sum runs in its own fixed-order launch
// (deterministic).
#include <algorithm>
#include <type_traits>

#include "prefill.hpp"

namespace fmoe {
namespace prefill {

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_, int NBUF_, bool FP8_, Mode MODE_>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, SB = 128,
                       NBUF = NBUF_;
  static constexpr bool FP8 = FP8_;
  static constexpr Mode MODE = MODE_;
  static constexpr int NW = WAVES_M * WAVES_N, NT = NW * 64;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int MI = WM / 16, NI = WN / 16;
  static constexpr int UPB = SB / 64;                       // units per 16-row block
  static constexpr int A_UNITS = (BM / 16) * UPB, B_UNITS = (BN / 16) * UPB;
  // unit u of a stage is DMAed by wave u % NW: waves below REM (or all of
  // them when REM == 0) issue UPW units per stage, the others UPW - 1
  static constexpr int UNITS = A_UNITS + B_UNITS;
  static constexpr int UPW = (UNITS + NW - 1) / NW;
  static constexpr int REM = UNITS % NW;
  static constexpr int STAGE = UNITS * kUnit;
  // waves that DMA the activation scales (64 rows each): the last SA_WAVES
  // waves, which carry the fewer units when the split is uneven
  static constexpr int SA_WAVES = FP8 ? (BM + 63) / 64 : 0;
  static constexpr int SA_FIRST = NW - SA_WAVES;
  // 16-row weight blocks taken in pairs (see tile_col): a lane's results of a
  // pair are 8 consecutive output columns
  static constexpr bool PAIR = (MODE == Mode::kGemm1Silu ? NI / 2 : NI) % 2 == 0;
  // fp8 weight-scale stages held in LDS (the reduction dim is at most 128 KST)
  static constexpr int KST =
      NBUF * STAGE + NBUF * BM * 4 + WAVES_N * 2 * kMaxKStages * 4 <= 160 * 1024 ? kMaxKStages : 64;
  static_assert(BM % 16 == 0 && (A_UNITS % 2) == 0, "16-row blocks");
  static_assert(REM == 0 || REM <= SA_FIRST || !FP8, "a-scale waves carry the fewer units");
  static_assert(MODE != Mode::kGemm1Silu || NI % 2 == 0, "gate/up pairing needs even NI");
  static_assert(NBUF >= 2 && NBUF <= 4, "ring depth");
  static_assert(NBUF * STAGE + NBUF * BM * 4 + WAVES_N * 2 * KST * 4 <= 160 * 1024, "LDS budget");
  static_assert(SA_WAVES <= NW, "a-scale waves");
};

template <class C, int ACT>
__global__ __launch_bounds__(C::NT) void gemm_prefill_kernel(GemmParams p) {
  constexpr int BM = C::BM, BN = C::BN, WM = C::WM, WN = C::WN, MI = C::MI, NI = C::NI;
  constexpr int SB = C::SB, UPB = C::UPB, NW = C::NW, NBUF = C::NBUF;
  constexpr bool FP8 = C::FP8;
  constexpr Mode MODE = C::MODE;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NBUF][C::STAGE];
  __shared__ __attribute__((aligned(256))) float sa_lds[NBUF][FP8 ? BM : 1];
  __shared__ float sb_lds[C::WAVES_N][2][FP8 ? C::KST : 1];

  const int tid = threadIdx.x, lane = tid % kWave;
  const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wid / C::WAVES_N, wn = wid % C::WAVES_N;

  // ---- which (split, expert M-tile, N-tile): workgroup ids are made
  // XCD-contiguous, then mapped by tile_of (or its precomputed table).
  const int64_t kbytes = FP8 ? p.Kred : p.Kred * 2;  // bytes per operand row
  const int nk_all = static_cast<int>(kbytes / SB);
  Work w;
  if (!locate<BM, MODE>(p, nk_all, lane, w)) return;
  const int split = w.split, n_splits = w.n_splits, tail = w.tail;
  const int e = w.e, nt = w.nt, row_beg = w.row_beg, row_end = w.row_end;

  // An expert's last M-tile is often nearly empty (Mixtral M=4096: ~1024 +- 30
  // slots per expert, so about half the experts add a fifth 256-row tile of a
  // few dozen rows; Qwen3 M=8192: a fifth of all tile rows are padding).
  // Waves whose rows are all padding skip their fragment reads and MFMAs, and
  // bf16 tiles do not fetch the DMA units of padding rows (their LDS rows hold
  // whatever was there; a slot row's results depend on its own operand row
  // only).  fp8 GEMM1 does neither (its 160-row tiles are mostly full: DSV3
  // M=4096 +3% with both).
  const bool wave_live = C::WAVES_M == 1 || (FP8 && MODE == Mode::kGemm1Silu) ||
                         __builtin_amdgcn_readfirstlane(row_end - row_beg > wm * WM);

  const int ksb = static_cast<int>(p.Kred / 128);      // fp8 scale blocks per row
  // split-K: this workgroup reduces stages [k0, k0 + nk)
  const int per_k = (nk_all + n_splits - 1) / n_splits;
  const int k0 = min(nk_all, split * per_k);
  const int nk = min(nk_all, k0 + per_k) - k0;

  auto a_src_row = [&](int r) -> int64_t {
    int s = row_beg + r;
    if (s >= row_end) s = row_beg;  // padding row: any valid row, result discarded
    return MODE == Mode::kGemm1Silu ? p.topk_indx[s] / p.top_k : s;
  };
  // ---- DMA sources: unit u = NW i + wid of the stage (A units first, then
  // B units) in the layout of frag_off.
  const uint8_t* Be = p.B + static_cast<int64_t>(e) * p.Nout * kbytes;
  const uint8_t* src[C::UPW];
  int loff[C::UPW];
  // the units this wave issues: UPW or UPW - 1, less those of padding rows
  uint32_t units = C::REM == 0 || wid < C::REM ? (1u << C::UPW) - 1 : (1u << (C::UPW - 1)) - 1;
  if constexpr (!FP8) {
#pragma unroll
    for (int i = 0; i < C::UPW; ++i) {
      const int u = NW * i + wid;
      if (u < C::A_UNITS && u * (16 / UPB) >= row_end - row_beg) units &= ~(1u << i);
    }
  }
  units = __builtin_amdgcn_readfirstlane(units);
#pragma unroll
  for (int i = 0; i < C::UPW; ++i) {
    const int u = min(NW * i + wid, C::UNITS - 1);
    const int b = u / UPB;
    const int ru = lane >> 3;
    const int lr = (u % 2) * 8 + ru;               // row within the 16-row block
    const int coff = ((lane & 7) ^ ru) * 16;       // byte offset in the row slice
    loff[i] = u * kUnit;
    if (u < C::A_UNITS) {
      src[i] = p.A + a_src_row(b * 16 + lr) * kbytes + static_cast<int64_t>(k0) * SB + coff;
    } else {
      const int r = tile_row<C::PAIR>(b - BM / 16, lr);  // row of the B tile
      int64_t brow;
      if (MODE == Mode::kGemm1Silu) {
        const int w = r / WN, within = r % WN;
        int64_t j = static_cast<int64_t>(nt) * (BN / 2) + w * (WN / 2) + (within % (WN / 2));
        if (j >= p.N_act) j = p.N_act - 1;  // past the last column (BN / 2 need not divide N)
        brow = gemm1_row(ACT, p.N_act, j, within < WN / 2 ? 0 : 1);
      } else {
        brow = static_cast<int64_t>(nt) * BN + r;
        if (brow >= p.Nout) brow = p.Nout - 1;
      }
      src[i] = Be + brow * kbytes + static_cast<int64_t>(k0) * SB + coff;
    }
  }
  // fp8: waves SA_FIRST + j DMA the activation scales of rows 64 j + lane
  // (lanes past BM stay idle)
  const int sa_j = wid - C::SA_FIRST;
  const bool sa_wave = FP8 && sa_j >= 0;
  const bool sa_lane = sa_wave && 64 * sa_j + lane < BM;
  const float* sa_src = nullptr;
  if (sa_wave) sa_src = p.a_scale + a_src_row(min(64 * sa_j + lane, BM - 1)) * ksb + k0;
  int sb_split = NI;  // GEMM2: 16-row blocks of the wave under its first weight-scale block
  // unit i of stage kt
  auto issue_unit = [&](int kt, int i) {
    if ((FP8 && i + 1 < C::UPW) || (units >> i & 1)) dma16(src[i] + static_cast<int64_t>(kt) * SB, lds[kt % NBUF] + loff[i]);
  };
  auto issue = [&](int kt) {
#pragma unroll
    for (int i = 0; i < C::UPW; ++i) issue_unit(kt, i);
    if (sa_wave) {
      if (64 * (sa_j + 1) <= BM) {
        dma4(sa_src + kt, &sa_lds[kt % NBUF][64 * sa_j]);
      } else if (sa_lane) {  // partial last 64-row group: masked lanes write nothing
        dma4(sa_src + kt, &sa_lds[kt % NBUF][64 * sa_j]);
      }
    }
  };

  f32x4_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // per-lane fragment offsets within a 16-row block's units
  const int foff0 = frag_off(lane, lane >> 4);
  const int foff1 = frag_off(lane, 4 + (lane >> 4));
  // DMA instructions per stage for this wave: its operand units, plus one
  // a-scale load
  const int per = __builtin_popcount(units) + (sa_wave ? 1 : 0);
  // this wave's part of a stage has landed once at most `newer` younger stages
  // are in flight; the whole stage after the barrier
  auto wait_full = [&](auto newer) {  // a full ring: a constant count first
    constexpr int N = decltype(newer)::value;
    wait_loads<N * (C::UPW + (FP8 ? 1 : 0))>(N * per);
    barrier_nofence();
  };
  auto wait_stage = [&](int newer) {
    wait_loads<(NBUF - 1) * (C::UPW + (FP8 ? 1 : 0))>(newer * per);
    barrier_nofence();
  };
  using Ring2 = std::integral_constant<int, NBUF - 2>;

  if constexpr (FP8) {
    // ring: up to NBUF-2 stages newer than kt stay in flight while kt is consumed
#pragma unroll
    for (int s = 0; s < NBUF - 1; ++s)
      if (s < nk) issue(s);
    // weight scales of the whole k range, staged once in LDS -- after the
    // first stages' DMA is issued, so the two round trips overlap
    const int64_t nrb = p.Nout / 128;
    const float* se = p.b_scale + static_cast<int64_t>(e) * nrb * ksb;
    const float* s0;
    const float* s1;
    if (MODE == Mode::kGemm1Silu) {
      // the wave's gate rows (and up rows) lie in one 128-row scale block
      const int64_t j = static_cast<int64_t>(nt) * (BN / 2) + wn * (WN / 2);
      s0 = se + (gemm1_row(ACT, p.N_act, j, 0) / 128) * ksb;
      s1 = se + (gemm1_row(ACT, p.N_act, j, 1) / 128) * ksb;
    } else {
      // the wave's rows span at most two 128-row scale blocks (WN <= 128):
      // 16-row blocks j < sb_split use the first one
      int64_t j = static_cast<int64_t>(nt) * BN + wn * WN;
      if (j >= p.Nout) j = p.Nout - 1;
      const int64_t jl = min(j + WN - 1, p.Nout - 1);
      s0 = se + (j / 128) * ksb;
      s1 = se + (jl / 128) * ksb;
      if (jl / 128 != j / 128) sb_split = static_cast<int>((128 - j % 128) / 16);
    }
    if (wm == 0)
      for (int kk = lane; kk < nk; kk += kWave) {
        sb_lds[wn][0][kk] = s0[k0 + kk];
        sb_lds[wn][1][kk] = s1[k0 + kk];
      }
    __syncthreads();
    // GEMM2 raises the wave's issue priority for its fragment reads and MFMAs
    // (DSV3 M=4096 -1.3%); GEMM1 keeps one level (+3.6% with it)
    constexpr int kPrio = MODE == Mode::kGemm1Silu ? 0 : 1;
    for (int kt = 0; kt < nk; ++kt) {
      if (kt + NBUF - 1 < nk) {
        wait_full(Ring2{});
        issue(kt + NBUF - 1);
      } else {
        wait_stage(min(NBUF - 2, nk - 1 - kt));
      }
      if (!wave_live) continue;
      if (kPrio) __builtin_amdgcn_s_setprio(kPrio);
      const uint8_t* As = lds[kt % NBUF] + (wm * MI) * UPB * kUnit;
      const uint8_t* Bs = lds[kt % NBUF] + (C::A_UNITS + wn * NI * UPB) * kUnit;
      i32x8_t fa[MI], fb[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        i32x4_t lo = lds16(As + (2 * i) * kUnit + foff0), hi = lds16(As + (2 * i) * kUnit + foff1);
        fa[i] = i32x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        i32x4_t lo = lds16(Bs + (2 * j) * kUnit + foff0), hi = lds16(Bs + (2 * j) * kUnit + foff1);
        fb[j] = i32x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
      const float sb0 = sb_lds[wn][0][kt], sb1 = sb_lds[wn][1][kt];
      const float* sa_st = sa_lds[kt % NBUF];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const float sa = sa_st[wm * WM + i * 16 + (lane & 15)];
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          f32x4_t t = {0.f, 0.f, 0.f, 0.f};
          t = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa[i], t, 0, 0, 0, 0, 0, 0);
          const float sb = (MODE == Mode::kGemm1Silu ? j >= NI / 2 : j >= sb_split) ? sb1 : sb0;
          const float sab = sa * sb;
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] += t[r] * sab;
        }
      }
      if (kPrio) __builtin_amdgcn_s_setprio(0);
    }
  } else {
    // bf16.  A step is 32 reduction elements: MI x NI MFMAs on fragments that
    // were read from LDS during the step before, so the matrix cores do not
    // wait for fragment reads.  Between a stage's last two steps its reads
    // are over and the next stage's begin; there, one wait and one barrier
    // both publish stage kt + 1 and free the slot of stage kt, whose DMA
    // (stage kt + NBUF) goes out between that step's MFMAs.  Against reading
    // a stage's first fragments after the barrier that publishes it and
    // issuing the DMA in one go (and without the padding rows' share above),
    // outputs bit-identical, same process: Mixtral M=4096 2614 -> 2530 us a
    // call, Qwen3 M=8192 820 -> 779 us, reference sweep M=2048 622 -> 601 us.
    // What bounds the 256 x 256 kernel now (Mixtral GEMM1 1750 us): with every
    // operand line an L2 hit 1519 us, without the DMA 1353 us, without
    // fragment reads as well 1230 us, the MFMAs alone 1.0 ms at 2.07 GHz.
    constexpr int kMfma = MI * NI, NF = MI + NI;
    // The f-th of n reads (DMA units) goes before MFMA at(f, n, gap): every
    // second MFMA for reads, every third for DMA units (2 / 3 / 4 measured at
    // 256 x 256: Mixtral M=4096 2607 / 2562 / 2610 us a call; back to back
    // they hold up the MFMAs, further apart they arrive late for a 2-deep
    // ring), closer where a step has too few MFMAs for that.
    auto at = [](int f, int n, int gap) { return gap * n <= kMfma ? gap * f : f * kMfma / n; };
    bf16x8_t fa[2][MI], fb[2][NI];
    // fragment f of step h of the stage in slot st, into register set q
    auto read_frag = [&](const uint8_t* st, int h, int q, int f) {
      const int fo = h == 0 ? foff0 : foff1;
      if (f >= 1 && f <= NI)
        fb[q][f - 1] = __builtin_bit_cast(bf16x8_t, lds16(st + (C::A_UNITS + (wn * NI + f - 1) * UPB) * kUnit + fo));
      else
        fa[q][f == 0 ? 0 : f - NI] =
            __builtin_bit_cast(bf16x8_t, lds16(st + (wm * MI + (f == 0 ? 0 : f - NI)) * UPB * kUnit + fo));
    };
    // one step on register set q; READ: fragments of step h of slot st go to
    // set 1 - q; DMA: stage kd goes out
    auto step = [&](int q, auto rd, const uint8_t* st, int h, auto dm, int kd) {
      constexpr bool READ = decltype(rd)::value, DMA = decltype(dm)::value;
#pragma unroll
      for (int m = 0; m < kMfma; ++m) {
        const int i = m / NI, j = m % NI;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (READ) {
#pragma unroll
          for (int f = 0; f < NF; ++f)
            if (at(f, NF, 2) == m) read_frag(st, h, 1 - q, f);
        }
        if constexpr (DMA) {
#pragma unroll
          for (int u = 0; u < C::UPW; ++u)
            if (at(u, C::UPW, 3 * C::UPW <= kMfma ? 3 : 2) == m) issue_unit(kd, u);
        }
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[q][j], fa[q][i], acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    using T = std::true_type;
    using F = std::false_type;
    auto done_reading = [&] { __builtin_amdgcn_s_waitcnt(0xc07f); };  // lgkmcnt(0)

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
#pragma unroll
      for (int f = 0; f < NF; ++f) read_frag(lds[0], 0, 0, f);
      int kt = 0;
      for (; kt + NBUF < nk; ++kt) {
        step(0, T{}, lds[kt % NBUF], 1, F{}, 0);
        done_reading();
        wait_full(Ring2{});
        step(1, T{}, lds[(kt + 1) % NBUF], 0, T{}, kt + NBUF);
      }
      for (; kt + 1 < nk; ++kt) {
        step(0, T{}, lds[kt % NBUF], 1, F{}, 0);
        done_reading();
        wait_stage(min(NBUF - 2, nk - 2 - kt));
        step(1, T{}, lds[(kt + 1) % NBUF], 0, F{}, 0);
      }
      step(0, T{}, lds[kt % NBUF], 1, F{}, 0);
      step(1, F{}, nullptr, 0, F{}, 0);
    }
  }

  // ---- epilogue.  The lane holds slot row lane % 16 of each 16-row block i
  // and output columns tile_col(j, lane) + 0..3 of each weight block j.
  const int orow = lane & 15;
  // Routing weights of the lane's rows, loaded and waited for before the
  // first store.  On gfx9 loads and stores share the vmcnt counter and the
  // compiler treats them as completing out of order, so a use of a load that
  // is still pending after a store waits for every store before it
  // (vmcnt(0) at each of the tile's stores): the empty asm with the values as
  // operands makes the compiler complete the loads here, once.
  float gv[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int s = row_beg + wm * WM + i * 16 + orow;
    gv[i] = (p.gamma && s < row_end) ? p.gate_scal[s] : 1.0f;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) asm volatile("" ::"v"(gv[i]));
  // GEMM2 bias of the lane's columns (split 0 only), loaded the same way
  float bv[MODE == Mode::kGemm2 ? NI : 1][4] = {};
  if (MODE == Mode::kGemm2 && p.bias && split == 0) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int64_t col = static_cast<int64_t>(nt) * BN + wn * WN + tile_col<C::PAIR>(j, lane);
      if (col < p.Nout) {
        const float* b = p.bias + static_cast<int64_t>(e) * p.Nout + col;
#pragma unroll
        for (int c = 0; c < 4; ++c) bv[j][c] = b[c];
      }
    }
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int c = 0; c < 4; ++c) asm volatile("" ::"v"(bv[j][c]));
  }
  if constexpr (FP8 && MODE == Mode::kGemm1Silu && BN / 2 == 128) {
    if (p.act_q) {
      // Activation quantized here, exactly as fmoe_quant_fp8_group would do
      // it on the bf16 activation: the tile's 128 activation columns are one
      // 1x128 group of each row.  Row amax: the lane's values, the 4 lanes
      // holding the row's other columns of this wave, then the WAVES_N waves
      // through LDS (the operand ring is free once every wave has left the
      // main loop).
      __syncthreads();
      float* amax_lds = reinterpret_cast<float*>(&lds[0][0]);  // [BM][WAVES_N]
      float v[MI][NI / 2][4];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const float g = gv[i];
        float amax = 0.f;
#pragma unroll
        for (int j = 0; j < NI / 2; ++j) {
          const int64_t col = static_cast<int64_t>(nt) * (BN / 2) + wn * (WN / 2) + tile_col<C::PAIR>(j, lane);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            float gb, ub;
            gemm1_bias<ACT>(p, e, col + c, gb, ub);
            v[i][j][c] = gemm1_act<ACT>(p, acc[i][j][c], acc[i][j + NI / 2][c], gb, ub, g);
          }
          round_bf16x2(v[i][j][0], v[i][j][1]);
          round_bf16x2(v[i][j][2], v[i][j][3]);
#pragma unroll
          for (int c = 0; c < 4; ++c) amax = fmaxf(amax, fabsf(v[i][j][c]));
        }
        amax = fmaxf(amax, __shfl_xor(amax, 16, kWave));
        amax = fmaxf(amax, __shfl_xor(amax, 32, kWave));
        if (lane < 16) amax_lds[(wm * WM + i * 16 + orow) * C::WAVES_N + wn] = amax;
      }
      __syncthreads();
      const int64_t ngrp = p.N_act / 128;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int r = wm * WM + i * 16 + orow;
        const int s = row_beg + r;
        float amax = 0.f;
#pragma unroll
        for (int w = 0; w < C::WAVES_N; ++w) amax = fmaxf(amax, amax_lds[r * C::WAVES_N + w]);
        const float sc = fmaxf(amax, kFp8Eps) / kFp8Max;
        const float inv = 1.0f / sc;
        if (s >= row_end) continue;
        uint8_t* q = p.act_q + static_cast<int64_t>(s) * p.N_act + static_cast<int64_t>(nt) * (BN / 2) + wn * (WN / 2);
        uint32_t w[NI / 2];
#pragma unroll
        for (int j = 0; j < NI / 2; ++j)
          w[j] = pack_e4m3x4(fp8_qdiv(v[i][j][0], sc, inv), fp8_qdiv(v[i][j][1], sc, inv),
                             fp8_qdiv(v[i][j][2], sc, inv), fp8_qdiv(v[i][j][3], sc, inv));
        if constexpr (C::PAIR) {
#pragma unroll
          for (int j = 0; j < NI / 2; j += 2)
            *reinterpret_cast<uint2*>(q + tile_col<true>(j, lane)) = make_uint2(w[j], w[j + 1]);
        } else {
#pragma unroll
          for (int j = 0; j < NI / 2; ++j) *reinterpret_cast<uint32_t*>(q + tile_col<false>(j, lane)) = w[j];
        }
        if (wn == 0 && lane < 16) p.act_qs[static_cast<int64_t>(s) * ngrp + nt] = sc;
      }
      return;
    }
  }
  const bool y_rows_bf16 = p.y_bf16 && tail < 0;  // whole tile, one split: bf16 slot rows
  // four bf16 columns of blocks j (and j + 1) of a row: one 16- or 8-byte store
  auto store_bf16 = [&](uint16_t* row, int64_t c0, int j, const uint32_t* w) {
    uint16_t* dst = row + c0 + tile_col<C::PAIR>(j, lane);
    if constexpr (C::PAIR)
      *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
    else
      *reinterpret_cast<uint2*>(dst) = make_uint2(w[0], w[1]);
  };
  constexpr int JS = C::PAIR ? 2 : 1;  // blocks per store
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int s = row_beg + wm * WM + i * 16 + orow;
    const bool ok = s < row_end;
    const float g = gv[i];
    if (MODE == Mode::kGemm1Silu) {
      uint16_t* act = static_cast<uint16_t*>(p.out) + static_cast<int64_t>(s) * p.N_act;
      const int64_t c0 = static_cast<int64_t>(nt) * (BN / 2) + wn * (WN / 2);
#pragma unroll
      for (int j = 0; j < NI / 2; j += JS) {
        uint32_t w[2 * JS];
#pragma unroll
        for (int h = 0; h < 2 * JS; ++h) {
          const int jj = j + h / 2, c = 2 * (h % 2);
          const int64_t col = c0 + tile_col<C::PAIR>(jj, lane) + c;
          float a[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float gb, ub;
            gemm1_bias<ACT>(p, e, col + u, gb, ub);
            a[u] = gemm1_act<ACT>(p, acc[i][jj][c + u], acc[i][jj + NI / 2][c + u], gb, ub, g);
          }
          w[h] = pack_bf16x2(a[0], a[1]);
        }
        if (ok && c0 + tile_col<C::PAIR>(j, lane) < p.N_act) store_bf16(act, c0, j, w);
      }
    } else {
      // fp32 destination row: a split plane's slot row, or the tile's row of
      // its tail-split partial ([BM][BN] within the tile; the row pointer is
      // taken back by the tile's first column, which `col` adds again, so
      // both cases share one store)
      float* y = tail >= 0 ? p.tail_part + static_cast<int64_t>(tail) * (BM * BN) +
                                 (wm * WM + i * 16 + orow) * BN - static_cast<int64_t>(nt) * BN
                           : static_cast<float*>(p.out) + split * p.out_split_stride +
                                 static_cast<int64_t>(s) * p.Nout;
      uint16_t* yb = static_cast<uint16_t*>(p.out) + static_cast<int64_t>(s) * p.Nout;
      const int64_t c0 = static_cast<int64_t>(nt) * BN + wn * WN;
#pragma unroll
      for (int j = 0; j < NI; j += JS) {
        f32x4_t v[JS];
#pragma unroll
        for (int h = 0; h < JS; ++h) {
          v[h] = acc[i][j + h];
          if (p.bias && split == 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c) v[h][c] += bv[j + h][c];
          }
#pragma unroll
          for (int c = 0; c < 4; ++c) v[h][c] *= g;
        }
        const int64_t col = c0 + tile_col<C::PAIR>(j, lane);
        if (ok && col < p.Nout) {
          if (y_rows_bf16) {
            // one split: the row goes out as bf16, like SGLang's per-slot
            // intermediate before its top-k sum
            uint32_t w[2 * JS];
#pragma unroll
            for (int h = 0; h < 2 * JS; ++h) w[h] = pack_bf16x2(v[h / 2][2 * (h % 2)], v[h / 2][2 * (h % 2) + 1]);
            store_bf16(yb, c0, j, w);
          } else {
#pragma unroll
            for (int h = 0; h < JS; ++h)
              *reinterpret_cast<float4*>(y + col + 4 * h) = make_float4(v[h][0], v[h][1], v[h][2], v[h][3]);
          }
        }
      }
    }
  }
}

template <class C>
int launch(const GemmParams& p, hipStream_t s) {
  if (C::FP8 && p.Kred / 128 > C::KST)
    return fmoe_host::fail(FMOE_ERR_UNSUPPORTED, "prefill fp8: reduction dim %lld is not supported",
                           static_cast<long long>(p.Kred));
  Kernel k = gemm_prefill_kernel<C, kActSilu>;
  if (C::MODE == Mode::kGemm1Silu && p.act == kActGelu) k = gemm_prefill_kernel<C, kActGelu>;
  if (C::MODE == Mode::kGemm1Silu && p.act == kActSwiglu) k = gemm_prefill_kernel<C, kActSwiglu>;
  return launch_tiles<C>(p, s, static_cast<int>((C::FP8 ? p.Kred : 2 * p.Kred) / C::SB), k);
}

}  // namespace prefill

// Host launcher: picks the instantiation for the tile height.
//   bf16: BM 256 -> 256x256, 4x2 waves, 128-byte stages, 2-deep ring
//         BM 160 -> 160x256, 2x4 waves, 128-byte stages, 3-deep ring
//         BM 128 -> 128x256, 2x4 waves, 128-byte stages, 3-deep ring
//         BM  64 ->  64x128, 1x4 waves, 128-byte stages, 3-deep ring
//         BM  32 ->  32x128, 1x4 waves, 128-byte stages, 4-deep ring
//         (72 and 80 KiB of LDS: two workgroups per CU, so one streams while
//         the other starts or ends, with 48 / 60 KiB each in flight; 64x256
//         with 64-byte stages in a 4-deep ring, one workgroup per CU, took 346
//         us against 297 on the reference sweep's M=128, 563 against 501 on
//         Mixtral M=100)
//   fp8 : BM 160 -> GEMM1 160x256, 3-deep ring; GEMM2 160x384, 2-deep ring;
//                   2x4 waves, 128-byte stages (K, N <= 8192)
//         BM 128 -> 128x256, 2x4 waves, 128-byte stages, 3-deep ring
//         BM  64 ->  64x256, 1x8 waves, 128-byte stages, 3-deep ring
int launch_prefill(WType wt, Mode mode, int bm, const GemmParams& p, hipStream_t s) {
  using namespace prefill;
  const bool fp8 = wt == WType::kFp8;
#define L(BM, BN, WMS, WNS, NB, F8)                                                          \
  (mode == Mode::kGemm1Silu ? launch<Cfg<BM, BN, WMS, WNS, NB, F8, Mode::kGemm1Silu>>(p, s) \
                            : launch<Cfg<BM, BN, WMS, WNS, NB, F8, Mode::kGemm2>>(p, s))
  if (!fp8) {
    if (bm == 256) return L(256, 256, 4, 2, 2, false);
    if (bm == 160) return L(160, 256, 2, 4, 3, false);
    if (bm == 128) return L(128, 256, 2, 4, 3, false);
    if (bm == 64) return L(64, 128, 1, 4, 3, false);
    if (bm == 32) return L(32, 128, 1, 4, 4, false);
  } else {
    // GEMM2 with 160-row tiles: 384-wide output tiles (2-deep ring of 68 KiB
    // stages), so the activation tile is re-read by a third fewer N-tiles
    // (13% fewer operand requests per output; DSV3 GEMM2 M=4096 -5%, M=8192 -7%)
    if (bm == 160)
      return mode == Mode::kGemm2 ? launch<Cfg<160, 384, 2, 4, 2, true, Mode::kGemm2>>(p, s)
                                  : launch<Cfg<160, 256, 2, 4, 3, true, Mode::kGemm1Silu>>(p, s);
    if (bm == 128) return L(128, 256, 2, 4, 3, true);
    if (bm == 64) return L(64, 256, 1, 8, 3, true);
  }
#undef L
  return fmoe_host::fail(FMOE_ERR_UNSUPPORTED,
                         "prefill: block_m=%d is not supported for this weight type", bm);
}

// Bytes of the tail-split partial buffer for a fused prefill GEMM2 of this
// weight type and tile height (the configuration launch_prefill picks).
size_t prefill_tail_bytes(WType wt, int bm, int64_t max_tiles, int64_t Nout) {
  using namespace prefill;
#define T(BM, BN, WMS, WNS, NB, F8) \
  static_cast<size_t>(tail_pairs_for<Cfg<BM, BN, WMS, WNS, NB, F8, Mode::kGemm2>>( \
      gemm_prefill_kernel<Cfg<BM, BN, WMS, WNS, NB, F8, Mode::kGemm2>, kActSilu>, max_tiles, Nout)) * BM * BN * 4
  if (wt != WType::kFp8) {
    if (wt != WType::kBf16) return 0;
    if (bm == 256) return T(256, 256, 4, 2, 2, false);
    if (bm == 160) return T(160, 256, 2, 4, 3, false);
    if (bm == 128) return T(128, 256, 2, 4, 3, false);
    if (bm == 64) return T(64, 128, 1, 4, 3, false);
    if (bm == 32) return T(32, 128, 1, 4, 4, false);
  } else {
    if (bm == 160) return T(160, 384, 2, 4, 2, true);
    if (bm == 128) return T(128, 256, 2, 4, 3, true);
    if (bm == 64) return T(64, 256, 1, 8, 3, true);
  }
#undef T
  return 0;
}

}  // namespace fmoe
