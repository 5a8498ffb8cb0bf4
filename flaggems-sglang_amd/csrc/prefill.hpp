// Pieces shared by the prefill GEMM kernels (gemm_prefill.hip, gemm_w4.hip):
// direct-to-LDS DMA and its waits, LDS unit layout, tile order, the table of
// tiles and the tail split.
#pragma once

#include <algorithm>

#include "gemm.hpp"

namespace fmoe {
namespace prefill {

constexpr int kUnit = 1024;       // one DMA wave-instruction: 64 lanes x 16 B
constexpr int kMaxKStages = 128;  // fp8: reduction dims up to 16384 (64 stages when LDS is short)
constexpr int kGroupTiles = 32;   // tiles per rasterization window (~ one XCD's CUs)

typedef __attribute__((address_space(3))) void* lds_ptr_t;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 0xf) | ((N >> 4) << 14) | (0x7 << 4) | (0xf << 8));
}

// wait until at most n of this wave's loads are in flight (n uniform, 0..MAX)
template <int MAX>
__device__ __forceinline__ void wait_loads(int n) {
  if constexpr (MAX == 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= MAX) wait_vmcnt<MAX>();
    else wait_loads<MAX - 1>(n);
  }
}

__device__ __forceinline__ void barrier_nofence() { asm volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_addr(const void* l) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)(l)));
}
// lane i's 16 (or 4) bytes land at LDS address l + 16 i (4 i)
__device__ __forceinline__ void dma16(const uint8_t* g, uint8_t* l) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_addr(l));
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(g), "s"(m0) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const float* g, float* l) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_addr(l));
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :: "v"(g), "s"(m0) : "memory", "m0");
}

// LDS unit layout (1 KiB = one DMA wave-instruction, lane i -> bytes 16i): a
// unit is 8 rows x 128 bytes (rows 0-7 or 8-15 of a 16-row block); DMA lane i
// reads row i / 8, chunk (i % 8) ^ (row), so 8 consecutive lanes read one
// row's 128 contiguous bytes.
// The MFMA fragment of lane L is row L % 16, 16-byte chunk c (c = L / 16 and
// 4 + L / 16); with the swizzle every 8 consecutive lanes of a fragment read
// hit 8 distinct 16-byte columns of a 128-byte window, which ds_read_b128
// serves at the contiguous rate (measured: plain row-major or a (row / 4)
// swizzle run at 70% of it).
__device__ __forceinline__ int frag_off(int L, int c) {
  const int r = L & 15, ru = r & 7;
  return (r >> 3) * 1024 + 16 * (8 * ru + (c ^ ru));
}

__device__ __forceinline__ i32x4_t lds16(const uint8_t* p) { return *reinterpret_cast<const i32x4_t*>(p); }

// Expert e with offs_pad[e] * nn <= key < offs_pad[e + 1] * nn (offs_pad is
// non-decreasing, offs_pad[0] = 0, key < offs_pad[E] * nn): two rounds of 64
// parallel probes and a ballot, instead of a serial binary search.
__device__ __forceinline__ int find_expert(const int32_t* offs_pad, int E, int key, int nn, int lane) {
  const int S = (E + 1 + kWave - 1) / kWave;
  const int i1 = min(lane * S, E);
  uint64_t b = __ballot(offs_pad[i1] * nn <= key);
  const int base = (63 - __builtin_clzll(b)) * S;
  const int i2 = min(base + lane, E);
  b = __ballot(lane < S && offs_pad[i2] * nn <= key);
  return base + (63 - __builtin_clzll(b));
}

// Which weight row of a tile sits in row lr of its 16-row LDS block b.  The
// MFMA takes the weight fragment as its first operand, so a lane ends with
// four consecutive weight rows 4 * (lane / 16) + 0..3 (output columns) of one
// slot row, lane % 16: what a row store wants, with no exchange between lanes.
// With PAIR, the rows of blocks 2p and 2p + 1 are dealt out four by four, so
// a lane's two blocks are 8 consecutive columns (one 16-byte bf16 store, and
// 64 contiguous bytes per row and instruction).  fp8: one activation scale
// per lane and row block instead of four.  Against the opposite operand order
// with 4x4 lane transposes and integer bf16 rounding in the epilogue, outputs
// bit-identical: Mixtral bf16 M=4096 2707 -> 2626 us a call, Qwen3 M=8192
// 891 -> 817 us, reference sweep M=1024 436 -> 416 us, DSV3 fp8 M=4096
// 2991 -> 2724 us.
template <bool PAIR>
__device__ __forceinline__ int tile_row(int b, int lr) {
  if constexpr (PAIR) return (b >> 1) * 32 + (lr >> 2) * 8 + (b & 1) * 4 + (lr & 3);
  return b * 16 + lr;
}
// First of the lane's four output columns of block j (same numbering).
template <bool PAIR>
__device__ __forceinline__ int tile_col(int j, int lane) {
  return tile_row<PAIR>(j, (lane >> 4) * 4);
}

// Logical tile L (within one split) -> expert, N-tile and rows.  Per expert,
// windows of all its T M-tiles x G N-tiles (T * G ~ group_tiles, about what
// one XCD runs at once) are enumerated M-fastest, so the tiles that share a
// weight panel run together on one XCD and the panel is fetched from HBM
// once.  Called by one whole wave (find_expert ballots).
struct Tile {
  int e, nt, row_beg, row_end;
};
template <int BM>
__device__ __forceinline__ Tile tile_of(const GemmParams& p, int L, int lane) {
  const int nn = p.n_ntiles;
  Tile t;
  t.e = find_expert(p.offs_pad, p.n_experts, L, nn, lane);
  const int t0 = p.offs_pad[t.e];
  const int T = p.offs_pad[t.e + 1] - t0;
  const int local = L - t0 * nn;
  const int G = max(1, p.group_tiles / T);
  const int grp = local / (T * G);
  const int rr = local - grp * T * G;
  const int blk = rr % T;
  t.nt = grp * G + rr / T;
  t.row_beg = p.offs_raw[t.e] + blk * BM;
  t.row_end = min(p.offs_raw[t.e + 1], t.row_beg + BM);
  return t;
}

// Tail split of XCD x (GEMM2, p.tail_split > 1): the XCD's logical tiles are
// [base, base + Tx) (xcd_remap's partition of the T live tiles).  Whole
// tiles fill rounds of `slots` workgroups; the tl = Tx % slots tiles of the
// last partial round are split S = min(max_split, slots / tl, stages) ways,
// so their tl * S workgroups fill at most one round.  S = 1: no split, every
// tile whole.  The GEMM and tail_fold_kernel derive the same plan.
struct TailPlan {
  int base, full, tl, S;
};
__device__ __forceinline__ TailPlan tail_plan(int T, int x, int max_split, int slots, int stages) {
  const int q = T / kNumXcd, r8 = T % kNumXcd;
  const int Tx = q + (x < r8 ? 1 : 0);
  TailPlan t;
  t.base = x * q + min(x, r8);
  t.tl = Tx % slots;
  t.S = t.tl > 0 ? min(min(max_split, slots / t.tl), stages) : 1;
  if (t.S < 2) {
    t.S = 1;
    t.tl = 0;
  }
  t.full = Tx - t.tl;
  return t;
}
// Index of XCD x's first tail pair: the pairs of XCDs 0 .. x-1 come first.
__device__ __forceinline__ int tail_offset(int T, int x, int max_split, int slots, int stages) {
  int off = 0;
  for (int y = 0; y < x; ++y) {
    const TailPlan t = tail_plan(T, y, max_split, slots, stages);
    off += t.tl * t.S;
  }
  return off;
}

// Fills p.tile_lut for every live logical tile: one wave per tile.
template <int BM>
__global__ __launch_bounds__(256) void tile_lut_kernel(GemmParams p) {
  const int lane = threadIdx.x % kWave;
  const int L = blockIdx.x * 4 + threadIdx.x / kWave;
  if (L >= *p.n_tiles * p.n_ntiles) return;
  const Tile t = tile_of<BM>(p, L, lane);
  if (lane == 0) p.tile_lut[L] = int4{t.e, t.nt, t.row_beg, t.row_end};
}

// A workgroup's work: expert, N-tile, slot rows, part `split` of `n_splits` of
// the reduction, and its pair index in p.tail_part (-1: a whole tile or a
// split plane).  Workgroup ids are made XCD-contiguous, then mapped by
// tile_of (or its precomputed table).  False: nothing to do.  `stages`: ring
// stages of the whole reduction.
struct Work {
  int e, nt, row_beg, row_end, split, n_splits, tail;
};
template <int BM, Mode MODE>
__device__ __forceinline__ bool locate(const GemmParams& p, int stages, int lane, Work& w) {
  const int per_split = *p.n_tiles * p.n_ntiles;
  int L;
  w.n_splits = p.splits;
  w.tail = -1;
  if (MODE == Mode::kGemm2 && p.tail_split > 1) {
    const TailPlan t = tail_plan(per_split, static_cast<int>(blockIdx.x) % kNumXcd, p.tail_split,
                                 p.tail_slots, stages);
    const int i = static_cast<int>(blockIdx.x) / kNumXcd;  // dispatch position within the XCD
    if (i < t.full) {
      L = t.base + i;
      w.split = 0;
      w.n_splits = 1;
    } else {
      const int j = i - t.full;
      if (j >= t.tl * t.S) return false;
      L = t.base + t.full + j / t.S;
      w.split = j % t.S;
      w.n_splits = t.S;
      w.tail = tail_offset(per_split, static_cast<int>(blockIdx.x) % kNumXcd, p.tail_split, p.tail_slots,
                           stages) + j;
      if (w.tail >= p.tail_pairs) return false;  // the host sizes tail_part for every pair
    }
  } else {
    const int live = per_split * p.splits;
    if (static_cast<int>(blockIdx.x) >= live) return false;
    L = xcd_remap(blockIdx.x, live);
    w.split = L / per_split;
    L -= w.split * per_split;
  }
  if (p.tile_lut) {
    const int4 v = p.tile_lut[L];
    w.e = v.x;
    w.nt = v.y;
    w.row_beg = v.z;
    w.row_end = v.w;
  } else {
    const Tile t = tile_of<BM>(p, L, lane);
    w.e = t.e;
    w.nt = t.nt;
    w.row_beg = t.row_beg;
    w.row_end = t.row_end;
  }
  return true;
}

// Adds the tail-split partials of each split tile in split order and writes
// the tile's rows (bf16 or fp32, [slot][Nout]): one workgroup per (XCD,
// tail tile, 16-row chunk), every partial of the chunk loaded before the
// adds.  Bias and routing weight are already in the partials.
constexpr int kFoldRows = 16;
template <int BM, int BN>
__global__ __launch_bounds__(256) void tail_fold_kernel(GemmParams p, int stages) {
  constexpr int kChunks = BM / kFoldRows;
  constexpr int kVec = kFoldRows * BN / (4 * 256);  // float4 per thread and partial
  static_assert(kFoldRows * BN % (4 * 256) == 0, "fold chunk");
  const int rc = blockIdx.x % kChunks;
  const int xt = blockIdx.x / kChunks;
  const int x = xt / p.tail_slots, t = xt % p.tail_slots;
  const int T = *p.n_tiles * p.n_ntiles;
  const TailPlan pl = tail_plan(T, x, p.tail_split, p.tail_slots, stages);
  if (t >= pl.tl) return;
  const int pair0 = tail_offset(T, x, p.tail_split, p.tail_slots, stages) + t * pl.S;
  if (pair0 + pl.S > p.tail_pairs) return;
  const int L = pl.base + pl.full + t;
  int nt, rb, re;
  if (p.tile_lut) {
    const int4 v = p.tile_lut[L];
    nt = v.y;
    rb = v.z;
    re = v.w;
  } else {
    const Tile tt = tile_of<BM>(p, L, threadIdx.x % kWave);
    nt = tt.nt;
    rb = tt.row_beg;
    re = tt.row_end;
  }
  const int r0 = rc * kFoldRows;
  if (r0 >= re - rb) return;
  const int64_t c0 = static_cast<int64_t>(nt) * BN;
  const int cols = static_cast<int>(min(static_cast<int64_t>(BN), p.Nout - c0));
  const float* part = p.tail_part + static_cast<int64_t>(pair0) * (BM * BN) + r0 * BN;
  float4 a[kVec];
#pragma unroll
  for (int v = 0; v < kVec; ++v) a[v] = *reinterpret_cast<const float4*>(part + (threadIdx.x + v * 256) * 4);
  for (int sp = 1; sp < pl.S; ++sp) {
    float4 b[kVec];
#pragma unroll
    for (int v = 0; v < kVec; ++v)
      b[v] = *reinterpret_cast<const float4*>(part + static_cast<int64_t>(sp) * (BM * BN) + (threadIdx.x + v * 256) * 4);
#pragma unroll
    for (int v = 0; v < kVec; ++v) {
      a[v].x += b[v].x;
      a[v].y += b[v].y;
      a[v].z += b[v].z;
      a[v].w += b[v].w;
    }
  }
#pragma unroll
  for (int v = 0; v < kVec; ++v) {
    const int idx = (threadIdx.x + v * 256) * 4;
    const int r = idx / BN, c = idx - (idx / BN) * BN;
    if (r0 + r >= re - rb || c >= cols) continue;
    const int64_t o = static_cast<int64_t>(rb + r0 + r) * p.Nout + c0 + c;
    if (p.y_bf16)
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + o) =
          make_uint2(pack_bf16x2(a[v].x, a[v].y), pack_bf16x2(a[v].z, a[v].w));
    else
      *reinterpret_cast<float4*>(static_cast<float*>(p.out) + o) = a[v];
  }
}

// Workgroup slots of one XCD for a configuration's kernel (workgroups per CU
// x CUs per XCD); 0 when the runtime cannot say (the tail split is then off).
using Kernel = void (*)(GemmParams);
template <class C>
int xcd_slots(Kernel kernel) {
  static const int slots = [kernel] {
    int dev = 0, cus = 0, occ = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, C::NT, 0) != hipSuccess) {
      (void)hipGetLastError();  // not left for the next launch's check to report
      return 0;
    }
    return (cus % kNumXcd == 0 && occ > 0) ? occ * (cus / kNumXcd) : 0;
  }();
  return slots;
}

// Partials the tail split of a GEMM2 launch may need: at most one round of
// an XCD's slots per XCD, and at most kTailMaxSplit per live tile.
template <class C>
int64_t tail_pairs_for(Kernel kernel, int64_t max_tiles, int64_t Nout) {
  const int slots = xcd_slots<C>(kernel);
  if (slots <= 0) return 0;
  const int64_t nn = (Nout + C::BN - 1) / C::BN;
  return std::min<int64_t>(static_cast<int64_t>(kNumXcd) * slots, max_tiles * nn * kTailMaxSplit);
}

// Launches `kernel` over every (expert tile, output tile): the table of tiles
// first, the tail split's fold after it.  `stages`: ring stages of the whole
// reduction.
template <class C>
int launch_tiles(const GemmParams& p0, hipStream_t s, int stages, Kernel kernel) {
  GemmParams p = p0;
  const int64_t ncols = C::MODE == Mode::kGemm1Silu ? p.N_act : p.Nout;
  const int per_tile = C::MODE == Mode::kGemm1Silu ? C::BN / 2 : C::BN;
  p.n_ntiles = static_cast<int>((ncols + per_tile - 1) / per_tile);
  if (p.group_tiles <= 0) p.group_tiles = kGroupTiles;
  if (p.splits < 1) p.splits = 1;
  int64_t grid = static_cast<int64_t>(p.max_tiles) * p.n_ntiles * p.splits;
  if (C::MODE == Mode::kGemm2 && p.tail_split > 1) {
    const int slots = xcd_slots<C>(kernel);
    const int64_t pairs = tail_pairs_for<C>(kernel, p.max_tiles, p.Nout);
    p.tail_pairs = static_cast<int64_t>(p.tail_bytes / (static_cast<size_t>(C::BM) * C::BN * sizeof(float)));
    if (slots <= 0 || !p.tail_part || pairs <= 0 || p.tail_pairs < pairs || p.splits != 1) {
      p.tail_split = 0;  // whole tiles only
    } else {
      p.tail_slots = slots;
      const int64_t per_xcd = (static_cast<int64_t>(p.max_tiles) * p.n_ntiles + kNumXcd - 1) / kNumXcd;
      grid = kNumXcd * (per_xcd + slots);  // whole tiles + one round of tail workgroups per XCD
    }
  }
  if (grid <= 0) return FMOE_OK;
  if (grid > 0x7fffffff) return fmoe_host::fail(FMOE_ERR_UNSUPPORTED, "prefill grid too large");
  if (p.tile_lut) {
    const int64_t lut_n = static_cast<int64_t>(p.max_tiles) * p.n_ntiles;
    tile_lut_kernel<C::BM><<<dim3(static_cast<unsigned>((lut_n + 3) / 4)), dim3(256), 0, s>>>(p);
  }
  kernel<<<dim3(static_cast<unsigned>(grid)), dim3(C::NT), 0, s>>>(p);
  if (C::MODE == Mode::kGemm2 && p.tail_split > 1)
    tail_fold_kernel<C::BM, C::BN>
        <<<dim3(static_cast<unsigned>(kNumXcd * p.tail_slots * (C::BM / kFoldRows))), dim3(256), 0, s>>>(p, stages);
  return fmoe_host::check_launch("prefill gemm");
}

}  // namespace prefill
}  // namespace fmoe
