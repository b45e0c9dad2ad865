// The fp16 MFMA GEMM mainloop shared by the lm_head kernels (lmhead.hip) and the projections'
// split-K product (gemm.hip): C[M, N] (+)= A[M, K] . op(B) on v_mfma_f32_32x32x16_f16, 256 x 256
// block tiles, blocks numbered XCD-aware, A always K-contiguous ([M, lda]) and B either
// K-contiguous ([N, ldb], op(B) = B^T) or N-contiguous ([K, ldb], op(B) = B), the second read
// out of LDS with gfx950's transposing ds_read_b64_tr_b16.
#pragma once

#include <type_traits>

#include "common.h"

namespace rus {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 256, kBN = 256, kBK = 64;
constexpr int kThreads = 256;
constexpr int kWM = 128, kWN = 128;
constexpr int kMT = kWM / 32, kNT = kWN / 32;
constexpr int kTileBytes = kBM * kBK * 2;  // 32 KiB
constexpr int kSmemBytes = 4 * kTileBytes;  // 128 KiB: the mainloop's four stages, the epilogues' staging

struct GemmArgs {
  const f16* A;  // [M, lda], rows K-contiguous
  const f16* B;  // [N, ldb] K-contiguous, or [K, ldb] N-contiguous (the KN mainloop)
  int64_t lda, ldb;
  int M, N;
  int K;            // multiple of kBK
  int k_per_split;  // multiple of kBK
  int splits;
  int tiles_m, tiles_n;
};

struct Tile {
  int m0, n0, split;
};

__device__ __forceinline__ bool tile_of(const GemmArgs& g, Tile& t) {
  const int total = g.tiles_m * g.tiles_n * g.splits;
  const int per_xcd = (total + 7) >> 3;
  const int local = blockIdx.x >> 3;
  const int work = (blockIdx.x & 7) * per_xcd + local;
  if (local >= per_xcd || work >= total) return false;
  const int tn = work % g.tiles_n;
  const int rest = work / g.tiles_n;
  t.m0 = (rest % g.tiles_m) * kBM;
  t.split = rest / g.tiles_m;
  t.n0 = tn * kBN;
  return true;
}

// acc[mt][nt] += A[m0 + wm*128 + mt*32 .. +32, k] . B[n0 + wn*128 + nt*32 .. +32, k]^T over the
// split's K range. Accumulator layout (v_mfma_f32_32x32x16_f16): register r of lane l holds
// row 8*(r/4) + 4*(l/32) + r%4, column l%32 of the 32x32 tile.
//
// Two pipelines. mainloop_t (the four-wave logit-gradient kernel) stages K 32 at a time through
// four LDS buffers of 32 KiB (A then B, 256 rows x 64 bytes each);
// mainloop_k64 (the eight-wave kernels) stages K 64 at a time, below. Global memory is copied
// straight into LDS (global_load_lds_dwordx4: each lane's 16 bytes land at buffer + lane * 16),
// three stages ahead of the MFMAs, so no register holds a tile in flight. The 16-byte chunk c of
// row r is stored at chunk c ^ ((r >> 2) & 3) of its 64-byte row, which a lane realises by loading
// the chunk that belongs at its position; the MFMAs' 16-byte fragment reads (16 consecutive rows
// per quarter wave, one chunk) then hit all 64 banks once. The fragment reads are explicit ds_read_b128 with
// explicit lgkmcnt waits (the compiler would otherwise wait for every LDS-bound global load before
// any LDS read); vmcnt waits and the one barrier per stage sit inside the stage's second K step,
// so the MFMA pipe keeps busy across stages.
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;

constexpr int kDK = 32;                  // K per LDS stage
constexpr int kStageBytes = 2 * kBM * kDK * 2;  // A + B: 32 KiB
constexpr int kNStages = 4;
static_assert(kNStages * kStageBytes == kSmemBytes, "stages fill the kernel's LDS");

template <int OFF>
__device__ __forceinline__ u32x4v lds_read16(uint32_t addr) {
  u32x4v v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(OFF));
  return v;
}

// The fragments of one K step of 16 from LDS addresses a / b (4 row groups of A and of B).
__device__ __forceinline__ void read_frags(uint32_t a, uint32_t b, u32x4v (&fa)[kMT],
                                           u32x4v (&fb)[kNT]) {
  fa[0] = lds_read16<0>(a);
  fa[1] = lds_read16<2048>(a);
  fa[2] = lds_read16<4096>(a);
  fa[3] = lds_read16<6144>(a);
  fb[0] = lds_read16<0>(b);
  fb[1] = lds_read16<2048>(b);
  fb[2] = lds_read16<4096>(b);
  fb[3] = lds_read16<6144>(b);
}

// Every LDS read issued so far has returned; ties the fragments so that no MFMA using them is
// scheduled before the wait.
__device__ __forceinline__ void wait_frags(u32x4v (&fa)[kMT], u32x4v (&fb)[kNT]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3]), "+v"(fb[0]), "+v"(fb[1]),
                 "+v"(fb[2]), "+v"(fb[3]));
}

__device__ __forceinline__ void mma16(const u32x4v (&fa)[kMT], const u32x4v (&fb)[kNT],
                                      f32x16 (&acc)[kMT][kNT]) {
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
      acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          __builtin_bit_cast(f16x8, fa[mt]), __builtin_bit_cast(f16x8, fb[nt]), acc[mt][nt], 0,
          0, 0);
}

// B stored [K][N] (N-contiguous) in LDS: 64 rows of 256 columns (512 bytes) per stage, the
// 16-byte chunk c of row r at chunk c ^ ((r & 3) << 2). ds_read_b64_tr_b16 lets each group of 16
// lanes read a 4 x 16 block and transposes it: lane i of the group receives the 16-bit element
// i % 4 of the 8 bytes read by lanes i / 4 + 4 e (e = 0..3) of the group. With lane j of the group
// pointing at row k0 + j / 4, columns n0 + 4 (j % 4) .. +4, lane i therefore holds
// B[k0 + e][n0 + i], e = 0..3: the low or high half of its MFMA B operand (8 consecutive K of
// column n0 + i). The four rows a group reads sit in four different 64-byte quarters of the
// 256-byte bank window, so a half wave's 32 lanes hit all 64 banks once.
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));

template <int OFF>
__device__ __forceinline__ u32x2v lds_read8_tr(uint32_t addr) {
  u32x2v v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(OFF));
  return v;
}

constexpr int kKNRowBytes = kBN * 2;  // one K row of the B stage: 512 bytes

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt not waited on).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Waits until at most `stages` (0..4) stages of PER copies each are still in flight.
template <int PER>
__device__ __forceinline__ void wait_stages(int stages) {
  if (stages >= 4)
    wait_vmcnt<4 * PER>();
  else if (stages == 3)
    wait_vmcnt<3 * PER>();
  else if (stages == 2)
    wait_vmcnt<2 * PER>();
  else if (stages == 1)
    wait_vmcnt<PER>();
  else
    wait_vmcnt<0>();
}

// Waves 2 (M halves) x 2 (N halves) of 128 x 128 (acc[4][4], one wave per SIMD).
__device__ __forceinline__ void mainloop_t(const GemmArgs& g, const Tile& tl, char* smem,
                                           f32x16 (&acc)[kMT][kNT]) {
  constexpr int CP = 4;  // copies per thread per operand and stage
  constexpr int PER = 2 * CP;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int kb = tl.split * g.k_per_split;
  const int ke = min(kb + g.k_per_split, g.K);
  const int KT = ke > kb ? (ke - kb) / kDK : 0;
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) acc[mt][nt] = f32x16{};
  if (KT == 0) {
    __syncthreads();
    return;
  }
  // Copies: instruction i of wave w fills bytes 1024 (4 i + w) .. +1024 of the stage's A and B
  // tiles: rows 64 i + 16 w .. +16 of 64 bytes; lane l covers row 64 i + 16 w + l/4 at position
  // l%4, i.e. the chunk (l%4) ^ ((l/16) & 3).
  const int lrow = 16 * wave + (lane >> 2);
  const int lchunk = (lane & 3) ^ ((lane >> 4) & 3);
  const char* gA = reinterpret_cast<const char*>(g.A);
  const char* gB = reinterpret_cast<const char*>(g.B);
  uint32_t oa[CP], ob[CP];
#pragma unroll
  for (int i = 0; i < CP; ++i) {
    // Rows past the matrix edge re-read the last one: finite values the epilogue discards.
    const int ra_ = min(tl.m0 + lrow + 64 * i, g.M - 1);
    const int rb_ = min(tl.n0 + lrow + 64 * i, g.N - 1);
    oa[i] = static_cast<uint32_t>((ra_ * g.lda + kb + lchunk * 8) * 2);
    ob[i] = static_cast<uint32_t>((rb_ * g.ldb + kb + lchunk * 8) * 2);
  }
  auto issue = [&](int k) {  // stage k's copies into buffer k % kNStages
    char* st = smem + (k % kNStages) * kStageBytes;
    const uint32_t bytes = k * (kDK * 2);
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      __builtin_amdgcn_global_load_lds(gA + oa[i] + bytes,
                                       (lds_void_ptr)(st + (4 * i + wave) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(gB + ob[i] + bytes,
                                       (lds_void_ptr)(st + kBM * 64 + (4 * i + wave) * 1024), 16,
                                       0, 0);
    }
  };
  const int pre = min(kNStages, KT);
  for (int k = 0; k < pre; ++k) issue(k);
  wait_stages<PER>(pre - 1);  // stage 0 landed (this wave's copies)
  __builtin_amdgcn_s_barrier();  // ... and every wave's
  // Fragment addresses: A row wm*128 + (l & 31), B row wn*128 + (l & 31) (+ 32 per MFMA tile,
  // immediate), chunk 2 kk + l/32 stored at chunk ^ ((l >> 2) & 3).
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_ptr)smem));
  const int sw = (lane >> 2) & 3, half = lane >> 5;
  const uint32_t c0 = ((0 + half) ^ sw) << 4, c1 = ((2 + half) ^ sw) << 4;
  const uint32_t arow = lds0 + (wm * kWM + (lane & 31)) * 64;
  const uint32_t a0 = arow + c0, a1 = arow + c1;
  const uint32_t brow = lds0 + kBM * 64 + (wn * kWN + (lane & 31)) * 64;
  const uint32_t b0 = brow + c0, b1 = brow + c1;
  u32x4v fa0[kMT], fb0[kNT], fa1[kMT], fb1[kNT];
  read_frags(a0, b0, fa0, fb0);
  wait_frags(fa0, fb0);
  for (int k = 0; k < KT; ++k) {
    const uint32_t sb = (k % kNStages) * kStageBytes;
    read_frags(a1 + sb, b1 + sb, fa1, fb1);  // step 1 of stage k
    __builtin_amdgcn_sched_barrier(0);
    mma16(fa0, fb0, acc);  // step 0 of stage k
    __builtin_amdgcn_sched_barrier(0);
    wait_frags(fa1, fb1);
    if (k + 1 < KT) {
      // Stage k + 1 has landed for every wave, and every wave has read stage k: its buffer
      // takes stage k + 4.
      wait_stages<PER>(min(kNStages - 2, KT - 2 - k));
      __builtin_amdgcn_s_barrier();
      if (k + kNStages < KT) issue(k + kNStages);
      const uint32_t nb = ((k + 1) % kNStages) * kStageBytes;
      read_frags(a0 + nb, b0 + nb, fa0, fb0);  // step 0 of stage k + 1
    }
    __builtin_amdgcn_sched_barrier(0);
    mma16(fa1, fb1, acc);  // step 1 of stage k
    __builtin_amdgcn_sched_barrier(0);
    if (k + 1 < KT) wait_frags(fa0, fb0);
  }
  __syncthreads();  // the epilogue reuses the LDS
}

// Eight waves (2 x 4 of 128 x 64) with K staged 64 at a time through two 64 KiB LDS buffers:
// every global -> LDS copy instruction then moves 8 whole 128-byte lines (8 rows x 64 K of a
// K-contiguous operand) instead of 16 half lines, which doubles what the copy path delivers per
// CU. Rows of 128 bytes, the 16-byte chunk c of row r stored at c ^ ((r >> 1) & 7): the 16 rows a
// quarter wave reads at one chunk then cover all 64 banks once. N-contiguous B: 64 K rows of 512
// bytes per stage (the chunk c of row r at c ^ ((r & 3) << 2), as in the 32-deep stages).
//
// A stage runs in four phases of eight MFMAs, one quadrant of the wave's tile (64 x 32) over all
// 64 K each: A0 B0, A0 B1, A1 B0, A1 B1. Every LDS read of a stage is then issued by the second
// phase and done before the third, so the stage's one barrier falls between them, with half of its
// MFMAs ready in registers: the copies of stage k + 2 (into the buffer just read) and the first
// reads of stage k + 1 go out between those MFMAs. Against one K step's fragments at a time, with
// the copies and the next reads issued in a burst after the barrier, before the stage's last MFMAs:
// 4096^3 127 -> 121 us (1,140 TFLOP/s), logits of 2,048 tokens x 32,768 rows 199 -> 186, of 744 x
// 76,544 204 -> 195, the split-K product at 707 tokens 47.8 -> 46.5 (same bits). What is left is
// power and the copies: with zero operands the same 4096^3 takes 83 us (the clock stays up), and
// without copies 8192^3 runs at 1,430 TFLOP/s on random and 2,145 on zero operands.
constexpr int kDK64 = 64;
constexpr int kStage64 = 2 * kBM * kDK64 * 2;  // 64 KiB
constexpr int kSmem64 = 2 * kStage64;          // 128 KiB

// Fragments of one 64-row half of A (2 MFMA tiles) or one 32-column tile of B, all four K steps.
struct FragA {
  u32x4v v[4][2];
};
template <bool KN>
struct FragB;
template <>
struct FragB<false> {
  u32x4v v[4];
  __device__ __forceinline__ f16x8 get(int kk) const { return __builtin_bit_cast(f16x8, v[kk]); }
};
template <>
struct FragB<true> {
  u32x2v lo[4], hi[4];
  __device__ __forceinline__ f16x8 get(int kk) const {
    const u32x4v b = {lo[kk].x, lo[kk].y, hi[kk].x, hi[kk].y};
    return __builtin_bit_cast(f16x8, b);
  }
};

// Every LDS read issued so far has returned; ties the fragments read since the last wait.
__device__ __forceinline__ void wait_set(FragA& f) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(f.v[0][0]), "+v"(f.v[0][1]), "+v"(f.v[1][0]), "+v"(f.v[1][1]),
                 "+v"(f.v[2][0]), "+v"(f.v[2][1]), "+v"(f.v[3][0]), "+v"(f.v[3][1]));
}
__device__ __forceinline__ void wait_set(FragB<false>& f) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.v[0]), "+v"(f.v[1]), "+v"(f.v[2]), "+v"(f.v[3]));
}
__device__ __forceinline__ void wait_set(FragB<true>& f) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(f.lo[0]), "+v"(f.lo[1]), "+v"(f.lo[2]), "+v"(f.lo[3]), "+v"(f.hi[0]),
                 "+v"(f.hi[1]), "+v"(f.hi[2]), "+v"(f.hi[3]));
}

// Wave w of eight's rows (128 wave8_m) and columns (64 wave8_n) of the tile. A wave with none of
// them inside the matrix takes part in the copies and barriers only, and so that the others still
// use four SIMDs (wave w is on SIMD w % 4), a tile that is not whole deals its waves so that those
// of either half of the rows, or of two neighbouring quarters of the columns, are on different
// ones. Such a tile then takes about half the time where its MFMAs count (345 tokens' statistics
// 262 -> 248 us, a training pass at 16 tokens 383 -> 342, at 100 465 -> 435, at 345 675 -> 642; the
// other deal costs a whole tile 0.5%). Leaving out the copies as well gave another 1-3% below 128
// tokens, at seven conditions in the loop.
__device__ __forceinline__ int wave8_m(int wave) { return wave >> 2; }
__device__ __forceinline__ int wave8_n(const GemmArgs& g, const Tile& tl, int wave) {
  const bool whole = tl.m0 + kWM < g.M && tl.n0 + 192 < g.N;
  return (wave & 3) ^ (whole ? 0 : (wave >> 2) << 1);
}

template <bool KN>
__device__ __forceinline__ void mainloop_k64(const GemmArgs& g, const Tile& tl, char* smem,
                                             f32x16 (&acc)[kMT][2]) {
  constexpr int CP = 4;  // copies per wave per operand and stage
  constexpr int PER = 2 * CP;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(t >> 6));
  const int wm = wave8_m(wave), wn = wave8_n(g, tl, wave);
  const int kb = tl.split * g.k_per_split;
  const int ke = min(kb + g.k_per_split, g.K);
  const int KT = ke > kb ? (ke - kb) / kDK64 : 0;
#pragma unroll
  for (int mt = 0; mt < kMT; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = f32x16{};
  if (KT == 0) {
    __syncthreads();
    return;
  }
  // Copies: instruction i of wave w fills bytes 1024 (8 i + w) .. +1024 of the stage's A tile
  // (rows 8 (8 i + w) .. +8; lane l covers row + l/8 at position l%8, i.e. the chunk
  // (l%8) ^ ((row >> 1) & 7)) and the same bytes of the B tile (K-contiguous as A; N-contiguous:
  // K rows 2 (8 i + w) + l/32 of 512 bytes, lane l at position l%32 of its row r, the chunk
  // (l%32) ^ ((r & 3) << 2), columns n0 + 8 chunk .. +8).
  const char* gA = reinterpret_cast<const char*>(g.A);
  const char* gB = reinterpret_cast<const char*>(g.B);
  uint32_t oa[CP], ob[CP];
#pragma unroll
  for (int i = 0; i < CP; ++i) {
    const int row = 8 * (8 * i + wave) + (lane >> 3);
    const int ch = (lane & 7) ^ ((row >> 1) & 7);
    // Rows (columns) past the matrix edge re-read the last one: finite values the epilogues
    // discard.
    const int ra_ = min(tl.m0 + row, g.M - 1);
    oa[i] = static_cast<uint32_t>((ra_ * g.lda + kb + ch * 8) * 2);
    if constexpr (KN) {
      const int krow = 2 * (8 * i + wave) + (lane >> 5);
      const int col = min(tl.n0 + 8 * ((lane & 31) ^ ((krow & 3) << 2)), g.N - 8);
      ob[i] = static_cast<uint32_t>(((kb + krow) * g.ldb + col) * 2);
    } else {
      const int rb_ = min(tl.n0 + row, g.N - 1);
      ob[i] = static_cast<uint32_t>((rb_ * g.ldb + kb + ch * 8) * 2);
    }
  }
  const uint32_t bstep = KN ? static_cast<uint32_t>(kDK64 * g.ldb * 2) : kDK64 * 2;
  auto copy = [&](int k, auto I) {  // copy I of stage k into buffer k % 2
    constexpr int i = decltype(I)::value;
    char* st = smem + (k & 1) * kStage64 + wave * 1024;
    __builtin_amdgcn_global_load_lds(gA + oa[i] + static_cast<uint32_t>(k) * (kDK64 * 2),
                                     (lds_void_ptr)(st + i * 8192), 16, 0, 0);
    __builtin_amdgcn_global_load_lds(gB + ob[i] + static_cast<uint32_t>(k) * bstep,
                                     (lds_void_ptr)(st + kBM * 128 + i * 8192), 16, 0, 0);
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;
  auto issue = [&](int k) {
    copy(k, C0{});
    copy(k, C1{});
    copy(k, C2{});
    copy(k, C3{});
  };
  // Fragment addresses. A: row wm*128 + (l & 31) (+ 32 per MFMA tile: immediate 4096), chunk
  // 2 kk + l/32 at position chunk ^ ((l >> 1) & 7) (the low row bits are those of l). B
  // K-contiguous likewise (rows wn*64 + ...); N-contiguous: lane l of group g = l/16 (j = l%16)
  // reads K row 16 kk + 8 (g/2) + j/4 (+ 4 for the high half), columns wn*64 + 32 nt + 16 (g%2)
  // + 4 (j%4).
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_ptr)smem));
  const int half = lane >> 5;
  const uint32_t c0 = static_cast<uint32_t>((half ^ ((lane >> 1) & 7)) << 4);
  const uint32_t arow = lds0 + (wm * kWM + (lane & 31)) * 128 + c0;  // kk: ^ (kk << 5)
  const uint32_t brow = lds0 + kBM * 128 + (wn * 64 + (lane & 31)) * 128 + c0;
  uint32_t bk[2];
  if constexpr (KN) {
    const int j = lane & 15, nh = (lane >> 4) & 1;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int col = wn * 64 + nt * 32 + 16 * nh + 4 * (j & 3);
      bk[nt] = lds0 + kBM * 128 + (8 * half + (j >> 2)) * kKNRowBytes +
               (((col >> 3) ^ ((j >> 2) << 2)) << 4) + (col & 7) * 2;
    }
  }
  FragA a0, a1;
  FragB<KN> b0, b1;
  auto read_a = [&](FragA& f, uint32_t sb, auto KK, auto H) {
    constexpr int kk = decltype(KK)::value, h = decltype(H)::value;
    const uint32_t a = (arow ^ (kk << 5)) + sb;
    f.v[kk][0] = lds_read16<h * 8192>(a);
    f.v[kk][1] = lds_read16<h * 8192 + 4096>(a);
  };
  auto read_b = [&](FragB<KN>& f, uint32_t sb, auto KK, auto N) {
    constexpr int kk = decltype(KK)::value, nt = decltype(N)::value;
    if constexpr (KN) {
      f.lo[kk] = lds_read8_tr<kk * 16 * kKNRowBytes>(bk[nt] + sb);
      f.hi[kk] = lds_read8_tr<kk * 16 * kKNRowBytes + 4 * kKNRowBytes>(bk[nt] + sb);
    } else {
      f.v[kk] = lds_read16<nt * 4096>((brow ^ (kk << 5)) + sb);
    }
  };
  auto mma = [&](const FragA& fa, const FragB<KN>& fb, auto KK, auto H, auto N) {
    constexpr int kk = decltype(KK)::value, h = decltype(H)::value, nt = decltype(N)::value;
#pragma unroll
    for (int m = 0; m < 2; ++m)
      acc[2 * h + m][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          __builtin_bit_cast(f16x8, fa.v[kk][m]), fb.get(kk), acc[2 * h + m][nt], 0, 0, 0);
  };
  auto each = [&](auto f) {  // the four K steps, kept apart so that what f interleaves stays so
    f(C0{});
    __builtin_amdgcn_sched_barrier(0);
    f(C1{});
    __builtin_amdgcn_sched_barrier(0);
    f(C2{});
    __builtin_amdgcn_sched_barrier(0);
    f(C3{});
    __builtin_amdgcn_sched_barrier(0);
  };
  issue(0);
  if (KT > 1) issue(1);
  if (KT > 1)
    wait_vmcnt<PER>();  // stage 0 landed (this wave's copies)
  else
    wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();  // ... and every wave's
  if (tl.m0 + wm * kWM >= g.M || tl.n0 + wn * 64 >= g.N) {  // the stages' copies and barriers
    for (int k = 0; k + 1 < KT; ++k) {
      wait_vmcnt<0>();
      __builtin_amdgcn_s_barrier();
      if (k + 2 < KT) issue(k + 2);
    }
    __syncthreads();
    return;
  }
  each([&](auto kk) { read_a(a0, 0, kk, C0{}); });
  each([&](auto kk) { read_b(b0, 0, kk, C0{}); });
  wait_set(a0);
  wait_set(b0);
  // MORE: stages beyond this one (0, 1, 2 = two or more: the copies of stage k + 2 go out).
  auto stage = [&](int k, auto MORE) {
    constexpr int more = decltype(MORE)::value;
    const uint32_t sb = (k & 1) * kStage64, sn = sb ^ kStage64;
    each([&](auto kk) {
      read_b(b1, sb, kk, C1{});
      mma(a0, b0, kk, C0{}, C0{});
    });
    wait_set(b1);
    each([&](auto kk) {
      read_a(a1, sb, kk, C1{});
      mma(a0, b1, kk, C0{}, C1{});
    });
    wait_set(a1);
    if constexpr (more > 0) {
      // Stage k + 1 has landed for every wave, and every wave has read stage k: its buffer
      // takes stage k + 2.
      wait_vmcnt<0>();
      __builtin_amdgcn_s_barrier();
    }
    each([&](auto kk) {
      mma(a1, b0, kk, C1{}, C0{});
      if constexpr (more > 0) read_a(a0, sn, kk, C0{});
      if constexpr (more > 1) copy(k + 2, kk);
    });
    if constexpr (more > 0) wait_set(a0);
    each([&](auto kk) {
      if constexpr (more > 0) read_b(b0, sn, kk, C0{});
      mma(a1, b1, kk, C1{}, C1{});
    });
    if constexpr (more > 0) wait_set(b0);
  };
  for (int k = 0; k + 2 < KT; ++k) stage(k, C2{});
  if (KT > 1) stage(KT - 2, C1{});
  stage(KT - 1, C0{});
  __syncthreads();  // the epilogues reuse the LDS
}

__device__ __forceinline__ void mainloop(const GemmArgs& g, const Tile& tl, char* smem,
                                         f32x16 (&acc)[kMT][4]) {
  mainloop_t(g, tl, smem, acc);
}

__device__ __forceinline__ void mainloop(const GemmArgs& g, const Tile& tl, char* smem,
                                         f32x16 (&acc)[kMT][2]) {
  mainloop_k64<false>(g, tl, smem, acc);
}

// The eight-wave mainloop with B stored [K, ldb] N-contiguous.
__device__ __forceinline__ void mainloop_kn(const GemmArgs& g, const Tile& tl, char* smem,
                                            f32x16 (&acc)[kMT][2]) {
  mainloop_k64<true>(g, tl, smem, acc);
}

// Eight waves (two per SIMD): the accumulators of a 128 x 64 wave tile leave room for a second
// wave per SIMD, whose MFMAs run while the first waits on its fragment reads and copies.
constexpr int kThreads8 = 512;

int launch_grid(const GemmArgs& g) {
  const int total = g.tiles_m * g.tiles_n * g.splits;
  return 8 * ((total + 7) / 8);
}

int check_operand(const char* fn, const void* p, int64_t ld, const char* name) {
  if (!p) return fail(RUS_ERR_INVALID, "%s: %s is null", fn, name);
  if (!aligned(p, 16) || ld % 8)
    return fail(RUS_ERR_INVALID, "%s: %s must be 16-byte aligned with a row stride multiple of 8",
                fn, name);
  return RUS_OK;
}

}  // namespace
}  // namespace rus
