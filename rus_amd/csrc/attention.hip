// Varlen causal GQA attention (forward and backward) on packed tokens for gfx950, head_dim 128.
//
// Reference behaviour (solution/ops.py:669-696, _run_packed_sdpa): per packed row, causal scaled
// dot-product attention with softmax scale 1/sqrt(head_dim) and K/V shared by h_q / h_kv query
// heads; its backward is torch's. Layout here: q [N, h_q, 128], k / v [N, h_kv, 128] token-major
// (the RoPE kernel's outputs), rows delimited by cu_seqlens [n_seq + 1] (int32, on the device).
//
// Design (CDNA4, v_mfma_f32_32x32x16_f16; operand / accumulator lane layouts as in mfma_gemm.h):
//   * one block of 4 waves per (row, 32-token block, query head); the waves split the loop over
//     the other operand's 32-token blocks and merge their partials through LDS at the end in a
//     fixed order (softmax partials rescaled by their running maxima);
//   * every operand tile (32 tokens x 128 dims) is copied straight into LDS by
//     global_load_lds_dwordx4 (whole 256-byte rows per 16 lanes; the block's own query tile
//     once, the waves' key / value tiles per loop step) and read from there as 16-byte row
//     fragments or, through ds_read_b64_tr_b16, as transposed fragments: no tile is held in
//     registers in flight, no transposed copy is written, and blocks fit two per CU;
//   * forward computes S^T = K Q^T, so a lane owns one query (column) and 16 of the block's 32
//     keys: the running max / sum and the O rescale are per-lane scalars, and P^T feeds the
//     O^T += V^T P^T product straight from the accumulator registers. An accumulator tile used
//     as an MFMA operand carries its reduction index in the order
//         k(h, i) = 16 s + 8 (i / 4) + 4 h + i % 4      (lane half h, slot i of step s),
//     which the transposed reads produce (two reads of 4 consecutive tokens per fragment);
//   * P and dS are rounded to fp16 for their MFMAs, as flash attention does; O, LSE, dQ, dK, dV
//     accumulate in fp32;
//   * backward: one launch runs the dK / dV blocks (row, key block, query head; fp32 dK / dV
//     partials per query head) and the dQ blocks (row, query block, head); each block forms
//     D = rowsum(dO o O) of the query rows it visits from the dO tile in LDS and O rows loaded
//     with that tile (no separate launch, no D array). The h_q / h_kv partials of a KV group are
//     summed in head order and rounded once, by a second launch or, in the engine's path, by the
//     RoPE backward that packs them (rus_qkv_rope_bwd_mid_parts);
//   * two layouts of both passes, chosen by size (wide() below): the 32-token blocks above, whose
//     waves split the other side's blocks, for batches that would leave the chip idle otherwise;
//     and 128-token blocks (attn_*_wide_kernel), whose four waves share each streamed tile.
#include <math.h>

#include <algorithm>

#include "common.h"

namespace rus {
namespace {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kHD = 128;       // head_dim
constexpr int kBlk = 32;       // tokens per block
constexpr int kW = 4;          // waves per block (one 32x32 head-dim tile each in the merges)
constexpr int kMaxGroup = 8;   // query heads per KV head (GQA group) the backward supports
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kLazy = 8.0f;  // lazy-rescale threshold (log2 units)

struct AttnArgs {
  const f16* q;
  const f16* k;
  const f16* v;
  const f16* o;    // forward output (backward input)
  const f16* dout;
  const int32_t* cu;
  f16* out;        // forward: O; backward kernel 1: dQ
  float* lse;      // [h_q, n_tok], natural log
  float* dk_part;  // [h_q, n_tok, 128]
  float* dv_part;
  f16* dk;         // [n_tok, h_kv, 128]
  f16* dv;
  int64_t n_tok;
  int n_seq, h_q, h_kv;
  int max_blocks;  // backward: blocks per pass (grid y of each pass)
  int n_blocks;    // wide kernels: bound of the 128-token blocks over all rows
  float scale, scale_log2;
};

// 2^x by the hardware instruction (v_exp_f32): 2^-inf = 0; results below the normal range
// flush to zero, far below what the fp16 operands they feed can hold.
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ f32x16 mfma(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Row bounds of row s (clamped to [0, n_tok] and non-decreasing, so a malformed cu_seqlens
// cannot send an access outside the token arrays) and its number of kB-token blocks.
struct RowInfo {
  int a, e, nb;
};

template <int kB>
__device__ __forceinline__ RowInfo row_info(const int32_t* cu, int s, int n_seq, int n_tok) {
  RowInfo r{0, 0, 0};
  if (s < n_seq) {
    r.a = min(max(cu[s], 0), n_tok);
    r.e = min(max(cu[s + 1], r.a), n_tok);
    r.nb = (r.e - r.a + kB - 1) / kB;
  }
  return r;
}

// Index of the n-th set bit of m (n < popcount(m)).
__device__ __forceinline__ int nth_bit(uint64_t m, int n) {
  for (int i = 0; i < n; ++i) m &= m - 1;
  return __ffsll(static_cast<unsigned long long>(m)) - 1;
}

// Block id -> (row start, row end, block start), heaviest blocks first. A row of nb blocks has
// one block of each work level w = 1 .. nb (the number of kB-token blocks on the other side of
// the causal loop): block w - 1 when the work grows towards the row's end (kDiagLast: forward
// and dQ, which loop over the keys up to the diagonal), block nb - w otherwise (dK/dV, which loop
// over the queries from the diagonal on). Ids run over levels from the highest down, rows in
// order within a level, so the longest blocks are dispatched first. Each lane holds one row of
// a 64-row chunk; false if blk is past the last block. Uniform over the block.
template <bool kDiagLast, int kB = kBlk>
__device__ __forceinline__ bool find_block(const int32_t* cu, int n_seq, int n_tok, int blk,
                                           int& start, int& end, int& b0) {
  const int lane = threadIdx.x & 63;
  const int n_chunks = (n_seq + 63) / 64;
  const RowInfo r0 = row_info<kB>(cu, lane, n_seq, n_tok);
  int max_nb = r0.nb;
  for (int c = 1; c < n_chunks; ++c) max_nb = max(max_nb, row_info<kB>(cu, 64 * c + lane, n_seq, n_tok).nb);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) max_nb = max(max_nb, __shfl_xor(max_nb, off, 64));
  for (int w = max_nb; w >= 1; --w) {
    for (int c = 0; c < n_chunks; ++c) {
      const RowInfo r = c == 0 ? r0 : row_info<kB>(cu, 64 * c + lane, n_seq, n_tok);
      const uint64_t mask = __ballot(r.nb >= w);
      const int cnt = __popcll(mask);
      if (blk < cnt) {
        const int src = nth_bit(mask, blk);
        start = __shfl(r.a, src, 64);
        end = __shfl(r.e, src, 64);
        const int nb = __shfl(r.nb, src, 64);
        b0 = start + (kDiagLast ? w - 1 : nb - w) * kB;
        return true;
      }
      blk -= cnt;
    }
  }
  return false;
}

// fp16 operand of k-step s from accumulator registers 8s .. 8s+7.
__device__ __forceinline__ f16x8 frag_acc(const f32x16& c, int s) {
  f16x8 r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = from_f32<f16>(c[8 * s + i]);
  return r;
}

// Accumulator row of register r for lane half h.
__device__ __forceinline__ int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// Partial accumulators of the block's kW waves, summed in a fixed order: every wave stores its
// four 32x32 tiles (the accumulator layout, lane-contiguous), then thread (wave w, lane) reads
// tile w of every wave. buf holds kW * 64 * 64 floats.
__device__ __forceinline__ void park(float* buf, const f32x16 (&acc)[4], int wave, int lane) {
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) buf[(wave * 64 + d * 16 + r) * 64 + lane] = acc[d][r];
}

__device__ __forceinline__ float parked(const float* buf, int w, int tile, int r, int lane) {
  return buf[(w * 64 + tile * 16 + r) * 64 + lane];
}

// fp16 store of the 16 accumulator values of tile d (head dims d*32 + 8 r4 + 4 h + i) of one
// query's row.
__device__ __forceinline__ void store_tile_row(f16* row, const float (&x)[16], int d, int h) {
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    f16x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = from_f32<f16>(x[4 * r4 + i]);
    *reinterpret_cast<f16x4*>(row + d * 32 + 8 * r4 + 4 * h) = w;
  }
}

constexpr int kParkBytes = kW * 64 * 64 * 4;             // 64 KiB
constexpr int kMax(int x, int y) { return x > y ? x : y; }

// ---------------------------------------------------------------------------------------------
// Operand tiles (32 tokens x 128 head dims of Q, dO, K or V) are copied straight from global
// memory into LDS (global_load_lds_dwordx4: 4 rows x 256 contiguous bytes per wave instruction,
// no registers in flight) and read from there both ways: 16-byte row fragments (ds_read_b128)
// and transposed fragments (ds_read_b64_tr_b16), so each tile is loaded once per use.
// ---------------------------------------------------------------------------------------------
constexpr int kTile = kBlk * kHD * 2;  // one 32 x 128 fp16 tile: 8 KiB
typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

// Tiles are row-major, 256 bytes per token row, with the 16-byte chunk c of row r stored at chunk
// c ^ swz(r): a quarter wave's 16-byte fragment reads (16 consecutive rows, one chunk) and a
// half wave's transposing reads (4 consecutive rows x 64 bytes) each cover the 64 banks once.
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// Issues copies i0 .. i0 + n - 1 of the 8 that fill a tile with token rows r0 .. r0 + 31 of a
// [*, stride] head slice (rows clamped into [lo, hi): rows past a row's end repeat its last token,
// finite values that the masks discard). Copy i fills tile rows 4 i .. 4 i + 3; lane l lands at
// row 4 i + l / 16, position l % 16, so it loads the chunk (l % 16) ^ swz(row).
__device__ __forceinline__ void tile_copy(char* tile, const f16* x, int64_t stride, int r0,
                                          int lo, int hi, int i0, int n) {
  const int lane = threadIdx.x & 63;
  for (int i = i0; i < i0 + n; ++i) {
    const int r = 4 * i + (lane >> 4);
    int t = r0 + r;
    t = t < hi ? t : hi - 1;
    t = t < lo ? lo : t;
    const int c = (lane & 15) ^ swz(r);
    __builtin_amdgcn_global_load_lds(x + static_cast<int64_t>(t) * stride + c * 8,
                                     (lds_void_ptr)(tile + i * 1024), 16, 0, 0);
  }
}

// s_waitcnt vmcnt(0): this wave's tile copies have landed (expcnt / lgkmcnt not waited on).
__device__ __forceinline__ void wait_copies() {
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
}

// This wave's LDS reads have returned: a copy may now overwrite the tiles they read.
__device__ __forceinline__ void wait_tile_reads() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), vmcnt / expcnt not waited on
  asm volatile("" ::: "memory");
}

// 16-byte fragment: head dims 8 c .. 8 c + 7 of tile row r.
__device__ __forceinline__ f16x8 tile_frag(const char* tile, int r, int c) {
  return *reinterpret_cast<const f16x8*>(tile + r * 256 + ((c ^ swz(r)) << 4));
}

// Transposed fragment of k-step s in the accumulator order k(h, i) = 16 s + 8 (i / 4) + 4 h +
// i % 4, head-dim tile d: lane l holds x[k(h, i)][32 d + l % 32], i = 0..7. ds_read_b64_tr_b16
// gives lane i of each 16-lane group element i % 4 of the 8 bytes read by lanes i / 4 + 4 e of
// the group, so lane j of a group reads row k0 + j / 4, head dims n0 + 4 (j % 4) .. +4, and lane i
// receives x[k0 + e][n0 + i], e = 0..3 (k0 = 16 s + 4 h, then + 8).
__device__ __forceinline__ f16x8 tile_frag_t(const char* tile, int s, int d) {
  const int lane = threadIdx.x & 63, j = lane & 15;
  const int col = 32 * d + (lane & 16) + 4 * (j & 3);
  const int r0 = 16 * s + 4 * (lane >> 5) + (j >> 2), r1 = r0 + 8;
  const int cb = (col & 7) * 2;
  const v4i16 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_v4i16*)(tile + r0 * 256 + (((col >> 3) ^ swz(r0)) << 4) + cb));
  const v4i16 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_v4i16*)(tile + r1 * 256 + (((col >> 3) ^ swz(r1)) << 4) + cb));
  const f16x4 a = __builtin_bit_cast(f16x4, x0), b = __builtin_bit_cast(f16x4, x1);
  return f16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}


// ---------------------------------------------------------------------------------------------
// Forward: O = softmax(Q K^T * scale, causal) V and LSE. Block = (row, query block, head); its
// kW waves take key blocks w, w + kW, ... with their own running max / sum, merged at the end.
// ---------------------------------------------------------------------------------------------
// At most 256 registers per lane (no spills) and 72 KiB of LDS (the block's Q tile, each wave's
// K and V tiles): two blocks share a CU, so the grid of (query block, head) blocks fits the chip
// in one round and one block's loads overlap another's MFMAs.
__global__ __launch_bounds__(64 * kW) __attribute__((amdgpu_waves_per_eu(2, 2))) void
attn_fwd_kernel(AttnArgs a) {
  constexpr int kBytes = kMax((1 + 2 * kW) * kTile, kParkBytes + kW * 64 * 4);
  __shared__ __attribute__((aligned(16))) char smem[kBytes];
  int start, end, q0;
  if (!find_block<true>(a.cu, a.n_seq, static_cast<int>(a.n_tok), blockIdx.y, start, end, q0)) return;
  const int head = blockIdx.x, g = head / (a.h_q / a.h_kv);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int64_t sq = static_cast<int64_t>(a.h_q) * kHD, skv = static_cast<int64_t>(a.h_kv) * kHD;
  const f16* kh = a.k + g * kHD;
  const f16* vh = a.v + g * kHD;
  char* qt = smem;
  char* kt = smem + (1 + 2 * wave) * kTile;
  char* vt = kt + kTile;

  const int qi = q0 + col;  // this lane's query
  const int nk = (q0 - start) / kBlk + 1;  // key blocks up to and including the diagonal
  tile_copy(qt, a.q + head * kHD, sq, q0, start, end, 2 * wave, 2);  // the 8 copies, 2 per wave
  if (wave < nk) {
    const int k0 = start + wave * kBlk;
    tile_copy(kt, kh, skv, k0, start, end, 0, 8);
    tile_copy(vt, vh, skv, k0, start, end, 0, 8);
  }
  wait_copies();
  __syncthreads();  // every wave's share of the Q tile has landed
  f16x8 qf[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) qf[s] = tile_frag(qt, col, 2 * s + h);
  f32x16 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = f32x16{};
  float m = -INFINITY, l = 0.0f;
  for (int kb = wave; kb < nk; kb += kW) {
    const int k0 = start + kb * kBlk;
    f32x16 st = f32x16{};  // S^T = K Q^T: rows keys, columns queries
#pragma unroll
    for (int s = 0; s < 8; ++s) st = mfma(tile_frag(kt, col, 2 * s + h), qf[s], st);
    // Only the diagonal block holds keys past the query or past the row's end.
    float mx = -INFINITY;
    if (kb == nk - 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + acc_row(r, h);
        st[r] = (key <= qi && key < end) ? st[r] * a.scale_log2 : -INFINITY;
        mx = fmaxf(mx, st[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        st[r] *= a.scale_log2;
        mx = fmaxf(mx, st[r]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));  // finite: key k0 <= q0 <= qi is always allowed
    // Lazy rescaling: the reference point m moves only when a block's maximum exceeds it by
    // more than 8 (log2 units), so p = 2^(s - m) <= 256 (exact in range for fp16) and O and l
    // share one reference, leaving O / l unchanged; the rescale of O is a wave-uniform branch
    // that is rarely taken after the first block.
    const bool bump = mx > m + kLazy;
    if (__ballot(bump)) {
      const float mn = bump ? mx : m;
      const float alpha = exp2_raw(m - mn);  // 0 on the first block (m = -inf)
      l *= alpha;
      m = mn;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = exp2_raw(st[r] - m);
      st[r] = p;
      rs += p;
    }
    rs += __shfl_xor(rs, 32, 64);
    l += rs;
    const f16x8 p0 = frag_acc(st, 0), p1 = frag_acc(st, 1);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      o[d] = mfma(tile_frag_t(vt, 0, d), p0, o[d]);  // O^T += V^T P^T
      o[d] = mfma(tile_frag_t(vt, 1, d), p1, o[d]);
    }
    if (kb + kW < nk) {  // the wave's next key block into its tiles
      wait_tile_reads();
      const int k1 = k0 + kW * kBlk;
      tile_copy(kt, kh, skv, k1, start, end, 0, 8);
      tile_copy(vt, vh, skv, k1, start, end, 0, 8);
      wait_copies();
    }
  }
  __syncthreads();  // all waves are done with their V^T tiles; the space is reused below
  float* buf = reinterpret_cast<float*>(smem);
  float* ml = buf + kW * 64 * 64;  // per wave: m of columns 0..31, then l
  park(buf, o, wave, lane);
  if (h == 0) {
    ml[wave * 64 + col] = m;
    ml[wave * 64 + 32 + col] = l;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < kW; ++w) M = fmaxf(M, ml[w * 64 + col]);
  float f[kW], L = 0.0f;
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const float mw = ml[w * 64 + col];
    f[w] = exp2_raw(mw - M);  // 0 for a wave without key blocks (mw = -inf)
    L += ml[w * 64 + 32 + col] * f[w];
  }
  if (qi < end) {
    const float inv = 1.0f / L;
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float acc = 0.0f;
#pragma unroll
      for (int w = 0; w < kW; ++w) acc += parked(buf, w, wave, r, lane) * f[w];
      x[r] = acc * inv;
    }
    store_tile_row(a.out + qi * sq + head * kHD, x, wave, h);
    if (wave == 0 && h == 0) a.lse[head * a.n_tok + qi] = (M + log2f(L)) * kLn2;
  }
}

// ---------------------------------------------------------------------------------------------
// Backward, on the LDS tiles: row fragments for S = Q K^T and dP = dO V^T, transposed fragments
// for dV += P^T dO, dK += dS^T Q and dQ^T += K^T dS^T. D = rowsum(dO o O) is formed by each block for
// the query rows it visits (below).
// ---------------------------------------------------------------------------------------------
// Waves per backward block: 4 (80 KiB of LDS and at most 256 registers, so two blocks share a
// CU and one block's waits overlap the other's work; 8 waves in one block per CU ran 13% slower).
constexpr int kWB = 4;
static_assert(kWB == 4 || kWB == 8, "4 or 8 waves per backward block");
constexpr int kCopiesPerWave = 8 / kWB;  // a shared tile's 8 copies over the block's waves
constexpr int kRegsPerWave = 64 / kWB;   // accumulator registers each wave sums in the merge
// LDS of a backward block: 2 shared tiles + 2 per wave; the merge reuses it as a buffer of every
// wave's four 32x32 fp32 accumulator tiles.
constexpr int kBwdBytes = (2 + 2 * kWB) * kTile;
static_assert(kWB * 64 * 64 * 4 <= kBwdBytes, "the merge buffer fits the tiles' LDS");

// Every wave's four 32x32 fp32 tiles into the merge buffer (the accumulator layout,
// lane-contiguous); thread (wave w, lane) then sums tile w % 4, registers kRegsPerWave (w / 4)
// .. + kRegsPerWave, over the waves in wave order.
__device__ __forceinline__ void park_b(float* buf, const f32x16 (&acc)[4], int wave, int lane) {
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) buf[(wave * 64 + d * 16 + r) * 64 + lane] = acc[d][r];
}

__device__ __forceinline__ void merge_b(const float* buf, int wave, int lane,
                                        float (&x)[kRegsPerWave]) {
  const int tile = wave & 3, r0 = kRegsPerWave * (wave >> 2);
#pragma unroll
  for (int r = 0; r < kRegsPerWave; ++r) {
    float acc = 0.0f;
#pragma unroll
    for (int w = 0; w < kWB; ++w) acc += buf[(w * 64 + tile * 16 + r0 + r) * 64 + lane];
    x[r] = acc;
  }
}

// D = rowsum(dO o O) of the 32 query rows of a block, formed where it is used: the dO tile is in
// LDS and the O rows come in registers (ORows, loaded with the tiles). Pass p covers rows 4 p ..
// 4 p + 3: lane l takes row 4 p + l / 16, head dims 8 (l % 16) .. + 8, sums their 8 fp32 products
// of fp16 values in dim order, then the 16 lanes of a row add by a butterfly (xor 8, 4, 2, 1);
// every lane of the group then holds the row's D. Rows past the row's end repeat its last token
// (as the tiles do), so they hold that token's D.
struct ORows {
  f16x8 v[8];
};

__device__ __forceinline__ void load_o_rows(ORows& o, const f16* oh, int64_t stride, int r0,
                                            int lo, int hi) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    int t = r0 + 4 * p + (lane >> 4);
    t = t < hi ? t : hi - 1;
    t = t < lo ? lo : t;
    o.v[p] = *reinterpret_cast<const f16x8*>(oh + static_cast<int64_t>(t) * stride +
                                             8 * (lane & 15));
  }
}

// x of the lane N places further round its 16-lane row (DPP row_ror: a VALU move, no LDS).
template <int N>
__device__ __forceinline__ float row_ror(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x),
                                                               0x120 + N, 0xF, 0xF, false));
}

// The butterfly adds lane c's sum to lane c ^ 8's, then c ^ 4's, c ^ 2's, c ^ 1's. After the
// step with 8 a lane's sum depends on c mod 8 only, so the lane c + 4 (mod 16) holds what c ^ 4
// holds; likewise for 2 and 1: rotations give the same sums as the xor exchanges.
__device__ __forceinline__ float row_dsum(const ORows& o, const char* dt, int p) {
  const int lane = threadIdx.x & 63;
  const f16x8 y = tile_frag(dt, 4 * p + (lane >> 4), lane & 15);
  float acc = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc += static_cast<float>(o.v[p][e]) * static_cast<float>(y[e]);
  acc += row_ror<8>(acc);
  acc += row_ror<4>(acc);
  acc += row_ror<2>(acc);
  acc += row_ror<1>(acc);
  return acc;
}

// D of the rows this lane's accumulator registers cover (register r: row acc_row(r, h)).
__device__ __forceinline__ void dsum_acc_rows(const ORows& o, const char* dt, int h,
                                              float (&d)[16]) {
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const float s = row_dsum(o, dt, p);
    // rows 4 p + g sit in lanes 16 g .. 16 g + 15; acc_row(4 j + g, h) = 4 (2 j + h) + g, so
    // the lanes of half h = p % 2 take them as registers 4 (p / 2) + g
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float v = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s), 16 * g));
      if ((p & 1) == h) d[4 * (p >> 1) + g] = v;
    }
  }
}

// D of tile row c (this lane's query column in the dQ blocks).
__device__ __forceinline__ float dsum_row(const ORows& o, const char* dt, int c) {
  float d = 0.0f;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const float s = __shfl(row_dsum(o, dt, p), 16 * (c & 3), 64);
    if ((c >> 2) == p) d = s;
  }
  return d;
}

// dQ = scale * dS K. Block = (row, query block, head): the Q and dO tiles of its 32 queries are
// shared; the kWB waves take key blocks w, w + kWB, ... (K and V tiles of their own) and their
// dQ partials are summed in wave order at the end.
__device__ __forceinline__ void attn_bwd_dq_block(const AttnArgs& a, int blk, char* smem) {
  int start, end, q0;
  if (!find_block<true>(a.cu, a.n_seq, static_cast<int>(a.n_tok), blk, start, end, q0)) return;
  const int head = blockIdx.x, g = head / (a.h_q / a.h_kv);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int64_t sq = static_cast<int64_t>(a.h_q) * kHD, skv = static_cast<int64_t>(a.h_kv) * kHD;
  const f16* kh = a.k + g * kHD;
  const f16* vh = a.v + g * kHD;
  char* qt = smem;
  char* dt = smem + kTile;
  char* kt = smem + (2 + 2 * wave) * kTile;
  char* vt = kt + kTile;
  const int nk = (q0 - start) / kBlk + 1;
  tile_copy(qt, a.q + head * kHD, sq, q0, start, end, kCopiesPerWave * wave, kCopiesPerWave);
  tile_copy(dt, a.dout + head * kHD, sq, q0, start, end, kCopiesPerWave * wave, kCopiesPerWave);
  if (wave < nk) {
    const int k0 = start + wave * kBlk;
    tile_copy(kt, kh, skv, k0, start, end, 0, 8);
    tile_copy(vt, vh, skv, k0, start, end, 0, 8);
  }
  ORows orow;
  load_o_rows(orow, a.o + head * kHD, sq, q0, start, end);
  const int qi = q0 + col, qr = qi < end ? qi : end - 1;
  const float lse2 = a.lse[head * a.n_tok + qr] * kLog2e;
  wait_copies();
  __syncthreads();  // every wave's share of the Q and dO tiles has landed
  const float dsum = dsum_row(orow, dt, col);  // D of this lane's query (tile row col)

  f32x16 dq[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) dq[d] = f32x16{};
  for (int kb = wave; kb < nk; kb += kWB) {
    const int k0 = start + kb * kBlk;
    f32x16 st = f32x16{}, dp = f32x16{};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      st = mfma(tile_frag(kt, col, 2 * s + h), tile_frag(qt, col, 2 * s + h), st);  // S^T = K Q^T
      dp = mfma(tile_frag(vt, col, 2 * s + h), tile_frag(dt, col, 2 * s + h), dp);  // dP^T = V dO^T
    }
    if (kb == nk - 1) {  // diagonal block: causal and row-end mask
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + acc_row(r, h);
        const float p = exp2_raw(st[r] * a.scale_log2 - lse2);
        st[r] = (key <= qi && key < end) ? p * (dp[r] - dsum) : 0.0f;  // dS^T
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) st[r] = exp2_raw(st[r] * a.scale_log2 - lse2) * (dp[r] - dsum);
    }
    const f16x8 s0 = frag_acc(st, 0), s1 = frag_acc(st, 1);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      dq[d] = mfma(tile_frag_t(kt, 0, d), s0, dq[d]);  // dQ^T += K^T dS^T
      dq[d] = mfma(tile_frag_t(kt, 1, d), s1, dq[d]);
    }
    if (kb + kWB < nk) {  // the wave's next key block into its tiles
      wait_tile_reads();
      const int k1 = k0 + kWB * kBlk;
      tile_copy(kt, kh, skv, k1, start, end, 0, 8);
      tile_copy(vt, vh, skv, k1, start, end, 0, 8);
      wait_copies();
    }
  }
  __syncthreads();  // every wave is done with the tiles; the space becomes the merge buffer
  float* buf = reinterpret_cast<float*>(smem);
  park_b(buf, dq, wave, lane);
  __syncthreads();
  if (qi < end) {
    float x[kRegsPerWave];
    merge_b(buf, wave, lane, x);
    // Register 4 r4 + i of tile d holds head dim 32 d + 8 r4 + 4 h + i.
    const int d = wave & 3, r4b = (kRegsPerWave / 4) * (wave >> 2);
    f16* row = a.out + qi * sq + head * kHD;
#pragma unroll
    for (int r4 = 0; r4 < kRegsPerWave / 4; ++r4) {
      f16x4 w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = from_f32<f16>(x[4 * r4 + i] * a.scale);
      *reinterpret_cast<f16x4*>(row + d * 32 + 8 * (r4b + r4) + 4 * h) = w;
    }
  }
}

// This query head's dK = scale * dS^T Q and dV = P^T dO for one 32-key block, fp32. Block = (row,
// key block, head): the K and V tiles are shared; the kWB waves take query blocks (Q and dO tiles
// of their own). Each query head stores its fp32 partials; attn_group_sum_kernel or the RoPE
// backward adds a KV group's.
__device__ __forceinline__ void attn_bwd_dkdv_block(const AttnArgs& a, int blk, char* smem) {
  int start, end, k0;
  if (!find_block<false>(a.cu, a.n_seq, static_cast<int>(a.n_tok), blk, start, end, k0)) return;
  const int head = blockIdx.x, g = head / (a.h_q / a.h_kv);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int64_t sq = static_cast<int64_t>(a.h_q) * kHD, skv = static_cast<int64_t>(a.h_kv) * kHD;
  const f16* qh = a.q + head * kHD;
  const f16* doh = a.dout + head * kHD;
  const float* lse = a.lse + head * a.n_tok;
  const f16* oh = a.o + head * kHD;
  char* kt = smem;
  char* vt = smem + kTile;
  char* qt = smem + (2 + 2 * wave) * kTile;
  char* dt = qt + kTile;
  const int nq = (end - k0 + kBlk - 1) / kBlk;  // query blocks from the diagonal to the row end
  tile_copy(kt, a.k + g * kHD, skv, k0, start, end, kCopiesPerWave * wave, kCopiesPerWave);
  tile_copy(vt, a.v + g * kHD, skv, k0, start, end, kCopiesPerWave * wave, kCopiesPerWave);
  ORows orow;  // the O rows of the wave's next query block, loaded with its tiles
  if (wave < nq) {
    const int q0 = k0 + wave * kBlk;
    tile_copy(qt, qh, sq, q0, start, end, 0, 8);
    tile_copy(dt, doh, sq, q0, start, end, 0, 8);
    load_o_rows(orow, oh, sq, q0, start, end);
  }
  const int kj = k0 + col;  // this lane's key (column of S = Q K^T)
  wait_copies();
  __syncthreads();  // every wave's share of the K and V tiles has landed
  // D of the query rows of this lane's registers, for the wave's current query block; formed
  // once its dO tile and O rows have landed, so the O rows are not held across the products
  float dsum[16] = {};
  if (wave < nq) dsum_acc_rows(orow, dt, h, dsum);

  f32x16 dk[4], dv[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    dk[d] = f32x16{};
    dv[d] = f32x16{};
  }
  for (int qb = wave; qb < nq; qb += kWB) {
    const int q0 = k0 + qb * kBlk;
    f32x16 st = f32x16{}, dp = f32x16{};
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      st = mfma(tile_frag(qt, col, 2 * s + h), tile_frag(kt, col, 2 * s + h), st);  // S = Q K^T
      dp = mfma(tile_frag(dt, col, 2 * s + h), tile_frag(vt, col, 2 * s + h), dp);  // dP = dO V^T
    }
    // Query rows past the row's end (last block) and before the key (diagonal block) are
    // masked; key columns past the row's end only feed dK / dV rows that are not written.
    const bool edge = q0 == k0 || q0 + kBlk > end;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int qi = q0 + acc_row(r, h);
      const int qc = qi < end ? qi : end - 1;
      float p = exp2_raw(st[r] * a.scale_log2 - lse[qc] * kLog2e);
      if (edge) p = (kj <= qi && qi < end) ? p : 0.0f;
      st[r] = p;                         // P
      dp[r] = p * (dp[r] - dsum[r]);     // dS
    }
    const f16x8 p0 = frag_acc(st, 0), p1 = frag_acc(st, 1);
    const f16x8 s0 = frag_acc(dp, 0), s1 = frag_acc(dp, 1);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      dv[d] = mfma(p0, tile_frag_t(dt, 0, d), dv[d]);  // dV += P^T dO
      dv[d] = mfma(p1, tile_frag_t(dt, 1, d), dv[d]);
      dk[d] = mfma(s0, tile_frag_t(qt, 0, d), dk[d]);  // dK += dS^T Q
      dk[d] = mfma(s1, tile_frag_t(qt, 1, d), dk[d]);
    }
    if (qb + kWB < nq) {  // the wave's next query block into its tiles
      wait_tile_reads();
      const int q1 = q0 + kWB * kBlk;
      tile_copy(qt, qh, sq, q1, start, end, 0, 8);
      tile_copy(dt, doh, sq, q1, start, end, 0, 8);
      load_o_rows(orow, oh, sq, q1, start, end);
      wait_copies();
      dsum_acc_rows(orow, dt, h, dsum);
    }
  }
  // Sum the waves' partials (dK, then dV through the same buffer) and store this head's fp32
  // partial. Rows are keys (accumulator rows), columns head dims (lanes); thread (wave w, lane)
  // writes head-dim tile w % 4, key rows of registers kRegsPerWave (w / 4) .. + kRegsPerWave.
  float* buf = reinterpret_cast<float*>(smem);
  const int dt4 = wave & 3, rb = kRegsPerWave * (wave >> 2);
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    __syncthreads();
    park_b(buf, pass == 0 ? dk : dv, wave, lane);
    __syncthreads();
    float x[kRegsPerWave];
    merge_b(buf, wave, lane, x);
    float* dst = pass == 0 ? a.dk_part : a.dv_part;
    const float sc = pass == 0 ? a.scale : 1.0f;
#pragma unroll
    for (int r = 0; r < kRegsPerWave; ++r) {
      const int key = k0 + acc_row(rb + r, h);
      if (key < end)
        store_partial(dst + (static_cast<int64_t>(head) * a.n_tok + key) * kHD + dt4 * 32 + col,
                      x[r] * sc);
    }
  }
}

// Both backward passes in one launch: blocks y < max_blocks are dK/dV blocks (the heavier ones,
// dispatched first), the rest dQ blocks.
__global__ __launch_bounds__(64 * kWB) __attribute__((amdgpu_waves_per_eu(2, 2))) void
attn_bwd_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[kBwdBytes];
  if (static_cast<int>(blockIdx.y) < a.max_blocks)
    attn_bwd_dkdv_block(a, blockIdx.y, smem);
  else
    attn_bwd_dq_block(a, blockIdx.y - a.max_blocks, smem);
}

// ---------------------------------------------------------------------------------------------
// Wide kernels, for batches with enough 128-token blocks to fill the chip: a block takes 128 tokens
// of one side (4 waves of 32, their fragments in registers) and streams the other side's 32-token
// tiles through double-buffered LDS, each tile copied once for all four waves while the previous
// one is used. The 32-token blocks copy 16 KiB per wave and 32 x 32 score tile and wait for it
// (9 TB/s of L2 reads at 8,161 tokens, and a memory latency per tile); here the copies are a
// quarter of that and off the critical path, and the LDS reads (16 KiB per wave and tile forward,
// 24-32 KiB backward, 128 B/clock per CU) and the exponentials bound it beside the MFMAs. Measured
// at 8,161 tokens in rows of 377 to 2,048, 12 / 2 heads: forward 129 -> 68 us (620 TFLOP/s of the
// causal half), backward with partials 398 -> 186, with the group sum 440 -> 204.
// ---------------------------------------------------------------------------------------------
constexpr int kWide = 128;  // tokens per block

// Block id -> (block index, head): the query heads of a KV group that work on one block index take
// ids 8 apart, i.e. one XCD (ids go round robin over the 8), so they read their shared K / V tiles
// from one L2. False past the last block.
__device__ __forceinline__ bool wide_item(const AttnArgs& a, int n_blocks, int& blk, int& head) {
  const int grp = a.h_q / a.h_kv, chunk = 8 * grp;
  const int t = blockIdx.x / chunk, r = blockIdx.x % chunk;
  const int item = t * chunk + (r & 7) * grp + (r >> 3);
  blk = item / a.h_q;
  head = item % a.h_q;
  return blk < n_blocks;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// This wave's two of the 8 copies that fill a shared tile (rows 8 wave .. + 8; see tile_copy for the
// layout). The tile's first row is a uniform pointer, so a lane's offsets are the same for every
// whole tile; rows past the row's end repeat its last token.
struct TileLane {
  int row[2];      // tile row of copy i
  uint32_t ch[2];  // byte offset of its chunk within the row
  uint32_t off[2];
  uint32_t stride;  // bytes per token

  __device__ __forceinline__ TileLane(int wave, int lane, int64_t stride_el)
      : stride(static_cast<uint32_t>(stride_el) * 2) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      row[i] = 8 * wave + 4 * i + (lane >> 4);
      ch[i] = ((lane & 15) ^ swz(row[i])) << 4;
      off[i] = row[i] * stride + ch[i];
    }
  }

  __device__ __forceinline__ uint32_t at(int i, int rows) const {  // rows: tokens left in the row
    return rows >= kBlk ? off[i] : min(row[i], rows - 1) * stride + ch[i];
  }

  // Copies the tile whose first row is x (uniform), with `rows` (>= 1) tokens left, into LDS. The
  // builtin's LDS target must be one of two __shared__ arrays of its own, so that the compiler
  // knows which LDS reads have to wait for it.
  __device__ __forceinline__ void copy(char* tile, int wave, const f16* x, int rows) const {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const char*>(x) + at(i, rows),
                                       (lds_void_ptr)(tile + (2 * wave + i) * 1024), 16, 0, 0);
  }
};

// A lane's LDS offsets for the fragments of a 32-row tile in tile_frag's and tile_frag_t's layout:
// both are one base per lane, changed by step and head-dim tile in a few bits only. The empty asm
// keeps the compiler from holding all sixteen combinations in registers across the loop (the
// dK / dV blocks need every register; an exclusive or per read is cheap).
struct FragLane {
  uint32_t row, tr;

  __device__ __forceinline__ explicit FragLane(int lane) {
    const int c = lane & 31, h = lane >> 5, j = lane & 15, r0 = 4 * h + (j >> 2);
    row = c * 256 + ((h ^ swz(c)) << 4);
    tr = r0 * 256 + (((((lane >> 4) & 1) * 2 + ((j & 3) >> 1)) ^ swz(r0)) << 4) + (j & 1) * 8;
  }
  __device__ __forceinline__ FragLane fresh() const {
    FragLane f = *this;
    asm("" : "+v"(f.row), "+v"(f.tr));
    return f;
  }
  // tile_frag(tile, lane % 32, 2 s + lane / 32)
  __device__ __forceinline__ f16x8 frag(const char* tile, int s) const {
    return *reinterpret_cast<const f16x8*>(tile + (row ^ (s << 5)));
  }
  // tile_frag_t(tile, s, d): row r0 + 8 differs from r0 in one bit of the swizzle
  __device__ __forceinline__ f16x8 frag_t(const char* tile, int s, int d) const {
    const v4i16 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_v4i16*)(tile + (tr ^ (d << 6)) + s * 4096));
    const v4i16 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_v4i16*)(tile + (tr ^ (d << 6) ^ 32) + s * 4096 + 2048));
    const f16x4 a = __builtin_bit_cast(f16x4, x0), b = __builtin_bit_cast(f16x4, x1);
    return f16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  }
};

// Every copy of this wave has landed and every LDS read of it has returned, then the block's barrier:
// the buffer just filled may be read, the buffer just read may be filled.
__device__ __forceinline__ void stage_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
  __syncthreads();
}

// The values of lanes l and l ^ 32 (in some order).
__device__ __forceinline__ float2 half_pair(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return float2{__builtin_bit_cast(float, static_cast<uint32_t>(p[0])),
                __builtin_bit_cast(float, static_cast<uint32_t>(p[1]))};
}

// fp16 row of one token, head dims 32 d + 8 r4 + 4 h + i from x[d][4 r4 + i] * f: the lane pair
// (l, l ^ 32) exchanges halves so that each stores 16 contiguous bytes.
__device__ __forceinline__ void store_row(f16* row, const f32x16 (&x)[4], float f, int h,
                                          bool valid) {
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f16x4 w0, w1;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w0[i] = from_f32<f16>(x[d][8 * b + i] * f);
        w1[i] = from_f32<f16>(x[d][8 * b + 4 + i] * f);
      }
      const u32x2 a = __builtin_bit_cast(u32x2, w0), c = __builtin_bit_cast(u32x2, w1);
      const auto p0 = __builtin_amdgcn_permlane32_swap(a.x, c.x, false, false);
      const auto p1 = __builtin_amdgcn_permlane32_swap(a.y, c.y, false, false);
      const u32x4 o = {static_cast<uint32_t>(p0[0]), static_cast<uint32_t>(p1[0]),
                       static_cast<uint32_t>(p0[1]), static_cast<uint32_t>(p1[1])};
      if (valid) *reinterpret_cast<u32x4*>(row + 32 * d + 16 * b + 8 * h) = o;
    }
}

// acc + the eight values of x, sums in fp32.
__device__ __forceinline__ float sum8(f16x8 x, float acc) {
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  const f16x2 one = {1, 1};
#pragma unroll
  for (int i = 0; i < 8; i += 2)
    acc = __builtin_amdgcn_fdot2(f16x2{x[i], x[i + 1]}, one, acc, false);
  return acc;
}

// Forward on 32 NT keys (tiles kt, kt + kTile; the last one holds the diagonal when `diag`). A query
// has one reference m here, where the 32-token blocks' four waves have one each and so round four of
// its largest P to exactly 1. To be as accurate, m is the running maximum at every step (moved
// lazily, the later large P took arbitrary roundings), and O is divided by lr, the sum of the rounded
// P, in which their common rounding cancels (l, of the unrounded, gives the lse). Error of O / dQ
// against float64, 16 rows of 512, scores of deviation 1 and 3: 32-token blocks 2.44e-4 / 3.12e-4 and
// 2.14e-4 / 6.69e-4, lazily with l 2.51 / 3.12 and 2.33 / 7.13, lazily with lr 2.49 / 3.11 and 2.09 /
// 6.56, this 2.44 / 3.11 and 2.06 / 6.51; rows of 2,048 64 us lazily with l, 68 this.
template <int NT>
__device__ __forceinline__ void fwd_keys(const FragLane& fl, const char* kt, const char* vt, const f16x8 (&qf)[8],
                                         f32x16 (&o)[4], float& m, float& l, float& lr, float sl2,
                                         bool diag, int k0, int qi, int end, int h) {
  f32x16 st[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    st[n] = f32x16{};
#pragma unroll
    for (int s = 0; s < 8; ++s)
      st[n] = mfma(fl.frag(kt + n * kTile, s), qf[s], st[n]);  // S^T = K Q^T
  }
  if (diag) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = k0 + 32 * (NT - 1) + acc_row(r, h);
      st[NT - 1][r] = (key <= qi && key < end) ? st[NT - 1][r] : -INFINITY;
    }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[n][r]);
  const float2 mp = half_pair(mx);
  mx = fmaxf(mp.x, mp.y) * sl2;  // scale > 0
  if (__ballot(mx > m)) {
    const float mn = fmaxf(m, mx);
    const float alpha = exp2_raw(m - mn);
    l *= alpha;
    lr *= alpha;
    m = mn;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    float rs = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = exp2_raw(__builtin_fmaf(st[n][r], sl2, -m));
      st[n][r] = p;
      rs += p;
    }
    l += rs;  // this lane's 16 keys; the other half's join at the end
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const f16x8 p0 = frag_acc(st[n], 0), p1 = frag_acc(st[n], 1);
    lr = sum8(p1, sum8(p0, lr));
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      o[d] = mfma(fl.frag_t(vt + n * kTile, 0, d), p0, o[d]);  // O^T += V^T P^T
      o[d] = mfma(fl.frag_t(vt + n * kTile, 1, d), p1, o[d]);
    }
  }
}

constexpr int kFwdTiles = 2;  // key tiles per stage

__global__ __launch_bounds__(64 * kW) __attribute__((amdgpu_waves_per_eu(2, 2))) void
attn_fwd_wide_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) char buf0[2 * kFwdTiles * kTile];
  __shared__ __attribute__((aligned(16))) char buf1[2 * kFwdTiles * kTile];
  int blk, head, start, end, q0;
  if (!wide_item(a, a.n_blocks, blk, head)) return;
  const int n_tok = static_cast<int>(a.n_tok);
  if (!find_block<true, kWide>(a.cu, a.n_seq, n_tok, blk, start, end, q0)) return;
  start = __builtin_amdgcn_readfirstlane(start);
  end = __builtin_amdgcn_readfirstlane(end);
  q0 = __builtin_amdgcn_readfirstlane(q0);
  const int g = head / (a.h_q / a.h_kv);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int64_t sq = static_cast<int64_t>(a.h_q) * kHD, skv = static_cast<int64_t>(a.h_kv) * kHD;
  const f16* kh = a.k + start * skv + g * kHD;  // the row's first token
  const f16* vh = a.v + start * skv + g * kHD;
  const int qw = q0 + 32 * wave, qi = qw + col;  // this wave's first query, this lane's
  const int last = min(q0 + kWide, end) - 1;
  const int tiles = (last - start) / 32 + 1;            // key tiles of the block
  const int mine = qw < end ? (qw - start) / 32 + 1 : 0;  // and of this wave
  const int stages = (tiles + kFwdTiles - 1) / kFwdTiles;

  const TileLane tl(wave, lane, skv);
  const FragLane fl0(lane);
  auto copy = [&](char* dst, int j) {
#pragma unroll
    for (int n = 0; n < kFwdTiles; ++n) {
      const int t = kFwdTiles * j + n;
      if (t >= tiles) break;
      const int rows = end - start - 32 * t;
      tl.copy(dst + n * kTile, wave, kh + 32 * t * skv, rows);
      tl.copy(dst + (kFwdTiles + n) * kTile, wave, vh + 32 * t * skv, rows);
    }
  };
  copy(buf0, 0);
  f16x8 qf[8];
  const f16* qrow = a.q + static_cast<int64_t>(min(qi, end - 1)) * sq + head * kHD;
#pragma unroll
  for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const f16x8*>(qrow + 8 * (2 * s + h));
  f32x16 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = f32x16{};
  float m = -INFINITY, l = 0.0f, lr = 0.0f;
  stage_barrier();
  auto stage = [&](const char* cur, char* next, int j) {
    if (j + 1 < stages) copy(next, j + 1);
    const char* vt = cur + kFwdTiles * kTile;
    const FragLane fl = fl0.fresh();
    const int left = mine - kFwdTiles * j;  // this wave's tiles from here on (wave-uniform)
    const int k0 = start + 32 * kFwdTiles * j;
    if (left >= 2)
      fwd_keys<2>(fl, cur, vt, qf, o, m, l, lr, a.scale_log2, left == 2, k0, qi, end, h);
    else if (left == 1)
      fwd_keys<1>(fl, cur, vt, qf, o, m, l, lr, a.scale_log2, true, k0, qi, end, h);
    stage_barrier();
  };
  for (int j = 0; j < stages; j += 2) {
    stage(buf0, buf1, j);
    if (j + 1 < stages) stage(buf1, buf0, j + 1);
  }
  if (mine == 0) return;
  const float2 lp = half_pair(l), rp = half_pair(lr);
  const float L = lp.x + lp.y;
  store_row(a.out + static_cast<int64_t>(qi) * sq + head * kHD, o, 1.0f / (rp.x + rp.y), h, qi < end);
  if (h == 0 && qi < end) a.lse[head * a.n_tok + qi] = (m + log2f(L)) * kLn2;
}

// LDS of the backward: the streamed tiles' two buffers (separate arrays, see TileLane::copy), and for
// the dK / dV blocks the block's V rows and the streamed queries' lse and D.
struct BwdLds {
  char* buf0;
  char* buf1;
  char* v;
  float* ld0;  // lse (log2 units) of 32 queries, then D
  float* ld1;
};

// dQ of 128 queries: key tiles stream through LDS, each wave owns 32 queries (Q and dO fragments in
// registers; D = rowsum(dO o O) from the same fragments).
__device__ __forceinline__ void bwd_wide_dq(const AttnArgs& a, int blk, int head, const BwdLds& lds) {
  int start, end, q0;
  if (!find_block<true, kWide>(a.cu, a.n_seq, static_cast<int>(a.n_tok), blk, start, end, q0)) return;
  start = __builtin_amdgcn_readfirstlane(start);
  end = __builtin_amdgcn_readfirstlane(end);
  q0 = __builtin_amdgcn_readfirstlane(q0);
  const int g = head / (a.h_q / a.h_kv);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int64_t sq = static_cast<int64_t>(a.h_q) * kHD, skv = static_cast<int64_t>(a.h_kv) * kHD;
  const f16* kh = a.k + start * skv + g * kHD;
  const f16* vh = a.v + start * skv + g * kHD;
  const int qw = q0 + 32 * wave, qi = qw + col;
  const int last = min(q0 + kWide, end) - 1;
  const int tiles = (last - start) / 32 + 1;
  const int mine = qw < end ? (qw - start) / 32 + 1 : 0;

  const TileLane tl(wave, lane, skv);
  const FragLane fl0(lane);
  auto copy = [&](char* dst, int j) {
    const int rows = end - start - 32 * j;
    tl.copy(dst, wave, kh + 32 * j * skv, rows);
    tl.copy(dst + kTile, wave, vh + 32 * j * skv, rows);
  };
  copy(lds.buf0, 0);
  const int qr = min(qi, end - 1);
  const int64_t off = static_cast<int64_t>(qr) * sq + head * kHD;
  f16x8 qf[8], df[8];
  float ds = 0.0f;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    qf[s] = *reinterpret_cast<const f16x8*>(a.q + off + 8 * (2 * s + h));
    df[s] = *reinterpret_cast<const f16x8*>(a.dout + off + 8 * (2 * s + h));
    const f16x8 ov = *reinterpret_cast<const f16x8*>(a.o + off + 8 * (2 * s + h));
#pragma unroll
    for (int e = 0; e < 8; ++e)
      ds = __builtin_fmaf(static_cast<float>(ov[e]), static_cast<float>(df[s][e]), ds);
  }
  const float2 dp2 = half_pair(ds);
  const float dsum = dp2.x + dp2.y;
  const float lse2 = a.lse[head * a.n_tok + qr] * kLog2e;
  f32x16 dq[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) dq[d] = f32x16{};
  stage_barrier();
  auto stage = [&](const char* kt, char* next, int j) {
    if (j + 1 < tiles) copy(next, j + 1);
    const char* vt = kt + kTile;
    const FragLane fl = fl0.fresh();
    if (j < mine) {
      f32x16 st = f32x16{}, dp = f32x16{};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        st = mfma(fl.frag(kt, s), qf[s], st);  // S^T = K Q^T
        dp = mfma(fl.frag(vt, s), df[s], dp);  // dP^T = V dO^T
      }
#pragma unroll
      for (int r = 0; r < 16; ++r)
        st[r] = exp2_raw(__builtin_fmaf(st[r], a.scale_log2, -lse2)) * (dp[r] - dsum);
      if (j == mine - 1) {  // the diagonal tile
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = start + 32 * j + acc_row(r, h);
          st[r] = (key <= qi && key < end) ? st[r] : 0.0f;
        }
      }
      const f16x8 s0 = frag_acc(st, 0), s1 = frag_acc(st, 1);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        dq[d] = mfma(fl.frag_t(kt, 0, d), s0, dq[d]);  // dQ^T += K^T dS^T
        dq[d] = mfma(fl.frag_t(kt, 1, d), s1, dq[d]);
      }
    }
    stage_barrier();
  };
  for (int j = 0; j < tiles; j += 2) {
    stage(lds.buf0, lds.buf1, j);
    if (j + 1 < tiles) stage(lds.buf1, lds.buf0, j + 1);
  }
  if (mine == 0) return;
  store_row(a.out + static_cast<int64_t>(qi) * sq + head * kHD, dq, a.scale, h, qi < end);
}

// dK and dV of 128 keys for one query head: Q and dO tiles stream through LDS with their lse and D,
// each wave owns 32 keys (K fragments in registers, V fragments from LDS).
__device__ __forceinline__ void bwd_wide_dkdv(const AttnArgs& a, int blk, int head,
                                              const BwdLds& lds) {
  int start, end, k0;
  if (!find_block<false, kWide>(a.cu, a.n_seq, static_cast<int>(a.n_tok), blk, start, end, k0)) return;
  start = __builtin_amdgcn_readfirstlane(start);
  end = __builtin_amdgcn_readfirstlane(end);
  k0 = __builtin_amdgcn_readfirstlane(k0);
  const int grp = a.h_q / a.h_kv, g = head / grp;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, h = lane >> 5, col = lane & 31;
  const int64_t sq = static_cast<int64_t>(a.h_q) * kHD, skv = static_cast<int64_t>(a.h_kv) * kHD;
  const f16* qh = a.q + k0 * sq + head * kHD;  // from the block's first key on
  const f16* doh = a.dout + k0 * sq + head * kHD;
  const f16* oh = a.o + k0 * sq + head * kHD;
  const float* lse = a.lse + head * a.n_tok + k0;
  const int kw = k0 + 32 * wave, kj = kw + col;
  const int tiles = (end - k0 + 31) / 32;

  const TileLane tl(wave, lane, sq);
  const FragLane fl0(lane);
  f16x8 orow[2];  // the O chunks of the dO chunks this lane copies
  float lr = 0.0f;
  auto copy = [&](char* dst, int j) {
    const int rows = end - k0 - 32 * j;
    tl.copy(dst, wave, qh + 32 * j * sq, rows);
    tl.copy(dst + kTile, wave, doh + 32 * j * sq, rows);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      orow[i] = *reinterpret_cast<const f16x8*>(reinterpret_cast<const char*>(oh + 32 * j * sq) +
                                                tl.at(i, rows));
    if (tid < kBlk) lr = lse[32 * j + min(tid, rows - 1)];
  };
  // D of the rows this wave copied (its copies have landed): each lane's 8 products, then the sum
  // over the 16 lanes of a row.
  auto finish = [&](const char* dst, float* ld) {
    __builtin_amdgcn_s_waitcnt(0x0070 | 0x0F00);  // vmcnt(0)
    if (tid < kBlk) ld[tid] = lr * kLog2e;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f16x8 y = *reinterpret_cast<const f16x8*>(dst + kTile + (2 * wave + i) * 1024 + lane * 16);
      float s = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        s = __builtin_fmaf(static_cast<float>(orow[i][e]), static_cast<float>(y[e]), s);
      s += row_ror<8>(s);
      s += row_ror<4>(s);
      s += row_ror<2>(s);
      s += row_ror<1>(s);
      if ((lane & 15) == 0) ld[kBlk + tl.row[i]] = s;
    }
  };
  copy(lds.buf0, 0);
  {
    const TileLane tv(wave, lane, skv);
#pragma unroll
    for (int n = 0; n < 4; ++n)
      if (k0 + 32 * n < end)
        tv.copy(lds.v + n * kTile, wave, a.v + (k0 + 32 * n) * skv + g * kHD, end - k0 - 32 * n);
  }
  f16x8 kf[8];
  const f16* krow = a.k + static_cast<int64_t>(min(kj, end - 1)) * skv + g * kHD;
#pragma unroll
  for (int s = 0; s < 8; ++s) kf[s] = *reinterpret_cast<const f16x8*>(krow + 8 * (2 * s + h));
  f32x16 dk[4], dv[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    dk[d] = f32x16{};
    dv[d] = f32x16{};
  }
  finish(lds.buf0, lds.ld0);
  stage_barrier();
  const char* vt = lds.v + wave * kTile;
  auto stage = [&](const char* qt, const float* ld, char* next, float* ldn, int j) {
    if (j + 1 < tiles) copy(next, j + 1);
    const char* dt = qt + kTile;
    const FragLane fl = fl0.fresh();
    if (j >= wave) {  // query tiles before the wave's keys see none of them
      f32x16 st = f32x16{}, dp = f32x16{};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        st = mfma(fl.frag(qt, s), kf[s], st);                          // S = Q K^T
        dp = mfma(fl.frag(dt, s), fl.frag(vt, s), dp);  // dP = dO V^T
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const f32x4 lv = *reinterpret_cast<const f32x4*>(ld + 8 * b + 4 * h);
        const f32x4 dd = *reinterpret_cast<const f32x4*>(ld + kBlk + 8 * b + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * b + i;
          const float p = exp2_raw(__builtin_fmaf(st[r], a.scale_log2, -lv[i]));
          st[r] = p;                    // P
          dp[r] = p * (dp[r] - dd[i]);  // dS
        }
      }
      if (j == wave || j == tiles - 1) {  // the diagonal tile, and rows past the row's end
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int qi = k0 + 32 * j + acc_row(r, h);
          const bool in = kj <= qi && qi < end;
          st[r] = in ? st[r] : 0.0f;
          dp[r] = in ? dp[r] : 0.0f;
        }
      }
      const f16x8 p0 = frag_acc(st, 0), p1 = frag_acc(st, 1);
      const f16x8 s0 = frag_acc(dp, 0), s1 = frag_acc(dp, 1);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        dv[d] = mfma(p0, fl.frag_t(dt, 0, d), dv[d]);  // dV += P^T dO
        dv[d] = mfma(p1, fl.frag_t(dt, 1, d), dv[d]);
        dk[d] = mfma(s0, fl.frag_t(qt, 0, d), dk[d]);  // dK += dS^T Q
        dk[d] = mfma(s1, fl.frag_t(qt, 1, d), dk[d]);
      }
    }
    if (j + 1 < tiles) finish(next, ldn);
    stage_barrier();
  };
  for (int j = 0; j < tiles; j += 2) {
    stage(lds.buf0, lds.ld0, lds.buf1, lds.ld1, j);
    if (j + 1 < tiles) stage(lds.buf1, lds.ld1, lds.buf0, lds.ld0, j + 1);
  }
  // This head's fp32 partial: keys are accumulator rows, head dims lanes.
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = kw + acc_row(r, h);
      if (key < end) {
        const int64_t o = (static_cast<int64_t>(head) * a.n_tok + key) * kHD + 32 * d + col;
        store_partial(a.dk_part + o, dk[d][r] * a.scale);
        store_partial(a.dv_part + o, dv[d][r]);
      }
    }
}

// dk / dv [key, g, :] = fp16(sum over the KV group's heads in head order) of the partials: a launch
// of its own. Summed by the last of a group's blocks to arrive it took 7 us with 32-token blocks and
// 24 us with 128-token ones (one block reading 128 keys x 6 heads from beyond its L2 at the end of
// the launch). Thread = 4 head dims of one key; y = dk, dv. The group's size is a template argument,
// so that the heads past the first four are in flight together too (one by one: 100 tokens of 14 / 2
// heads, whole backward, 12.1 us, this 11.7; 707 of 8 / 1 16.4, 15.7). All eight together gain
// another 0.2 us there and lose 1-2% from 8,161 tokens on, where the reads bound it (5.5 TB/s).
// Where 32-token blocks just fill the chip the last block's sum was partly hidden, which no launch
// after them is: 1,206 tokens of 12 / 2 27.5 us against 28.3 now, 2,048 of 8 / 1 28.6 against 30.4;
// beyond, 178 against 91. (The partials are stored past the L2, store_partial: with plain stores the
// launch's end waits for their write-back, 5-10% of the small batches.)
template <int kGrp>
__global__ __launch_bounds__(256) void attn_group_sum_kernel(AttnArgs a) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int c = 4 * static_cast<int>(t & 31), g = static_cast<int>((t >> 5) % a.h_kv);
  const int64_t key = (t >> 5) / a.h_kv;
  if (key >= a.n_tok) return;
  const float* src = (blockIdx.y == 0 ? a.dk_part : a.dv_part) +
                     (static_cast<int64_t>(g) * kGrp * a.n_tok + key) * kHD + c;
  constexpr int kDepth = 4;  // heads whose loads are in flight together
  f32x4 s;
#pragma unroll
  for (int j0 = 0; j0 < kGrp; j0 += kDepth) {
    f32x4 v[kDepth];
#pragma unroll
    for (int j = 0; j < kDepth; ++j)
      if (j0 + j < kGrp) v[j] = *reinterpret_cast<const f32x4*>(src + (j0 + j) * a.n_tok * kHD);
#pragma unroll
    for (int j = 0; j < kDepth; ++j)
      if (j0 + j < kGrp) s = j0 + j == 0 ? v[0] : s + v[j];
    __builtin_amdgcn_sched_barrier(0);
  }
  f16x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = from_f32<f16>(s[i]);
  *reinterpret_cast<f16x4*>((blockIdx.y == 0 ? a.dk : a.dv) + (key * a.h_kv + g) * kHD + c) = w;
}

// Blocks below n_blocks are dK / dV blocks (dispatched first), the rest dQ blocks.
__global__ __launch_bounds__(64 * kW) __attribute__((amdgpu_waves_per_eu(2, 2))) void
attn_bwd_wide_kernel(AttnArgs a) {
  __shared__ __attribute__((aligned(16))) char buf0[2 * kTile];
  __shared__ __attribute__((aligned(16))) char buf1[2 * kTile];
  __shared__ __attribute__((aligned(16))) char v[4 * kTile];
  __shared__ __attribute__((aligned(16))) float ld0[2 * kBlk];
  __shared__ __attribute__((aligned(16))) float ld1[2 * kBlk];
  int blk, head;
  if (!wide_item(a, 2 * a.n_blocks, blk, head)) return;
  const BwdLds lds{buf0, buf1, v, ld0, ld1};
  if (blk < a.n_blocks)
    bwd_wide_dkdv(a, blk, head, lds);
  else
    bwd_wide_dq(a, blk - a.n_blocks, head, lds);
}

// Whether a batch takes the wide kernels: when its 128-token blocks are at least min_blocks. How long
// its rows are is known on the device only (and changes from replay to replay of a captured graph),
// and a long row is what the wide kernels do worse: one block walks its whole length where the
// 32-token blocks' waves share it. So the lines are where no mixture of rows is slower (256 CUs, us,
// 32-token blocks -> wide). Backward with partials, 12 / 2 heads: 192 blocks 2,048 tokens in rows of
// 512 44 -> 33, as one row 112 -> 100, 800 + 18 rows of 64 48 -> 44 (but 156 blocks, 1,024 + 10 rows
// of 64, 51 -> 56). Forward: 300 blocks 1,500 + 27 rows of 64 42 -> 41, 1,024 + 35 rows of 64 34 ->
// 31, one row of 3,300 90 -> 83; 288 blocks one row of 4,600 with 8 heads 110 -> 112, 256 blocks two
// rows of 2,000 with 8 heads 46 -> 51. Below the lines rows of one length would gain (14 rows of 100
// forward 12.3 -> 10.2, backward 27 -> 17), one long row among short ones lose as much (1,024 + 13
// rows of 20 forward 21 -> 30, backward 46 -> 53). Scores are scaled after their maximum is taken,
// hence scale > 0.
constexpr int kFwdWideBlocks = 300, kBwdWideBlocks = 192;

bool wide(int64_t n_tok, int h_q, float scale, int min_blocks) {
  return scale > 0.0f && (n_tok + kWide - 1) / kWide * h_q >= min_blocks;
}

// Bound of the 128-token blocks over all rows (at most the caller's bound of 32-token blocks).
int wide_blocks(int64_t n_tok, int n_seq, int max_blocks) {
  return static_cast<int>(std::min<int64_t>((n_tok + kWide - 1) / kWide + n_seq, max_blocks));
}

unsigned wide_grid(int n_blocks, const AttnArgs& a) {
  const int64_t chunk = 8 * (a.h_q / a.h_kv), items = static_cast<int64_t>(n_blocks) * a.h_q;
  return static_cast<unsigned>((items + chunk - 1) / chunk * chunk);
}

int check(const char* fn, const void* q, const void* k, const void* v, const int32_t* cu,
          int64_t n_tok, int32_t n_seq, int32_t h_q, int32_t h_kv, int32_t head_dim,
          int32_t max_blocks) {
  if (!q || !k || !v || !cu) return fail(RUS_ERR_INVALID, "%s: null pointer argument", fn);
  if (head_dim != kHD) return fail(RUS_ERR_UNSUPPORTED, "%s: head_dim %d (only 128)", fn, head_dim);
  if (h_q <= 0 || h_kv <= 0 || h_q % h_kv)
    return fail(RUS_ERR_INVALID, "%s: h_q=%d must be a multiple of h_kv=%d", fn, h_q, h_kv);
  if (n_tok <= 0 || n_tok >= (int64_t(1) << 31) || n_seq <= 0 || max_blocks <= 0 ||
      max_blocks > 65535)
    return fail(RUS_ERR_INVALID, "%s: n_tok=%lld n_seq=%d max_blocks=%d", fn, (long long)n_tok,
                n_seq, max_blocks);
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16))
    return fail(RUS_ERR_INVALID, "%s: q/k/v must be 16-byte aligned", fn);
  return RUS_OK;
}

}  // namespace
}  // namespace rus

using rus::f16;

extern "C" int rus_attn_varlen_fwd(const void* q, const void* k, const void* v,
                                   const int32_t* cu_seqlens, int32_t n_seq, int64_t n_tokens,
                                   int32_t max_blocks, int32_t h_q, int32_t h_kv,
                                   int32_t head_dim, float scale, void* out, float* lse,
                                   void* stream) {
  using namespace rus;
  const char* fn = "rus_attn_varlen_fwd";
  if (int e = check(fn, q, k, v, cu_seqlens, n_tokens, n_seq, h_q, h_kv, head_dim, max_blocks))
    return e;
  if (!out || !lse || !aligned(out, 16)) return fail(RUS_ERR_INVALID, "%s: bad output", fn);
  AttnArgs a{};
  a.q = static_cast<const f16*>(q);
  a.k = static_cast<const f16*>(k);
  a.v = static_cast<const f16*>(v);
  a.cu = cu_seqlens;
  a.out = static_cast<f16*>(out);
  a.lse = lse;
  a.n_tok = n_tokens;
  a.n_seq = n_seq;
  a.h_q = h_q;
  a.h_kv = h_kv;
  a.scale = scale;
  a.scale_log2 = scale * kLog2e;
  if (wide(n_tokens, h_q, scale, kFwdWideBlocks)) {
    a.n_blocks = wide_blocks(n_tokens, n_seq, max_blocks);
    hipLaunchKernelGGL(attn_fwd_wide_kernel, dim3(wide_grid(a.n_blocks, a)), dim3(64 * kW), 0,
                       static_cast<hipStream_t>(stream), a);
    return check_launch(fn);
  }
  hipLaunchKernelGGL(attn_fwd_kernel, dim3(h_q, max_blocks), dim3(64 * kW), 0,
                     static_cast<hipStream_t>(stream), a);
  return check_launch(fn);
}

static int attn_bwd(const char* fn, const void* q, const void* k, const void* v,
                    const void* out, const void* dout, const float* lse,
                    const int32_t* cu_seqlens, int32_t n_seq, int64_t n_tokens,
                    int32_t max_blocks, int32_t h_q, int32_t h_kv, int32_t head_dim, float scale,
                    void* dq, void* dk, void* dv, float* workspace, int32_t* counters,
                    int64_t n_counters, bool group_sum, void* stream) {
  using namespace rus;
  if (int e = check(fn, q, k, v, cu_seqlens, n_tokens, n_seq, h_q, h_kv, head_dim, max_blocks))
    return e;
  if (!out || !dout || !lse || !dq || !workspace || !aligned(out, 16) || !aligned(dout, 16) ||
      !aligned(dq, 16) || !aligned(workspace, 16))
    return fail(RUS_ERR_INVALID, "%s: null or misaligned argument", fn);
  if (group_sum) {
    if (!dk || !dv || !aligned(dk, 16) || !aligned(dv, 16) || !aligned(counters, 4))
      return fail(RUS_ERR_INVALID, "%s: null or misaligned argument", fn);
    if (h_q / h_kv > kMaxGroup)
      return fail(RUS_ERR_UNSUPPORTED, "%s: %d query heads per KV head (at most %d)", fn,
                  h_q / h_kv, kMaxGroup);
    if ((counters || n_counters) && n_counters < static_cast<int64_t>(max_blocks) * h_kv)
      return fail(RUS_ERR_INVALID, "%s: %lld counters, need max_blocks * h_kv = %lld", fn,
                  static_cast<long long>(n_counters),
                  static_cast<long long>(max_blocks) * h_kv);
  }
  AttnArgs a{};
  a.q = static_cast<const f16*>(q);
  a.k = static_cast<const f16*>(k);
  a.v = static_cast<const f16*>(v);
  a.o = static_cast<const f16*>(out);
  a.dout = static_cast<const f16*>(dout);
  a.cu = cu_seqlens;
  a.lse = const_cast<float*>(lse);
  a.n_tok = n_tokens;
  a.n_seq = n_seq;
  a.h_q = h_q;
  a.h_kv = h_kv;
  a.scale = scale;
  a.scale_log2 = scale * kLog2e;
  // workspace: dk_part [h_q, n_tok, 128] | dv_part (alike)
  if (2 * static_cast<int64_t>(max_blocks) > 65535)
    return fail(RUS_ERR_UNSUPPORTED, "%s: max_blocks=%d (at most 32767)", fn, max_blocks);
  a.dk_part = workspace;
  a.dv_part = a.dk_part + static_cast<int64_t>(h_q) * n_tokens * kHD;
  hipStream_t st = static_cast<hipStream_t>(stream);
  a.out = static_cast<f16*>(dq);
  a.dk = static_cast<f16*>(dk);
  a.dv = static_cast<f16*>(dv);
  a.max_blocks = max_blocks;
  if (wide(n_tokens, h_q, scale, kBwdWideBlocks)) {
    a.n_blocks = wide_blocks(n_tokens, n_seq, max_blocks);
    hipLaunchKernelGGL(attn_bwd_wide_kernel, dim3(wide_grid(2 * a.n_blocks, a)), dim3(64 * kW), 0,
                       st, a);
  } else {
    hipLaunchKernelGGL(attn_bwd_kernel, dim3(h_q, 2 * max_blocks), dim3(64 * kWB), 0, st, a);
  }
  if (int e = check_launch(fn)) return e;
  if (!group_sum) return RUS_OK;
  const dim3 sum_grid(static_cast<unsigned>((n_tokens * h_kv * 32 + 255) / 256), 2);
#define RUS_GROUP_SUM(G) \
  case G: hipLaunchKernelGGL(attn_group_sum_kernel<G>, sum_grid, dim3(256), 0, st, a); break;
  switch (h_q / h_kv) {
    RUS_GROUP_SUM(1) RUS_GROUP_SUM(2) RUS_GROUP_SUM(3) RUS_GROUP_SUM(4)
    RUS_GROUP_SUM(5) RUS_GROUP_SUM(6) RUS_GROUP_SUM(7) RUS_GROUP_SUM(8)
  }
#undef RUS_GROUP_SUM
  return check_launch(fn);
}

extern "C" int rus_attn_varlen_bwd(const void* q, const void* k, const void* v, const void* out,
                                   const void* dout, const float* lse,
                                   const int32_t* cu_seqlens, int32_t n_seq, int64_t n_tokens,
                                   int32_t max_blocks, int32_t h_q, int32_t h_kv,
                                   int32_t head_dim, float scale, void* dq, void* dk, void* dv,
                                   float* workspace, int32_t* counters, int64_t n_counters,
                                   void* stream) {
  return attn_bwd("rus_attn_varlen_bwd", q, k, v, out, dout, lse, cu_seqlens, n_seq, n_tokens,
                  max_blocks, h_q, h_kv, head_dim, scale, dq, dk, dv, workspace, counters,
                  n_counters, true, stream);
}

extern "C" int rus_attn_varlen_bwd_parts(const void* q, const void* k, const void* v,
                                         const void* out, const void* dout, const float* lse,
                                         const int32_t* cu_seqlens, int32_t n_seq,
                                         int64_t n_tokens, int32_t max_blocks, int32_t h_q,
                                         int32_t h_kv, int32_t head_dim, float scale, void* dq,
                                         float* workspace, void* stream) {
  return attn_bwd("rus_attn_varlen_bwd_parts", q, k, v, out, dout, lse, cu_seqlens, n_seq,
                  n_tokens, max_blocks, h_q, h_kv, head_dim, scale, dq, nullptr, nullptr,
                  workspace, nullptr, 0, false, stream);
}
