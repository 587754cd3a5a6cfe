// Gated LoRA (mtp_glora/models/layers/gated_lora.py:51-53), the parts that
// are not plain GEMMs:
//
//   out = base(x) + s * B(A(dropout(x))) * gate
//
// The plain GEMMs (x W^T and dY W, accumulated onto the rank-r term, and d_a^T h
// when the forward kept h) go to hipBLASLt
// (mga_blas.hip). The kernels here fuse what a library GEMM cannot, or stream
// what it runs far from the HBM bound:
//
// * the products that stream a wide operand once (lora_stream_body): the
//   down-projection t = T(T(s * T(h A^T)) * gate), h = dropout(x) drawn on the
//   fly (written out only on request); lora_B's u = dY B and dB = dY^T t; and
//   lora_A's dA = d_a^T h, which draws the same mask again from x. fp32 split
//   sums are added in a fixed order by finishing kernels, which also form t and
//   d_a = T(T(T(u) * gate) * s).
// * lora_outer_kernel: the rank-r products that write a wide result once, the
//   up-projection T(t B^T) and the LoRA path's input gradient
//   L = T(mask * T(scale * T(d_a A))); the base product x W^T or dY W is then
//   accumulated on top by hipBLASLt (beta = 1), so the result is written once
//   here and read once inside that compute-bound GEMM. lora_dx_rows_kernel
//   serves the gradient at ranks above 128, columns not a multiple of 8 and
//   8-byte-aligned rows, one row per lane, from a transposed lora_A.
// * lora_scale_rows_kernel: d_a = T(T(u * gate) * s), u = dY B, when u comes
//   from hipBLASLt (ranks above 128, unaligned rows).
// * lora_transpose_kernel: A^T padded to a multiple of 32 ranks (for
//   lora_dx_rows_kernel, whose operand wants rank-contiguous rows).
//
// T rounds to bf16. With the scaling a power of two and gate values 0 / 1 (the
// reference's alpha = 2 * rank and clamped gate mask), applying s and the gate
// to t instead of to B(t) changes nothing but the rounding of B(t) itself.
//
// Dropout: keep / drop bits come from a counter-based hash, not from torch's
// generator (whose stream cannot be reproduced here): element pair j of the
// flattened [S, K] input (elements 2j, 2j + 1) gets
//   bits = fmix32(fmix32(lo(j) ^ lo(seed)) ^ hi(j) ^ hi(seed)),
// fmix32 being MurmurHash3's 32-bit finaliser; element 2j is kept when
// bits & 0xffff >= thr, element 2j + 1 when bits >> 16 >= thr, thr =
// round(p * 65536). Kept elements are multiplied by 1 / (1 - p), as
// torch's dropout does. The backward draws the same bits again.
#include <algorithm>
#include <type_traits>

#include "mga_common.hpp"
#include "mga_internal.hpp"

namespace mga {

namespace {

__device__ __forceinline__ uint32_t fmix32(uint32_t h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}

__device__ __forceinline__ uint32_t pair_bits(uint64_t seed, uint64_t pair) {
  return fmix32(fmix32((uint32_t)pair ^ (uint32_t)seed) ^ (uint32_t)(pair >> 32) ^ (uint32_t)(seed >> 32));
}

// Dropout of 8 consecutive elements, pair pj (a multiple of 4) the first:
// kept elements times keep_scale, rounded to bf16, the others 0. thr > 0; the
// compares are bits > thr - 1, on the low 16 bits and on the whole word, and
// the four pairs share the upper word of pj: about 140 cycles of VALU work a
// pair and wave, 64 of them the four quarter-rate multiplies.
__device__ __forceinline__ bf16x8 drop8(bf16x8 v, uint64_t pj, uint64_t seed, uint32_t thr, float keep_scale) {
  const uint32_t lo = (uint32_t)pj ^ (uint32_t)seed, hi = (uint32_t)(pj >> 32) ^ (uint32_t)(seed >> 32);
  const uint16_t t_lo = (uint16_t)(thr - 1);
  const uint32_t t_hi = ((thr - 1) << 16) | 0xffffu;
  i32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t bits = fmix32(fmix32(lo ^ (uint32_t)e) ^ hi);
    const float a = (uint16_t)bits > t_lo ? (float)v[2 * e] * keep_scale : 0.f;
    const float b = bits > t_hi ? (float)v[2 * e + 1] * keep_scale : 0.f;
    // asm: the compiler splits the pair into two conversions and a permute
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r[e]) : "v"(a), "v"(b));
  }
  return __builtin_bit_cast(bf16x8, r);
}

__device__ __forceinline__ float rnd(float v) { return (float)(bf16_t)v; }

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (bf16_t)0.f;
  return z;
}

}  // namespace

// out[s][c] = T(sum_r d[s][r] W(r, c)) of the rank-padded rows d (t or d_a) and
// a small weight, written once: the up-projection t B^T (W = lora_B [cols,
// rank]: COLMAJ) and the LoRA term d_a A of dX (W = lora_A [rank, cols]), there
// with the dropout's backward T(mask * T(.) / (1 - p)) applied (DROP). The base
// product is accumulated on top by the compute-bound base GEMM.
// Bound by the writes of out (and the hashes, 140 cycles a pair). A workgroup
// of up to 10 waves takes 128 columns, its W tile shared through LDS (COLMAJ:
// 128 rows of RP ranks, padded; else RP rows of 128 columns, swizzled, read
// transposed, so no transposed copy of lora_A is needed), and 32 rows a wave,
// two 32 x 32 blocks at a time; the rounded blocks go through a per-wave LDS
// tile so that each lane then owns 8 consecutive columns of one row: 16-byte
// stores (whole lines a wave), and each hash serves its element pair. The number of waves is chosen
// so that the workgroups fill whole rounds of the CUs (outer_waves). In the
// layer, at [5120, 6144] x rank 96, t B^T takes 17.7 us (hipBLASLt 25.6 us; a
// plain write of as much 10.7 us), and the dropped d_a A of 4 096 columns 23 us
// (20.4 + 5.1 us with a transposed copy of lora_A).
// cols a multiple of 8, out rows 16-byte aligned, NK = 16-rank steps of the
// padded rank (even).
constexpr int kOuterTs = 72;   // row stride of a wave's 32 x 64 result tile (144 bytes)
constexpr int kOuterWaves = 10;
template <int NK, bool COLMAJ>
constexpr int kOuterTile = COLMAJ ? 128 * (NK * 16 + 8) : 128 * NK * 16;   // elements of the W tile

template <int NK, bool COLMAJ, bool DROP>
__global__ __launch_bounds__(64 * kOuterWaves) void lora_outer_kernel(LoraOuter a) {
  constexpr int RP = NK * 16;          // padded rank
  constexpr int LS = RP + 8;           // COLMAJ: LDS row stride of the W tile (elements)
  extern __shared__ __attribute__((aligned(16))) bf16_t outer_lds[];
  bf16_t *sW = outer_lds;
  const int w = wave_id(), lane = threadIdx.x & 63, tid = threadIdx.x, nt = blockDim.x;
  bf16_t *tile = outer_lds + kOuterTile<NK, COLMAJ> + w * 32 * kOuterTs;
  const int l32 = lane & 31, hi = lane >> 5;
  const int c0 = blockIdx.x * 128;
  const int s0 = (blockIdx.y * (nt >> 6) + w) * 32;
  const bf16_t *wp = reinterpret_cast<const bf16_t *>(a.w);
  const int srow = min(s0 + l32, a.rows - 1);   // rows past the end: computed, never stored
  const bf16_t *dr = reinterpret_cast<const bf16_t *>(a.d) + (int64_t)srow * a.d_rs;
  bf16x8 dv[NK];
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    if constexpr (COLMAJ) {
      dv[j] = load8(dr + 16 * j + 8 * hi);
    } else {   // the k order of the transposed reads
      const i32x2 x = *reinterpret_cast<const i32x2 *>(dr + 16 * j + 4 * hi);
      const i32x2 y = *reinterpret_cast<const i32x2 *>(dr + 16 * j + 8 + 4 * hi);
      dv[j] = __builtin_bit_cast(bf16x8, i32x4{x[0], x[1], y[0], y[1]});
    }
  }
  // the W tile, four granules a thread in flight: each batch's loads are issued
  // before its first LDS write
  constexpr int kGran = 16 * RP, kPerRow = COLMAJ ? RP / 8 : 16;   // granules, granules of a tile row
  for (int i0 = 0; i0 < kGran; i0 += 4 * nt) {
    bf16x8 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * nt + tid, r = i / kPerRow, g = i % kPerRow;
      v[u] = zero8();
      if (COLMAJ ? (i < kGran && c0 + r < a.cols && 8 * g < a.rank) : (r < a.rank && c0 + 8 * g < a.cols))
        v[u] = load8(wp + (COLMAJ ? (int64_t)(c0 + r) * a.w_rs + 8 * g : (int64_t)r * a.w_rs + c0 + 8 * g));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u * nt + tid, r = i / kPerRow, g = i % kPerRow;
      if (COLMAJ && 8 * g + 8 > a.rank)   // the elements past the rank belong to the next row
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (8 * g + e >= a.rank) v[u][e] = (bf16_t)0.f;
      if (i < kGran)
        *reinterpret_cast<i32x4 *>(sW + (COLMAJ ? r * LS + 8 * g : tile_off<128>(r, g))) = __builtin_bit_cast(i32x4, v[u]);
    }
  }
  TrOffsets<128> tro;
  if constexpr (!COLMAJ) tro.init(lane);
  // epilogue ownership: lane -> rows er + 8 h, columns ec .. ec + 7 of a block
  // pair: eight lanes write a row's whole 128-byte line
  const int er = lane >> 3, ec = (lane & 7) * 8;
  bf16_t *out = reinterpret_cast<bf16_t *>(a.out);
  __syncthreads();
  if (s0 >= a.rows) return;
#pragma unroll
  for (int bp = 0; bp < 2; ++bp) {
#pragma unroll
    for (int bi = 0; bi < 2; ++bi) {
      const int blk = 2 * bp + bi;
      f32x16 acc = zero16();
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const bf16x8 wv = COLMAJ ? lds_read8(sW + (blk * 32 + l32) * LS + 16 * j + 8 * hi) : tro.operand(sW, 16 * j, blk);
        acc = mfma32<bf16_t>(dv[j], wv, acc);
      }
      // lane holds column l32 of rows 8 (q / 4) + 4 hi + q % 4
#pragma unroll
      for (int q = 0; q < 16; ++q)
        tile[(8 * (q >> 2) + 4 * hi + (q & 3)) * kOuterTs + 32 * bi + l32] = (bf16_t)acc[q];
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's tile writes done
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int r = er + 8 * h, s = s0 + r, c = c0 + bp * 64 + ec;
      bf16x8 v = lds_read8(tile + r * kOuterTs + ec);
      if (s < a.rows && c < a.cols) {
        if (DROP) v = drop8(v, ((uint64_t)s * (uint64_t)a.cols + (uint64_t)c) >> 1, a.seed, a.thr, a.keep_scale);
        *reinterpret_cast<i32x4 *>(out + (int64_t)s * a.out_rs + c) = __builtin_bit_cast(i32x4, v);
      }
    }
    __builtin_amdgcn_wave_barrier();   // the tile is rewritten by the next pair
  }
}

// General variant (any K multiple of 16, any rank). Grid: (ceil(K / 512),
// ceil(S / 32)), 4 waves; wave w covers 32 rows x 128 columns of dX. D^T[k][s] = sum_r A^T[k][r] d_a[s][r]; each lane holds one
// row s and four runs of four consecutive columns per 32-column block. Every
// load (its d_a row, the A^T rows of its four blocks) is issued before the
// first MFMA when the rank is at most 16 NK (larger ranks go in chunks of NK
// steps). d_a and A^T are zero-padded to a multiple of 32
// ranks, so the step count is even.
template <int NK>
__global__ __launch_bounds__(256) void lora_dx_rows_kernel(LoraDxArgs a) {
  const int w = wave_id(), lane = threadIdx.x & 63;
  const int l32 = lane & 31, hi = lane >> 5;
  const int s = blockIdx.y * 32 + l32;
  const bool s_ok = s < a.S;
  const int sc = s_ok ? s : a.S - 1;     // clamped rows: their sums are never stored
  const int rq = 8 * hi;
  const int kb0 = blockIdx.x * 512 + w * 128;
  bf16_t *dxr = reinterpret_cast<bf16_t *>(a.dx) + (int64_t)sc * a.dx_rs;
  const bf16_t *dar = reinterpret_cast<const bf16_t *>(a.da) + (int64_t)sc * a.da_rs + rq;
  const bf16_t *atr[4];
#pragma unroll
  for (int blk = 0; blk < 4; ++blk) {
    const int kr = kb0 + blk * 32 + l32;
    atr[blk] = reinterpret_cast<const bf16_t *>(a.At) + (int64_t)(kr < a.K ? kr : a.K - 1) * a.at_rs + rq;
  }
  f32x16 acc[4];
#pragma unroll
  for (int blk = 0; blk < 4; ++blk) acc[blk] = zero16();
  // ranks in chunks of NK steps (one chunk when the rank is at most 16 NK)
  const int nsteps = (a.rank + 31) / 32 * 2;
  for (int j0 = 0; j0 < nsteps; j0 += NK) {
    bf16x8 dv[NK], av[4][NK];
#pragma unroll
    for (int j = 0; j < NK; ++j) dv[j] = load8(dar + 16 * (j0 + j));
#pragma unroll
    for (int blk = 0; blk < 4; ++blk)
#pragma unroll
      for (int j = 0; j < NK; ++j) av[blk][j] = load8(atr[blk] + 16 * (j0 + j));
#pragma unroll
    for (int blk = 0; blk < 4; ++blk)
#pragma unroll
      for (int j = 0; j < NK; ++j) acc[blk] = mfma32<bf16_t>(av[blk][j], dv[j], acc[blk]);
  }
#pragma unroll
  for (int blk = 0; blk < 4; ++blk) {
    const int kbase = kb0 + blk * 32;
    if (!s_ok || kbase >= a.K) continue;
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int k = kbase + 8 * g4 + 4 * hi;
      if (k >= a.K) continue;
      const uint64_t pj = ((uint64_t)s * (uint64_t)a.K + (uint64_t)k) >> 1;
      const uint32_t b0 = pair_bits(a.seed, pj), b1 = pair_bits(a.seed, pj + 1);
      const bool keep[4] = {(b0 & 0xffffu) >= a.thr, (b0 >> 16) >= a.thr, (b1 & 0xffffu) >= a.thr,
                            (b1 >> 16) >= a.thr};
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float dh = rnd(acc[blk][4 * g4 + e]);                 // d(dropout(x)) = T(d_a A)
        o[e] = (bf16_t)(keep[e] ? dh * a.keep_scale : 0.f);         // dropout backward
      }
      *reinterpret_cast<bf16x4 *>(dxr + k) = o;
    }
  }
}

// d_a[s][r] = T(T(u[s][r] * gate[s]) * s) for r < rank, 0 up to rpad.
__global__ __launch_bounds__(256) void lora_scale_rows_kernel(const bf16_t *u, int64_t u_rs, const float *gate,
                                                              float scaling, int32_t S, int32_t rank, int32_t rpad,
                                                              bf16_t *da, int64_t da_rs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)S * rpad) return;
  const int s = (int)(i / rpad), r = (int)(i - (int64_t)s * rpad);
  float v = 0.f;
  if (r < rank) {
    const float g = gate ? gate[s] : 1.f;
    v = rnd(rnd((float)u[(int64_t)s * u_rs + r] * g) * scaling);
  }
  da[(int64_t)s * da_rs + r] = (bf16_t)v;
}

// At[k][r] = A[r][k] for r < rank, 0 up to rpad. 32 x 32 tiles through LDS.
__global__ __launch_bounds__(256) void lora_transpose_kernel(const bf16_t *A, int64_t a_rs, int32_t rank, int32_t K,
                                                             int32_t rpad, bf16_t *At, int64_t at_rs) {
  __shared__ bf16_t tile[32][33];
  const int k0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
  for (int y = ty; y < 32; y += 8) {
    const int r = r0 + y, k = k0 + tx;
    tile[y][tx] = (r < rank && k < K) ? A[(int64_t)r * a_rs + k] : (bf16_t)0.f;
  }
  __syncthreads();
  for (int y = ty; y < 32; y += 8) {
    const int k = k0 + y, r = r0 + tx;
    if (k < K && r < rpad) At[(int64_t)k * at_rs + r] = tile[tx][y];
  }
}


// ---- the rank-r products that stream a wide operand -------------------------
// X [rows, cols] (dY or the layer input x) is read once; the small matrix has
// one line of ranks per reduced entry (t, d_a, lora_B) or per rank (lora_A):
//   kDb:   part[split][n][r] = sum over the split's rows s of dY[s][n] t[s][r]
//   kU:    part[split][s][r] = sum over the split's columns n of dY[s][n] B[n][r]
//   kDa:   part[split][r][k] = sum over the split's rows s of d_a[s][r] h[s][k]
//   kDown: part[split][s][r] = sum over the split's columns k of h[s][k] A[r][k]
// with h = dropout(x) drawn on the fly (one hash per element pair). A workgroup
// of 8 waves owns 128 output lines (columns of X for kDb and kDa, rows for kU
// and kDown) and a share of the 64-wide chunks of the reduced dimension. Each
// chunk stages two 64 x 64 X tiles (rows, columns, swizzled), one per 64
// lines, and the chunk's part of the small matrix (64 compact rows of RP =
// 32 RB ranks; for kDown RP rows of 64 columns, swizzled), in a ring of four
// stages filled up to four chunks ahead by direct loads. Wave w takes k-step
// w % 4 (16 of the 64) of every chunk for its 64 lines (half w / 4) and all
// ranks:
//   kDb:   dB^T[r][n] += t^T[r][s] dY[s][n]      A: t^T, B: dY  (transposed LDS reads)
//   kU:    u^T[r][s]  += B^T[r][n] dY^T[n][s]    A: B^T (transposed read), B: dY rows (8-byte reads)
//   kDa:   dA^T[k][r] += h^T[k][s] d_a[s][r]     the operands of kDb exchanged
//   kDown: t^T[r][s]  += A[r][k] h^T[k][s]       A: lora_A rows, B: x rows (16-byte reads)
// kDown applies the dropout to the operand it read, whose 8 columns are 4
// pairs; kDa, whose operand holds one column of 8 rows, applies it in place to
// the 16-byte granules that the wave itself loaded, before the barrier that
// publishes them. A lane holds one output line and 16 ranks of each rank block
// (kDa: one rank and 16 columns), written as 16-byte runs. The waves' sums are
// added in a fixed order at the end.
// Bound by the workgroup's start and end (about 6 us: first loads, final sums)
// and 0.45 us a chunk, 0.65 us once all CUs stream (X from HBM, the small
// matrix from L2; the hashes of a chunk are 0.8 us of VALU work), so the splits
// give every CU one long workgroup where they can. 128 lines a workgroup bring
// 1.75 bytes into LDS per byte of X at rank 96 (64 lines: 2.5).
// kDb and kU at [5120, 6144] x rank 96 38 us, and 5.4 us to finish both (one
// launch per product with 64 lines: 28.7 + 5.4 and 25.6 + 6.2 us); at
// [1387, 4096] x rank 32 8.2 + 4.7 us (6.7 + 4.8 and 6.6 + 4.8 us).
// The hashes bound kDown and kDa there (1.2 us a chunk): [5120, 4096] x rank 96
// with dropout 26.3 + 5.3 and 26.5 + 5.0 us with the finishing launches (an
// earlier kernel with a packed copy of lora_A 5.1 + 26.5 + 5.4, staging through
// registers for dA 30.2 + 7.6 us).
// The loads are inline asm through buffer resources (the caller of the wait
// counts them: 2 X loads a wave and chunk, and the small matrix's 4 RB loads
// dealt to the 8 waves); rows past the end arrive as zeros, columns past the
// end as other elements of X, which are zeroed in the operand where they are
// reduced over and stay in lines that nothing reads otherwise. Rank columns
// past the rank hold junk that the finishing kernels do not read.
// FAR (kDa and kDown, row strides of 2^23 elements and more, which the loads'
// 32-bit lane offsets over a tile's rows do not reach): the same granules by
// 64-bit addresses through registers, rows and columns past the end as zeros.
enum { kDb = 0, kU = 1, kDa = 2, kDown = 3 };

template <int KIND, int RB, bool DROP, bool WRITE_H, bool FAR = false>
__device__ __forceinline__ void lora_stream_body(const LoraStream &a, int blk, int split, bf16_t *lds) {
  constexpr bool kCols = KIND == kDb || KIND == kDa;   // lines are columns of X, rows are reduced
  constexpr int RP = 32 * RB;                 // ranks of a small tile
  constexpr int YT = 64 * 64, MT = 64 * RP, STAGE = 2 * YT + MT;
  constexpr int MG = RP / 8;                  // granules per compact small-tile row
  constexpr int MIA = (RB + 1) / 2, MIB = RB / 2;   // small-tile loads of waves 0-3, of waves 4-7
  const int w = wave_id(), lane = threadIdx.x & 63;
  const int kq = w & 3, half = w >> 2;
  const int l32 = lane & 31, hi = lane >> 5;
  const int line0 = blk * 128 + 64 * half;    // the wave's first line
  const int nlines = kCols ? a.cols : a.rows;   // output lines
  const int kdim = kCols ? a.rows : a.cols;     // reduced dimension
  const int nall = (kdim + 63) / 64;
  const int c0 = (int)((int64_t)nall * split / a.ns);
  const int nch = (int)((int64_t)nall * (split + 1) / a.ns) - c0;
  const bf16_t *x = reinterpret_cast<const bf16_t *>(a.x);
  const bf16_t *sm = reinterpret_cast<const bf16_t *>(a.sm);
  const int mcols = (a.rank + 7) / 8 * 8;

  // Per-lane byte offsets. X tile: 8 granules per row, 8 rows per load, wave kq
  // of the half loads rows 16 kq .. 16 kq + 15 (two loads). Small tile, load i
  // of wave w: compact rows, slots 64 (w + 8 i) + lane (row slot / MG, granule
  // slot % MG; a granule past the rank reads the last one again); kDown, ranks
  // 8 (w + 8 i) + lane / 8.
  uint32_t yo[2], mo[MIA];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 16 * kq + 8 * i + (lane >> 3);
    yo[i] = opaque_u32((uint32_t)(r * a.x_rs * 2) + (uint32_t)(16 * ((lane & 7) ^ swz<64>(r))));
  }
#pragma unroll
  for (int i = 0; i < MIA; ++i) {
    if constexpr (KIND == kDown) {
      const int r = 8 * (w + 8 * i) + (lane >> 3);
      mo[i] = opaque_u32((uint32_t)(r * a.sm_rs * 2) + (uint32_t)(16 * ((lane & 7) ^ swz<64>(r))));
    } else {
      const int slot = 64 * (w + 8 * i) + lane;
      mo[i] = opaque_u32((uint32_t)((slot / MG) * a.sm_rs * 2) + (uint32_t)(16 * min(slot % MG, mcols / 8 - 1)));
    }
  }
  // Workgroups start their share at different chunks (rotated by the line
  // block), so that those streaming the same share at the same time do not all
  // read the same rows of the small matrix at once.
  const int rot = blk % max(nch, 1);
  auto chunk_of = [&](int c) { const int r = c + rot; return c0 + (r >= nch ? r - nch : r); };
  auto issue = [&](int c, bf16_t *st) {
    const int k0 = chunk_of(min(c, nch - 1)) * 64;   // past the share: its last chunk again
    const int r0 = kCols ? k0 : line0, n0 = kCols ? line0 : k0;
    if constexpr (FAR) {
      auto put = [&](bf16_t *dst, const bf16_t *base, int64_t rs, int r, int nr, int c, int nc) {
        const bf16x8 v = r < nr && c < nc ? load8(base + r * rs + c) : zero8();
        *reinterpret_cast<i32x4 *>(dst + lane * 8) = __builtin_bit_cast(i32x4, v);
      };
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * kq + 8 * i + (lane >> 3);
        put(st + half * YT + (16 * kq + 8 * i) * 64, x, a.x_rs, r0 + r, a.rows, n0 + 8 * ((lane & 7) ^ swz<64>(r)), a.cols);
      }
#pragma unroll
      for (int i = 0; i < MIA; ++i)
        if (i < MIB || w < 4) {
          const int r = 8 * (w + 8 * i) + (lane >> 3), slot = 64 * (w + 8 * i) + lane;
          bf16_t *dst = st + 2 * YT + 512 * (w + 8 * i);
          if constexpr (KIND == kDown) put(dst, sm, a.sm_rs, r, a.rank, k0 + 8 * ((lane & 7) ^ swz<64>(r)), a.cols);
          else put(dst, sm, a.sm_rs, k0 + slot / MG, kdim, min(8 * (slot % MG), mcols - 8), mcols);
        }
      return;
    }
    // resource ranges end with the last element of the tile's last existing row
    const int64_t yb = (int64_t)(min(64, a.rows - r0) - 1) * a.x_rs + a.cols - n0;
    const i32x4 ry =
        buf_rsrc(x + (r0 < a.rows ? (int64_t)r0 * a.x_rs + n0 : 0), r0 < a.rows && yb > 0 ? (uint32_t)(yb * 2) : 0u);
#pragma unroll
    for (int i = 0; i < 2; ++i) bdma16(ry, yo[i], st + half * YT + (16 * kq + 8 * i) * 64);
    i32x4 rm;
    if constexpr (KIND == kDown)
      rm = buf_rsrc(sm + k0, (uint32_t)(((int64_t)(min(a.rank, RP) - 1) * a.sm_rs + a.cols - k0) * 2));
    else
      rm = buf_rsrc(sm + (int64_t)k0 * a.sm_rs, (uint32_t)(((int64_t)(min(64, kdim - k0) - 1) * a.sm_rs + mcols) * 2));
#pragma unroll
    for (int i = 0; i < MIA; ++i)
      if (i < MIB || w < 4) bdma16(rm, mo[i], st + 2 * YT + 512 * (w + 8 * i));
  };
  // the loads of the three (two) newest chunks stay in flight; with the
  // dropout output's stores among them, which may retire out of order, none
  auto wait3 = [&]() {
    if (MIA == MIB || w < 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * (2 + MIA)) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * (2 + MIB)) : "memory");
  };
  auto wait2 = [&]() {
    if (WRITE_H) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (MIA == MIB || w < 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (2 + MIA)) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (2 + MIB)) : "memory");
  };
  // dropout of the 8 elements of row s from column k on (columns a multiple of 16)
  auto drop = [&](const bf16x8 &v, int s, int k) {
    return drop8(v, ((uint64_t)s * (uint64_t)a.cols + (uint64_t)k) >> 1, a.seed, a.thr, a.keep_scale);
  };
  // kDa: dropout, in place, of the granules of chunk c that this wave loaded
  auto drop_own = [&](int c, bf16_t *st) {
    if constexpr (KIND == kDa && DROP) {
      const int k0 = chunk_of(c) * 64;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * kq + 8 * i + (lane >> 3), g = (lane & 7) ^ swz<64>(r);
        bf16_t *p = st + half * YT + (16 * kq + 8 * i) * 64 + lane * 8;
        *reinterpret_cast<i32x4 *>(p) = __builtin_bit_cast(i32x4, drop(lds_read8(p), k0 + r, line0 + 8 * g));
      }
    }
  };

  // small operand from a compact k-major tile (rows k, RP columns): lane (l32,
  // hi) takes column 32 rb + l32 at rows k0 + 4 hi + 0..3 and k0 + 8 + 4 hi +
  // 0..3 (the k order of TrLane), by two transposed reads
  const int ti = lane & 15;
  const uint32_t mro[2] = {
      opaque_u32((uint32_t)(((16 * kq + 4 * hi + (ti >> 2)) * RP + 16 * ((lane >> 4) & 1) + 4 * (ti & 3)) * 2)),
      opaque_u32((uint32_t)(((16 * kq + 8 + 4 * hi + (ti >> 2)) * RP + 16 * ((lane >> 4) & 1) + 4 * (ti & 3)) * 2))};
  auto m_operand = [&](const bf16_t *tM, int rb) {
    if constexpr (KIND == kDown) return lds_read8(tM + tile_off<64>(32 * rb + l32, 2 * kq + hi));
    const char *p = reinterpret_cast<const char *>(tM) + 64 * rb;
    return join8(lds_tr4(reinterpret_cast<const bf16_t *>(p + mro[0])),
                 lds_tr4(reinterpret_cast<const bf16_t *>(p + mro[1])));
  };
  TrOffsets<64> try_;
  if constexpr (kCols) try_.init(lane);
  f32x16 acc[RB][2];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[rb][0] = acc[rb][1] = zero16();

  auto operands = [&](int c, const bf16_t *st, bf16x8 (&av)[RB], bf16x8 (&bv)[2]) {
    const bf16_t *tY = st + half * YT, *tM = st + 2 * YT;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) av[rb] = m_operand(tM, rb);
    if constexpr (kCols) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) bv[nb] = try_.operand(tY, 16 * kq, nb);
    } else {
      const int kb = chunk_of(c) * 64 + 16 * kq;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb) {
        const int r = 32 * sb + l32;
        if constexpr (KIND == kU) {
          // dY columns kb + 4 hi + 0..3 and kb + 8 + 4 hi + 0..3 of row r
          bv[sb] = lds_read4x2(tY + tile_off<64>(r, 2 * kq) + 4 * hi, tY + tile_off<64>(r, 2 * kq + 1) + 4 * hi);
          if (kb + 16 > kdim)
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (kb + 4 * hi + (e & 3) + 8 * (e >> 2) >= kdim) bv[sb][e] = (bf16_t)0.f;
        } else {
          // x columns kb + 8 hi + 0..7 of row r (the columns are a multiple of 16)
          bv[sb] = lds_read8(tY + tile_off<64>(r, 2 * kq + hi));
          if (DROP) bv[sb] = drop(bv[sb], line0 + r, kb + 8 * hi);
          if (kb >= kdim) bv[sb] = zero8();
          if (WRITE_H && DROP && kb < kdim && line0 + r < a.rows)
            *reinterpret_cast<i32x4 *>(reinterpret_cast<bf16_t *>(a.h) + (int64_t)(line0 + r) * a.h_rs + kb + 8 * hi) =
                __builtin_bit_cast(i32x4, bv[sb]);
        }
      }
      if (KIND == kDown && kb >= kdim)   // lora_A's elements there belong to the next rank
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) av[rb] = zero8();
    }
  };

  // chunk c: its operands were read in the turn before, so its stage is free
  // behind a barrier. This wave's loads of chunk c + 1 landed, then a barrier
  // behind this wave's LDS reads (every wave's part of c + 1 is in, and every
  // wave has read c), the loads of chunk c + 4 into c's stage, the operand reads
  // of c + 1, and the products of c under them.
  bf16x8 av[2][RB], bv[2][2];
  if (nch > 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) issue(q, lds + q * STAGE);
    wait3();
    drop_own(0, lds);
    lds_barrier();
    operands(0, lds, av[0], bv[0]);
    for (int cb = 0; cb < nch; cb += 4)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (cb + q < nch) {
          if (cb + q + 1 < nch) {
            wait2();
            drop_own(cb + q + 1, lds + ((q + 1) & 3) * STAGE);
            lds_barrier();
            issue(cb + q + 4, lds + q * STAGE);
            operands(cb + q + 1, lds + ((q + 1) & 3) * STAGE, av[(q + 1) & 1], bv[(q + 1) & 1]);
          }
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int lb = 0; lb < 2; ++lb)
              acc[rb][lb] = KIND == kDa ? mfma32<bf16_t>(bv[q & 1][lb], av[q & 1][rb], acc[rb][lb])
                                        : mfma32<bf16_t>(av[q & 1][rb], bv[q & 1][lb], acc[rb][lb]);
        }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the ring's trailing loads
  __syncthreads();

  // fixed-order sum of the four k-step waves of each half through LDS, 32 lines
  // at a time: every wave parks its accumulators, then wave kq adds the four
  // waves' registers 4 kq .. 4 kq + 3 and writes them as this split's partial:
  // lane = line 32 lb + l32, ranks 32 rb + 8 kq + 4 hi + 0..3 (kDa: rank
  // 32 rb + l32, lines 32 lb + 8 kq + 4 hi + 0..3)
  f32x4 *park = reinterpret_cast<f32x4 *>(lds) + half * (4 * RB * 4 * 64);
#pragma unroll
  for (int lb = 0; lb < 2; ++lb) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x16 &c = acc[rb][lb];
        park[((kq * RB + rb) * 4 + q) * 64 + lane] = f32x4{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      f32x4 v = park[(rb * 4 + kq) * 64 + lane];
#pragma unroll
      for (int k = 1; k < 4; ++k) {
        const f32x4 y = park[((k * RB + rb) * 4 + kq) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += y[e];
      }
      if constexpr (KIND == kDa) {
        const int line = line0 + 32 * lb + 8 * kq + 4 * hi;   // the columns are a multiple of 16
        if (line < nlines)
          *reinterpret_cast<f32x4 *>(a.part + ((int64_t)split * RP + 32 * rb + l32) * nlines + line) = v;
      } else {
        const int line = line0 + 32 * lb + l32;
        if (line < nlines)
          *reinterpret_cast<f32x4 *>(a.part + ((int64_t)split * nlines + line) * RP + 32 * rb + 8 * kq + 4 * hi) = v;
      }
    }
    __syncthreads();
  }
}

template <int RB>
constexpr int kStreamLds = 4 * (2 * 64 * 64 + 64 * 32 * RB);   // elements

// kU over u, kDb over b (ns = 0: not wanted)
template <int RB>
__global__ __launch_bounds__(512, 1) void lora_skinny_kernel(LoraStream u, LoraStream b) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[kStreamLds<RB>];
  const int nbu = (u.rows + 127) / 128, nbb = (b.cols + 127) / 128;
  const int i = blockIdx.x;
  if (i < nbu * u.ns) lora_stream_body<kU, RB, false, false>(u, i % nbu, i / nbu, lds);
  else lora_stream_body<kDb, RB, false, false>(b, (i - nbu * u.ns) % nbb, (i - nbu * u.ns) / nbb, lds);
}

template <int RB, bool FAR>
__global__ __launch_bounds__(512, 1) void lora_da_kernel(LoraStream a) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[kStreamLds<RB>];
  const int nb = (a.cols + 127) / 128;
  lora_stream_body<kDa, RB, true, false, FAR>(a, blockIdx.x % nb, blockIdx.x / nb, lds);
}

template <int RB, bool DROP, bool WRITE_H, bool FAR>
__global__ __launch_bounds__(512, 1) void lora_down_kernel(LoraStream a) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[kStreamLds<RB>];
  const int nb = (a.rows + 127) / 128;
  lora_stream_body<kDown, RB, DROP, WRITE_H, FAR>(a, blockIdx.x % nb, blockIdx.x / nb, lds);
}

// t[s][r] = T(T(s * T(sum over the splits, in order)) * gate), 0 for rank <= r
// < 32 RB. Four ranks a thread.
__global__ __launch_bounds__(256) void lora_down_finish_kernel(LoraStream a, int rp, const float *gate, float scaling,
                                                               bf16_t *t, int64_t t_rs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)a.rows * (rp / 4)) return;
  const int s = (int)(i / (rp / 4)), r = 4 * (int)(i - (int64_t)s * (rp / 4));
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int y = 0; y < a.ns; ++y) {
    const f32x4 x = *reinterpret_cast<const f32x4 *>(a.part + ((int64_t)y * a.rows + s) * rp + r);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += x[e];
  }
  const float g = gate ? gate[s] : 1.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = r + e < a.rank ? rnd(rnd(v[e]) * scaling) * g : 0.f;
  bf16_t *out = t + (int64_t)s * t_rs + r;
  if ((t_rs & 3) == 0 && ((uintptr_t)t & 7) == 0) store4(out, v[0], v[1], v[2], v[3]);
  else
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = (bf16_t)v[e];
}

// dA[r][k] = T(sum over the splits, in order) for r < rank. Four columns a thread.
__global__ __launch_bounds__(256) void lora_da_finish_kernel(LoraStream a, int rp, bf16_t *dA, int64_t dA_rs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)a.rank * (a.cols / 4)) return;
  const int r = (int)(i / (a.cols / 4)), k = 4 * (int)(i - (int64_t)r * (a.cols / 4));
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int y = 0; y < a.ns; ++y) {
    const f32x4 x = *reinterpret_cast<const f32x4 *>(a.part + ((int64_t)y * rp + r) * a.cols + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += x[e];
  }
  bf16_t *out = dA + (int64_t)r * dA_rs + k;
  if ((dA_rs & 3) == 0 && ((uintptr_t)dA & 7) == 0) store4(out, v[0], v[1], v[2], v[3]);
  else
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = (bf16_t)v[e];
}

// d_a[s][r] = T(T(T(u) * gate[s]) * scaling), u = the sum over the splits in
// order; 0 for rank <= r < rp (the roundings of the chain dY B (bf16), then
// lora_scale_rows); dB[n][r] = T(sum over the splits, in order), r < rank
// (nsb > 0). Four ranks a thread.
__global__ __launch_bounds__(256) void lora_skinny_finish_kernel(LoraStream u, LoraStream b, int rp, const float *gate,
                                                                 float scaling, bf16_t *da, int64_t da_rs, bf16_t *db,
                                                                 int64_t db_rs) {
  const int64_t nu = (int64_t)u.rows * (rp / 4), nb = b.ns > 0 ? (int64_t)b.cols * (rp / 4) : 0;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool isb = i >= nu;
  if (isb) i -= nu;
  if (isb && i >= nb) return;
  const int line = (int)(i / (rp / 4)), r = 4 * (int)(i - (int64_t)line * (rp / 4));
  const int nlines = isb ? b.cols : u.rows, ns = isb ? b.ns : u.ns;
  const float *p = (isb ? b.part : u.part) + (int64_t)line * rp + r;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int y = 0; y < ns; ++y) {
    const f32x4 x = *reinterpret_cast<const f32x4 *>(p + (int64_t)y * nlines * rp);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += x[e];
  }
  if (isb) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (r + e < b.rank) db[(int64_t)line * db_rs + r + e] = (bf16_t)v[e];
    return;
  }
  const float g = gate ? gate[line] : 1.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = r + e < u.rank ? rnd(rnd(rnd(v[e]) * g) * scaling) : 0.f;
  store4(da + (int64_t)line * da_rs + r, v[0], v[1], v[2], v[3]);
}

// The general form of the LoRA term of dX (ranks above 128, columns a multiple
// of 16 only, 8-byte aligned rows), from a transposed copy of lora_A.
void launch_lora_dx_rows(const LoraDxArgs &a, hipStream_t st) {
  const dim3 grid((unsigned)((a.K + 511) / 512), (unsigned)((a.S + 31) / 32)), block(256);
  switch ((a.rank + 31) / 32) {
    case 1: hipLaunchKernelGGL((lora_dx_rows_kernel<2>), grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL((lora_dx_rows_kernel<4>), grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL((lora_dx_rows_kernel<6>), grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL((lora_dx_rows_kernel<8>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((lora_dx_rows_kernel<2>), grid, block, 0, st, a); break;   // 2-step chunks
  }
}

namespace {

// Waves of an outer-product workgroup, 6 to 10: the count that leaves the CUs
// the least uneven number of waves (workgroups per CU, rounded up, times
// waves), the larger of equals. Each workgroup copies the W tile: [3000, 24576]
// x rank 64 takes 64 us with 1 wave, 39 with 2, 27 with 4 to 10; [5120, 6144] x
// rank 96 takes 49, 26, 19 (4), 17.8 (6) and 15.5 us (10).
int outer_waves(int row_blocks, int col_blocks) {
  const int cus = device_cu_count();
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int w = std::min(row_blocks, 6); w <= std::min(row_blocks, kOuterWaves); ++w) {
    const int64_t wgs = (int64_t)((row_blocks + w - 1) / w) * col_blocks;
    const int64_t cost = (wgs + cus - 1) / cus * w;
    if (cost <= best_cost) {
      best_cost = cost;
      best = w;
    }
  }
  return best;
}

template <int NK, bool COLMAJ, bool DROP>
void outer_launch(const LoraOuter &a, hipStream_t st) {
  const int rb = (a.rows + 31) / 32, cb = (a.cols + 127) / 128;
  const int w = outer_waves(rb, cb);
  const size_t lds = 2 * ((size_t)kOuterTile<NK, COLMAJ> + (size_t)w * 32 * kOuterTs);
  hipLaunchKernelGGL((lora_outer_kernel<NK, COLMAJ, DROP>), dim3((unsigned)cb, (unsigned)((rb + w - 1) / w)),
                     dim3(64 * w), lds, st, a);
}

template <bool COLMAJ, bool DROP>
void outer_rank(const LoraOuter &a, hipStream_t st) {
  switch ((a.rank + 31) / 32) {
    case 1: outer_launch<2, COLMAJ, DROP>(a, st); break;
    case 2: outer_launch<4, COLMAJ, DROP>(a, st); break;
    case 3: outer_launch<6, COLMAJ, DROP>(a, st); break;
    default: outer_launch<8, COLMAJ, DROP>(a, st); break;
  }
}

}  // namespace

void launch_lora_outer(const LoraOuter &a, bool colmaj, hipStream_t st) {
  if (colmaj) outer_rank<true, false>(a, st);
  else if (a.thr > 0) outer_rank<false, true>(a, st);
  else outer_rank<false, false>(a, st);
}

void launch_lora_scale_rows(const void *u, int64_t u_rs, const float *gate, float scaling, int32_t S, int32_t rank,
                            int32_t rpad, void *da, int64_t da_rs, hipStream_t st) {
  const int64_t n = (int64_t)S * rpad;
  hipLaunchKernelGGL(lora_scale_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<const bf16_t *>(u), u_rs, gate, scaling, S, rank, rpad,
                     reinterpret_cast<bf16_t *>(da), da_rs);
}

void launch_lora_transpose(const void *A, int64_t a_rs, int32_t rank, int32_t K, int32_t rpad, void *At,
                           int64_t at_rs, hipStream_t st) {
  hipLaunchKernelGGL(lora_transpose_kernel, dim3((unsigned)((K + 31) / 32), (unsigned)(rpad / 32)), dim3(256), 0, st,
                     reinterpret_cast<const bf16_t *>(A), a_rs, rank, K, rpad, reinterpret_cast<bf16_t *>(At), at_rs);
}

// ---- the general path (fp16 / fp32 operands) ------------------------------
// HBM-bound elementwise kernels: one thread per element pair (dropout) or
// element (scale rows); the products run in hipBLASLt.

namespace {

template <typename T> __device__ __forceinline__ float to_f(T v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f(float v) { return (T)v; }

template <typename T>
__global__ __launch_bounds__(256) void lora_gen_dropout_kernel(const T *x, int64_t x_rs, int32_t S, int32_t K,
                                                               uint32_t thr, float ks, uint64_t seed, T *h,
                                                               int64_t h_rs, int32_t in_place) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;   // element pair of the flattened [S, K]
  if (j >= (int64_t)S * K / 2) return;
  const int64_t e = 2 * j;
  const int s = (int)(e / K), k = (int)(e - (int64_t)s * K);   // K is even: the pair stays in the row
  const uint32_t bits = pair_bits(seed, (uint64_t)j);
  const T *xr = in_place ? h + (int64_t)s * h_rs : x + (int64_t)s * x_rs;
  T *hr = h + (int64_t)s * h_rs;
  const float v0 = to_f(xr[k]), v1 = to_f(xr[k + 1]);
  hr[k] = (bits & 0xffffu) >= thr ? from_f<T>(v0 * ks) : from_f<T>(0.f);
  hr[k + 1] = (bits >> 16) >= thr ? from_f<T>(v1 * ks) : from_f<T>(0.f);
}

// rows of rank entries, then zeros up to rpad (the padded columns the bf16
// kernels write as zeros too)
template <typename T>
__global__ __launch_bounds__(256) void lora_gen_scale_rows_kernel(const T *u, int64_t u_rs, const float *gate,
                                                                  float scaling, int32_t gate_first, int32_t S,
                                                                  int32_t rank, int32_t rpad, T *out, int64_t out_rs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)S * rpad) return;
  const int s = (int)(i / rpad), r = (int)(i - (int64_t)s * rpad);
  float w = 0.f;
  if (r < rank) {
    const float g = gate ? gate[s] : 1.f;
    const float v = to_f(u[(int64_t)s * u_rs + r]);
    w = gate_first ? to_f(from_f<T>(to_f(from_f<T>(v * g)) * scaling))
                   : to_f(from_f<T>(to_f(from_f<T>(v * scaling)) * g));
  }
  out[(int64_t)s * out_rs + r] = from_f<T>(w);
}

template <typename T>
void gen_launch(int64_t n, void (*k)(const T *, int64_t, int32_t, int32_t, uint32_t, float, uint64_t, T *, int64_t, int32_t),
                const void *x, int64_t x_rs, int32_t S, int32_t K, uint32_t thr, float ks, uint64_t seed, void *h,
                int64_t h_rs, int32_t in_place, hipStream_t st) {
  hipLaunchKernelGGL(k, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, reinterpret_cast<const T *>(x), x_rs, S,
                     K, thr, ks, seed, reinterpret_cast<T *>(h), h_rs, in_place);
}

}  // namespace

void launch_lora_gen_dropout(int dtype, const void *x, int64_t x_rs, int32_t S, int32_t K, uint32_t thr,
                             float keep_scale, uint64_t seed, void *h, int64_t h_rs, hipStream_t st) {
  const int64_t n = (int64_t)S * K / 2;
  if (dtype == kDtF32) gen_launch<float>(n, lora_gen_dropout_kernel<float>, x, x_rs, S, K, thr, keep_scale, seed, h, h_rs, 0, st);
  else gen_launch<f16_t>(n, lora_gen_dropout_kernel<f16_t>, x, x_rs, S, K, thr, keep_scale, seed, h, h_rs, 0, st);
}

void launch_lora_gen_dx_mask(int dtype, void *dx, int64_t dx_rs, int32_t S, int32_t K, uint32_t thr, float keep_scale,
                             uint64_t seed, hipStream_t st) {
  const int64_t n = (int64_t)S * K / 2;
  if (dtype == kDtF32) gen_launch<float>(n, lora_gen_dropout_kernel<float>, dx, dx_rs, S, K, thr, keep_scale, seed, dx, dx_rs, 1, st);
  else gen_launch<f16_t>(n, lora_gen_dropout_kernel<f16_t>, dx, dx_rs, S, K, thr, keep_scale, seed, dx, dx_rs, 1, st);
}

void launch_lora_gen_scale_rows(int dtype, const void *u, int64_t u_rs, const float *gate, float scaling, bool gate_first,
                                int32_t S, int32_t rank, int32_t rpad, void *out, int64_t out_rs, hipStream_t st) {
  const int64_t n = (int64_t)S * rpad;
  const dim3 grid((unsigned)((n + 255) / 256));
  if (dtype == kDtF32)
    hipLaunchKernelGGL(lora_gen_scale_rows_kernel<float>, grid, dim3(256), 0, st, reinterpret_cast<const float *>(u),
                       u_rs, gate, scaling, (int32_t)gate_first, S, rank, rpad, reinterpret_cast<float *>(out), out_rs);
  else
    hipLaunchKernelGGL(lora_gen_scale_rows_kernel<f16_t>, grid, dim3(256), 0, st, reinterpret_cast<const f16_t *>(u),
                       u_rs, gate, scaling, (int32_t)gate_first, S, rank, rpad, reinterpret_cast<f16_t *>(out), out_rs);
}

namespace {

// Splits of the reduced dimensions of one or two streaming products (line
// blocks, chunks): rounds of one workgroup per CU with the smallest number of
// chunks from the first to the last, kStreamStart chunks' time going into a
// workgroup's first loads and final sums (7 to 14 measure level).
void stream_plan(int64_t nb0, int ch0, int32_t *ns0, int64_t nb1, int ch1, int32_t *ns1) {
  constexpr int kStreamStart = 8, kMaxSplit = 16;
  const int cus = device_cu_count();
  int64_t best = INT64_MAX;
  for (int len = 1; len <= std::max(ch0, ch1); ++len) {
    const int a = (ch0 + len - 1) / len, b = (ch1 + len - 1) / len;
    if (a > kMaxSplit || b > kMaxSplit) continue;
    const int64_t wgs = nb0 * a + nb1 * b;
    const int64_t cost = ((wgs + cus - 1) / cus) * (len + kStreamStart);
    if (cost < best) {
      best = cost;
      *ns0 = a;
      *ns1 = b;
    }
  }
}

int blocks128(int n) { return (n + 127) / 128; }
int chunks64(int n) { return (n + 63) / 64; }
int32_t stream_split(int lines, int kdim) {
  int32_t ns = 1, none = 0;
  stream_plan(blocks128(lines), chunks64(kdim), &ns, 0, 0, &none);
  return ns;
}
void skinny_plan(int32_t S, int32_t N, bool with_b, int32_t *nsu, int32_t *nsb) {
  stream_plan(blocks128(S), chunks64(N), nsu, with_b ? blocks128(N) : 0, with_b ? chunks64(S) : 0, nsb);
}

template <int RB, bool FAR>
void down_rb(const LoraStream &a, bool drop, hipStream_t st) {
  const dim3 grid((unsigned)(blocks128(a.rows) * a.ns)), blk(512);
  if (drop && a.h) hipLaunchKernelGGL((lora_down_kernel<RB, true, true, FAR>), grid, blk, 0, st, a);
  else if (drop) hipLaunchKernelGGL((lora_down_kernel<RB, true, false, FAR>), grid, blk, 0, st, a);
  else hipLaunchKernelGGL((lora_down_kernel<RB, false, false, FAR>), grid, blk, 0, st, a);
}

template <bool FAR>
void down_rank(const LoraStream &a, bool drop, hipStream_t st) {
  switch ((a.rank + 31) / 32) {
    case 1: down_rb<1, FAR>(a, drop, st); break;
    case 2: down_rb<2, FAR>(a, drop, st); break;
    case 3: down_rb<3, FAR>(a, drop, st); break;
    default: down_rb<4, FAR>(a, drop, st); break;
  }
}

template <bool FAR>
void da_rank(const LoraStream &a, hipStream_t st) {
  const dim3 grid((unsigned)(blocks128(a.cols) * a.ns)), blk(512);
  switch ((a.rank + 31) / 32) {
    case 1: hipLaunchKernelGGL((lora_da_kernel<1, FAR>), grid, blk, 0, st, a); break;
    case 2: hipLaunchKernelGGL((lora_da_kernel<2, FAR>), grid, blk, 0, st, a); break;
    case 3: hipLaunchKernelGGL((lora_da_kernel<3, FAR>), grid, blk, 0, st, a); break;
    default: hipLaunchKernelGGL((lora_da_kernel<4, FAR>), grid, blk, 0, st, a); break;
  }
}

bool far_rows(const LoraStream &a) { return a.x_rs >= kMaxStreamStride || a.sm_rs >= kMaxStreamStride; }

}  // namespace

// Partial sums of every streaming product of a layer (one at a time, but for u
// and dB): ranks up to 128 at a time.
int64_t lora_part_floats(int32_t S, int32_t K, int32_t N, int32_t rank) {
  const int64_t rp = (std::min(rank, 128) + 31) / 32 * 32;
  int32_t nsu = 1, nsb = 1, nsu1 = 1, none = 0;
  skinny_plan(S, N, true, &nsu, &nsb);
  skinny_plan(S, N, false, &nsu1, &none);
  return rp * std::max({(int64_t)nsu * S + (int64_t)nsb * N, (int64_t)nsu1 * S, (int64_t)stream_split(S, K) * S,
                        (int64_t)stream_split(K, S) * K});
}

// Ranks in launches of up to 128; the dropout output is written by the first
// (every launch draws the same bits).
void launch_lora_down(const LoraDownArgs &d, hipStream_t st) {
  for (int r0 = 0; r0 < d.rank; r0 += 128) {
    LoraStream a = {};
    a.x = d.x; a.x_rs = d.x_rs; a.rows = d.S; a.cols = d.K;
    a.sm = reinterpret_cast<const bf16_t *>(d.A) + (int64_t)r0 * d.a_rs; a.sm_rs = d.a_rs;
    a.part = d.part; a.rank = std::min(d.rank - r0, 128); a.ns = stream_split(d.S, d.K);
    a.keep_scale = d.keep_scale; a.thr = d.thr; a.seed = d.seed;
    a.h = r0 == 0 ? d.h : nullptr; a.h_rs = d.h_rs;
    const int rb = (a.rank + 31) / 32;
    if (far_rows(a)) down_rank<true>(a, d.thr > 0, st);
    else down_rank<false>(a, d.thr > 0, st);
    const int64_t n = (int64_t)d.S * (8 * rb);
    hipLaunchKernelGGL(lora_down_finish_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, 32 * rb,
                       d.gate, d.scaling, reinterpret_cast<bf16_t *>(d.t) + r0, d.t_rs);
  }
}

void launch_lora_da(const LoraDaArgs &d, hipStream_t st) {
  for (int r0 = 0; r0 < d.rank; r0 += 128) {
    LoraStream a = {};
    a.x = d.x; a.x_rs = d.x_rs; a.rows = d.S; a.cols = d.K;
    a.sm = reinterpret_cast<const bf16_t *>(d.da) + r0; a.sm_rs = d.da_rs;
    a.part = d.part; a.rank = std::min(d.rank - r0, 128); a.ns = stream_split(d.K, d.S);
    a.keep_scale = d.keep_scale; a.thr = d.thr; a.seed = d.seed;
    const int rb = (a.rank + 31) / 32;
    if (far_rows(a)) da_rank<true>(a, st);
    else da_rank<false>(a, st);
    const int64_t n = (int64_t)a.rank * (d.K / 4);
    hipLaunchKernelGGL(lora_da_finish_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, 32 * rb,
                       reinterpret_cast<bf16_t *>(d.dA) + (int64_t)r0 * d.dA_rs, d.dA_rs);
  }
}

void launch_lora_grad_ub(const LoraSkinnyArgs &d, float *part, const float *gate, float scaling, void *da,
                         int64_t da_rs, void *db, int64_t db_rs, hipStream_t st) {
  LoraStream u = {}, b = {};
  u.x = b.x = d.dy; u.x_rs = b.x_rs = d.dy_rs; u.rows = b.rows = d.S; u.cols = b.cols = d.N;
  u.rank = b.rank = d.rank;
  u.sm = d.b; u.sm_rs = d.b_rs; b.sm = d.t; b.sm_rs = d.t_rs;
  skinny_plan(d.S, d.N, db != nullptr, &u.ns, &b.ns);
  const int rb = (d.rank + 31) / 32;
  u.part = part;
  b.part = part + (int64_t)u.ns * d.S * (32 * rb);
  const dim3 grid((unsigned)(blocks128(d.S) * u.ns + blocks128(d.N) * b.ns)), blk(512);
  switch (rb) {
    case 1: hipLaunchKernelGGL(lora_skinny_kernel<1>, grid, blk, 0, st, u, b); break;
    case 2: hipLaunchKernelGGL(lora_skinny_kernel<2>, grid, blk, 0, st, u, b); break;
    case 3: hipLaunchKernelGGL(lora_skinny_kernel<3>, grid, blk, 0, st, u, b); break;
    default: hipLaunchKernelGGL(lora_skinny_kernel<4>, grid, blk, 0, st, u, b); break;
  }
  const int64_t n = ((int64_t)d.S + (b.ns > 0 ? d.N : 0)) * (8 * rb);
  hipLaunchKernelGGL(lora_skinny_finish_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, u, b, 32 * rb,
                     gate, scaling, reinterpret_cast<bf16_t *>(da), da_rs, reinterpret_cast<bf16_t *>(db), db_rs);
}

}  // namespace mga
