// MTP block-mask construction on the GPU: per-token codes, 128x128 tile
// classes, and the eight ordered BlockMask index tensors.
//
// The tensors equal what create_block_mask returns for the reference's
// mask_mod (mtp_glora/data_utils/collator.py:290-363): tiles are padded with
// False to a multiple of 128 ([torch]nn/attention/flex_attention.py:979-1022),
// a tile is "full" when all 128*128 entries are allowed and "partial" when some
// are, and every index row is the selected tiles ascending followed by the
// rest ascending (the stable descending argsort of :429-436; the q-major lists
// are the transposes of :439-441).
#include "mga_common.hpp"
#include "mga_internal.hpp"

namespace mga {

// ---- codes ----------------------------------------------------------------
// code[i] = -1 pad, -2 regular, else P + #(gate == 0 in [0, i]) -- the
// num_prefix_x of collator.py:320 for a mask token (the P cached tokens are
// all regular, collator.py:311-318). Latency bound: two rounds of loads and one
// barrier; 5120 tokens in 4.5 us (5.7 us with a segment per thread and a scan
// of 10 steps over the threads' counts).
__global__ __launch_bounds__(1024) void mtp_codes_kernel(const int64_t *__restrict__ gate,
                                                         int64_t stride, int32_t n, int64_t P,
                                                         int32_t *__restrict__ code) {
  __shared__ int sums[16];
  const int lane = threadIdx.x & 63;
  const WaveSpan s = scan_flags(n, sums, [&](int i) { return gate[(int64_t)i * stride] == 0; });
  int run = s.before;   // zeros before these 64 tokens
  for (int i0 = s.begin; i0 < s.end; i0 += 512) {
    int64_t g[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) g[u] = gate[(int64_t)min(i0 + 64 * u + lane, n - 1) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + 64 * u + lane;
      const bool x = g[u] == 0 && i < s.end;
      const uint64_t m = __ballot(x);
      const int upto = run + __popcll(m & lanes_below()) + x;
      if (i < s.end) code[i] = g[u] == -1 ? kCodePad : (x ? kCodeX : (int)(P + upto));
      run += __popcll(m);
    }
  }
}

// ---- tile classes -----------------------------------------------------------
// grid (1 + chunk tiles, nQ); class 0 empty, 1 partial, 2 full. Column 0 takes
// all tiles of cached tokens, which have one class per query tile: a key there
// is visible to every query that is no pad. The others count the visible pairs
// of 64 rows x 64 keys per wave from two 64-bit masks, regular keys (visible
// if not later than the query: one popcount a row) and mask keys (visible to
// the mask queries of their own block: compared one by one). Bound by the
// launch and the reduction. Per-pair compares with a workgroup for every tile:
// 12.3 us for 5120 tokens after 8192, so: 4.6 us.
__global__ __launch_bounds__(256) void tile_class_kernel(const int32_t *__restrict__ code, int32_t S,
                                                         int32_t P, int32_t L, int32_t nKV,
                                                         int8_t *__restrict__ cls) {
  __shared__ int red[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int q0 = blockIdx.y * kBlock, cached = P / kBlock;
  const int kt = cached + (int)blockIdx.x - 1;
  const int k0 = kt * kBlock;
  int8_t *row_cls = cls + (int64_t)blockIdx.y * nKV;
  if (blockIdx.x > 0 && k0 > min(q0 + kBlock, S) - 1 + P) {
    // every key follows every query of the tile: causally empty
    if (t == 0) row_cls[kt] = 0;
    return;
  }
  const int row = q0 + (wave & 1) * 64 + lane;
  const int qc = row < S ? code[row] : kCodePad;
  int cnt = 0;
  if (blockIdx.x == 0) {
    cnt = qc != kCodePad ? kBlock / 2 : 0;   // two waves per row
  } else {
    const int key = k0 + (wave >> 1) * 64;
    const int kc = key_code(code, key + lane, P, L);
    const uint64_t keys_x = __ballot(kc == kCodeX);
    uint64_t keys_m = __ballot(kc != kCodeX && kc != kCodePad);
    const int seen = min(row + P - key + 1, 64);   // keys not later than the query
    const uint64_t causal = seen <= 0 ? 0 : ~uint64_t(0) >> (64 - seen);
    if (qc != kCodePad) cnt = __popcll(keys_x & causal);
    if (__ballot(qc != kCodePad && qc != kCodeX))
      while (keys_m) {
        const int j = __builtin_ctzll(keys_m);
        keys_m &= keys_m - 1;
        cnt += (int)(__builtin_amdgcn_readlane(kc, j) == qc && (causal >> j & 1));
      }
  }
  for (int off = 32; off > 0; off >>= 1) cnt += __shfl_down(cnt, off, 64);
  if (lane == 0) red[wave] = cnt;
  __syncthreads();
  const int tot = red[0] + red[1] + red[2] + red[3];
  const int8_t c = tot == kBlock * kBlock ? 2 : (tot > 0 ? 1 : 0);
  if (blockIdx.x == 0) {
    for (int i = t; i < cached; i += 256) row_cls[i] = c;
  } else if (t == 0) {
    row_cls[kt] = c;
  }
}

// ---- ordered lists ------------------------------------------------------------
// Block-wide exclusive scan of one flag per thread (256 threads).
__device__ __forceinline__ int block_excl_scan(int f, int *buf, int &total) {
  const int wave = threadIdx.x >> 6;
  const uint64_t m = __ballot(f);
  if ((threadIdx.x & 63) == 0) buf[wave] = __popcll(m);
  __syncthreads();
  int before = __popcll(m & lanes_below());
  total = 0;
  for (int w = 0; w < 4; ++w) {
    before += w < wave ? buf[w] : 0;
    total += buf[w];
  }
  __syncthreads();
  return before;
}

// Writes num = #selected and idx[0..n) = selected ascending then the rest ascending.
__device__ void ordered_row(const int8_t *cls, int64_t step, int n, int want, int32_t *num,
                            int32_t *idx, int *buf) {
  int tot_sel = 0;
  for (int b = 0; b < n; b += 256) {
    const int j = b + threadIdx.x;
    const int f = (j < n) && cls[j * step] == want;
    int chunk_tot;
    block_excl_scan(f, buf, chunk_tot);
    tot_sel += chunk_tot;
  }
  int carry = 0;
  for (int b = 0; b < n; b += 256) {
    const int j = b + threadIdx.x;
    const int f = (j < n) && cls[j * step] == want;
    int chunk_tot;
    const int before = block_excl_scan(f, buf, chunk_tot);
    if (j < n) {
      const int sel_before = carry + before;
      const int pos = f ? sel_before : tot_sel + (j - sel_before);
      idx[pos] = j;
    }
    carry += chunk_tot;
  }
  if (threadIdx.x == 0) *num = tot_sel;
}

// grid nQ + nKV: rows (kv lists per q tile) then columns (q lists per kv tile).
__global__ __launch_bounds__(256) void block_lists_kernel(
    const int8_t *__restrict__ cls, int32_t nQ, int32_t nKV, int32_t *kv_num, int32_t *kv_idx,
    int32_t *full_kv_num, int32_t *full_kv_idx, int32_t *q_num, int32_t *q_idx,
    int32_t *full_q_num, int32_t *full_q_idx) {
  __shared__ int buf[4];
  const int b = blockIdx.x;
  if (b < nQ) {
    const int8_t *row = cls + (int64_t)b * nKV;
    ordered_row(row, 1, nKV, 1, kv_num + b, kv_idx + (int64_t)b * nKV, buf);
    ordered_row(row, 1, nKV, 2, full_kv_num + b, full_kv_idx + (int64_t)b * nKV, buf);
  } else {
    const int c = b - nQ;
    const int8_t *col = cls + c;
    ordered_row(col, nKV, nQ, 1, q_num + c, q_idx + (int64_t)c * nQ, buf);
    ordered_row(col, nKV, nQ, 2, full_q_num + c, full_q_idx + (int64_t)c * nQ, buf);
  }
}

void launch_mtp_block_mask(const int64_t *gate, int64_t gate_stride, int32_t S, int64_t P,
                           int32_t *code, int8_t *cls, int32_t *kv_num, int32_t *kv_idx,
                           int32_t *full_kv_num, int32_t *full_kv_idx, int32_t *q_num,
                           int32_t *q_idx, int32_t *full_q_num, int32_t *full_q_idx,
                           hipStream_t stream) {
  const int L = (int)(P + S);
  const int nQ = (S + kBlock - 1) / kBlock;
  const int nKV = (L + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(mtp_codes_kernel, dim3(1), dim3(1024), 0, stream, gate, gate_stride, S, P,
                     code);
  hipLaunchKernelGGL(tile_class_kernel, dim3(1 + nKV - (int)(P / kBlock), nQ), dim3(256), 0, stream, code, S, (int)P, L,
                     nKV, cls);
  hipLaunchKernelGGL(block_lists_kernel, dim3(nQ + nKV), dim3(256), 0, stream, cls, nQ, nKV, kv_num,
                     kv_idx, full_kv_num, full_kv_idx, q_num, q_idx, full_q_num, full_q_idx);
}

}  // namespace mga
