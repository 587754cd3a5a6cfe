// Stable soft cross-entropy of the MTP sampler loss (student logits x, teacher
// logits t, one row per drafted position) for gfx950. HBM-bound: each kernel
// streams its rows once.
//
// Forward, two or three launches:
//   soft_ce_partial_kernel  - grid (row, column split): one pass over a column
//       range of x and t keeps the online statistics of both rows at once,
//       (mx, dx) of x and (mt, dt, S = sum e^{t - mt} x) of t, and writes
//       them per split;
//   soft_ce_combine_kernel  - merges the splits of each row in a fixed order,
//       writes ce = -S / dt + mx + log dx and (mx, dx, mt, dt), and, at few
//       rows, sums the row losses (soft_ce_sum_kernel at many).
// The reference reads x twice (an x pass, then a fused t + x pass,
// mtp_glora/core/loss.py:63-124); here both rows are read once.
// Backward: grad_x = go * (e^{x - mx} / dx - e^{t - mt} / dt), written in the
// student's dtype (loss.py:188-222, 307-330).
// Exponentials are exp2 of log2(e)-scaled arguments; the clamps of dx and dt
// at 1e-20 follow loss.py:85, 112, 203-205.
#include "mga_common.hpp"
#include "mga_internal.hpp"

namespace mga {

namespace {

constexpr int kThreads = 256;
constexpr float kL2E = 1.4426950408889634f;
constexpr float kClamp = 1e-20f;
constexpr float kNegInf = -__builtin_huge_valf();
constexpr int kChunkQuantum = 2048;   // column split granularity (a multiple of every vector width)

__device__ __forceinline__ float ex2(float v) { return __builtin_amdgcn_exp2f(v); }

// Online statistics of one row segment: x: (mx, dx); t: (mt, dt, s).
struct Stats {
  float mx = kNegInf, dx = 0.f, mt = kNegInf, dt = 0.f, s = 0.f;

  // a group of n consecutive (x, t) values
  template <int N>
  __device__ __forceinline__ void add(const float (&x)[N], const float (&t)[N]) {
    float gx = x[0], gt = t[0];
#pragma unroll
    for (int i = 1; i < N; ++i) {
      gx = fmaxf(gx, x[i]);
      gt = fmaxf(gt, t[i]);
    }
    if (gx > mx) {   // never true for an all -inf group
      dx *= ex2((mx - gx) * kL2E);   // 0 while mx = -inf
      mx = gx;
    }
    if (gt > mt) {
      const float sc = ex2((mt - gt) * kL2E);
      dt *= sc;
      s *= sc;
      mt = gt;
    }
    // nothing but -inf so far: exponents of -inf, not of -inf + inf
    const float mxl = mx == kNegInf ? 0.f : mx * kL2E, mtl = mt == kNegInf ? 0.f : mt * kL2E;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      dx += ex2(__builtin_fmaf(x[i], kL2E, -mxl));
      const float e = ex2(__builtin_fmaf(t[i], kL2E, -mtl));
      dt += e;
      s = __builtin_fmaf(e, x[i], s);
    }
  }

  __device__ __forceinline__ void merge(const Stats &o) {
    const float nx = fmaxf(mx, o.mx);
    if (nx != kNegInf) {
      dx = dx * ex2((mx - nx) * kL2E) + o.dx * ex2((o.mx - nx) * kL2E);
      mx = nx;
    }
    const float nt = fmaxf(mt, o.mt);
    if (nt != kNegInf) {
      const float a = ex2((mt - nt) * kL2E), b = ex2((o.mt - nt) * kL2E);
      dt = dt * a + o.dt * b;
      s = s * a + o.s * b;
      mt = nt;
    }
  }

  __device__ __forceinline__ Stats shfl_xor(int m) const {
    Stats o;
    o.mx = __shfl_xor(mx, m, 64);
    o.dx = __shfl_xor(dx, m, 64);
    o.mt = __shfl_xor(mt, m, 64);
    o.dt = __shfl_xor(dt, m, 64);
    o.s = __shfl_xor(s, m, 64);
    return o;
  }
};

// 16-byte vectors of the element type <-> fp32.
template <typename T>
struct Vec {   // bf16 and fp16
  static constexpr int W = 8;
  __device__ __forceinline__ static void unpack(const i32x4 &r, float *v) {
    const auto a = __builtin_bit_cast(typename Elem<T>::v8, r);
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = (float)a[i];
  }
  __device__ __forceinline__ static i32x4 pack(const float (&v)[W]) {
    typename Elem<T>::v8 a;
#pragma unroll
    for (int i = 0; i < W; ++i) a[i] = (T)v[i];
    return __builtin_bit_cast(i32x4, a);
  }
};
template <>
struct Vec<float> {
  static constexpr int W = 4;
  __device__ __forceinline__ static void unpack(const i32x4 &r, float *v) {
    const f32x4 a = __builtin_bit_cast(f32x4, r);
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = a[i];
  }
  __device__ __forceinline__ static i32x4 pack(const float (&v)[W]) {
    return __builtin_bit_cast(i32x4, f32x4{v[0], v[1], v[2], v[3]});
  }
};

}  // namespace

// VEC: 16-byte vector loads (row starts 16-byte aligned); else element loads.
template <typename T, bool VEC>
__global__ __launch_bounds__(kThreads) void soft_ce_partial_kernel(const T *__restrict__ x, int64_t xs,
                                                                 const T *__restrict__ t, int64_t ts,
                                                                 int32_t V, int32_t chunk, int32_t nsplit,
                                                                 float *__restrict__ part) {
  const int tid = threadIdx.x;
  const int row = blockIdx.x / nsplit, sp = blockIdx.x - row * nsplit;
  const int c0 = sp * chunk, c1 = min(V, c0 + chunk);
  const T *xr = x + (int64_t)row * xs;
  const T *tr = t + (int64_t)row * ts;
  Stats st;
  int cs = c0;   // first column left for the element loop
  if constexpr (VEC) {
    // two vectors of x and of t per turn, the next turn's loads issued before
    // this turn's arithmetic (about 75 cycles of VALU work per wave and pair
    // against the streams' 100): [52, 151936] 11.0 -> 9.4 us, level at 1 024
    // rows, where the streams alone bound it (5.4 TB/s by itself, 4.5 TB/s
    // behind a backward whose gradient is still being written back)
    constexpr int W = Vec<T>::W;
    const int nvec = (c1 - c0) / W;
    const int nturn = nvec / (2 * kThreads);
    const i32x4 *xp = reinterpret_cast<const i32x4 *>(xr + c0) + tid;
    const i32x4 *tp = reinterpret_cast<const i32x4 *>(tr + c0) + tid;
    if (nturn > 0) {
      i32x4 xa = xp[0], ta = tp[0], xb = xp[kThreads], tb = tp[kThreads];
      for (int i = 1; i <= nturn; ++i) {
        const int n = min(i, nturn - 1) * 2 * kThreads;   // the last turn reads its own vectors again
        const i32x4 xc = xp[n], tc = tp[n], xd = xp[n + kThreads], td = tp[n + kThreads];
        float xv[2 * W], tv[2 * W];
        Vec<T>::unpack(xa, xv);
        Vec<T>::unpack(ta, tv);
        Vec<T>::unpack(xb, xv + W);
        Vec<T>::unpack(tb, tv + W);
        st.add(xv, tv);
        xa = xc; ta = tc; xb = xd; tb = td;
      }
    }
    for (int i = nturn * 2 * kThreads + tid; i < nvec; i += kThreads) {
      float xv[W], tv[W];
      Vec<T>::unpack(xp[i - tid], xv);
      Vec<T>::unpack(tp[i - tid], tv);
      st.add(xv, tv);
    }
    cs = c0 + nvec * W;
  }
  for (int c = cs + tid; c < c1; c += kThreads) {
    const float xv[1] = {(float)xr[c]}, tv[1] = {(float)tr[c]};
    st.add(xv, tv);
  }
  // wave, then workgroup (fixed order)
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) st.merge(st.shfl_xor(m));
  __shared__ float wst[kThreads / 64][5];
  if ((tid & 63) == 0) {
    float *o = wst[tid >> 6];
    o[0] = st.mx;
    o[1] = st.dx;
    o[2] = st.mt;
    o[3] = st.dt;
    o[4] = st.s;
  }
  __syncthreads();
  if (tid == 0) {
    Stats acc;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {
      Stats o;
      o.mx = wst[w][0];
      o.dx = wst[w][1];
      o.mt = wst[w][2];
      o.dt = wst[w][3];
      o.s = wst[w][4];
      acc.merge(o);
    }
    float *o = part + (int64_t)blockIdx.x * 5;
    o[0] = acc.mx;
    o[1] = acc.dx;
    o[2] = acc.mt;
    o[3] = acc.dt;
    o[4] = acc.s;
  }
}

// Sum of the workgroup's values, in a fixed order; on thread 0.
__device__ __forceinline__ float block_sum(float v) {
  const int tid = threadIdx.x;
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  __shared__ float wsum[16];
  if ((tid & 63) == 0) wsum[tid >> 6] = v;
  __syncthreads();
  v = tid < 16 ? wsum[tid] : 0.f;
  for (int m = 8; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// tpr (a power of two) neighbouring lanes take a row's splits and merge them in
// a fixed order. With sum (one workgroup then) the row losses are summed too, in
// a fixed order. Latency-bound (at most a few hundred KB): the splits' loads of
// a row run side by side, 10.8 us for one thread a row at 52 rows of 19 splits
// against 5.2 us, and the separate sum's launch is gone.
__global__ __launch_bounds__(1024) void soft_ce_combine_kernel(const float *__restrict__ part, int32_t N,
                                                               int32_t nsplit, int32_t tpr,
                                                               float *__restrict__ loss, float *__restrict__ stats,
                                                               float *__restrict__ sum) {
  const int tid = threadIdx.x, j = tid & (tpr - 1), rows = 1024 / tpr;
  float total = 0.f;
  for (int64_t r0 = (int64_t)blockIdx.x * rows; r0 < N; r0 += (int64_t)gridDim.x * rows) {
    const int64_t row = r0 + tid / tpr;
    Stats acc;
    if (row < N)
      for (int sp = j; sp < nsplit; sp += tpr) {
        const float *p = part + (row * nsplit + sp) * 5;
        Stats o;
        o.mx = p[0];
        o.dx = p[1];
        o.mt = p[2];
        o.dt = p[3];
        o.s = p[4];
        acc.merge(o);
      }
    for (int m = tpr >> 1; m >= 1; m >>= 1) acc.merge(acc.shfl_xor(m));
    if (row < N && j == 0) {
      const float dx = fmaxf(acc.dx, kClamp), dt = fmaxf(acc.dt, kClamp);
      const float ce = -(acc.s / dt) + acc.mx + logf(dx);
      total += ce;
      loss[row] = ce;
      stats[row] = acc.mx;
      stats[N + row] = dx;
      stats[2 * (int64_t)N + row] = acc.mt;
      stats[3 * (int64_t)N + row] = dt;
    }
  }
  if (!sum) return;
  total = block_sum(total);
  if (tid == 0) *sum = total;
}

// *sum = the row losses added in a fixed order, eight loads in flight a thread.
__global__ __launch_bounds__(1024) void soft_ce_sum_kernel(const float *__restrict__ loss, int32_t N,
                                                           float *__restrict__ sum) {
  float total = 0.f;
  for (int64_t r0 = 0; r0 < N; r0 += 8 * 1024) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t r = r0 + u * 1024 + threadIdx.x;
      v[u] = r < N ? loss[r] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) total += v[u];
  }
  total = block_sum(total);
  if (threadIdx.x == 0) *sum = total;
}

// Bound by the streams. The forward walks every row's columns upwards, all rows
// side by side, so what the last-level cache (256 MB) still holds of x and t are
// the last columns: this kernel starts at the end and walks down. NT: the
// gradient is written past the cache, so that it does not push them out (the rule
// is at kCachedBytes). The next turn's loads are issued before this turn's
// arithmetic, as in the forward. Loss + gradient, bf16 x 151 936, upwards with
// ordinary stores / downwards / downwards past the cache: 1 024 rows 318 / 287 /
// 267 us, 400 rows 109 / 109 / 99 us, 200 rows 59 / 57 / 57 us.
template <typename T, bool VEC, bool NT>
__global__ __launch_bounds__(kThreads) void soft_ce_bwd_kernel(const T *__restrict__ x, int64_t xs,
                                                             const T *__restrict__ t, int64_t ts, int32_t V,
                                                             int32_t chunk, int32_t nsplit, int32_t N,
                                                             const float *__restrict__ grad_out,
                                                             const float *__restrict__ stats,
                                                             T *__restrict__ g, int64_t gs) {
  const int tid = threadIdx.x;
  const int b = gridDim.x - 1 - blockIdx.x;
  const int row = b / nsplit, sp = b - row * nsplit;
  const int c0 = sp * chunk, c1 = min(V, c0 + chunk);
  const T *xr = x + (int64_t)row * xs;
  const T *tr = t + (int64_t)row * ts;
  T *gr = g + (int64_t)row * gs;
  const float go = *grad_out;
  const float mxl = stats[row] * kL2E, mtl = stats[2 * N + row] * kL2E;
  // saved values are clamped already; clamping again matches loss.py:203-205
  const float ax = go / fmaxf(stats[N + row], kClamp), at = go / fmaxf(stats[3 * N + row], kClamp);
  constexpr int W = Vec<T>::W;
  const int nvec = VEC ? (c1 - c0) / W : 0;
  for (int c = c0 + nvec * W + tid; c < c1; c += kThreads) {
    const float xv = (float)xr[c], tv = (float)tr[c];
    gr[c] = (T)(ax * ex2(__builtin_fmaf(xv, kL2E, -mxl)) - at * ex2(__builtin_fmaf(tv, kL2E, -mtl)));
  }
  if constexpr (VEC) {
    const i32x4 *xp = reinterpret_cast<const i32x4 *>(xr + c0) + tid;
    const i32x4 *tp = reinterpret_cast<const i32x4 *>(tr + c0) + tid;
    T *gp = gr + c0 + tid * W;
    auto put = [&](int i, const i32x4 &xa, const i32x4 &ta) {
      float xv[W], tv[W], gv[W];
      Vec<T>::unpack(xa, xv);
      Vec<T>::unpack(ta, tv);
#pragma unroll
      for (int e = 0; e < W; ++e)
        gv[e] = ax * ex2(__builtin_fmaf(xv[e], kL2E, -mxl)) - at * ex2(__builtin_fmaf(tv[e], kL2E, -mtl));
      i32x4 *out = reinterpret_cast<i32x4 *>(gp + (int64_t)i * W);
      if constexpr (NT) __builtin_nontemporal_store(Vec<T>::pack(gv), out);
      else *out = Vec<T>::pack(gv);
    };
    const int nturn = nvec / (2 * kThreads);
    for (int i = nturn * 2 * kThreads; i + tid < nvec; i += kThreads) put(i, xp[i], tp[i]);
    if (nturn > 0) {
      int n = (nturn - 1) * 2 * kThreads;
      i32x4 xa = xp[n], ta = tp[n], xb = xp[n + kThreads], tb = tp[n + kThreads];
      while (n > 0) {
        n -= 2 * kThreads;
        const i32x4 xc = xp[n], tc = tp[n], xd = xp[n + kThreads], td = tp[n + kThreads];
        put(n + 3 * kThreads, xb, tb);
        put(n + 2 * kThreads, xa, ta);
        xa = xc; ta = tc; xb = xd; tb = td;
      }
      put(kThreads, xb, tb);
      put(0, xa, ta);
    }
  }
}

// Column split of the rows: enough workgroups to fill the chip (about 1024),
// each over a multiple of kChunkQuantum columns.
void soft_ce_plan(int32_t N, int32_t V, int32_t *nsplit, int32_t *chunk) {
  const int64_t want = (1024 + N - 1) / N;
  const int64_t maxs = (V + 4095) / 4096;
  int64_t s = want < maxs ? want : maxs;
  if (s < 1) s = 1;
  int64_t c = (V + s - 1) / s;
  c = (c + kChunkQuantum - 1) / kChunkQuantum * kChunkQuantum;
  *chunk = (int32_t)c;
  *nsplit = (int32_t)((V + c - 1) / c);
}

int64_t soft_ce_workspace_floats(int32_t N, int32_t V) {
  int32_t ns, ch;
  soft_ce_plan(N, V, &ns, &ch);
  return (int64_t)N * ns * 5;
}

// Passes over the rows up to which one workgroup combines and sums them; beyond,
// every pass is a workgroup and the sum a launch of its own. Whole forward, bf16
// x 1 024 columns (a pass is 1 024 rows), one workgroup / one a pass: 2 048 rows
// 10.8 / 11.6 us, 3 072 rows 13.3 / 13.3, 4 096 rows 15.9 / 15.1, 16 384 rows 46.7 /
// 36.6; 65 536 rows of 512 columns 152 / 105 us.
constexpr int kOneGroupPasses = 3;

template <typename T>
static void fwd_typed(const void *x, int64_t xs, const void *t, int64_t ts, int32_t N, int32_t V, bool vec,
                      float *loss, float *stats, float *sum, float *ws, hipStream_t st) {
  int32_t ns, ch;
  soft_ce_plan(N, V, &ns, &ch);
  const dim3 grid((unsigned)((int64_t)N * ns));
  if (vec)
    hipLaunchKernelGGL((soft_ce_partial_kernel<T, true>), grid, dim3(kThreads), 0, st, (const T *)x, xs,
                       (const T *)t, ts, V, ch, ns, ws);
  else
    hipLaunchKernelGGL((soft_ce_partial_kernel<T, false>), grid, dim3(kThreads), 0, st, (const T *)x, xs,
                       (const T *)t, ts, V, ch, ns, ws);
  int tpr = 1;
  while (tpr < ns && tpr < 64) tpr *= 2;
  const int passes = (int)(((int64_t)N * tpr + 1023) / 1024);   // of one workgroup over the rows
  const bool one = sum && passes <= kOneGroupPasses;
  hipLaunchKernelGGL(soft_ce_combine_kernel, dim3(one ? 1 : passes), dim3(1024), 0, st, ws, N, ns, tpr, loss, stats,
                     one ? sum : nullptr);
  if (sum && !one) hipLaunchKernelGGL(soft_ce_sum_kernel, dim3(1), dim3(1024), 0, st, loss, N, sum);
}

// Bytes of x, t and their gradient up to which the last-level cache holds all
// three: the gradient is then written into it, where the next operation (the
// head's backward) finds it. Loss + gradient + a copy of the gradient, bf16 x
// 151 936, ordinary / past the cache: 52 rows 30.4 / 31.6 us, 200 rows (182 MB)
// 74.5 / 78.7, 250 rows (228 MB) 93.5 / 95.5, without the copy 66.7 / 66.6, with x
// just written too 126 / 117; 300 rows 124 / 116 us.
constexpr int64_t kCachedBytes = 200 << 20;

template <typename T>
static void bwd_typed(const void *x, int64_t xs, const void *t, int64_t ts, int32_t N, int32_t V, bool vec,
                      const float *go, const float *stats, void *g, int64_t gs, hipStream_t st) {
  int32_t ns, ch;
  soft_ce_plan(N, V, &ns, &ch);
  const dim3 grid((unsigned)((int64_t)N * ns));
  const bool nt = 3 * (int64_t)N * V * (int64_t)sizeof(T) > kCachedBytes;
  auto run = [&](auto k) {
    hipLaunchKernelGGL(k, grid, dim3(kThreads), 0, st, (const T *)x, xs, (const T *)t, ts, V, ch, ns, N, go, stats,
                       (T *)g, gs);
  };
  if (vec && nt) run(soft_ce_bwd_kernel<T, true, true>);
  else if (vec) run(soft_ce_bwd_kernel<T, true, false>);
  else run(soft_ce_bwd_kernel<T, false, false>);
}

void launch_soft_ce_fwd(const void *x, int64_t xs, const void *t, int64_t ts, int32_t N, int32_t V, int dtype,
                        bool vec, float *loss, float *stats, float *sum, float *ws, hipStream_t st) {
  if (dtype == kDtF32) fwd_typed<float>(x, xs, t, ts, N, V, vec, loss, stats, sum, ws, st);
  else if (dtype == kDtF16) fwd_typed<f16_t>(x, xs, t, ts, N, V, vec, loss, stats, sum, ws, st);
  else fwd_typed<bf16_t>(x, xs, t, ts, N, V, vec, loss, stats, sum, ws, st);
}

void launch_soft_ce_bwd(const void *x, int64_t xs, const void *t, int64_t ts, int32_t N, int32_t V, int dtype,
                        bool vec, const float *go, const float *stats, void *g, int64_t gs, hipStream_t st) {
  if (dtype == kDtF32) bwd_typed<float>(x, xs, t, ts, N, V, vec, go, stats, g, gs, st);
  else if (dtype == kDtF16) bwd_typed<f16_t>(x, xs, t, ts, N, V, vec, go, stats, g, gs, st);
  else bwd_typed<bf16_t>(x, xs, t, ts, N, V, vec, go, stats, g, gs, st);
}

}  // namespace mga
