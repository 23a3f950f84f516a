// Packed depthwise causal conv1d, forward and backward (the GatedDelta layer's
// short conv over q/k/v channels, ops/gated_delta_net.py:252-289; the
// reference runs causal_conv1d_fn / causal_conv1d_bwd, models/backbone_qwen35.py
// keeps the CPU form F.conv1d(padding = K - 1) per document).
//
//   pre[t][c] = sum_{i<K} w[c][i] * x[t - (K-1) + i][c]   (rows of the same document only)
//   y = silu(pre) with the activation, else pre
//
// x, y, dy, dx: bf16 [T][C] (time-first, B = 1, packed documents); w: bf16
// [C][K], K <= 4.  Row u of x may be read through a row map (x row xrows[u],
// xs elements apart) and row t of dx written through its own map (dx row
// dxrows[t], dxs apart; null: row t):
// the layer's content gather updates = raw.index_select(0, content_order)
// (models/backbone_qwen35.py:167) and its backward, consumed in the loads and
// stores.  A thread owns 8 consecutive channels (16-byte accesses, a
// wave covers 512 channels of one row: 1 KB per load or store); a tap on a row
// of another document contributes nothing.  The forward requests every row of
// a CONV_ROWS tile (with the K - 1 row halo) before computing; the backward
// (CONV_BWD_CH channels per thread) streams longer strips with its loads one
// row group ahead, so that it writes few dw partials.  Both passes are
// HBM-bound.
#include "gdn_common.hpp"
#include "gdn_kernels.hpp"

#include <climits>

namespace cqgdn {

constexpr int CONV_ROWS = 16;     // rows per workgroup
constexpr int CONV_THREADS = 256; // 2048 channels per workgroup

// first index i with bounds[i] >= v (bounds ascending, n + 1 entries)
__device__ __forceinline__ int lower_bound(const int32_t* __restrict__ bounds, int n, int v) {
  int lo = 0, hi = n + 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (bounds[mid] < v) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Tracks the start of the document holding row u as u increases from u0.
// The next bound is kept in a register (nb), so a row that crosses no document
// boundary costs a compare, not a load and its wait.
struct DocCursor {
  const int32_t* bounds;
  int n, next, start, nb;  // nb = bounds[next], or INT_MAX past the last bound
  __device__ DocCursor(const int32_t* b, int n_docs, int u0) : bounds(b), n(n_docs) {
    int i = lower_bound(b, n_docs, u0 + 1) - 1;  // last bound <= u0
    i = max(i, 0);
    start = b[i];
    next = i + 1 <= n_docs ? i + 1 : n_docs;
    nb = next <= n ? b[next] : INT_MAX;
  }
  __device__ __forceinline__ void advance_to(int u) {
    while (nb <= u) {
      start = nb;
      ++next;
      nb = next <= n ? bounds[next] : INT_MAX;
    }
  }
};

// sigmoid through v_rcp_f32 (1 ulp) rather than an IEEE divide; exp(-x) = inf gives 0
__device__ __forceinline__ float sigmoid_f(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x * sigmoid_f(x); }
__device__ __forceinline__ float dsilu_f(float x) {
  const float s = sigmoid_f(x);
  return s * (1.f + x * (1.f - s));
}

template <int K>
__global__ __launch_bounds__(CONV_THREADS) void conv_fwd_kernel(const bf16* __restrict__ x, const int32_t* __restrict__ xrows,
                                                               int64_t xs, const bf16* __restrict__ w,
                                                               const int32_t* __restrict__ bounds, int n_docs,
                                                               int T, int C, int act, bf16* __restrict__ y) {
  const int c = (blockIdx.y * CONV_THREADS + threadIdx.x) * 8;
  if (c >= C) return;
  const int s = blockIdx.x * CONV_ROWS;
  const int u0 = s - (K - 1);
  // every row of the tile and its halo is requested before any is used
  bf16x8 xr[CONV_ROWS + K - 1];
#pragma unroll
  for (int i = 0; i < CONV_ROWS + K - 1; ++i) {
    const int u = min(max(u0 + i, 0), T - 1);  // rows outside [0, T) are never used
    xr[i] = ld8(x + (xrows ? (int64_t)xrows[u] : (int64_t)u) * xs + c);
  }
  f32x8 wk[K];
  {
    const bf16* wc = w + (size_t)c * K;  // 8 channels x K taps, contiguous
#pragma unroll
    for (int ch = 0; ch < 8; ++ch)
#pragma unroll
      for (int i = 0; i < K; ++i) wk[i][ch] = (float)wc[ch * K + i];
  }
  DocCursor doc(bounds, n_docs, max(s, 0));
#pragma unroll
  for (int r = 0; r < CONV_ROWS; ++r) {
    const int t = s + r;
    if (t >= T) break;
    doc.advance_to(t);
    f32x8 acc = f32x8{};
#pragma unroll
    for (int i = 0; i < K; ++i)  // tap i reads row t - (K-1) + i = xr[r + i]
      if (t - (K - 1) + i >= doc.start) acc += wk[i] * cvtf8(xr[r + i]);
    if (act) {
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) acc[ch] = silu_f(acc[ch]);
    }
    st8(y + (size_t)t * C + c, cvt8(acc));
  }
}

// Backward: a wave streams a strip of rows [s, e) for 64 * CONV_BWD_CH channels, walking u =
// s - (K-1) .. e + K - 2 in groups of K rows whose x and dy rows are requested while the previous
// group computes (a gathered x row's index one group before that).  Per row u:
//   pre[u] from the last K x rows, dpre[u] = dy[u] * silu'(pre[u]),
//   dw partials over u in [s, e),
//   dx[t] = sum_j w[K-1-j] * dpre[t + j] over rows t + j of t's document.
// The last K x rows (fp32) and dpre rows sit in rings indexed by the row's
// place in its group, so the windows advance without register moves.  A strip
// whose rows u0 .. uend-1 hold no document boundary (0 and T included) runs
// without any per-row document test (DOCS = false).  A workgroup is four
// neighbouring strips, whose rows overlap by K - 1 on each side: it sums their dw
// partials in LDS, in strip order, and writes one [C][K] part; colsum_kernel (event_sums_kernel in a layer)
// sums the parts.  Bound by the memory traffic: 8192 rows of 6144 channels take 65.7 us (58 at a large copy's rate),
// 2048 rows 23.5; a one-wave workgroup and a part per strip took 69.7 and 25.5.
constexpr int CONV_STRIPS = 128;  // row strips per 64 * CONV_BWD_CH channels, at least
constexpr int CONV_MIN_GROUPS = 512;  // workgroups to ask for in all: two per CU
constexpr int CONV_BWD_WAVES = 4; // strips per workgroup
constexpr int CONV_BWD_CH = 4;    // channels per thread in the backward

template <int CH> struct ConvVec;
template <> struct ConvVec<8> { typedef bf16x8 b; typedef f32x8 f; };
template <> struct ConvVec<4> { typedef bf16x4 b; typedef f32x4 f; };

template <int K, int CH, bool DOCS>
__device__ __forceinline__ void conv_bwd_strip(const bf16* __restrict__ x, const int32_t* __restrict__ rows,
                                               int64_t xstr, const typename ConvVec<CH>::f (&wk)[K],
                                               const bf16* __restrict__ dy, const int32_t* __restrict__ bounds,
                                               int n_docs, int T, int C, int c, int s, int e, int act,
                                               bf16* __restrict__ dx, const int32_t* __restrict__ dxrows, int64_t dxs,
                                               typename ConvVec<CH>::f (&dwa)[K]) {
  typedef typename ConvVec<CH>::b bv;
  typedef typename ConvVec<CH>::f fv;
  const int u0 = s - (K - 1), uend = e + K - 1;
  bv nx[K], nd[K];  // the next group's rows (clamped into [0, T); rows outside are never used)
  int nr[K];        // the x rows of the group after it
  auto place = [&](int u) { return min(max(u, 0), T - 1); };
  auto index = [&](int ub) {
#pragma unroll
    for (int j = 0; j < K; ++j) nr[j] = rows ? rows[place(ub + j)] : place(ub + j);
  };
  auto request = [&](int ub) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      nx[j] = *reinterpret_cast<const bv*>(x + (int64_t)nr[j] * xstr + c);
      nd[j] = *reinterpret_cast<const bv*>(dy + (int64_t)place(ub + j) * C + c);
    }
    index(ub + K);
  };
  index(u0);
  request(u0);
  // ring slot j holds the row at place j of the current group (rows before u0 are never read)
  fv xs[K], dp[K];
  int st[K];  // document start of each dpre ring row (-1: no row)
#pragma unroll
  for (int i = 0; i < K; ++i) {
    dp[i] = fv{};
    st[i] = -1;
  }
  DocCursor doc(bounds, n_docs, s);
  for (int ub = u0; ub < uend; ub += K) {
    bv cx[K], cd[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      cx[j] = nx[j];
      cd[j] = nd[j];
    }
    if (ub + K < uend) request(ub + K);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int u = ub + j;
      // slot j still holds row u - K until here: the taps of the rows before u read it
      xs[j] = __builtin_convertvector(cx[j], fv);
      if (u >= uend) break;
      if (u < s) continue;
      fv dpu = fv{};
      int stu = 0;
      if (!DOCS || u < T) {
        if (DOCS) {
          doc.advance_to(u);
          stu = __builtin_amdgcn_readfirstlane(doc.start);
        }
        // tap i reads row u - (K-1) + i, ring slot (j + 1 + i) % K
        fv pre = wk[K - 1] * xs[j];
#pragma unroll
        for (int i = 0; i < K - 1; ++i)
          if (!DOCS || u - (K - 1) + i >= stu) pre += wk[i] * xs[(j + 1 + i) % K];
        dpu = __builtin_convertvector(cd[j], fv);
        if (act) {
#pragma unroll
          for (int ch = 0; ch < CH; ++ch) dpu[ch] *= dsilu_f(pre[ch]);
        }
        if (u < e) {
          dwa[K - 1] += dpu * xs[j];
#pragma unroll
          for (int i = 0; i < K - 1; ++i)
            if (!DOCS || u - (K - 1) + i >= stu) dwa[i] += dpu * xs[(j + 1 + i) % K];
        }
      } else {
        stu = -1;
      }
      dp[j] = dpu;
      if (DOCS) st[j] = stu;
      const int t = u - (K - 1);
      if (t >= s && t < e) {  // dpre[t + m] is ring slot (j + 1 + m) % K, tap K-1-m, same document only
        fv acc = wk[K - 1] * dp[(j + 1) % K];
#pragma unroll
        for (int m = 1; m < K; ++m)
          if (!DOCS || st[(j + 1 + m) % K] == st[(j + 1) % K]) acc += wk[K - 1 - m] * dp[(j + 1 + m) % K];
        *reinterpret_cast<bv*>(dx + (dxrows ? (int64_t)dxrows[t] : (int64_t)t) * dxs + c) =
            __builtin_convertvector(acc, bv);
      }
    }
  }
}

template <int K>
__global__ __launch_bounds__(64 * CONV_BWD_WAVES) void conv_bwd_kernel(
    const bf16* __restrict__ x, const int32_t* __restrict__ xrows, int64_t xs, const bf16* __restrict__ w,
    const bf16* __restrict__ dy, const int32_t* __restrict__ bounds, int n_docs, int T, int C, int rows, int act,
    bf16* __restrict__ dx, const int32_t* __restrict__ dxrows, int64_t dxs, float* __restrict__ dw_part) {
  constexpr int CH = CONV_BWD_CH;
  typedef typename ConvVec<CH>::f fv;
  __shared__ fv red[CONV_BWD_WAVES - 1][K][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = (blockIdx.y * 64 + lane) * CH;
  const int s = (blockIdx.x * CONV_BWD_WAVES + wave) * rows, e = min(s + rows, T);
  fv dwa[K];
#pragma unroll
  for (int i = 0; i < K; ++i) dwa[i] = fv{};
  if (c < C && s < T) {
    fv wk[K];
    const bf16* wc = w + (size_t)c * K;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch)
#pragma unroll
      for (int i = 0; i < K; ++i) wk[i][ch] = (float)wc[ch * K + i];
    // a boundary b with u0 < b < uend separates two rows of the walk (b = 0 and b = T included)
    const int u0 = s - (K - 1), uend = e + K - 1;
    const int i = lower_bound(bounds, n_docs, u0 + 1);
    const bool docs = __builtin_amdgcn_readfirstlane(i <= n_docs && bounds[i] < uend);
    if (docs)
      conv_bwd_strip<K, CH, true>(x, xrows, xs, wk, dy, bounds, n_docs, T, C, c, s, e, act, dx, dxrows, dxs, dwa);
    else
      conv_bwd_strip<K, CH, false>(x, xrows, xs, wk, dy, bounds, n_docs, T, C, c, s, e, act, dx, dxrows, dxs, dwa);
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < K; ++i) red[wave - 1][i][lane] = dwa[i];
  }
  __syncthreads();
  if (wave > 0 || c >= C) return;
#pragma unroll
  for (int v = 0; v < CONV_BWD_WAVES - 1; ++v)
#pragma unroll
    for (int i = 0; i < K; ++i) dwa[i] += red[v][i][lane];
  float* part = dw_part + ((size_t)blockIdx.x * C + c) * K;
#pragma unroll
  for (int ch = 0; ch < CH; ++ch)
#pragma unroll
    for (int k = 0; k < K; ++k) part[ch * K + k] = dwa[k][ch];
}

// dw[j] = sum over strips of the partials [strips][n] (n % 4 == 0; the conv's dw
// and the other per-workgroup parameter-gradient partials): a lane owns 4
// consecutive j (16-byte loads), a workgroup 256 j; its 4 waves sum strips
// b = wave, wave + 4, ... with 8 loads in flight, and the four sums are added
// in wave order (fixed order: deterministic).
__global__ __launch_bounds__(256) void colsum_kernel(const float* __restrict__ part, int strips, int n,
                                                    float* __restrict__ dw) {
  __shared__ f32x4 red[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = (blockIdx.x * 64 + lane) * 4;
  f32x4 acc = f32x4{};
  if (j < n) {
    const f32x4* p = reinterpret_cast<const f32x4*>(part + j);
    const size_t stride = (size_t)n / 4;
    int b = wave;
    for (; b + 28 < strips; b += 32) {
      f32x4 v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = p[(size_t)(b + 4 * q) * stride];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc += v[q];
    }
    for (; b < strips; b += 4) acc += p[(size_t)b * stride];
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && j < n) {
    const f32x4 r = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
#pragma unroll
    for (int q = 0; q < 4; ++q) dw[j + q] = r[q];
  }
}

// Rows of a strip: 16 at least (2 (K - 1) more are read), else T over the strips.  Where
// CONV_STRIPS strips in fours make fewer workgroups than CONV_MIN_GROUPS (below 4096 channels) there are
// as many more strips as make that many: with CONV_STRIPS alone whole CUs had nothing to read
// (65536 rows of 512 / 1536 / 2048 / 3072 channels 266 / 296 / 299 / 337 us, now 53 / 161 / 190 / 309; 8192 rows 43 / 44 / 45 /
// 50, now 21 / 31 / 32 / 45; with 256 workgroups 78 / 226 / 299 / 337).
int conv_strip_rows(int64_t T, int C) {
  const int blocks = (C + 64 * CONV_BWD_CH - 1) / (64 * CONV_BWD_CH);
  const int strips = std::max(CONV_STRIPS, (CONV_MIN_GROUPS + blocks - 1) / blocks * CONV_BWD_WAVES);
  return (int)std::max<int64_t>(16, (T + strips - 1) / strips);
}

int conv_parts(int64_t T, int C) {
  const int64_t rows = (int64_t)conv_strip_rows(T, C) * CONV_BWD_WAVES;
  return (int)((T + rows - 1) / rows);
}

void launch_conv_fwd(const bf16* x, const int32_t* xrows, int64_t xs, const bf16* w, const int32_t* bounds,
                     int n_docs, int T, int C, int K, int act, bf16* y, hipStream_t stream) {
  const dim3 grid((T + CONV_ROWS - 1) / CONV_ROWS, (C / 8 + CONV_THREADS - 1) / CONV_THREADS);
  switch (K) {
    case 2: hipLaunchKernelGGL(conv_fwd_kernel<2>, grid, dim3(CONV_THREADS), 0, stream, x, xrows, xs, w, bounds, n_docs, T, C, act, y); break;
    case 3: hipLaunchKernelGGL(conv_fwd_kernel<3>, grid, dim3(CONV_THREADS), 0, stream, x, xrows, xs, w, bounds, n_docs, T, C, act, y); break;
    default: hipLaunchKernelGGL(conv_fwd_kernel<4>, grid, dim3(CONV_THREADS), 0, stream, x, xrows, xs, w, bounds, n_docs, T, C, act, y); break;
  }
}

void launch_conv_bwd(const bf16* x, const int32_t* xrows, int64_t xs, const bf16* w, const bf16* dy,
                     const int32_t* bounds, int n_docs, int T, int C, int K, int act, bf16* dx, const int32_t* dxrows,
                     int64_t dxs, float* part, hipStream_t stream) {
  const int rows = conv_strip_rows(T, C), parts = conv_parts(T, C);
  const dim3 grid(parts, (C / CONV_BWD_CH + 63) / 64), block(64 * CONV_BWD_WAVES);
  switch (K) {
    case 2: hipLaunchKernelGGL(conv_bwd_kernel<2>, grid, block, 0, stream, x, xrows, xs, w, dy, bounds, n_docs, T, C, rows, act, dx, dxrows, dxs, part); break;
    case 3: hipLaunchKernelGGL(conv_bwd_kernel<3>, grid, block, 0, stream, x, xrows, xs, w, dy, bounds, n_docs, T, C, rows, act, dx, dxrows, dxs, part); break;
    default: hipLaunchKernelGGL(conv_bwd_kernel<4>, grid, block, 0, stream, x, xrows, xs, w, dy, bounds, n_docs, T, C, rows, act, dx, dxrows, dxs, part); break;
  }
}

// The same sums for few columns (n % 4 == 0) and many parts: a workgroup of 1024 threads
// takes the four float4 columns from 16 blk on (64 bytes of a part's row, one quad of lanes) and sums parts
// stripe, stripe + 256, ... in each of 256 stripes (8 loads in flight), then the stripes
// pairwise (a fixed order).  With one workgroup for all columns, one CU read everything:
// 2048 parts of 32 columns, or 1024 of 128, took 6.7 us; with a workgroup per 16 columns 4.4.
constexpr int SUM_THREADS = 1024;
__device__ __forceinline__ void narrow_sum(const float* __restrict__ part, int parts, int n, int blk, f32x4* red,
                                           float* __restrict__ out) {
  const int n4 = n / 4, c4 = 4 * blk + (threadIdx.x & 3), stripe = threadIdx.x >> 2;
  f32x4 acc = f32x4{};
  if (c4 < n4) {
    const f32x4* p = reinterpret_cast<const f32x4*>(part) + c4;
    int b = stripe;
    for (; b + 7 * 256 < parts; b += 8 * 256) {
      f32x4 v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = p[(size_t)(b + q * 256) * n4];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc += v[q];
    }
    for (; b < parts; b += 256) acc += p[(size_t)b * n4];
  }
  red[threadIdx.x] = acc;
  __syncthreads();
#pragma unroll
  for (int half = SUM_THREADS / 2; half >= 4; half >>= 1) {
    if ((int)threadIdx.x < half) red[threadIdx.x] += red[threadIdx.x + half];
    __syncthreads();
  }
  if (threadIdx.x < 4 && c4 < n4) {
    const f32x4 r = red[threadIdx.x];
#pragma unroll
    for (int k = 0; k < 4; ++k) out[c4 * 4 + k] = r[k];
  }
}

__global__ __launch_bounds__(SUM_THREADS) void colsum_narrow_kernel(const float* __restrict__ part, int parts, int n,
                                                                   float* __restrict__ out) {
  __shared__ f32x4 red[SUM_THREADS];
  narrow_sum(part, parts, n, blockIdx.x, red, out);
}

// The parameter gradients of the event inputs in one launch.  Workgroups below `wide` take
// 256 columns of dw [n]: the conv's parts and, for the q channels (the first nq columns),
// the query conv's, rows wave, wave + 16, ... in each of 16 waves, then the waves in order.
// The others take 16 columns each of dgate [ng] (narrow_sum).  A handful of loads per lane,
// so a launch costs its latency, not its bytes: the three launches before it (the conv's
// sum, the queries' added to it, the gates') took 4.7, 4.7 and 4.6 us, this one 5.0.
__global__ __launch_bounds__(SUM_THREADS) void event_sums_kernel(const float* __restrict__ cpart, int cparts, int n,
                                                                const float* __restrict__ qpart, int qparts, int nq,
                                                                float* __restrict__ dw, int wide,
                                                                const float* __restrict__ gpart, int gparts, int ng,
                                                                float* __restrict__ dgate) {
  __shared__ f32x4 red[SUM_THREADS];
  if ((int)blockIdx.x >= wide) {
    narrow_sum(gpart, gparts, ng, blockIdx.x - wide, red, dgate);
    return;
  }
  constexpr int WAVES = SUM_THREADS / 64, AHEAD = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = (blockIdx.x * 64 + lane) * 4;
  f32x4 acc = f32x4{};
  // rows past the end re-read the last one and are left out of the sum
  auto add = [&](const float* part, int parts, int width) {
    const f32x4* p = reinterpret_cast<const f32x4*>(part + j);
    const size_t stride = (size_t)width / 4;
    for (int b = wave; b < parts; b += WAVES * AHEAD) {
      f32x4 v[AHEAD];
#pragma unroll
      for (int q = 0; q < AHEAD; ++q) v[q] = p[(size_t)min(b + WAVES * q, parts - 1) * stride];
#pragma unroll
      for (int q = 0; q < AHEAD; ++q)
        if (b + WAVES * q < parts) acc += v[q];
    }
  };
  if (j < n) add(cpart, cparts, n);
  if (j < nq) add(qpart, qparts, nq);
  red[threadIdx.x] = acc;
  __syncthreads();
  if (wave == 0 && j < n) {
#pragma unroll
    for (int w = 1; w < WAVES; ++w) acc += red[64 * w + lane];
#pragma unroll
    for (int q = 0; q < 4; ++q) dw[j + q] = acc[q];
  }
}

void launch_colsum(const float* part, int parts, int n, float* out, hipStream_t stream) {
  if (n <= 256 && parts > 64)
    hipLaunchKernelGGL(colsum_narrow_kernel, dim3((n + 15) / 16), dim3(SUM_THREADS), 0, stream, part, parts, n, out);
  else
    hipLaunchKernelGGL(colsum_kernel, dim3((n / 4 + 63) / 64), dim3(256), 0, stream, part, parts, n, out);
}

void launch_event_sums(const float* cpart, int cparts, int n, const float* qpart, int qparts, int nq, float* dw,
                       const float* gpart, int gparts, int ng, float* dgate, hipStream_t stream) {
  const int wide = (n / 4 + 63) / 64, narrow = (ng + 15) / 16;
  hipLaunchKernelGGL(event_sums_kernel, dim3(wide + narrow), dim3(SUM_THREADS), 0, stream, cpart, cparts, n, qpart,
                     qparts, nq, dw, wide, gpart, gparts, ng, dgate);
}

}  // namespace cqgdn
