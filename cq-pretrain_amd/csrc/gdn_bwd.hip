// GDN backward on gfx950.
//
// Per chunk (C events, S_c the state entering it, dS_{c+1} the gradient of the
// state leaving it), with Gam_ij = exp(G_i - G_j) on i >= j, gam = exp(G),
// kdec_i = exp(G_last - G_i), P = (Qn Kn^T) * Gam:
//
//   bwd_local  (grid NC x H)  dv_local = scale P^T dO ;  X = scale (gam Qn)^T dO
//   bwd_scan   (serial, reverse)  dVn = dv_local + kdec * (Kn dS_{c+1})
//                                 dS_c = exp(G_last) dS_{c+1} + X - W^T dVn
//   bwd_dkw    (grid NC x H), in one workgroup:
//              dQn = scale gam (dO S_c^T) + (scale dP Gam) Kn   (dP = dO Vn^T); l2norm backward of dq
//              dKn(part) = (scale dP Gam)^T Qn + kdec (Vn dS_{c+1}^T)
//              dW = -dVn S_c^T ; dG terms of the output and state update
//              dT = dW (beta gam Kn)^T + dVn (beta V)^T ; dA = -(T^T dT T^T)
//              dKn += beta (dA Gam) Kn + (dA Gam)^T (beta Kn) + beta gam (T^T dW)
//              dV = beta (T^T dVn) ; dbeta ; dG ; reverse cumsum -> dg ; l2norm backward of dk
//
// This is the reference's backward op chain (ops/gated_delta_net.py:188-214:
// chunk_bwd_dv_local, chunk_gated_delta_rule_bwd_dhu, chunk_bwd_dqkwg,
// prepare_wy_repr_bwd_da/_full, reverse_cumsum, l2_bwd) regrouped into three
// kernels.  All reductions run in a fixed order (no atomics), so results are
// bitwise reproducible from run to run.
//
// E is the operand type: bf16, or fp16 for fp16 inputs.  In fp16 every quantity is
// carried in exact power-of-two scales that keep it inside fp16's range: the
// forward's scale s_v of V (h and v_new carry it; the V rows read here are scaled
// by it too) and the scale s_d of dO.  s_d brings max|dO| below 2^e with
// T 2^e <= 2^15: with unit-norm q rows a state gradient satisfies |dS| <= T max|dO|,
// so dS and dVn stay below about 2^15.  dv_local, X, dS, dVn and dv carry s_d; dP,
// dW, dT, dA, dq, dk, dg and dbeta carry s_d s_v.  Each output is divided by its
// scale in fp32 before it is stored.
//
// bwd_dkw may run on a second stream beside the reverse scan (launch_bwd): the
// scan then stores each chunk's dS / dVn at device scope and announces the chunk
// with an atomic count, and bwd_dkw takes the chunks in the order the scan
// finishes them, each waiting (bounded) for its count.  The atomics only order
// the hand-off; every value is computed as in the sequential order, so the
// results are the same bits either way.
#include "gdn_common.hpp"
#include "gdn_layout.hpp"
#include "gdn_kernels.hpp"

namespace cqgdn {

constexpr int LDK = 136;  // bf16 row stride, 64 x 128 tiles
constexpr int LDT = 72;   // bf16 row stride, 128 x 64 and 64 x 64 tiles

// ---------------------------------------------------------------------------
// bwd_local
// ---------------------------------------------------------------------------
// dscale: null in bf16; in fp16 the scale s_d of dO, which this kernel forms from the
// partial maxima after dscale[0] (range_scale, target ds_target) and stores in
// dscale[0] for bwd_dkw
template <class E>
__global__ __launch_bounds__(256, 3) void bwd_local_kernel(
    const E* __restrict__ q, const E* __restrict__ k, int normalize,
    const float* __restrict__ rk, const E* __restrict__ dout, const float* __restrict__ gc,
    const float* __restrict__ beta, const E* __restrict__ Tm,
    const int32_t* __restrict__ chunks, int H, float scale, float* __restrict__ dscale, int ds_target,
    E* __restrict__ dvlT, E* __restrict__ XT, E* __restrict__ knP, E* __restrict__ WT, int* __restrict__ sync) {
  typedef typename Vec<E>::x8 X8;
  constexpr bool F16 = __is_same(E, f16);
  // grid (H, NC), chunks dispatched first to last: the reverse state scan that
  // follows reads the last chunks first, and they are then the most recently
  // written (still in the memory-side cache).  The scan's other two operands,
  // kdec Kn and -W^T, are made here for the same reason.
  const HeadChunk hc = xcd_head_chunk(gridDim.x, gridDim.y);  // all heads of a chunk on one XCD
  const int h = hc.h, c = hc.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q4 = lane >> 4;
  const ChunkInfo ci = chunk_info(chunks, c);
  const size_t cb = (size_t)c * H + h;
  // the counts of the reverse scan's hand-off to bwd_dkw start at zero: this (chunk,
  // head)'s, and (one workgroup) the count of resident scan workgroups after them
  if (tid == 0) {
    sync[cb] = 0;
    if (c == 0 && h == 0) sync[(size_t)gridDim.y * H] = 0;
  }

  // Row tiles only (every transposed operand is read with ds_read_b64_tr_b16),
  // 52 KB, so three workgroups share a CU.  The outputs are staged over them
  // once they are read and stored as whole rows: X^T over Qs | Ks, dv_local^T
  // (64-element rows, 16-byte columns XOR-swizzled by row) over dOs.
  __shared__ __attribute__((aligned(16))) E QK[2 * 64 * LDK];  // Qs | Ks, then X^T [v][k]
  __shared__ __attribute__((aligned(16))) E dOs[64 * LDK];     // dO rows, then dv_local^T [v][s]
  __shared__ __attribute__((aligned(16))) float Gs[64];
  __shared__ __attribute__((aligned(16))) float Bs[64];
  __shared__ float red[4];
  E* Qs = QK;
  E* Ks = QK + 64 * LDK;
  static_assert(64 * LDK >= 128 * 64, "dv_local^T fits the dO tile");
  // fp16: this thread's partial maximum of |dO|, requested before the other loads
  const float dpart = F16 ? range_partial4(dscale + 1) : 0.f;
  float ds = 1.f;  // s_d (fp16), formed once the input loads are in flight

  // T rows t = 16 wave + r, for -W^T below (requested with the inputs)
  X8 at[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) at[kb] = ld8(Tm + cb * (CH * CH) + (16 * wave + r) * CH + 32 * kb + 8 * q4);
  {
    const int t = tid >> 2, p = tid & 3;
    const bool in = t < ci.len;
    const int tc = clamp_row(t, ci.len);
    const size_t ev = (size_t)(ci.start + tc) * H + h, row = ev * D;
    const float rkt = rk[ev];
    // q and k non-temporally: what this kernel writes (the reverse scan's operands,
    // 188 MB at T = 9216, H = 16) and what the scan writes do not both fit the
    // 256 MB memory-side cache, and q, k are read next only by bwd_dkw, after the scan
    X8 xq[4], xk[4], xd[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * j + 8 * p;
      xq[j] = ld8_nt(q + row + col);
      xk[j] = ld8_nt(k + row + col);
      xd[j] = ld8(dout + row + col);
    }
    if (p == 0) {
      Gs[t] = gc[ev];
      Bs[t] = keep_if(in, beta[ev]);
    }
    const float rqt = normalize ? row_rnorm(xq) : 1.f;
    if constexpr (F16) {  // dO s_d (exact: a power of two, in range)
      ds = range_scale(dpart, ds_target, red);
#pragma unroll
      for (int j = 0; j < 4; ++j) xd[j] = to8<E>(cvtf8(xd[j]) * ds);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * j + 8 * p;
      st8(Qs + t * LDK + col, keep_if(in, scaled8<E>(xq[j], rqt)));
      st8(Ks + t * LDK + col, keep_if(in, scaled8<E>(xk[j], rkt)));
      st8(dOs + t * LDK + col, keep_if(in, xd[j]));
    }
  }
  __syncthreads();

  // kdec_t Kn_t (kdec_t = exp(G_last - G_t), the decay the reverse scan applies to Kn dS)
  // in the order the scan reads it: fragment (t / 16, k / 32), and in it 16-byte granule
  // 16 g + r holding row t = 16 (t / 16) + r, k = 32 (k / 32) + 8 g ..
  {
    E* kp = knP + cb * (CH * D) + 8 * tid;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * i + r;
      const float kd = __expf(Gs[ci.len - 1] - Gs[t]);
      st8(kp + 2048 * i, to8<E>(cvtf8(ld8(Ks + t * LDK + 32 * wave + 8 * q4)) * kd));
    }
  }

  // per-lane event factors at s = 32 kb + 8 q4 + e: beta_s gam_s (for W) and gam_s (for X)
  f32x8 fbg[2], fg[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int s = 32 * kb + 8 * q4 + e;
      fg[kb][e] = __expf(Gs[s]);
      fbg[kb][e] = Bs[s] * fg[kb][e];
    }

  // -W^T with W = T (beta gam K): t-tile = wave, k-tiles n; beta gam K is read transposed
  // from the K rows and scaled per event s on the way.  Stored in the order the reverse
  // scan reads it: fragment (k / 32, (k / 4) % 2, t / 32), and in it granule 16 g + i
  // holding row k = .. + 8 (i / 4) + i % 4 at the four-runs g of both halves of the 32
  // events (perm32)
  {
    E* wt = WT + cb * (D * CH) + (64 * (2 * ((r >> 2) & 1) + (wave >> 1)) + 16 * q4 + 4 * (r >> 3) + (r & 3)) * 8 +
            4 * (wave & 1);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      f32x4 aw = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        if (kb == 0 || wave >= 2)  // T[t][s] = 0 for s > t
          aw = mfma(at[kb], to8<E>(cvtf8(ld8_tr(Ks, LDK, 32 * kb, 16 * n)) * fbg[kb]), aw);
      st4(wt + (n >> 1) * 2048 + (n & 1) * 64, -aw);
    }
  }

  // P tiles (t-tile tt >= s-tile = wave), causal and gated, kept in registers:
  // pp[tt][i] = P[t = 16 tt + 4 q4 + i][s = 16 wave + r]
  f32x4 pp[4];
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    pp[tt] = zero4();
    if (tt >= wave) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        pp[tt] = mfma(ld8(Qs + (16 * tt + r) * LDK + 32 * kb + 8 * q4), ld8(Ks + (16 * wave + r) * LDK + 32 * kb + 8 * q4),
                      pp[tt]);
      const int s = 16 * wave + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * tt + 4 * q4 + i;
        pp[tt][i] = (s <= t) ? pp[tt][i] * __expf(Gs[t] - Gs[s]) : 0.f;
      }
    }
  }

  // dv_local^T (s rows 16 wave + 4 q4 .., 8 value tiles) = P^T dO: P^T comes from
  // the P tiles (pack_permv, events in perm32 order), dO is read transposed in the
  // same order; only t >= s contributes
  f32x4 dvl[8];
  {
    const int kb0 = wave >= 2 ? 1 : 0;
    X8 a[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) a[kb] = pack_permv<E>(pp[2 * kb], pp[2 * kb + 1]);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      dvl[n] = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        if (kb >= kb0) dvl[n] = mfma(a[kb], ld8_trp(dOs, LDK, 32 * kb, 16 * n), dvl[n]);
    }
  }
  // X^T (k-tiles 2w, 2w+1 x 8 value tiles) = (gam Q)^T dO, both read transposed
  f32x4 xt[2][8];
#pragma unroll
  for (int mm = 0; mm < 2; ++mm) {
    const int m = 2 * wave + mm;
    X8 a[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) a[kb] = to8<E>(cvtf8(ld8_tr(Qs, LDK, 32 * kb, 16 * m)) * fg[kb]);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      xt[mm][n] = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) xt[mm][n] = mfma(a[kb], ld8_tr(dOs, LDK, 32 * kb, 16 * n), xt[mm][n]);
    }
  }
  __syncthreads();  // the input tiles are read: they take the output tiles
  E* xts = QK;      // X^T [v][k], row stride LDK
  E* dvs = dOs;     // dv_local^T [v][s], 64-element rows, 16-byte column c at c ^ (v & 7)
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int v = 16 * n + r, sc = 2 * wave + (q4 >> 1);
    st4(dvs + v * 64 + 8 * (sc ^ (v & 7)) + 4 * (q4 & 1), dvl[n] * scale);
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) st4(xts + v * LDK + 16 * (2 * wave + mm) + 4 * q4, xt[mm][n] * scale);
  }
  __syncthreads();
  {
    E* out = dvlT + cb * (D * CH);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int seg = 256 * i + tid, v = seg >> 3, part = seg & 7;
      st8(out + v * CH + 8 * part, ld8(dvs + v * 64 + 8 * (part ^ (v & 7))));
    }
  }
  {
    E* out = XT + cb * (D * D);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int seg = 256 * i + tid, v = seg >> 4, part = seg & 15;
      st8(out + v * D + 8 * part, ld8(xts + v * LDK + 8 * part));
    }
  }
  if (F16 && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) dscale[0] = ds;  // for bwd_dkw
}

// ---------------------------------------------------------------------------
// bwd_scan: the reverse scan, four waves per (head, 16-wide value slice, document)
// ---------------------------------------------------------------------------
// Organised as fwd_scan (gdn_fwd.hip): wave w holds rows 32 w .. of the slice's dS and
// does a quarter of each contraction, dS and dVn pass through LDS with a barrier after
// each.  bwd_local writes both matrices, kdec Kn and -W^T, in fragment order, so their
// loads are 1 KB of contiguous operands; X^T and dv_local^T are read by quads and
// exchanged between lanes; dS and dVn are read back from LDS transposed, as whole blocks
// of the value-slice-major outputs.  The tiles' rows are k = 32 w + 8 (i / 4) + 4 m + i % 4,
// so a lane's eight values of dS are consecutive in k: one 16-byte LDS write, and one
// 16-byte piece of X^T.
//
// Measured in the kernel trace of whole steps, bwd_dkw after it (H = 16, one document of 144
// chunks / 15 documents, 520 chunks): 121 -> 97 us, 326 -> 298 us; 36 chunks 32.9 -> 23.7;
// four heads, 144 chunks 113.5 -> 77.1.
//
// The outputs are stored with the non-temporal hint: the scan still has the earlier chunks'
// operands to read (bwd_local wrote them first to last, so they are the oldest in the
// memory-side cache).  With bwd_dkw beside it (SC1) the stores are device-scope, and the
// waves run at a raised priority (four heads: a step 270 -> 266 us; no change at 16).
// One slice's dS / dVn of chunk c are stored (their stores have completed): add to
// the chunk's count, which bwd_dkw waits to see at 8, from one lane.
__device__ __forceinline__ void bwd_publish(int* __restrict__ ready, int c, int H, int h, int lane) {
  asm volatile("" ::: "memory");
  if (lane == 0) count_add(ready + (size_t)c * H + h);
  asm volatile("" ::: "memory");
}

// LDS that a scan workgroup with a bwd_dkw beside it takes in addition, unused: with it no
// bwd_dkw workgroup (81 KB) shares its CU.  On a shared CU the two halve each other (H = 16,
// 144 chunks: scan 180 us, step 432; alone on its CU 137 and 426; 512 chunks of 8 heads:
// step 1064 and 1028).
constexpr int BESIDE_LDS = 88 * 1024;

// Vector memory operations of one full step of one wave: 8 operand fragments, X, dv_local,
// two stores.  A step's chunk is announced BWD_ANNOUNCE steps later.
constexpr int BWD_STEP_OPS = 12, BWD_ANNOUNCE = 3;

template <class E, bool SC1, bool WIDE>
__global__ __launch_bounds__(SCAN_THREADS, 2) void bwd_scan_kernel(
    // without __restrict__ where loads are requested ahead: the barriers then pin their place
    const E* knP, const float* gc, const E* dvlT, const E* XT, const E* WT, const int32_t* chunks,
    const int32_t* __restrict__ doc_chunk, int H, E* dhS, E* dVnS, int* ready, int* resident) {
  // SC1: a bwd_dkw runs beside this scan (each workgroup adds one to resident when it
  // starts, and one to a chunk's ready count once its outputs of that chunk are stored)
  typedef typename Vec<E>::x8 X8;
  typedef typename Vec<E>::x4 X4;
  const int h = blockIdx.x % H, slice = blockIdx.x / H, d = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q4 = lane >> 4;
  const int v0 = 16 * slice;
  constexpr int OUT = CPOL_NT | (SC1 ? CPOL_SC1 : 0);
  if constexpr (SC1) __builtin_amdgcn_s_setprio(3);

  __shared__ __attribute__((aligned(16))) E Sx[16 * SCAN_SROW];  // dS's operand copy, [v][k]
  __shared__ __attribute__((aligned(16))) E Vx[16 * SCAN_VROW];  // dVn, [v][perm32(t)]

  const int c_begin = __builtin_amdgcn_readfirstlane(doc_chunk[d]);
  const int c_last = __builtin_amdgcn_readfirstlane(doc_chunk[d + 1]) - 1, n = c_last + 1 - c_begin;
  if (SC1 && threadIdx.x == 0) count_add(resident);
  if (n <= 0) return;
  // step tau handles chunk c_last - tau
  f32x4 dS[2];  // dS[m][i] = dState[k = 32 wave + 8 q4 + 4 m + i][v = v0 + r]
#pragma unroll
  for (int m = 0; m < 2; ++m) dS[m] = zero4();
  ScanTable tab(chunks, gc, nullptr, c_last, -1, n, H, h, lane);
  const size_t cb = (size_t)c_last * H + h;
  const int64_t tile = (int64_t)H * D * CH * 2;  // bytes from one chunk's [D][64] tile to the next chunk's
  ScanBlocks<true, WIDE> kb(knP + cb * (D * CH), tile, n);
  ScanBlocks<true, WIDE> wb(WT + (cb + H) * (D * CH), tile, n + 1);  // one step behind: its first block is step -1's
  ScanBlocks<true, WIDE> lb(dvlT + cb * (D * CH) + v0 * CH, tile, n), xb(XT + cb * (D * D) + v0 * D, 2 * tile, n);
  ScanBlocks<true, WIDE> sb(dhS + cb * (D * D) + slice * (D * 16), 2 * tile, n);
  ScanBlocks<true, WIDE> nb(dVnS + cb * (CH * D) + slice * (CH * 16), tile, n);
  // per-lane parts of the addresses, the same for every chunk (bytes of global memory;
  // elements of LDS)
  const int q = (lane >> 2) & 3, p = lane & 3, from = tile_source(lane);
  const int f_off = 4096 * wave + 16 * lane;                        // fragments (wave, m, b) of -W^T
  int n_off[4];                                                     // fragments (wave, j) of Kn, this wave's own k first
#pragma unroll
  for (int j = 0; j < 4; ++j) n_off[j] = f_off + 1024 * ((wave + j) & 3);
  const int l_off = (4 * q4 + q) * CH * 2 + 32 * wave + 8 * p;      // dv_local^T row 4 q4 + q, t = 16 wave + 4 p ..
  const int x_off = (4 * q4 + q) * D * 2 + 64 * wave + 16 * p;      // X^T row 4 q4 + q, k = 32 wave + 8 p ..
  const int s_own = r * SCAN_SROW + 32 * wave + 8 * q4;
  const int v_own = r * SCAN_VROW + 32 * (wave >> 1) + 8 * q4 + 4 * (wave & 1), v_in = r * SCAN_VROW + 8 * q4;
  // the outputs, read transposed: dS [k][16] rows 32 wave .., dVn [t][16] rows 16 wave ..
  const E* v_tr = Vx + (4 * q4 + (r >> 2)) * SCAN_VROW + 32 * (wave >> 1) + 8 * (r & 3) + 4 * (wave & 1);
  const int s_out = ((32 * wave + 16 * (q4 >> 1) + r) * 16 + 8 * (q4 & 1)) * 2, v_out = ((16 * wave + r) * 16 + 4 * q4) * 2;
  X8 fn[SCAN_DEPTH][4], fw[SCAN_DEPTH][2][2], fx[SCAN_DEPTH], x;
  X4 fl[SCAN_DEPTH], dvl;
  float gl[SCAN_DEPTH];
  // l: the step's place after the table's and the blocks' first
  auto issue_n = [&](int slot, int l) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) fn[slot][j] = buf_ld16<X8>(kb.buffer(l), n_off[j], kb.offset(l));
    fl[slot] = buf_ld8<X4>(lb.buffer(l), l_off, lb.offset(l));
    fx[slot] = buf_ld16<X8>(xb.buffer(l), x_off, xb.offset(l));
  };
  auto issue_w = [&](int slot, int l) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int b = 0; b < 2; ++b) fw[slot][m][b] = buf_ld16<X8>(wb.buffer(l), f_off + 2048 * m + 1024 * b, wb.offset(l));
  };
  auto next_inputs = [&](int slot) __attribute__((always_inline)) {
    dvl = tile_exchange(fl[slot], from);
    x = tile_exchange(fx[slot], from);
  };
  X8 own = to8<E>(f32x8{});
  st8(Sx + s_own, own);
#pragma unroll
  for (int i = 0; i < SCAN_DEPTH; ++i) {
    issue_n(i, i);
    if (i > 0) issue_w(i - 1, i);
    if (i == 0) {
      // the first step's requests go out before the wait for the chunk table (documents of one chunk:
      // the backward of 512 of them, 16 heads, 1097 -> 1053 us)
      __builtin_amdgcn_sched_barrier(0);
      tab.open();
      __builtin_amdgcn_sched_barrier(0);
    }
    gl[i] = tab.glast(i);
  }
  kb.advance();
  wb.advance();
  lb.advance();
  xb.advance();
  float g_now = __expf(gl[0]);
  next_inputs(0);
  lds_barrier();
  auto step = [&](auto place, auto more) __attribute__((always_inline)) {
    constexpr int s = decltype(place)::value;
    // dVn = dv_local + (kdec Kn) dS_{c+1}, this wave's own block of k first
    f32x4 acc = mfma(fn[s][0], own, cvtf4(dvl));
    X8 sx[3];
#pragma unroll
    for (int j = 1; j < 4; ++j) sx[j - 1] = ld8(Sx + r * SCAN_SROW + 32 * ((wave + j) & 3) + 8 * q4);
    const X8 ds_out = ld8_tr16(Sx, SCAN_SROW, 32 * wave);
    if constexpr (decltype(more)::value) issue_w((s + SCAN_DEPTH - 1) % SCAN_DEPTH, s);
#pragma unroll
    for (int j = 1; j < 4; ++j) acc = mfma(fn[s][j], sx[j - 1], acc);
    buf_st16<OUT>(sb.buffer(s), s_out + sb.offset(s), ds_out);
    // the first two terms of dS_c = exp(G_last) dS_{c+1} + X + (-W^T) dVn
    const f32x8 xf = cvtf8(x);
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) dS[m][i] = dS[m][i] * g_now + xf[4 * m + i];
    *reinterpret_cast<X4*>(Vx + v_own) = to4<E>(acc);
    lds_barrier();
    const X8 b0 = ld8(Vx + v_in), b1 = ld8(Vx + v_in + 32);
    typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
    const X4 dv_out = __builtin_bit_cast(X4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)v_tr));
    constexpr int next = (s + 1) % SCAN_DEPTH;
    g_now = __expf(gl[next]);
    next_inputs(next);
    if constexpr (decltype(more)::value) {
      issue_n(s, s);
      gl[s] = tab.glast(s);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) dS[m] = mfma(fw[s][m][0], b0, dS[m]);
#pragma unroll
    for (int m = 0; m < 2; ++m) dS[m] = mfma(fw[s][m][1], b1, dS[m]);
    buf_st8<OUT>(nb.buffer(s), v_out, nb.offset(s), dv_out);
    own = to8<E>(f32x8{dS[0][0], dS[0][1], dS[0][2], dS[0][3], dS[1][0], dS[1][1], dS[1][2], dS[1][3]});
    st8(Sx + s_own, own);
    if constexpr (SC1 && decltype(more)::value) {
      // the stores of BWD_ANNOUNCE steps ago have completed: that many full steps were issued after them
      asm volatile("" ::: "memory");
      wait_vmem_le<BWD_ANNOUNCE * BWD_STEP_OPS>();
    }
    lds_barrier();
  };
  int announced = 0;  // steps whose chunks are announced
  auto round = [&](int tau, auto first) __attribute__((always_inline)) {
    tab.advance(tau + SCAN_DEPTH);
    auto announced_step = [&](auto place) __attribute__((always_inline)) {
      step(place, Int<1>());
      // every wave has waited for its stores of step tau + place - BWD_ANNOUNCE
      if constexpr (SC1 && (!decltype(first)::value || decltype(place)::value >= BWD_ANNOUNCE)) {
        if (wave == 0) bwd_publish(ready, c_last - announced, H, h, lane);
        ++announced;
      }
    };
    announced_step(Int<0>());
    announced_step(Int<1>());
    announced_step(Int<2>());
    announced_step(Int<3>());
    kb.advance();
    wb.advance();
    lb.advance();
    xb.advance();
    sb.advance();
    nb.advance();
  };
  int tau = 0;
  if (n >= SCAN_DEPTH) {
    round(0, Int<1>());
    for (tau = SCAN_DEPTH; tau + SCAN_DEPTH <= n; tau += SCAN_DEPTH) round(tau, Int<0>());
  }
  if (tau < n) step(Int<0>(), Int<0>());
  if (tau + 1 < n) step(Int<1>(), Int<0>());
  if (tau + 2 < n) step(Int<2>(), Int<0>());
  if constexpr (SC1) {
    wait_vmem_all();
    lds_barrier();
    if (wave == 0)
      for (; announced < n; ++announced) bwd_publish(ready, c_last - announced, H, h, lane);
  }
}

// ---------------------------------------------------------------------------
// bwd_dkw: the dq/dK/dW part and then the WY part in one workgroup per (chunk, head), so the
// dK partial (registers), dW (LDS), the dG partial (a register of wave 0) and the
// K tile never leave the chip.  LDS regions are reused as their first users die
// (81,408 bytes: two workgroups per CU):
//   R1  Q rows            -> V rows (wy)
//   R2  K rows            (both parts)
//   R3  dPm^T             -> T (wy)
//   R4a dO rows           -> dVn tile (value-slice-major) + q.dq row dots
//                         -> dT^T / (beta dM)^T staging + beta, dbeta and k.dK partials (wy)
//   R4b v_new^T           -> dW rows [t][k]   -> Y^T staging (wy)
// dPm and the wy staging tiles are stored transposed: an MFMA result fragment
// holds 4 consecutive rows of one column per lane, which then leave as one
// 8-byte write instead of four 2-byte writes (readers swap row and transposed
// reads accordingly).
// The l2norm backward of dq runs on the phase-2 registers (per-wave row dots in
// LDS), so no fp32 staging tile is needed and dQ's registers carry the dK partial.
// h is read by whole row pieces and turned in LDS (columns_from_rows), and dq, dk and dv
// leave as whole rows, dq through the dO rows' place before the dVn copy, dk and dv from
// the K and V rows' places, whose values only their lane still reads: column gathers and
// 8-byte stores from lanes on 16 different rows keep the vector memory unit 3 and 2.5
// times as long.  H = 16, 144 chunks / 520 chunks of 15 documents / 36 chunks, in a step's kernel
// trace: 133 -> 130 / 424 -> 415 / 44.0 -> 42.2 us.
// Barriers order LDS only (s_waitcnt lgkmcnt(0); s_barrier): global stores stay
// in flight across them, and the one barrier that needs the dVn tile's copies
// waits for vector memory explicitly.
constexpr int DKW_R1 = 0, DKW_R2 = 64 * LDK * 2, DKW_R3 = DKW_R2 + 64 * LDK * 2, DKW_R4A = DKW_R3 + 64 * LDT * 2,
              DKW_R4B = DKW_R4A + 64 * LDK * 2, DKW_BYTES = DKW_R4B + 128 * LDT * 2;

template <class E>  // dscale, vscale: null in bf16; in fp16 the device scalars s_d and s_v
__global__ __launch_bounds__(256, 2) void bwd_dkw_kernel(
    const E* __restrict__ q, const E* __restrict__ k,
    const float* __restrict__ rk, const float* __restrict__ gc, const E* __restrict__ hT,
    const E* __restrict__ vnT, const E* __restrict__ dout, const E* __restrict__ dh,
    const E* __restrict__ dVn, const E* __restrict__ vin, const float* __restrict__ beta,
    const E* __restrict__ Tm, const int32_t* __restrict__ chunks, int H, float scale, int normalize,
    const float* __restrict__ dscale, const float* __restrict__ vscale,
    E* __restrict__ dq, E* __restrict__ dk, E* __restrict__ dv, float* __restrict__ dg,
    float* __restrict__ dbeta, const int* __restrict__ ready, int ready_target, int ready_polls) {
  // grid (H, NC).  After the reverse scan: chunks first to last (the scan wrote the
  // first chunks last, so they are the likeliest still in the memory-side cache).
  // Beside the scan (ready != null): chunks last to first, the order the scan
  // finishes them, each workgroup waiting for its chunk's count after phase 1.
  typedef typename Vec<E>::x8 X8;
  constexpr bool F16 = __is_same(E, f16);
  // fp16: dq, dk, dg and dbeta leave divided by s_d s_v, dv by s_d (powers of two: exact)
  float inv_dv = 1.f, inv_d = 1.f, vs = 1.f;
  if constexpr (F16) {
    vs = *vscale;
    inv_d = 1.f / *dscale;
    inv_dv = inv_d / vs;
  }
  const HeadChunk hc = xcd_head_chunk(gridDim.x, gridDim.y);  // all heads of a chunk on one XCD
  const int h = hc.h, c = ready ? gridDim.y - 1 - hc.p : hc.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q4 = lane >> 4;
  const ChunkInfo ci = chunk_info(chunks, c);
  const size_t cb = (size_t)c * H + h;

  // One array per region: the compiler then sees that the dVn tile's
  // asynchronous copy writes R4a only, and lets phase 3's reads of the other
  // regions run while it is in flight (with a single array it waited for the
  // copy, and every store before it, ahead of phase 3's first LDS read).
  __shared__ __attribute__((aligned(16))) uint8_t r1[DKW_R2 - DKW_R1];
  __shared__ __attribute__((aligned(16))) uint8_t r2[DKW_R3 - DKW_R2];
  __shared__ __attribute__((aligned(16))) uint8_t r3[DKW_R4A - DKW_R3];
  __shared__ __attribute__((aligned(16))) uint8_t r4a[DKW_R4B - DKW_R4A];
  __shared__ __attribute__((aligned(16))) uint8_t r4b[DKW_BYTES - DKW_R4B];
  __shared__ __attribute__((aligned(16))) float Gs[64];
  __shared__ float dgw[4][64];
  __shared__ __attribute__((aligned(16))) float Rs[64];  // rsqrt norms of q (1 without normalize)
  __shared__ int stale_s;  // nonzero when the wait for the reverse scan gave up
  E* Qs = reinterpret_cast<E*>(r1);
  E* Ks = reinterpret_cast<E*>(r2);
  E* dPm = reinterpret_cast<E*>(r3);
  E* dOs = reinterpret_cast<E*>(r4a);
  E* VnT = reinterpret_cast<E*>(r4b);  // v_new^T [v][t], read transposed as v_new rows
  E* dVs = dOs;                        // dVn tile, from phase 3 on
  float* dqdot = reinterpret_cast<float*>(r4a + CH * D * 2);  // [64][4 waves] after the dVn tile
  E* dWs = VnT;                        // dW rows [t][k], from phase 4 on

  // This wave's state fragments: rows k = 16 (2 wave + mm) + r of h
  // (columns of h^T, turned in LDS) and of dS_{c+1}, value block kb.
  const E* ht = hT + cb * (D * D);
  X8 bh[2][4], bd[2][4];
  // Every prologue load is issued before the first wait: h^T by row pieces, the
  // gate and k-norm values (unconditional: rk is allocated either way), the
  // v_new^T rows and the Q, K, dO rows; h^T is turned last.  The q norm is formed
  // from the Q rows (row_rnorm).
  {
    const int t = tid >> 2, p = tid & 3;
    X8 gh[8];  // h^T row v = 16 i + lane / 4, piece p of the wave's columns k = 32 wave ..
#pragma unroll
    for (int i = 0; i < 8; ++i) gh[i] = row_piece(ht, D, 16 * i + (lane >> 2), 32 * wave);
    const bool in = t < ci.len;
    const int tc = clamp_row(t, ci.len);
    const size_t ev = (size_t)(ci.start + tc) * H + h, row = ev * D;
    const float gv = gc[ev];
    const float rkv = rk[ev];
    const E* vt = vnT + cb * (D * CH);
    X8 xv[4], xq[4], xk[4], xo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int seg = 256 * i + tid, v = seg >> 3, part = seg & 7;
      xv[i] = ld8(vt + v * CH + 8 * part);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * j + 8 * p;
      xq[j] = ld8(q + row + col);
      xk[j] = ld8(k + row + col);
      xo[j] = ld8(dout + row + col);
    }
    dgw[wave][lane] = 0.f;
    const float rv = normalize ? row_rnorm(xq) : 1.f;
    if (p == 0) {
      Gs[t] = gv;
      Rs[t] = rv;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int seg = 256 * i + tid, v = seg >> 3, part = seg & 7;
      st8(VnT + v * LDT + 8 * part, xv[i]);
    }
    if constexpr (F16) {  // dO s_d (exact: a power of two, in range)
      const float ds = *dscale;
#pragma unroll
      for (int j = 0; j < 4; ++j) xo[j] = to8<E>(cvtf8(xo[j]) * ds);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * j + 8 * p;
      st8(Qs + t * LDK + col, keep_if(in, scaled8<E>(xq[j], rv)));
      st8(Ks + t * LDK + col, keep_if(in, scaled8<E>(xk[j], rkv)));
      st8(dOs + t * LDK + col, keep_if(in, xo[j]));
    }
    // through dPm's region, whose first use is after the barrier
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      X8 y[2];
      columns_from_rows(dPm + 1024 * wave, gh[2 * kb], gh[2 * kb + 1], y);
      bh[0][kb] = y[0];
      bh[1][kb] = y[1];
    }
  }
  lds_barrier();
  const float glast = Gs[ci.len - 1];
  float* dgl = dgw[wave];

  // ---- phase 1: P, dP over the ten causal (t-tile, s-tile) pairs: wave w takes t-tile w with
  //      s-tiles 0 .. min(w, 2) and wave 0 also the (3, 3) diagonal, at most three pairs a wave ----
  // The gates Gam[t][s] of this wave's pairs stay in registers for the wy phase 3, which
  // takes the same pairs in the same fragment layout: gk[n] for s-tile n of t-tile wave,
  // gk[3] for wave 0's (3, 3) tile.
  f32x4 gk[4];
  {
    // dPm of t-tile tt, s-tile n; its row sums are added to rowE, its column sums to dgl
    auto pair = [&](int tt, int n, float(&rowE)[4], f32x4& gout) -> f32x4 {
      f32x4 p = zero4(), dp = zero4();
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        p = mfma(ld8(Qs + (16 * tt + r) * LDK + 32 * kb + 8 * q4), ld8(Ks + (16 * n + r) * LDK + 32 * kb + 8 * q4), p);
        dp = mfma(ld8(dOs + (16 * tt + r) * LDK + 32 * kb + 8 * q4), ld8_tr(VnT, LDT, 32 * kb, 16 * n), dp);
      }
      const int s = 16 * n + r;
      const f32x4 g4 = *reinterpret_cast<const f32x4*>(&Gs[16 * tt + 4 * q4]);
      const float gs = Gs[s];
      float colE = 0.f;
      f32x4 dpm;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * tt + 4 * q4 + i;
        const float gam = (s <= t) ? __expf(g4[i] - gs) : 0.f;
        gout[i] = gam;
        dpm[i] = scale * dp[i] * gam;
        const float e = dpm[i] * p[i];
        rowE[i] += e;
        colE += e;
      }
      colE = sum_rows4(colE);
      if (q4 == 0) dgl[s] -= colE;
      return dpm;
    };
    float rowE[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      if (n == 3 && wave == 3) continue;  // the (3, 3) tile is wave 0's
      const f32x4 dpm = (n <= wave) ? pair(wave, n, rowE, gk[n]) : zero4();
      st4(dPm + (16 * n + r) * LDT + 16 * wave + 4 * q4, dpm);  // transposed: dPm^T[s][t], 4 rows t in 8 bytes
    }
    sum16x4(rowE);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r == 0) dgl[16 * wave + 4 * q4 + i] += rowE[i];
    if (wave == 0) {
      float rowE3[4] = {0.f, 0.f, 0.f, 0.f};
      st4(dPm + (48 + r) * LDT + 48 + 4 * q4, pair(3, 3, rowE3, gk[3]));
      sum16x4(rowE3);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (r == 0) dgl[48 + 4 * q4 + i] += rowE3[i];
    }
  }
  // dS_{c+1} and dVn are the reverse scan's: beside it, wait until all eight value
  // slices of this chunk are stored (wave 1 has the fewest phase-1 pairs).  If the
  // wait gives up, dS_{c+1} and dVn are taken as NaN, which turns every output that
  // depends on them (dk, dv, dg, dbeta) to NaN; dq does not depend on them.
  if (wave == 1) {
    bool ok = true;
    if (ready && lane == 0) ok = count_wait_ge(ready + cb, ready_target, ready_polls);
    if (lane == 0) stale_s = ok ? 0 : 1;
  }
  lds_barrier();
  const bool stale = stale_s != 0;
  const __amdgpu_buffer_rsrc_t dh_rs = buf_rsrc(dh + cb * (D * D), D * D * 2);

  // (device-scope loads beside the scan, which may still be running)
#pragma unroll
  for (int mm = 0; mm < 2; ++mm)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int i = (2 * kb + (q4 >> 1)) * (D * 16) + (16 * (2 * wave + mm) + r) * 16 + 8 * (q4 & 1);
      bd[mm][kb] = ready ? buf_ld16_sc1<X8>(dh_rs, i * 2) : ld8(dh + cb * (D * D) + i);
    }
  if (stale) {
    asm volatile("");  // a branch, not selects
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) bd[mm][kb] = to8<E>(f32x8{NAN, NAN, NAN, NAN, NAN, NAN, NAN, NAN});
  }

  // ---- phase 2: dQ^T (k-tiles 2w, 2w+1 as rows, t columns); dG_t from the output term ----
  // Each MFMA takes the operands of dQ = dO h^T + (dP Gam) K swapped, so a lane holds 4
  // consecutive k of one row t: dQ[mm][n][i] = dq[t = 16 n + r][k = 16 (2w + mm) + 4 q4 + i].
  // The row's gate and norm are then one value per lane, and its sums over k run over the
  // 4 lanes of a column (permlane swaps).
  f32x4 dQ[2][4];
  f32x4 qrow[4][2];  // q[t = 16 n + r][k = 16 (2w + mm) + 4 q4 + i], kept for the dq stores
  float pdot[4];     // this wave's parts of the row dots q_t . dQ_t (l2norm backward of dq)
  {
    f32x4 a1[2][4];
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
#pragma unroll
      for (int n = 0; n < 4; ++n) a1[mm][n] = dQ[mm][n] = zero4();
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const X8 a = ld8(dOs + (16 * n + r) * LDK + 32 * kb + 8 * q4);
#pragma unroll
        for (int mm = 0; mm < 2; ++mm) a1[mm][n] = mfma(bh[mm][kb], a, a1[mm][n]);
      }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        if (n < 2 * kb) continue;
        const X8 a = ld8_tr(dPm, LDT, 32 * kb, 16 * n);  // dPm rows t = 16 n + r
#pragma unroll
        for (int mm = 0; mm < 2; ++mm)
          dQ[mm][n] = mfma(ld8_tr(Ks, LDK, 32 * kb, 16 * (2 * wave + mm)), a, dQ[mm][n]);
      }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const float f = scale * __expf(Gs[16 * n + r]);
#pragma unroll
      for (int mm = 0; mm < 2; ++mm) qrow[n][mm] = cvtf4(ld4(Qs + (16 * n + r) * LDK + 16 * (2 * wave + mm) + 4 * q4));
      float x = 0.f, y = 0.f;  // x: the output term's dG_t part; y: q_t . dQ_t (dQ complete here)
#pragma unroll
      for (int mm = 0; mm < 2; ++mm)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float inter = a1[mm][n][i] * f;
          dQ[mm][n][i] += inter;
          x += qrow[n][mm][i] * inter;
          y += qrow[n][mm][i] * dQ[mm][n][i];
        }
      x = sum_rows4(x);
      if (q4 == 0) dgl[16 * n + r] += x;
      pdot[n] = sum_rows4(y);
    }
  }
  lds_barrier();  // every read of the dO rows is done: the row dots and then the dVn tile may replace them
  if (q4 == 0) {
#pragma unroll
    for (int n = 0; n < 4; ++n) dqdot[4 * (16 * n + r) + wave] = pdot[n];  // after the tile's 16 KB
  }
  lds_barrier();
  // The dS fragments (bd) requested after phase 1 have landed long since: wait
  // for them here, where nothing else is in flight, so that their first use in
  // phase 3 does not wait for the dq stores and the dVn copy issued below (the
  // copy stands in a branch, so the compiler counts the path without it).
  wait_vmem_all();
  // dq = rq (dQ - q (q . dQ)): each lane holds 4 consecutive k of row t = 16 n + r
  const int rowb = H * D * 2;  // bytes per event row
  {
  // dq's rows over the dO rows (256-byte rows, 16-byte columns XORed with t % 16), then
  // whole rows to memory: a store whose lanes are rows costs 2.5 times the whole rows' time
  const __amdgpu_buffer_rsrc_t dq_rs = chunk_rows_rsrc(dq, ci.start, ci.len, H, h);
  E* dqs = dOs;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int t = 16 * n + r;
    const float rs = Rs[t];
    const f32x4 d4 = *reinterpret_cast<const f32x4*>(&dqdot[4 * t]);
    const float dot = d4[0] + d4[1] + d4[2] + d4[3];
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int k0 = 16 * (2 * wave + mm) + 4 * q4;
      const f32x4 x = normalize ? (dQ[mm][n] - qrow[n][mm] * dot) * rs : dQ[mm][n];
      st4(dqs + t * D + 8 * ((k0 >> 3) ^ r) + (k0 & 4), F16 ? x * inv_dv : x);  // row t, columns k0 .. k0 + 3
    }
  }
  lds_barrier();
  X8 rows[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) rows[i] = ld8(dqs + 512 * (4 * i + wave) + 8 * lane);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = 16 * i + 4 * wave + q4;
    buf_st16(dq_rs, t * rowb + 16 * (r ^ (t & 15)), rows[i]);
  }
  // this wave's pieces are read: the dVn copies below take exactly their places
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  // the dVn tile, copied global -> LDS while phase 3 runs (after the dq stores, which retire first)
  {
    const E* dvs = dVn + cb * (CH * D);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (stale)
        st8(dVs + 512 * (4 * i + wave) + 8 * lane, to8<E>(f32x8{NAN, NAN, NAN, NAN, NAN, NAN, NAN, NAN}));
      else if (ready)
        dma16_sc1(dvs + 512 * (4 * i + wave) + 8 * lane, dVs + 512 * (4 * i + wave));
      else
        dma16(dvs + 512 * (4 * i + wave) + 8 * lane, dVs + 512 * (4 * i + wave));
    }
  }

  // ---- phase 3: dK^T partial (k rows, t columns), kept in registers for the wy part ----
  f32x4 fkp[2][4];
  {
    float esum = 0.f;
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int m = 2 * wave + mm;
      f32x4 a3[4], a4[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) a3[n] = a4[n] = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const X8 a = ld8_tr(Qs, LDK, 32 * kb, 16 * m);
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          if (n > 2 * kb + 1) continue;
          a3[n] = mfma(a, ld8(dPm + (16 * n + r) * LDT + 32 * kb + 8 * q4), a3[n]);  // dPm^T rows s
        }
      }
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int n = 0; n < 4; ++n) a4[n] = mfma(bd[mm][kb], ld8_tr(VnT, LDT, 32 * kb, 16 * n), a4[n]);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int t = 16 * n + r;
        const float kd = __expf(glast - Gs[t]);
        const f32x4 st = a4[n] * kd;
        const f32x4 kk = cvtf4(ld4(Ks + t * LDK + 16 * m + 4 * q4));
        float e = st[0] * kk[0] + st[1] * kk[1] + st[2] * kk[2] + st[3] * kk[3];
        e = sum_rows4(e);
        if (q4 == 0) dgl[t] -= e;
        esum += (q4 == 0) ? e : 0.f;
        fkp[mm][n] = keep_if(t < ci.len, a3[n] + st);
      }
    }
    esum = sum16(esum);
    // <h, dS_{c+1}> over this wave's quarter of both
    float x = 0.f;
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) x = dot8(bh[mm][kb], bd[mm][kb], x);
    x = sum16(x);
    x = sum_rows4(x);
    if (lane == 0) dgl[ci.len - 1] += esum + __expf(glast) * x;
  }
  wait_vmem_all();  // the dVn tile has landed (the dq stores issued before it have retired too)
  lds_barrier();    // every read of Q, dPm and v_new^T is done

  // the wy part's V rows, T rows and beta, requested now and stored over Q and dPm after phase 4
  X8 pv[4], pt[2];
  float pb;
  {
    const int t = tid >> 2, p = tid & 3;
    const bool in = t < ci.len;
    const int tc = clamp_row(t, ci.len);
    const size_t row = ((size_t)(ci.start + tc) * H + h) * D;
    pb = keep_if(in, beta[(size_t)(ci.start + tc) * H + h]);
#pragma unroll
    for (int j = 0; j < 4; ++j) pv[j] = keep_if(in, ld8(vin + row + 32 * j + 8 * p));
    const E* tm = Tm + cb * (CH * CH);
#pragma unroll
    for (int j = 0; j < 2; ++j) pt[j] = ld8(tm + t * CH + 32 * j + 8 * p);
  }

  // ---- phase 4: dW = -dVn S^T into LDS rows [t][k]; the wy part's dVn fragments ----
  X8 fdv[4], fvt[2][2];
  {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int t = 16 * n + r;
      X8 av[4];  // dVn row t, value block kb
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) av[kb] = ld8(dVs + (2 * kb + (q4 >> 1)) * (CH * 16) + t * 16 + 8 * (q4 & 1));
#pragma unroll
      for (int mm = 0; mm < 2; ++mm) {
        const int m = 2 * wave + mm;
        f32x4 w = zero4();  // -dW^T[k = 16 m + 4 q4 + i][t] = (dVn S^T)^T, zero past the chunk
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) w = mfma(bh[mm][kb], av[kb], w);
        st4(dWs + t * LDK + 16 * m + 4 * q4, keep_if(t < ci.len, w));
      }
    }
    const int t = 16 * wave + r;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      fdv[kb] = keep_if(t < ci.len, ld8(dVs + (2 * kb + (q4 >> 1)) * (CH * 16) + t * 16 + 8 * (q4 & 1)));
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) fvt[mm][kb] = ld8_tr(dVs + (2 * wave + mm) * (CH * 16), 16, 32 * kb, 0);
  }
  lds_barrier();  // -dW rows complete, dG partials complete, the dVn tile consumed

  // ---- the WY part, on the chip-resident operands ----
  const float dgp_t = (tid < 64) ? dgw[0][tid] + dgw[1][tid] + dgw[2][tid] + dgw[3][tid] : 0.f;
  E* Vs = Qs;
  E* Ts = dPm;
  E* S1 = dOs;  // transposed: dT^T[s][t], then (beta dM)^T [j][i]
  E* S2 = VnT;                                                              // Y^T[j][t], over dW rows
  float* Bs = reinterpret_cast<float*>(r4a + 64 * LDT * 2);                   // after S1
  float* dbw = Bs + 64;                                                        // [4][64]
  float* dkdot = dbw + 256;                                                    // [64][4 waves]
  {
    const int t = tid >> 2, p = tid & 3;
    if (p == 0) Bs[t] = pb;
#pragma unroll
    for (int j = 0; j < 4; ++j)  // fp16: V s_v, in the scale of the forward's v_new and U
      st8(Vs + t * LDK + 32 * j + 8 * p, F16 ? to8<E>(cvtf8(pv[j]) * vs) : pv[j]);
#pragma unroll
    for (int j = 0; j < 2; ++j) st8(Ts + t * LDT + 32 * j + 8 * p, pt[j]);
  }
  lds_barrier();  // dgp_t has been read everywhere it is needed
  dgw[wave][lane] = 0.f;
  dbw[wave * 64 + lane] = 0.f;
  lds_barrier();
  float* dbl = dbw + wave * 64;

  // ---- wy phase 1: dT = dW (beta gam K)^T + dVn (beta V)^T -> S1 = dT[t][s]; dW fragments ----
  X8 fwt[2][2];
#pragma unroll
  for (int mm = 0; mm < 2; ++mm)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) fwt[mm][kb] = ld8_tr(dWs, LDK, 32 * kb, 16 * (2 * wave + mm));
  {
    X8 fdw[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) fdw[kb] = ld8(dWs + (16 * wave + r) * LDK + 32 * kb + 8 * q4);
    f32x4 ak[4], av[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) ak[n] = av[n] = zero4();
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        ak[n] = mfma(fdw[kb], ld8(Ks + (16 * n + r) * LDK + 32 * kb + 8 * q4), ak[n]);
        av[n] = mfma(fdv[kb], ld8(Vs + (16 * n + r) * LDK + 32 * kb + 8 * q4), av[n]);
      }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int s = 16 * n + r;
      const float fk = -(Bs[s] * __expf(Gs[s])), fv = Bs[s];  // ak holds -dW (beta gam K)^T
      st4(S1 + s * LDT + 16 * wave + 4 * q4, ak[n] * fk + av[n] * fv);
    }
  }
  float rsn[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const float x = rk[(size_t)(ci.start + clamp_row(16 * n + r, ci.len)) * H + h];  // allocated either way
    rsn[n] = normalize ? x : 1.f;
  }
  lds_barrier();  // S1 complete; every wave holds its dW fragments (S2 may overwrite the rows)

  // ---- wy phase 2: Y = dT T^T -> S2 = Y^T[j][t] ----
  {
    X8 a[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) a[kb] = ld8_tr(S1, LDT, 32 * kb, 16 * wave);  // dT rows t = 16 wave + r
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      f32x4 acc = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        if (n < 2 * kb) continue;  // T[j][b] = 0 for b > j
        acc = mfma(a[kb], ld8(Ts + (16 * n + r) * LDT + 32 * kb + 8 * q4), acc);
      }
      st4(S2 + (16 * n + r) * LDT + 16 * wave + 4 * q4, acc);
    }
  }
  lds_barrier();

  // ---- wy phase 3: dA = -T^T Y, dM, dbeta and dG from A, over the causal (i-tile, j-tile) pairs
  //      shared out as in phase 1 ----
  {
    // (beta dM)^T of i-tile it, j-tile n (at, ak: T^T and K fragments of i-tile it; gam: the
    // tile's gates from phase 1, whose diagonal 1 is masked here by dA's strict mask)
    auto pair = [&](int it, int n, const X8(&at)[2], const X8(&ak)[4], const f32x4& gam,
                    float(&rowB)[4], float(&rowE)[4]) -> f32x4 {
      f32x4 da = zero4(), kk = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        if (kb >= (it >= 2 ? 1 : 0)) da = mfma(at[kb], ld8(S2 + (16 * n + r) * LDT + 32 * kb + 8 * q4), da);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) kk = mfma(ak[kb], ld8(Ks + (16 * n + r) * LDK + 32 * kb + 8 * q4), kk);
      const int j = 16 * n + r;
      const f32x4 b4 = *reinterpret_cast<const f32x4*>(&Bs[16 * it + 4 * q4]);
      float colE = 0.f;
      f32x4 dmp;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * it + 4 * q4 + e;
        const bool strict = j < i;
        const float dA = strict ? -da[e] : 0.f;
        const float dM = dA * gam[e];
        const float Aij = b4[e] * kk[e] * gam[e];
        dmp[e] = b4[e] * dM;
        rowB[e] += dM * kk[e];
        const float e2 = dA * Aij;
        rowE[e] += e2;
        colE += e2;
      }
      colE = sum_rows4(colE);
      if (q4 == 0) dgl[j] -= colE;
      return dmp;
    };
    auto rows = [&](int it, const float(&rowB)[4], const float(&rowE)[4]) {
      float xb[4] = {rowB[0], rowB[1], rowB[2], rowB[3]}, xe[4] = {rowE[0], rowE[1], rowE[2], rowE[3]};
      sum16x4(xb);
      sum16x4(xe);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (r == 0) {
          dbl[16 * it + 4 * q4 + e] += xb[e];
          dgl[16 * it + 4 * q4 + e] += xe[e];
        }
      }
    };
    {
      X8 at[2], ak[4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) at[kb] = ld8_tr(Ts, LDT, 32 * kb, 16 * wave);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) ak[kb] = ld8(Ks + (16 * wave + r) * LDK + 32 * kb + 8 * q4);
      float rowB[4] = {0.f, 0.f, 0.f, 0.f}, rowE[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        if (n == 3 && wave == 3) continue;  // the (3, 3) tile is wave 0's
        const f32x4 dmp = (n <= wave) ? pair(wave, n, at, ak, gk[n], rowB, rowE) : zero4();
        st4(S1 + (16 * n + r) * LDT + 16 * wave + 4 * q4, dmp);
      }
      rows(wave, rowB, rowE);
    }
    if (wave == 0) {
      X8 at[2], ak[4];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) at[kb] = ld8_tr(Ts, LDT, 32 * kb, 48);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) ak[kb] = ld8(Ks + (48 + r) * LDK + 32 * kb + 8 * q4);
      float rowB[4] = {0.f, 0.f, 0.f, 0.f}, rowE[4] = {0.f, 0.f, 0.f, 0.f};
      st4(S1 + (48 + r) * LDT + 48 + 4 * q4, pair(3, 3, at, ak, gk[3], rowB, rowE));
      rows(3, rowB, rowE);
    }
  }
  lds_barrier();

  // ---- wy phase 4b: dv = beta (T^T dVn) ----
  {
    float colB[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int m = 2 * wave + mm;
      f32x4 acc[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[n] = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const X8 a = fvt[mm][kb];
#pragma unroll
        for (int n = 0; n < 4; ++n)
          if (kb >= 1 || n < 2) acc[n] = mfma(a, ld8_tr(Ts, LDT, 32 * kb, 16 * n), acc[n]);
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int s = 16 * n + r;
        const f32x4 vv = cvtf4(ld4(Vs + s * LDK + 16 * m + 4 * q4));
        colB[n] += acc[n][0] * vv[0] + acc[n][1] * vv[1] + acc[n][2] * vv[2] + acc[n][3] * vv[3];
        // over the V values that only this lane reads from here on
        st4(Vs + s * LDK + 16 * m + 4 * q4, acc[n] * (F16 ? Bs[s] * inv_d : Bs[s]));
      }
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      float xb = colB[n];
      xb = sum_rows4(xb);
      if (q4 == 0) dbl[16 * n + r] += xb;
    }
  }

  // ---- wy phase 4a: dK in registers ----
  f32x4 dkr[2][4];
  f32x4 krow[4][2];  // k[t = 16 n + r][16 (2w + mm) + 4 q4 + i], kept for the dk stores
  float pdk[4] = {0.f, 0.f, 0.f, 0.f};  // this wave's parts of the row dots k_t . dK_t
  {
    float colB[4] = {0.f, 0.f, 0.f, 0.f}, colG[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int m = 2 * wave + mm;
      f32x4 ak[4], aw[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) ak[n] = aw[n] = zero4();
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const X8 a = ld8_tr(Ks, LDK, 32 * kb, 16 * m);
        const X8 w = fwt[mm][kb];
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          if (n >= 2 * kb) ak[n] = mfma(a, ld8_tr(S1, LDT, 32 * kb, 16 * n), ak[n]);
          if (kb >= 1 || n < 2) {
            ak[n] = mfma(a, ld8(S1 + (16 * n + r) * LDT + 32 * kb + 8 * q4), ak[n]);
            aw[n] = mfma(w, ld8_tr(Ts, LDT, 32 * kb, 16 * n), aw[n]);
          }
        }
      }
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int t = 16 * n + r;
        const float bg = Bs[t] * __expf(Gs[t]);
        const f32x4 kk = krow[n][mm] = cvtf4(ld4(Ks + t * LDK + 16 * m + 4 * q4));
        // aw holds -(T^T dW): every use takes its sign back
        const float x = aw[n][0] * kk[0] + aw[n][1] * kk[1] + aw[n][2] * kk[2] + aw[n][3] * kk[3];
        colB[n] -= __expf(Gs[t]) * x;
        colG[n] -= bg * x;
        dkr[mm][n] = ak[n] + aw[n] * -bg + fkp[mm][n];
        pdk[n] += kk[0] * dkr[mm][n][0] + kk[1] * dkr[mm][n][1] + kk[2] * dkr[mm][n][2] + kk[3] * dkr[mm][n][3];
      }
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      float xb = colB[n], xg = colG[n];
      xb = sum_rows4(xb);
      xg = sum_rows4(xg);
      if (q4 == 0) {
        dbl[16 * n + r] += xb;
        dgl[16 * n + r] += xg;
      }
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const float pd = sum_rows4(pdk[n]);
      if (q4 == 0) dkdot[4 * (16 * n + r) + wave] = pd;
    }
  }
  lds_barrier();

  // ---- wy phase 5: l2norm backward of dk; dg (reverse cumsum of the chunk's dG); dbeta ----
  // dv and dk leave as whole rows, dv from the V rows' place, dk from the K rows'
  const __amdgpu_buffer_rsrc_t dk_rs = chunk_rows_rsrc(dk, ci.start, ci.len, H, h);
  const __amdgpu_buffer_rsrc_t dv_rs = chunk_rows_rsrc(dv, ci.start, ci.len, H, h);
  const int row_l = (tid >> 2) * LDK + 8 * (tid & 3), row_g = (tid >> 2) * rowb + 16 * (tid & 3);
#pragma unroll
  for (int j = 0; j < 4; ++j) buf_st16(dv_rs, row_g + 64 * j, ld8(Vs + row_l + 32 * j));
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int t = 16 * n + r;
    const f32x4 d4 = *reinterpret_cast<const f32x4*>(&dkdot[4 * t]);
    const float dot = d4[0] + d4[1] + d4[2] + d4[3];
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int m = 2 * wave + mm;
      const f32x4 out = normalize ? (dkr[mm][n] - krow[n][mm] * dot) * rsn[n] : dkr[mm][n];
      st4(Ks + t * LDK + 16 * m + 4 * q4, F16 ? out * inv_dv : out);
    }
  }
  lds_barrier();
#pragma unroll
  for (int j = 0; j < 4; ++j) buf_st16(dk_rs, row_g + 64 * j, ld8(Ks + row_l + 32 * j));
  if (tid < 64) {
    const int t = tid;
    const bool in = t < ci.len;
    float x = keep_if(in, dgp_t + dgw[0][t] + dgw[1][t] + dgw[2][t] + dgw[3][t]);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float o = __shfl_down(x, off, 64);
      if (t + off < 64) x += o;
    }
    if (in) {
      const float db = dbw[t] + dbw[64 + t] + dbw[128 + t] + dbw[192 + t];
      dg[(size_t)(ci.start + t) * H + h] = F16 ? x * inv_dv : x;
      dbeta[(size_t)(ci.start + t) * H + h] = F16 ? db * inv_dv : db;
    }
  }
}

// ---------------------------------------------------------------------------
// One wave on bwd_dkw's stream that ends once every reverse-scan workgroup has
// started (each adds one to *resident), so that bwd_dkw, launched behind it, can
// only take the CUs the scan leaves free and never holds one a scan workgroup
// still waits for.  Bounded: after COUNT_SPIN_LIMIT polls it ends anyway, and
// bwd_dkw's own bounded waits then decide.
__global__ __launch_bounds__(64) void scan_resident_gate_kernel(const int* __restrict__ resident, int expected) {
  if (threadIdx.x == 0) count_wait_ge<4>(resident, expected, COUNT_SPIN_LIMIT * 4);  // one wave: polls fast
}

static void launch_resident_gate(const int* resident, int expected, hipStream_t stream) {
  hipLaunchKernelGGL(scan_resident_gate_kernel, dim3(1), dim3(64), 0, stream, resident, expected);
}

// The scale target of dO: max|dO s_d| < 2^e with T 2^e <= 2^15, at most 2^1.
static int dout_scale_target(int T) {
  int lg = 0;
  while (lg < 31 && (1LL << lg) < (long long)T) ++lg;  // 2^lg >= T
  return 15 - lg < 1 ? 15 - lg : 1;
}

template <class E>
static hipError_t launch_bwd_t(const BwdArgs& a, hipStream_t stream) {
  auto F = [&](int i) { return reinterpret_cast<const E*>(a.fws + a.foff[i]); };
  auto Ff = [&](int i) { return reinterpret_cast<const float*>(a.fws + a.foff[i]); };
  auto B = [&](int i) { return reinterpret_cast<E*>(a.bws + a.boff[i]); };
  const E* q = static_cast<const E*>(a.q);
  const E* k = static_cast<const E*>(a.k);
  const E* v = static_cast<const E*>(a.v);
  const E* dout = static_cast<const E*>(a.dout);
  E* dq = static_cast<E*>(a.dq);
  E* dk = static_cast<E*>(a.dk);
  E* dv = static_cast<E*>(a.dv);
  const dim3 grid_p(a.H, a.n_chunks);  // chunk-major dispatch (the kernels pick the chunk order)
  int* sync = reinterpret_cast<int*>(a.bws + a.boff[B_SYNC]);
  int* ready = sync;                                 // [NC][H]
  int* resident = sync + (size_t)a.n_chunks * a.H;  // one count
  const bool beside = a.side != nullptr;
  // fp16: the scales s_d (partial maxima here, the scale itself in bwd_local) and s_v (the forward's)
  float* dsc = nullptr;
  const float* vsc = nullptr;
  if (__is_same(E, f16)) {
    dsc = reinterpret_cast<float*>(a.bws + a.boff[B_DSC]);
    vsc = Ff(F_VSC);
    launch_range_partials(a.dout, true, (size_t)a.T * a.H * (D / 8), nullptr, 0, dsc, stream);
  }
  {
    TimedLaunch tl(K_BWD_LOCAL, stream);
    hipLaunchKernelGGL(bwd_local_kernel<E>, dim3(a.H, a.n_chunks), dim3(256), 0, stream, q, k, (int)a.normalize, Ff(F_RK),
                       dout, Ff(F_GC), a.beta, F(F_TM), a.chunks, a.H, a.scale, dsc, dout_scale_target(a.T), B(B_DVLT),
                       B(B_XT), B(B_KNP), B(B_WT), sync);
  }
  if (beside) {
    if (const hipError_t e = hipEventRecord(a.side_fork, stream)) return e;
    if (const hipError_t e = hipStreamWaitEvent(a.side, a.side_fork, 0)) return e;
  }
  {
    TimedLaunch tl(K_BWD_SCAN, stream);
    // beside, every workgroup is resident at once: far fewer heads than scan_wide's
    const auto kernel = beside            ? bwd_scan_kernel<E, true, false>
                        : scan_wide(a.H) ? bwd_scan_kernel<E, false, true>
                                         : bwd_scan_kernel<E, false, false>;
    hipLaunchKernelGGL(kernel, dim3(a.H * (D / 16), a.n_docs), dim3(SCAN_THREADS), beside ? BESIDE_LDS : 0, stream,
                       B(B_KNP), Ff(F_GC), B(B_DVLT), B(B_XT), B(B_WT), a.chunks, a.doc_chunk, a.H, B(B_DH), B(B_DVN),
                       ready, resident);
  }
  if (beside) {
    launch_resident_gate(resident, a.H * (D / 16) * a.n_docs, a.side);
    {
      TimedLaunch tl(K_BWD_DKW, a.side);
      hipLaunchKernelGGL(bwd_dkw_kernel<E>, grid_p, dim3(256), 0, a.side, q, k, Ff(F_RK), Ff(F_GC),
                         F(F_HT), F(F_VNT), dout, B(B_DH), B(B_DVN), v, a.beta, F(F_TM), a.chunks, a.H, a.scale,
                         (int)a.normalize, (const float*)dsc, vsc, dq, dk, dv, a.dg, a.dbeta, (const int*)ready,
                         a.dkw_never_ready ? D / 16 + 1 : D / 16, a.dkw_never_ready ? 4 : COUNT_SPIN_LIMIT);
    }
    if (const hipError_t e = hipEventRecord(a.side_join, a.side)) return e;
    return hipStreamWaitEvent(stream, a.side_join, 0);
  }
  if (a.dkw_after)
    if (const hipError_t e = hipStreamWaitEvent(stream, a.dkw_after, 0)) return e;
  TimedLaunch tl(K_BWD_DKW, stream);
  hipLaunchKernelGGL(bwd_dkw_kernel<E>, grid_p, dim3(256), 0, stream, q, k, Ff(F_RK), Ff(F_GC), F(F_HT),
                     F(F_VNT), dout, B(B_DH), B(B_DVN), v, a.beta, F(F_TM), a.chunks, a.H, a.scale, (int)a.normalize,
                     (const float*)dsc, vsc, dq, dk, dv, a.dg, a.dbeta, (const int*)nullptr, 0, 0);
  return hipSuccess;
}

hipError_t launch_bwd(const BwdArgs& a, hipStream_t stream) {
  return a.fp16 ? launch_bwd_t<f16>(a, stream) : launch_bwd_t<bf16>(a, stream);
}

}  // namespace cqgdn
