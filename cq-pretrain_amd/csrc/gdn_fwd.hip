// GDN forward on gfx950: chunk preparation, inter-chunk state scan, output.
//
// Math (per document, chunks of C = 64 events, state S in R^{K x V} fp32):
//   G = chunk-local cumsum(g), gam = exp(G), Gam_ij = exp(G_i - G_j) (i >= j)
//   A = strict_lower(beta_i * (k_i . k_j) * Gam_ij),  T = (I + A)^-1
//   W = T (beta*gam*K),  U = T (beta*V)
//   Vn = U - W S,  O = scale * [ (gam*Q) S + ((Q K^T) * Gam) Vn ]
//   S <- exp(G_last) S + (K * exp(G_last - G))^T Vn
// (reference_modeling_qwen3_5.py:344-411; the reference's op chain is the
//  K-b..K-g set of ops/gated_delta_net.py:144-183).
//
// Kernels:
//   fwd_prep   grid (NC, H), 4 waves: l2norm q,k; cumsum g; A via MFMA; the unit
//              lower-triangular inverse in LDS (fp32); W, U via MFMA.
//   fwd_scan   grid (H * 8 value slices, docs), 4 waves: the serial scan, a 128x16
//              fp32 state slice held in registers across all chunks of a document.
//   fwd_out    grid (NC, H), 4 waves: O^T = gam * (h^T Qn^T) + Vn^T P^T, all MFMA.
#include "gdn_common.hpp"
#include "gdn_layout.hpp"
#include "gdn_kernels.hpp"

namespace cqgdn {

constexpr int LDK = 136;  // row stride (elements) of 64 x 128 tiles in LDS
constexpr int LDT = 72;   // row stride (elements) of 128 x 64 and 64 x 64 tiles in LDS
constexpr int LDA = 65;   // row stride (fp32) of the 64 x 64 solve matrix

// ---------------------------------------------------------------------------
// fwd_prep
// ---------------------------------------------------------------------------
// I: input element type of q, k, v (bf16 or f16).  E: operand element type (bf16,
// or f16 for the precise forward and for fp16 inputs).  vscale: with f16 operands,
// the power-of-two factor applied to V (fp16 range), which this kernel forms from
// the partial maxima after vscale[0] (range_scale, target vs_target) and stores in
// vscale[0] for the scan and the output kernel; null with bf16 operands.
template <class I, class E, bool NORMALIZE>
__global__ __launch_bounds__(256, 3) void fwd_prep_kernel(
    const I* __restrict__ k, const I* __restrict__ v,
    const float* __restrict__ g, const float* __restrict__ beta, const int32_t* __restrict__ chunks,
    int H, float* __restrict__ vscale, int vs_target,
    float* __restrict__ rk, float* __restrict__ gc, E* __restrict__ Tm, E* __restrict__ W,
    E* __restrict__ UT, E* __restrict__ KgT) {
  typedef typename Vec<E>::x8 X8;
  typedef typename Vec<E>::x4 X4;
  // grid (H, NC), chunks dispatched last to first: the state scan reads the
  // first chunks first, and they are then the most recently written (still in
  // the memory-side cache)
  const HeadChunk hc = xcd_head_chunk(gridDim.x, gridDim.y);  // all heads of a chunk on one XCD
  const int h = hc.h, c = gridDim.y - 1 - hc.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q4 = lane >> 4;
  const ChunkInfo ci = chunk_info(chunks, c);
  const size_t cb = (size_t)c * H + h;

  __shared__ __attribute__((aligned(16))) float Gs[64];
  __shared__ __attribute__((aligned(16))) float Bs[64];
  __shared__ __attribute__((aligned(16))) E Ks[64 * LDK];      // K rows, then (beta gam K) rows
  __shared__ __attribute__((aligned(16))) float Af[64 * LDA];  // the solve's matrix, then the KgT tile
  __shared__ __attribute__((aligned(16))) E Ts[64 * LDT];
  __shared__ float red[4];
  // fp16 operands (the only ones with a scale): this thread's partial maximum of
  // |V|, requested before the other loads
  constexpr bool SCALED = __is_same(E, f16);
  const float vpart = SCALED ? range_partial4(vscale + 1) : 0.f;

  // Every global load is issued first, before any store (a wait for a load
  // also waits for every store issued before it), so the kernel pays one memory
  // round trip: the gates (wave 0), this thread's pieces of its k row,
  // and the columns 32 wave .. of V for U = T (beta V) (rows past the chunk re-read
  // its last row; their beta is zero).  Each phase waits only for what it reads, and
  // the stores of the row phase go through buffer resources (rows past the chunk dropped by the range
  // check), so no store is conditional and the compiler can count what is in flight.
  // k is loaded non-temporally: nothing reads it again before the state scan,
  // whose operands (written here) then keep more of the memory-side cache.  q is
  // not read here: its l2 scale is formed by each kernel that reads q (row_rnorm).
  const int t_r = tid >> 2, p_r = tid & 3;  // row phase: thread (t, p) owns columns 8p + 32j, j = 0..3
  const size_t row_r = ((size_t)(ci.start + clamp_row(t_r, ci.len)) * H + h) * D;
  float gv = 0.f, bv = 0.f;
  if (wave == 0) {
    const size_t ev = (size_t)(ci.start + clamp_row(lane, ci.len)) * H + h;
    gv = g[ev];
    bv = beta[ev];
  }
  typename Vec<I>::x8 lk[4];
  typename Vec<I>::x8 vr[4], vg[2][2];  // V rows 16 i + lane / 4 by quads, then the fragments (tile nn, t block kb)
#pragma unroll
  for (int j = 0; j < 4; ++j) lk[j] = ld8_nt(k + row_r + 32 * j + 8 * p_r);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    vr[i] = row_piece(v + ((size_t)ci.start * H + h) * D, (size_t)H * D, clamp_row(16 * i + (lane >> 2), ci.len), 32 * wave);
  // the scale of V, while the loads above are in flight (stored for the kernels
  // after this one at the end, where the store holds up no wait for a load)
  float vs = 1.f;
  if constexpr (SCALED) vs = range_scale(vpart, vs_target, red);
  const int rowe = H * D * (int)sizeof(E);  // bytes per event row of W
  const int rows_bytes = ((ci.len - 1) * H + 1) * D * (int)sizeof(E);
  const int gate_bytes = ((ci.len - 1) * H + 1) * (int)sizeof(float);

  // ---- gates: chunk-local cumsum of g (wave 0, one event per lane) ----
  if (wave == 0) {
    const bool in = lane < ci.len;
    gv = keep_if(in, gv);
    bv = keep_if(in, bv);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float o = __shfl_up(gv, off, 64);
      if (lane >= off) gv += o;
    }
    Gs[lane] = gv;
    Bs[lane] = bv;
    buf_stf(buf_rsrc(gc + (size_t)ci.start * H + h, gate_bytes), lane * H * 4, 0, gv);  // rows past the chunk dropped
  }
  __syncthreads();
  const float glast = Gs[ci.len - 1];

  // ---- rows ----
  // Kg = K exp(G_last - G) is kept in registers and leaves through LDS after the
  // solve (coalesced rows of KgT instead of 2-byte scattered stores); beta gam K
  // (rounded once, from fp32) replaces K in LDS once A has been formed.
  X8 kg8[4], kb8[4];
  {
    const int t = t_r, p = p_r;
    const bool in = t < ci.len;
    const float gam_t = __expf(Gs[t]);
    const float kdec_t = __expf(glast - Gs[t]);
    const float b_t = Bs[t];
    const __amdgpu_buffer_rsrc_t rk_rs = buf_rsrc(rk + (size_t)ci.start * H + h, gate_bytes);
    // k
    {
      f32x8 x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = keep_if(in, cvtf8(lk[j]));
      float rs = 1.f;
      if (NORMALIZE) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int s = 0; s < 8; ++s) ss += x[j][s] * x[j][s];
        ss = sum4(ss);
        rs = rsqrtf(ss + 1e-6f);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x8 xn = x[j] * rs;
        const X8 xb = to8<E>(xn);
        const int col = 32 * j + 8 * p;
        st8(Ks + t * LDK + col, xb);
        kb8[j] = to8<E>(xn * (b_t * gam_t));
        kg8[j] = to8<E>(xn * kdec_t);
      }
      buf_stf(rk_rs, t * H * 4, 0, rs);
    }
  }
  // the V fragments, through the place of T (written after the solve)
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    typename Vec<I>::x8 y[2];
    columns_from_rows(reinterpret_cast<I*>(Ts) + 1024 * wave, vr[2 * kb], vr[2 * kb + 1], y);
    vg[0][kb] = y[0];
    vg[1][kb] = y[1];
  }
  __syncthreads();

  // ---- A = strict_lower(beta_t (k_t . k_s) Gam_ts): t-tile = wave, s-tiles <= wave ----
  {
    f32x4 acc[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[n] = zero4();
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const X8 a = ld8(Ks + (16 * wave + r) * LDK + 32 * kb + 8 * q4);
#pragma unroll
      for (int n = 0; n < 4; ++n)
        if (n <= wave) acc[n] = mfma(a, ld8(Ks + (16 * n + r) * LDK + 32 * kb + 8 * q4), acc[n]);
    }
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int s = 16 * n + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * wave + 4 * q4 + i;
        Af[t * LDA + s] = (s < t) ? Bs[t] * acc[n][i] * __expf(Gs[t] - Gs[s]) : 0.f;
      }
    }
  }
  __syncthreads();
  // every read of K is done: beta gam K takes its rows (read again only after the solve)
#pragma unroll
  for (int j = 0; j < 4; ++j) st8(Ks + t_r * LDK + 32 * j + 8 * p_r, kb8[j]);

  // ---- T = (I + A)^-1, blocked by 16, in fp32 ----
  // The four diagonal blocks by forward substitution (column c = tid/4 of block
  // c/16, lanes p split the sums), then the blocks below the diagonal level by
  // level (i - j = 1, 2, 3):  X_ij = sum_{k=j}^{i-1} A_ik T_kj,  T_ij = -T_ii X_ij.
  // Af then holds T_ii in the diagonal blocks and T_ij^T (i > j) in block
  // (j, i) above the diagonal (A's upper triangle is zero and unused); the
  // blocks below the diagonal still hold A.
  {
    const int col = tid >> 2, p = tid & 3, b0 = col & ~15, lc = col & 15;
    float tc[4];  // T[b0 + 4 jj + p][col]
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) tc[jj] = (4 * jj + p == lc) ? 1.f : 0.f;
#pragma unroll
    for (int i = 1; i < 16; ++i) {
      float part = 0.f;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) part += Af[(b0 + i) * LDA + b0 + 4 * jj + p] * tc[jj];
      part = sum4(part);
      const float val = (i > lc) ? -part : ((i == lc) ? 1.f : 0.f);
      if ((i & 3) == p) tc[i >> 2] = val;
    }
    __syncthreads();  // every read of A's diagonal blocks is done
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) Af[(b0 + 4 * jj + p) * LDA + col] = tc[jj];
  }
  // The levels below the diagonal, d = 1, 2, 3, on fp32 MFMA (16x16x4): wave w <
  // 4 - d owns the target block (ib, jb) = (w + d, w).  X = sum_{k=jb}^{ib-1}
  // A_{ib,k} T_{k,jb} reads only lower levels (T_{jb,jb} in its diagonal block,
  // T_{k,jb}, k > jb, transposed in block (jb, k)); X goes to the wave's own
  // block (jb, ib), transposed, and comes back as the operand of T_{ib,jb} =
  // -T_{ib,ib} X, which replaces it.  The block is the wave's alone (its LDS
  // operations complete in order), so the levels need one barrier each.
#pragma unroll
  for (int d = 1; d < 4; ++d) {
    __syncthreads();  // the diagonal blocks and the lower levels are complete
    if (wave < 4 - d) {
      const int jb = wave, ib = wave + d;
      const float* arow = Af + (16 * ib + r) * LDA + q4;  // A_{ib, .} row r at this lane's k (4 kk + q4)
      f32x4 x = zero4();
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        x = mfma4(arow[16 * jb + 4 * kk], Af[(16 * jb + 4 * kk + q4) * LDA + 16 * jb + r], x);
      for (int kb = jb + 1; kb < ib; ++kb)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          x = mfma4(arow[16 * kb + 4 * kk], Af[(16 * jb + r) * LDA + 16 * kb + 4 * kk + q4], x);
      float* blk = Af + (16 * jb + r) * LDA + 16 * ib;  // block (jb, ib), row r: X^T, then T_{ib,jb}^T
#pragma unroll
      for (int i = 0; i < 4; ++i) blk[4 * q4 + i] = x[i];
      const float* trow = Af + (16 * ib + r) * LDA + 16 * ib + q4;  // T_{ib,ib} row r at k = 4 kk + q4
      f32x4 y = zero4();
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) y = mfma4(trow[4 * kk], blk[4 * kk + q4], y);
#pragma unroll
      for (int i = 0; i < 4; ++i) blk[4 * q4 + i] = -y[i];
    }
  }
  __syncthreads();
  {
    // T in the operand type: Ts rows [t][s], then the global copy from those rows.
    // The lanes of a wave run along one row (rows 4 jj + wave), so every read and
    // write of the copy touches 32 distinct banks (the solve matrix's row stride
    // is 65 words: its transposed blocks are read down consecutive rows).
    const int col = tid & 63, bcb = col >> 4;
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
      const int t = 4 * jj + wave, bt = t >> 4;
      const float val = (bt == bcb) ? Af[t * LDA + col]
                                    : (bt > bcb ? Af[(16 * bcb + (col & 15)) * LDA + 16 * bt + (t & 15)] : 0.f);
      Ts[t * LDT + col] = (E)val;
    }
  }
  __syncthreads();
  {
    E* tm = Tm + cb * (CH * CH);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int seg = 256 * i + tid, row = seg >> 3, part = seg & 7;
      st8(tm + row * CH + 8 * part, ld8(Ts + row * LDT + 8 * part));
    }
  }

  // Kg^T over the solve's matrix (free now), in the order the scan reads it (stored
  // below): fragment (k / 16, t / 32), and in it 16-byte granule 16 g + r holding row
  // k = 16 (k / 16) + r at the four-runs g of both halves of the 32 events (perm32).  A
  // granule's low three bits are XORed with g + 4 (r / 8): the 16 (event run, quarter)
  // pairs that write together then spread over all the banks, and the reads stay
  // conflict-free.
  E* kgs = reinterpret_cast<E*>(Af);
  static_assert(sizeof(Af) >= D * CH * sizeof(E), "the KgT tile must fit the solve matrix");
  {
    const int t = tid >> 2, p = tid & 3, tp = perm32(t), g = (tp >> 3) & 3;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int k = 32 * j + 8 * p + s, gran = 16 * g + ((k & 15) ^ (g + 4 * (p & 1)));
        kgs[((2 * (k >> 4) + (t >> 5)) * 64 + gran) * 8 + (tp & 7)] = kg8[j][s];
      }
  }

  // ---- W = T (beta gam K) -> W rows, U = T (beta V) -> U^T storage ----
  // beta gam K is read transposed from its rows (ld8_tr); beta V comes from the
  // V fragments gathered at the start, scaled here.  (-W^T, the reverse scan's
  // operand, is formed by bwd_local.)
  X4 uo[2][4], wo[2][4];
  {
    X8 bvf[2][2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const f32x4 b0 = *reinterpret_cast<const f32x4*>(Bs + 32 * kb + 8 * q4);
      const f32x4 b1 = *reinterpret_cast<const f32x4*>(Bs + 32 * kb + 8 * q4 + 4);
      const f32x8 bb = f32x8{b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]} * vs;
#pragma unroll
      for (int nn = 0; nn < 2; ++nn) bvf[nn][kb] = to8<E>(cvtf8(vg[nn][kb]) * bb);
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      X8 a[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) a[kb] = ld8(Ts + (16 * tt + r) * LDT + 32 * kb + 8 * q4);
#pragma unroll
      for (int nn = 0; nn < 2; ++nn) {
        f32x4 au = zero4();
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          if (kb == 0 || tt >= 2) au = mfma(a[kb], bvf[nn][kb], au);  // T[t][s] = 0 for s > t
        uo[nn][tt] = to4<E>(au);
      }
    }
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int m = 2 * wave + mm;
      X8 ak[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) ak[kb] = ld8_trv<E>(Ks, LDK, 32 * kb, 16 * m);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        f32x4 acc = zero4();
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) acc = mfma(ak[kb], ld8(Ts + (16 * n + r) * LDT + 32 * kb + 8 * q4), acc);
        wo[mm][n] = to4<E>(-acc);
      }
    }
  }
  // The outputs leave as whole rows through LDS (a store whose lanes are rows takes the
  // vector memory unit 2.5 times as long; with V read by row pieces instead of column
  // gathers: H = 16, 144 / 520 / 36 / 5 chunks 62.6 -> 55.2 / 196 -> 160 / 21.0 -> 19.2 /
  // 13.4 -> 12.3 us in a step's kernel trace, 3.8 and 4.7 TB/s on the two long ones): Kg^T from the
  // solve's region, -W through the K rows' place, then U^T through the solve's region.
  __syncthreads();  // the KgT tile is complete, every read of beta gam K is done
  {
    E* kgt = KgT + cb * (D * CH);
    X8 x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int seg = 256 * i + tid;
      x[i] = ld8(kgs + (seg ^ (((seg >> 4) & 3) + 4 * ((seg >> 3) & 1))) * 8);
    }
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)  // row t = 16 n + r, columns k = 16 (2 wave + mm) + 4 q4 .. in perm32 order
#pragma unroll
      for (int n = 0; n < 4; ++n)
        *reinterpret_cast<X4*>(Ks + (16 * n + r) * LDK + perm32(16 * (2 * wave + mm) + 4 * q4)) = wo[mm][n];
#pragma unroll
    for (int i = 0; i < 4; ++i) st8(kgt + (256 * i + tid) * 8, x[i]);
  }
  lds_barrier();  // every read of the KgT tile is done, -W is complete
  {
    const __amdgpu_buffer_rsrc_t w_rs = buf_rsrc(W + ((size_t)ci.start * H + h) * D, rows_bytes);
    X8 x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = ld8(Ks + t_r * LDK + 32 * j + 8 * p_r);
#pragma unroll
    for (int nn = 0; nn < 2; ++nn)  // U^T row v = 16 (2 wave + nn) + r, t = 16 tt + 4 q4 ..
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
        *reinterpret_cast<X4*>(kgs + (16 * (2 * wave + nn) + r) * CH + 8 * ((2 * tt + (q4 >> 1)) ^ (r & 7)) + 4 * (q4 & 1)) =
            uo[nn][tt];
#pragma unroll
    for (int j = 0; j < 4; ++j) buf_st16(w_rs, t_r * rowe + 64 * j + 16 * p_r, x[j]);  // rows past the chunk fall outside w_rs
  }
  lds_barrier();
  {
    E* ut = UT + cb * (D * CH);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int seg = 256 * i + tid;  // row v = seg / 8, 16-byte column seg % 8
      st8(ut + seg * 8, ld8(kgs + (seg ^ ((seg >> 3) & 7)) * 8));
    }
  }
  if (SCALED && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) vscale[0] = vs;
}

// ---------------------------------------------------------------------------
// fwd_scan: the serial scan, four waves per (head, 16-wide value slice, document)
// ---------------------------------------------------------------------------
// The scan is a chain of dependent chunk steps.  A workgroup serves one 16-wide value
// slice of one head; wave w holds rows 32 w .. 32 w + 31 of the slice's fp32 state in two
// C tiles and does a quarter of each contraction:
//   v_new rows t = 16 w ..  = U + (-W rows) S      needs all of S, in the operand type
//   S rows k = 32 w ..      = e^G S + Kg^T v_new   needs all of v_new
// so a step passes the operand copy of S (4 KB) and v_new (2 KB) through LDS, with a
// barrier after each, and its chain is 4 + 2 dependent MFMAs and two LDS round trips:
// 48 us over 144 steps with no operand traffic.  (One wave doing it all needs 32 MFMAs in
// a row and reads 34 KB of operands from LDS; with two loader waves feeding it the kernel
// took 102 us.)
//
// What bounds a step now is what one CU's vector memory takes in: every workgroup of a
// head reads all of -W and Kg^T, 34 KB a step, and writes 6 KB.  Each lane group has to
// read whole 64-byte pieces for that (see "the vector memory unit" in gdn_common.hpp):
//   Kg^T  is stored in fragment order by fwd_prep: 1 KB of contiguous lanes' operands a load;
//   -W    rows go to LDS by asynchronous copies of four 256-byte rows (16-byte columns
//         XOR-swizzled by row), each wave its own 16 rows, and come back as fragments;
//   U^T   is read by quads and exchanged between lanes (tile_exchange);
//   h^T, v_new^T leave as whole rows, read back from the LDS copies; h^T with the
//   non-temporal hint: its 32 KB a chunk-head would push the operands of the chunks still
//   to come, and then bwd_local's, out of the memory-side cache (a training step of 144
//   chunks 477 -> 464 us, packed 1496 -> 1484, 36 chunks 140.1 -> 139.4; v_new^T as well
//   slowed fwd_out by 3 us and gained nothing more on a step).
// With fragments read straight from the row-major matrices the same kernel took 173 us.
// Operands are requested SCAN_DEPTH steps ahead into registers (and four LDS rings);
// 3, 5 or 6 steps measured the same.  Half of a step's requests go out in each of its
// two waits (Kg^T a step later than -W): all at once they filled the memory unit's queue
// and held up the wave's MFMAs (each scan alone, H = 16 / 4, 144 chunks: 84.5 -> 80.7 /
// 74.6 -> 72.8 us, the reverse scan 93.4 -> 92 / 83.5 -> 77.9; 36 chunks 23.1 -> 22.0,
// 25.3 -> 24.2).  No step computes an address (ScanBlocks, ScanTable)
// and nothing in a round is conditional, so the compiler's own waits leave every later
// request in flight; the first round is peeled because a loop entered with fewer
// operations in flight than it runs with waits as strictly as its entry.
//
// Measured in the kernel trace of whole steps (H = 16, one document of 144 chunks / 15
// documents, 520 chunks): 107 -> 85 us, 298 -> 249 us; 36 chunks 29.7 -> 22.0; four heads,
// 144 chunks 98.6 -> 73.3.  LDS
// went from 136 KB to 72 KB a workgroup, so two share a CU.
//
// The waits for -W: loads, copies and stores of a wave retire in issue order, so a copy
// has landed once at most as many operations are in flight as were surely issued after
// it.  Counted are the operations of whole windows between barriers (the compiler may
// reorder a window's own): a full step issues 11 (9 loads, 2 stores), and the Kg^T loads
// and the store of h^T of its own step precede the wait.
constexpr int FWD_STEP_OPS = 11, FWD_LOAD_OPS = 9;

// LDS that a workgroup of a scan on the side stream takes in addition, unused: with it none of
// the reverse scan (SCAN_EXCHANGE_BYTES), which runs beside it, shares its CU.  On a shared CU
// the two halve each other: the backward with its forward rebuilt, us, H = 16 / 4 / 8, one document
// of 144 / 144 / 512 chunks: 482 / 208 / 1134, alone on its CU 412 / 160 / 860 (two loader waves and
// 136 KB a workgroup, which never shared, 434 / 199 / 924).
constexpr int FWD_RING_BYTES = SCAN_DEPTH * 64 * D * 2, FWD_ALONE_LDS = 84 * 1024;
static_assert(FWD_RING_BYTES + SCAN_EXCHANGE_BYTES + FWD_ALONE_LDS + SCAN_EXCHANGE_BYTES > LDS_BYTES &&
                  FWD_RING_BYTES + SCAN_EXCHANGE_BYTES + FWD_ALONE_LDS <= LDS_BYTES,
              "one forward scan workgroup fits a CU, a reverse scan workgroup no longer");
template <class E, bool WIDE>
__global__ __launch_bounds__(SCAN_THREADS, 2) void fwd_scan_kernel(
    // without __restrict__ where loads are requested ahead: the barriers then pin their place
    const E* W, const E* UT, const E* KgT, const float* gc, const int32_t* chunks,
    const int32_t* __restrict__ doc_chunk, int H, const float* __restrict__ vscale,
    const float* __restrict__ init_state, float* __restrict__ final_state, E* hT, E* vnT) {
  typedef typename Vec<E>::x8 X8;
  typedef typename Vec<E>::x4 X4;
  // blockIdx.x = slice * H + h: the slices of one head land on one XCD when H % 8 == 0
  const int h = blockIdx.x % H, slice = blockIdx.x / H, d = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q4 = lane >> 4;
  const int v0 = 16 * slice;

  __shared__ __attribute__((aligned(16))) E Sx[16 * SCAN_SROW];  // the state's operand copy, [v][perm32(k)]
  __shared__ __attribute__((aligned(16))) E Vx[16 * SCAN_VROW];  // v_new, [v][perm32(t)]
  // -W rows of SCAN_DEPTH chunks, each wave's 16 rows its own
  __shared__ __attribute__((aligned(16))) E W0[64 * D], W1[64 * D], W2[64 * D], W3[64 * D];
  static_assert(SCAN_DEPTH == 4, "four rings, and the waits below");

  const int c_begin = __builtin_amdgcn_readfirstlane(doc_chunk[d]);
  const int n = __builtin_amdgcn_readfirstlane(doc_chunk[d + 1]) - c_begin;
  const float vs = vscale ? *vscale : 1.f;  // the state is carried in the scale of V
  f32x4 S[2];  // S[m][i] = state[k = 32 wave + 16 m + 4 q4 + i][v = v0 + r]
#pragma unroll
  for (int m = 0; m < 2; ++m) S[m] = zero4();
  if (init_state) {
    const float* s0 = init_state + ((size_t)d * H + h) * D * D;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[m][i] = s0[(32 * wave + 16 * m + 4 * q4 + i) * D + v0 + r] * vs;
  }
  if (n > 0) {
    ScanTable tab(chunks, gc, W, c_begin, 1, n, H, h, lane);
    tab.open();
    const size_t cb = (size_t)c_begin * H + h;
    const int64_t tile = (int64_t)H * D * CH * 2;  // bytes from one chunk's [D][64] tile to the next chunk's
    ScanBlocks<false, WIDE> ub(UT + cb * (D * CH) + v0 * CH, tile, n);
    ScanBlocks<false, WIDE> kb(KgT + (cb - H) * (D * CH), tile, n + 1);  // one step behind: its first block is step -1's
    ScanBlocks<false, WIDE> vb(vnT + cb * (D * CH) + v0 * CH, tile, n), hb(hT + cb * (D * D) + v0 * D, 2 * tile, n);
    // per-lane parts of the addresses, the same for every chunk (bytes of global
    // memory; elements of LDS)
    const int q = (lane >> 2) & 3, p = lane & 3, from = tile_source(lane);
    int w_off[4], w_in[4];  // -W rows 16 wave + 4 i + q4, column r ^ row; fragment j: row 16 wave + r, column 4 q4 + j
#pragma unroll
    for (int i = 0; i < 4; ++i) w_off[i] = (16 * wave + 4 * i + q4) * H * D * 2 + 16 * (r ^ (4 * i + q4));
    E* const ring[SCAN_DEPTH] = {W0, W1, W2, W3};
#pragma unroll
    for (int j = 0; j < 4; ++j) w_in[j] = (16 * wave + r) * D + 8 * ((4 * q4 + j) ^ r);
    const int k_off = 4096 * wave + 16 * lane;                    // fragments (wave, m, b) of KgT
    const int u_off = (4 * q4 + q) * CH * 2 + 32 * wave + 8 * p;  // U^T row 4 q4 + q, t = 16 wave + 4 p ..
    const int s_own = r * SCAN_SROW + 32 * wave + 8 * q4, s_in = r * SCAN_SROW + 32 * q4;
    const int v_own = r * SCAN_VROW + 32 * (wave >> 1) + 8 * q4 + 4 * (wave & 1), v_in = r * SCAN_VROW + 8 * q4;
    // the outputs as rows: h^T row 4 wave + q4, k = 8 r .. 8 r + 7 (two runs of four in
    // perm32 order), v_new^T row 4 wave + q4, t = 4 r .. 4 r + 3
    const int s_row = (4 * wave + q4) * SCAN_SROW, s_lo = s_row + perm32(8 * r), s_hi = s_row + perm32(8 * r + 4);
    const int v_row = (4 * wave + q4) * SCAN_VROW + perm32(4 * r);
    const int h_off = 1024 * wave + 16 * lane, vn_off = 512 * wave + 8 * lane;
    X8 fk[SCAN_DEPTH][2][2];
    X4 fu[SCAN_DEPTH], u;
    X8 w[4];
    float gl[SCAN_DEPTH];
    // l: the step's place after the table's and the blocks' first
    auto issue_w = [&](int slot, int l) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t wr = tab.rows(l), ur = ub.buffer(l);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void_ptr)(ring[slot] + (16 * wave + 4 * i) * D), 16,
                                                 w_off[i], 0, 0, 0);
      fu[slot] = buf_ld8<X4>(ur, u_off, ub.offset(l));
      gl[slot] = tab.glast(l);
    };
    auto issue_k = [&](int slot, int l) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t kr = kb.buffer(l);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int b = 0; b < 2; ++b) fk[slot][m][b] = buf_ld16<X8>(kr, k_off + 2048 * m + 1024 * b, kb.offset(l));
    };
    st8(Sx + s_own, pack_permv<E>(S[0], S[1]));
#pragma unroll
    for (int x = 0; x < SCAN_DEPTH; ++x) {
      issue_w(x, x);
      if (x > 0) issue_k(x - 1, x);
      __builtin_amdgcn_sched_barrier(0);  // in this order: the waits count on it
    }
    // -W of the next step, once at most `flight` operations are in flight
    auto take_w = [&](auto flight, int slot) __attribute__((always_inline)) {
      wait_vmem_le<decltype(flight)::value>();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = ld8(ring[slot] + w_in[j]);
    };
    float g_now = __expf(gl[0]);
    u = tile_exchange(fu[0], from);
    take_w(Int<3 * FWD_LOAD_OPS>(), 0);
    ub.advance();
    kb.advance();
    lds_barrier();
    // one step: its -W, U and decay are in w, u and g_now; place: its place in the round;
    // more: not one of the last steps, whose requests would all lie past the end; flight:
    // operations surely issued after the next step's -W
    auto step = [&](auto place, auto more, auto flight) __attribute__((always_inline)) {
      constexpr int s = decltype(place)::value;
      // v_new = U + (-W) S
      X8 sx[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) sx[j] = ld8(Sx + s_in + 8 * j);
      const X8 h_out = cat(ld4(Sx + s_lo), ld4(Sx + s_hi));
      if constexpr (decltype(more)::value) issue_k((s + SCAN_DEPTH - 1) % SCAN_DEPTH, s);
      f32x4 acc = cvtf4(u);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = mfma(w[j], sx[j], acc);
      buf_st16<CPOL_NT>(hb.buffer(s), h_off + hb.offset(s), h_out);
#pragma unroll
      for (int m = 0; m < 2; ++m) S[m] *= g_now;
      *reinterpret_cast<X4*>(Vx + v_own) = to4<E>(acc);
      lds_barrier();
      // S <- exp(G_last) S + (K exp(G_last - G))^T v_new
      const X8 b0 = ld8(Vx + v_in), b1 = ld8(Vx + v_in + 32);
      const X4 v_out = ld4(Vx + v_row);
      const int next = (s + 1) % SCAN_DEPTH;
      g_now = __expf(gl[next]);
      take_w(flight, next);
      u = tile_exchange(fu[next], from);
#pragma unroll
      for (int m = 0; m < 2; ++m) S[m] = mfma(fk[s][m][0], b0, S[m]);
#pragma unroll
      for (int m = 0; m < 2; ++m) S[m] = mfma(fk[s][m][1], b1, S[m]);
      if constexpr (decltype(more)::value) issue_w(s, s);
      buf_st8(vb.buffer(s), vn_off, vb.offset(s), v_out);
      st8(Sx + s_own, pack_permv<E>(S[0], S[1]));
      lds_barrier();
    };
    // SCAN_DEPTH steps a round, so that the operand ring's registers are named by constants
    auto round = [&](int tau, auto flight) __attribute__((always_inline)) {
      tab.advance(tau + SCAN_DEPTH);
      step(Int<0>(), Int<1>(), flight);
      step(Int<1>(), Int<1>(), flight);
      step(Int<2>(), Int<1>(), flight);
      step(Int<3>(), Int<1>(), flight);
      ub.advance();
      kb.advance();
      vb.advance();
      hb.advance();
    };
    int tau = 0;
    if (n >= SCAN_DEPTH) {
      // its first step's next -W has two more slots' loads after it and this step's store
      round(0, Int<2 * FWD_LOAD_OPS + 1>());
      for (tau = SCAN_DEPTH; tau + SCAN_DEPTH <= n; tau += SCAN_DEPTH) round(tau, Int<2 * FWD_STEP_OPS + 5>());
    }
    // the last steps issue their two stores only (and n < SCAN_DEPTH never issued more than the first loads)
    if (tau < n) step(Int<0>(), Int<0>(), Int<2 * FWD_LOAD_OPS + 1>());
    if (tau + 1 < n) step(Int<1>(), Int<0>(), Int<FWD_LOAD_OPS + 3>());
    if (tau + 2 < n) step(Int<2>(), Int<0>(), Int<5>());
  }
  if (final_state) {
    float* sf = final_state + ((size_t)d * H + h) * D * D;
    const float inv = 1.f / vs;  // exact: vs is a power of two
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) sf[(32 * wave + 16 * m + 4 * q4 + i) * D + v0 + r] = S[m][i] * inv;
  }
}

// ---------------------------------------------------------------------------
// fwd_out: O^T (v rows, t columns) per chunk and head.  h^T and v_new^T come in by row
// pieces (operand_from_rows) and O leaves as whole rows: H = 16, 144 / 520 / 36 / 5 chunks
// 44.3 -> 41.7 / 152 -> 144 / 16.2 -> 15.2 / 7.1 -> 7.2 us in a step's kernel trace, against
// fragments read and O stored with lanes on 16 different rows.  Bound by HBM on the long ones:
// 228 MB at 5.5 TB/s, some of it from the memory-side cache (a large copy reaches 5.2).
// ---------------------------------------------------------------------------
template <class I, class E>  // I: element type of q, k and o; E: operand type (as fwd_prep)
__global__ __launch_bounds__(256) void fwd_out_kernel(
    const I* __restrict__ q, const I* __restrict__ k, int normalize,
    const float* __restrict__ rk, const float* __restrict__ gc, const E* __restrict__ hT,
    const E* __restrict__ vnT, const int32_t* __restrict__ chunks, int H,
    float scale, const float* __restrict__ vscale, I* __restrict__ o) {
  typedef typename Vec<E>::x8 X8;
  // grid (H, NC), chunks last to first: the state scan wrote the last chunks
  // last, so they are the likeliest still in the memory-side cache
  const HeadChunk hc = xcd_head_chunk(gridDim.x, gridDim.y);  // all heads of a chunk on one XCD
  const int h = hc.h, c = gridDim.y - 1 - hc.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q4 = lane >> 4;
  const ChunkInfo ci = chunk_info(chunks, c);
  const size_t cb = (size_t)c * H + h;

  __shared__ __attribute__((aligned(16))) E Qs[64 * LDK];
  __shared__ __attribute__((aligned(16))) E Ks[64 * LDK];
  __shared__ __attribute__((aligned(16))) E Ps[64 * LDT];  // P[t][s], causal, gated
  __shared__ float Gs[64];

  const E* ht = hT + cb * (D * D);
  const E* vt = vnT + cb * (D * CH);
  // requested with the inputs, by quads: rows v = 16 (2 wave + mm) .. of v_new^T (t block
  // kb) and of h^T (k block kb)
  X8 av[2][2], ah[2][4];
#pragma unroll
  for (int mm = 0; mm < 2; ++mm) {
    const int v = 16 * (2 * wave + mm) + (lane >> 2);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) av[mm][kb] = row_piece(vt, CH, v, 32 * kb);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) ah[mm][kb] = row_piece(ht, D, v, 32 * kb);
  }
  {
    const int t = tid >> 2, p = tid & 3;
    const bool in = t < ci.len;
    const size_t ev = (size_t)(ci.start + clamp_row(t, ci.len)) * H + h, row = ev * D;
    const float rkt = rk[ev];
    typename Vec<I>::x8 xq[4], xk[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * j + 8 * p;
      xq[j] = ld8(q + row + col);
      xk[j] = ld8(k + row + col);
    }
    if (p == 0) Gs[t] = gc[ev];
    const float rqt = normalize ? row_rnorm(xq) : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = 32 * j + 8 * p;
      st8(Qs + t * LDK + col, keep_if(in, scaled8<E>(xq[j], rqt)));
      st8(Ks + t * LDK + col, keep_if(in, scaled8<E>(xk[j], rkt)));
    }
  }
  // to the operands' layout through the place of P
#pragma unroll
  for (int mm = 0; mm < 2; ++mm) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) av[mm][kb] = operand_from_rows(Ps + 1024 * wave + 512 * (kb & 1), av[mm][kb]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) ah[mm][kb] = operand_from_rows(Ps + 1024 * wave + 512 * (kb & 1), ah[mm][kb]);
  }
  __syncthreads();

  // P^T tiles: s-tile a = wave, t-tiles b >= a
  {
    const int a = wave;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f32x4 acc = zero4();
      if (b >= a) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
          acc = mfma(ld8(Ks + (16 * a + r) * LDK + 32 * kb + 8 * q4), ld8(Qs + (16 * b + r) * LDK + 32 * kb + 8 * q4),
                     acc);
        const int t = 16 * b + r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = 16 * a + 4 * q4 + i;
          acc[i] = (s <= t) ? acc[i] * __expf(Gs[t] - Gs[s]) : 0.f;
        }
      }
      st4(Ps + (16 * b + r) * LDT + 16 * a + 4 * q4, acc);
    }
  }
  __syncthreads();

  // O^T = (h^T Qn^T) * gam_t + Vn^T P^T ; wave owns value tiles 2w, 2w+1
  f32x4 acc[2][4];
#pragma unroll
  for (int mm = 0; mm < 2; ++mm)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[mm][n] = zero4();
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    X8 bq[4];
#pragma unroll
    for (int n = 0; n < 4; ++n) bq[n] = ld8(Qs + (16 * n + r) * LDK + 32 * kb + 8 * q4);
#pragma unroll
    for (int mm = 0; mm < 2; ++mm)
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[mm][n] = mfma(ah[mm][kb], bq[n], acc[mm][n]);
  }
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const float gam = __expf(Gs[16 * n + r]);
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) acc[mm][n] *= gam;
  }
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      if (n < 2 * kb) continue;  // t-tile n holds no s in this block (s > t)
      const X8 b = ld8(Ps + (16 * n + r) * LDT + 32 * kb + 8 * q4);
#pragma unroll
      for (int mm = 0; mm < 2; ++mm) acc[mm][n] = mfma(av[mm][kb], b, acc[mm][n]);
    }
  }
  const float osc = vscale ? scale / *vscale : scale;  // undo the power-of-two scale of V
  // O leaves as whole rows, through the Q rows' place
  static_assert(sizeof(I) == sizeof(E), "O rows fit the Q rows");
  I* Os = reinterpret_cast<I*>(Qs);
  lds_barrier();
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) st4(Os + (16 * n + r) * LDK + 16 * (2 * wave + mm) + 4 * q4, acc[mm][n] * osc);
  lds_barrier();
  const __amdgpu_buffer_rsrc_t o_rs = chunk_rows_rsrc(o, ci.start, ci.len, H, h);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    buf_st16(o_rs, (tid >> 2) * H * D * 2 + 64 * j + 16 * (tid & 3), ld8(Os + (tid >> 2) * LDK + 32 * j + 8 * (tid & 3)));
}

// ---------------------------------------------------------------------------
// Power-of-two scale of V for the fp16 forwards.  The recurrence is linear in
// (V, initial state): scaling both by vs scales W-free quantities (U, v_new,
// every state, O) by vs exactly, so the kernels carry them scaled and divide O
// and the final state by vs.  vs brings max(|V|, |S0|) into [2^(t-1), 2^t):
// t = 6 for inference, far inside fp16's range (65504) for U, v_new and the
// state; t = 3 for training, where the backward multiplies V-scaled by
// dO-scaled quantities (dP, dW) and keeps their products in fp16 too.  The same
// kernels give the backward's scale of dO (launch_range_partials, then bwd_local).
// ---------------------------------------------------------------------------
constexpr int VS_BLOCKS = kVscaleBlocks;

__device__ __forceinline__ float block_max(float m, float* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

template <class I>
__global__ __launch_bounds__(256) void vscale_partial_kernel(const I* __restrict__ v, size_t nv8,
                                                             const float* __restrict__ s0, size_t ns,
                                                             float* __restrict__ part) {
  __shared__ float red[4];
  float m = 0.f;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  // eight 16-byte loads in flight per thread: one at a time, the loop waits out a
  // memory round trip per load and reads at about a quarter of HBM's rate
  // (the last round's loads past the end are skipped lane by lane, all in one round trip)
  constexpr int U = 8;
  for (; i < nv8; i += U * stride) {
    typename Vec<I>::x8 x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = i + u * stride < nv8 ? ld8(v + 8 * (i + u * stride)) : zero8v<I>();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const f32x8 f = cvtf8(x[u]);
#pragma unroll
      for (int s = 0; s < 8; ++s) m = fmaxf(m, fabsf(f[s]));
    }
  }
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < ns; i += stride) m = fmaxf(m, fabsf(s0[i]));
  m = block_max(m, red);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
template <class I, class E>
static hipError_t launch_fwd_t(const FwdArgs& a, float* vscale, int vs_target, hipStream_t stream) {
  E* ws[F_COUNT];
  for (int i = 0; i < F_COUNT; ++i) ws[i] = reinterpret_cast<E*>(a.ws + a.off[i]);
  float* rk = reinterpret_cast<float*>(ws[F_RK]);
  float* gcum = reinterpret_cast<float*>(ws[F_GC]);
  const I* q = static_cast<const I*>(a.q);
  const I* k = static_cast<const I*>(a.k);
  const I* v = static_cast<const I*>(a.v);
  {
    TimedLaunch tl(K_FWD_PREP, stream);
    const dim3 grid_p(a.H, a.n_chunks);
    if (a.normalize)
      hipLaunchKernelGGL((fwd_prep_kernel<I, E, true>), grid_p, dim3(256), 0, stream, k, v, a.g, a.beta,
                         a.chunks, a.H, vscale, vs_target, rk, gcum, ws[F_TM], ws[F_W],
                         ws[F_UT], ws[F_KGT]);
    else
      hipLaunchKernelGGL((fwd_prep_kernel<I, E, false>), grid_p, dim3(256), 0, stream, k, v, a.g, a.beta,
                         a.chunks, a.H, vscale, vs_target, rk, gcum, ws[F_TM], ws[F_W],
                         ws[F_UT], ws[F_KGT]);
  }
  const dim3 grid_s(a.H * (D / 16), a.n_docs);
  hipStream_t ss = stream;
  if (a.scan_stream) {
    if (const hipError_t e = hipEventRecord(a.scan_fork, stream)) return e;
    if (const hipError_t e = hipStreamWaitEvent(a.scan_stream, a.scan_fork, 0)) return e;
    ss = a.scan_stream;
  }
  {
    TimedLaunch tl(K_FWD_SCAN, ss);
    const auto kernel = scan_wide(a.H) ? fwd_scan_kernel<E, true> : fwd_scan_kernel<E, false>;
    hipLaunchKernelGGL(kernel, grid_s, dim3(SCAN_THREADS), a.scan_stream ? FWD_ALONE_LDS : 0, ss, ws[F_W], ws[F_UT], ws[F_KGT], gcum,
                       a.chunks, a.doc_chunk, a.H, vscale, a.initial_state, a.final_state, ws[F_HT], ws[F_VNT]);
  }
  if (a.scan_stream)
    if (const hipError_t e = hipEventRecord(a.scan_join, a.scan_stream)) return e;
  if (a.no_output) return hipSuccess;
  TimedLaunch tl(K_FWD_OUT, stream);
  hipLaunchKernelGGL((fwd_out_kernel<I, E>), dim3(a.H, a.n_chunks), dim3(256), 0, stream, q, k, (int)a.normalize, rk, gcum,
                     ws[F_HT], ws[F_VNT], a.chunks, a.H, a.scale, vscale, static_cast<I*>(a.o));
  return hipSuccess;
}

void launch_range_partials(const void* x, bool fp16, size_t n8, const float* s0, size_t ns, float* out,
                           hipStream_t stream) {
  static_assert(VS_BLOCKS == 4 * 256, "range_partial4 takes four partials per thread of a 256-thread workgroup");
  if (fp16)
    hipLaunchKernelGGL(vscale_partial_kernel<f16>, dim3(VS_BLOCKS), dim3(256), 0, stream,
                       static_cast<const f16*>(x), n8, s0, ns, out + 1);
  else
    hipLaunchKernelGGL(vscale_partial_kernel<bf16>, dim3(VS_BLOCKS), dim3(256), 0, stream,
                       static_cast<const bf16*>(x), n8, s0, ns, out + 1);
}

hipError_t launch_fwd(const FwdArgs& a, hipStream_t stream) {
  if (!a.precise && !a.fp16) return launch_fwd_t<bf16, bf16>(a, nullptr, 0, stream);
  float* vsc = reinterpret_cast<float*>(a.ws + a.off[F_VSC]);
  const size_t nv8 = (size_t)a.T * a.H * (D / 8);
  const size_t ns = a.initial_state ? (size_t)a.n_docs * a.H * D * D : 0;
  launch_range_partials(a.v, a.fp16, nv8, a.initial_state, ns, vsc, stream);
  const int target = a.training ? kVscaleTargetTraining : kVscaleTarget;
  return a.fp16 ? launch_fwd_t<f16, f16>(a, vsc, target, stream) : launch_fwd_t<bf16, f16>(a, vsc, target, stream);
}

}  // namespace cqgdn
