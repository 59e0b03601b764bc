// Kernels of the widths without a compile-time instance (33 to kMaxBlockW = 128), and of what the
// vectorised kernels do not address at the widths below (fp64 x, one channel, batch slabs past
// 32-bit offsets). One lane owns one channel; a workgroup of kBlkNW waves walks a segment of rows of
// 64 channels in steps of kBlkStep rows, 16 rows to a wave.
//
// What bounds them is the arithmetic: W multiply-adds per element in the forward and 3 W in the
// backward. A lane therefore holds 16 output rows (or 16 dweight taps) in registers and takes 16
// taps (or rows) at a time against a register window of 32 rows: 256 multiply-adds for 32 LDS reads.
// The rows (x, and in the backward g) sit in LDS rings of 16-row blocks that move on with the walk,
// so each is read from memory once per segment plus the window, and the weights once per segment.
// The rows of the next step are requested before a step is computed.
//
// Measured against one lane walking one row at a time with weights, x, g and the dweight sums in LDS
// (four LDS accesses per tap; the kernels these replaced): B=2 T=4096 D=1024 W=64 bf16 fwd+bwd 5012
// -> 138 us, forward alone 657 -> 36; with the segments of generic_tiling 30.
//
// Rows are numbered in taps of the padded window: with Pp = W - 1 rounded up to whole blocks, tap
// k sits at position k + (Pp - P), so that every block of 16 positions meets whole row blocks. The
// arithmetic per value and its order (w[P] first, then k = 0 .. P-1, the bias last) are those of
// causal_conv1d.py:129-138 and :290-302.
#pragma once

#include "ccv1d_generic.h"

namespace ccv1d {

// 16 rows of one channel from a ring of NB blocks, the `i`-th block from slot `slot`.
template <typename E>
__device__ __forceinline__ void ring_block(const E* ring, int NB, int slot, int i, int lane,
                                           float (&v)[kBlk]) {
  int s = slot + i;
  s = s >= NB ? s - NB : s;
  const E* p = ring + s * (kBlk * 64) + lane;
#pragma unroll
  for (int r = 0; r < kBlk; ++r) v[r] = static_cast<float>(p[r * 64]);
}

// acc[r] += w[tap(q)] * (row r + q of lo:hi) for the positions q in [first, last] of a block of 16;
// wk points at position 0's weight, `dir` weights apart per position (65: ascending taps).
template <int DIR>
__device__ __forceinline__ void block_taps(const float* wk, int first, int last,
                                           const float (&lo)[kBlk], const float (&hi)[kBlk],
                                           float (&acc)[kBlk]) {
#pragma unroll
  for (int q = 0; q < kBlk; ++q) {
    if (q < first || q > last) continue;
    const float w = wk[q * DIR];
#pragma unroll
    for (int r = 0; r < kBlk; ++r)
      acc[r] = fmaf(w, q + r < kBlk ? lo[q + r < kBlk ? q + r : 0] : hi[q + r < kBlk ? 0 : q + r - kBlk],
                    acc[r]);
  }
}

// Pre-activations (without the bias) of the 16 rows whose window starts at block `slot` of the ring.
template <typename E>
__device__ __forceinline__ void block_conv(const float* wl, const E* ring, int NB, int slot, int W,
                                           int lane, float (&z)[kBlk]) {
  const int P = W - 1, NC = blk_window(W) / kBlk, sh = blk_window(W) - P;
  const float* wk = wl + lane - sh * kBlkWPitch;  // position q: tap q - sh
  float a[kBlk], b[kBlk];
  ring_block(ring, NB, slot, NC, lane, a);
  const float wp = wl[P * kBlkWPitch + lane];
#pragma unroll
  for (int r = 0; r < kBlk; ++r) z[r] = wp * a[r];
  ring_block(ring, NB, slot, 0, lane, a);
  ring_block(ring, NB, slot, 1, lane, b);
  block_taps<kBlkWPitch>(wk, sh, kBlk - 1, a, b, z);
#pragma unroll 1
  for (int c = 1; c < NC; c += 2) {
    ring_block(ring, NB, slot, c + 1, lane, a);
    block_taps<kBlkWPitch>(wk + c * kBlk * kBlkWPitch, 0, kBlk - 1, b, a, z);
    if (c + 1 < NC) {
      ring_block(ring, NB, slot, c + 2, lane, b);
      block_taps<kBlkWPitch>(wk + (c + 1) * kBlk * kBlkWPitch, 0, kBlk - 1, a, b, z);
    }
  }
}

// dx (without dfinal) of the 16 rows at block `slot` of the g ring: w[P] g[u] + sum_j w[P-j] g[u+j].
__device__ __forceinline__ void block_dx(const float* wl, const float* ring, int NB, int slot, int W,
                                         int lane, float (&dx)[kBlk]) {
  const int P = W - 1, NC = P / kBlk + 1;
  const float* wk = wl + P * kBlkWPitch + lane;  // position j: tap P - j
  float a[kBlk], b[kBlk];
  ring_block(ring, NB, slot, 0, lane, a);
  ring_block(ring, NB, slot, 1, lane, b);
  const float wp = wk[0];
#pragma unroll
  for (int r = 0; r < kBlk; ++r) dx[r] = wp * a[r];
  block_taps<-kBlkWPitch>(wk, 1, NC == 1 ? P : kBlk - 1, a, b, dx);
#pragma unroll 1
  for (int c = 1; c < NC; ++c) {
    // The last block's rows past its last tap are not used (its second half need not be written yet).
#pragma unroll
    for (int r = 0; r < kBlk; ++r) a[r] = b[r];
    ring_block(ring, NB, slot, c + 1, lane, b);
    const float* wc = wk - c * kBlk * kBlkWPitch;
    if (c + 1 < NC) block_taps<-kBlkWPitch>(wc, 0, kBlk - 1, a, b, dx);
    else block_taps<-kBlkWPitch>(wc, 0, P - c * kBlk, a, b, dx);
  }
}

// Ring row of the row `d` rows after the start of block `slot`.
__device__ __forceinline__ int ring_row(int NB, int slot, int d) {
  const int r = slot * kBlk + d;
  return r >= NB * kBlk ? r - NB * kBlk : r;
}

// Whether the rows d0 .. d1-1 after the start of block `slot` (d1 - d0 <= 192) carry one sequence id.
__device__ __forceinline__ bool ring_one_id(const int32_t* sid, int NB, int slot, int d0, int d1,
                                            int lane) {
  const int32_t id0 = sid[ring_row(NB, slot, d0)];
  bool ok = true;
#pragma unroll
  for (int h = 0; h < 3; ++h) {
    const int d = d0 + h * 64 + lane;
    ok = ok && (d >= d1 || sid[ring_row(NB, slot, d < d1 ? d : d0)] == id0);
  }
  return __all(ok);
}

// The weights of 64 channels from c0 in LDS, tap k of channel c at [k][c - c0]. The 64 * W weights
// are read in memory order, so neighbouring threads write different taps of one channel: with 65
// floats per tap they meet different banks.
// A thread requests 8 of them at a time (one load and its use at a time cost a memory round trip each,
// 16 of them at W = 64: forward alone B=2 T=4096 D=1024 W=64 36.2
// -> 33.9 us).
__device__ __forceinline__ void stage_weights(const void* w, int w_dt, int c0, int D, int W,
                                              float* wl) {
  constexpr int N = 8, NT = kBlkNW * 64;
  const int n = min(64, D - c0) * W;
  const int dc = NT / W, dk = NT - dc * W;  // NT weights further on: dc channels and dk taps
  int c = threadIdx.x / W, k = threadIdx.x - c * W;
  auto each = [&](auto* q) {
    q += (int64_t)c0 * W;
#pragma unroll 1
    for (int i = threadIdx.x; i < n; i += N * NT) {
      float v[N];
#pragma unroll
      for (int u = 0; u < N; ++u) v[u] = static_cast<float>(q[min(i + u * NT, n - 1)]);
#pragma unroll
      for (int u = 0; u < N; ++u) {
        if (i + u * NT < n) wl[k * kBlkWPitch + c] = v[u];
        k += dk;
        c += dc;
        if (k >= W) {
          k -= W;
          ++c;
        }
      }
    }
  };
  switch (w_dt) {
    case DT_F32: each(static_cast<const float*>(w)); break;
    case DT_F16: each(static_cast<const _Float16*>(w)); break;
    case DT_BF16: each(static_cast<const __bf16*>(w)); break;
    default: each(static_cast<const double*>(w)); break;
  }
}

// One channel of concat(initial_states, x): rows -P .. -1 from the states (or zero), rows past the
// end repeat the last one (their values are never used), rows before -P are zero (never used).
template <typename TX, typename E>
struct BlkRows {
  GenRow<TX> xx;
  int T;
  __device__ __forceinline__ void load(int row0, E (&v)[kBlk]) const {
    if (row0 >= 0) {
#pragma unroll
      for (int r = 0; r < kBlk; ++r)
        v[r] = static_cast<E>(xx.xb[(int64_t)min(row0 + r, T - 1) * xx.s_xt]);
    } else {
#pragma unroll
      for (int r = 0; r < kBlk; ++r) {
        const int row = row0 + r;
        v[r] = row < -xx.P ? static_cast<E>(0.0f) : static_cast<E>(xx(min(row, T - 1)));
      }
    }
  }
};

template <typename TX, typename P>
__device__ __forceinline__ GenRow<TX> gen_rows(const P& p, int b, int c) {
  GenRow<TX> xx;
  xx.xb = static_cast<const TX*>(p.x) + (int64_t)b * p.s_xb + c;
  xx.s_xt = p.s_xt;
  xx.P = p.W - 1;
  xx.D = p.D;
  xx.i_dt = p.i_dt;
  xx.initb = p.has_init ? static_cast<const char*>(p.init) +
                              ((int64_t)b * xx.P * p.D + c) * dt_size(p.i_dt)
                        : nullptr;
  return xx;
}

// E: the LDS element of x, TX itself for 16-bit x, else float (also for 16-bit x whose initial states
// have another type, which need not be exact in TX).
template <typename TX, typename E>
__global__ __launch_bounds__(kBlkNW * 64, 2) void fwd_block_kernel(const FwdParams p) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int T = p.T, D = p.D, W = p.W, P = W - 1;
  const int Pp = blk_window(W), NC = Pp / kBlk, NB = blk_ring(W);
  const int tile = blockIdx.x % p.tl.nT;
  const int b = blockIdx.x / p.tl.nT;
  const int c0 = blockIdx.y * 64;
  const bool active = c0 + lane < D;
  const int c = min(c0 + lane, D - 1);  // lanes past the last channel compute it again, unstored
  const int t0 = tile * p.tl.L;
  const int t1 = min(t0 + p.tl.L, T);
  float* wl = lds;
  int32_t* sid = reinterpret_cast<int32_t*>(wl + W * kBlkWPitch);
  E* xr = reinterpret_cast<E*>(sid + NB * kBlk);
  const int32_t* sb = p.seq ? p.seq + (int64_t)b * T : nullptr;
  const BlkRows<TX, E> rows{gen_rows<TX>(p, b, c), T};
  const float bias = p.has_bias ? ld_any(p.bias, c, p.b_dt) : 0.0f;
  TX* ob = static_cast<TX*>(p.out) + (int64_t)b * T * D + c;

  auto put = [&](int slot, int row0, const E (&v)[kBlk]) {
    E* q = xr + slot * (kBlk * 64) + lane;
#pragma unroll
    for (int r = 0; r < kBlk; ++r) q[r * 64] = v[r];
    if (sb && lane < kBlk) sid[slot * kBlk + lane] = seq_at(sb, row0 + lane, T, p.has_init);
  };

  E nxt[kBlk];
  rows.load(t0 + wave * kBlk, nxt);
  for (int i = wave; i < NC; i += kBlkNW) {
    E v[kBlk];
    rows.load(t0 - Pp + i * kBlk, v);
    put(i, t0 - Pp + i * kBlk, v);
  }
  stage_weights(p.w, p.w_dt, c0, D, W, wl);

  // Slot of the block Pp rows before this wave's block, which the next NC blocks follow.
  int slot = wave >= NB ? wave - NB : wave;
  for (int a = t0; a < t1; a += kBlkStep) {
    const int r0 = a + wave * kBlk;
    int own = slot + NC;
    own = own >= NB ? own - NB : own;
    put(own, r0, nxt);
    lds_barrier();
    if (a + kBlkStep < t1) rows.load(r0 + kBlkStep, nxt);
    if (r0 < t1) {
      float z[kBlk];
      // Rows of one sequence (the window's included): every mask is 1.
      if (!sb || ring_one_id(sid, NB, slot, Pp - P, Pp + kBlk, lane)) {
        block_conv(wl, xr, NB, slot, W, lane, z);
      } else {
#pragma unroll
        for (int r = 0; r < kBlk; ++r) {
          const int32_t st = sid[ring_row(NB, slot, Pp + r)];
          float v = wl[P * kBlkWPitch + lane] *
                    static_cast<float>(xr[ring_row(NB, slot, Pp + r) * 64 + lane]);
          for (int k = 0; k < P; ++k) {
            const int q = ring_row(NB, slot, Pp + r - P + k);
            if (sid[q] == st) v = fmaf(wl[k * kBlkWPitch + lane], static_cast<float>(xr[q * 64 + lane]), v);
          }
          z[r] = v;
        }
      }
#pragma unroll
      for (int r = 0; r < kBlk; ++r) {
        float v = z[r];
        if (p.has_bias) v += bias;
        if (sb && sid[ring_row(NB, slot, Pp + r)] < 0) v = 0.0f;
        if (p.silu) v = v * sigmoid_f(v);
        if (active && r0 + r < t1) ob[(int64_t)(r0 + r) * D] = to_store<TX>(v);
      }
    }
    lds_barrier();  // the step's oldest blocks are overwritten next
    slot += kBlkNW;
    slot = slot >= NB ? slot - NB : slot;
  }
  if (p.has_final && t1 == T && active) {
    TX* fb = static_cast<TX*>(p.fin) + (int64_t)b * P * D + c;
    for (int q = wave; q < P; q += kBlkNW) fb[(int64_t)q * D] = to_store<TX>(rows.xx(T - P + q));
  }
}

// Backward. Step by step the workgroup forms g = dout * silu'(z) of 64 new rows (rows past the
// segment too, as far as its last dx rows reach) and completes dx of the 64 rows Pp before them;
// dweight's taps are shared out among the waves in blocks of 16, each wave taking its blocks over
// all of a step's rows; tap P and dbias belong to the wave of the row. A step's sums start from zero
// and are added to the segment's, which become the partial row b * nT + tile.
template <typename TX, typename E>
__global__ __launch_bounds__(kBlkNW * 64, 2) void bwd_block_kernel(const BwdParams p) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int T = p.T, D = p.D, W = p.W, P = W - 1;
  const int Pp = blk_window(W), NC = Pp / kBlk, NB = blk_ring(W);
  const int tile = blockIdx.x % p.tl.nT;
  const int b = blockIdx.x / p.tl.nT;
  const int c0 = blockIdx.y * 64;
  const bool active = c0 + lane < D;
  const int c = min(c0 + lane, D - 1);
  const int t0 = tile * p.tl.L;
  const int own_end = min(t0 + p.tl.L, T);
  const int emit_lo = (tile == 0 && p.need_dinit) ? -P : t0;
  float* wl = lds;
  float* gr = wl + W * kBlkWPitch;
  int32_t* sid = reinterpret_cast<int32_t*>(gr + NB * kBlk * 64);
  E* xr = reinterpret_cast<E*>(sid + NB * kBlk);
  const int32_t* sb = p.seq ? p.seq + (int64_t)b * T : nullptr;
  const BlkRows<TX, E> rows{gen_rows<TX>(p, b, c), T};
  const float bias = p.has_bias ? ld_any(p.bias, c, p.b_dt) : 0.0f;
  const TX* yb = static_cast<const TX*>(p.dy) + (int64_t)b * p.s_yb + c;
  TX* dxb = static_cast<TX*>(p.dx) + (int64_t)b * p.s_dxb + c;
  const int isz = dt_size(p.i_dt);
  void* dinitb =
      p.need_dinit ? static_cast<char*>(p.dinit) + ((int64_t)b * P * D + c) * isz : nullptr;
  const TX* dfb = p.has_dfinal ? static_cast<const TX*>(p.dfin) + (int64_t)b * P * D + c : nullptr;

  auto put = [&](int slot, int row0, const E (&v)[kBlk]) {
    E* q = xr + slot * (kBlk * 64) + lane;
#pragma unroll
    for (int r = 0; r < kBlk; ++r) q[r * 64] = v[r];
    if (sb && lane < kBlk) sid[slot * kBlk + lane] = seq_at(sb, row0 + lane, T, p.has_init);
  };
  E nx[kBlk];
  TX ny[kBlk];
  auto load = [&](int row0) {
    rows.load(row0, nx);
#pragma unroll
    for (int r = 0; r < kBlk; ++r) ny[r] = yb[(int64_t)min(row0 + r, T - 1) * p.s_yt];
  };
  load(t0 + wave * kBlk);
  for (int i = wave; i < NC; i += kBlkNW) {
    E v[kBlk];
    rows.load(t0 - Pp + i * kBlk, v);
    put(i, t0 - Pp + i * kBlk, v);
    // Rows before the segment: their g belongs to the previous one (or is 0 before row 0).
#pragma unroll
    for (int r = 0; r < kBlk; ++r) gr[(i * kBlk + r) * 64 + lane] = 0.0f;
  }
  stage_weights(p.w, p.w_dt, c0, D, W, wl);

  // dweight sums of this wave's tap blocks (position block wave, wave + 4), of tap P and of dbias.
  constexpr int NOWN = (blk_window(kMaxBlockW) / kBlk + kBlkNW - 1) / kBlkNW;
  float dw[NOWN][kBlk];
#pragma unroll
  for (int n = 0; n < NOWN; ++n)
#pragma unroll
    for (int q = 0; q < kBlk; ++q) dw[n][q] = 0.0f;
  float dwp = 0.0f, db = 0.0f;
  // fp64 x comes here at every width: where the taps are one block, the waves share out the rows
  // instead, and positions before the first tap are left out (fwd+bwd B=8 T=4096 D=1024 W=2 404 -> 374
  // us, W=4 407 -> 378, W=16 436 -> 417).
  const bool by_rows = sizeof(TX) == 8 && NC == 1;
  static_assert(2 * kBlkNW * 64 + kBlkNW * kBlk * 64 <= blk_ring(2) * kBlk * 64, "sums in the g ring");

  int base = 0;  // slot of the block Pp rows before the step's first
  for (int a = t0; a - Pp < own_end; a += kBlkStep) {
    const int r0 = a + wave * kBlk;
    int slot = base + wave;
    slot = slot >= NB ? slot - NB : slot;
    int own = slot + NC;
    own = own >= NB ? own - NB : own;
    E cx[kBlk];
    TX cy[kBlk];
#pragma unroll
    for (int r = 0; r < kBlk; ++r) {
      cx[r] = nx[r];
      cy[r] = ny[r];
    }
    put(own, r0, cx);
    lds_barrier();
    if (a + kBlkStep - Pp < own_end) load(r0 + kBlkStep);

    float g[kBlk];
    if (r0 < T) {
      if (p.silu) {
        float z[kBlk];
        if (!sb || ring_one_id(sid, NB, slot, Pp - P, Pp + kBlk, lane)) {
          block_conv(wl, xr, NB, slot, W, lane, z);
        } else {
#pragma unroll
          for (int r = 0; r < kBlk; ++r) {
            const int32_t st = sid[ring_row(NB, slot, Pp + r)];
            float v = wl[P * kBlkWPitch + lane] *
                      static_cast<float>(xr[ring_row(NB, slot, Pp + r) * 64 + lane]);
            for (int k = 0; k < P; ++k) {
              const int q = ring_row(NB, slot, Pp + r - P + k);
              if (sid[q] == st)
                v = fmaf(wl[k * kBlkWPitch + lane], static_cast<float>(xr[q * 64 + lane]), v);
            }
            z[r] = v;
          }
        }
#pragma unroll
        for (int r = 0; r < kBlk; ++r) {
          if (p.has_bias) z[r] += bias;
          g[r] = dsilu_times(static_cast<float>(cy[r]), z[r]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < kBlk; ++r) g[r] = static_cast<float>(cy[r]);
      }
      float sw = 0.0f, sd = 0.0f;
#pragma unroll
      for (int r = 0; r < kBlk; ++r) {
        if (r0 + r >= T || (sb && sid[ring_row(NB, slot, Pp + r)] < 0)) g[r] = 0.0f;
        if (r0 + r < own_end) {
          sw = fmaf(g[r], static_cast<float>(cx[r]), sw);
          sd += g[r];
        }
      }
      dwp += sw;
      db += sd;
    } else {
#pragma unroll
      for (int r = 0; r < kBlk; ++r) g[r] = 0.0f;
    }
    {
      float* q = gr + own * (kBlk * 64) + lane;
#pragma unroll
      for (int r = 0; r < kBlk; ++r) q[r * 64] = g[r];
    }
    lds_barrier();

    // dx of the rows Pp before this wave's.
    const int u0 = r0 - Pp;
    if (u0 + kBlk > emit_lo && u0 < own_end) {
      float dx[kBlk];
      if (!sb || ring_one_id(sid, NB, slot, 0, kBlk + P, lane)) {
        block_dx(wl, gr, NB, slot, W, lane, dx);
      } else {
#pragma unroll
        for (int r = 0; r < kBlk; ++r) {
          const int32_t q0 = sid[ring_row(NB, slot, r)];
          float v = wl[P * kBlkWPitch + lane] * gr[ring_row(NB, slot, r) * 64 + lane];
          for (int j = 1; j <= P; ++j) {
            const int q = ring_row(NB, slot, r + j);
            if (sid[q] == q0) v = fmaf(wl[(P - j) * kBlkWPitch + lane], gr[q * 64 + lane], v);
          }
          dx[r] = v;
        }
      }
#pragma unroll
      for (int r = 0; r < kBlk; ++r) {
        const int row = u0 + r;
        if (row < emit_lo || row >= own_end || !active) continue;
        float v = dx[r];
        if (dfb) {
          const int f = row - (T - P);
          if (f >= 0 && f < P) v += static_cast<float>(dfb[(int64_t)f * D]);
        }
        if (row >= 0) dxb[(int64_t)row * p.s_dxt] = to_store<TX>(v);
        else st_any(dinitb, (int64_t)(row + P) * D, p.i_dt, v);
      }
    }

    // dweight of this wave's tap blocks over the step's own rows.
    if (a < own_end) {
      const bool one = !sb || ring_one_id(sid, NB, base, Pp - P, Pp + kBlkStep, lane);
#pragma unroll
      for (int n = 0; n < NOWN; ++n) {
        const int cb = by_rows ? n : wave + n * kBlkNW;
        if (cb >= NC) continue;
        float acc[kBlk];
#pragma unroll
        for (int q = 0; q < kBlk; ++q) acc[q] = 0.0f;
#pragma unroll 1
        for (int i = by_rows ? wave : 0; i < (by_rows ? wave + 1 : kBlkNW); ++i) {
          const int rows_left = own_end - (a + i * kBlk);
          if (rows_left <= 0) break;
          float gv[kBlk], lo[kBlk], hi[kBlk];
          ring_block(gr, NB, base, NC + i, lane, gv);
          if (one) {
            ring_block(xr, NB, base, i + cb, lane, lo);
            ring_block(xr, NB, base, i + cb + 1, lane, hi);
            if (by_rows && rows_left >= kBlk) {
#pragma unroll
              for (int q = 0; q < kBlk; ++q) {
                if (q < Pp - P) continue;
#pragma unroll
                for (int r = 0; r < kBlk; ++r)
                  acc[q] = fmaf(gv[r], q + r < kBlk ? lo[q + r < kBlk ? q + r : 0]
                                                    : hi[q + r < kBlk ? 0 : q + r - kBlk], acc[q]);
              }
            } else if (rows_left >= kBlk) {
#pragma unroll
              for (int r = 0; r < kBlk; ++r)
#pragma unroll
                for (int q = 0; q < kBlk; ++q)
                  acc[q] = fmaf(gv[r], q + r < kBlk ? lo[q + r < kBlk ? q + r : 0]
                                                    : hi[q + r < kBlk ? 0 : q + r - kBlk], acc[q]);
            } else {
#pragma unroll
              for (int r = 0; r < kBlk; ++r) {
                if (r >= rows_left) continue;
#pragma unroll
                for (int q = 0; q < kBlk; ++q)
                  acc[q] = fmaf(gv[r], q + r < kBlk ? lo[q + r < kBlk ? q + r : 0]
                                                    : hi[q + r < kBlk ? 0 : q + r - kBlk], acc[q]);
              }
            }
          } else {
            for (int r = 0; r < min(rows_left, kBlk); ++r) {
              const int32_t st = sid[ring_row(NB, base, Pp + i * kBlk + r)];
              const float gt = gr[ring_row(NB, base, Pp + i * kBlk + r) * 64 + lane];
#pragma unroll
              for (int q = 0; q < kBlk; ++q) {
                const int xq = ring_row(NB, base, (i + cb) * kBlk + r + q);
                if (sid[xq] == st) acc[q] = fmaf(gt, static_cast<float>(xr[xq * 64 + lane]), acc[q]);
              }
            }
          }
        }
#pragma unroll
        for (int q = 0; q < kBlk; ++q) dw[n][q] += acc[q];
      }
    }
    lds_barrier();  // the step's oldest blocks are overwritten next
    base += kBlkNW;
    base = base >= NB ? base - NB : base;
  }

  // Tap P and dbias: the waves' sums in wave order (the LDS of the weights, and where they are few of
  // the g ring after them, is free now).
  wl[wave * 64 + lane] = dwp;
  wl[(kBlkNW + wave) * 64 + lane] = db;
  float* const waves = gr + 2 * kBlkNW * 64;  // [wave][position][64], by_rows
  if (by_rows) {
#pragma unroll
    for (int q = 0; q < kBlk; ++q) waves[(wave * kBlk + q) * 64 + lane] = dw[0][q];
  }
  lds_barrier();
  float* pp = p.part + ((int64_t)b * p.tl.nT + tile) * (W + 1) * D + c;
  if (!active) return;
  const int sh = Pp - P;
  if (by_rows) {
    for (int q = sh + wave; q < kBlk; q += kBlkNW) {
      float s = waves[q * 64 + lane];
#pragma unroll
      for (int v = 1; v < kBlkNW; ++v) s += waves[(v * kBlk + q) * 64 + lane];
      pp[(int64_t)(q - sh) * D] = s;
    }
  } else {
#pragma unroll
    for (int n = 0; n < NOWN; ++n)
#pragma unroll
      for (int q = 0; q < kBlk; ++q) {
        const int k = (wave + n * kBlkNW) * kBlk + q - sh;
        if (k >= 0 && k < P) pp[(int64_t)k * D] = dw[n][q];
      }
  }
  if (wave == 0 || (wave == 1 && p.has_bias)) {
    float s = wl[wave * kBlkNW * 64 + lane];
#pragma unroll
    for (int v = 1; v < kBlkNW; ++v) s += wl[(wave * kBlkNW + v) * 64 + lane];
    pp[(int64_t)(P + wave) * D] = s;
  }
}

}  // namespace ccv1d
