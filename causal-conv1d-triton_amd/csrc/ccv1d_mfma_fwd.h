// Forward with silu on the matrix cores, for bf16 x (widths 33 to kMaxBlockW = 128, no seq_idx): z of
// 256 rows of a channel as the product of ccv1d_mfma.h, three bf16 pieces of the fp32 weights times x.
//
// A workgroup takes 32 channels and walks a segment of rows in steps of 256 or 512. Rows are
// transposed in registers into per-channel LDS rows; a wave takes 4 of the channels and leaves out in x's place,
// which the thread that staged those rows reads back, transposes and stores. The weights are the
// products' left operand, so that a lane ends up with 4 consecutive rows (one 8-byte LDS write). A
// channel with infinities or NaN in reach is computed row by row, by its own values alone as in the
// backward. A row's sum is grouped by its place in its block of 16 rows from the call's first row on
// (segments are multiples of 16), whatever the segment: chunks cut elsewhere round about 1 value of
// out in 10^4 differently (so do calls under 16 rows, which mfma_pays may give to the block kernels).
//
// Measured, forward alone B=2 T=4096 D=1024 against fwd_block_kernel: W=33 21.8 -> 13.2 us, W=64
// 30.3 -> 14.8, W=128 47 -> 18.4 (memory: about 6). No unit is busy half of that at W=64 (LDS 5 us,
// vector instructions 3.3, matrix units 2; the waves wait 38 % of their time on memory and LDS and
// 35 % to issue). The weights' fragments start at any element, 5 words and 4 shifts each, so segments
// above 256 rows take steps of SUB = 2 and use each fragment twice (W=64 16.6 -> 14.8 us); below, half
// of such a step would be empty (B=1 T=512 W=64 6.6 us against 8.6). At width 32 the register-window
// kernel takes 14.2 us, at 24 11.0.
#pragma once

#include <type_traits>

#include "ccv1d_mfma.h"

namespace ccv1d {

// LDS layout for windows of NC blocks of 16 rows, in 16-bit elements as in MmShape, and
// steps of SUB x 256 rows.
template <int NC, int SUB>
struct MmFwdShape {
  static constexpr int ROWS = SUB * kMmRows;
  static constexpr int PP = MmShape<NC>::PP;
  static constexpr int KB = MmShape<NC>::KB;
  static constexpr int XP = MmShape<NC>::XP + (SUB - 1) * kMmRows;
  static constexpr int WL = MmShape<NC>::WL;
  static constexpr int WP = kMmCh * XP;
  static constexpr int FLAG = WP + kMmCh * 3 * WL;  // one word per wave
  static constexpr int BYTES = 2 * FLAG + 4 * kMmNW;
  static_assert(XP % 8 == 0 && WP % 8 == 0 && FLAG % 2 == 0 && PP <= kMmRows, "layout");
  static_assert(BYTES <= 80 * 1024, "two workgroups per CU");
};

// v as three bf16 pieces cut off one after the other: each has v's sign, none is larger than v, so the
// pieces of every finite v are finite. False if v is not.
__device__ __forceinline__ bool cut3(float v, uint16_t (&p)[3]) {
  float r = v;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const uint32_t h = __float_as_uint(r) & 0xffff0000u;
    p[i] = (uint16_t)(h >> 16);
    r -= __uint_as_float(h);
  }
  if (finite_f(v)) return true;
  p[0] |= v != v ? 0x40 : 0;  // a NaN stays one whose payload is in the bits cut off
  p[1] = p[2] = 0;
  return false;
}

// At least two workgroups (4 waves per SIMD) per CU.
template <int NC, int SUB>
__global__ __launch_bounds__(kMmNW * 64, 4) void fwd_mfma_kernel(const FwdParams p) {
  using S = MmFwdShape<NC, SUB>;
  constexpr int PP = S::PP, KB = S::KB, ROWS = S::ROWS;
  extern __shared__ __align__(16) uint16_t mlds[];
  uint16_t* const xs = mlds;
  uint16_t* const wp = mlds + S::WP;
  int32_t* const flag = reinterpret_cast<int32_t*>(mlds + S::FLAG);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lq = lane >> 4;
  const int T = p.T, D = p.D, W = p.W, P = W - 1, sh = PP - P;

  // Channel blocks, their order and the last one of a dim that 32 does not divide: as in the backward.
  constexpr int kChunk = 512;
  const int first = blockIdx.x / kChunk * kChunk;
  const int blk = first + xcd_remap(blockIdx.x - first, min(kChunk, p.tl.nBlk - first));
  const int cb = blk % p.tl.nGW;
  const int rest = blk / p.tl.nGW;
  const int tile = rest % p.tl.nT;
  const int b = rest / p.tl.nT;
  const int c0 = min(cb * kMmCh, D - kMmCh);
  const int t0 = tile * p.tl.L;
  const int t1 = min(t0 + p.tl.L, T);

  // Staging: a thread takes 8 rows of 2 channels of each 256.
  const int oct = tid >> 4, ch2 = 2 * (tid & 15);
  const uint32_t coff = (uint32_t)(c0 + ch2) * 2u;
  const uint16_t* const xb = static_cast<const uint16_t*>(p.x) + (int64_t)b * p.s_xb;
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(xb), 0, (int)p.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      static_cast<uint16_t*>(p.out) + (int64_t)b * T * D, 0, (int)p.o_bytes, 0x00020000);
  const uint32_t xrow = (uint32_t)p.s_xt * 2u, orow = (uint32_t)D * 2u;
  uint32_t rx[SUB][8];
  auto load = [&](int a) {
#pragma unroll
    for (int h = 0; h < SUB; ++h) {
      const int r0 = a + h * kMmRows + 8 * oct;
      if (a + (h + 1) * kMmRows <= T) {
        const uint32_t xo = (uint32_t)r0 * xrow + coff;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          rx[h][e] = __builtin_amdgcn_raw_buffer_load_b32(xrs, xo, e * xrow, kCachePlain);
      } else {  // rows past the end repeat the last one
#pragma unroll
        for (int e = 0; e < 8; ++e)
          rx[h][e] = __builtin_amdgcn_raw_buffer_load_b32(
              xrs, (uint32_t)min(r0 + e, T - 1) * xrow + coff, 0, kCachePlain);
      }
    }
  };
  uint32_t bad = 0;
  auto put = [&](const uint32_t (&r)[8], int at) {
    u32x4 lo, hi;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] = __builtin_amdgcn_perm(r[2 * e + 1], r[2 * e], 0x05040100u);
      hi[e] = __builtin_amdgcn_perm(r[2 * e + 1], r[2 * e], 0x07060302u);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) bad |= (r[e] & 0x7fff7fffu) + 0x00800080u;
    uint16_t* const dst = xs + ch2 * S::XP + at + 8 * oct;
    *reinterpret_cast<u32x4*>(dst) = lo;
    *reinterpret_cast<u32x4*>(dst + S::XP) = hi;
  };

  // Requested together: the first step, the window before the segment, the weights, the biases.
  load(t0);
  uint32_t rw[8];
  if (oct < 2 * NC) {
    const int r0 = t0 - PP + 8 * oct;
    if (t0 >= PP) {
      const uint32_t o = (uint32_t)r0 * xrow + coff;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        rw[e] = __builtin_amdgcn_raw_buffer_load_b32(xrs, o, e * xrow, kCachePlain);
    } else {  // t0 == 0 (segments are at least a window long): the initial states or zeros
      const uint16_t* const q =
          static_cast<const uint16_t*>(p.init) + ((int64_t)b * P + r0 + P) * D + c0 + ch2;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        rw[e] = 0;
        if (p.has_init && r0 + e >= -P)
          rw[e] = (uint32_t)q[(int64_t)e * D] | ((uint32_t)q[(int64_t)e * D + 1] << 16);
      }
    }
  }
  const int wc = tid >> 4, wk = tid & 15;  // this thread's channel and first tap of the weights
  float wv[NC + 1];
  mm_weights<NC>(p.w, p.w_dt, (int64_t)(c0 + wc) * W, wk, P, wv);
  const float bias_v = p.has_bias ? ld_any(p.bias, c0 + (lane & 31), p.b_dt) : 0.0f;

  constexpr int XPAD = S::XP - (PP + ROWS);
  for (int i = tid; i < kMmCh * XPAD; i += kMmNW * 64)
    xs[i / XPAD * S::XP + PP + ROWS + i % XPAD] = 0;
  for (int i = tid; i < kMmCh * 3 * S::WL / 2; i += kMmNW * 64)
    reinterpret_cast<uint32_t*>(wp)[i] = 0;
  lds_barrier();
  if (oct < 2 * NC) put(rw, 0);
  bool wbad = false;
#pragma unroll
  for (int j = 0; j <= NC; ++j) {
    const int k = wk + 16 * j;
    if (k <= P) {
      uint16_t pc[3];
      wbad = !cut3(wv[j], pc) || wbad;
#pragma unroll
      for (int i = 0; i < 3; ++i) wp[(wc * 3 + i) * S::WL + k + sh + 15] = pc[i];
    }
  }

  const uint32_t bad_taps = mm_bad_taps(wbad, wave);
  int slow_prev = 0;  // channels computed row by row by the step before, whose last rows are the window
#pragma unroll 1
  for (int a = t0; a < t1; a += ROWS) {
#pragma unroll
    for (int h = 0; h < SUB; ++h) put(rx[h], PP + h * kMmRows);
    const uint32_t mine = mm_bad_rows(bad) | bad_taps;
    if (lane == 0) flag[wave] = (int32_t)mine;
    bad = 0;
    lds_barrier();
    if (a + ROWS < t1) load(a + ROWS);
    int f = 0;
#pragma unroll
    for (int v = 0; v < kMmNW; ++v) f |= flag[v];
    f = __builtin_amdgcn_readfirstlane(f);
    const uint32_t slow = mm_wave_bits((uint32_t)(slow_prev | f), wave);
    slow_prev = f;

    auto channel = [&](int n, auto by_row) {
      const int ch = wave + n * kMmNW;
      uint16_t* const xc = xs + ch * S::XP;
      const float bias = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(bias_v), ch));
      float o[SUB][4];
      if constexpr (!decltype(by_row)::value) {
        // 8 weights of a lane from any element on: aligned words, shifted where the start is odd.
        const uint32_t* const wq = reinterpret_cast<const uint32_t*>(
            wp + ch * 3 * S::WL + ((8 * lq - li + 15) & ~1));
        const uint32_t wshift = (li & 1) ? 0 : 16;
        f4v z[SUB];
#pragma unroll
        for (int h = 0; h < SUB; ++h) z[h] = f4v{bias, bias, bias, bias};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          bf8v xa[SUB];
#pragma unroll
          for (int h = 0; h < SUB; ++h)
            xa[h] = *reinterpret_cast<const bf8v*>(xc + h * kMmRows + 16 * li + 32 * kb + 8 * lq);
#pragma unroll
          for (int j = 2; j >= 0; --j) {
            const uint32_t* q = wq + j * (S::WL / 2) + 16 * kb;
            uint32_t d[5];
#pragma unroll
            for (int e = 0; e < 5; ++e) d[e] = q[e];
            u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = __builtin_amdgcn_alignbit(d[e + 1], d[e], wshift);
#pragma unroll
            for (int h = 0; h < SUB; ++h)
              z[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, w), xa[h],
                                                             z[h], 0, 0, 0);
          }
        }
#pragma unroll
        for (int h = 0; h < SUB; ++h) {
#pragma unroll
          for (int v = 0; v < 4; ++v) o[h][v] = z[h][v] * sigmoid_f(z[h][v]);
        }
      } else {  // infinities or NaN in the channel's reach: every row in its own window alone
        const uint16_t* const wq = wp + ch * 3 * S::WL + sh + 15;
#pragma unroll
        for (int h = 0; h < SUB; ++h) {
          const uint16_t* const xr = xc + h * kMmRows + 16 * li + 4 * lq + sh;
#pragma unroll
          for (int v = 0; v < 4; ++v) o[h][v] = bias;
          for (int k = 0; k < W; ++k) {
            const float w = bf_one(wq[k]) + (bf_one(wq[S::WL + k]) + bf_one(wq[2 * S::WL + k]));
#pragma unroll
            for (int v = 0; v < 4; ++v) o[h][v] = fmaf(w, bf_one(xr[k + v]), o[h][v]);
          }
#pragma unroll
          for (int v = 0; v < 4; ++v) o[h][v] = o[h][v] * sigmoid_f(o[h][v]);
        }
      }
      // The step's last PP rows are the next one's window; then out takes the rows' place.
      mm_fence();
      if (lane < 2 * NC)
        *reinterpret_cast<u32x4*>(xc + 8 * lane) =
            *reinterpret_cast<const u32x4*>(xc + ROWS + 8 * lane);
      mm_fence();
#pragma unroll
      for (int h = 0; h < SUB; ++h)
        *reinterpret_cast<u32x2*>(xc + PP + h * kMmRows + 16 * li + 4 * lq) =
            u32x2{bf_pack(o[h][0], o[h][1]), bf_pack(o[h][2], o[h][3])};
      mm_fence();
    };
    // Without a branch between the channels where no channel needs it. One after the other: their
    // instructions interleaved over the loop were slower (W=64 B=32 T=16 D=2560 35.2 -> 36.1 us).
    if ((slow & 0x1111u) == 0) {
#pragma unroll
      for (int n = 0; n < kMmPerWave; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        channel(n, std::false_type{});
      }
    } else {
#pragma unroll 1
      for (int n = 0; n < kMmPerWave; ++n) {
        if (slow >> (4 * n) & 1) channel(n, std::true_type{});
        else channel(n, std::false_type{});
      }
    }
    lds_barrier();

#pragma unroll
    for (int h = 0; h < SUB; ++h) {
      const uint16_t* const src = xs + ch2 * S::XP + PP + h * kMmRows + 8 * oct;
      const u32x4 lo = *reinterpret_cast<const u32x4*>(src);
      const u32x4 hi = *reinterpret_cast<const u32x4*>(src + S::XP);
      uint32_t r[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[2 * e] = __builtin_amdgcn_perm(hi[e], lo[e], 0x05040100u);
        r[2 * e + 1] = __builtin_amdgcn_perm(hi[e], lo[e], 0x07060302u);
      }
      const int r0 = a + h * kMmRows + 8 * oct;
      if (a + (h + 1) * kMmRows <= t1) {
        const uint32_t off = (uint32_t)r0 * orow + coff;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          __builtin_amdgcn_raw_buffer_store_b32(r[e], ors, off, e * orow, kCachePlain);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (r0 + e < t1)
            __builtin_amdgcn_raw_buffer_store_b32(r[e], ors, (uint32_t)(r0 + e) * orow + coff, 0,
                                                  kCachePlain);
        }
      }
    }
  }

  if (p.has_final && t1 == T) {
    uint16_t* const fb = static_cast<uint16_t*>(p.fin) + (int64_t)b * P * D + c0;
    const uint16_t* const ib = static_cast<const uint16_t*>(p.init) + (int64_t)b * P * D + c0;
    for (int i = tid; i < P * kMmCh; i += kMmNW * 64) {
      const int q = i / kMmCh, c = i % kMmCh, row = T - P + q;
      uint16_t v = 0;
      if (row >= 0) v = xb[(int64_t)row * p.s_xt + c0 + c];
      else if (p.has_init) v = ib[(int64_t)(row + P) * D + c];
      fb[(int64_t)q * D + c] = v;
    }
  }
}

}  // namespace ccv1d
