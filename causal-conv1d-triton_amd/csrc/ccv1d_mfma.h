// Backward with silu on the matrix cores, for bf16 x (widths 33 to kMaxBlockW = 128, no seq_idx).
//
// Along one channel every sum of the backward is a product with a Toeplitz or Hankel matrix of
// W + 15 distinct values: 256 rows t = 16 b + i of z are Z[b][i] = sum_s X[b][s] Wt[s][i] with
// X[b][s] = x[16 b - Pp + s] and Wt[s][i] = w[s - i - (Pp - P)], K = Pp + 16 deep (Pp: P = W - 1
// rounded up to 16); dx is the same product with the rows of g in reverse, so it takes the same
// weight fragments; and dweight's lags l = i - j + 16 m are the entries (i, j) of
// sum_b g[16 b + i] x[16 (b - m) + j]. Each is a few v_mfma_f32_16x16x32_bf16 per 256 elements of
// a channel where the vector units need 3 W multiply-adds per element.
//
// fp32 operands (the weights and g) are the exact sum of three bf16 pieces of 8 bits each: products
// of pieces are exact in fp32 and the matrix cores add them in fp32. z takes 3 products (x is bf16),
// dweight 3, dx the 6 of its 9 whose size is above 2^-25 of the result. Against 64-bit results the
// sums are no further off than those of the register-window kernels.
//
// Zeros of the Toeplitz matrix meet rows outside an output's window, so an infinity or NaN there would
// spread: a channel whose x, dout, weights or g in reach are not all finite is computed with vector
// arithmetic in its window alone (mm_slow). Each channel goes by its own values, never by those of
// the 31 it shares a workgroup with: its results do not depend on them, and the two workgroups that
// share channels where 32 does not divide dim store the same bits.
//
// A workgroup takes 32 channels and walks a segment of rows in steps of 256. Rows are read channels
// last, transposed in registers (8 rows x 2 channels per lane) and kept per channel in time order in
// LDS, where the operands are 16-byte reads; dweight's operand of x, 4 rows 16 apart, is a
// transposing read. A wave takes 4 of the channels. dx is written PP rows behind the rows of a step.
//
// Measured, fwd+bwd B=2 T=4096 D=1024 against the block kernels (ccv1d_block.h) in the backward:
// W=33 107 -> 85 us, W=64 139 -> 108, W=100 306 -> 138, W=128 351 -> 158; then, with segments that fill
// rounds and the matrix-core forward at 68.5, 85.7, 107.6 and 121.7, the weights' fragments kept from z
// to dx (64.9, 82.2, 101.7) and no dweight products in a segment's last step where that holds dx rows
// alone (63.7, 80.5, 98.7, 119.1; leaving z out there too past the end of x: T=256 W=40 121.4 -> 118.2, but
// W=33 63.7 -> 64.4). These are graphs of many steps; one step per graph replay takes 85 us at W=64.
// What bounds it is latency: at W=64 (66 us under the counters) the matrix units are busy 9 us, the
// vector units about 17 (504 instructions per 256 elements), LDS 26 (8 of them bank conflicts), and the
// waves wait 45 % of their time, 2 per SIMD in phases between barriers. A second workgroup per CU
// fits neither the LDS (from NC = 3) nor the registers. At widths 9-32 the register-window kernels
// are faster (B=4 T=8192 D=1024 W=16 95 us against 150, W=32 159 against 210).
#pragma once

#include "ccv1d_device.h"

namespace ccv1d {

constexpr int kMmNW = 8;
constexpr int kMmPerWave = kMmCh / kMmNW;

typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4v lds_s4v;

// LDS layout for windows of NC blocks of 16 rows (16-bit elements; every row a multiple of 16 bytes).
template <int NC>
struct MmShape {
  static constexpr int PP = 16 * NC;
  static constexpr int KB = (PP + 16 + 31) / 32;  // k-blocks of 32
  static constexpr int XP = 248 + 32 * KB;        // x: rows a - PP .. a + 255, zeros to 240 + 32 KB
  static constexpr int YP = kMmRows + 8;          // dout of the step, then its dx
  static constexpr int GP = 240 + 32 * KB;        // one piece of g: row a + 255 - r at r, PP rows back
  static constexpr int WL = 32 * KB + 16;         // one piece of the weights: tap k at k + PP - P + 15
  static constexpr int X = 0;
  static constexpr int Y = X + kMmCh * XP;
  static constexpr int G = Y + kMmCh * YP;              // per wave
  static constexpr int GT = G + kMmNW * 3 * GP;         // per channel: g of the step's last PP rows
  static constexpr int WP = GT + kMmCh * 3 * PP;
  static constexpr int FLAG = WP + kMmCh * 3 * WL;      // one word per wave
  static constexpr int SUM = FLAG + 2 * kMmNW;          // floats [32][SP]: sums of mm_slow (dbias last)
  static constexpr int SP = PP + 2;
  static constexpr int TAPS = SUM + 2 * kMmCh * SP;     // floats [32][SP]: weights of mm_slow (bias last)
  static constexpr int BYTES = 2 * TAPS + 4 * kMmCh * SP;
  static_assert(XP >= PP + kMmRows && GP >= PP + kMmRows && FLAG % 8 == 0, "layout");
  static_assert((kMaxBlockW + 1) * kMmCh * 2 <= kMmCh * YP, "dweight sums reuse the dout rows");
  static_assert(16 * 17 * 2 <= 3 * GP, "one tile of dweight lags reuses a wave's g rows");
};

// LDS reads and writes of different types to the same memory: keeps the compiler from reordering them
// (the hardware runs a wave's LDS operations in order).
__device__ __forceinline__ void mm_fence() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ float bf_one(uint16_t u) { return __uint_as_float((uint32_t)u << 16); }
__device__ __forceinline__ uint32_t bf_pack(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2v){a, b}, bf2v));
}
__device__ __forceinline__ bool finite_f(float v) {
  return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u;
}

// Sets of a workgroup's 32 channels: channel ch is bit ch / 2 of its half, the even channels in the
// lower 16 bits, so that the channels of one wave (wave + n * kMmNW) are every fourth bit from
// mm_bit(wave) on.
__device__ __forceinline__ int mm_bit(int ch) { return (ch >> 1) + ((ch & 1) << 4); }
__device__ __forceinline__ uint32_t mm_wave_bits(uint32_t set, int wave) {
  return set >> mm_bit(wave);  // bit 4 n: channel wave + n * kMmNW
}
static_assert(kMmNW == 8 && kMmCh == 32, "every fourth bit of a half");

// The wave's channels whose staged rows hold an infinity or NaN: a thread has rows of channels
// 2 (lane % 16) and the one after it, `bad` says so of them in bits 15 and 31.
__device__ __forceinline__ uint32_t mm_bad_rows(uint32_t bad) {
  if (!__any((bad & 0x80008000u) != 0)) return 0;
  const uint64_t e = __ballot((bad & 0x8000u) != 0), o = __ballot((bad & 0x80000000u) != 0);
  uint32_t lo = (uint32_t)e | (uint32_t)(e >> 32), hi = (uint32_t)o | (uint32_t)(o >> 32);
  lo |= lo >> 16;
  hi |= hi << 16;
  return (lo & 0xffffu) | (hi & 0xffff0000u);
}

// Those whose weights do: 16 lanes have the taps of one of the wave's 4 channels.
__device__ __forceinline__ uint32_t mm_bad_taps(bool bad, int wave) {
  const uint64_t b = __ballot(bad);
  if (b == 0) return 0;
  uint32_t set = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if ((b >> (16 * q)) & 0xffffu) set |= 1u << mm_bit(4 * wave + q);
  return set;
}

// v as three bf16 pieces (bits) whose sum is v; false if v or its first piece is not finite.
__device__ __forceinline__ bool split3(float v, uint16_t (&p)[3]) {
  float r = v;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const uint16_t h = (uint16_t)(bf_pack(r, 0.0f) & 0xffffu);
    p[i] = h;
    r -= bf_one(h);
  }
  if (finite_f(bf_one(p[0]))) return true;
  p[1] = p[2] = 0;
  return false;
}

// Taps wk, wk + 16, ... of the weights from element `off`, those past tap P repeated (not used).
template <int NC>
__device__ __forceinline__ void mm_weights(const void* w, int dt, int64_t off, int wk, int P,
                                           float (&v)[NC + 1]) {
  auto each = [&](auto* q) {
#pragma unroll
    for (int j = 0; j <= NC; ++j) v[j] = static_cast<float>(q[off + min(wk + 16 * j, P)]);
  };
  switch (dt) {
    case DT_F32: each(static_cast<const float*>(w)); break;
    case DT_F16: each(static_cast<const _Float16*>(w)); break;
    case DT_BF16: each(static_cast<const __bf16*>(w)); break;
    default: each(static_cast<const double*>(w)); break;
  }
}

// 4 values down a column of a row-major 16-column block of 16-bit elements: lane l gets elements
// (4 (l / 16) + v, l % 16), v = 0 .. 3; `p` is the block's first element.
__device__ __forceinline__ u32x2 mm_column(const uint16_t* p, int lane) {
  const s4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_s4v*)(const_cast<uint16_t*>(p) + 4 * lane));
  return __builtin_bit_cast(u32x2, v);
}

// One channel of one step in its rows' own windows, with vector arithmetic: g~ = -ln2 g of the step's
// rows (its pieces to `g`, whose last PP rows hold the previous ones), dx to `yc`, the sums of dweight
// and dbias added to `sum`. rows_t: rows of the step before T; own: its own rows. `taps` (the bias
// last) and pre-activations are the unscaled ones: times log2(e) as in the products, those above
// 2.36e38 would be infinite.
template <int NC, typename DF>
__device__ __forceinline__ void mm_slow(const uint16_t* xc, uint16_t* yc, uint16_t* g,
                                        const float* taps, int W, int rows_t, int own, int lane,
                                        float* sum, const DF& dfinal) {
  using S = MmShape<NC>;
  const int P = W - 1, sh = S::PP - P;
  auto g_at = [&](int r) {  // row r of the window (0 .. PP + 255)
    const uint16_t* q = g + S::PP + kMmRows - 1 - r;
    return bf_one(q[0]) + (bf_one(q[S::GP]) + bf_one(q[2 * S::GP]));
  };
  float db = 0.0f;
#pragma unroll 1
  for (int r = lane; r < kMmRows; r += 64) {
    float z = taps[P] * bf_one(xc[r + sh + P]);
    for (int k = 0; k < P; ++k) z = fmaf(taps[k], bf_one(xc[r + sh + k]), z);
    const float gv = r < rows_t ? -kLn2 * dsilu_times(bf_one(yc[r]), z + taps[W]) : 0.0f;
    uint16_t pc[3];
    split3(gv, pc);
#pragma unroll
    for (int i = 0; i < 3; ++i) g[i * S::GP + kMmRows - 1 - r] = pc[i];
    if (r < own) db += gv;
  }
  mm_fence();
#pragma unroll 1
  for (int r = lane; r < kMmRows; r += 64) {
    float d = 0.0f;
    for (int j = 0; j <= P; ++j) d = fmaf(taps[P - j], g_at(r + j), d);
    d = fmaf(d, kNegLog2e, dfinal(r));
    yc[r] = (uint16_t)(bf_pack(d, 0.0f) & 0xffffu);
  }
  const int rows = min(own, kMmRows);
#pragma unroll 1
  for (int k = lane; k < W; k += 64) {
    float s = 0.0f;
    for (int r = 0; r < rows; ++r) s = fmaf(g_at(S::PP + r), bf_one(xc[r + sh + k]), s);
    sum[k] += s;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) db += __shfl_xor(db, o);
  if (lane == 0) sum[W] += db;
  mm_fence();
}

// Two waves per SIMD: the dweight tiles alone take 16 (NC + 1) registers, and LDS from NC = 3 on holds
// one workgroup per CU.
template <int NC>
__global__ __launch_bounds__(kMmNW * 64, 2) void bwd_mfma_kernel(const BwdParams p) {
  using S = MmShape<NC>;
  constexpr int PP = S::PP, KB = S::KB;
  extern __shared__ __align__(16) uint16_t mlds[];
  uint16_t* const xs = mlds + S::X;
  uint16_t* const ys = mlds + S::Y;
  uint16_t* const gt = mlds + S::GT;
  uint16_t* const wp = mlds + S::WP;
  int32_t* const flag = reinterpret_cast<int32_t*>(mlds + S::FLAG);
  float* const slow_sum = reinterpret_cast<float*>(mlds + S::SUM);
  float* const slow_taps = reinterpret_cast<float*>(mlds + S::TAPS);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lq = lane >> 4;
  uint16_t* const g = mlds + S::G + wave * 3 * S::GP;
  const int T = p.T, D = p.D, W = p.W, P = W - 1, sh = PP - P;

  // Neighbouring channel blocks of one range of rows are consecutive and run on one XCD at about the
  // same time: a row's 128-byte line holds two of them.
  constexpr int kChunk = 512;
  const int first = blockIdx.x / kChunk * kChunk;
  const int blk = first + xcd_remap(blockIdx.x - first, min(kChunk, p.tl.nBlk - first));
  const int cb = blk % p.tl.nGW;
  const int rest = blk / p.tl.nGW;
  const int tile = rest % p.tl.nT;
  const int b = rest / p.tl.nT;
  // The last block of a dim that is not a multiple of 32 is its last 32 channels: it shares channels with
  // the block before, and both store the same bits for them (a channel's arithmetic, the choice of
  // mm_slow included, depends on its own values alone).
  const int c0 = min(cb * kMmCh, D - kMmCh);
  const int t0 = tile * p.tl.L;
  const int own_end = min(t0 + p.tl.L, T);
  const int emit_lo = (tile == 0 && p.need_dinit) ? -P : t0;
  const int need_end = min(own_end + PP, T);
  const int steps = (own_end - t0 + PP + kMmRows - 1) / kMmRows;

  // Staging: a thread takes 8 rows of 2 channels.
  const int cp = tid & 15, oct = tid >> 4;
  const int ch2 = 2 * cp;
  const uint32_t coff = (uint32_t)(c0 + ch2) * 2u;
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(static_cast<const uint16_t*>(p.x) + (int64_t)b * p.s_xb), 0,
      (int)p.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(static_cast<const uint16_t*>(p.dy) + (int64_t)b * p.s_yb), 0,
      (int)p.y_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc(
      static_cast<uint16_t*>(p.dx) + (int64_t)b * p.s_dxb, 0, (int)p.o_bytes, 0x00020000);
  const uint32_t xrow = (uint32_t)p.s_xt * 2u, yrow = (uint32_t)p.s_yt * 2u,
                 drow = (uint32_t)p.s_dxt * 2u;
  uint32_t rx[8], ry[8];
  auto load = [&](int a) {
    int tid_ = tid;
    asm volatile("" : "+v"(tid_));
    const int r0 = a + 8 * (tid_ >> 4);
    const uint32_t coff = (uint32_t)(c0 + 2 * (tid_ & 15)) * 2u;
    if (a + kMmRows <= need_end) {
      const uint32_t xo = (uint32_t)r0 * xrow + coff, yo = (uint32_t)r0 * yrow + coff;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        rx[e] = __builtin_amdgcn_raw_buffer_load_b32(xrs, xo, e * xrow, kCacheNT);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        ry[e] = __builtin_amdgcn_raw_buffer_load_b32(yrs, yo, e * yrow, kCacheNT);
    } else {  // rows past the last one needed repeat it; past T their g is 0
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t r = (uint32_t)min(r0 + e, need_end - 1);
        rx[e] = __builtin_amdgcn_raw_buffer_load_b32(xrs, r * xrow + coff, 0, kCacheNT);
        ry[e] = __builtin_amdgcn_raw_buffer_load_b32(yrs, r * yrow + coff, 0, kCacheNT);
      }
    }
  };
  // 8 rows of 2 channels to their channels' rows `at`; the bits of `bad` say whether all are finite.
  auto put = [&](const uint32_t (&r)[8], uint16_t* dst, int pitch, int at, uint32_t& bad) {
    int tid_ = tid;
    asm volatile("" : "+v"(tid_));
    const int ch2 = 2 * (tid_ & 15);
    at += 8 * (tid_ >> 4);
    u32x4 lo, hi;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      lo[e] = __builtin_amdgcn_perm(r[2 * e + 1], r[2 * e], 0x05040100u);
      hi[e] = __builtin_amdgcn_perm(r[2 * e + 1], r[2 * e], 0x07060302u);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) bad |= (r[e] & 0x7fff7fffu) + 0x00800080u;
    *reinterpret_cast<u32x4*>(dst + ch2 * pitch + at) = lo;
    *reinterpret_cast<u32x4*>(dst + (ch2 + 1) * pitch + at) = hi;
  };

  // Everything the start needs from memory is requested before the first of it is used: the first
  // step, the window before the segment, the weights (16 lanes to a channel) and the biases.
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
  const float bias_u = p.has_bias ? ld_any(p.bias, c0 + (lane & 31), p.b_dt) : 0.0f;
  const float bias_v = kNegLog2e * bias_u;

  constexpr int XPAD = S::XP - (PP + kMmRows), GPAD = S::GP - (PP + kMmRows);
  for (int i = tid; i < kMmCh * XPAD; i += kMmNW * 64)
    xs[i / XPAD * S::XP + PP + kMmRows + i % XPAD] = 0;
  if constexpr (GPAD > 0) {
    for (int i = lane; i < 3 * GPAD; i += 64) g[i / GPAD * S::GP + PP + kMmRows + i % GPAD] = 0;
  }
  for (int i = tid; i < kMmCh * 3 * PP / 2; i += kMmNW * 64) reinterpret_cast<uint32_t*>(gt)[i] = 0;
  for (int i = tid; i < kMmCh * 3 * S::WL / 2; i += kMmNW * 64)
    reinterpret_cast<uint32_t*>(wp)[i] = 0;
  for (int i = tid; i < kMmCh * S::SP; i += kMmNW * 64) slow_sum[i] = 0.0f;
  lds_barrier();
  uint32_t bad = 0;
  if (oct < 2 * NC) put(rw, xs, S::XP, 0, bad);
  // Weights times -log2(e) (dsilu_scaled) in pieces, among the zeros, and as they are for mm_slow.
  if (tid < kMmCh) slow_taps[tid * S::SP + W] = bias_u;
  bool wbad = false;
#pragma unroll
  for (int j = 0; j <= NC; ++j) {
    const int k = wk + 16 * j;
    if (k <= P) {
      uint16_t pc[3];
      wbad = !split3(kNegLog2e * wv[j], pc) || wbad;
      slow_taps[wc * S::SP + k] = wv[j];
#pragma unroll
      for (int i = 0; i < 3; ++i) wp[(wc * 3 + i) * S::WL + k + sh + 15] = pc[i];
    }
  }

  f4v acc[kMmPerWave][NC + 1];
  float db[kMmPerWave];
  uint32_t gbad = 0;  // bit n: g of channel n in the window before the step is not all finite
#pragma unroll
  for (int n = 0; n < kMmPerWave; ++n) {
#pragma unroll
    for (int m = 0; m <= NC; ++m) acc[n][m] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    db[n] = 0.0f;
  }

  const uint32_t bad_taps = mm_bad_taps(wbad, wave);
  int slow_prev = 0;  // channels of mm_slow by the step before, whose last rows are the window
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    const int a = t0 + s * kMmRows;
    put(rx, xs, S::XP, PP, bad);
    put(ry, ys, S::YP, 0, bad);
    const uint32_t mine = mm_bad_rows(bad) | bad_taps;
    if (lane == 0) flag[wave] = (int32_t)mine;
    bad = 0;
    lds_barrier();
    if (s + 1 < steps) load(a + kMmRows);
    int f = 0;
#pragma unroll
    for (int v = 0; v < kMmNW; ++v) f |= flag[v];
    f = __builtin_amdgcn_readfirstlane(f);
    const uint32_t slow = mm_wave_bits((uint32_t)(slow_prev | f), wave);
    slow_prev = f;
    const int rows_t = T - a;      // rows of the step before T (may be <= 0)
    const int own = own_end - a;   // its own rows (may be <= 0: only dx rows are left)
    const int row0 = a - PP;       // row of the step's first dx

    auto dfinal = [&](int ch, int r) {  // of the step's dx row r
      const int q = row0 + r - (T - P);
      return q >= 0 && q < P
                 ? bf_one(static_cast<const uint16_t*>(p.dfin)[((int64_t)b * P + q) * D + c0 + ch])
                 : 0.0f;
    };
    const bool with_dfinal = p.has_dfinal && row0 + kMmRows > T - P;
    // g of the PP rows before the step, and the last PP rows on to the next step's window.
    auto tails_in = [&](int ch, int lane) {
      const int tp = lane / (2 * NC), t8 = lane % (2 * NC) * 8;
      if (lane < 6 * NC)
        *reinterpret_cast<u32x4*>(g + tp * S::GP + kMmRows + t8) =
            *reinterpret_cast<const u32x4*>(gt + (ch * 3 + tp) * PP + t8);
      mm_fence();
    };
    auto tails_out = [&](int ch, int lane) {
      const int tp = lane / (2 * NC), t8 = lane % (2 * NC) * 8;
      mm_fence();
      if (lane < 6 * NC)
        *reinterpret_cast<u32x4*>(gt + (ch * 3 + tp) * PP + t8) =
            *reinterpret_cast<const u32x4*>(g + tp * S::GP + t8);
      if (lane < 2 * NC)
        *reinterpret_cast<u32x4*>(xs + ch * S::XP + 8 * lane) =
            *reinterpret_cast<const u32x4*>(xs + ch * S::XP + kMmRows + 8 * lane);
      mm_fence();
    };
    uint32_t todo = 0;  // channels for mm_slow
    const uint32_t flip = ((s + tile + b) & 1) ? 0x80008000u : 0u;
    const float sign = ((s + tile + b) & 1) ? -1.0f : 1.0f;

#pragma unroll
    for (int n = 0; n < kMmPerWave; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      int ch = wave + n * kMmNW;
      // Recomputed per channel and step: 4 channels' addresses would not stay within the registers.
      int ln = lane;
      asm volatile("" : "+s"(ch), "+v"(ln));
      const int li = ln & 15, lq = ln >> 4;
      bool fast = !(slow >> (4 * n) & 1) && !(gbad >> n & 1);
      const uint16_t* const xc = xs + ch * S::XP;
      uint16_t* const yc = ys + ch * S::YP;
      // A lane's 8 weights start at any element: 5 aligned words, shifted by one element where the
      // start is odd.
      const uint32_t* const wc = reinterpret_cast<const uint32_t*>(
          wp + ch * 3 * S::WL + ((8 * lq - li + 15) & ~1));
      const uint32_t wshift = (li & 1) ? 0 : 16;
      auto weights_at = [&](int kb, int j) {
        const uint32_t* q = wc + j * (S::WL / 2) + 16 * kb;
        uint32_t d[5];
#pragma unroll
        for (int e = 0; e < 5; ++e) d[e] = q[e];
        u32x4 f;
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = __builtin_amdgcn_alignbit(d[e + 1], d[e], wshift);
        return __builtin_bit_cast(bf8v, f);
      };
      // Kept from z to dx up to 7 window blocks (at 8 they spill: W=128 121.7 -> 125.5 us).
      constexpr bool kKeepW = NC <= 7;
      bf8v wf[KB][3];
      if constexpr (kKeepW) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int j = 0; j < 3; ++j) wf[kb][j] = weights_at(kb, j);
      }
      auto weights = [&](int kb, int j) {
        if constexpr (kKeepW) return wf[kb][j];
        else return weights_at(kb, j);
      };
      float gv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      u32x2 hi = {0u, 0u}, mid = {0u, 0u}, lo = {0u, 0u};
      if (fast) {
        const float zf =
            __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(bias_v), ch));
        f4v z = {zf, zf, zf, zf};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const bf8v xa = *reinterpret_cast<const bf8v*>(xc + 16 * li + 32 * kb + 8 * lq);
#pragma unroll
          for (int j = 2; j >= 0; --j) {
            z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, weights(kb, j), z, 0, 0, 0);
          }
        }
        const u32x2 yv = mm_column(yc, ln);
        gv[0] = dsilu_scaled(bf_lo(yv[0]), z[0]);
        gv[1] = dsilu_scaled(bf_hi(yv[0]), z[1]);
        gv[2] = dsilu_scaled(bf_lo(yv[1]), z[2]);
        gv[3] = dsilu_scaled(bf_hi(yv[1]), z[3]);
        if (rows_t < kMmRows) {
#pragma unroll
          for (int v = 0; v < 4; ++v) gv[v] = 64 * lq + 16 * v + li < rows_t ? gv[v] : 0.0f;
        }
        hi = u32x2{bf_pack(gv[0], gv[1]), bf_pack(gv[2], gv[3])};
        const float r0 = gv[0] - bf_lo(hi[0]), r1 = gv[1] - bf_hi(hi[0]);
        const float r2 = gv[2] - bf_lo(hi[1]), r3 = gv[3] - bf_hi(hi[1]);
        mid = u32x2{bf_pack(r0, r1), bf_pack(r2, r3)};
        lo = u32x2{bf_pack(r0 - bf_lo(mid[0]), r1 - bf_hi(mid[0])),
                   bf_pack(r2 - bf_lo(mid[1]), r3 - bf_hi(mid[1]))};
        // 0 unless a g or its first piece is not finite.
        const float chk = fmaf(r0, 0.0f, fmaf(r1, 0.0f, fmaf(r2, 0.0f, r3 * 0.0f)));
        fast = __all(chk == 0.0f);
        if (fast) {
          tails_in(ch, ln);
          uint16_t* const gw = g + kMmRows - 1 - 64 * lq - li;
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const u32x2 pc = j == 0 ? hi : j == 1 ? mid : lo;
            gw[j * S::GP] = (uint16_t)pc[0];
            gw[j * S::GP - 16] = (uint16_t)(pc[0] >> 16);
            gw[j * S::GP - 32] = (uint16_t)pc[1];
            gw[j * S::GP - 48] = (uint16_t)(pc[1] >> 16);
          }
        } else {
          gv[0] = gv[1] = gv[2] = gv[3] = 0.0f;
          hi = mid = lo = u32x2{0u, 0u};
        }
      }
      if (own > 0) {  // else a step of dx rows alone (the segment's window)
        if (own < kMmRows) {  // rows past the segment count in dx only
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const bool in = 64 * lq + 16 * v + li < own;
            const uint32_t keep = in ? 0xffffffffu : (v & 1) ? 0x0000ffffu : 0xffff0000u;
            hi[v >> 1] &= keep;
            mid[v >> 1] &= keep;
            lo[v >> 1] &= keep;
            gv[v] = in ? gv[v] : 0.0f;
          }
        }
        db[n] += (gv[0] + gv[1]) + (gv[2] + gv[3]);
        // K slots of a lane: rows b = 4 lq + v once with the first piece and once with the second.
        const bf8v ga = __builtin_bit_cast(bf8v, (u32x4){hi[0], hi[1], mid[0], mid[1]});
        const bf8v gb = __builtin_bit_cast(bf8v, (u32x4){lo[0], lo[1], 0u, 0u});
#pragma unroll
        for (int m = 0; m <= NC; ++m) {
          const u32x2 xv = mm_column(xc + 16 * (NC - m), ln);
          const uint32_t x0 = fast ? xv[0] ^ flip : 0u, x1 = fast ? xv[1] ^ flip : 0u;
          const bf8v xb = __builtin_bit_cast(bf8v, (u32x4){x0, x1, x0, x1});
          // A step's products are summed from zero and the steps by vector adds. The matrix cores'
          // sums are biased downwards by about 1 % of an ulp, which grows with the number of rows
          // where the rounding errors themselves average out: every other step takes x negated, counted
          // over the segments and the batch too, since short rows have one step each (dweight against
          // 64 bits, counted without the batch: B=16 T=100 D=512 W=33 2.0e-7 -> 1.3e-7, B=8 T=64
          // D=1024 W=64 1.7e-7 -> 1.2e-7).
          f4v t = {0.0f, 0.0f, 0.0f, 0.0f};
          t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gb, xb, t, 0, 0, 0);
          t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, xb, t, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            float sum = fmaf(sign, t[v], acc[n][m][v]);
            asm volatile("" : "+v"(sum));  // added here: the adds would sink past dx, all t held
            acc[n][m][v] = sum;
          }
        }
      }
      mm_fence();
      if (fast) {
        f4v d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          bf8v gp[3], w[3];
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            gp[j] = *reinterpret_cast<const bf8v*>(g + j * S::GP + 240 - 16 * li + 32 * kb + 8 * lq);
            w[j] = weights(kb, j);
          }
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[0], gp[2], d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2], gp[0], d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[1], gp[1], d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[0], gp[1], d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[1], gp[0], d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[0], gp[0], d, 0, 0, 0);
        }
        // Entry (4 lq + v, li) is dx row 16 li + 15 - 4 lq - v.
        const int u = 16 * li + 12 - 4 * lq;
        if (with_dfinal) {
#pragma unroll
          for (int v = 0; v < 4; ++v) d[v] += dfinal(ch, u + 3 - v);
        }
        *reinterpret_cast<u32x2*>(yc + u) = u32x2{bf_pack(d[3], d[2]), bf_pack(d[1], d[0])};
        tails_out(ch, ln);
      } else {
        todo |= 1u << n;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    gbad = 0;
#pragma unroll 1
    for (; todo; todo &= todo - 1) {
      const int n = __builtin_ctz(todo);
      const int ch = wave + n * kMmNW;
      tails_in(ch, lane);
      mm_slow<NC>(xs + ch * S::XP, ys + ch * S::YP, g, slow_taps + ch * S::SP, W, rows_t, own, lane,
                  slow_sum + ch * S::SP,
                  [&](int r) { return with_dfinal ? dfinal(ch, r) : 0.0f; });
      // Whether the next step's window holds a g that is not finite.
      bool ok = true;
      for (int r = lane; r < PP; r += 64) ok = ok && finite_f(bf_one(g[r]));
      if (!__all(ok)) gbad |= 1u << n;
      tails_out(ch, lane);
    }
    lds_barrier();

    // dx rows, transposed back.
    int tid_ = tid;
    asm volatile("" : "+v"(tid_));
    const int ch2 = 2 * (tid_ & 15), oct = tid_ >> 4;
    const uint32_t coff = (uint32_t)(c0 + ch2) * 2u;
    const u32x4 lo = *reinterpret_cast<const u32x4*>(ys + ch2 * S::YP + 8 * oct);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(ys + (ch2 + 1) * S::YP + 8 * oct);
    uint32_t r[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[2 * e] = __builtin_amdgcn_perm(hi[e], lo[e], 0x05040100u);
      r[2 * e + 1] = __builtin_amdgcn_perm(hi[e], lo[e], 0x07060302u);
    }
    const int d0 = row0 + 8 * oct;
    if (row0 >= t0 && row0 + kMmRows <= own_end) {
      const uint32_t off = (uint32_t)d0 * drow + coff;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        __builtin_amdgcn_raw_buffer_store_b32(r[e], drs, off, e * drow, kCacheSC1NT);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int row = d0 + e;
        if (row < emit_lo || row >= own_end) continue;
        if (row >= 0) {
          __builtin_amdgcn_raw_buffer_store_b32(r[e], drs, (uint32_t)row * drow + coff, 0, kCacheSC1NT);
        } else {
          uint16_t* q = static_cast<uint16_t*>(p.dinit) + ((int64_t)b * P + row + P) * D + c0 + ch2;
          q[0] = (uint16_t)r[e];
          q[1] = (uint16_t)(r[e] >> 16);
        }
      }
    }
  }

  // The lags' entries are summed along the diagonals of their tiles: lag l = i - j + 16 m.
  lds_barrier();
  float* const dwl = reinterpret_cast<float*>(ys);  // [W + 1][32]
  float* const tb = reinterpret_cast<float*>(g);    // [16][17]
#pragma unroll
  for (int n = 0; n < kMmPerWave; ++n) {
    const int ch = wave + n * kMmNW;
    for (int k = lane; k < W; k += 64) dwl[k * kMmCh + ch] = slow_sum[ch * S::SP + k];
    mm_fence();
#pragma unroll
    for (int m = 0; m <= NC; ++m) {
#pragma unroll
      for (int v = 0; v < 4; ++v) tb[(4 * lq + v) * 17 + li] = acc[n][m][v];
      mm_fence();
      const int k = P - (16 * m - 15 + lane);
      if (lane < 31 && k >= 0 && k <= P) {
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int i = lane - 15 + j;
          const float t = tb[min(max(i, 0), 15) * 17 + j];
          sum += i >= 0 && i < 16 ? t : 0.0f;
        }
        dwl[k * kMmCh + ch] += sum;
      }
      mm_fence();
    }
    float sb = db[n];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sb += __shfl_xor(sb, o);
    if (lane == 0) dwl[W * kMmCh + ch] = sb + slow_sum[ch * S::SP + W];
  }
  lds_barrier();
  float* const pp = p.part + ((int64_t)b * p.tl.nT + tile) * (W + 1) * D + c0;
  const int n_out = (p.has_bias ? W + 1 : W) * kMmCh;
  for (int i = tid; i < n_out; i += kMmNW * 64)
    pp[(int64_t)(i / kMmCh) * D + i % kMmCh] = dwl[i] * kNegLog2e;
}

}  // namespace ccv1d
