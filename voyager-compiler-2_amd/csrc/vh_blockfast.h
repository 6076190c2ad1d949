// Block-scaled quantization of bf16 tensors to the reference form (bf16 codes
// and scales), one map and mode per kernel: the same arithmetic as k_rows and
// k_cols (vh_blockscale.hip), which decide every step at run time.
//
// What bounds them: HBM, once the arithmetic per element is small.  The
// general kernels spend it on branches (mode, dtype, NaN, the rare exact
// division, each element's map), and their column form reads two bytes a lane
// and every element twice.  Here a block whose maximum is finite and whose
// divisor is normal takes straight-line code, two elements an instruction
// where they fit: the quotients by x * (1 / s) with the hardware's rounding
// (a row of eight goes back to the exact division when one lies near a
// rounding midpoint), block extremes on 16-bit keys, maps without branches.
// Any other block takes element_code, element by element.
#pragma once

#include "vh_blockscale.h"
#include "vh_device.h"

namespace {

typedef unsigned short fu16x2 __attribute__((ext_vector_type(2)));
typedef short fi16x2 __attribute__((ext_vector_type(2)));

VH_DEV uint32_t pk_umax16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t,
                            __builtin_elementwise_max(__builtin_bit_cast(fu16x2, a), __builtin_bit_cast(fu16x2, b)));
}

// Keys of two bf16 patterns for the block's extremes, as unsigned 16-bit
// integers.  MX: the magnitude's bits (NaN above infinity).  AFFINE: ordered
// as the values, -NaN below -infinity, +NaN above +infinity.
VH_DEV uint32_t affine_keys(uint32_t w) {
  const uint32_t neg = __builtin_bit_cast(uint32_t, __builtin_bit_cast(fi16x2, w) >> 15);
  return w ^ (neg | 0x80008000u);
}
VH_DEV uint32_t affine_bits(uint32_t key) { return (key & 0x8000u) ? key ^ 0x8000u : ~key & 0xffffu; }

// A block's extremes from its keys: MX: hi = amax; AFFINE: the maximum and,
// from the maximum of the complemented keys, the minimum; NaN if one is in it.
template <int MODE>
VH_DEV void extremes(uint32_t mx, uint32_t mn, float& hi, float& lo, bool& finite) {
  if constexpr (MODE == AFFINE) {
    const uint32_t mi = ~mn & 0xffffu;
    const bool nan = mx > 0xff80u || mi < 0x007fu;
    finite = mx < 0xff80u && mi > 0x007fu;
    hi = nan ? __uint_as_float(0x7fc00000u) : bf2f(affine_bits(mx));
    lo = nan ? __uint_as_float(0x7fc00000u) : bf2f(affine_bits(mi));
  } else {
    finite = mx < 0x7f80u;
    hi = bf2f(mx);
    lo = 0.0f;
  }
}

// What x is multiplied by: the exact inverse of a power of two, else the
// hardware's reciprocal; 0 where the block needs element_code.
template <int MODE>
VH_DEV float fast_inverse(const BlockScale& bs, bool finite) {
  if constexpr (MODE == MX_POT) return finite ? bs.inv : 0.0f;
  const float a = fabsf(bs.el_scale);
  const bool ok = finite && a >= 0x1p-126f && a <= 0x1p126f && fabsf(bs.zp) < __builtin_inff();
  return ok ? __builtin_amdgcn_rcpf(bs.el_scale) : 0.0f;
}

// A minifloat's value of a finite bf16 x (fmt_minifloat): the nearest
// multiple of the binade's step by adding 1.5 * 2**23 steps and taking them
// off again.
VH_DEV float fast_mini(float x, const vh_format& f) {
  const float a = fminf(fabsf(x), f.clamp_bf16);
  const uint32_t eb = umax32(__float_as_uint(a) & 0x7f800000u, (uint32_t)(f.emin + 127) << 23);
  const float c = __uint_as_float((eb + ((uint32_t)(23 - f.p1) << 23)) | 0x400000u);
  const float r = fminf((a + c) - c, f.max_norm);
  return x == 0.0f ? 0.0f : copysignf(r, x);
}

// Reference-form codes (bf16 pairs) of eight quotients, given as bf16 pairs.
// keys: the thresholds of a table of at most 15, padded (steps_level_padded);
// vals: its 16 entries.
template <int KIND>
VH_DEV uint4 fast_codes(const uint32_t (&q)[4], const vh_format& f, const uint16_t* keys, const uint16_t* vals) {
  uint32_t o[4];
  if constexpr (KIND == K_STEPS) {
    uint32_t key[8], pos[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      key[j] = bf_key(j & 1 ? q[j >> 1] >> 16 : q[j >> 1] & 0xffffu);
      pos[j] = 0;
    }
#pragma unroll
    for (int step = 8; step >= 1; step >>= 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j) pos[j] = (uint32_t)keys[pos[j] + step - 1] <= key[j] ? pos[j] + step : pos[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (uint32_t)vals[pos[2 * j]] | ((uint32_t)vals[pos[2 * j + 1]] << 16);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v0 = __uint_as_float(q[j] << 16), v1 = __uint_as_float(q[j] & 0xffff0000u);
      if constexpr (KIND == K_INT) {
        v0 = fmt_int(v0, f);
        v1 = fmt_int(v1, f);
      } else if constexpr (KIND == K_E4M3) {
        // + 0: an exact zero takes code 0 whatever its sign
        const float c0 = fminf(fmaxf(v0, -448.0f), 448.0f) + 0.0f, c1 = fminf(fmaxf(v1, -448.0f), 448.0f) + 0.0f;
        const int c = __builtin_amdgcn_cvt_pk_fp8_f32(c0, c1, 0, false);
        v0 = __builtin_amdgcn_cvt_f32_fp8(c, 0);
        v1 = __builtin_amdgcn_cvt_f32_fp8(c, 1);
      } else {
        v0 = fast_mini(v0, f);
        v1 = fast_mini(v1, f);
      }
      o[j] = f2bf2_hw(v0, v1);
    }
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// Eight elements of finite blocks: the codes, and whether a quotient lies too
// near a rounding midpoint for its approximation to decide (then they are not
// valid).  Each column's multiplier r (fast_inverse) and zero point z; UNIFORM:
// index 0 for all.
template <int MODE, int KIND, bool UNIFORM>
VH_DEV uint4 fast_elements(const uint4& raw, const float* r, const float* z, const vh_format& f, const uint16_t* keys,
                           const uint16_t* vals, bool& near) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
  uint32_t q[4];
  near = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float q0 = __uint_as_float(w[j] << 16) * r[UNIFORM ? 0 : 2 * j];
    const float q1 = __uint_as_float(w[j] & 0xffff0000u) * r[UNIFORM ? 0 : 2 * j + 1];
    if constexpr (MODE != MX_POT) {
      near |= ((__float_as_uint(q0) - 0x7ffcu) & 0xffffu) <= 8u;
      near |= ((__float_as_uint(q1) - 0x7ffcu) & 0xffffu) <= 8u;
    }
    q[j] = f2bf2_hw(q0, q1);
  }
  if constexpr (MODE == AFFINE) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      q[j] = f2bf2_hw(__uint_as_float(q[j] << 16) + z[UNIFORM ? 0 : 2 * j],
                      __uint_as_float(q[j] & 0xffff0000u) + z[UNIFORM ? 0 : 2 * j + 1]);
  }
  return fast_codes<KIND>(q, f, keys, vals);
}

// The general parameters with the fields these kernels fix as constants.
template <int MODE>
VH_DEV Params fast_params(const Params& in) {
  Params P = in;
  P.mode = MODE;
  P.cdt = VH_BF16;
  P.codes_dtype = VH_BF16;
  P.scale_dtype = VH_BF16;
  P.code_lut = nullptr;
  P.gs = nullptr;
  P.scale_t16 = 0;
  return P;
}

// Eight elements by element_code, each column's divisor s and zero point z.
template <int KIND, bool UNIFORM>
VH_DEV uint4 slow_elements(const uint4& raw, const float* s, const float* z, const Params& P, const uint16_t* lds) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
  uint32_t o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    BlockScale bs;
    bs.el_scale = s[UNIFORM ? 0 : j];
    bs.zp = z[UNIFORM ? 0 : j];
    bs.inv = 0.0f;  // divides: the same quotient
    float v;
    uint32_t c;
    element_code<KIND>(bf2f(j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xffffu), bs, P, lds, nullptr, &v, &c);
    o[j] = f2bf(v);
  }
  return make_uint4(o[0] | (o[1] << 16), o[2] | (o[3] << 16), o[4] | (o[5] << 16), o[6] | (o[7] << 16));
}

// A steps table in LDS, as stage_steps lays it out, its thresholds padded with
// 0xFFFF from nsteps to the 16th.
VH_DEV void stage_steps16(const vh_format& f, uint16_t* lds) {
  if (threadIdx.x < VH_MAX_STEPS) {
    const int i = (int)threadIdx.x;
    lds[i] = i < 16 && i >= f.nsteps ? 0xFFFFu : f.thr_key[i];
    lds[VH_MAX_STEPS + i] = f.val[i];
  }
  __syncthreads();
}

// Blocks along rows of the innermost dimension: eight consecutive elements a
// lane, g = block / 8 lanes a block (as k_rows<8>).  WHOLE: L is a multiple of
// the block, so a lane's block is its index over g.  1777 x 14336 to MX FP8
// with its codes and scales in bf16: 48.0 us by k_rows, 20.3 here (5.1 TB/s);
// 2000 x 14336 to MX-int8 23.1 (28.9 by the row kernel it had); the KIVI
// values below 79.4 -> 36.0.
template <int MODE, int KIND, int SKIND, bool WHOLE>
__global__ void __launch_bounds__(256)
k_fast_rows(const uint16_t* __restrict__ x, uint32_t threads, uint32_t L, FastDiv tpr, int g, Params Pin,
            uint16_t* __restrict__ scale_out, uint16_t* __restrict__ zp_out, uint16_t* __restrict__ codes_out) {
  const Params P = fast_params<MODE>(Pin);
  __shared__ uint16_t lds[2 * VH_MAX_STEPS];
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  bool live = t < threads;
  int64_t base = (int64_t)t * 8;
  if constexpr (!WHOLE) {
    const uint32_t row = fast_div(t, tpr), v = t - row * tpr.d;
    live = live && v * 8u < L;
    base = (int64_t)row * L + v * 8u;
  }
  uint4 raw = make_uint4(0u, 0u, 0u, 0u);  // zero padding of a partial block
  if (live) raw = ld_stream16(x + base);
  if constexpr (KIND == K_STEPS) stage_steps16(Pin.fmt, lds);
  uint32_t mx, mn = 0u;
  if constexpr (MODE == AFFINE) {
    const uint32_t k0 = affine_keys(raw.x), k1 = affine_keys(raw.y), k2 = affine_keys(raw.z), k3 = affine_keys(raw.w);
    const uint32_t a = pk_umax16(pk_umax16(k0, k1), pk_umax16(k2, k3));
    const uint32_t b = pk_umax16(pk_umax16(~k0, ~k1), pk_umax16(~k2, ~k3));
    mx = umax32(a & 0xffffu, a >> 16);
    mn = group_umax_rt(umax32(b & 0xffffu, b >> 16), g);
  } else {
    constexpr uint32_t M = 0x7fff7fffu;
    const uint32_t a = pk_umax16(pk_umax16(raw.x & M, raw.y & M), pk_umax16(raw.z & M, raw.w & M));
    mx = umax32(a & 0xffffu, a >> 16);
  }
  mx = group_umax_rt(mx, g);
  if (t >= threads) return;
  float hi, lo;
  bool finite;
  extremes<MODE>(mx, mn, hi, lo, finite);
  const BlockScale bs = block_scale<SKIND>(hi, lo, P, nullptr);
  if ((t & (uint32_t)(g - 1)) == 0u) {  // (threads of a row and g are multiples of g)
    const uint32_t si = t >> __builtin_ctz((unsigned)g);
    scale_out[si] = (uint16_t)f2bf(bs.scale);
    if constexpr (MODE == AFFINE) zp_out[si] = (uint16_t)f2bf(bs.zp);
  }
  if (!live) return;
  const float r = fast_inverse<MODE>(bs, finite);
  bool near;
  uint4 o = fast_elements<MODE, KIND, true>(raw, &r, &bs.zp, P.fmt, lds, lds + VH_MAX_STEPS, near);
  if (near | (r == 0.0f)) o = slow_elements<KIND, true>(raw, &bs.el_scale, &bs.zp, P, lds);
  st_stream16(codes_out + base, o);
}

// Blocks along another dimension, of 4 ROWS rows, inner a multiple of 8: a
// lane takes eight consecutive columns, wave w of the workgroup rows w ROWS ..
// of the block, in registers (one read of each element, 16 bytes a lane, all
// of a wave's loads in flight).  The waves' extremes meet in LDS, wave w turns
// those of columns 2 w and 2 w + 1 into scales for all four, and each writes
// its rows.  Keys of 8 x 8 x 3968 x 128 with the KIVI formats: 118 us by
// k_cols, 29.6 here (4.7 TB/s).
template <int MODE, int KIND, int SKIND, int ROWS>
__global__ void __launch_bounds__(256)
k_fast_cols(const uint16_t* __restrict__ x, uint32_t total, int64_t L, int64_t inner, FastDiv inner8, FastDiv nblk,
            Params Pin, uint16_t* __restrict__ scale_out, uint16_t* __restrict__ zp_out,
            uint16_t* __restrict__ codes_out) {
  const Params P = fast_params<MODE>(Pin);
  constexpr bool AFF = MODE == AFFINE;
  __shared__ uint16_t lds[2 * VH_MAX_STEPS];
  __shared__ uint32_t s_key[4][AFF ? 8 : 4][64];
  __shared__ float s_div[8][64], s_inv[8][64], s_zp[AFF ? 8 : 1][AFF ? 64 : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t idx = blockIdx.x * 64u + (uint32_t)lane;
  const uint32_t ob = fast_div(idx, inner8), i = idx - ob * inner8.d;
  const uint32_t o = fast_div(ob, nblk), b = ob - o * nblk.d;
  const int64_t row0 = (int64_t)b * (4 * ROWS) + wave * ROWS;
  const int64_t base = ((int64_t)o * L + row0) * inner + (int64_t)i * 8;
  const int64_t left = idx < total ? L - row0 : 0;
  const int rows = left < 0 ? 0 : left < ROWS ? (int)left : ROWS;
  uint4 raw[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)  // zero padding of a partial block
    raw[r] = r < rows ? ld_stream16(x + base + r * inner) : make_uint4(0u, 0u, 0u, 0u);
  uint32_t mx[4] = {0u, 0u, 0u, 0u}, mn[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const uint32_t w[4] = {raw[r].x, raw[r].y, raw[r].z, raw[r].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t k = AFF ? affine_keys(w[j]) : w[j] & 0x7fff7fffu;
      mx[j] = pk_umax16(mx[j], k);
      if constexpr (AFF) mn[j] = pk_umax16(mn[j], ~k);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    s_key[wave][j][lane] = mx[j];
    if constexpr (AFF) s_key[wave][4 + j][lane] = mn[j];
  }
  if constexpr (KIND == K_STEPS) stage_steps16(Pin.fmt, lds);
  else __syncthreads();
  {
    const uint32_t a = pk_umax16(pk_umax16(s_key[0][wave][lane], s_key[1][wave][lane]),
                                 pk_umax16(s_key[2][wave][lane], s_key[3][wave][lane]));
    uint32_t n = 0u;
    if constexpr (AFF)
      n = pk_umax16(pk_umax16(s_key[0][4 + wave][lane], s_key[1][4 + wave][lane]),
                    pk_umax16(s_key[2][4 + wave][lane], s_key[3][4 + wave][lane]));
    uint32_t sb = 0u, zb = 0u;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float hi, lo;
      bool finite;
      extremes<MODE>((a >> (16 * h)) & 0xffffu, (n >> (16 * h)) & 0xffffu, hi, lo, finite);
      const BlockScale bs = block_scale<SKIND>(hi, lo, P, nullptr);
      s_div[2 * wave + h][lane] = bs.el_scale;
      s_inv[2 * wave + h][lane] = fast_inverse<MODE>(bs, finite);
      if constexpr (AFF) s_zp[2 * wave + h][lane] = bs.zp;
      sb |= f2bf(bs.scale) << (16 * h);
      zb |= f2bf(bs.zp) << (16 * h);
    }
    if (idx < total) {
      const int64_t si = (int64_t)ob * inner + (int64_t)i * 8 + 2 * wave;
      *(uint32_t*)(scale_out + si) = sb;
      if constexpr (AFF) *(uint32_t*)(zp_out + si) = zb;
    }
  }
  __syncthreads();
  float inv[8], zp[8];
  uint32_t redo = 0u;  // rows that go element by element
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    inv[j] = s_inv[j][lane];
    zp[j] = AFF ? s_zp[AFF ? j : 0][AFF ? lane : 0] : 0.0f;
    redo |= inv[j] == 0.0f ? (1u << ROWS) - 1u : 0u;
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    bool near;
    const uint4 c = fast_elements<MODE, KIND, false>(raw[r], inv, zp, P.fmt, lds, lds + VH_MAX_STEPS, near);
    redo |= near ? 1u << r : 0u;
    if (r < rows && !((redo >> r) & 1u)) st_stream16(codes_out + base + r * inner, c);
  }
#pragma unroll 1
  for (int r = 0; r < rows; ++r) {
    if (!((redo >> r) & 1u)) continue;
    float div[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) div[j] = s_div[j][lane];
    st_stream16(codes_out + base + r * inner,
                slow_elements<KIND, false>(ld_stream16(x + base + r * inner), div, zp, P, lds));
  }
}

// Whether a map has a fast form.
inline bool fast_map(const vh_format& f) {
  switch (kernel_kind(&f)) {
    case K_INT: case K_E4M3: return true;
    case K_MINI:
      return (f.flags & VH_FMT_SIGNED) && f.p1 >= 0 && f.p1 <= 10 && f.emin >= -100 && f.max_norm < 0x1p100f &&
             f.clamp_bf16 < 0x1p100f;
    case K_STEPS: return f.nsteps <= 15;
    default: return false;
  }
}

// Calls fn(MODE, KIND, SKIND) with the constants of a call that has a fast
// kernel; false for the others.
template <typename F>
bool dispatch_fast(const Params& P, F&& fn) {
  if (P.cdt != VH_BF16 || P.codes_dtype != VH_BF16 || P.scale_dtype != VH_BF16 || P.code_lut || P.gs || P.scale_t16 ||
      !P.has_fmt || !fast_map(P.fmt))
    return false;
  const int k = kernel_kind(&P.fmt), s = P.has_sfmt ? kernel_kind(&P.sfmt) : (int)K_NONE;
#define VH_FAST(M, K, S)                                                                                    \
  if (P.mode == M && k == K && (M == MX_POT || s == S)) {                                                   \
    fn(std::integral_constant<int, M>{}, std::integral_constant<int, K>{}, std::integral_constant<int, S>{}); \
    return true;                                                                                            \
  }
  VH_FAST(MX_POT, K_INT, K_NONE)
  VH_FAST(MX_POT, K_E4M3, K_NONE)
  VH_FAST(MX_POT, K_MINI, K_NONE)
  VH_FAST(MX_SCALED, K_MINI, K_E4M3)
  VH_FAST(MX_SCALED, K_MINI, K_MINI)
  VH_FAST(MX_SCALED, K_STEPS, K_E4M3)
  VH_FAST(MX_SCALED, K_STEPS, K_MINI)
  VH_FAST(AFFINE, K_INT, K_MINI)
  VH_FAST(AFFINE, K_INT, K_NONE)
#undef VH_FAST
  return false;
}

}  // namespace
