// GEMM of at most 64 activation rows: C[M, N] = epilogue(A[M, K] . B[N, K]^T)
// with the weight B streamed once from memory.
//
// What bounds it: the weight's bytes.  So the matrix roles are turned round:
// a wave's MFMA takes 16 weight rows as its row operand and the activation's
// rows as its 16 columns.  A workgroup owns a tile of 16 NT weight rows and
// the whole of K; its eight waves take every eighth group of 64 CHUNKS bytes
// of each row and add their sums through LDS once, at the end, in wave order.
// Two groups per wave are in flight (64 to 128 KB a workgroup, against the
// ~40 KB a CU that 5 TB/s needs at 2 us of latency).  NT is the smallest for
// which one round of the CUs takes all tiles: a workgroup's first latency and
// its sum are about 1 us each, and every further round repeats them (16 rows
// of K = 4096, N = 14336 in E4M3: 18.4 us in two rounds, 15.4 in one).  Loads
// take whole 128-byte lines, eight consecutive lanes each, and reach the
// MFMA's layout (lane: one row, one chunk) through LDS of the wave's own:
// loaded in that layout directly, every lane of an access lies in another line
// than its neighbours, and 64 rows took 33.5 us where this takes 23.3.
//
// FUSED (at most 8 rows): the activation comes as bf16 and each wave
// quantizes the part of it that it multiplies, a group at a time under the
// next group's loads: the group's chunks of 16 elements are dealt over the
// lanes, so the work grows with M and not with the 16 columns of the MFMA.
// Every workgroup repeats it, which costs less than the launch that a quantize
// of its own takes as long as the rows are few: 8 rows of K = N = 4096 in a
// graph, two launches / one: E4M3 10.1 / 8.9 us, MX-int8 13.2 / 9.6; K =
// 14336: 17.3 / 19.1 (4 rows 17.0 / 14.9), 22.7 / 21.1.  Quantized once per
// workgroup into LDS before the loop, it took 1.5 us more at K = 4096 and 5 at
// K = 14336 (4 rows): nothing ran beside it.
#include "vh_skinny.h"

#include <hip/hip_runtime.h>

#include "vh_device.h"
#include "vh_epilogue.h"
#include "vh_host.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int WAVES = 8;
// 16-byte chunks per lane, row and group: the registers and LDS of two groups
// of many rows only fit with half-size groups
constexpr int chunks(int mt, int nt) { return mt >= 4 || nt >= 4 ? 2 : 4; }
constexpr int MAX_ROWS = 64;
constexpr int CUS = 256;


struct SkinnyArgs {
  const uint8_t* A;  // FUSED: bf16 rows; else rows of the stored format
  const uint8_t* B;
  void* C;
  int64_t N, lda, ldb, ldc;  // lda, ldb: row pitch in bytes; ldc: elements
  int M, K;                  // K: stored bytes of a row
  const uint8_t *a_scale, *b_scale;
  int lds_a, lds_b;          // OP_MXI8: scale bytes per row
  int a_bias, b_bias;
  const void* xs;            // FUSED FP8: the activation's scale
  int xs_dtype;
  int64_t sa, sb, sc;        // batch strides: bytes of A, B, elements of C
  vh_epilogue epi;
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t rsrc(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes > 0x7fffffff ? 0x7fffffff : (int)bytes,
                                           0x00020000);
}

__device__ __forceinline__ uint4 load16(rsrc_t r, int off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// The scale bytes of a group of n chunks (4 n bytes), in the low words.
template <int n>
__device__ __forceinline__ uint4 load_scales(rsrc_t r, int off) {
  if constexpr (n == 4) return load16(r, off);
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
  return make_uint4(v[0], v[1], 0u, 0u);
}

constexpr int PAST = (int)0x80000000;  // an offset past every resource: reads zero

// Sixteen int8 codes times a power of two as bf16, exact.
__device__ __forceinline__ void mxi8_bf16x16(const uint4& w, float s, uint32_t (&o)[8]) {
  const uint32_t d[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float f0 = (float)(int8_t)(d[i] & 0xffu) * s, f1 = (float)(int8_t)((d[i] >> 8) & 0xffu) * s;
    const float f2 = (float)(int8_t)((d[i] >> 16) & 0xffu) * s, f3 = (float)(int8_t)(d[i] >> 24) * s;
    o[2 * i] = f2bf2_hw(f0, f1);
    o[2 * i + 1] = f2bf2_hw(f2, f3);
  }
}

// quantize(x, s, qmap=fp8_e4m3) of sixteen bf16 values to E4M3 bytes: the
// steps of k_quantize_e4m3_pt (x * rcp(s) with the hardware bf16 rounding
// and fp8 converter; a product near a bf16 rounding midpoint, a NaN or an
// unusual scale sends the chunk to the correctly rounded division).
__device__ __forceinline__ uint4 e4m3_chunk(const uint4& lo, const uint4& hi, float s, float r, bool fast) {
  const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  uint32_t o[4] = {0u, 0u, 0u, 0u};
  bool slow = !fast;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float q0 = __uint_as_float(w[j] << 16) * r, q1 = __uint_as_float(w[j] & 0xffff0000u) * r;
    slow |= ((__float_as_uint(q0) - 0x7ffcu) & 0xffffu) <= 8u;
    slow |= ((__float_as_uint(q1) - 0x7ffcu) & 0xffffu) <= 8u;
    const uint32_t b = f2bf2_hw(q0, q1);
    const float v0 = __uint_as_float(b << 16), v1 = __uint_as_float(b & 0xffff0000u);
    slow |= (v0 != v0) | (v1 != v1);
    // + 0: an exact zero takes code 0 whatever its sign
    const float f0 = fminf(fmaxf(v0, -448.0f), 448.0f) + 0.0f, f1 = fminf(fmaxf(v1, -448.0f), 448.0f) + 0.0f;
    if (j & 1) o[j >> 1] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f0, f1, (int)o[j >> 1], true);
    else o[j >> 1] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f0, f1, (int)o[j >> 1], false);
  }
  if (slow) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = 0u;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float x = bf2f(j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xffffu);
      o[j >> 2] |= e4m3_hw_code(rbf(x / s)) << (8 * (j & 3));
    }
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// quantize_mx(x, int8, [-1], 16, 127, power-of-two scales) of one block of
// sixteen bf16 values, decoded: code * 2**e in bf16 (the steps of
// k_mx_pot_int_rows8, and of the decode of its packed codes, in which NaN
// is code 0).
__device__ __forceinline__ void mxi8_block(const uint4& lo, const uint4& hi, uint32_t (&o)[8]) {
  const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  // the amax as its bf16 bits: ordered as the values, NaN above infinity
  uint32_t m = 0u;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    m = umax32(m, w[j] & 0x7fffu);
    m = umax32(m, (w[j] >> 16) & 0x7fffu);
  }
  // (a block of zeros is zeros at any scale; rows past M are such blocks)
  float s = 1.0f;
  if (m != 0u && m < 0x7f80u) s = rbf(ldexpf(1.0f, floor_log2(bf2f(m)) - 6));
  if (!(s > 0.0f)) s = 1.0f;
  float q[16];
  if (m >= 0x7f80u || s < 0x1p-126f) {
    // NaN or infinite blocks, subnormal scales: element by element
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float x = bf2f(j & 1 ? w[j >> 1] >> 16 : w[j >> 1] & 0xffffu);
      const float v = m == 0x7f80u ? 0.0f : div_bf16(x, s);
      q[j] = v != v ? 0.0f : fminf(fmaxf(rintf(v), -128.0f), 127.0f);
    }
  } else {
    // |x| < 2**(E + 1): quotients are under 128 before rounding, so only
    // +128 can leave the range
    const float inv = __uint_as_float((254u << 23) - __float_as_uint(s));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t b = f2bf2_hw(__uint_as_float(w[j] << 16) * inv, __uint_as_float(w[j] & 0xffff0000u) * inv);
      q[2 * j] = fminf(rintf(__uint_as_float(b << 16)), 127.0f);
      q[2 * j + 1] = fminf(rintf(__uint_as_float(b & 0xffff0000u)), 127.0f);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = f2bf2_hw(q[2 * j] * s, q[2 * j + 1] * s);
}

// Waits for this wave's LDS accesses only (the weight loads in flight stay
// so), then meets the workgroup.
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Bytes of an activation row in a wave's LDS, and of the whole of that.
constexpr int x_pitch(int fmt, bool fused, int group) { return (fused && fmt == OP_MXI8 ? 2 : 1) * group + 16; }
constexpr int wave_lds(int fmt, int mt, int nt, bool fused) {
  const int group = 64 * chunks(mt, nt), scales = fmt == OP_MXI8 ? 16 : 0;
  return 16 * (nt * (group + 16 + scales) + mt * (x_pitch(fmt, fused, group) + (fused ? 0 : scales)));
}

// FMT: the stored format of the weight (and of the activation unless FUSED).
// MT: tiles of 16 activation rows; NT: tiles of 16 weight rows per workgroup.
// CH (FUSED, else 0): passes of the wave over a group's activation.
template <int FMT, int MT, int NT, int CH>
__global__ void __launch_bounds__(WAVES * 64) k_skinny(SkinnyArgs g) {
  constexpr bool FUSED = CH > 0;
  static_assert(!FUSED || (MT == 1 && FMT != OP_BF16), "the fused forms");
  constexpr int CHUNKS = chunks(MT, NT);
  constexpr int GROUP = 64 * CHUNKS;  // stored bytes of a row per group
  // A wave's LDS: its weight rows of one group, its activation rows (as
  // stored, or FUSED: E4M3 bytes or decoded bf16) and the scale bytes; rows
  // padded by one chunk, so that 16 rows' reads of one chunk hit all banks.
  // At the end it holds the sums.
  constexpr int P = GROUP + 16;
  constexpr int XP = x_pitch(FMT, FUSED, GROUP);
  constexpr int SP = FMT == OP_MXI8 ? 16 : 0;
  constexpr int AT_X = NT * 16 * P, AT_SW = AT_X + MT * 16 * XP, AT_SX = AT_SW + NT * 16 * SP;
  constexpr int WAVE_LDS = wave_lds(FMT, MT, NT, FUSED);
  static_assert(WAVE_LDS >= MT * NT * 1024 && WAVE_LDS == AT_SX + (FUSED ? 0 : MT * 16 * SP), "the wave's LDS");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];  // WAVES of them
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15, quad = lane >> 4;   // the MFMA's layout
  const int lrow = lane >> 3, lchunk = lane & 7; // the loads': eight lanes a line
  uint8_t* const lds = smem + wave * WAVE_LDS;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * NT);
  const int64_t bat = blockIdx.y;
  const int64_t rows_b = g.N - n0 < 16 * NT ? g.N - n0 : 16 * NT;
  const rsrc_t rb = rsrc(g.B + bat * g.sb + n0 * g.ldb, rows_b * g.ldb);
  const rsrc_t ra = rsrc(g.A + bat * g.sa, g.M * g.lda);
  rsrc_t rbs = rb, ras = ra;
  if constexpr (FMT == OP_MXI8) {
    // A group's scale bytes go past a row's end where K is no whole group:
    // the resource ends with the last row's own (in whole dwords, as the
    // pitch is), since a padded view's storage may end there too.
    const int64_t last = (g.K / 16 + 3) & ~3;
    rbs = rsrc(g.b_scale + n0 * g.lds_b, (rows_b - 1) * g.lds_b + last);
    if constexpr (!FUSED) ras = rsrc(g.a_scale, (int64_t)(g.M - 1) * g.lds_a + last);
  }

  struct Set {
    uint4 w[NT][CHUNKS], ws[NT];
    uint4 x[FUSED ? 1 : MT][CHUNKS], xs[FUSED ? 1 : MT];
  };
  // Group gi.  Load j of 16 rows: eight rows of the line j / 2 (j even: the
  // first eight).  Past K: zeros, with no memory access.
  const int woff = lrow * (int)g.ldb + lchunk * 16, xoff = lrow * (int)g.lda + lchunk * 16;
  auto load = [&](Set& s, int gi) __attribute__((always_inline)) {
    const int k0 = gi * GROUP;
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
      const int at = k0 + (j >> 1) * 128, r = (j & 1) * 8;
      const bool in = at + lchunk * 16 < g.K;
#pragma unroll
      for (int t = 0; t < NT; ++t) s.w[t][j] = load16(rb, in ? woff + (t * 16 + r) * (int)g.ldb + at : PAST);
      if constexpr (!FUSED) {
#pragma unroll
        for (int t = 0; t < MT; ++t) s.x[t][j] = load16(ra, in ? xoff + (t * 16 + r) * (int)g.lda + at : PAST);
      }
    }
    if constexpr (FMT == OP_MXI8) {  // lanes 0 .. 15: a row's scale bytes of the group
      const bool in = k0 < g.K && lane < 16;
#pragma unroll
      for (int t = 0; t < NT; ++t) s.ws[t] = load_scales<CHUNKS>(rbs, in ? (row + t * 16) * g.lds_b + k0 / 16 : PAST);
      if constexpr (!FUSED) {
#pragma unroll
        for (int t = 0; t < MT; ++t) s.xs[t] = load_scales<CHUNKS>(ras, in ? (row + t * 16) * g.lds_a + k0 / 16 : PAST);
      }
    }
  };
  // FUSED: lane takes chunk lane % CPR (16 elements) of row i RPP + lane / CPR
  constexpr int CPR = GROUP / 16, RPP = 64 / CPR;
  const int qrow = lane / CPR, qchunk = lane % CPR;
  uint4 xr[FUSED ? CH : 1][2];
  auto load_x = [&](int gi) __attribute__((always_inline)) {
    if constexpr (FUSED) {
      const int k = gi * GROUP + qchunk * 16;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int off = k < g.K ? (i * RPP + qrow) * (int)g.lda + k * 2 : PAST;
        xr[i][0] = load16(ra, off);
        xr[i][1] = load16(ra, k < g.K ? off + 16 : PAST);
      }
    }
  };
  float xs = 1.0f, xinv = 1.0f;
  bool fast = true;
  // The wave's LDS accesses execute in order; this keeps the compiler from
  // moving one lane's past another's.
  auto in_order = []() __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // A loaded group into the wave's LDS, behind its reads of the last one.
  auto stage = [&](const Set& s) __attribute__((always_inline)) {
    in_order();
#pragma unroll
    for (int j = 0; j < CHUNKS; ++j) {
      const int at = ((j & 1) * 8 + lrow) * P + (j >> 1) * 128 + lchunk * 16;
#pragma unroll
      for (int t = 0; t < NT; ++t) *(uint4*)(lds + t * 16 * P + at) = s.w[t][j];
      if constexpr (!FUSED) {
#pragma unroll
        for (int t = 0; t < MT; ++t) *(uint4*)(lds + AT_X + t * 16 * P + at) = s.x[t][j];
      }
    }
    if constexpr (FMT == OP_MXI8) {
      if (lane < 16) {
#pragma unroll
        for (int t = 0; t < NT; ++t) *(uint4*)(lds + AT_SW + (t * 16 + lane) * 16) = s.ws[t];
        if constexpr (!FUSED) {
#pragma unroll
          for (int t = 0; t < MT; ++t) *(uint4*)(lds + AT_SX + (t * 16 + lane) * 16) = s.xs[t];
        }
      }
    }
    if constexpr (FUSED) {
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        uint8_t* d = lds + AT_X + (i * RPP + qrow) * XP;
        if constexpr (FMT == OP_FP8) {
          *(uint4*)(d + qchunk * 16) = e4m3_chunk(xr[i][0], xr[i][1], xs, xinv, fast);
        } else {
          uint32_t o[8];
          mxi8_block(xr[i][0], xr[i][1], o);
          *(uint4*)(d + qchunk * 32) = make_uint4(o[0], o[1], o[2], o[3]);
          *(uint4*)(d + qchunk * 32 + 16) = make_uint4(o[4], o[5], o[6], o[7]);
        }
      }
    }
    in_order();
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const uint8_t* const wl = lds + row * P + quad * 16;          // chunk c at + 64 c
  // (an activation row past M holds anything: nobody reads its sums)
  const uint8_t* const xl = lds + AT_X + row * XP + quad * (FUSED && FMT == OP_MXI8 ? 32 : 16);
  auto compute = [&]() __attribute__((always_inline)) {
    if constexpr (FMT == OP_FP8) {
      auto two = [](const uint8_t* p) {
        const uint4 a = *(const uint4*)p, b = *(const uint4*)(p + 64);
        return i32x8{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, (int)b.z, (int)b.w};
      };
#pragma unroll
      for (int p = 0; p < CHUNKS / 2; ++p) {
        i32x8 x[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) x[i] = two(xl + i * 16 * P + 128 * p);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const i32x8 w = two(wl + j * 16 * P + 128 * p);
#pragma unroll
          for (int i = 0; i < MT; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x[i], acc[i][j], 0, 0, 0, 127, 0, 127);
        }
      }
    } else if constexpr (FMT == OP_BF16) {
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) {
        bf16x8 x[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) x[i] = *(const bf16x8*)(xl + i * 16 * P + 64 * c);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const bf16x8 w = *(const bf16x8*)(wl + j * 16 * P + 64 * c);
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x[i], acc[i][j], 0, 0, 0);
        }
      }
    } else {
      // a chunk is one block of 16: the first eight elements in one MFMA,
      // the others in the next
      auto scale = [&](int at, int tile, int c, int bias) {
        return ldexpf(1.0f, (int)lds[at + (tile * 16 + row) * 16 + 4 * c + quad] - bias);
      };
      auto half = [](const uint32_t* o) { return __builtin_bit_cast(bf16x8, make_uint4(o[0], o[1], o[2], o[3])); };
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) {
        uint32_t x[MT][8];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          if constexpr (FUSED) {
            const uint4 a = *(const uint4*)(xl + 128 * c), b = *(const uint4*)(xl + 128 * c + 16);
            x[i][0] = a.x, x[i][1] = a.y, x[i][2] = a.z, x[i][3] = a.w;
            x[i][4] = b.x, x[i][5] = b.y, x[i][6] = b.z, x[i][7] = b.w;
          } else {
            mxi8_bf16x16(*(const uint4*)(xl + i * 16 * P + 64 * c), scale(AT_SX, i, c, g.a_bias), x[i]);
          }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          uint32_t w[8];
          mxi8_bf16x16(*(const uint4*)(wl + j * 16 * P + 64 * c), scale(AT_SW, j, c, g.b_bias), w);
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(half(w), half(x[i]), acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(half(w + 4), half(x[i] + 4), acc[i][j], 0, 0, 0);
          }
        }
      }
    }
  };

  const int groups = (g.K + GROUP - 1) / GROUP;
  Set s0, s1;
  load_x(wave);  // ahead of the weight's loads: no wait for it waits for those
  load(s0, wave);
  load(s1, wave + WAVES);
  if constexpr (FUSED && FMT == OP_FP8) {
    xs = g.xs_dtype == VH_BF16 ? bf2f(*(const uint16_t*)g.xs)
         : g.xs_dtype == VH_F16 ? __half2float(*(const __half*)g.xs) : *(const float*)g.xs;
    fast = fabsf(xs) >= 0x1p-126f && fabsf(xs) <= 0x1p126f;
    xinv = __builtin_amdgcn_rcpf(xs);
  }
  __builtin_amdgcn_sched_barrier(0);
  for (int gi = wave; gi < groups; gi += 2 * WAVES) {
    stage(s0);
    load_x(gi + WAVES);
    load(s0, gi + 2 * WAVES);
    __builtin_amdgcn_sched_barrier(0);
    compute();
    if (gi + WAVES < groups) {
      stage(s1);
      load_x(gi + 2 * WAVES);
      load(s1, gi + 3 * WAVES);
      __builtin_amdgcn_sched_barrier(0);
      compute();
    }
  }

  // the waves' sums, each in its own LDS
  in_order();
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) *(f32x4*)(lds + (i * NT + j) * 1024 + lane * 16) = acc[i][j];
  const vh_epilogue& e = g.epi;
  const float sc = epi_scale(e);
  lds_sync();
  for (int t = threadIdx.x; t < MT * NT * 64; t += WAVES * 64) {
    // MFMA output: lane holds weight rows 4 (lane / 16) .. + 3 of activation row lane % 16
    const int tile = t >> 6;
    const int m = tile / NT * 16 + (t & 15);
    const int64_t n = n0 + (tile % NT) * 16 + ((t >> 4) & 3) * 4;
    if (m >= g.M) continue;
    f32x4 v = *(const f32x4*)(smem + t * 16);
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += *(const f32x4*)(smem + w * WAVE_LDS + t * 16);
    const int64_t at = bat * g.sc + m * g.ldc + n;
    float r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = n + u < g.N ? epi_value(e, v[u], sc, epi_bias(e, n + u)) : 0.0f;
    if (e.out_dtype == VH_BF16) {
      uint16_t* c = (uint16_t*)g.C + at;
      const uint32_t b0 = f2bf(r[0]) | (f2bf(r[1]) << 16), b1 = f2bf(r[2]) | (f2bf(r[3]) << 16);
      if (n + 4 <= g.N && ((uintptr_t)c & 7) == 0) {
        *(uint2*)c = make_uint2(b0, b1);
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (n + u < g.N) c[u] = (uint16_t)((u & 2 ? b1 : b0) >> (16 * (u & 1)));
      }
    } else {
      float* c = (float*)g.C + at;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (n + u < g.N) c[u] = r[u];
    }
  }
}

template <int FMT, int MT, int NT, int CH>
int launch_as(const SkinnyArgs& g, int64_t batch, vh_stream_t stream, const char* what) {
  const int64_t wgs = (g.N + 16 * NT - 1) / (16 * NT);
  VH_REQUIRE(wgs < (1ll << 31), "%s: N too large", what);
  constexpr int smem = WAVES * wave_lds(FMT, MT, NT, CH > 0);
  static_assert(smem <= 160 * 1024, "LDS");
  static const hipError_t reserved =
      hipFuncSetAttribute((const void*)k_skinny<FMT, MT, NT, CH>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (reserved != hipSuccess) {
    vh::set_error("%s: cannot reserve %d bytes of LDS", what, smem);
    return VH_ELAUNCH;
  }
  hipLaunchKernelGGL((k_skinny<FMT, MT, NT, CH>), dim3((unsigned)wgs, (unsigned)batch), dim3(WAVES * 64), smem,
                     vh::as_stream(stream), g);
  return vh::check_launch(what);
}

// The smallest NT that takes one round of the CUs (64 rows: as far as the
// registers go).  FUSED: the activation's passes over a group, which is half
// as long at NT = 4.
template <int FMT, int MT, bool FUSED>
int launch(const SkinnyArgs& g, int64_t batch, vh_stream_t stream, const char* what) {
  const int64_t tiles = (g.N + 15) / 16 * batch;
  const bool two = FUSED && g.M > 4;  // (g.M <= 8)
  if constexpr (MT < 4) {
    if (tiles > 2 * CUS) return launch_as<FMT, MT, 4, FUSED ? 1 : 0>(g, batch, stream, what);
  }
  if constexpr (FMT != OP_MXI8 || MT < 4) {
    if (tiles > CUS) {
      if constexpr (FUSED) {
        if (two) return launch_as<FMT, MT, 2, 2>(g, batch, stream, what);
      }
      return launch_as<FMT, MT, 2, FUSED ? 1 : 0>(g, batch, stream, what);
    }
  }
  if constexpr (FUSED) {
    if (two) return launch_as<FMT, MT, 1, 2>(g, batch, stream, what);
  }
  return launch_as<FMT, MT, 1, FUSED ? 1 : 0>(g, batch, stream, what);
}

template <int FMT>
int launch_rows(const SkinnyArgs& g, int64_t batch, vh_stream_t stream, const char* what) {
  if (g.M <= 16) return launch<FMT, 1, false>(g, batch, stream, what);
  if (g.M <= 32) return launch<FMT, 2, false>(g, batch, stream, what);
  return launch<FMT, 4, false>(g, batch, stream, what);
}

// A scale byte's power of two as bf16 operands take it: 2**(byte - bias)
// finite in float32 (bias >= 128) and code * 2**(byte - bias) exact in bf16
// (bias <= 133), as int8's 133 is.
bool bias_ok(int bias) { return bias >= 128 && bias <= 133; }

int check_epilogue(const vh_epilogue* e, int mode, const char* what) {
  VH_REQUIRE(e->mode == mode && (e->out_dtype == VH_BF16 || e->out_dtype == VH_F32), "%s: unsupported epilogue", what);
  VH_REQUIRE(!e->scale || e->scale_dtype == VH_BF16 || e->scale_dtype == VH_F32, "%s: scale must be bf16 or float32",
             what);
  VH_REQUIRE(!e->bias || e->bias_dtype == VH_BF16 || e->bias_dtype == VH_F32, "%s: bias must be bf16 or float32", what);
  return VH_OK;
}

int check_rows8(const void* x, int64_t ldx, const uint8_t* w, int64_t ldw, int64_t M, int64_t N, int64_t K,
                 const vh_epilogue* epi, const void* y, int64_t ldy, int mode, const char* what) {
  VH_REQUIRE(x && w && epi && y, "%s: null argument", what);
  VH_REQUIRE(M >= 1 && M <= 8, "%s: M must be in [1, 8] (got %lld)", what, (long long)M);
  VH_REQUIRE(N > 0 && K > 0 && K % 16 == 0, "%s: needs K a multiple of 16", what);
  VH_REQUIRE(ldx >= K && ldx % 8 == 0 && ldw >= K && ldw % 16 == 0 && ldy >= N, "%s: bad row pitch", what);
  VH_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0, "%s: misaligned operand", what);
  VH_REQUIRE(ldx * 512 < (1ll << 31) && ldw * 256 < (1ll << 31), "%s: rows too long for 32-bit offsets", what);
  return check_epilogue(epi, mode, what);
}

SkinnyArgs rows8_args(const uint16_t* x, int64_t ldx, const uint8_t* w, int64_t ldw, int64_t M, int64_t N, int64_t K,
                       const vh_epilogue* epi, void* y, int64_t ldy) {
  SkinnyArgs g{};
  g.A = (const uint8_t*)x;
  g.B = w;
  g.C = y;
  g.M = (int)M;
  g.N = N;
  g.K = (int)K;
  g.lda = ldx * 2;
  g.ldb = ldw;
  g.ldc = ldy;
  g.epi = *epi;
  return g;
}

}  // namespace

namespace vh {

bool skinny_fits(const vh_gemm_desc* d) {
  if (d->M > MAX_ROWS || d->a_fmt != d->b_fmt || d->lda % 16 || d->ldb % 16 || d->K <= 0) return false;
  if (d->a_fmt == OP_FP8 || d->a_fmt == OP_BF16) return true;
  if (d->a_fmt != OP_MXI8) return false;
  auto al = [](const void* p, int64_t ld) { return (uintptr_t)p % 4 == 0 && ld % 4 == 0; };
  return d->batch <= 1 && d->a_block == 16 && d->b_block == 16 && d->K % 16 == 0 && bias_ok(d->a_bias) &&
         bias_ok(d->b_bias) && al(d->a_scale, d->a_scale_ld) && al(d->b_scale, d->b_scale_ld) &&
         d->a_scale_ld < (1 << 20) && d->b_scale_ld < (1 << 20);
}

bool skinny_taken(const vh_gemm_desc* d) {
  // Measured on MI355X, weights from HBM: this kernel / the tiled ones in us (*
  // where those are taken).
  //                    K   N = 4096                   14336                      32768
  //                        16 rows       64           16            64           16            64
  //   E4M3           512    4.0 /  4.8    4.8 /  5.0    5.2 /  5.1*   9.1 /  5.3*   9.3 /  6.4*  16.9 /  7.1*
  //                 2048    4.9 /  7.3    6.5 /  7.7    9.2 /  9.9   13.8 /  9.3*  16.9 / 13.7*  26.9 / 14.4*
  //                 4096    6.8 / 12.2    9.7 / 15.2   12.9 / 13.0   19.2 / 13.7*  26.1 / 22.7*  39.4 / 24.1*
  //                14336   12.6 / 27.9   19.1 / 32.3   31.6 / 32.9   42.3 / 36.2*
  //   bf16           512    4.2 /  5.2    5.2 /  5.4    6.7 /  6.6*  11.5 /  7.0*  12.4 /  9.6*  22.0 / 10.5*
  //                 2048    7.1 / 13.0   10.2 / 13.7   15.7 / 16.6   23.4 / 17.4*  31.9 / 34.5*  46.1 / 35.3*
  //                 4096   10.1 / 22.2   15.9 / 23.6   26.4 / 29.1   37.8 / 30.7*  55.7 / 61.6   76.4 / 62.7*
  //                14336   26.5 / 69.0   46.8 / 75.7   80.0 / 94.2    118 /  100*
  //   MX-int8        128    4.3 /  5.3    5.4 /  5.4*   5.5 /  6.0   17.3 /  6.2*   9.2 / 10.4*  32.7 / 11.1*
  //                  512    4.7 /  9.2    5.9 / 10.9    6.2 / 11.4   18.3 / 16.1*  11.3 / 17.2   34.8 / 17.9*
  //                 4096    9.2 / 15.9   15.8 / 19.2   18.4 / 33.4   53.2 / 36.0*  36.3 / 75.8    111 / 77.7*
  //                14336   18.8 / 30.8   37.1 / 31.9*  41.5 / 95.7    135 / 98.0*
  //   batches of bf16      1 row         16           32            64
  //   256 of (1024, 128)    47.1 / 31.0*  48.2 / 31.9*  54.9 / 33.1*   103 / 36.2*
  //   32 of (1024, 512)     12.4 /  9.8*  12.9 /  9.9*  14.5 / 10.4*  22.4 / 11.7*
  //   8 of (512, 512)        4.2 /  5.2    4.3 /  5.2    4.8 /  5.3*   5.5 /  5.5*
  //   32 of (1024, 4096)    54.1 / 68.0   56.3 / 68.0   58.4 / 68.2   80.6 / 70.0*
  // One round of the CUs at NT = 1 (256 weight tiles) pays at any K; a second
  // set of columns or a second round repeats each workgroup's latency and sum
  // (about 2 us) and needs a K whose stream covers it; from a third on the
  // last round has to be nearly full as well, and E4M3's tiles, twice as fast
  // as bf16's, are then even or better.  More rows cost this kernel more than
  // the tiles, most of all in a batch, whose every product has its own.  Over
  // 7035 sizes (K = 64 .. 14336, N = 64 .. 65536, 1 .. 64 rows, batches of 1
  // .. 256) the choice is 0.6% above the faster kernel on average; any K and,
  // to 32 rows, any grid, as before, 9.7%.
  if (d->tile_hint == VH_GEMM_TILE_SKINNY) return skinny_fits(d);
  if (d->tile_hint != 0 || d->split_k != 0 || d->N <= 0 || !skinny_fits(d)) return false;
  const int64_t batch = d->batch < 1 ? 1 : d->batch, K = d->K, N = d->N;
  const int64_t t = (N + 15) / 16 * batch;  // tiles of 16 weight rows
  const bool many = d->M > 16, most = d->M > 32;
  const int64_t rounds = (t + 4 * CUS - 1) / (4 * CUS);  // at NT = 4
  const int64_t fill = t * 20 / (rounds * 4 * CUS);      // of them, in twentieths
  if (d->a_fmt == OP_MXI8) {
    if (most && (N > 4096 || K > 4096)) return false;
    return K >= (rounds > 1 && fill < 18 ? 1024 : many || rounds > 1 ? 256 : 128);
  }
  if (K < 2048) {
    if (t <= CUS) return batch == 1 || t <= (most ? 64 : many ? 128 : CUS);
    return t <= 2 * CUS && !many;
  }
  if (t <= CUS) return !most || batch == 1 || N >= 512 || t <= 128;
  if (t <= 2 * CUS) return !most || batch == 1 || N >= 1024;
  if (most) return false;
  return rounds == 1 || (d->a_fmt == OP_BF16 && K >= 4096 && fill >= 17);
}

int skinny_gemm(const vh_gemm_desc* d, vh_stream_t stream) {
  SkinnyArgs g{};
  g.A = (const uint8_t*)d->A;
  g.B = (const uint8_t*)d->B;
  g.C = d->C;
  g.M = (int)d->M;
  g.N = d->N;
  g.K = (int)(d->a_fmt == OP_BF16 ? d->K * 2 : d->K);
  g.lda = d->lda;
  g.ldb = d->ldb;
  g.ldc = d->ldc;
  g.a_scale = (const uint8_t*)d->a_scale;
  g.b_scale = (const uint8_t*)d->b_scale;
  g.lds_a = (int)d->a_scale_ld;
  g.lds_b = (int)d->b_scale_ld;
  g.a_bias = d->a_bias;
  g.b_bias = d->b_bias;
  g.sa = d->batch_stride_a;
  g.sb = d->batch_stride_b;
  g.sc = d->batch_stride_c;
  g.epi = d->epi;
  const int64_t batch = d->batch < 1 ? 1 : d->batch;
  if (d->a_fmt == OP_FP8) return launch_rows<OP_FP8>(g, batch, stream, "vh_gemm");
  if (d->a_fmt == OP_BF16) return launch_rows<OP_BF16>(g, batch, stream, "vh_gemm");
  return launch_rows<OP_MXI8>(g, batch, stream, "vh_gemm");
}

}  // namespace vh

extern "C" int vh_linear_fp8_rows8(const uint16_t* x, int64_t ldx, const void* x_scale, int32_t x_scale_dtype,
                                    const uint8_t* w, int64_t ldw, int64_t M, int64_t N, int64_t K,
                                    const vh_epilogue* epi, void* y, int64_t ldy, vh_stream_t stream) {
  const char* what = "vh_linear_fp8_rows8";
  int rc;
  if ((rc = check_rows8(x, ldx, w, ldw, M, N, K, epi, y, ldy, EPI_ROUND_SCALE, what))) return rc;
  VH_REQUIRE(x_scale && vh::is_float_dtype(x_scale_dtype), "%s: needs a float scale", what);
  SkinnyArgs g = rows8_args(x, ldx, w, ldw, M, N, K, epi, y, ldy);
  g.xs = x_scale;
  g.xs_dtype = x_scale_dtype;
  return launch<OP_FP8, 1, true>(g, 1, stream, what);
}

extern "C" int vh_linear_mxint8_rows8(const uint16_t* x, int64_t ldx, const uint8_t* w, int64_t ldw,
                                       const uint8_t* w_scale, int64_t ldws, int32_t w_bias, int64_t M, int64_t N,
                                       int64_t K, const vh_epilogue* epi, void* y, int64_t ldy, vh_stream_t stream) {
  const char* what = "vh_linear_mxint8_rows8";
  int rc;
  if ((rc = check_rows8(x, ldx, w, ldw, M, N, K, epi, y, ldy, EPI_PLAIN, what))) return rc;
  VH_REQUIRE(w_scale && (uintptr_t)w_scale % 4 == 0 && ldws % 4 == 0 && ldws >= K / 16 && ldws < (1 << 20),
             "%s: scale rows must be 4-byte aligned and hold K / 16 bytes", what);
  VH_REQUIRE(bias_ok(w_bias), "%s: scale bias must be in [128, 133]", what);
  SkinnyArgs g = rows8_args(x, ldx, w, ldw, M, N, K, epi, y, ldy);
  g.b_scale = w_scale;
  g.lds_b = (int)ldws;
  g.b_bias = w_bias;
  return launch<OP_MXI8, 1, true>(g, 1, stream, what);
}
