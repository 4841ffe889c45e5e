// hh_gemm_f4.hip — batched (prefill) GEMM of the 1- and 2-bit weight formats on
// the f8f6f4 matrix instructions of gfx950.
//
// Semantics: out[s*n + r] = dot_fn(w + r*row_bytes, x + s*q8_stride, K) for
// every token s < seq and row r < n: par_dot_rows_batched with DotFn / DotFn2
// (pool.rs:40-80, :568-618; matmul.rs:580-674), whose paired kernels are
// bit-identical to the single-token dot (q2_0.rs:936-986).  Here too: every
// 32-element sub-block dot is exact, and the fp32 combine follows the scalar
// kernels (q2_0.rs:537-574, q1_0g128.rs:1113-1152):
//   block_acc = ((i0*da0 + i1*da1) + i2*da2) + i3*da3;  sum += block_acc * dw
// so each output equals the decode GEMV's bit for bit.
//
// One v_mfma_scale_f32_32x32x64_f8f6f4 gives the sub-block dots of 32 weight
// rows x 32 tokens as floats.  An int8 activation a is sign * (16 h + l) with
// h <= 8 and l <= 15; the FP6 e2m3 code sign:n, n < 16, is sign * n / 8, so the
// instruction's K = 64 takes the 32 h codes (block scale 2^7) and the 32 l
// codes (2^3), each against the sub-block's 32 weights in FP4 (-0.5, 0, 0.5, 1
// with block scale 2).  Products are integers and every sum stays below 2^24:
// the result is the sub-block's exact dot, already the float that the combine
// multiplies (the int8 instructions needed a convert per output).
//
// What bounds it: the combine, 6 VALU operations per output and 128-weight block (the
// int8 form took 9); the matrix pipe is busy about a third as long.  8B gate+up
// (24576 x 4096, Q2_0) over 2048 tokens: int8 form 791 us, here 417 us, of which the
// combine alone would take 0.25 ms.
#include "hh_kernels.h"

#include <algorithm>

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32x3_a4 __attribute__((ext_vector_type(3), aligned(4)));

// Activation tile: 32 tokens x 128 columns, the same bytes in memory and LDS.
//   [sub 4][half 2][token 32] 16 B : slots 0..20 of the half's 32 FP6 codes and 2 bits
//   [sub 4][half 2][token 32]  8 B : the rest (24 B are 32 codes, slot j at bit 6j)
//   [token 32][sub 4] f32          : the Q8_0 scales
// Every lane group of an operand read is then contiguous (no bank conflicts),
// and a workgroup's token groups of one column block are one contiguous copy.
constexpr int AT_HI = 4096, AT_D = 6144, AT_BYTES = 6656;
static_assert(AT_BYTES == HH_ACT_TILE_BYTES, "activation tile size");

// Slot order of the 32 codes of a sub-block: what the weight format's bit
// extraction yields.  Slot 8j + i is nibble i of the operand's dword j:
//   Q2 : element 16 (j / 2) + 2 i + j % 2     ((D >> 2 (j % 2)) & 0x33333333)
//   Q1 : element 4 i + j                      ((D >> j) & 0x11111111)
//   PT : element 16 (i % 2) + 4 j + i / 2     (two dwords of byte-wide trits)
HH_DEV void slot_words(int fmt, const uint32_t w[8], uint32_t s[8]) {   // 4 slots (bytes) per word
  if (fmt == FMT_Q2) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int b = 4 * (j / 2) + 2 * q;
        s[2 * j + q] = __builtin_amdgcn_perm(w[b + 1], w[b], j % 2 ? 0x07050301u : 0x06040200u);
      }
  } else if (fmt == FMT_Q1) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {   // 4x4 byte transposes
      const uint32_t a = w[4 * q], b = w[4 * q + 1], c = w[4 * q + 2], d = w[4 * q + 3];
      const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u), ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
      const uint32_t cd0 = __builtin_amdgcn_perm(d, c, 0x05010400u), cd1 = __builtin_amdgcn_perm(d, c, 0x07030602u);
      s[0 + q] = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
      s[2 + q] = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
      s[4 + q] = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
      s[6 + q] = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[2 * j] = __builtin_amdgcn_perm(w[4 + j], w[j], 0x05010400u);
      s[2 * j + 1] = __builtin_amdgcn_perm(w[4 + j], w[j], 0x07030602u);
    }
  }
}

// 4 bytes of 6 bits -> 24 bits.
HH_DEV uint32_t pack6(uint32_t b) {
  const uint32_t t = (b & 0x003f003fu) | ((b >> 2) & 0x0fc00fc0u);
  return (t & 0xfffu) | ((t >> 4) & 0xfff000u);
}

// One sub-block of one token into its tile.  w: 32 int8, element order.
HH_DEV void put_sub_block(uint8_t* __restrict__ tile, int fmt, int sub, int tok, const uint32_t w[8], float d) {
  uint32_t s[8], u[2][8];
  slot_words(fmt, w, s);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t sg = (s[i] >> 7) & 0x01010101u;
    const uint32_t m = (s[i] ^ (sg * 0xffu)) + sg;   // |a| per byte (128 for -128; no carries)
    u[0][i] = pack6(((m >> 4) & 0x0f0f0f0fu) | (sg << 5));
    u[1][i] = pack6((m & 0x0f0f0f0fu) | (sg << 5));
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t* v = u[h];
    const uint32_t d0 = v[0] | (v[1] << 24), d1 = (v[1] >> 8) | (v[2] << 16), d2 = (v[2] >> 16) | (v[3] << 8);
    const uint32_t d3 = v[4] | (v[5] << 24), d4 = (v[5] >> 8) | (v[6] << 16), d5 = (v[6] >> 16) | (v[7] << 8);
    const int at = (sub * 2 + h) * 32 + tok;
    *(uint4*)(tile + at * 16) = make_uint4(d0, d1, d2, d3);
    *(uint2*)(tile + AT_HI + at * 8) = make_uint2(d4, d5);
  }
  *(float*)(tile + AT_D + (tok * 4 + sub) * 4) = d;
}

// Activation rows -> tiles, tile (kb, token group) at (kb * n_groups + group).
// STD: standard Q8_0 blocks (x); else int8 rows xq and f32 scales xd.  Rows past
// seq are zeros.  One workgroup per tile, one lane per (token, sub-block).
template <int FMT, bool STD>
__global__ __launch_bounds__(128) void k_act_tiles(const uint8_t* __restrict__ x, const int8_t* __restrict__ xq,
                                                   const float* __restrict__ xd, int K, int seq,
                                                   int n_groups, uint8_t* __restrict__ tiles) {
  const int kb = blockIdx.x / n_groups, g = blockIdx.x % n_groups;
  const int tok = threadIdx.x & 31, sub = threadIdx.x >> 5, s = g * 32 + tok;
  uint32_t w[8];
  float d = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) w[i] = 0;
  if (s < seq) {
    const size_t b = (size_t)s * (K / 32) + kb * 4 + sub;
    if constexpr (STD) {
      const uint8_t* blk = x + b * 34;
      const u32x4_a2 a0 = *(const u32x4_a2*)(blk + 2), a1 = *(const u32x4_a2*)(blk + 18);
#pragma unroll
      for (int i = 0; i < 4; ++i) { w[i] = a0[i]; w[4 + i] = a1[i]; }
      d = h2f(*(const uint16_t*)blk);
    } else {
      const uint4 a0 = *(const uint4*)(xq + b * 32), a1 = *(const uint4*)(xq + b * 32 + 16);
      w[0] = a0.x; w[1] = a0.y; w[2] = a0.z; w[3] = a0.w;
      w[4] = a1.x; w[5] = a1.y; w[6] = a1.z; w[7] = a1.w;
      d = xd[b];
    }
  }
  put_sub_block(tiles + (size_t)blockIdx.x * AT_BYTES, FMT, sub, tok, w, d);
}

// ---- weights: one row's 128-weight block -> FP4 operand words ----
// FP4 e2m1 nibbles at half scale: 0x9 = -0.5, 0x0 = 0, 0x1 = 0.5, 0x2 = 1.
constexpr uint32_t FP4_OF_CODE = 0x02010009u;   // byte c: code c (value (c - 1) / 2)

template <int FMT> constexpr int blk_bytes() { return FMT == FMT_Q1 ? 18 : FMT == FMT_PT ? 28 : 34; }
template <int FMT> constexpr int scale_off() { return FMT == FMT_PT ? 26 : 0; }

// Half a block (sub-blocks 2 half, 2 half + 1) as loaded.
template <int FMT> struct WRaw { uint32_t v[FMT == FMT_Q2 ? 4 : FMT == FMT_Q1 ? 2 : 7]; };

template <int FMT> HH_DEV void w_load(WRaw<FMT>& R, const uint8_t* __restrict__ blk, int half) {
  if constexpr (FMT == FMT_Q2) {
    const u32x4_a2 a = *(const u32x4_a2*)(blk + 2 + 16 * half);
#pragma unroll
    for (int i = 0; i < 4; ++i) R.v[i] = a[i];
  } else if constexpr (FMT == FMT_Q1) {
    const u32x2_a2 a = *(const u32x2_a2*)(blk + 2 + 8 * half);
    R.v[0] = a[0]; R.v[1] = a[1];
  } else {
    const u32x4_a4 a = *(const u32x4_a4*)blk;
    const u32x3_a4 b = *(const u32x3_a4*)(blk + 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) R.v[i] = a[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) R.v[4 + i] = b[i];
  }
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// PTQ1_0 (ptq1_0.rs:1-13): trit n of byte b is ((b * 3^n mod 256) * 3) >> 8.
// The trits n of 4 bytes as 4 bytes, from the bytes' even and odd 16-bit lanes
// already multiplied by 3^n mod 256.
HH_DEV uint32_t pt_trits(u16x2 lo, u16x2 hi) {
  const u16x2 three = {3, 3}, eight = {8, 8};
  return __builtin_bit_cast(uint32_t, (u16x2)((lo * three) >> eight)) |
         (__builtin_bit_cast(uint32_t, (u16x2)((hi * three) >> eight)) << 8);
}
HH_DEV uint32_t pt_at(uint32_t q, int pow3) {   // trits of the 4 bytes of q at 3^n = pow3
  const unsigned short p = (unsigned short)pow3;
  const u16x2 m = {p, p};
  const u16x2 lo = __builtin_bit_cast(u16x2, q & 0x00ff00ffu) * m;
  const u16x2 hi = __builtin_bit_cast(u16x2, (q >> 8) & 0x00ff00ffu) * m;
  return pt_trits(__builtin_bit_cast(u16x2, __builtin_bit_cast(uint32_t, lo) & 0x00ff00ffu),
                  __builtin_bit_cast(u16x2, __builtin_bit_cast(uint32_t, hi) & 0x00ff00ffu));
}
// two dwords of 4 trits -> 8 FP4 nibbles (a in the even, b in the odd)
HH_DEV uint32_t pt_word(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(0u, FP4_OF_CODE, a) | (__builtin_amdgcn_perm(0u, FP4_OF_CODE, b) << 4);
}

// The operand words of sub-blocks 2 half and 2 half + 1: out[4 sub + j].
template <int FMT> HH_DEV void w_expand(const WRaw<FMT>& R, int half, uint32_t out[8]) {
  if constexpr (FMT == FMT_Q2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t p[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)   // codes k, k + 4, k + 8, k + 12 of the dword
        p[k] = __builtin_amdgcn_perm(0u, FP4_OF_CODE, (R.v[i] >> (2 * k)) & 0x03030303u);
      out[2 * i] = p[0] | (p[2] << 4);       // codes 0, 2, 4, ..
      out[2 * i + 1] = p[1] | (p[3] << 4);   // codes 1, 3, 5, ..
    }
  } else if constexpr (FMT == FMT_Q1) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t nb = ~R.v[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) out[4 * i + k] = ((nb << (3 - k)) & 0x88888888u) | 0x11111111u;
    }
  } else {
    // half 0: trits 0..3 of bytes 0..15 (elements 0..63); half 1: trit 4 of those, the
    // trits of bytes 16..23 (elements 64..119) and the 4 trits of bytes 24, 25 (element
    // 120 + 2n + h) from the dword e of the bytes and their 3-multiples.  The lane picks
    // the inputs, so both halves run the same 16 unpackings.
    const bool hi = half != 0;
    auto pick = [&](uint32_t q0, int p0, uint32_t q1, int p1) { return pt_at(hi ? q1 : q0, hi ? p1 : p0); };
    const uint32_t qh = R.v[6] & 0xffffu;
    const u16x2 q3 = __builtin_bit_cast(u16x2, (qh & 0xffu) | ((qh & 0xff00u) << 8)) * u16x2{3, 3};
    const uint32_t q3w = __builtin_bit_cast(uint32_t, q3);
    const uint32_t e = qh | ((q3w & 0xffu) << 16) | ((q3w & 0xff0000u) << 8);
    const uint32_t* v = R.v;
    out[0] = pt_word(pick(v[0], 1, v[0], 81), pick(v[0], 3, v[4], 1));
    out[1] = pt_word(pick(v[1], 1, v[1], 81), pick(v[1], 3, v[5], 1));
    out[2] = pt_word(pick(v[2], 1, v[2], 81), pick(v[2], 3, v[4], 3));
    out[3] = pt_word(pick(v[3], 1, v[3], 81), pick(v[3], 3, v[5], 3));
    out[4] = pt_word(pick(v[0], 9, v[4], 9), pick(v[0], 27, v[4], 81));
    out[5] = pt_word(pick(v[1], 9, v[5], 9), pick(v[1], 27, v[5], 81));
    out[6] = pt_word(pick(v[2], 9, v[4], 27), pick(v[2], 27, e, 1));
    out[7] = pt_word(pick(v[3], 9, v[5], 27), pick(v[3], 27, e, 9));
  }
}

HH_DEV i32x8 op_fp4(u32x4 v) { return i32x8{(int)v[0], (int)v[1], (int)v[2], (int)v[3], 0, 0, 0, 0}; }
HH_DEV i32x8 op_fp6(u32x4 v, u32x2 t) {
  return i32x8{(int)v[0], (int)v[1], (int)v[2], (int)v[3], (int)t[0], (int)t[1], 0, 0};
}

// Sub-block dots of 32 rows (weights a) x 32 tokens (activations b): lane l holds
// token l % 32, rows 8 (i / 4) + 4 (l / 32) + i % 4.  scale_b: 2^7 for the lanes
// of the h codes (l < 32), 2^3 for those of the l codes.
HH_DEV f32x16 sub_dots(i32x8 a, i32x8 b, int scale_b) {
  const f32x16 z = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, z, 4, 2, 0, 128, 0, scale_b);
}

// The block accumulator of output i: |dot| <= 2^13 and da has an f16's 11
// significant bits, so dot * da is exact in f32 and each fma rounds once, as the
// scalar order's add does.
HH_DEV float block_sum(const f32x16 c[4], int i, f32x4 da) {
  float acc = c[0][i] * da[0];
  acc = fmaf(c[1][i], da[1], acc);
  acc = fmaf(c[2][i], da[2], acc);
  return fmaf(c[3][i], da[3], acc);
}

// A 32 x 32 tile of outputs (rows row0.., tokens tok0..); vec: n % 4 == 0 and out
// 16-byte aligned.
HH_DEV void store_tile(float* __restrict__ out, const f32x16& v, int row0, int tok0, int n, int seq, int vec) {
  const int l32 = threadIdx.x & 31, lh = (threadIdx.x >> 5) & 1, s = tok0 + l32, row = row0 + 4 * lh;
  if (s >= seq) return;
  float* o = out + (size_t)s * n + row;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (vec) {
      if (row + 8 * q < n) *(float4*)(o + 8 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (row + 8 * q + j < n) o[8 * q + j] = v[4 * q + j];
    }
  }
}

// The product straight from the GGUF blocks: WR waves of 32 rows,
// all on the same 32 tokens.  Per 128-column step the activation tile is copied to
// LDS and the weight blocks are expanded there; two LDS buffers, the next step's
// global loads in registers over the whole compute of the current one.
template <int FMT, int WR>
__global__ __launch_bounds__(64 * WR, 2) void k_gemm_f4(const uint8_t* __restrict__ w,
                                                        const uint8_t* __restrict__ tiles, float* __restrict__ out,
                                                        int n, int K, int seq, int n_groups, int vec_out) {
#pragma clang fp contract(off)
  constexpr int NT = 64 * WR, R = 32 * WR, NP = AT_BYTES / 16, PL = (NP + NT - 1) / NT;
  struct Stage {
    uint8_t a[AT_BYTES];
    uint32_t w[4][R][4];   // [sub][row] FP4 operand
    float dw[R];
  };
  __shared__ __align__(16) Stage st[2];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, l32 = lane & 31, lh = lane >> 5;
  const int n_rows = (n + R - 1) / R, r0 = blockIdx.x % n_rows * R, g = blockIdx.x / n_rows;
  const int nsteps = K / 128, scale_b = lh ? 130 : 134;
  const int row = tid % R, half = tid / R;   // this lane's half block per step (the half is wave-uniform)
  const uint8_t* ab = tiles + (size_t)g * AT_BYTES;
  const size_t a_step = (size_t)n_groups * AT_BYTES;
  const uint8_t* wp = w + (size_t)min(r0 + row, n - 1) * ((size_t)(K / 128) * blk_bytes<FMT>());
  u32x4 av[PL];
  WRaw<FMT> wv;
  uint32_t ws = 0;
  auto load = [&](int kb) {
    const uint8_t* blk = wp + (size_t)kb * blk_bytes<FMT>();
    w_load<FMT>(wv, blk, half);
    ws = *(const uint16_t*)(blk + scale_off<FMT>());
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const uint8_t* base = ab + (size_t)kb * a_step + 16 * NT * i;   // uniform
      const int p = (i + 1) * NT <= NP ? tid : min(tid, NP - 1 - NT * i);
      av[i] = *(const u32x4*)(base + (uint32_t)(16 * p));
    }
  };
  auto store = [&](Stage& S) {
    uint32_t o[8];
    w_expand<FMT>(wv, half, o);
    *(uint4*)S.w[2 * half][row] = make_uint4(o[0], o[1], o[2], o[3]);
    *(uint4*)S.w[2 * half + 1][row] = make_uint4(o[4], o[5], o[6], o[7]);
    if (half == 0) S.dw[row] = h2f(ws);
#pragma unroll
    for (int i = 0; i < PL; ++i)
      if (tid + NT * i < NP) *(u32x4*)(S.a + (tid + NT * i) * 16) = av[i];
  };
  f32x16 sum;
#pragma unroll
  for (int i = 0; i < 16; ++i) sum[i] = 0.0f;
  load(0);
  store(st[0]);
  if (nsteps > 1) load(1);
  __syncthreads();
  for (int kb = 0; kb < nsteps; ++kb) {
    const Stage& S = st[kb & 1];
    if (kb + 1 < nsteps) store(st[(kb + 1) & 1]);
    if (kb + 2 < nsteps) load(kb + 2);
    f32x16 c[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int p = (s * 2 + lh) * 32 + l32;
      c[s] = sub_dots(op_fp4(*(const u32x4*)S.w[s][wid * 32 + l32]),
                      op_fp6(*(const u32x4*)(S.a + p * 16), *(const u32x2*)(S.a + AT_HI + p * 8)), scale_b);
    }
    const f32x4 da = *(const f32x4*)(S.a + AT_D + l32 * 16);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 dw = *(const f32x4*)(S.dw + wid * 32 + 8 * q + 4 * lh);
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[4 * q + j] += block_sum(c, 4 * q + j, da) * dw[j];
    }
    __syncthreads();
  }
  store_tile(out, sum, r0 + wid * 32, g * 32, n, seq, vec_out);
}

// The same for a grid too small to fill the CUs that way: one 32 x 32 tile per
// workgroup of 8 waves.  A round takes 16 column blocks, two per wave: the wave loads
// and expands its own weights and activations, and leaves its block accumulators in
// LDS; after the barrier every lane adds its two outputs' 16 block products in block
// order (sum += acc * dw, the scalar order).  So a short prompt still spreads a
// matrix over all CUs, with one memory round trip per 2048 columns.
template <int FMT>
__global__ __launch_bounds__(512, 2) void k_gemm_f4s(const uint8_t* __restrict__ w,
                                                     const uint8_t* __restrict__ tiles, float* __restrict__ out,
                                                     int n, int K, int seq, int n_groups, int vec_out) {
#pragma clang fp contract(off)
  constexpr int NB = 16;
  __shared__ __align__(16) float acc[NB][4][64][4];   // [block][output / 4][lane][output % 4]
  __shared__ float dws[NB][32];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, l32 = lane & 31, lh = lane >> 5;
  const int n_rt = (n + 31) / 32, r0 = blockIdx.x % n_rt * 32, g = blockIdx.x / n_rt;
  const int nkb = K / 128, scale_b = lh ? 130 : 134;
  const uint8_t* wrow = w + (size_t)min(r0 + l32, n - 1) * ((size_t)nkb * blk_bytes<FMT>());
  const int q = wid >> 1, j0 = 2 * (wid & 1);   // this lane's outputs 4 q + j0, + 1
  float s0 = 0.0f, s1 = 0.0f;
  for (int base = 0; base < nkb; base += NB) {
    const int nb = min(NB, nkb - base);
    WRaw<FMT> R[2];
    uint32_t sc[2];
    u32x4 b16[2][4];
    u32x2 b8[2][4];
    f32x4 da[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {   // blocks past the end re-read the last (not added)
      const int kb = min(base + 2 * wid + i, nkb - 1);
      const uint8_t* blk = wrow + (size_t)kb * blk_bytes<FMT>();
      w_load<FMT>(R[i], blk, lh);
      sc[i] = *(const uint16_t*)(blk + scale_off<FMT>());
      const uint8_t* at = tiles + ((size_t)kb * n_groups + g) * AT_BYTES;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int p = (s * 2 + lh) * 32 + l32;
        b16[i][s] = *(const u32x4*)(at + p * 16);
        b8[i][s] = *(const u32x2*)(at + AT_HI + p * 8);
      }
      da[i] = *(const f32x4*)(at + AT_D + l32 * 16);
    }
    if (base) __syncthreads();   // the last round's accumulators have been read
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t o[8];
      w_expand<FMT>(R[i], lh, o);
      i32x8 a[4] = {};
#pragma unroll
      for (int k = 0; k < 8; ++k) {   // both halves' words to all lanes
        const auto r = __builtin_amdgcn_permlane32_swap(o[k], o[k], false, false);
        a[k >> 2][k & 3] = (int)r[0];
        a[2 + (k >> 2)][k & 3] = (int)r[1];
      }
      f32x16 c[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) c[s] = sub_dots(a[s], op_fp6(b16[i][s], b8[i][s]), scale_b);
      const int slot = 2 * wid + i;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = block_sum(c, 4 * k + j, da[i]);
        *(f32x4*)acc[slot][k][lane] = v;
      }
      if (lh == 0) dws[slot][l32] = h2f(sc[i]);
    }
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < nb; ++k) {
      const float2 v = *(const float2*)&acc[k][q][lane][j0], dw = *(const float2*)&dws[k][8 * q + 4 * lh + j0];
      s0 += v.x * dw.x;
      s1 += v.y * dw.y;
    }
  }
  const int tok = g * 32 + l32, row = r0 + 8 * q + 4 * lh + j0;
  if (tok >= seq) return;
  float* o = out + (size_t)tok * n + row;
  if (vec_out) {
    if (row < n) *(float2*)o = make_float2(s0, s1);   // n % 4 == 0
  } else {
    if (row < n) o[0] = s0;
    if (row + 1 < n) o[1] = s1;
  }
}

// ---- expanded weights ----
// Weight tile: 32 rows x 128 columns of FP4 operand words and f32 scales,
//   [sub 4][row 32] 16 B, then the f16 scales, [half 2][16]: half h holds the rows
//   8 (i / 4) + 4 h + i % 4 of a lane's 16 outputs,
// tile (kb, row group) at (kb * row_groups + group).  Rows past n repeat row n - 1.
constexpr int WT_D = 2048, WT_BYTES = 2112;

template <int FMT>
__global__ __launch_bounds__(256) void k_weight_tiles(const uint8_t* __restrict__ w, int n, int K,
                                                      uint8_t* __restrict__ tiles) {
  // a wave: 32 rows x the two halves of a block; 4 column blocks per workgroup
  const int lane = threadIdx.x & 63, kb = blockIdx.x * 4 + (threadIdx.x >> 6), nkb = K / 128;
  const int g = blockIdx.y, row = lane & 31, half = lane >> 5;
  if (kb >= nkb) return;
  const uint8_t* blk = w + ((size_t)min(g * 32 + row, n - 1) * nkb + kb) * blk_bytes<FMT>();
  WRaw<FMT> R;
  w_load<FMT>(R, blk, half);
  uint32_t o[8];
  w_expand<FMT>(R, half, o);
  uint8_t* t = tiles + ((size_t)kb * gridDim.y + g) * WT_BYTES;
  *(uint4*)(t + ((2 * half) * 32 + row) * 16) = make_uint4(o[0], o[1], o[2], o[3]);
  *(uint4*)(t + ((2 * half + 1) * 32 + row) * 16) = make_uint4(o[4], o[5], o[6], o[7]);
  if (half == 0) {
    const int at = ((row >> 2) & 1) * 16 + (row >> 3) * 4 + (row & 3);
    *(uint16_t*)(t + WT_D + at * 2) = *(const uint16_t*)(blk + scale_off<FMT>());
  }
}

// The product from expanded weights: WR x WT waves, each RT x TT tiles of 32 rows x
// 32 tokens.  A step's tiles (128 columns) go from memory straight to LDS, NS - 1
// steps ahead: one step is shorter than a loaded memory round trip, and the
// operands of several steps would not fit the registers.
template <int WG, int TG> struct StageX {
  uint8_t a[TG * AT_BYTES];
  uint8_t w[WG * WT_BYTES];
};
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// At most N vector memory operations still in flight, and no LDS read (of a buffer
// that another wave may copy into after the barrier that follows).
template <int N> HH_DEV void wait_copies() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

template <int RT, int TT, int WR, int WT, int NS>
__global__ __launch_bounds__(64 * WR * WT, 2) void k_gemm_f4x(const uint8_t* __restrict__ wtiles,
                                                              const uint8_t* __restrict__ tiles,
                                                              float* __restrict__ out, int row0, int n, int K,
                                                              int seq, int n_rgroups, int n_groups, int vec_out) {
#pragma clang fp contract(off)
  constexpr int NW = WR * WT, NT = 64 * NW, WG = RT * WR, TG = TT * WT;
  constexpr int NPA = TG * (AT_BYTES / 16), PA = (NPA + NT - 1) / NT;   // 16-byte pieces; copies per wave
  constexpr int NPW = WG * (WT_BYTES / 16), PW = (NPW + NT - 1) / NT;
  constexpr int PER = PA + PW;
  typedef StageX<WG, TG> Stage;
  __shared__ __align__(16) Stage s0, s1, s2, s3;   // distinct objects: a read waits for its own copies only
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31,
            lh = lane >> 5;
  const int wr = wid % WR, wt = wid / WR;
  const int rg0 = blockIdx.x * WG, g0 = blockIdx.y * TG;   // n_rgroups, n_groups: multiples of WG, TG
  const int nsteps = K / 128, scale_b = lh ? 130 : 134;
  const uint8_t* ab = tiles + (size_t)g0 * AT_BYTES;
  const uint8_t* wb = wtiles + (size_t)rg0 * WT_BYTES;
  const size_t a_step = (size_t)n_groups * AT_BYTES, w_step = (size_t)n_rgroups * WT_BYTES;
  // every wave issues PER copies (the last ones overlap where the pieces do not divide)
  auto copy = [&](Stage& S, int kb) {
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const int p = min(wid * 64 + NT * i, NPA - 64);
      __builtin_amdgcn_global_load_lds((gptr_t)(ab + (size_t)kb * a_step + (size_t)(p * 16) + (uint32_t)(lane * 16)),
                                       (lptr_t)(S.a + p * 16), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      const int p = min(wid * 64 + NT * i, NPW - 64);
      __builtin_amdgcn_global_load_lds((gptr_t)(wb + (size_t)kb * w_step + (size_t)(p * 16) + (uint32_t)(lane * 16)),
                                       (lptr_t)(S.w + p * 16), 16, 0, 0);
    }
  };
  f32x16 sum[RT][TT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[r][t][i] = 0.0f;

  // one step from S; N: the buffer of step kb + NS - 1 (read last in step kb - 1)
  auto step = [&](const Stage& S, Stage& N, int kb) {
    copy(N, min(kb + NS - 1, nsteps - 1));   // past the end: into a buffer that no one reads again
    const uint8_t* wp = S.w + wr * RT * WT_BYTES;
    const uint8_t* ap = S.a + wt * TT * AT_BYTES;
    i32x8 a[4], b[TT][4];
    f32x4 da[TT];
    f16x8 dw[2];
    auto load_a = [&](int r, int s) { a[s] = op_fp4(*(const u32x4*)(wp + r * WT_BYTES + (s * 32 + l32) * 16)); };
    auto load_b = [&](int t, int s) {
      const int p = (s * 2 + lh) * 32 + l32;
      uint32_t tail = AT_HI + p * 8;
      asm("" : "+v"(tail));   // keeps two subs' 8-byte reads from being merged into one (and moved apart again)
      b[t][s] = op_fp6(*(const u32x4*)(ap + t * AT_BYTES + p * 16), *(const u32x2*)(ap + t * AT_BYTES + tail));
    };
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      load_a(0, s);
      load_b(0, s);
    }
    da[0] = *(const f32x4*)(ap + AT_D + l32 * 16);
    f32x16 c[2], acc;
    c[0] = sub_dots(a[0], b[0][0], scale_b);
#pragma unroll
    for (int j = 0; j < RT * TT * 4; ++j) {   // each product is issued one ahead of its combine
      const int s = j & 3, t = (j >> 2) % TT, r = (j >> 2) / TT;
      if (j + 1 < RT * TT * 4) c[(j + 1) & 1] = sub_dots(a[(j + 1) & 3], b[((j + 1) >> 2) % TT][(j + 1) & 3], scale_b);
      if (t == TT - 1 && r + 1 < RT) load_a(r + 1, s);   // this sub's operand is free: the next row tile's
      if (r == 0 && t + 1 < TT) load_b(t + 1, s);
      if (r == 0 && s == 1 && t + 1 < TT) da[t + 1] = *(const f32x4*)(ap + (t + 1) * AT_BYTES + AT_D + l32 * 16);
      if (t == 0 && s == 0) {
        uint32_t at = WT_D + lh * 32 + 16;
        asm("" : "+v"(at));   // kept apart: the halves of a merged read would wait for every copy in flight
        dw[0] = *(const f16x8*)(wp + r * WT_BYTES + WT_D + lh * 32);
        dw[1] = *(const f16x8*)(wp + r * WT_BYTES + at);
      }
      __builtin_amdgcn_sched_barrier(0x74);   // global memory and scalar operations may cross
      const f32x16& cj = c[j & 1];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        acc[i] = s == 0 ? cj[i] * da[t][0] : fmaf(cj[i], da[t][s], acc[i]);
        if (s == 3) sum[r][t][i] += fmaf(acc[i], (float)dw[i >> 3][i & 7], 0.0f);
      }
      __builtin_amdgcn_sched_barrier(0x74);
    }
    // this wave's copies of step kb + 1 have landed; after the barrier everyone's have
    wait_copies<(NS - 2) * PER>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  copy(s0, 0);
  if (NS > 2) copy(s1, min(1, nsteps - 1));
  if (NS > 3) copy(s2, min(2, nsteps - 1));
  wait_copies<(NS - 2) * PER>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int kb = 0;
  if constexpr (NS == 2) {
    for (; kb + 2 <= nsteps; kb += 2) {
      step(s0, s1, kb);
      step(s1, s0, kb + 1);
    }
    if (kb < nsteps) step(s0, s1, kb);
  } else if constexpr (NS == 3) {
    for (; kb + 3 <= nsteps; kb += 3) {
      step(s0, s2, kb);
      step(s1, s0, kb + 1);
      step(s2, s1, kb + 2);
    }
    if (kb < nsteps) step(s0, s2, kb);
    if (kb + 1 < nsteps) step(s1, s0, kb + 1);
  } else {
    for (; kb + 4 <= nsteps; kb += 4) {
      step(s0, s3, kb);
      step(s1, s0, kb + 1);
      step(s2, s1, kb + 2);
      step(s3, s2, kb + 3);
    }
    if (kb < nsteps) step(s0, s3, kb);
    if (kb + 1 < nsteps) step(s1, s0, kb + 1);
    if (kb + 2 < nsteps) step(s2, s1, kb + 2);
  }
  wait_copies<0>();   // the copies past the end
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t)
      store_tile(out, sum[r][t], row0 + (rg0 + wr * RT + r) * 32, (g0 + wt * TT + t) * 32, n, seq, vec_out);
}

}  // namespace

// 32-token groups of a tile buffer: whole workgroup tiles of the widest launch.
static int act_groups(int seq) { return (seq + 127) / 128 * 4; }

size_t hh_act_tiles_bytes(int K, int seq) {
  return (size_t)(K / 128) * act_groups(seq) * AT_BYTES;
}

int hh_act_tiles_launch(int fmt, const uint8_t* x, const int8_t* xq, const float* xd, int K, int seq, uint8_t* tiles,
                        hipStream_t s) {
  if (K <= 0 || K % 128 != 0 || seq <= 0) return 1;
  const int ng = act_groups(seq);
  const dim3 grid((unsigned)(K / 128) * ng);
#define HH_TILES(F)                                                                                     \
  if (x) hipLaunchKernelGGL((k_act_tiles<F, true>), grid, dim3(128), 0, s, x, xq, xd, K, seq, ng, tiles);   \
  else hipLaunchKernelGGL((k_act_tiles<F, false>), grid, dim3(128), 0, s, x, xq, xd, K, seq, ng, tiles)
  switch (fmt) {
    case FMT_Q2: HH_TILES(FMT_Q2); break;
    case FMT_Q1: HH_TILES(FMT_Q1); break;
    case FMT_PT: HH_TILES(FMT_PT); break;
    default: return 1;
  }
#undef HH_TILES
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

// The forms of a product and the time each takes, from which the launcher chooses.
// A form costs a start, its workgroups' loads and stores against each other, and for
// each of its rounds (the workgroups that fit the 256 CUs at once) a fixed part and a
// part per 128 columns.  The figures are fits to 6153 measured products (K 128 ..
// 17408, 1024 .. 34816 rows, 2 .. 2048 tokens, the three formats, weights cold); the
// choice by them takes 0.1% longer than the fastest form on average, and 17% at most
// from K = 1024 (more than 5% in 25 of 5082).  (Thresholds on the tokens and the grid
// alone, set at K = 4096, took up to 57% longer, and at K = 1024 longer than an int8
// MFMA kernel: Q2_0, 6144 x 1024, 224 tokens 13.2 us expanded in 128 x 64 tiles, 12.3
// int8, 10.4 straight from the blocks, the form chosen here.  int8 keeps one corner,
// PTQ1_0 of some 8192 .. 16384 rows at 65 .. 256 tokens with K 1024 .. 1536, where no
// form here reaches it, by 2 to 9%: 16384 x 1024, 128 tokens 14.8, here 15.5; and with
// 16384 rows and K = 17408, past one slab, 187, here 207.)
enum : int { F4_TILE, F4_ROWS, X_128x64_8, X_128x64_4, X_128x128, X_256x128, N_FORMS };
constexpr int FORM_ROWS[N_FORMS] = {5, 7, 7, 7, 7, 8};     // log2 rows and
constexpr int FORM_GROUPS[N_FORMS] = {0, 0, 1, 1, 2, 2};   // 32-token groups per workgroup

// us of one pass over n rows in a form (the expanded ones without their expansion).
static double form_us(int form, int fmt, int n, int K, int ng) {
  const int rl = FORM_ROWS[form], gl = FORM_GROUPS[form];
  const long g = (long)((n + (1 << rl) - 1) >> rl) * ((ng + (1 << gl) - 1) >> gl);
  const double u = K >> 7, r = g * (1.0 / 512);
  const double waves = (double)((g + 255) >> 8);                // rounds at one workgroup per CU
  const double pairs = (double)((g >> 9) + ((g & 511) > 256));  // at two, but for
  const double tail = (g & 511) != 0 && (g & 511) <= 256;       // a last one of one per CU
  switch (form) {
    case F4_TILE: {   // 16 column blocks are one memory round trip
      const double trip = fmt == FMT_Q1 ? 3.65 : fmt == FMT_Q2 ? 3.99 : 4.39;
      return 1.2 + waves * trip * ((K + 2047l) >> 11);
    }
    case F4_ROWS:   // unpacks its weights in every workgroup: by format
      if (fmt == FMT_Q1)
        return 2.118 + 0.89 * r + (g <= 256 ? 0.7 * u : 0.116 * u + pairs * 0.707 * u + tail * 0.393 * u);
      if (fmt == FMT_Q2)
        return 2.2 + 1.1 * r + (g <= 256 ? 0.745 * u : 0.084 * u + pairs * 0.828 * u + tail * 0.432 * u);
      return 1.251 + 1.474 * r + (g <= 256 ? 1.301 * u : 0.443 * u + pairs * 1.09 * u + tail * 0.519 * u);
    case X_128x64_8: return 3.277 + 6.4 * r + waves * (0.721 + 0.535 * u);
    case X_128x64_4: return 4.234 + 4.454 * r + tail * 0.612 * u + pairs * (1.2 + 0.963 * u);
    case X_128x128: return 4.053 + 6.65 * r + tail * 1.123 * u + pairs * 1.774 * u;
    default: return 5.922 + 18.534 * r + waves * (3.41 + 1.673 * u);
  }
}

// Expanded weights: the whole matrix's where they fit F4X_SLAB, else that many rows
// at a time.  An expansion reads its blocks and writes 2112 bytes per 32 x 128.
constexpr size_t F4X_SLAB = (size_t)128 << 20;
static int slab_rows(int n, int K) {   // rows per expansion: whole 256-row tiles
  const size_t per = (size_t)(K / 128) * 8 * WT_BYTES;
  return (int)std::min<size_t>((n + 255) / 256, std::max<size_t>(1, F4X_SLAB / per)) * 256;
}
static double expand_us(int n, int K) { return 2.223 + 0.161e-6 * n * K; }
static int best_expanded(int fmt, int n, int K, int ng, double* us) {
  int best = X_128x64_8;
  *us = form_us(best, fmt, n, K, ng);
  for (int f = best + 1; f < N_FORMS; ++f) {
    const double t = form_us(f, fmt, n, K, ng);
    if (t < *us) { *us = t; best = f; }
  }
  return best;
}

// The form without expanded weights, and the one that is chosen (for the first slab).
static int direct_form(int fmt, int n, int K, int ng, double* us) {
  *us = form_us(F4_ROWS, fmt, n, K, ng);
  // past 16 rounds the row form always wins
  if ((long)((n + 31) / 32) * ng > 4096) return F4_ROWS;
  const double tile = form_us(F4_TILE, fmt, n, K, ng);
  if (!(tile < *us)) return F4_ROWS;
  *us = tile;
  return F4_TILE;
}

int hh_gemm_f4_form(int fmt, int n, int K, int seq) {
  const int ng = (seq + 31) / 32;
  double limit, us = 0.0, t;
  const int direct = direct_form(fmt, n, K, ng, &limit);
  if (ng < 2) return direct;   // one group leaves half of every expanded tile empty
  // (a grid dimension holds 2^32 lanes: the row form's tiles may be more)
  if ((long)((n + 127) / 128) * ng >= (1l << 24)) limit = 1e30;
  const int slab = slab_rows(n, K);
  int first = -1;
  for (int r0 = 0; r0 < n && us < limit; r0 += slab) {
    const int nr = std::min(slab, n - r0), f = best_expanded(fmt, nr, K, ng, &t);
    if (first < 0) first = f;
    us += expand_us(nr, K) + t;
  }
  return us < limit ? first : direct;
}

int hh_gemm_f4_pass_rows(int form, int n, int K) { return form >= X_128x64_8 ? std::min(slab_rows(n, K), n) : n; }

size_t hh_gemm_f4_wbytes(int form, int n, int K) {
  return form >= X_128x64_8 ? (size_t)(slab_rows(n, K) / 32) * (K / 128) * WT_BYTES : 0;
}

int hh_gemm_f4_launch(int fmt, int form, const uint8_t* w, int n, int K, const uint8_t* tiles, int seq,
                      uint8_t* wtiles, float* out, hipStream_t s) {
  if (K <= 0 || K % 128 != 0 || n <= 0 || seq <= 0 || (fmt != FMT_Q2 && fmt != FMT_Q1 && fmt != FMT_PT)) return 1;
  const int ng = (seq + 31) / 32, ngp = act_groups(seq);
  const int vec = n % 4 == 0 && ((uintptr_t)out & 15) == 0;
  double us;
  if (form >= X_128x64_8 && !wtiles) form = direct_form(fmt, n, K, ng, &us);
  if (form < X_128x64_8) {
    const bool small = form == F4_TILE;
    const dim3 grid(small ? (unsigned)((n + 31) / 32) * ng : (unsigned)((n + 127) / 128) * ng);
#define HH_F4(F)                                                                                                   \
  if (small) hipLaunchKernelGGL((k_gemm_f4s<F>), grid, dim3(512), 0, s, w, tiles, out, n, K, seq, ngp, vec);        \
  else hipLaunchKernelGGL((k_gemm_f4<F, 4>), grid, dim3(256), 0, s, w, tiles, out, n, K, seq, ngp, vec)
    switch (fmt) {
      case FMT_Q2: HH_F4(FMT_Q2); break;
      case FMT_Q1: HH_F4(FMT_Q1); break;
      default: HH_F4(FMT_PT); break;
    }
#undef HH_F4
    return hipGetLastError() == hipSuccess ? 0 : 1;
  }
  const int slab = slab_rows(n, K);
  for (int r0 = 0; r0 < n; r0 += slab) {
    const int nr = std::min(slab, n - r0), rg = (nr + 255) / 256 * 8;   // its own rows, in whole 256-row tiles
    const uint8_t* ws = w + (size_t)r0 * (K / 128) * (fmt == FMT_Q1 ? 18 : fmt == FMT_PT ? 28 : 34);
    const dim3 wgrid((K / 128 + 3) / 4, rg);
#define HH_WT(F) hipLaunchKernelGGL((k_weight_tiles<F>), wgrid, dim3(256), 0, s, ws, nr, K, wtiles)
    if (fmt == FMT_Q2) HH_WT(FMT_Q2);
    else if (fmt == FMT_Q1) HH_WT(FMT_Q1);
    else HH_WT(FMT_PT);
#undef HH_WT
#define HH_F4X(RT, TT, WR, WT, NS)                                                                               \
  hipLaunchKernelGGL((k_gemm_f4x<RT, TT, WR, WT, NS>),                                                           \
                     dim3((nr + 32 * RT * WR - 1) / (32 * RT * WR), (ng + TT * WT - 1) / (TT * WT)),             \
                     dim3(64 * WR * WT), 0, s, wtiles, tiles, out, r0, n, K, seq, rg, ngp, vec)
    switch (best_expanded(fmt, nr, K, ng, &us)) {
      case X_128x64_8: HH_F4X(1, 1, 4, 2, 4); break;
      case X_128x64_4: HH_F4X(2, 1, 2, 2, 3); break;
      case X_128x128: HH_F4X(2, 2, 2, 2, 2); break;
      default: HH_F4X(4, 1, 2, 4, 3);
    }
#undef HH_F4X
    if (hipGetLastError() != hipSuccess) return 1;
  }
  return 0;
}
