// hh_gemm.hip — batched GEMM of Q8_0 weights on int8 MFMA for gfx950 (the 1- and
// 2-bit formats: hh_gemm_f4.hip).
//
// Semantics: out[s*n + r] = dot_fn(w + r*row_bytes, x + s*q8_stride, K) for
// every token s < seq_len and row r < n: par_dot_rows_batched with DotFn /
// DotFn2 (pool.rs:40-80, :568-618; matmul.rs:580-674), whose paired kernels
// are bit-identical to the single-token dot (q2_0.rs:936-986).  Here too:
// every 32-element sub-block dot is an exact int32 from
// v_mfma_i32_16x16x32_i8, and the fp32 combine follows the scalar kernels
// (q8_0.rs:154-171): sum += ((float)i * dw) * da per 32-weight block,
// so each output equals the decode GEMV's bit for bit.
//
// Tiling: a 512-lane workgroup owns 128 tokens x 64 rows; wave w owns tokens
// [16w, 16w+16) and all rows as four 16x16 MFMA tiles.  Per 128-column step the
// workgroup stages the activation bytes and scales of its tokens and the weight
// blocks of its rows in LDS (double-buffered: the next step's global loads are
// issued before this step's MFMAs).  Activations come split (int8 rows + f32 block
// scales, k_q8_split), so staging is plain 16-byte copies.  Operand layouts
// (checked on the device): A lane l = row l%16, k = 8*(l/16) .. +8; B lane l =
// column l%16, same k; C lane l = column l%16, rows 4*(l/16) .. +4.
#include "hh_kernels.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int NTG = 512;       // lanes per workgroup (8 waves, two per SIMD)
constexpr int TM = 128;        // tokens per workgroup
constexpr int TN = 64;         // rows per workgroup
constexpr int KS = 128;        // columns per step
// LDS bytes per token / weight row: 34 dwords (= 2 mod 32 banks), so the 16
// rows of an MFMA operand read (8 bytes per lane) fall on distinct bank pairs;
// rows are 8-byte aligned, so tile stores are 8 bytes wide.
constexpr int AROW = KS + 8;

// Per step a lane copies two 16-byte pieces of the 128 x 128 int8 tile and one
// scale.
struct Stage {
  int8_t a[TM * AROW];     // activations
  int8_t w[TN * AROW];     // weights
  float da[4 * TM];        // activation scale per (sub-block, token)
  float dw[TN * 4];        // weight scale per (row, sub-block)
};

constexpr int CU = 64;                  // u16 code units per row and step
constexpr int WREGS = TN * CU / NTG;    // per lane
constexpr int STEP_BYTES = 136;         // four 34-byte blocks

struct Regs {
  uint4 a[2];
  float ad;
  uint32_t w[WREGS];
  uint32_t ws;
};

HH_DEV void stage_load(Regs& R, const uint8_t* __restrict__ w, const int8_t* __restrict__ xq,
                       const float* __restrict__ xd, int n, int seq, int K, int r0, int s0, int kb) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + NTG * i, t = idx >> 3, piece = idx & 7;
    const int sidx = min(s0 + t, seq - 1);
    R.a[i] = *(const uint4*)(xq + (size_t)sidx * K + (size_t)kb * KS + 16 * piece);
  }
  {
    const int t = tid >> 2, sub = tid & 3;
    const int sidx = min(s0 + t, seq - 1);
    R.ad = xd[(size_t)sidx * (K / 32) + kb * 4 + sub];
  }
  const size_t row_bytes = (size_t)K / 32 * 34;
#pragma unroll
  for (int i = 0; i < WREGS; ++i) {
    const int idx = tid + NTG * i;
    const int rr = idx / CU, u = idx % CU, r = min(r0 + rr, n - 1);
    const uint8_t* base = w + (size_t)r * row_bytes + (size_t)kb * STEP_BYTES;
    R.w[i] = *(const uint16_t*)(base + (u / 16) * 34 + 2 + 2 * (u % 16));
  }
  if (tid < TN * 4) {   // waves 0-3: uniform
    const int rr = tid / 4, b = tid % 4, r = min(r0 + rr, n - 1);
    R.ws = *(const uint16_t*)(w + (size_t)r * row_bytes + (size_t)kb * STEP_BYTES + 34 * b);
  }
}

HH_DEV void stage_store(Stage& st, const Regs& R) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + NTG * i, t = idx >> 3, piece = idx & 7;
    uint2* dst = (uint2*)(st.a + t * AROW + 16 * piece);
    dst[0] = make_uint2(R.a[i].x, R.a[i].y);
    dst[1] = make_uint2(R.a[i].z, R.a[i].w);
  }
  st.da[(tid & 3) * TM + (tid >> 2)] = R.ad;        // loaded as (t = tid / 4, sub = tid % 4)
#pragma unroll
  for (int i = 0; i < WREGS; ++i) {
    const int idx = tid + NTG * i, rr = idx / CU, u = idx % CU;
    *(uint16_t*)(st.w + rr * AROW + 32 * (u / 16) + 2 * (u % 16)) = (uint16_t)R.w[i];
  }
  if (tid < TN * 4) st.dw[tid] = h2f(R.ws);
}

__global__ __launch_bounds__(NTG) void k_gemm(const uint8_t* __restrict__ w, const int8_t* __restrict__ xq,
                                              const float* __restrict__ xd, float* __restrict__ out, int n, int K,
                                              int seq) {
#pragma clang fp contract(off)
  __shared__ Stage st[2];
  constexpr int NTT = TN / 16;   // MFMA tiles per wave
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int r0 = blockIdx.x * TN, s0 = blockIdx.y * TM;
  const int nsteps = K / KS;
  float sum[NTT][4];
#pragma unroll
  for (int t = 0; t < NTT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) sum[t][r] = 0.0f;

  // Two register sets: at the end of step kb, step kb + 1 (loaded two steps
  // earlier) is written to the free LDS buffer and the global loads of step
  // kb + 3 are issued into the register set just freed, so every load has two
  // steps' compute to land.
  Regs R0, R1;
  stage_load(R0, w, xq, xd, n, seq, K, r0, s0, 0);
  if (nsteps > 1) stage_load(R1, w, xq, xd, n, seq, K, r0, s0, 1);
  stage_store(st[0], R0);
  if (nsteps > 2) stage_load(R0, w, xq, xd, n, seq, K, r0, s0, 2);
  __syncthreads();
  const int arow = 16 * wid + (lane & 15);   // A operand token (within the tile)
  const int kg = 8 * (lane >> 4);            // k offset within a sub-block
  const int tok0 = 16 * wid + 4 * (lane >> 4);
  auto step = [&](int kb, Regs& Rn) {   // Rn holds step kb + 1
    const Stage& S = st[kb & 1];
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
      const long a = *(const long*)(S.a + arow * AROW + sub * 32 + kg);
      const float4 da4 = *(const float4*)(S.da + sub * TM + tok0);
      const float da[4] = {da4.x, da4.y, da4.z, da4.w};
#pragma unroll
      for (int t = 0; t < NTT; ++t) {
        const int col = 16 * t + (lane & 15);
        const long b = *(const long*)(S.w + col * AROW + sub * 32 + kg);
        v4i c = {0, 0, 0, 0};
        c = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0);
        const float dw = S.dw[col * 4 + sub];
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[t][r] += ((float)c[r] * dw) * da[r];
      }
    }
    if (kb + 1 < nsteps) stage_store(st[(kb + 1) & 1], Rn);
    if (kb + 3 < nsteps) stage_load(Rn, w, xq, xd, n, seq, K, r0, s0, kb + 3);
    __syncthreads();
  };
  for (int kb = 0; kb < nsteps; kb += 2) {
    step(kb, R1);
    if (kb + 1 < nsteps) step(kb + 1, R0);
  }
#pragma unroll
  for (int t = 0; t < NTT; ++t) {
    const int r = r0 + 16 * t + (lane & 15);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int s = s0 + tok0 + q;
      if (r < n && s < seq) out[(size_t)s * n + r] = sum[t][q];
    }
  }
}

// Standard Q8_0 rows -> split layout (int8 [seq][K], f32 scales [seq][K/32]).
__global__ void k_q8_split(const uint8_t* __restrict__ x, int64_t nblocks, int8_t* __restrict__ xq,
                           float* __restrict__ xd) {
  const int64_t b = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
  const int l = threadIdx.x & 31;
  if (b >= nblocks) return;
  const uint8_t* blk = x + b * 34;
  xq[b * 32 + l] = (int8_t)blk[2 + l];
  if (l == 0) xd[b] = h2f((uint32_t)blk[0] | ((uint32_t)blk[1] << 8));
}

}  // namespace

int hh_gemm_launch(const uint8_t* w, int n, int K, const int8_t* xq, const float* xd, int seq, float* out,
                   hipStream_t s) {
  if (K % KS != 0 || n <= 0 || seq <= 0) return 1;
  hipLaunchKernelGGL(k_gemm, dim3((n + TN - 1) / TN, (seq + TM - 1) / TM), dim3(NTG), 0, s, w, xq, xd, out, n, K, seq);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

int hh_q8_split_launch(const uint8_t* x, int64_t nblocks, int8_t* xq, float* xd, hipStream_t s) {
  if (nblocks <= 0) return 0;
  hipLaunchKernelGGL(k_q8_split, dim3((unsigned)((nblocks + 7) / 8)), dim3(256), 0, s, x, nblocks, xq, xd);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}
