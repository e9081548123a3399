// Exact fp32 FlashAttention (forward and backward) on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32: fp32 operands, fp32 accumulate).
//
// This is the path for float32 inputs: the reference checks its fp32 results
// against SDPA at 1e-3 and runs gradcheck in fp32
// (kernels/tests/test_flash_attention.py:49-53,
// kernels/tests/test_flash_attention_backward.py:44-65), so nothing here is
// rounded to a narrower type. Arbitrary element strides and any head_dim
// <= 128 (zero-padded to DP = 32, 64 or 128) are accepted.
//
// Math is the same as the bf16/fp16 kernels (kernels/flash_attention.py:
// 135-179, kernels/flash_attention_backward.py:290-330), with a row max per
// 32-key block (standard online softmax) and exponentials in base 2.
//
// Operand layouts of v_mfma_f32_32x32x2_f32 (checked on the device): lane l
// supplies A[l % 32][l / 32] and B[l / 32][l % 32]; register i of lane l
// holds C[8 (i / 4) + 4 (l / 32) + i % 4][l % 32]. With hh = l / 32:
//   - a product over the head dim takes step kk (0 .. DP/2 - 1) as the dims
//     kk (hh = 0) and kk + DP/2 (hh = 1); the row operand (K, Q or dO rows)
//     is read from LDS, four steps per ds_read_b128, and the column operand
//     (Q, dO, K or V of the lane's own row) is held in registers;
//   - a product over a 32-row block of the score tile takes step j (0..15)
//     as rows 8 (j / 4) + 4 hh + j % 4, which is exactly register j of the
//     score tile: the B operand is the score register itself, and the A
//     operand is one row per half-wave of a V, K, dO or Q tile (32
//     consecutive floats per half-wave, one ds_read_b32).
// The first three kernels take any strides; the wave kernels below them, for
// rows that 16-byte loads can address, are several times faster.
// Tiles are staged through LDS with padded rows: row stride DP + 4 floats
// for tiles read four steps at a time by 16 rows (every 16-byte read of a
// quarter-wave hits distinct banks), DP + 8 for tiles read one row per
// half-wave (the two rows of a read, 4 apart, land 32 banks apart).
#include "fa_common.hpp"

namespace lsfa {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2f = 0.6931471805599453f;

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Stage rows [r0, r0 + R) of a strided fp32 matrix (rows x D valid) into LDS
// rows of stride LD (zero outside the matrix or past D).
template <int R, int DP, int LD>
__device__ __forceinline__ void stage_rows(float* dst, const float* src, int64_t srow, int64_t scol, int r0, int rows,
                                           int D, int tid, int nthreads) {
  for (int idx = tid; idx < R * DP; idx += nthreads) {
    const int r = idx / DP, c = idx - r * DP, g = r0 + r;
    dst[r * LD + c] = (g < rows && c < D) ? src[(int64_t)g * srow + (int64_t)c * scol] : 0.f;
  }
}

// Column operand of a head-dim product: this lane's row, dims kk + hh * DP/2.
template <int DP>
__device__ __forceinline__ void load_row_operand(float (&reg)[DP / 2], const float* src, int64_t srow, int64_t scol,
                                                 int row, int rows, int D, int hh) {
#pragma unroll
  for (int kk = 0; kk < DP / 2; ++kk) {
    const int d = kk + hh * (DP / 2);
    reg[kk] = (row < rows && d < D) ? src[(int64_t)row * srow + (int64_t)d * scol] : 0.f;
  }
}

// C = (rows of A tile) x reg^T over the head dim: 32 tile rows (LDS, stride
// LD, first row base) against this lane's register row.
template <int DP, int LD>
__device__ __forceinline__ f32x16 dim_product(const float* base, const float (&reg)[DP / 2], int l32, int hh) {
  f32x16 c = f32x16{};
  const float* row = base + l32 * LD + hh * (DP / 2);
#pragma unroll
  for (int k4 = 0; k4 < DP / 8; ++k4) {
    const f32x4 a = *(const f32x4*)(row + 4 * k4);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = mfma_f32(a[e], reg[4 * k4 + e], c);
  }
  return c;
}

// acc[dt] += (tile rows)^T x scores over a 32-row block: tile rows r_j (LDS,
// stride LD) times register j of the score tile s.
template <int DT, int LD>
__device__ __forceinline__ void block_product(f32x16 (&acc)[DT], const float* tile, const f32x16& s, int l32, int hh) {
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float* row = tile + (8 * (j >> 2) + 4 * hh + (j & 3)) * LD + l32;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = mfma_f32(row[32 * dt], s[j], acc[dt]);
  }
}

__device__ __forceinline__ float hmax(float x) { return half_max(x); }
__device__ __forceinline__ float hsum(float x) { return half_sum(x); }

// Forward: workgroup = 4 waves x 32 queries; keys in blocks of 32. S^T = K Q^T
// (lane = query, registers = keys), O^T += V^T P^T.
template <int DP, bool VARLEN>
__global__ __launch_bounds__(256) void fa_fwd_f32_kernel(const FwdParams p, int causal, float scale) {
  constexpr int BM = 128, BN = 32, DT = DP / 32, LDK = DP + 4, LDV = DP + 8;
  __shared__ __attribute__((aligned(16))) float Ks[BN * LDK];
  __shared__ __attribute__((aligned(16))) float Vs[BN * LDV];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int bh = blockIdx.y, b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / (p.Hq / p.Hkv);
  int nq = p.Nq, nk = p.Nk;
  int64_t rq0 = 0, rk0 = 0;
  if (VARLEN) {
    rq0 = p.cu_q[b];
    nq = p.cu_q[b + 1] - (int)rq0;
    rk0 = p.cu_k[b];
    nk = p.cu_k[b + 1] - (int)rk0;
  }
  const int q0 = blockIdx.x * BM;
  if (q0 >= nq) return;  // uniform, before any barrier
  const int off = nk - nq, D = p.D;
  const float* Q = (const float*)p.q + (VARLEN ? 0 : (int64_t)b * p.sqb) + (int64_t)h * p.sqh + rq0 * p.sqn;
  const float* K = (const float*)p.k + (VARLEN ? 0 : (int64_t)b * p.skb) + (int64_t)hk * p.skh + rk0 * p.skn;
  const float* V = (const float*)p.v + (VARLEN ? 0 : (int64_t)b * p.svb) + (int64_t)hk * p.svh + rk0 * p.svn;
  float* O = (float*)p.o + (VARLEN ? 0 : (int64_t)b * p.sob) + (int64_t)h * p.soh + rq0 * p.son;
  const int qw = q0 + 32 * wave, qrow = qw + l32;
  const float sl2 = scale * kLog2e;

  float qreg[DP / 2];
  load_row_operand<DP>(qreg, Q, p.sqn, p.sqd, qrow, nq, D, hh);
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  float m = -INFINITY, l = 0.f;  // log2 units

  int kv_end = nk;
  if (causal) kv_end = min(nk, q0 + BM + off);
  for (int kt = 0; kt < kv_end; kt += BN) {
    __syncthreads();
    stage_rows<BN, DP, LDK>(Ks, K, p.skn, p.skd, kt, nk, D, tid, 256);
    stage_rows<BN, DP, LDV>(Vs, V, p.svn, p.svd, kt, nk, D, tid, 256);
    __syncthreads();
    if (causal && kt > qw + 31 + off) continue;  // wave-uniform: no key of the block is visible
    f32x16 s = dim_product<DP, LDK>(Ks, qreg, l32, hh);
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kt + 8 * (i >> 2) + 4 * hh + (i & 3);
      float x = s[i] * sl2;
      if (key >= nk || (causal && key > qrow + off)) x = -INFINITY;
      s[i] = x;
      mx = fmaxf(mx, x);
    }
    const float m_new = fmaxf(m, hmax(mx));
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2f(m - m_use);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = exp2f(s[i] - m_use);
      sum += s[i];
    }
    l = l * alpha + hsum(sum);
    m = m_new;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
    block_product<DT, LDV>(acc, Vs, s, l32, hh);
  }
  if (qrow < nq) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = 32 * dt + 8 * (i >> 2) + 4 * hh + (i & 3);
        if (d < D) O[(int64_t)qrow * p.son + (int64_t)d * p.sod] = acc[dt][i] * inv;
      }
    if (p.lse != nullptr && hh == 0) {
      float* L = p.lse + (VARLEN ? 0 : (int64_t)b * p.slb) + (int64_t)h * p.slh + (rq0 + qrow) * p.sln;
      *L = l > 0.f ? (m + __log2f(l)) * kLn2f : -INFINITY;
    }
  }
}

// Query-stationary dQ (and delta = rowsum(dO * O), stored beside L for the
// dK/dV kernel): S^T = K Q^T, dP^T = V dO^T, dS^T = P^T (dP^T - delta),
// dQ^T += K^T dS^T.
template <int DP>
__global__ __launch_bounds__(256) void fa_bwd_dq_f32_kernel(const BwdParams p, int causal) {
  constexpr int BM = 128, BN = 32, DT = DP / 32, LDK = DP + 4, LDV = DP + 4;
  __shared__ __attribute__((aligned(16))) float Ks[BN * LDK];
  __shared__ __attribute__((aligned(16))) float Vs[BN * LDV];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int bh = blockIdx.y, b = bh / p.H, h = bh - b * p.H;
  const int nq = p.Nq, nk = p.Nk, D = p.D, off = nk - nq;
  const int q0 = blockIdx.x * BM;
  const float* Q = (const float*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const float* K = (const float*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const float* V = (const float*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  const float* Og = (const float*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh;
  const float* dO = (const float*)p.dout + (int64_t)b * p.sdob + (int64_t)h * p.sdoh;
  float* dQ = (float*)p.dq + (int64_t)b * p.sdqb + (int64_t)h * p.sdqh;
  const float* Lg = p.lse + (int64_t)b * p.slb + (int64_t)h * p.slh;
  float* Dg = p.ld + (int64_t)b * p.sldb + (int64_t)h * p.sldh + 1;  // delta of query q at Dg[2q]
  const int qw = q0 + 32 * wave, qrow = qw + l32;
  const bool valid = qrow < nq;

  float qreg[DP / 2], doreg[DP / 2];
  load_row_operand<DP>(qreg, Q, p.sqn, p.sqd, qrow, nq, D, hh);
  load_row_operand<DP>(doreg, dO, p.sdon, p.sdod, qrow, nq, D, hh);
  float dpart = 0.f;
#pragma unroll
  for (int kk = 0; kk < DP / 2; ++kk) {
    const int d = kk + hh * (DP / 2);
    if (valid && d < D) dpart += doreg[kk] * Og[(int64_t)qrow * p.son + (int64_t)d * p.sod];
  }
  const float delta = hsum(dpart);
  float L2 = valid ? Lg[(int64_t)qrow * p.sln] : INFINITY;
  if (L2 == -INFINITY) L2 = INFINITY;  // a row that sees no key: P = 0
  L2 *= kLog2e;
  if (valid && hh == 0) Dg[2 * (int64_t)qrow] = delta;
  const float sl2 = p.scale * kLog2e;

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  int kv_end = nk;
  if (q0 < nq && causal) kv_end = min(nk, q0 + BM + off);
  if (q0 >= nq) kv_end = 0;
  for (int kt = 0; kt < kv_end; kt += BN) {
    __syncthreads();
    stage_rows<BN, DP, LDK>(Ks, K, p.skn, p.skd, kt, nk, D, tid, 256);
    stage_rows<BN, DP, LDV>(Vs, V, p.svn, p.svd, kt, nk, D, tid, 256);
    __syncthreads();
    if (causal && kt > qw + 31 + off) continue;
    f32x16 s = dim_product<DP, LDK>(Ks, qreg, l32, hh);
    const f32x16 dp = dim_product<DP, LDV>(Vs, doreg, l32, hh);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kt + 8 * (i >> 2) + 4 * hh + (i & 3);
      float pr = exp2f(s[i] * sl2 - L2);
      if (key >= nk || (causal && key > qrow + off)) pr = 0.f;
      s[i] = pr * (dp[i] - delta);
    }
    block_product<DT, LDK>(acc, Ks, s, l32, hh);
  }
  if (valid) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = 32 * dt + 8 * (i >> 2) + 4 * hh + (i & 3);
        if (d < D) dQ[(int64_t)qrow * p.sdqn + (int64_t)d * p.sdqd] = acc[dt][i] * p.scale;
      }
  }
}

// Key-stationary dK, dV: S = Q K^T and dP = dO V^T with the keys as the
// columns (lane = key, registers = queries), dV^T += dO^T P, dK^T += Q^T dS.
template <int DP>
__global__ __launch_bounds__(256) void fa_bwd_dkdv_f32_kernel(const BwdParams p, int causal) {
  constexpr int BK = 128, BM = 32, DT = DP / 32, LDQ = DP + 4;
  __shared__ __attribute__((aligned(16))) float Qs[BM * LDQ];
  __shared__ __attribute__((aligned(16))) float dOs[BM * LDQ];
  __shared__ float Ls[BM], Ds[BM];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  const int bh = blockIdx.y, b = bh / p.H, h = bh - b * p.H;
  const int nq = p.Nq, nk = p.Nk, D = p.D, off = nk - nq;
  const int k0 = blockIdx.x * BK;
  const float* Q = (const float*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const float* K = (const float*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const float* V = (const float*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  const float* dO = (const float*)p.dout + (int64_t)b * p.sdob + (int64_t)h * p.sdoh;
  float* dK = (float*)p.dk + (int64_t)b * p.sdkb + (int64_t)h * p.sdkh;
  float* dV = (float*)p.dv + (int64_t)b * p.sdvb + (int64_t)h * p.sdvh;
  const float* Lg = p.lse + (int64_t)b * p.slb + (int64_t)h * p.slh;
  const float* Dg = p.ld + (int64_t)b * p.sldb + (int64_t)h * p.sldh + 1;  // delta of query q at Dg[2q]
  const int kw = k0 + 32 * wave, krow = kw + l32;

  float kreg[DP / 2], vreg[DP / 2];
  load_row_operand<DP>(kreg, K, p.skn, p.skd, krow, nk, D, hh);
  load_row_operand<DP>(vreg, V, p.svn, p.svd, krow, nk, D, hh);
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dk[dt] = f32x16{};
    dv[dt] = f32x16{};
  }
  const float sl2 = p.scale * kLog2e;
  int q_lo = (causal && k0 < nk) ? max(0, k0 - off) : 0;
  q_lo = (q_lo / BM) * BM;
  const int q_end = k0 < nk ? nq : 0;
  for (int qt = q_lo; qt < q_end; qt += BM) {
    __syncthreads();
    stage_rows<BM, DP, LDQ>(Qs, Q, p.sqn, p.sqd, qt, nq, D, tid, 256);
    stage_rows<BM, DP, LDQ>(dOs, dO, p.sdon, p.sdod, qt, nq, D, tid, 256);
    if (tid < BM) {
      const int q = qt + tid;
      float lv = q < nq ? Lg[(int64_t)q * p.sln] : INFINITY;
      if (lv == -INFINITY) lv = INFINITY;
      Ls[tid] = lv * kLog2e;
      Ds[tid] = q < nq ? Dg[2 * (int64_t)q] : 0.f;
    }
    __syncthreads();
    if (causal && kw > qt + BM - 1 + off) continue;  // wave-uniform: no query of the block sees these keys
    f32x16 s = dim_product<DP, LDQ>(Qs, kreg, l32, hh);
    f32x16 dp = dim_product<DP, LDQ>(dOs, vreg, l32, hh);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 8 * (i >> 2) + 4 * hh + (i & 3), q = qt + r;
      float pr = exp2f(s[i] * sl2 - Ls[r]);
      if (q >= nq || krow >= nk || (causal && krow > q + off)) pr = 0.f;
      s[i] = pr;
      dp[i] = pr * (dp[i] - Ds[r]);
    }
    block_product<DT, LDQ>(dv, dOs, s, l32, hh);
    block_product<DT, LDQ>(dk, Qs, dp, l32, hh);
  }
  if (krow < nk) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int d = 32 * dt + 8 * (i >> 2) + 4 * hh + (i & 3);
        if (d < D) {
          dK[(int64_t)krow * p.sdkn + (int64_t)d * p.sdkd] = dk[dt][i] * p.scale;
          dV[(int64_t)krow * p.sdvn + (int64_t)d * p.sdvd] = dv[dt][i];
        }
      }
  }
}

// ---------------------------------------------------------------------------
// Kernels for rows that 16-byte loads can address (unit head-dim stride, D and
// every other stride a multiple of 4, 16-byte aligned bases), which every
// contiguous tensor and projection view with D % 4 == 0 is.
//
// A 32 x 32 x 2 fp32 MFMA takes 64 cycles for 4 KFLOP, so a 32-row block's
// products (two in the forward, three or four in the backward, DP/2 MFMAs
// each) take 4096 cycles apiece at DP = 128, and one wave per SIMD keeps the
// matrix cores busy provided its tiles are there in time. So each wave works
// alone, with no barrier in its loop: it owns 32 stationary rows and streams
// 32-row tiles of the two other operands through two LDS buffers of its own,
// by direct 1 KB loads (buffer_load ... lds). Each buffer is refilled as soon
// as its last product has read it and lands under the products that use the
// other one. (The kernels above stage element by element between two barriers:
// the loads' latency took three quarters of a tile's time.)
// Launches of fewer waves than the GPU has SIMDs give a block of stationary
// rows to KS = 2 or 4 waves of a workgroup, which take its tiles in turn and
// merge through LDS.
// Measured (us, before -> after): forward 1x4x256x64 causal 44.3 -> 10.4,
// 1x8x2048x128 817 -> 170 (101 TFLOP/s; a library GEMM reaches 140);
// forward + backward 1x4x1500x128 2214 -> 283, 2x8x513x64 causal 378 ->
// 79.
// Tiles are [32][DP] floats, 16-byte segments XOR-swizzled per row (swz4) so
// that the reads of four dims of 16 rows and those of 32 floats of rows r and
// r + 4 touch every bank once.
template <int DP>
__device__ __forceinline__ int swz4(int row) {
  if constexpr (DP == 32) return (row >> 1) & 7;
  return (row & 3) | ((row >> 1) & 4) | ((row << 1) & 8);
}
constexpr int kF32Waves = 4;
template <int DP> constexpr int kF32Tile = 32 * DP * 4;  // bytes of a tile

// (Restrict, once inlined, keeps the compiler from waiting for every direct
// load before each LDS read; the waits are explicit.)
__device__ __forceinline__ f32x4 lds_f4(const LDS_AS char* __restrict__ p) { return *(const LDS_AS f32x4*)p; }
__device__ __forceinline__ float lds_f1(const LDS_AS char* __restrict__ p) { return *(const LDS_AS float*)p; }

// Direct load of rows r0 .. r0 + 31 of a matrix (row stride sn elements; rows
// past `rows` and columns past D read as zero) into the tile at dst: DP / 8
// loads of this wave, always.
template <int DP>
__device__ __forceinline__ void load_tile_f32(LDS_AS char* dst, const float* src, int64_t sn, int r0, int rows, int D,
                                              int lane) {
  const int n = min(rows - r0, 32);
  const __amdgpu_buffer_rsrc_t rs = tile_rsrc(n > 0 ? src + (int64_t)r0 * sn : src, n > 0 ? (int)(n * sn * 4) : 0);
#pragma unroll
  for (int c = 0; c < DP / 8; ++c) {
    const int byte = c * 1024 + lane * 16;
    const int row = byte / (DP * 4), seg = ((byte % (DP * 4)) / 16) ^ swz4<DP>(row);
    dma16(rs, (LDS_AS void*)(dst + c * 1024), seg * 4 < D ? (int)(row * sn * 4) + seg * 16 : (int)0x80000000);
  }
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// This wave's LDS reads are done (their buffer may be refilled).
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// This lane's row as a column operand (dims kk + hh * DP/2), 16 bytes a load:
// zero past the matrix and past D (read in bounds, then masked: no branches).
template <int DP>
__device__ __forceinline__ void load_row_f32(float (&reg)[DP / 2], const float* src, int64_t sn, int row, int rows, int D,
                                             int hh) {
  const float* r = src + (int64_t)min(row, rows - 1) * sn;
#pragma unroll
  for (int k4 = 0; k4 < DP / 8; ++k4) {
    const int d = hh * (DP / 2) + 4 * k4;
    const f32x4 v = *(const f32x4*)(r + min(d, D - 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) reg[4 * k4 + e] = row < rows && d < D ? v[e] : 0.f;
  }
}
// dim_product and block_product (above) on a swizzled tile.
template <int DP>
__device__ __forceinline__ f32x16 tile_dims(const LDS_AS char* tile, const float (&reg)[DP / 2], int l32, int hh) {
  f32x16 c = f32x16{};
  const LDS_AS char* row = tile + l32 * DP * 4;
  const int s = swz4<DP>(l32);
#pragma unroll
  for (int k4 = 0; k4 < DP / 8; ++k4) {
    const f32x4 a = lds_f4(row + ((hh * (DP / 8) + k4) ^ s) * 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = mfma_f32(a[e], reg[4 * k4 + e], c);
  }
  return c;
}
template <int DP>
__device__ __forceinline__ void tile_block(f32x16 (&acc)[DP / 32], const LDS_AS char* tile, const f32x16& s, int l32,
                                           int hh) {
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int r = 8 * (j >> 2) + 4 * hh + (j & 3), z = swz4<DP>(r);
#pragma unroll
    for (int dt = 0; dt < DP / 32; ++dt)
      acc[dt] = mfma_f32(lds_f1(tile + r * DP * 4 + ((8 * dt + (l32 >> 2)) ^ z) * 16 + (l32 & 3) * 4), s[j], acc[dt]);
  }
}
// Sums of the KS waves of a row block: wave ks leaves its accumulators (scaled
// by its weight) in its own LDS, [register][lane], and takes every KS-th group
// of four registers of the total.
template <int DP>
__device__ __forceinline__ void put_acc(LDS_AS char* base, const f32x16 (&acc)[DP / 32], float w, int lane) {
#pragma unroll
  for (int dt = 0; dt < DP / 32; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *(LDS_AS f32x4*)(base + ((dt * 4 + g) * 64 + lane) * 16) =
          f32x4{acc[dt][4 * g] * w, acc[dt][4 * g + 1] * w, acc[dt][4 * g + 2] * w, acc[dt][4 * g + 3] * w};
}
// f(column of the group, four values) for this wave's groups of the total.
template <int DP, int KS, typename F>
__device__ __forceinline__ void for_total(const LDS_AS char* base0, int stride, int ks, int lane, F f) {
#pragma unroll
  for (int q = 0; q < DP / 8 / KS; ++q) {
    const int grp = q * KS + ks;
    f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < KS; ++w) t += *(const LDS_AS f32x4*)(base0 + w * stride + (grp * 64 + lane) * 16);
    f(32 * (grp >> 2) + 8 * (grp & 3) + 4 * (lane >> 5), t);
  }
}

template <int DP, bool VARLEN, int KS>
__global__ __launch_bounds__(256, DP == 128 ? 1 : 2) void fa_fwd_f32_wave_kernel(const FwdParams p, int causal,
                                                                                float scale) {
  constexpr int DT = DP / 32, NL = DP / 8, QB = kF32Waves / KS;
  __shared__ __attribute__((aligned(1024))) char f32_smem[kF32Waves * 2 * kF32Tile<DP>];  // per wave: K tile, V tile
  __shared__ float st_m[kF32Waves][32], st_l[kF32Waves][32];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5, ks = wave % KS;
  const int bh = blockIdx.x, b = bh / p.Hq, h = bh - b * p.Hq;
  const int hk = h / (p.Hq / p.Hkv);
  int nq = p.Nq, nk = p.Nk;
  int64_t rq0 = 0, rk0 = 0;
  if (VARLEN) {
    rq0 = p.cu_q[b];
    nq = p.cu_q[b + 1] - (int)rq0;
    rk0 = p.cu_k[b];
    nk = p.cu_k[b + 1] - (int)rk0;
  }
  const int q0 = (gridDim.y - 1 - blockIdx.y) * 32 * QB;  // causal: the longest first
  if (q0 >= nq) return;  // uniform, before any barrier
  const int off = nk - nq, D = p.D;
  const float* Q = (const float*)p.q + (VARLEN ? 0 : (int64_t)b * p.sqb) + (int64_t)h * p.sqh + rq0 * p.sqn;
  const float* K = (const float*)p.k + (VARLEN ? 0 : (int64_t)b * p.skb) + (int64_t)hk * p.skh + rk0 * p.skn;
  const float* V = (const float*)p.v + (VARLEN ? 0 : (int64_t)b * p.svb) + (int64_t)hk * p.svh + rk0 * p.svn;
  const int qw = q0 + 32 * (wave / KS), qrow = qw + l32;
  const float sl2 = scale * kLog2e;
  LDS_AS char* Ks = (LDS_AS char*)f32_smem + wave * 2 * kF32Tile<DP>;
  LDS_AS char* Vs = Ks + kF32Tile<DP>;

  int kv_end = qw < nq ? nk : 0;
  if (causal) kv_end = min(kv_end, qw + 32 + off);
  const int nt = kv_end > 0 ? (kv_end + 31) / 32 : 0;
  load_tile_f32<DP>(Ks, K, p.skn, 32 * ks, ks < nt ? nk : 0, D, lane);
  load_tile_f32<DP>(Vs, V, p.svn, 32 * ks, ks < nt ? nk : 0, D, lane);
  float qreg[DP / 2];
  load_row_f32<DP>(qreg, Q, p.sqn, qrow, nq, D, hh);
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  float m = -INFINITY, l = 0.f;  // log2 units
  if (ks < nt) wait_vm<0>();
  for (int t = ks; t < nt; t += KS) {
    const int kt = 32 * t, next = t + KS < nt ? nk : 0;
    wait_vm<NL>();  // K has landed; V may still be in flight
    f32x16 s = tile_dims<DP>(Ks, qreg, l32, hh);
    wait_lds();
    load_tile_f32<DP>(Ks, K, p.skn, kt + 32 * KS, next, D, lane);
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kt + 8 * (i >> 2) + 4 * hh + (i & 3);
      float x = s[i] * sl2;
      if (key >= nk || (causal && key > qrow + off)) x = -INFINITY;
      s[i] = x;
      mx = fmaxf(mx, x);
    }
    const float m_new = fmaxf(m, hmax(mx));
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2f(m - m_use);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = exp2f(s[i] - m_use);
      sum += s[i];
    }
    l = l * alpha + hsum(sum);
    m = m_new;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] *= alpha;
    wait_vm<NL>();  // V has landed; the next K may still be in flight
    tile_block<DP>(acc, Vs, s, l32, hh);
    wait_lds();
    load_tile_f32<DP>(Vs, V, p.svn, kt + 32 * KS, next, D, lane);
  }
  wait_vm<0>();  // the last refills (empty) are done with LDS
  float* O = (float*)p.o + (VARLEN ? 0 : (int64_t)b * p.sob) + (int64_t)h * p.soh + (rq0 + qrow) * p.son;
  float* L = p.lse == nullptr ? nullptr
                              : p.lse + (VARLEN ? 0 : (int64_t)b * p.slb) + (int64_t)h * p.slh + (rq0 + qrow) * p.sln;
  if constexpr (KS == 1) {
    if (qrow < nq) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d = 32 * dt + 8 * g + 4 * hh;
          if (d < D)
            *(f32x4*)(O + d) = f32x4{acc[dt][4 * g] * inv, acc[dt][4 * g + 1] * inv, acc[dt][4 * g + 2] * inv,
                                     acc[dt][4 * g + 3] * inv};
        }
      if (L != nullptr && hh == 0) *L = l > 0.f ? (m + __log2f(l)) * kLn2f : -INFINITY;
    }
  } else {
    if (hh == 0) {
      st_m[wave][l32] = m;
      st_l[wave][l32] = l;
    }
    __syncthreads();
    const int w0 = wave - ks;
    float M = -INFINITY, total = 0.f;
#pragma unroll
    for (int w = 0; w < KS; ++w) M = fmaxf(M, st_m[w0 + w][l32]);
    const float Mu = M == -INFINITY ? 0.f : M;
#pragma unroll
    for (int w = 0; w < KS; ++w) total += st_l[w0 + w][l32] * exp2f(st_m[w0 + w][l32] - Mu);
    put_acc<DP>(Ks, acc, exp2f(m - Mu) * (total > 0.f ? 1.f / total : 0.f), lane);
    __syncthreads();
    const LDS_AS char* base0 = (const LDS_AS char*)f32_smem + w0 * 2 * kF32Tile<DP>;
    for_total<DP, KS>(base0, 2 * kF32Tile<DP>, ks, lane, [&](int d, f32x4 v) {
      if (qrow < nq && d < D) *(f32x4*)(O + d) = v;
    });
    if (L != nullptr && hh == 0 && ks == 0 && qrow < nq) *L = total > 0.f ? (M + __log2f(total)) * kLn2f : -INFINITY;
  }
}

// dQ, and (lse * log2e, delta) pairs of every query row of the block for the
// dK/dV kernel (+inf and 0 where a row sees no key or is past nq).
template <int DP, int KS>
__global__ __launch_bounds__(256, DP == 128 ? 1 : 2) void fa_bwd_dq_f32_wave_kernel(const BwdParams p, int causal) {
  constexpr int DT = DP / 32, NL = DP / 8, QB = kF32Waves / KS;
  __shared__ __attribute__((aligned(1024))) char f32_smem[kF32Waves * 2 * kF32Tile<DP>];  // per wave: K tile, V tile
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5, ks = wave % KS;
  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H;
  const int nq = p.Nq, nk = p.Nk, D = p.D, off = nk - nq;
  const float* K = (const float*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const float* V = (const float*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh;
  const int qw = (gridDim.y - 1 - blockIdx.y) * 32 * QB + 32 * (wave / KS), qrow = qw + l32;
  const bool valid = qrow < nq;
  LDS_AS char* Ks = (LDS_AS char*)f32_smem + wave * 2 * kF32Tile<DP>;
  LDS_AS char* Vs = Ks + kF32Tile<DP>;
  int kv_end = qw < nq ? nk : 0;
  if (causal) kv_end = min(kv_end, qw + 32 + off);
  const int nt = kv_end > 0 ? (kv_end + 31) / 32 : 0;
  load_tile_f32<DP>(Vs, V, p.svn, 32 * ks, ks < nt ? nk : 0, D, lane);
  load_tile_f32<DP>(Ks, K, p.skn, 32 * ks, ks < nt ? nk : 0, D, lane);
  float qreg[DP / 2], doreg[DP / 2];
  load_row_f32<DP>(qreg, (const float*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh, p.sqn, qrow, nq, D, hh);
  load_row_f32<DP>(doreg, (const float*)p.dout + (int64_t)b * p.sdob + (int64_t)h * p.sdoh, p.sdon, qrow, nq, D,
                   hh);
  float dpart = 0.f;
  {
    float oreg[DP / 2];
    load_row_f32<DP>(oreg, (const float*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh, p.son, qrow, nq, D, hh);
#pragma unroll
    for (int kk = 0; kk < DP / 2; ++kk) dpart += doreg[kk] * oreg[kk];
  }
  const float delta = hsum(dpart);
  float L2 = valid ? p.lse[(int64_t)b * p.slb + (int64_t)h * p.slh + (int64_t)qrow * p.sln] : INFINITY;
  if (L2 == -INFINITY) L2 = INFINITY;  // a row that sees no key: P = 0
  L2 *= kLog2e;
  if (hh == 0 && ks == 0 && qrow < p.nq_pad)
    *(float2*)(p.ld + (int64_t)b * p.sldb + (int64_t)h * p.sldh + 2 * (int64_t)qrow) = float2{L2, valid ? delta : 0.f};
  const float sl2 = p.scale * kLog2e;
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  if (ks < nt) wait_vm<0>();
  for (int t = ks; t < nt; t += KS) {
    const int kt = 32 * t, next = t + KS < nt ? nk : 0;
    wait_vm<NL>();  // V has landed; K may still be in flight
    const f32x16 dp = tile_dims<DP>(Vs, doreg, l32, hh);
    wait_lds();
    load_tile_f32<DP>(Vs, V, p.svn, kt + 32 * KS, next, D, lane);
    wait_vm<NL>();  // K has landed
    f32x16 s = tile_dims<DP>(Ks, qreg, l32, hh);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kt + 8 * (i >> 2) + 4 * hh + (i & 3);
      float pr = exp2f(s[i] * sl2 - L2);
      if (key >= nk || (causal && key > qrow + off)) pr = 0.f;
      s[i] = pr * (dp[i] - delta);
    }
    tile_block<DP>(acc, Ks, s, l32, hh);
    wait_lds();
    load_tile_f32<DP>(Ks, K, p.skn, kt + 32 * KS, next, D, lane);
  }
  wait_vm<0>();
  float* dQ = (float*)p.dq + (int64_t)b * p.sdqb + (int64_t)h * p.sdqh + (int64_t)qrow * p.sdqn;
  if constexpr (KS > 1) {
    put_acc<DP>(Ks, acc, p.scale, lane);
    __syncthreads();
    for_total<DP, KS>((const LDS_AS char*)f32_smem + (wave - ks) * 2 * kF32Tile<DP>, 2 * kF32Tile<DP>, ks, lane,
                      [&](int d, f32x4 v) {
                        if (valid && d < D) *(f32x4*)(dQ + d) = v;
                      });
  } else if (valid) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * dt + 8 * g + 4 * hh;
        if (d < D)
          *(f32x4*)(dQ + d) = f32x4{acc[dt][4 * g] * p.scale, acc[dt][4 * g + 1] * p.scale, acc[dt][4 * g + 2] * p.scale,
                                    acc[dt][4 * g + 3] * p.scale};
      }
  }
}

// dK, dV of 32 keys per wave (or per KS waves) over the query tiles.
template <int DP, int KS>
__global__ __launch_bounds__(256, 1) void fa_bwd_dkdv_f32_wave_kernel(const BwdParams p, int causal) {
  constexpr int DT = DP / 32, NL = DP / 8, KB = kF32Waves / KS;
  constexpr int WB = 2 * kF32Tile<DP> + 256;  // Q tile, dO tile, their (L, delta) pairs
  __shared__ __attribute__((aligned(1024))) char f32_smem[kF32Waves * WB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5, ks = wave % KS;
  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H;
  const int nq = p.Nq, nk = p.Nk, D = p.D, off = nk - nq;
  const float* Q = (const float*)p.q + (int64_t)b * p.sqb + (int64_t)h * p.sqh;
  const float* dO = (const float*)p.dout + (int64_t)b * p.sdob + (int64_t)h * p.sdoh;
  const float* LD = p.ld + (int64_t)b * p.sldb + (int64_t)h * p.sldh;
  const int kw = blockIdx.y * 32 * KB + 32 * (wave / KS), krow = kw + l32;
  LDS_AS char* Qs = (LDS_AS char*)f32_smem + wave * WB;
  LDS_AS char* Ds = Qs + kF32Tile<DP>;
  LDS_AS char* Ls = Ds + kF32Tile<DP>;
  const int t0 = causal ? max(0, kw - off) / 32 : 0;  // first tile with a query that sees the block
  const int nt = kw < nk ? (nq + 31) / 32 : 0;
  // (lse * log2e, delta) of the 32 queries of tile t, 256 bytes: one 4-byte
  // direct load. nq_pad is a multiple of 32, so whole tiles of pairs exist.
  auto load_ld = [&](int t) {
    const bool live = t < nt;
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(live ? LD + 64 * (int64_t)t : LD, live ? 256 : 0);
    dma4(rs, (LDS_AS void*)Ls, lane * 4);
  };
  int t = t0 + ks;
  load_tile_f32<DP>(Qs, Q, p.sqn, 32 * t, t < nt ? nq : 0, D, lane);
  load_tile_f32<DP>(Ds, dO, p.sdon, 32 * t, t < nt ? nq : 0, D, lane);
  load_ld(t);
  float kreg[DP / 2], vreg[DP / 2];
  load_row_f32<DP>(kreg, (const float*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh, p.skn, krow, nk, D, hh);
  load_row_f32<DP>(vreg, (const float*)p.v + (int64_t)b * p.svb + (int64_t)h * p.svh, p.svn, krow, nk, D, hh);
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dk[dt] = f32x16{};
    dv[dt] = f32x16{};
  }
  const float sl2 = p.scale * kLog2e;
  wait_vm<0>();
  for (; t < nt; t += KS) {
    const int qt = 32 * t, tn = t + KS, next = tn < nt ? nq : 0;
    wait_vm<NL + 1>();  // Q has landed; dO and the pairs may still be in flight
    f32x16 s = tile_dims<DP>(Qs, kreg, l32, hh);
    wait_vm<0>();  // so have they
    f32x16 dp = tile_dims<DP>(Ds, vreg, l32, hh);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 8 * (i >> 2) + 4 * hh + (i & 3), q = qt + r;
      const LDS_AS char* pair = Ls + r * 8;
      float pr = exp2f(s[i] * sl2 - lds_f1(pair));
      if (q >= nq || krow >= nk || (causal && krow > q + off)) pr = 0.f;
      s[i] = pr;
      dp[i] = pr * (dp[i] - lds_f1(pair + 4));
    }
    tile_block<DP>(dk, Qs, dp, l32, hh);
    wait_lds();
    load_tile_f32<DP>(Qs, Q, p.sqn, 32 * tn, next, D, lane);
    tile_block<DP>(dv, Ds, s, l32, hh);
    wait_lds();
    load_tile_f32<DP>(Ds, dO, p.sdon, 32 * tn, next, D, lane);
    load_ld(tn);
  }
  wait_vm<0>();
  const bool valid = krow < nk;
  float* dK = (float*)p.dk + (int64_t)b * p.sdkb + (int64_t)h * p.sdkh + (int64_t)krow * p.sdkn;
  float* dV = (float*)p.dv + (int64_t)b * p.sdvb + (int64_t)h * p.sdvh + (int64_t)krow * p.sdvn;
  if constexpr (KS > 1) {
    put_acc<DP>(Qs, dk, p.scale, lane);
    put_acc<DP>(Ds, dv, 1.f, lane);
    __syncthreads();
    const LDS_AS char* base0 = (const LDS_AS char*)f32_smem + (wave - ks) * WB;
    for_total<DP, KS>(base0, WB, ks, lane, [&](int d, f32x4 v) {
      if (valid && d < D) *(f32x4*)(dK + d) = v;
    });
    for_total<DP, KS>(base0 + kF32Tile<DP>, WB, ks, lane, [&](int d, f32x4 v) {
      if (valid && d < D) *(f32x4*)(dV + d) = v;
    });
  } else if (valid) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * dt + 8 * g + 4 * hh;
        if (d < D) {
          *(f32x4*)(dK + d) = f32x4{dk[dt][4 * g] * p.scale, dk[dt][4 * g + 1] * p.scale, dk[dt][4 * g + 2] * p.scale,
                                    dk[dt][4 * g + 3] * p.scale};
          *(f32x4*)(dV + d) = f32x4{dv[dt][4 * g], dv[dt][4 * g + 1], dv[dt][4 * g + 2], dv[dt][4 * g + 3]};
        }
      }
  }
}

// Whether 16-byte loads can address a tensor's rows: unit head-dim stride,
// 16-byte aligned base, other strides multiples of 4, rows that do not
// overlap, and 32 of them within the 2^31 bytes of a buffer descriptor.
static bool rows16(const void* ptr, int D, int64_t sb, int64_t sh, int64_t sn, int64_t sd) {
  return sd == 1 && (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0 && sb % 4 == 0 && sh % 4 == 0 && sn % 4 == 0 &&
         sn >= D && sn <= (int64_t(1) << 22);
}
// Waves per block of 32 stationary rows: as many as keep the launch within one
// wave per SIMD (1024), or two when causal, where the longest block takes twice
// the mean: 2x16x1024x128 causal (1024 blocks), forward + backward, 728 us at one
// wave per block, 430 at four.
static int f32_wave_split(long long blocks, int causal) {
  const long long simds = causal ? 2048 : 1024;
  return blocks * 4 <= simds ? 4 : (blocks * 2 <= simds ? 2 : 1);
}
// Blocks are the y axis of the grid (the heads the x axis, so that every
// head's longest blocks start first).
static bool f32_grid_ok(int rows) { return rows <= 65535 * 32; }

template <int DP, bool VARLEN>
static hipError_t launch_fwd_f32_wave(const FwdParams& p, int causal, float scale, hipStream_t s) {
  const int blocks = (p.Nq + 31) / 32, bh = p.B * p.Hq;
  switch (f32_wave_split((long long)blocks * bh, causal)) {
    case 4:
      hipLaunchKernelGGL((fa_fwd_f32_wave_kernel<DP, VARLEN, 4>), dim3(bh, blocks), dim3(256), 0, s, p, causal, scale);
      break;
    case 2:
      hipLaunchKernelGGL((fa_fwd_f32_wave_kernel<DP, VARLEN, 2>), dim3(bh, (blocks + 1) / 2), dim3(256), 0, s, p, causal, scale);
      break;
    default:
      hipLaunchKernelGGL((fa_fwd_f32_wave_kernel<DP, VARLEN, 1>), dim3(bh, (blocks + 3) / 4), dim3(256), 0, s, p, causal, scale);
  }
  return hipGetLastError();
}

template <int DP>
static hipError_t launch_fwd_f32(const FwdParams& p, bool causal, bool varlen, float scale, hipStream_t s) {
  const int D = p.D;
  if (D % 4 == 0 && f32_grid_ok(p.Nq) && rows16(p.q, D, p.sqb, p.sqh, p.sqn, p.sqd) &&
      rows16(p.k, D, p.skb, p.skh, p.skn, p.skd) && rows16(p.v, D, p.svb, p.svh, p.svn, p.svd) &&
      rows16(p.o, D, p.sob, p.soh, p.son, p.sod))
    return varlen ? launch_fwd_f32_wave<DP, true>(p, causal, scale, s) : launch_fwd_f32_wave<DP, false>(p, causal, scale, s);
  dim3 grid((p.Nq + 127) / 128, p.B * p.Hq);
  if (varlen)
    hipLaunchKernelGGL((fa_fwd_f32_kernel<DP, true>), grid, dim3(256), 0, s, p, (int)causal, scale);
  else
    hipLaunchKernelGGL((fa_fwd_f32_kernel<DP, false>), grid, dim3(256), 0, s, p, (int)causal, scale);
  return hipGetLastError();
}

hipError_t fwd_f32(const FwdParams& p, int dp, bool causal, bool varlen, float scale, hipStream_t s) {
  switch (dp) {
    case 32: return launch_fwd_f32<32>(p, causal, varlen, scale, s);
    case 64: return launch_fwd_f32<64>(p, causal, varlen, scale, s);
    default: return launch_fwd_f32<128>(p, causal, varlen, scale, s);
  }
}

template <int DP, int KS>
static hipError_t launch_dq_f32_wave(const BwdParams& p, int causal, hipStream_t s) {
  hipLaunchKernelGGL((fa_bwd_dq_f32_wave_kernel<DP, KS>), dim3(p.B * p.H, (p.Nq + 128 / KS - 1) / (128 / KS)), dim3(256), 0, s,
                     p, causal);
  return hipGetLastError();
}
template <int DP, int KS>
static hipError_t launch_dkdv_f32_wave(const BwdParams& p, int causal, hipStream_t s) {
  hipLaunchKernelGGL((fa_bwd_dkdv_f32_wave_kernel<DP, KS>), dim3(p.B * p.H, (p.Nk + 128 / KS - 1) / (128 / KS)), dim3(256), 0,
                     s, p, causal);
  return hipGetLastError();
}
template <int DP>
static hipError_t launch_bwd_f32_wave(const BwdParams& p, int causal, hipStream_t s) {
  hipError_t e = hipSuccess;
  const long long bh = (long long)p.B * p.H;
  if (p.Nq > 0) {
    const int ks = f32_wave_split(bh * ((p.Nq + 31) / 32), causal);
    e = ks == 4 ? launch_dq_f32_wave<DP, 4>(p, causal, s)
                : (ks == 2 ? launch_dq_f32_wave<DP, 2>(p, causal, s) : launch_dq_f32_wave<DP, 1>(p, causal, s));
    if (e != hipSuccess) return e;
  }
  if (p.Nk > 0) {
    const int ks = f32_wave_split(bh * ((p.Nk + 31) / 32), causal);
    e = ks == 4 ? launch_dkdv_f32_wave<DP, 4>(p, causal, s)
                : (ks == 2 ? launch_dkdv_f32_wave<DP, 2>(p, causal, s) : launch_dkdv_f32_wave<DP, 1>(p, causal, s));
  }
  return e;
}

template <int DP>
static hipError_t launch_bwd_f32(const BwdParams& p, bool causal, hipStream_t s) {
  const int D = p.D;
  if (D % 4 == 0 && f32_grid_ok(p.Nq) && f32_grid_ok(p.Nk) && rows16(p.q, D, p.sqb, p.sqh, p.sqn, p.sqd) &&
      rows16(p.k, D, p.skb, p.skh, p.skn, p.skd) && rows16(p.v, D, p.svb, p.svh, p.svn, p.svd) &&
      rows16(p.o, D, p.sob, p.soh, p.son, p.sod) &&
      rows16(p.dout, D, p.sdob, p.sdoh, p.sdon, p.sdod) && rows16(p.dq, D, p.sdqb, p.sdqh, p.sdqn, p.sdqd) &&
      rows16(p.dk, D, p.sdkb, p.sdkh, p.sdkn, p.sdkd) && rows16(p.dv, D, p.sdvb, p.sdvh, p.sdvn, p.sdvd))
    return launch_bwd_f32_wave<DP>(p, causal, s);
  if (p.Nq > 0) {
    hipLaunchKernelGGL((fa_bwd_dq_f32_kernel<DP>), dim3((p.Nq + 127) / 128, p.B * p.H), dim3(256), 0, s, p,
                       (int)causal);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (p.Nk > 0) {
    hipLaunchKernelGGL((fa_bwd_dkdv_f32_kernel<DP>), dim3((p.Nk + 127) / 128, p.B * p.H), dim3(256), 0, s, p,
                       (int)causal);
    return hipGetLastError();
  }
  return hipSuccess;
}

hipError_t bwd_f32(const BwdParams& p, int dp, bool causal, hipStream_t s) {
  switch (dp) {
    case 32: return launch_bwd_f32<32>(p, causal, s);
    case 64: return launch_bwd_f32<64>(p, causal, s);
    default: return launch_bwd_f32<128>(p, causal, s);
  }
}

}  // namespace lsfa
