// Skinny GEMM on MFMA, 3 rows and more: y[M, N] = x[M, K] @ W[K, N] (W in the
// model's [in, out] row-major layout, bf16/fp16, fp32 accumulate, one rounding),
// for the decode steps of a batch, where the VALU kernel (fa_gemv.hip) spends
// more time on its products than on the weight bytes.
//
// The product is a pass over W (2 M FLOP per 2-byte weight, M <= 32), so it is
// bound by HBM as long as W streams without gaps. W therefore goes from memory
// straight into registers, two steps deep, with no LDS, barrier or reuse
// between a wave's load and its use:
//   A wave owns 128 columns and walks K in steps of 32 rows. Lane (c, kg) =
//   (l % 16, l / 16) loads 16 bytes (columns 8c .. 8c+7) of the eight rows
//   8 kg .. 8 kg + 7 of a step, so a load instruction covers four 256-byte row
//   segments and a step is eight instructions, 8 KB. The lane then holds an
//   8 x 8 block with K across its registers; 32 v_perm_b32 turn it into eight
//   operands of eight K values, one per column, and operand j of the wave is
//   the W^T tile {8 c + j} x {32 rows} of v_mfma_f32_16x16x32 (an operand's
//   rows may be any 16 columns, so the stride of 8 costs nothing; the permutes
//   take 128 issue cycles per 8 KB, and a CU's share of HBM delivers 8 KB in
//   about 750).
//   x^T is the B operand: lane (row l % 16, kg) loads 16 bytes of its row.
//   The four waves of a workgroup take the steps of its K-range in turn and
//   add their sums through LDS.
//   Grid (N / 128 column blocks, splits). With one split a workgroup rounds its
//   sums into y; otherwise partial sums, arrival counters and the last
//   workgroup's reduction work as in fa_gemv.hip (device-scope atomic stores
//   and loads, no cache maintenance).
// Measured at 8 rows, bf16, graph replays over weights that no cache holds, in
// us, against W through LDS in one-shot workgroups of 256 rows x 128 columns:
//   4096 -> 4096+1024+1024 (50 MB): 21.4 -> 13.5    4096 -> 4096 (34 MB): 16.9 -> 10.9
//   4096 -> 2 x 14336 (235 MB): 68.3 -> 42.3 (5.6 TB/s)    14336 -> 4096: 44.4 -> 23.1
//   4096 -> 128256 (1.05 GB): 286 -> 165 (6.4 TB/s)
// and at 32 rows 37.1 -> 16.4, 31.3 -> 13.7, 99.4 -> 46.2, 85.5 -> 27.2, 406 -> 177.
// Three or four steps in flight, or eight waves, change nothing (+-3%): what is
// left on the small products is the launch's own latency and the reduction.
//
// Above 32 rows (grid z, blocks of 64 rows, eight waves) the same kernel serves
// products whose tiles fit the GPU once, where a library GEMM's larger tiles
// leave most CUs idle: us against hipBLASLt at 64 / 128 / 256 / 512 rows,
//   4096 -> 4096+1024+1024: 22.5 / 28 / 37.5 / - against 82 / 78 / 64 (three launches)
//   4096 -> 4096: 18.9 / 20.5 / 26.0 / 35.4 against 28.2 / 39.6 / 25.7 / 39.4
//   14336 -> 4096: 36.5 / 46.5 / 68.0 / 110 against 103 / 124 / 98.5 / 124
//   2048 -> 2048: 15.7 / 15.7 / 14.2 / 16.4 against 15.6 / 12.6 / 13.0 / 14.1: left to
//   the library, as is what has more tiles than CUs (4096 -> 2 x 14336 at 128 rows 92
//   against 86, at 512 288 against 148).
// There it is bound by its loads: every wave reads x rows of its own steps, in
// 64-byte pieces, and W passes L1 once per row block (with both from L1 the same
// loop runs at 950 TFLOP/s). Four waves of twice the steps: 4% slower; 128-row
// blocks (512 VGPRs): slower everywhere.
#include "fa_common.hpp"

namespace lsfa {

constexpr int kMfmaCols = 128;   // columns per workgroup
constexpr int kMfmaStep = 32;    // rows of W per step
constexpr int kMfmaDepth = 2;    // steps of a wave in flight
constexpr int kMfmaLd = kMfmaCols + 4;  // row stride of the wave sums in LDS (floats)
constexpr int kMfmaCounterSlots = 16;

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// 16-byte loads, the first non-temporal; lanes whose offset is out of range read zero.
__device__ __forceinline__ u32x4 load16_nt(__amdgpu_buffer_rsrc_t rs, int voff, int soff) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 2));
}
__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t rs, int voff, int soff) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 0));
}

// MT: blocks of 16 rows (M <= 16 MT). GATE: x stands for silu(xg) * x.
template <typename T, int MT, int NW, bool GATE>
__global__ __launch_bounds__(64 * NW, 2) void fa_gemv_mfma_kernel(const GemvParams p) {
  constexpr int DEPTH = kMfmaDepth;
  constexpr bool WNT = MT <= 2;  // one row block: W is read once
  using X8 = typename VecT<T>::x8;
  extern __shared__ __attribute__((aligned(16))) float wave_sums[];  // [NW / 2][16 MT][kMfmaLd]
  __shared__ int last_arrival;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int split = blockIdx.y;
  const int m0 = blockIdx.z * 16 * MT;  // first row of the row block
  const int rows = min(p.M - m0, 16 * MT);
  const int k_begin = split * p.kc;
  const int k_len = max(0, min(p.K, k_begin + p.kc) - k_begin);

  // Matrix of this column block (every matrix's width is a multiple of 128).
  const int n_blk = blockIdx.x * kMfmaCols;  // virtual column
  const int g = (n_blk >= p.col_off[1]) + (n_blk >= p.col_off[2]) + (n_blk >= p.col_off[3]);
  const int col_off = g == 0 ? p.col_off[0] : (g == 1 ? p.col_off[1] : (g == 2 ? p.col_off[2] : p.col_off[3]));
  const T* w = (const T*)(g == 0 ? p.w[0] : (g == 1 ? p.w[1] : (g == 2 ? p.w[2] : p.w[3])));
  T* y = (T*)(g == 0 ? p.y[0] : (g == 1 ? p.y[1] : (g == 2 ? p.y[2] : p.y[3])));
  const int64_t sw = g == 0 ? p.sw[0] : (g == 1 ? p.sw[1] : (g == 2 ? p.sw[2] : p.sw[3]));
  const int64_t sy = g == 0 ? p.sy[0] : (g == 1 ? p.sy[1] : (g == 2 ? p.sy[2] : p.sy[3]));
  const int n_local = n_blk - col_off;

  // Rows of x past M repeat the last one: their sums are never stored.
  int xo[MT], go[GATE ? MT : 1];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = min(16 * t + c, rows - 1);
    xo[t] = (int)(m * p.sx * 2) + 16 * kg;
    if (GATE) go[t] = (int)(m * p.sxg * 2) + 16 * kg;
  }
  const T* xk = (const T*)p.x + (int64_t)m0 * p.sx + k_begin;
  const T* gk = GATE ? (const T*)p.xg + (int64_t)m0 * p.sxg + k_begin : nullptr;
  const T* wk = w + (int64_t)k_begin * sw + n_local;
  const int row_bytes = (int)(sw * 2);
  const int lane_off = 8 * kg * row_bytes + 16 * c;

  struct Step {
    u32x4 w[8];
    u32x4 x[MT];
    u32x4 g[GATE ? MT : 1];
  };
  // The loads of one step, always the same number of them, so that the wait
  // before a step's use counts the next step's loads as still in flight. K is
  // a multiple of 8, so a lane's eight rows are inside the K-range or past it
  // together; past it W and x read as zero (offset out of range: no memory
  // access).
  auto load = [&](int step, Step& s) {
    const int k = step * kMfmaStep, kc = min(k, k_len);
    // (or-ed into the offsets: a select of offsets turns into branches around the loads)
    const int past = k + 8 * kg < k_len ? 0 : (int)0x80000000;
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(wk + (int64_t)kc * sw, 0x7fffffff);
    const int voff = lane_off | past;
#pragma unroll
    for (int r = 0; r < 8; ++r) s.w[r] = WNT ? load16_nt(rs, voff, r * row_bytes) : load16(rs, voff, r * row_bytes);
    const __amdgpu_buffer_rsrc_t xs = tile_rsrc(xk + kc, 0x7fffffff);
#pragma unroll
    for (int t = 0; t < MT; ++t) s.x[t] = load16(xs, xo[t] | past, 0);
    if constexpr (GATE) {
      const __amdgpu_buffer_rsrc_t gs = tile_rsrc(gk + kc, 0x7fffffff);
#pragma unroll
      for (int t = 0; t < MT; ++t) s.g[t] = load16(gs, go[t] | past, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[MT][8];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto use = [&](const Step& s) {
    X8 xb[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      u32x4 raw = s.x[t];
      if (GATE) {
        // silu(gate) rounded to T, times x rounded to T: the two roundings of
        // F.silu(gate) * up.
        const X8 up = __builtin_bit_cast(X8, raw), gt = __builtin_bit_cast(X8, s.g[t]);
        X8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float gv = (float)gt[e];
          const float act = (float)(T)(gv / (1.0f + expf(-gv)));
          o[e] = (T)(act * (float)up[e]);
        }
        raw = __builtin_bit_cast(u32x4, o);
      }
      xb[t] = __builtin_bit_cast(X8, raw);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // columns 2q and 2q + 1 of the lane's eight
      u32x4 lo, hi;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[e] = __builtin_amdgcn_perm(s.w[2 * e + 1][q], s.w[2 * e][q], 0x05040100u);
        hi[e] = __builtin_amdgcn_perm(s.w[2 * e + 1][q], s.w[2 * e][q], 0x07060302u);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        acc[t][2 * q] = mfma16(__builtin_bit_cast(X8, lo), xb[t], acc[t][2 * q]);
        acc[t][2 * q + 1] = mfma16(__builtin_bit_cast(X8, hi), xb[t], acc[t][2 * q + 1]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  if (k_len > 0) {  // uniform: an empty K-range reads neither x nor W
    const int steps = (k_len + kMfmaStep - 1) / kMfmaStep;
    Step s[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(wave + d * NW, s[d]);
    for (int st = wave; st < steps; st += DEPTH * NW) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        use(s[d]);
        load(st + (DEPTH + d) * NW, s[d]);
      }
    }
  }

  // acc[t][j] register i holds row 16 t + l % 16 of column 32 kg + 8 i + j. The
  // upper half of the waves hands its sums to the lower half, which adds them
  // to its own, so that LDS holds NW / 2 blocks.
  constexpr int HW = NW / 2;
  auto slot = [&](int t) { return wave_sums + ((wave % HW) * 16 * MT + 16 * t + c) * kMfmaLd + 32 * kg; };
  if (wave >= HW) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        *(f32x4*)(slot(t) + 8 * i) = f32x4{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
        *(f32x4*)(slot(t) + 8 * i + 4) = f32x4{acc[t][4][i], acc[t][5][i], acc[t][6][i], acc[t][7][i]};
      }
  }
  __syncthreads();
  if (wave < HW) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        *(f32x4*)(slot(t) + 8 * i) += f32x4{acc[t][0][i], acc[t][1][i], acc[t][2][i], acc[t][3][i]};
        *(f32x4*)(slot(t) + 8 * i + 4) += f32x4{acc[t][4][i], acc[t][5][i], acc[t][6][i], acc[t][7][i]};
      }
  }
  __syncthreads();
  // The block's sums in pairs of columns, row by row: thread tid takes pairs
  // tid, tid + 64 NW, ...
  constexpr int IT = 16 * MT * (kMfmaCols / 2) / (64 * NW);
  const int pairs = rows * (kMfmaCols / 2);
  const int64_t sstride = (int64_t)p.N * p.M / 2;
  uint64_t* base = (uint64_t*)(p.partial + (int64_t)n_blk * p.M + (int64_t)m0 * kMfmaCols);
  auto put = [&](int pair, float s0, float s1) {
    T* dst = y + (int64_t)(m0 + pair / (kMfmaCols / 2)) * sy + n_local + 2 * (pair % (kMfmaCols / 2));
    dst[0] = (T)s0;
    dst[1] = (T)s1;
  };
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int pair = tid + it * 64 * NW;
    if (pair < pairs) {
      const float* src = wave_sums + (pair / (kMfmaCols / 2)) * kMfmaLd + 2 * (pair % (kMfmaCols / 2));
      float s0 = src[0], s1 = src[1];
#pragma unroll
      for (int wv = 1; wv < HW; ++wv) {
        s0 += src[wv * 16 * MT * kMfmaLd];
        s1 += src[wv * 16 * MT * kMfmaLd + 1];
      }
      if (p.splits == 1)
        put(pair, s0, s1);
      else
        __hip_atomic_store(base + split * sstride + pair,
                           (uint64_t)__float_as_uint(s0) | (uint64_t)__float_as_uint(s1) << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (p.splits == 1) return;
  // Handoff to the workgroup that arrives last, built on gfx950's device
  // coherence rather than on release/acquire fences: the partials are
  // agent-scope atomic stores (write-through to the device-coherent level,
  // sc1), every wave waits for their completion (vmcnt(0)) before the
  // barrier and thread 0's agent-scope counter RMWs, and the last workgroup
  // reads them with agent-scope atomic loads (sc1: never a stale line of its
  // own XCD's L2) issued only after its RMW has returned. Release/acquire
  // fences at agent scope would be the HIP memory model's way; they lower to
  // a whole-L2 write-back (buffer_wbl2 sc1) per arrival and an invalidate
  // (buffer_inv sc1) per acquire, and measured 1.4-1.9x slower on the
  // LM-head product (6.7 -> 3.6-4.8 TB/s), more on the narrow decode
  // projections whose ~1000 workgroups each would pay a write-back.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the partials have reached device scope
  __syncthreads();
  if (tid == 0) {
    int* ctr = p.counters + (blockIdx.z * gridDim.x + blockIdx.x) * kMfmaCounterSlots;
    // One counter for up to eight splits (the arrivals are spread over more
    // than the 175 ns that each takes), two levels above.
    bool last = true;
    if (p.splits > 8) {
      const int group = split & 7;
      const int group_size = (p.splits - group + 7) >> 3;
      last = __hip_atomic_fetch_add(ctr + group, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == group_size - 1;
      if (last) __hip_atomic_store(ctr + group, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (last) {
      last = __hip_atomic_fetch_add(ctr + 8, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == min(p.splits, 8) - 1;
      if (last) __hip_atomic_store(ctr + 8, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    last_arrival = last;
  }
  __syncthreads();
  if (!last_arrival) return;
  // The last workgroup adds the block's partials, contiguous per split, in
  // split order, the loads of up to four splits in flight together.
  float t0[IT], t1[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) t0[it] = t1[it] = 0.f;
  constexpr int SB = IT <= 4 ? 4 : 2;
  for (int s0 = 0; s0 < p.splits; s0 += SB) {
    uint64_t v[SB][IT];
#pragma unroll
    for (int b = 0; b < SB; ++b)
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        const int pair = tid + it * 64 * NW;
        v[b][it] = (s0 + b < p.splits && pair < pairs)
                       ? __hip_atomic_load(base + (s0 + b) * sstride + pair, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                       : 0;
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < SB; ++b)
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        t0[it] += __uint_as_float((uint32_t)v[b][it]);
        t1[it] += __uint_as_float((uint32_t)(v[b][it] >> 32));
      }
  }
#pragma unroll
  for (int it = 0; it < IT; ++it)
    if (tid + it * 64 * NW < pairs) put(tid + it * 64 * NW, t0[it], t1[it]);
}

template <typename T, int MT, int NW, bool GATE>
static hipError_t launch_gemv_mfma(const GemvParams& p, hipStream_t s) {
  const dim3 grid((unsigned)(p.N / kMfmaCols), (unsigned)p.splits, (unsigned)((p.M + 16 * MT - 1) / (16 * MT)));
  const size_t lds = (size_t)(NW / 2) * 16 * MT * kMfmaLd * 4;
  hipLaunchKernelGGL((fa_gemv_mfma_kernel<T, MT, NW, GATE>), grid, dim3(64 * NW), lds, s, p);
  return hipGetLastError();
}

template <typename T>
static hipError_t dispatch_gemv_mfma(const GemvParams& p, hipStream_t s) {
  if (p.M <= 16) return p.xg ? launch_gemv_mfma<T, 1, 4, true>(p, s) : launch_gemv_mfma<T, 1, 4, false>(p, s);
  if (p.M <= 32) return p.xg ? launch_gemv_mfma<T, 2, 4, true>(p, s) : launch_gemv_mfma<T, 2, 4, false>(p, s);
  return launch_gemv_mfma<T, 4, 8, false>(p, s);
}

// Host entry used by the C ABI layer: arguments validated, every matrix's
// width a multiple of 128, K and kc multiples of 8, M >= 3, no gate above 32
// rows.
hipError_t gemv_mfma(const GemvParams& p, bool is_bf16, hipStream_t s) {
  if (p.M == 0 || p.N == 0) return hipSuccess;
  return is_bf16 ? dispatch_gemv_mfma<__bf16>(p, s) : dispatch_gemv_mfma<_Float16>(p, s);
}

}  // namespace lsfa
