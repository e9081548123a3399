// FlashAttention backward for gfx950 (bf16/fp16 operands, fp32 accumulate).
//
// Math (kernels/flash_attention_backward.py:290-330): with the saved
// L = m + ln(l), P = exp(S*scale - L) is recomputed exactly; then
//   delta_i = rowsum(dO_i * O_i)                       (:211-229)
//   dV += P^T dO      (P rounded to the input dtype, :316)
//   dP  = dO V^T
//   dS  = P * (dP - delta)  (rounded to the input dtype, :319)
//   dK += dS^T Q * scale,   dQ += dS K * scale.
//
// Unlike the reference (one key-stationary kernel with fp32 atomic adds into
// a dq workspace, :323-325, followed by a cast, :382), the work is split into
// two kernels; by default
//   fa_bwd_dq_kernel   : query-stationary. Its prologue does the reference's
//                        preprocess (:341-350): L*log2(e) and -delta per query
//                        row into the workspace. Then dQ = scale * dS K over
//                        all visible key tiles, stored straight in the input
//                        dtype;
//   fa_bwd_dkdv_kernel : key-stationary; dK, dV over all visible query tiles
//                        (runs after the dq kernel, which feeds it).
// Both kernels recompute S and dP. The stored-dS path instead runs
//   fa_bwd_prep_kernel : the preprocess (delta, L*log2(e)) on its own;
//   fa_bwd_dkdv_kernel<..., DS = true> : as above, also storing dS;
//   fa_bwd_dq_ds_kernel : dQ = scale * dS K over the stored dS,
// which computes S and dP once but moves dS through HBM twice.
// There are no atomics and no fp32 dq buffer, so results are deterministic.
// Every dP accumulation starts from -delta (the MFMA's C input), so that
// dS = P (dP - delta) costs one multiply per score.
#include "fa_common.hpp"
#include <algorithm>

namespace lsfa {

constexpr float kLog2eB = 1.4426950408889634f;
// Cache-policy operand of the buffer builtins: the non-temporal (streaming) hint.
constexpr int kCacheNT = 2;

// ---------------------------------------------------------------------------
// dQ. Workgroup = 4 waves x 32 query rows, at most 256 registers
// per wave so two workgroups share a CU. K/V tiles of 64 keys go global ->
// LDS with buffer_load ... lds (double-buffered, zero past the sequence end).
// Per key tile and wave:
//   S^T  = K Q^T          A = K rows (LDS),  B = Q^T  (registers)
//   dP^T = V dO^T         A = V rows (LDS),  B = dO^T (registers)
//   dS^T = P^T (dP^T - delta)  -> rounded into B operands
//   dQ^T += K^T dS^T      A = K^T via transpose reads of the same LDS tile
// ---------------------------------------------------------------------------
template <typename T, int DP, bool CAUSAL, bool VARLEN = false>
__global__ __launch_bounds__(256, 2) void fa_bwd_dq_kernel(const BwdParams p) {
  using X8 = typename VecT<T>::x8;
  using X4 = typename VecT<T>::x4;
  constexpr int NW = 4, BM = NW * 32, BN = 64;
  constexpr int TILE = BN * DP;
  constexpr int LDI = TILE * 2 / 1024 / NW;
  constexpr int KSTEPS = DP / 16;
  constexpr int DT = DP / 32;
  constexpr int KB = BN / 32;
  static_assert(LDI >= 1, "tile too small for the workgroup");

  __shared__ __attribute__((aligned(1024))) T smem_raw[4 * TILE];  // K0 K1 V0 V1
  LDS_AS char* sm = (LDS_AS char*)smem_raw;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (SGPR)
  const int l32 = lane & 31, hh = lane >> 5;
  int b, h, qt;
  if (VARLEN && p.ranked_tokens >= 0 && p.cu_q[p.B] - p.cu_q[0] <= p.ranked_tokens) {
    // Sequences differ in length: (sequence, query tile) items longest first,
    // workgroup L taking rank L / H and head slot L % H (ranked_head).
    const int rank = blockIdx.x / p.H;
    h = ranked_head(blockIdx.x - rank * p.H, p.H);
    int tq = 0, nk = 0, off = 0;
    if (lane < p.B) {
      const int nq = min(max(p.cu_q[lane + 1] - p.cu_q[lane], 0), p.Nq);
      nk = min(max(p.cu_k[lane + 1] - p.cu_k[lane], 0), p.Nk);
      tq = (nq + BM - 1) / BM;
      off = nk - nq;
    }
    int d;
    b = ranked_item(p.B, rank, lane, tq, (nk + 63) >> 6, [&](int x) { return tiles_above<CAUSAL, BM>(x, tq, nk, off); },
                    d);
    if (b < 0) return;  // uniform, before any barrier
    qt = __builtin_amdgcn_readlane(tq, b) - 1 - d;
  } else {
    int bh;
    map_tile(p.num_tiles, gridDim.x, p.heads_per_group, bh, qt, CAUSAL);
    b = bh / p.H;
    h = bh - b * p.H;
  }
  int nq = p.Nq, nk = p.Nk;
  int64_t rq0 = 0, rk0 = 0;  // varlen: the sequence's first query / key row
  if (VARLEN) {  // lengths clamped to the longest the grid and the workspace were sized for
    rq0 = p.cu_q[b];
    nq = min(max(p.cu_q[b + 1] - (int)rq0, 0), p.Nq);
    rk0 = p.cu_k[b];
    nk = min(max(p.cu_k[b + 1] - (int)rk0, 0), p.Nk);
  }
  const int D = p.D;
  const int q0 = qt * BM;
  // Past this sequence's queries (varlen grids cover the longest one); its
  // workspace rows are never read. Uniform, before any barrier.
  if (VARLEN && q0 >= nq) return;
  const int off = nk - nq;

  const int hk = h / p.G;  // KV head of this query head
  const int64_t bq = VARLEN ? 0 : b, bk = VARLEN ? 0 : b;
  const T* Q = (const T*)p.q + bq * p.sqb + (int64_t)h * p.sqh + rq0 * p.sqn;
  const T* K = (const T*)p.k + bk * p.skb + (int64_t)hk * p.skh + rk0 * p.skn;
  const T* V = (const T*)p.v + bk * p.svb + (int64_t)hk * p.svh + rk0 * p.svn;
  const T* Og = (const T*)p.o + bq * p.sob + (int64_t)h * p.soh + rq0 * p.son;
  const T* dO = (const T*)p.dout + bq * p.sdob + (int64_t)h * p.sdoh + rq0 * p.sdon;
  T* dQ = (T*)p.dq + bq * p.sdqb + (int64_t)h * p.sdqh + rq0 * p.sdqn;

  const int qw_lo = q0 + wave * 32;
  const int qrow = qw_lo + l32;
  const bool qvalid = qrow < nq;

  // Lane byte offset of chunk lc of a row-major tile (rows of 2*DP bytes):
  // lane t fills LDS bytes [16t, 16t+16) of the chunk, i.e. stored segment
  // (byte % 2DP)/16 of a row, which holds logical segment stored ^
  // seg_swz(row). Logical columns at or past D get an offset past any
  // descriptor's end, so they read as zero.
  auto row_voff = [&](int lc, int64_t sn) -> int {
    const int byte = lc * 1024 + lane * 16;
    const int row = byte / (DP * 2);
    const int seg = ((byte % (DP * 2)) / 16) ^ seg_swz<DP>(row);
    return seg * 8 < D ? (int)(row * sn * 2) + seg * 16 : (int)0x80000000;
  };
  const int tr_row = 4 * hh + ((lane & 15) >> 2);
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  int troff[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    troff[dt][0] = swz_off<DP>(tr_row, 32 * dt + tr_col) * 2;
    troff[dt][1] = swz_off<DP>(tr_row + 8, 32 * dt + tr_col) * 2;
  }

  // Prologue (the backward's per-query-row pass): the tile's Q and dO rows
  // go to LDS (rows past nq and columns past D as zero), then
  //   - Q^T and dO^T B operands of this kernel come from LDS;
  //   - delta = rowsum(dO * O) and L*log2e are written to the workspace for
  //     the dK/dV kernel.
  constexpr int TB = BM * DP * 2;  // bytes of one 128-row tile
  static_assert(2 * TB <= 4 * TILE * 2, "Q/dO tiles must fit in the K/V buffers");
  {
    constexpr int CPW = 2 * TB / 1024 / NW;  // chunks per wave (waves 0..1: Q, 2..3: dO)
    const bool w_do = wave >= NW / 2;
    const int64_t sn = w_do ? p.sdon : p.sqn;
    const int rows = min(nq - q0, BM);
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc((w_do ? dO : Q) + (int64_t)q0 * sn, (int)(rows * sn * 2));
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int c = wave * CPW + i;
      const int vo = row_voff(c % (TB / 1024), sn);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LDS_AS void*)(sm + c * 1024), 16, vo, 0, 0, 0);
    }
  }
  u32x4 oraw[KSTEPS];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) {
    const int col = 16 * kk + 8 * hh;
    oraw[kk] = u32x4{0, 0, 0, 0};
    if (qvalid && col < D) oraw[kk] = ldg16(Og + (int64_t)qrow * p.son + col);
  }
  float lraw = -INFINITY;
  if (qvalid) lraw = p.lse[bq * p.slb + (int64_t)h * p.slh + (rq0 + qrow) * p.sln];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  X8 qreg[KSTEPS], doreg[KSTEPS];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) {
    const int o = swz_off<DP>(32 * wave + l32, 16 * kk + 8 * hh) * 2;
    qreg[kk] = *(const LDS_AS X8*)(sm + o);
    doreg[kk] = *(const LDS_AS X8*)(sm + TB + o);
  }
  __syncthreads();  // the K/V tiles below reuse the Q/dO buffers

  int kv_end = nk;
  if (CAUSAL) kv_end = min(nk, q0 + BM + off);
  const int ntiles = kv_end > 0 ? (kv_end + BN - 1) / BN : 0;

  // Direct tile loads of K and V (see row_voff). The buffer descriptor is
  // rebuilt per tile (scalar work) and clipped to the rows that exist, so
  // the per-lane byte offsets are loop-invariant and rows past nk read as zero.
  int kvo[LDI], vvo[LDI];
#pragma unroll
  for (int c = 0; c < LDI; ++c) {
    kvo[c] = row_voff(wave * LDI + c, p.skn);
    vvo[c] = row_voff(wave * LDI + c, p.svn);
  }
  auto tile_load = [&](const T* base, int64_t sn, const int* vo, int j, int buf) {
    const int rows = min(nk - j * BN, BN);
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(base + (int64_t)j * BN * sn, (int)(rows * sn * 2));
    LDS_AS char* dst = sm + buf * TILE * 2;
#pragma unroll
    for (int c = 0; c < LDI; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LDS_AS void*)(dst + (wave * LDI + c) * 1024), 16, vo[c], 0, 0, 0);
  };
  // The first K/V tiles load while delta is computed.
  if (ntiles > 0) {
    tile_load(K, p.skn, kvo, 0, 0);
    tile_load(V, p.svn, vvo, 0, 2);
  }

  float dpart = 0.f;
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) {
    const X8 ov = __builtin_bit_cast(X8, oraw[kk]);
#pragma unroll
    for (int s = 0; s < 8; ++s) dpart += (float)doreg[kk][s] * (float)ov[s];
  }
  const float delta = half_sum(dpart);
  const float l2 = lraw == -INFINITY ? INFINITY : lraw * kLog2eB;  // no visible key / padding: P == 0
  if (hh == 0) {
    float* w = p.ld + (int64_t)b * p.sldb + (int64_t)h * p.sldh + (qrow >> 6) * 128 + (qrow & 63);
    w[0] = l2;
    w[64] = -delta;
  }
  // dP^T - delta accumulates from -delta (this lane's query in every
  // register), so dS = P (dP - delta) is one multiply per score.
  f32x16 negd;
#pragma unroll
  for (int i = 0; i < 16; ++i) negd[i] = -delta;

  int koff[KSTEPS];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) koff[kk] = swz_off<DP>(l32, 16 * kk + 8 * hh) * 2;

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};
  const float sl2 = p.scale_log2;

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // One key tile j; the loop below runs it twice per iteration (j even,
  // then odd), so the buffer parity is known at compile time and every LDS
  // operand address is a lane offset plus an immediate.
  auto key_tile = [&](int j) {
    if (j + 1 < ntiles) {
      tile_load(K, p.skn, kvo, j + 1, (j + 1) & 1);
      tile_load(V, p.svn, vvo, j + 1, 2 + ((j + 1) & 1));
    }
    const int kbase = j * BN;
    const bool active = !CAUSAL || (kbase <= qw_lo + 31 + off);
    if (active) {
      const LDS_AS char* Ks = sm + (j & 1) * TILE * 2;
      const LDS_AS char* Vs = sm + (2 + (j & 1)) * TILE * 2;
      f32x16 s[KB], dp[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        s[kb] = f32x16{};
        dp[kb] = negd;
      }
#pragma unroll
      for (int kk = 0; kk < KSTEPS; ++kk) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const int o = kb * 32 * DP * 2 + koff[kk];
          s[kb] = mfma32(*(const LDS_AS X8*)(Ks + o), qreg[kk], s[kb]);
          dp[kb] = mfma32(*(const LDS_AS X8*)(Vs + o), doreg[kk], dp[kb]);
        }
      }
      // K / V operand reads run 4 MFMAs ahead of their MFMA (the compiler's
      // order reads one ahead and waits out an LDS latency per MFMA; eight
      // ahead no longer fits beside the -delta block).
      {
        constexpr int NM = 2 * KSTEPS * KB, RA = 4;
#pragma unroll
        for (int i = 0; i < RA; ++i) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (m + RA < NM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float pv = fast_exp2(fmaf(s[kb][i], sl2, -l2));
          s[kb][i] = pv * dp[kb][i];
        }
      if (CAUSAL && kbase + BN - 1 > qw_lo + off) {  // tile crosses the diagonal
        const int lim = qrow + off - kbase - 4 * hh;  // masked if 32kb + 8(i/4) + i%4 > lim
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[kb][i] = (32 * kb + 8 * (i >> 2) + (i & 3) > lim) ? 0.f : s[kb][i];
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
        for (int ks = 0; ks < 2 * KB; ++ks) {
          const LDS_AS char* base = Ks + ks * 16 * DP * 2;
          const X8 a = cat4<X8, X4>(lds_read_tr((const LDS_AS T*)(base + troff[dt][0])),
                                    lds_read_tr((const LDS_AS T*)(base + troff[dt][1])));
          acc[dt] = mfma32(a, pack8<T>(s[ks >> 1], 8 * (ks & 1)), acc[dt]);
        }
      }
      // K^T transpose reads run 4 MFMAs ahead.
      {
        constexpr int NM = DT * 2 * KB, RA = 4;
#pragma unroll
        for (int i = 0; i < RA; ++i) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (m + RA < NM) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  int j = 0;
  for (; j + 1 < ntiles; j += 2) {
    key_tile(j);
    key_tile(j + 1);
  }
  if (j < ntiles) key_tile(j);

  // dQ (times sm_scale) leaves through LDS, four whole rows per store
  // instruction (as dK/dV below); the loop's closing barrier has retired
  // every K/V read.
  {
    constexpr int BLK = 32 * DP * 2;  // bytes of one wave's 32 rows
    LDS_AS char* wb = sm + wave * BLK;
    const float sc = p.scale;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        X4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (T)(acc[dt][4 * g + e] * sc);
        *(LDS_AS X4*)(wb + swz_off<DP>(l32, 32 * dt + 8 * g + 4 * hh) * 2) = v;
      }
#pragma unroll
    for (int c = 0; c < BLK / 1024; ++c) {
      const int byte = c * 1024 + lane * 16;
      const int row = byte / (DP * 2), seg = (byte % (DP * 2)) / 16;
      const X8 v = *(const LDS_AS X8*)(wb + row * DP * 2 + ((seg ^ seg_swz<DP>(row)) << 4));
      const int q = qw_lo + row;
      if (q < nq && seg * 8 < D) *(X8*)(dQ + (int64_t)q * p.sdqn + seg * 8) = v;
    }
  }
}

// ---------------------------------------------------------------------------
// dK, dV. Workgroup = 4 waves, one per SIMD, over 128 keys of one KV head
// (with GQA the tiles of the head's G query heads follow one another through
// the ring, summing into the same dK/dV registers); wave w owns keys
// 32w..32w+31 and keeps their K and V rows in registers for the whole kernel
// (the B operands of S = Q K^T and dP = dO V^T). Q, dO and the rows'
// L*log2e and -delta blocks stream through three LDS stages of 64-row tiles by
// direct buffer loads. Each wave walks the 32-row halves of the tiles in
// order, software-pipelined so that its own MFMA and VALU work overlap (a
// wave's MFMAs run beside its own independent VALU instructions, not beside
// another wave's):
//   iteration h:  S, dP of half h+1 (16 MFMAs, A = Q / dO rows from LDS)
//                 beside P = exp2(S*scale*log2e - L*log2e), dS = P (dP - delta)
//                 of half h (VALU), then
//                 dV^T += dO^T P and dK^T += Q^T dS of half h (16 MFMAs, A =
//                 dO^T / Q^T through transpose reads of the same row tiles).
// A tile's stage is refilled after every wave has finished its second half
// (one barrier per tile); a tile is loaded three halves-iterations before its
// first use. Query rows beyond the sequence have L = +inf in the workspace
// (written by the dq kernel's prologue or the preprocess kernel), so their P
// is exactly 0; head-dim columns at or past D load as zero. dK is scaled by
// sm_scale at the end.
// With DS, the wave also stores dS (in the input dtype: the exact values its
// dK MFMAs take) for fa_bwd_dq_ds_kernel, as 2 KB blocks of 32 keys x 32
// queries in register order: a half's G0 words of all 64 lanes fill the
// block's first KB, its G1 words the second, lane l's 16 bytes at unit
// l ^ 8 (l / 32) (^ 4 in the second KB) so that the reader's transpose reads
// spread over all LDS banks. Each store instruction writes 1 KB of
// contiguous memory. Keys at or past nk are stored as zero, masked (causal)
// entries are zero already.
// ---------------------------------------------------------------------------
// s_waitcnt immediate: wait until at most n vector-memory operations of the
// wave are outstanding (expcnt and lgkmcnt left at their maxima).
constexpr int vmcnt_enc(int n) { return 0x0F70 | (n & 15) | (((n >> 4) & 3) << 14); }

template <typename T, int DP, bool CAUSAL, bool DS, bool GQA = false, bool VARLEN = false>
__global__ __launch_bounds__(256, 1) void fa_bwd_dkdv_kernel(const BwdParams p) {
  using X8 = typename VecT<T>::x8;
  using X4 = typename VecT<T>::x4;
  constexpr int NW = 4, BNK = 128, BMQ = 64, NST = 3;
  constexpr int KSTEPS = DP / 16, DT = DP / 32;
  constexpr int R_B = BMQ * DP * 2;     // bytes of a row-major Q (or dO) tile
  constexpr int RS_B = 2 * R_B + 1024;  // one stage: Q | dO | 64 L*log2e | 64 -delta, 1 KB aligned
  constexpr int KV_B = 4 * R_B;        // the prologue's K / V rows, from stage 2 on
  constexpr int LDS_B = (NST - 1) * RS_B + KV_B;
  constexpr int CR = 2 * R_B / 1024 / NW;  // 1 KB chunks per wave per tile (Q|dO)
  static_assert(CR >= 1, "tile too small for the workgroup");
  static_assert(LDS_B <= 160 * 1024, "LDS budget");

  __shared__ __attribute__((aligned(1024))) char sm_raw[LDS_B];
  LDS_AS char* sm = (LDS_AS char*)sm_raw;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int kb = wave;
  const bool w_hi = wave >= NW / 2;  // waves 2, 3 load dO; 0, 1 load Q
  // One workgroup per (batch, KV head, key tile). With GQA (G query heads
  // per KV head) the query tiles of the group's G heads stream through the
  // ring one head after another, into the same dK/dV sums.
  static_assert(!((GQA || VARLEN) && DS), "the stored-dS path has no GQA or varlen");
  const int G = GQA ? p.G : 1, Hkv = p.H / G;
  int bh, kt, b, hk;
  if (VARLEN && p.ranked_tokens >= 0 && p.cu_k[p.B] - p.cu_k[0] <= p.ranked_tokens) {
    // Longest first, as in fa_bwd_dq_kernel: key tile kt of a sequence takes
    // the query tiles from max(0, 128 kt - off) / 64 on, so more than x of
    // them iff 128 kt < 64 (tiles - x) + off.
    const int rank = blockIdx.x / Hkv;
    hk = ranked_head(blockIdx.x - rank * Hkv, Hkv);
    int tk = 0, tiles = 0, off = 0;
    if (lane < p.B) {
      const int nq = min(max(p.cu_q[lane + 1] - p.cu_q[lane], 0), p.Nq);
      const int nk = min(max(p.cu_k[lane + 1] - p.cu_k[lane], 0), p.Nk);
      tk = (nk + BNK - 1) / BNK;
      tiles = (nq + BMQ - 1) / BMQ;
      off = nk - nq;
    }
    b = ranked_item(p.B, rank, lane, tk, tiles, [&](int x) {
      if (x < 0) return tk;
      if (x >= tiles) return 0;
      if (!CAUSAL) return tk;
      const int y = BMQ * (tiles - x) + off;
      return y <= 0 ? 0 : min(tk, (y + BNK - 1) / BNK);
    }, kt);
    if (b < 0) return;  // uniform, before any barrier
    bh = b * Hkv + hk;
  } else {
    map_tile(p.num_tiles, gridDim.x, p.heads_per_group, bh, kt, false);  // low key tiles see the most queries
    bh += p.bh0;
    b = bh / Hkv;
    hk = bh - b * Hkv;
  }
  const int h0 = hk * G;
  int nq = p.Nq, nk = p.Nk;
  int64_t rq0 = 0, rk0 = 0;  // varlen: the sequence's first query / key row
  if (VARLEN) {  // lengths clamped to the longest the grid and the workspace were sized for
    rq0 = p.cu_q[b];
    nq = min(max(p.cu_q[b + 1] - (int)rq0, 0), p.Nq);
    rk0 = p.cu_k[b];
    nk = min(max(p.cu_k[b + 1] - (int)rk0, 0), p.Nk);
  }
  const int D = p.D;
  const int k0 = kt * BNK;
  if (VARLEN && k0 >= nk) return;  // past this sequence's keys; uniform, before any barrier
  const int off = nk - nq;

  const int64_t bb = VARLEN ? 0 : b;
  const T* K = (const T*)p.k + bb * p.skb + (int64_t)hk * p.skh + rk0 * p.skn;
  const T* V = (const T*)p.v + bb * p.svb + (int64_t)hk * p.svh + rk0 * p.svn;
  const T* Q = (const T*)p.q + bb * p.sqb + (int64_t)h0 * p.sqh + rq0 * p.sqn;
  const T* dO = (const T*)p.dout + bb * p.sdob + (int64_t)h0 * p.sdoh + rq0 * p.sdon;
  const float* LD = p.ld + (int64_t)b * p.sldb + (int64_t)h0 * p.sldh;

  const int n_qt = (nq + BMQ - 1) / BMQ;  // every tile starts below nq
  int t_begin = 0;
  if (CAUSAL) t_begin = max(0, k0 - off) / BMQ;  // first tile holding a query that sees key k0
  const int n_t = max(0, n_qt - t_begin);  // visible query tiles per query head
  const int n_all = G * n_t;               // ... over the group's heads
  // Linear tile index -> (query head of the group, tile within the head).
  auto head_of = [&](int tt) { return GQA ? tt / n_t : 0; };
  const int kcol = k0 + 32 * kb + l32;  // this lane's key

  // dS blocks: this wave's 32 keys are block row kblk of the head, blocks
  // [kblk][query / 32] of 1024 elements; a wave with no key below nk stores
  // nothing (empty descriptor).
  __amdgpu_buffer_rsrc_t dsr;
  int dso0 = 0, dso1 = 0;
  if constexpr (DS) {
    const int nqb = (int)(p.ds_ldq >> 5);
    const T* base = (const T*)p.ds + (int64_t)(bh - p.bh0) * p.ds_sbh + (int64_t)((k0 >> 5) + kb) * nqb * 1024;
    dsr = tile_rsrc(base, k0 + 32 * kb < nk ? nqb * 2048 : 0);
    dso0 = 16 * (lane ^ (8 * hh));
    dso1 = 1024 + 16 * (lane ^ (8 * hh) ^ 4);
  }
  // The G0 (g = 0) or G1 (g = 1) words of the half whose first query is qfirst.
  auto store_ds = [&](int qfirst, const u32x4& w, int g) {
    if constexpr (DS) {
      const u32x4 v = kcol < nk ? w : u32x4{0u, 0u, 0u, 0u};
      // nt: dS is read once, by another kernel, long after it leaves L2
      __builtin_amdgcn_raw_buffer_store_b128(v, dsr, (qfirst >> 5) * 2048 + (g ? dso1 : dso0), 0, kCacheNT);
    }
  };

  // Row-major tile loads (see fa_bwd_dq_kernel's row_voff).
  auto row_voff = [&](int lc, int64_t sn) -> int {
    const int byte = lc * 1024 + lane * 16;
    const int row = byte / (DP * 2);
    const int seg = ((byte % (DP * 2)) / 16) ^ seg_swz<DP>(row);
    return seg * 8 < D ? (int)(row * sn * 2) + seg * 16 : (int)0x80000000;
  };
  int rvo[CR];
#pragma unroll
  for (int i = 0; i < CR; ++i) rvo[i] = row_voff((wave % (NW / 2)) * CR + i, w_hi ? p.sdon : p.sqn);
  auto load_tile = [&](int tt, int stage, const int* vo) {
    const int g = head_of(tt);
    const int q0 = (t_begin + tt - g * n_t) * BMQ;
    const int rows = min(nq - q0, BMQ);
    const int64_t sn = w_hi ? p.sdon : p.sqn;
    const T* src = w_hi ? dO + (int64_t)g * p.sdoh : Q + (int64_t)g * p.sqh;
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(src + (int64_t)q0 * sn, (int)(rows * sn * 2));
    LDS_AS char* base = sm + stage * RS_B + (w_hi ? R_B : 0);
#pragma unroll
    for (int i = 0; i < CR; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LDS_AS void*)(base + ((wave % (NW / 2)) * CR + i) * 1024), 16,
                                               vo[i], 0, 0, 0);
    if (wave == 0 && lane < BMQ * 8 / 16) {
      const __amdgpu_buffer_rsrc_t lrs = tile_rsrc(LD + (int64_t)g * p.sldh + 2 * (int64_t)q0, BMQ * 8);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(lrs, (LDS_AS void*)(sm + stage * RS_B + 2 * R_B), 16, lane * 16, 0, 0,
                                               0);
    }
  };
  // Prologue only: the rows of tile tt (an empty descriptor past the last
  // tile, whose loads then write zeros to a stage read by no one), and the
  // tile's L*log2e / -delta pairs (wave 0).
  auto load_rows_pro = [&](int tt, int stage) {
    const bool live = tt < n_all;
    const int g = live ? head_of(tt) : 0;
    const int q0 = live ? (t_begin + tt - g * n_t) * BMQ : 0;
    const int rows = live ? min(nq - q0, BMQ) : 0;
    const int64_t sn = w_hi ? p.sdon : p.sqn;
    const T* src = w_hi ? dO + (int64_t)g * p.sdoh : Q + (int64_t)g * p.sqh;
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(src + (int64_t)q0 * sn, (int)(rows * sn * 2));
    LDS_AS char* base = sm + stage * RS_B + (w_hi ? R_B : 0);
#pragma unroll
    for (int i = 0; i < CR; ++i) dma16(rs, (LDS_AS void*)(base + ((wave % (NW / 2)) * CR + i) * 1024), rvo[i]);
  };
  auto load_ld_pro = [&](int tt, int stage) {
    if (wave == 0 && lane < BMQ * 8 / 16) {
      const int g = head_of(tt);
      const int q0 = (t_begin + tt - g * n_t) * BMQ;
      const __amdgpu_buffer_rsrc_t lrs = tile_rsrc(LD + (int64_t)g * p.sldh + 2 * (int64_t)q0, BMQ * 8);
      dma16(lrs, (LDS_AS void*)(sm + stage * RS_B + 2 * R_B), lane * 16);
    }
  };
  // Prologue. The first tile goes into stage 0, the workgroup's 128 K and
  // 128 V rows into the space from stage 2 on, then the second tile into
  // stage 1, all by direct 1 KB loads of whole rows (each 128-byte line is
  // requested once; per-lane register loads of 16 bytes from 32 rows
  // touched every line four times and took most of the prologue). Wave w
  // loads K (w < 2) or V (w >= 2) rows 64 (w % 2) .. +63, swizzled like a Q
  // tile; rows at or past nk and columns at or past D read as zero. The
  // first scores wait for the first tile and K / V only; the second tile
  // lands under them.
  if (n_all > 0) load_tile(0, 0, rvo);
  if (1 < n_all) load_ld_pro(1, 1);
  {
    const int r0 = 64 * (wave % 2);
    const int rows = max(0, min(nk - k0 - r0, BMQ));
    const int64_t sn = w_hi ? p.svn : p.skn;
    const T* src = (w_hi ? V : K) + (int64_t)(k0 + r0) * sn;
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(src, (int)(rows * sn * 2));
    LDS_AS char* base = sm + (NST - 1) * RS_B + (w_hi ? 2 : 0) * R_B + (wave % 2) * R_B;
#pragma unroll
    for (int i = 0; i < R_B / 1024; ++i) dma16(rs, (LDS_AS void*)(base + i * 1024), row_voff(i, sn));
  }
  // Issued on every path (no branch from here to the wait, so that the
  // count below is exact): the wave's CR row loads of the second tile.
  load_rows_pro(1, 1);
  // The first tile and K / V have landed once at most those CR loads are
  // outstanding (a wave's loads retire in order); a plain barrier, since
  // __syncthreads() would also wait for the second tile.
  __builtin_amdgcn_s_waitcnt(vmcnt_enc(CR));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // K and V rows of this lane's key as B operands: columns 16kk + 8hh .. +7.
  X8 kreg[KSTEPS], vreg[KSTEPS];
  {
    const LDS_AS char* kr = sm + (NST - 1) * RS_B + (kb / 2) * R_B + 32 * (kb % 2) * DP * 2;
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) {
      const int o = swz_off<DP>(l32, 16 * kk + 8 * hh) * 2;
      // straight into accumulation registers, where the loop's MFMAs read
      // them as B operands (a VGPR result would be parked there and copied
      // back before every use)
      const uint32_t ka = (uint32_t)(uintptr_t)(kr + o), va = (uint32_t)(uintptr_t)(kr + 2 * R_B + o);
      asm volatile("ds_read_b128 %0, %1" : "=a"(kreg[kk]) : "v"(ka) : "memory");
      asm volatile("ds_read_b128 %0, %1" : "=a"(vreg[kk]) : "v"(va) : "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  int roff[KSTEPS];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) roff[kk] = swz_off<DP>(l32, 16 * kk + 8 * hh) * 2;
  const int tr_row = 4 * hh + ((lane & 15) >> 2);
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  int troff[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    troff[dt][0] = swz_off<DP>(tr_row, 32 * dt + tr_col) * 2;
    troff[dt][1] = swz_off<DP>(tr_row + 8, 32 * dt + tr_col) * 2;
  }

  // Lane offsets for the third stage, whose addresses pass the 16-bit
  // immediate: the same offsets plus 64 KB (kept opaque so that they stay in
  // registers instead of being re-added per read).
  int roffH[KSTEPS], troffH[DT][2];
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) {
    roffH[kk] = roff[kk] + 65536;
    asm volatile("" : "+v"(roffH[kk]));
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j2 = 0; j2 < 2; ++j2) {
      troffH[dt][j2] = troff[dt][j2] + 65536;
      asm volatile("" : "+v"(troffH[dt][j2]));
    }
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dk[dt] = f32x16{};
    dv[dt] = f32x16{};
  }
  const float sl2 = p.scale_log2;

  // Half (t, q): rows 32 q .. 32 q + 31 of tile t_begin + t, which sits in
  // LDS stage t % NST. The loop below is unrolled over the stages so that
  // every LDS address is a lane offset plus an immediate. Within a wave the
  // work of two halves is interleaved in fenced chunks (the scheduler keeps
  // each chunk's instructions together and in order), so that the wave's
  // MFMAs issue beside its own independent VALU and LDS instructions:
  //   phase X: 16 chunks of (S or dP MFMA of the next half, operand read
  //            PF chunks ahead; P and dS of one score of this half; at
  //            chunks 8..15 one conversion of P0 / G0),
  //   phase Y: 16 chunks of (two transpose reads PF chunks ahead; one dV or
  //            dK MFMA of this half, the 16-query step ks = 0 first; at
  //            chunks 0..7 one conversion of P1 / G1).
  // Register i of a score tile holds query 32 q + 8 (i / 4) + 4 hh + i % 4.
  constexpr int PF = 3;
  typedef __attribute__((ext_vector_type(2))) T T2;
  auto cvt2 = [](float a, float b) -> uint32_t { return __builtin_bit_cast(uint32_t, T2{(T)a, (T)b}); };
  u32x4 p0w, g0w, p1w, g1w;  // P0, G0, P1, G1 as packed words
  X8 P0, P1, G0, G1;

  // Phase X has NCX = 2 KSTEPS MFMA chunks and EPC = 16 / NCX scores per
  // chunk; phase Y has NCY = 4 DT chunks, the first 2 DT of them (step ks = 0)
  // carrying the 8 conversions of P1 / G1 that the rest need.
  constexpr int NCX = 2 * KSTEPS, EPC = 16 / NCX, NCY = 4 * DT, CPY = 8 / (2 * DT);
  // -delta of the 16 queries a lane's score registers hold in half q of the
  // tile in stage st (register i: query 32 q + 8 (i / 4) + 4 hh + i % 4),
  // the start of its dP - delta accumulation: four 16-byte reads.
  auto neg_delta = [&](const LDS_AS char* st, int q) -> f32x16 {
    const LDS_AS f32x4* d = (const LDS_AS f32x4*)(st + 2 * R_B + 256 + (32 * q + 4 * hh) * 4);
    f32x16 r;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 v = d[2 * g];
#pragma unroll
      for (int e = 0; e < 4; ++e) r[4 * g + e] = v[e];
    }
    return r;
  };
  auto phase_x = [&](const LDS_AS char* nst, bool nhi, int nq, f32x16& sn, f32x16& dn, const LDS_AS char* stg, int t, int q,
                     f32x16& s, f32x16& dp) {
    const LDS_AS char* an = nst + 32 * nq * DP * 2;
    // operand c: kk = c / 2; even c reads a Q row (S), odd c a dO row (dP)
    auto opread = [&](int c) -> X8 {
      return *(const LDS_AS X8*)((nhi ? an - 65536 : an) + (c & 1) * R_B + (nhi ? roffH[c >> 1] : roff[c >> 1]));
    };
    // L*log2e of queries 8g + 4hh .. +3 (group g = scores 4g .. 4g+3): one
    // 16-byte read, issued four chunks before the group's first score is
    // scaled.
    const LDS_AS f32x4* ldp = (const LDS_AS f32x4*)(stg + 2 * R_B + (32 * q + 4 * hh) * 4);
    f32x4 lda[4];
    auto lead = [](int g) { return 4 * g / EPC - 4; };
    auto l2_of = [&](int i) { return lda[i >> 2][i & 3]; };
    // Each score goes through three steps two chunks apart (x = s*scale*log2e
    // - L*log2e; p = exp2(x); dS = p (dP - delta)), so the VALU instructions
    // of one chunk never wait on each other.
    auto step_a = [&](int cc) {
      if (cc < NCX)
#pragma unroll
        for (int u = 0; u < EPC; ++u) { const int i = cc * EPC + u; s[i] = fmaf(s[i], sl2, -l2_of(i)); }
    };
    auto step_b = [&](int cc) {
      if (cc < NCX)
#pragma unroll
        for (int u = 0; u < EPC; ++u) { const int i = cc * EPC + u; s[i] = fast_exp2(s[i]); }
    };
    auto step_c = [&](int cc) {
#pragma unroll
      for (int u = 0; u < EPC; ++u) { const int i = cc * EPC + u; dp[i] = s[i] * dp[i]; }
    };
    X8 op[PF + 1];
#pragma unroll
    for (int c = 0; c < PF && c < NCX; ++c) op[c] = opread(c);
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (lead(g) < 0) lda[g] = ldp[2 * g];
    sn = f32x16{};
    dn = neg_delta(nst, nq);
    step_a(0);
    step_a(1);
    step_b(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NCX; ++c) {
      if (c + PF < NCX) op[(c + PF) % (PF + 1)] = opread(c + PF);
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (lead(g) == c) lda[g] = ldp[2 * g];
      if (c & 1)
        dn = mfma32(op[c % (PF + 1)], vreg[c >> 1], dn);
      else
        sn = mfma32(op[c % (PF + 1)], kreg[c >> 1], sn);
      step_a(c + 2);
      step_b(c + 1);
      step_c(c);
      if (c >= NCX / 2) {  // scores 0..7 are final: P0 / G0 words
#pragma unroll
        for (int u = 0; u < EPC; ++u) {
          const int k = (c - NCX / 2) * EPC + u, w = k >> 1;
          if ((k & 1) == 0) p0w[w] = cvt2(s[2 * w], s[2 * w + 1]);
          else g0w[w] = cvt2(dp[2 * w], dp[2 * w + 1]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const int q0 = (t_begin + t) * BMQ + 32 * q;
    if (CAUSAL && k0 + 32 * kb + 31 > q0 + off) {  // block crosses the diagonal
      // (the empty volatile asm keeps this a branch: the selects below would
      // otherwise be hoisted out of it and run on every half)
      asm volatile("" ::: "memory");
      const int lim = kcol - (q0 + 4 * hh + off);  // masked if 8*(i/4) + i%4 < lim
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bool m = 8 * (i >> 2) + (i & 3) < lim;
        s[i] = m ? 0.f : s[i];
        dp[i] = m ? 0.f : dp[i];
      }
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        p0w[w] = cvt2(s[2 * w], s[2 * w + 1]);
        g0w[w] = cvt2(dp[2 * w], dp[2 * w + 1]);
      }
    }
    P0 = __builtin_bit_cast(X8, p0w);
    G0 = __builtin_bit_cast(X8, g0w);
    store_ds(q0, g0w, 0);
  };
  auto phase_y = [&](const LDS_AS char* stg, bool chi, int t, int q, const f32x16& s, const f32x16& dp) {
    const LDS_AS char* st = stg + 32 * q * DP * 2;
    // MFMA c: ks = c / (2 DT), dt = (c / 2) % DT; even c is dV (dO^T), odd c dK (Q^T)
    auto opread = [&](int c) -> X8 {
      const LDS_AS char* qb = st + 16 * (c / (2 * DT)) * DP * 2 + ((c & 1) ? 0 : R_B);
      const int dt = (c >> 1) % DT;
      const LDS_AS char* qh = chi ? qb - 65536 : qb;
      return cat4<X8, X4>(lds_read_tr((const LDS_AS T*)(qh + (chi ? troffH[dt][0] : troff[dt][0]))),
                          lds_read_tr((const LDS_AS T*)(qh + (chi ? troffH[dt][1] : troff[dt][1]))));
    };
    X8 op[PF + 1];
#pragma unroll
    for (int c = 0; c < PF && c < NCY; ++c) op[c] = opread(c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NCY; ++c) {
      if (c + PF < NCY) op[(c + PF) % (PF + 1)] = opread(c + PF);
      if (c < 2 * DT) {  // scores 8..15: P1 / G1 words
#pragma unroll
        for (int u = 0; u < CPY; ++u) {
          const int k = c * CPY + u, w = k >> 1;
          if ((k & 1) == 0) p1w[w] = cvt2(s[8 + 2 * w], s[9 + 2 * w]);
          else g1w[w] = cvt2(dp[8 + 2 * w], dp[9 + 2 * w]);
        }
        if (c == 2 * DT - 1) {
          P1 = __builtin_bit_cast(X8, p1w);
          G1 = __builtin_bit_cast(X8, g1w);
          store_ds((t_begin + t) * BMQ + 32 * q, g1w, 1);
        }
      }
      const int dt = (c >> 1) % DT, ks = c / (2 * DT);
      if (c & 1)
        dk[dt] = mfma32(op[c % (PF + 1)], ks == 0 ? G0 : G1, dk[dt]);
      else
        dv[dt] = mfma32(op[c % (PF + 1)], ks == 0 ? P0 : P1, dv[dt]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // S and dP of the first half (not interleaved).
  auto scores = [&](const LDS_AS char* stg, int q, f32x16& s, f32x16& dp) {
    const LDS_AS char* st = stg + 32 * q * DP * 2;
    s = f32x16{};
    dp = neg_delta(stg, q);
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) {
      s = mfma32(*(const LDS_AS X8*)(st + roff[kk]), kreg[kk], s);
      dp = mfma32(*(const LDS_AS X8*)(st + R_B + roff[kk]), vreg[kk], dp);
    }
  };

  f32x16 sa, da, sb, db;  // S / dP of the current and the next half
  if (n_all > 0) scores(sm, 0, sa, da);
  // The second tile has landed and every wave holds its K / V rows; then
  // stage 2 takes its tile (which lands by the first iteration's closing
  // wait, one tile before its use).
  __syncthreads();
  if (NST - 1 < n_all) load_tile(NST - 1, NST - 1, rvo);
  // Per tile: the second half's S/dP beside the first half's softmax, the
  // first half's dV/dK; the next tile's first-half S/dP beside the second
  // half's softmax (past the last tile they read a stale stage and are
  // discarded), the second half's dV/dK; then the tile-end barrier: every
  // wave is done with this stage, which takes the tile NST ahead, and the
  // tile loaded at the previous barrier has landed.
  for (int t0 = 0; t0 < n_all; t0 += NST) {
#pragma unroll
    for (int si = 0; si < NST; ++si) {
      const int tt = t0 + si;
      if (tt >= n_all) break;
      const int t = tt - head_of(tt) * n_t;  // tile within its head (masking, dS blocks)
      const LDS_AS char* stg = sm + si * RS_B;
      const LDS_AS char* nstg = sm + ((si + 1) % NST) * RS_B;
      const bool chi = si == 2, nhi = (si + 1) % NST == 2;
      phase_x(stg, chi, 1, sb, db, stg, t, 0, sa, da);
      phase_y(stg, chi, t, 0, sa, da);
      phase_x(nstg, nhi, 0, sa, da, stg, t, 1, sb, db);
      phase_y(stg, chi, t, 1, sb, db);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tt + NST < n_all) load_tile(tt + NST, si, rvo);
    }
  }

  // dK (times sm_scale) and dV leave through LDS: a lane's accumulators hold
  // 4-column pieces of one key's row, so direct stores would scatter 8-byte
  // pieces over 32 rows per instruction. Each wave writes its two 32-row
  // blocks (swizzled 16-byte segments) into its own LDS region, reads them
  // back row-major and stores 16 bytes per lane, four whole rows per
  // instruction. The loop's closing barrier has retired every ring read.
  {
    constexpr int BLK = 32 * DP * 2;  // bytes of one 32-row block
    LDS_AS char* wb = sm + wave * 2 * BLK;
    const float sc = p.scale;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        X4 ck, cv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ck[e] = (T)(dk[dt][4 * g + e] * sc);
          cv[e] = (T)dv[dt][4 * g + e];
        }
        const int o = swz_off<DP>(l32, 32 * dt + 8 * g + 4 * hh) * 2;
        *(LDS_AS X4*)(wb + o) = ck;
        *(LDS_AS X4*)(wb + BLK + o) = cv;
      }
    T* rk = (T*)p.dk + bb * p.sdkb + (int64_t)hk * p.sdkh + rk0 * p.sdkn;
    T* rv = (T*)p.dv + bb * p.sdvb + (int64_t)hk * p.sdvh + rk0 * p.sdvn;
#pragma unroll
    for (int c = 0; c < BLK / 1024; ++c) {
      const int byte = c * 1024 + lane * 16;
      const int row = byte / (DP * 2), seg = (byte % (DP * 2)) / 16;
      const int o = row * DP * 2 + ((seg ^ seg_swz<DP>(row)) << 4);
      const X8 vk = *(const LDS_AS X8*)(wb + o);
      const X8 vv = *(const LDS_AS X8*)(wb + BLK + o);
      const int key = k0 + 32 * kb + row;
      if (key < nk && seg * 8 < D) {
        *(X8*)(rk + (int64_t)key * p.sdkn + seg * 8) = vk;
        *(X8*)(rv + (int64_t)key * p.sdvn + seg * 8) = vv;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Preprocess of the stored-dS path (kernels/flash_attention_backward.py:
// 341-350): per query row delta = rowsum(dO * O) (products of the input-dtype
// values in fp32) and L * log2(e) into the ld workspace (L * log2(e) and
// -delta); rows Nq .. nq_pad-1 and rows whose L is -inf get (+inf, 0), so
// that their P is exactly 0.
// Block = 64 rows x 4 lanes; lane part of a row sums the 16-byte chunks
// part, part + 4, ... of both rows.
// ---------------------------------------------------------------------------
template <typename T, int DP>
__global__ __launch_bounds__(256) void fa_bwd_prep_kernel(const BwdParams p) {
  using X8 = typename VecT<T>::x8;
  constexpr int LPR = 4, RPB = 256 / LPR;
  constexpr int CH = (DP / 8 + LPR - 1) / LPR;
  const int tiles = p.nq_pad / RPB;
  const int bh = blockIdx.x / tiles, rt = blockIdx.x - bh * tiles;
  const int b = bh / p.H, h = bh - b * p.H;
  const int row = rt * RPB + (int)threadIdx.x / LPR, part = threadIdx.x % LPR;
  float acc = 0.f, l2 = INFINITY;
  if (row < p.Nq) {
    const T* orow = (const T*)p.o + (int64_t)b * p.sob + (int64_t)h * p.soh + (int64_t)row * p.son;
    const T* drow = (const T*)p.dout + (int64_t)b * p.sdob + (int64_t)h * p.sdoh + (int64_t)row * p.sdon;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int col = 8 * (c * LPR + part);
      if (col < p.D) {
        const X8 ov = __builtin_bit_cast(X8, ldg16(orow + col));
        const X8 dv = __builtin_bit_cast(X8, ldg16(drow + col));
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += (float)dv[e] * (float)ov[e];
      }
    }
    const float lse = p.lse[(int64_t)b * p.slb + (int64_t)h * p.slh + (int64_t)row * p.sln];
    if (lse != -INFINITY) l2 = lse * kLog2eB;
  }
  acc += __shfl_xor(acc, 1);
  acc += __shfl_xor(acc, 2);
  if (part == 0) {
    float* w = p.ld + (int64_t)b * p.sldb + (int64_t)h * p.sldh + (row >> 6) * 128 + (row & 63);
    w[0] = l2;
    w[64] = -acc;
  }
}

// ---------------------------------------------------------------------------
// dQ of the stored-dS path: dQ = scale * dS K, a GEMM over the dS blocks that
// fa_bwd_dkdv_kernel<..., DS> stored, so S and dP are not computed a second
// time. Workgroup = 8 waves x 32 query rows (256 queries of one (batch,
// head)); key tiles of 64 go global -> LDS by direct buffer loads through NST
// stages: the tile's 16 dS blocks (2 block rows x 8 query blocks, each block
// row 16 KB of contiguous memory) and the K tile [64][DP]. Per tile and wave
// (wave w owns query block w):
//   dQ^T += K^T dS^T   A = K^T (transpose reads of K rows), B = dS^T
// with the 16-key MFMA steps in natural key order: lane l of the B operand
// needs keys 8 (l / 32) + 0..7 of query l % 32, and each 8-byte piece of a
// block holds 4 consecutive queries of one key, so a transpose read of 4
// pieces (4 keys) per 16-lane group delivers them. Keys at or past nk are
// zero (stored so, and K rows past nk load as zero). Causal: a wave skips
// the tiles wholly above its diagonal, and zeroes the dS entries with
// key > query + (Nk - Nq) in the tiles it crosses (there the dK/dV kernel
// stored zeros or, in blocks left of its first query tile, nothing).
// ---------------------------------------------------------------------------
template <typename T, int DP, bool CAUSAL>
__global__ __launch_bounds__(512, 1) void fa_bwd_dq_ds_kernel(const BwdParams p) {
  using X8 = typename VecT<T>::x8;
  using X4 = typename VecT<T>::x4;
  constexpr int NW = 8, BM = NW * 32, BN = 64, NST = 3;
  constexpr int DS_B = BN * BM * 2;           // dS bytes of a tile (16 blocks)
  constexpr int K_B = BN * DP * 2;            // K tile bytes
  constexpr int STG_B = DS_B + K_B;           // one stage
  constexpr int NCH = STG_B / 1024;           // 1 KB load chunks per stage
  constexpr int CPW = (NCH + NW - 1) / NW;    // chunk slots per wave
  constexpr int DT = DP / 32;
  static_assert(K_B % 1024 == 0, "K tile must be whole 1 KB chunks");
  static_assert(NST * STG_B <= 160 * 1024, "LDS budget");

  __shared__ __attribute__((aligned(1024))) char sm_raw[NST * STG_B];
  LDS_AS char* sm = (LDS_AS char*)sm_raw;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5;
  int bh, qt;
  map_tile(p.num_tiles, gridDim.x, p.heads_per_group, bh, qt, CAUSAL);
  bh += p.bh0;
  const int b = bh / p.H, h = bh - b * p.H;
  const int nq = p.Nq, nk = p.Nk, D = p.D;
  const int q0 = qt * BM;
  const int off = nk - nq;
  const int nqb = (int)(p.ds_ldq >> 5);  // query blocks per block row
  const int nkb = (nk + 31) >> 5;        // block rows

  const T* K = (const T*)p.k + (int64_t)b * p.skb + (int64_t)h * p.skh;
  const T* dS = (const T*)p.ds + (int64_t)(bh - p.bh0) * p.ds_sbh + (int64_t)(q0 >> 5) * 1024;
  T* dQ = (T*)p.dq + (int64_t)b * p.sdqb + (int64_t)h * p.sdqh;

  const int qw_lo = q0 + wave * 32;
  const int qrow = qw_lo + (lane & 31);

  int kv_end = nk;
  if (CAUSAL) kv_end = min(nk, q0 + BM + off);
  const int ntiles = kv_end > 0 ? (kv_end + BN - 1) / BN : 0;

  // Chunk slot i of this wave is stage chunk c = wave + NW i: chunks
  // 0 .. DS_B/1024 - 1 copy the two 16 KB block rows as they are (chunk c
  // of the stage = KB c % 16 of block row c / 16), the rest fill the K tile
  // (lane t writes the chunk's bytes [16 t, 16 t + 16), i.e. stored segment
  // (byte % row) / 16 of a row, which holds logical segment stored ^
  // seg_swz(row)).
  int cvo[CPW];
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const int c = wave + NW * i;
    if (c < DS_B / 1024) {
      cvo[i] = (c >> 4) * nqb * 2048 + (c & 15) * 1024 + lane * 16;
    } else {
      const int byte = (c - DS_B / 1024) * 1024 + lane * 16;
      const int row = byte / (DP * 2);
      const int seg = ((byte % (DP * 2)) / 16) ^ seg_swz<DP>(row);
      cvo[i] = seg * 8 < D ? (int)(row * p.skn * 2) + seg * 16 : (int)0x80000000;
    }
  }
  // (the offsets come in as a pointer parameter: indexing the captured array
  // itself in the builtin's argument makes clang's host pass drop the
  // kernel's launch stub)
  auto load_tile = [&](int j, int stage, const int* vo) {
    const int rows = min(nk - j * BN, BN);
    const int brows = min(nkb - 2 * j, 2);  // block rows of this tile below nk
    const __amdgpu_buffer_rsrc_t rd =
        tile_rsrc(dS + (int64_t)2 * j * nqb * 1024, (brows - 1) * nqb * 2048 + DS_B / 2);
    const __amdgpu_buffer_rsrc_t rk = tile_rsrc(K + (int64_t)j * BN * p.skn, (int)(rows * p.skn * 2));
    LDS_AS char* dst = sm + stage * STG_B;
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int c = wave + NW * i;
      if (c < DS_B / 1024)  // dS streams through once: nt keeps it from displacing K in L2
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rd, (LDS_AS void*)(dst + c * 1024), 16, vo[i], 0, 0, kCacheNT);
      else if (c < NCH)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (LDS_AS void*)(dst + c * 1024), 16, vo[i], 0, 0, 0);
    }
  };

  // Transpose-read offsets. Inside 16-lane group G (g = G % 2 picks the
  // block's KB, i.e. queries 16 g .. 16 g + 15; hh = G / 2 the MFMA's key
  // half), lane 4 j + r addresses the piece of key 8 hh + j (+ 4 for the
  // second read) holding queries 16 g + 8 (r / 2) + 4 (r % 2) .. + 3: unit
  // key + 32 (r % 2), swizzled as stored, byte 8 (r / 2) of it.
  const int G = lane >> 4, jj = (lane & 15) >> 2, rr = lane & 3, gq = G & 1;
  auto unit = [&](int key) { return (key + 32 * (rr & 1)) ^ (8 * (rr & 1)) ^ (4 * gq); };
  const int dsb0 = wave * 2048 + gq * 1024 + 16 * unit(8 * hh + jj) + 8 * (rr >> 1);
  const int dsb1 = wave * 2048 + gq * 1024 + 16 * unit(8 * hh + 4 + jj) + 8 * (rr >> 1);
  // K^T in the same key order: rows 8 hh + j and 8 hh + 4 + j.
  const int tr_row = 8 * hh + ((lane & 15) >> 2);
  const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  int troff[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    troff[dt][0] = swz_off<DP>(tr_row, 32 * dt + tr_col) * 2;
    troff[dt][1] = swz_off<DP>(tr_row + 4, 32 * dt + tr_col) * 2;
  }

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x16{};

#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < ntiles) load_tile(i, i, cvo);

  for (int j0 = 0; j0 < ntiles; j0 += NST) {
#pragma unroll
    for (int si = 0; si < NST; ++si) {
      const int j = j0 + si;
      if (j >= ntiles) break;
      // Tile j has landed once at most the next tile's loads are
      // outstanding (loads complete in order; waves with one more chunk slot
      // wait a little longer); then every wave is past tile j - 1, whose
      // stage takes tile j + NST - 1.
      if (j + 1 < ntiles)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NCH / NW) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (j + NST - 1 < ntiles) load_tile(j + NST - 1, (si + NST - 1) % NST, cvo);
      const int kbase = j * BN;
      const bool active = !CAUSAL || (kbase <= qw_lo + 31 + off);
      if (active) {
        const LDS_AS char* st = sm + si * STG_B;
        const LDS_AS char* kt = st + DS_B;
        // slot s of the B operand is key kbase + 16 ks + 8 hh + s: masked if
        // 16 ks + s > lim
        const bool need_mask = CAUSAL && kbase + BN - 1 > qw_lo + off;
        const int lim = qrow + off - kbase - 8 * hh;
#pragma unroll
        for (int ks = 0; ks < BN / 16; ++ks) {
          const LDS_AS char* db = st + (ks >> 1) * (DS_B / 2) + (ks & 1) * 256;
          X8 bop = cat4<X8, X4>(lds_read_tr((const LDS_AS T*)(db + dsb0)), lds_read_tr((const LDS_AS T*)(db + dsb1)));
          if (need_mask) {
            asm volatile("" ::: "memory");
            u32x4 w = __builtin_bit_cast(u32x4, bop);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int k_lo = 16 * ks + 2 * e;
              const uint32_t m = (k_lo > lim ? 0u : 0xffffu) | (k_lo + 1 > lim ? 0u : 0xffff0000u);
              w[e] &= m;
            }
            bop = __builtin_bit_cast(X8, w);
          }
          const LDS_AS char* kb = kt + ks * 16 * DP * 2;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const X8 a = cat4<X8, X4>(lds_read_tr((const LDS_AS T*)(kb + troff[dt][0])),
                                      lds_read_tr((const LDS_AS T*)(kb + troff[dt][1])));
            acc[dt] = mfma32(a, bop, acc[dt]);
          }
        }
      }
    }
  }

  if (qrow < nq) {
    T* row = dQ + (int64_t)qrow * p.sdqn;
    const float sc = p.scale;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * dt + 8 * g + 4 * hh;
        if (d < D) {
          X4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (T)(acc[dt][4 * g + e] * sc);
          *(X4*)(row + d) = v;
        }
      }
    }
  }
}

// Stored-dS path (head dim 128; phases: bit 0 dQ, bit 1 dK/dV):
// fa_bwd_prep_kernel, then per chunk of p.nbh heads fa_bwd_dkdv_kernel
// storing dS into p.ds and fa_bwd_dq_ds_kernel reading it back.
template <typename T, bool CAUSAL>
static hipError_t launch_bwd_ds(BwdParams p, int phases, hipStream_t s) {
  hipError_t e = hipSuccess;
  const int BH = p.B * p.H;
  const int ktiles = (p.Nk + 127) / 128, qtiles = (p.Nq + 255) / 256;
  if ((phases & 2) && p.nq_pad > 0) {
    hipLaunchKernelGGL((fa_bwd_prep_kernel<T, 128>), dim3(BH * (p.nq_pad / 64)), dim3(256), 0, s, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  for (int bh0 = 0; bh0 < BH; bh0 += p.nbh) {
    BwdParams c = p;
    c.bh0 = bh0;
    const int n = BH - bh0 < p.nbh ? BH - bh0 : p.nbh;
    if ((phases & 2) && ktiles > 0) {
      c.num_tiles = ktiles;
      c.heads_per_group = heads_per_group_for((long long)p.Nq * 128 * 2 * 2);  // Q and dO rows of a head
      hipLaunchKernelGGL((fa_bwd_dkdv_kernel<T, 128, CAUSAL, true>), dim3(ktiles * n), dim3(256), 0, s, c);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if ((phases & 1) && qtiles > 0) {
      c.num_tiles = qtiles;
      c.heads_per_group = heads_per_group_for((long long)p.Nk * 128 * 2);  // K rows of a head (dS streams once)
      hipLaunchKernelGGL((fa_bwd_dq_ds_kernel<T, 128, CAUSAL>), dim3(qtiles * n), dim3(512), 0, s, c);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
  }
  return e;
}

// BwdParams::ranked_tokens of a varlen launch of B sequences of up to num_tiles
// tiles (`longest` tokens) on `heads` heads (heads_kv K/V heads).
// Longest first keeps the XCDs and the tail level where lengths differ, but it
// streams the rows of all sequences at once, so that an L2 holds none of them for
// long once many K/V heads take part, and each workgroup pays 1 to 2 us for its
// rank. Measured on 688 packed batches of 2..64 sequences (head dims 64 and 128,
// 16/16, 32/8 and 16/2 heads, shortest 16 tokens, half, 0.85 or all of the longest),
// map_tile's order (batch, then head) against longest first, us:
//   one or two tiles, or no more items than CUs: 82 -> 108 (64 x 250, 16/16), 18 -> 20;
//   few sequences: 87 -> 72 (3 x 1000, 16/16), 826 -> 387 (8 of 16..2000, 32/8), 1552 -> 1061
//   (8 of 16..4000, 16/16), but 157 -> 165 (8 x 1000, 16/16);
//   many: 1769 -> 1501 (33 of 16..2000, 32/8), 2187 -> 2026 (33 x 2000, 16/2), but 1159 -> 1265
//   (33 x 1000, 32/8), 2099 -> 2624 (33 x 2000, 16/16), 1.2 times (64 of 1000..2000, 16/16).
// So the share of the tokens that may be there falls with the K/V heads in all
// sequences: 92% at 128 of them, 84% at 264, 67% at 528.
static int ranked_tokens_for(int B, int heads, int heads_kv, int num_tiles, int longest) {
  const long long grid = (long long)B * num_tiles * heads, streams = (long long)B * heads_kv;
  if (B > 64 || num_tiles < 3 || grid <= 256) return -1;
  if (grid <= 1024 && num_tiles >= 8 && streams < 64) return 0x7fffffff;
  const long long percent = std::min(97LL, 100 - streams / 16) - (num_tiles < 5 ? 15 : 0);
  return (int)std::min(0x7fffffffLL, (long long)B * longest * std::max(40LL, percent) / 100);
}

// phases: bit 0 dQ, bit 1 dK/dV. With p.ds set, the stored-dS path above;
// otherwise the recompute path: fa_bwd_dq_kernel (whose prologue writes the
// ld blocks), then fa_bwd_dkdv_kernel.
template <typename T, int DP, bool CAUSAL>
static hipError_t launch_bwd(BwdParams p, int phases, hipStream_t s) {
  if (p.ds != nullptr) {
    if constexpr (DP == 128) return launch_bwd_ds<T, CAUSAL>(p, phases, s);
    return hipErrorInvalidValue;  // the host takes the stored-dS path only at head dim 128
  }
  // An empty axis means an empty grid: that kernel has nothing to write
  // (with no queries dK = dV = 0 still needs the dK/dV kernel, which then
  // runs no query tile).
  hipError_t e = hipSuccess;
  const int BH = p.B * p.H;
  p.bh0 = 0;
  p.nbh = BH;
  p.num_tiles = (p.Nq + 127) / 128;
  p.heads_per_group = heads_per_group_for((long long)p.Nk * DP * 2 * 2);  // K and V rows of a head
  const bool varlen = p.cu_q != nullptr;  // grids over the longest sequence; shorter ones exit early
  p.ranked_tokens = varlen ? ranked_tokens_for(p.B, p.H, p.H / p.G, p.num_tiles, p.Nq) : -1;
  if ((phases & 1) && p.num_tiles > 0) {
    if (varlen)
      hipLaunchKernelGGL((fa_bwd_dq_kernel<T, DP, CAUSAL, true>), dim3(p.num_tiles * BH), dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL((fa_bwd_dq_kernel<T, DP, CAUSAL>), dim3(p.num_tiles * BH), dim3(256), 0, s, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  p.num_tiles = (p.Nk + 127) / 128;
  // one workgroup per (b, KV head, key tile); it streams the Q and dO rows of the group's G heads
  p.heads_per_group = heads_per_group_for((long long)p.Nq * DP * 2 * 2 * p.G);
  p.ranked_tokens = varlen ? ranked_tokens_for(p.B, p.H / p.G, p.H / p.G, p.num_tiles, p.Nk) : -1;
  if ((phases & 2) && p.num_tiles > 0) {
    const dim3 grid(p.num_tiles * (BH / p.G));
    if (varlen && p.G > 1)
      hipLaunchKernelGGL((fa_bwd_dkdv_kernel<T, DP, CAUSAL, false, true, true>), grid, dim3(256), 0, s, p);
    else if (varlen)
      hipLaunchKernelGGL((fa_bwd_dkdv_kernel<T, DP, CAUSAL, false, false, true>), grid, dim3(256), 0, s, p);
    else if (p.G > 1)
      hipLaunchKernelGGL((fa_bwd_dkdv_kernel<T, DP, CAUSAL, false, true>), grid, dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL((fa_bwd_dkdv_kernel<T, DP, CAUSAL, false>), grid, dim3(256), 0, s, p);
    e = hipGetLastError();
  }
  return e;
}

template <typename T>
static hipError_t dispatch_bwd_t(const BwdParams& p, int dp, bool causal, int ph, hipStream_t s) {
  switch (dp) {
    case 32: return causal ? launch_bwd<T, 32, true>(p, ph, s) : launch_bwd<T, 32, false>(p, ph, s);
    case 64: return causal ? launch_bwd<T, 64, true>(p, ph, s) : launch_bwd<T, 64, false>(p, ph, s);
    default: return causal ? launch_bwd<T, 128, true>(p, ph, s) : launch_bwd<T, 128, false>(p, ph, s);
  }
}

hipError_t bwd_mfma(const BwdParams& p, bool is_bf16, int dp, bool causal, int phases, hipStream_t s) {
  if (is_bf16) return dispatch_bwd_t<__bf16>(p, dp, causal, phases, s);
  return dispatch_bwd_t<_Float16>(p, dp, causal, phases, s);
}

}  // namespace lsfa
