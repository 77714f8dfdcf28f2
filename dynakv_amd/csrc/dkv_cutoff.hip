// Cutoff head: the per-token retained-dimension count r and the masked coefficients that feed
// the cache append, for K and V in one call.
//
// Reference behaviour: src/dynakv/kernels/compressed_attention.py:84-119 (kv_process_fused):
//   logits = b + x @ W                      (addmm in the compute dtype, :92-93)
//   mask   = flip(cumsum(softmax(logits)))  (:99)
//   hard   = mask >= 0.1                    (:100; 0.1 compared in the compute dtype)
//   hard[..., low_rank:] = 0                (:106-107)
//   len    = sum(hard) (int32), out = x * hard (:113-117)
// Here every group g of a row (G groups of D dims; G = 1 is the reference's joint 1024-d head,
// G = 8 with D = 128 its per-head form) has its own W_g and b_g.
//
// Because cumsum of the non-negative softmax is non-decreasing, flip(cumsum) >= thr is a prefix
// mask: its length is the number of positions m whose prefix sum c_m reaches thr, and
// out = x on the first len dims (min(len, low_rank)), x * 0 after them.
//
// Kernels, by the shape of the call:
//   cutoff_small_kernel   D <= 128, a decode step's rows: one launch of 8 waves per 16 rows;
//   cutoff_fused_kernel   D <= 128, a prompt's rows: one launch, a wave takes 16 rows through
//                         logits, softmax, count and masked copy with a row in four lanes;
//   cutoff_logits_ks_kernel (few rows) or cutoff_logits_tile_kernel, then cutoff_rows_kernel
//                         D >= 256 (the joint head): the logits into the caller's workspace,
//                         then one wave per (row, group, K|V).
// Every path rounds as the reference does: bias added in fp32 and the sum rounded to the compute
// dtype (addmm's output), softmax in fp32 of the rounded logits with the probabilities rounded
// to the compute dtype (as torch.softmax returns them), prefix sums accumulated in fp32 and
// rounded to the compute dtype, counted against the threshold rounded to the compute dtype. The
// rounded logits are left in the caller's workspace.
// W is taken transposed, Wt[g][n][k] = W_g[k][n] (the input dimension contiguous), so both MFMA
// operands are 16-byte row loads; the Python layer prepares that copy once per weight.
#include "dkv_internal.h"

namespace {

constexpr int CT_ROWS = 16;   // rows per logits workgroup
constexpr int CT_COLS = 64;   // logits per workgroup (16 per wave)

struct CutoffMat {
  const uint16_t* x;   // (M, G*D) rows, stride x_ld
  const uint16_t* wt;  // (G, D, D): wt[g][n][k]
  const uint16_t* b;   // (G, D)
  uint16_t* out;       // (M, G*D) rows, stride out_ld
  int* lens;           // (M, G) rows, stride len_ld
  uint16_t* logits;    // workspace (M, G, D)
};

struct CutoffParams {
  CutoffMat mat[2];
  long long x_ld, out_ld, len_ld;
  int M, G, D, low_rank;
  float count_min;     // smallest fp32 value whose rounding to the compute dtype is >= the
                       // threshold (itself rounded to the compute dtype)
  int vec;             // 16-byte stores of out and logits are aligned
};

template <int DT>
__device__ __forceinline__ dkv_f32x4 mfma_16x16x32(const dkv_u32x4& a, const dkv_u32x4& b,
                                                   dkv_f32x4 c) {
  if constexpr (DT == DKV_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dkv_bf16x8, a),
                                                   __builtin_bit_cast(dkv_bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(dkv_f16x8, a),
                                                  __builtin_bit_cast(dkv_f16x8, b), c, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ float elt_f32(uint16_t v) {
  if constexpr (DT == DKV_BF16)
    return dkv_bf16_bits_to_f32(v);
  else
    return dkv_f16_bits_to_f32(v);
}
template <int DT>
__device__ __forceinline__ uint16_t f32_elt(float v) {
  if constexpr (DT == DKV_BF16)
    return (uint16_t)dkv_f32_to_bf16_bits(v);
  else
    return (uint16_t)dkv_f32_to_f16_bits(v);
}

// One wave: logits n0 .. n0 + 15 of rows row0 .. row0 + 15.
// MFMA operands: A = x rows (lane: row i = lane % 16, inputs 8*(lane/16) .. +8 of the k-step),
// B = Wt rows (lane: output n = lane % 16, the same inputs); the result lane holds rows
// 4*(lane/16) + u of output column lane % 16.
template <int DT>
__device__ __forceinline__ void logits_tile(const CutoffParams& p, int mat, int g, int row0,
                                            int n0, int lane) {
  const int i = lane & 15, kg = lane >> 4;
  const CutoffMat& cm = p.mat[mat];
  const int D = p.D;
  const int xrow = min(row0 + i, p.M - 1);  // rows past M compute a copy of the last row
  const uint16_t* xa = cm.x + (long long)xrow * p.x_ld + (long long)g * D + 8 * kg;
  const uint16_t* wb = cm.wt + ((long long)g * D + n0 + i) * D + 8 * kg;
  dkv_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int k = 0;
  for (; k + 128 <= D; k += 128) {
    dkv_u32x4 a[4], b[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      a[s] = *(const dkv_u32x4*)(xa + k + 32 * s);
      b[s] = *(const dkv_u32x4*)(wb + k + 32 * s);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma_16x16x32<DT>(a[s], b[s], acc);
  }
  for (; k < D; k += 32)
    acc = mfma_16x16x32<DT>(*(const dkv_u32x4*)(xa + k), *(const dkv_u32x4*)(wb + k), acc);
  const float bias = elt_f32<DT>(cm.b[(long long)g * D + n0 + i]);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int m = row0 + 4 * kg + u;
    if (m < p.M)
      cm.logits[((long long)m * p.G + g) * D + n0 + i] = f32_elt<DT>(acc[u] + bias);
  }
}
// Split-K logits for wide heads (D = 128 * STEPS, the joint 1024-d head: STEPS = 8): grid
// (D / 16, ceil(M / 16), 2 * G), one workgroup per 16 logits of 16 rows; wave w takes the
// quarter w of the input dimension, issues every operand load of its STEPS k-steps before the
// first product, and the four partial sums are added in wave order through LDS (one memory
// round trip per workgroup instead of one per k-step).
template <int DT, int STEPS>
__global__ __launch_bounds__(256) void cutoff_logits_ks_kernel(CutoffParams p) {
  __shared__ dkv_f32x4 sP[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int mat = blockIdx.z & 1, g = blockIdx.z >> 1;
  const int row0 = blockIdx.y * CT_ROWS, n0 = blockIdx.x * 16;
  const int i = lane & 15, kg = lane >> 4;
  const CutoffMat& cm = p.mat[mat];
  const int D = p.D;
  const int k0 = wave * STEPS * 32;
  const int xrow = min(row0 + i, p.M - 1);  // rows past M compute a copy of the last row
  const uint16_t* xa = cm.x + (long long)xrow * p.x_ld + (long long)g * D + k0 + 8 * kg;
  const uint16_t* wb = cm.wt + ((long long)g * D + n0 + i) * D + k0 + 8 * kg;
  dkv_u32x4 a[STEPS], b[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    a[s] = *(const dkv_u32x4*)(xa + 32 * s);
    b[s] = *(const dkv_u32x4*)(wb + 32 * s);
  }
  dkv_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < STEPS; ++s) acc = mfma_16x16x32<DT>(a[s], b[s], acc);
  sP[wave][lane] = acc;
  __syncthreads();
  if (wave == 0) {
    dkv_f32x4 t = sP[0][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) t += sP[w][lane];
    const float bias = elt_f32<DT>(cm.b[(long long)g * D + n0 + i]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = row0 + 4 * kg + u;
      if (m < p.M) cm.logits[((long long)m * p.G + g) * D + n0 + i] = f32_elt<DT>(t[u] + bias);
    }
  }
}

// 16 bytes per lane from a buffer resource straight to LDS, lane l's at lds_base + 16 * l.
__device__ __forceinline__ void ct_lds_load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds_base,
                                              uint32_t byte_off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               ::"s"(lds_base), "v"(byte_off), "s"(rsrc)
               : "memory", "m0");
}
__device__ __forceinline__ uint32_t ct_lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

constexpr int CG_TN = 128;  // logits per tiled workgroup
constexpr int CG_KS = 64;   // inputs per staged step

// Logits of wide heads for many rows (a prompt), D = 128 * STEPS: workgroup = TM rows x 128
// logits, four waves of TM/2 x 64, the inputs staged in LDS 64 at a time (two to four buffers,
// direct-to-LDS loads, 16-byte chunk c of a row at position c ^ (row % 8)). A = W rows, staged in
// the order that gives lane (row n, g) the 16 consecutive logits 16g .. of its wave's 64 (LDS row
// 16 * blk + i is logit 16 * (i / 4) + 4 * blk + i % 4), B = x rows. The products of each quarter
// of the inputs are summed by themselves and the quarters added in order, as
// cutoff_logits_ks_kernel adds its waves' partial sums: the same logits bit for bit.
// Bound: LDS operand reads (32 x 64 products per wave) and the barrier per step. D = 1024, 3001
// rows: about 20 us for K and V, 0.6 PFLOP/s (110 us in 16 x 16 tiles).
template <int DT, int STEPS, int TM>
__global__ __launch_bounds__(256, 2) void cutoff_logits_tile_kernel(CutoffParams p) {
  constexpr int D = 128 * STEPS, NC = D / CG_TN, NK = D / CG_KS, RB = TM / 32;
  constexpr int NBUF = TM == 32 ? 4 : 2;       // steps in LDS
  constexpr int LOADS = CG_TN / 32 + TM / 32;  // loads per wave and step
  __shared__ __attribute__((aligned(16))) uint8_t sW[NBUF][CG_TN * CG_KS * 2];
  __shared__ __attribute__((aligned(16))) uint8_t sX[NBUF][TM * CG_KS * 2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  // ids go to the 8 XCDs round-robin: XCD = (K | V) x (every fourth row tile), a row tile's
  // column tiles consecutive on it, so an L2 takes in one matrix and a quarter of the rows
  const int rt_n = (p.M + TM - 1) / TM, nrg = (rt_n + 3) / 4;
  const int xcd = blockIdx.x & 7, rank = blockIdx.x >> 3;
  const int mat = xcd & 1;
  const int ct = rank % NC, rt = rank / NC % nrg * 4 + (xcd >> 1), grp = rank / NC / nrg;
  if (rt >= rt_n) return;
  const int col0 = ct * CG_TN, row0 = rt * TM;
  const CutoffMat& cm = p.mat[mat];
  const int rows = min(TM, p.M - row0);

  const __amdgpu_buffer_rsrc_t rx =
      dkv_make_rsrc(cm.x + (long long)row0 * p.x_ld + (long long)grp * D,
                    (uint32_t)(((long long)(rows - 1) * p.x_ld + D) * 2));
  const __amdgpu_buffer_rsrc_t rw =
      dkv_make_rsrc(cm.wt + ((long long)grp * D + col0) * D, (uint32_t)(CG_TN * D * 2));
  // loads of step k (past the last step: the last one again, into a buffer nobody reads):
  // instruction c of wave w fills LDS rows 8 * (4c + w) .. + 7, lane l row l / 8's chunk
  // position l % 8
  auto issue = [&](int k) {
    const int buf = k % NBUF, k0 = min(k, NK - 1) * CG_KS;
#pragma unroll
    for (int c = 0; c < CG_TN / 32; ++c) {
      const int r8 = 8 * (4 * c + wave), r = r8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (r & 7);
      const int i = r & 15, blk = (r >> 4) & 3;
      const int col = (r & 64) + 16 * (i >> 2) + 4 * blk + (i & 3);
      ct_lds_load16(rw, ct_lds_addr(&sW[buf][r8 * CG_KS * 2]),
                    (uint32_t)((col * D + k0 + 8 * chunk) * 2));
    }
#pragma unroll
    for (int c = 0; c < TM / 32; ++c) {
      const int r8 = 8 * (4 * c + wave), r = r8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (r & 7);
      // rows past M read the last row
      ct_lds_load16(rx, ct_lds_addr(&sX[buf][r8 * CG_KS * 2]),
                    (uint32_t)(((long long)min(r, rows - 1) * p.x_ld + k0 + 8 * chunk) * 2));
    }
  };
  const int wr = (wave >> 1) * (TM / 2), wc = (wave & 1) * 64;
  dkv_f32x4 acc[RB][4], tot[RB][4];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      acc[rb][blk] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
      tot[rb][blk] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
  for (int k = 0; k < NBUF - 1; ++k) issue(k);
#pragma unroll 1
  for (int q = 0; q < 4; ++q) {
#pragma unroll 1
    for (int kk = 0; kk < NK / 4; ++kk) {
      const int k = q * (NK / 4) + kk;
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 2) * LOADS) : "memory");  // step k's loads are done
      __syncthreads();  // step k is in LDS for every wave; the buffer of step k - 1 is free
      issue(k + NBUF - 1);
      const uint8_t *wt = sW[k % NBUF], *xt = sX[k % NBUF];
#pragma unroll
      for (int s = 0; s < CG_KS / 32; ++s) {
        const int pos = 16 * ((4 * s + g) ^ (n & 7));
        dkv_u32x4 a[4], b[RB];
#pragma unroll
        for (int blk = 0; blk < 4; ++blk)
          a[blk] = *(const dkv_u32x4*)(wt + (wc + 16 * blk + n) * (CG_KS * 2) + pos);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          b[rb] = *(const dkv_u32x4*)(xt + (wr + 16 * rb + n) * (CG_KS * 2) + pos);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int blk = 0; blk < 4; ++blk)
            acc[rb][blk] = mfma_16x16x32<DT>(a[blk], b[rb], acc[rb][blk]);
      }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        tot[rb][blk] += acc[rb][blk];
        acc[rb][blk] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int n0 = col0 + wc + 16 * g;  // this lane's 16 logits
  float bias[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) bias[e] = elt_f32<DT>(cm.b[(long long)grp * D + n0 + e]);
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int m = row0 + wr + 16 * rb + n;
    if (m >= p.M) continue;
    uint32_t w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int blk = e >> 1, u = 2 * (e & 1);
      w[e] = (uint32_t)f32_elt<DT>(tot[rb][blk][u] + bias[2 * e]) |
             ((uint32_t)f32_elt<DT>(tot[rb][blk][u + 1] + bias[2 * e + 1]) << 16);
    }
    uint16_t* lo = cm.logits + ((long long)m * p.G + grp) * D + n0;
    if (p.vec) {
      *(dkv_u32x4*)lo = dkv_u32x4{w[0], w[1], w[2], w[3]};
      *(dkv_u32x4*)(lo + 8) = dkv_u32x4{w[4], w[5], w[6], w[7]};
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) lo[e] = (uint16_t)(w[e / 2] >> (16 * (e & 1)));
    }
  }
}

// a / s rounded to fp32, from r = 1 / s (correctly rounded): the product and one correction step by
// the exact remainder, which rounds as the division does (Markstein's theorem) while the remainder
// does not underflow (quotients above about 2^-100; smaller ones only a threshold as small could
// see). The empty asm keeps the fp32 quotient a value of its own: the compiler otherwise folds the
// last fma and the conversion to fp16 that follows into one v_fma_mixlo_f16, which rounds once, and
// probabilities beside an fp16 tie come out as the other neighbour.
__device__ __forceinline__ float cf_div(float a, float s, float r) {
  const float q = a * r;
  float v = __builtin_fmaf(__builtin_fmaf(-q, s, a), r, q);
  asm("" : "+v"(v));
  return v;
}

// The retained count of one (row m, group g) of a matrix, computed by one wave from the
// row's rounded logits (global workspace or LDS). Lane l owns the E = D / 64 consecutive
// positions l*E .. l*E + E - 1 of the row.
template <int DT, int E>
__device__ __forceinline__ int cutoff_row_len(const CutoffParams& p, const uint16_t* row,
                                              int lane) {
  const uint16_t* lg = row + lane * E;

  float x[E];
  if constexpr (E >= 8) {
    // 16-byte loads (the row and each lane's E elements are 16-byte aligned)
#pragma unroll
    for (int v = 0; v < E / 8; ++v) {
      const dkv_u32x4 w = *(const dkv_u32x4*)(lg + 8 * v);
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        x[8 * v + e] = elt_f32<DT>((uint16_t)(ww[e >> 1] >> (16 * (e & 1))));
    }
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = elt_f32<DT>(lg[e]);
  }
  float mx = x[0];
#pragma unroll
  for (int e = 1; e < E; ++e) mx = fmaxf(mx, x[e]);
  mx = dkv_wave_max_fast(mx);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    x[e] = expf(x[e] - mx);
    s += x[e];
  }
  s = dkv_wave_sum_fast(s);
  // probabilities in the compute dtype, then their prefix sums accumulated in fp32
  const float rcp = 1.0f / s;
  float run = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    run += dkv_round_to<DT>(cf_div(x[e], s, rcp));
    x[e] = run;  // inclusive prefix within the lane
  }
  const float inc = dkv_wave_scan_fast(run);  // inclusive scan of the lane totals
  const float excl = inc - run;
  int cnt = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) cnt += excl + x[e] >= p.count_min ? 1 : 0;
  cnt = dkv_wave_sum_fast_i(cnt);
  return min(cnt, max(p.low_rank, 0));
}

// One wave per (row m, group g, K|V): the count and the masked copy of the row.
template <int DT, int E>
__device__ __forceinline__ void row_task(const CutoffParams& p, int mat, long long rg, int lane) {
  const int m = (int)(rg / p.G), g = (int)(rg % p.G);
  const CutoffMat& cm = p.mat[mat];
  const int D = p.D;
  const int len = cutoff_row_len<DT, E>(p, cm.logits + rg * D, lane);

  const uint16_t* xs = cm.x + (long long)m * p.x_ld + (long long)g * D + lane * E;
  uint16_t* xo = cm.out + (long long)m * p.out_ld + (long long)g * D + lane * E;
  uint16_t xv[E];
  if constexpr (E >= 8) {
    // 16-byte loads of the input (x rows are 16-byte aligned: checked by the host)
#pragma unroll
    for (int v = 0; v < E / 8; ++v) {
      const dkv_u32x4 w = *(const dkv_u32x4*)(xs + 8 * v);
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) xv[8 * v + e] = (uint16_t)(ww[e >> 1] >> (16 * (e & 1)));
    }
  } else {
#pragma unroll
    for (int e = 0; e < E; ++e) xv[e] = xs[e];
  }
  // x * 1 or x * 0 in the compute dtype, written out bitwise: x * 0 is a zero with x's sign,
  // or NaN for an infinite or NaN x (a multiply would do the same, but the compiler may turn
  // it into an fma with a +0 addend, which loses the sign of -0)
  constexpr uint16_t EXP = DT == DKV_BF16 ? 0x7f80 : 0x7c00;
  constexpr uint16_t QNAN = DT == DKV_BF16 ? 0x7fc0 : 0x7e00;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const uint16_t xb = xv[e];
    const uint16_t zb = (xb & EXP) == EXP ? QNAN : (uint16_t)(xb & 0x8000);
    xo[e] = lane * E + e < len ? xb : zb;
  }
  if (lane == 0) cm.lens[(long long)m * p.len_ld + g] = len;
}
template <int DT, int E>
__global__ __launch_bounds__(256) void cutoff_rows_kernel(CutoffParams p) {
  const int lane = threadIdx.x & 63;
  const long long task = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const long long n_rows = (long long)p.M * p.G;
  if (task >= 2 * n_rows) return;
  row_task<DT, E>(p, (int)(task / n_rows), task % n_rows, lane);
}

// Few rows of D <= 128 (a decode step) in one launch of 8 waves per (16 rows, group, K|V): the
// logits of the rows go to LDS (wave w: output columns 16w .. 16w+15; every operand load issued
// before the first product, the masked copies' inputs loaded ahead as well), then wave w takes
// rows w and w + 8: count, masked copy, length. One memory round trip before the stores.
constexpr int CS_WAVES = 8;

template <int DT>
__device__ __forceinline__ void small_logits(const CutoffParams& p, int mat, int g, int wave,
                                             int lane, uint16_t (*sLog)[128], int row0) {
  const int n0 = 16 * wave;
  if (n0 >= p.D) return;
  const int i = lane & 15, kg = lane >> 4;
  const CutoffMat& cm = p.mat[mat];
  const int D = p.D;
  const uint16_t* xa =
      cm.x + (long long)min(row0 + i, p.M - 1) * p.x_ld + (long long)g * D + 8 * kg;
  const uint16_t* wb = cm.wt + ((long long)g * D + n0 + i) * D + 8 * kg;
  dkv_u32x4 a[4], b[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int k = min(32 * s, D - 32);  // D = 64: the last two steps are loaded but not used
    a[s] = *(const dkv_u32x4*)(xa + k);
    b[s] = *(const dkv_u32x4*)(wb + k);
  }
  const float bias = elt_f32<DT>(cm.b[(long long)g * D + n0 + i]);
  dkv_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; ++s)
    if (32 * s < D) acc = mfma_16x16x32<DT>(a[s], b[s], acc);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int m = row0 + 4 * kg + u;
    if (m < p.M) {
      const uint16_t v = f32_elt<DT>(acc[u] + bias);
      sLog[m - row0][n0 + i] = v;
      cm.logits[((long long)m * p.G + g) * D + n0 + i] = v;  // the workspace copy, as the
                                                               // two-kernel path leaves it
    }
  }
}

template <int DT, int E>
__global__ __launch_bounds__(64 * CS_WAVES) void cutoff_small_kernel(CutoffParams p) {
  __shared__ uint16_t sLog[CT_ROWS][128];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int mat = blockIdx.x & 1, g = blockIdx.x >> 1, row0 = blockIdx.y * CT_ROWS;
  const CutoffMat& cm = p.mat[mat];
  const int D = p.D;
  uint16_t xr[2][E];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int m = min(row0 + wave + CS_WAVES * r, p.M - 1);
    const uint16_t* xs = cm.x + (long long)m * p.x_ld + (long long)g * D + lane * E;
#pragma unroll
    for (int e = 0; e < E; ++e) xr[r][e] = xs[e];
  }
  small_logits<DT>(p, mat, g, wave, lane, sLog, row0);
  __syncthreads();
  constexpr uint16_t EXP = DT == DKV_BF16 ? 0x7f80 : 0x7c00;
  constexpr uint16_t QNAN = DT == DKV_BF16 ? 0x7fc0 : 0x7e00;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int m = row0 + wave + CS_WAVES * r;
    if (m >= p.M) break;
    const int len = cutoff_row_len<DT, E>(p, &sLog[m - row0][0], lane);
    uint16_t* xo = cm.out + (long long)m * p.out_ld + (long long)g * D + lane * E;
    // x * 1 or x * 0 written bitwise, as row_task writes them
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint16_t xb = xr[r][e];
      const uint16_t zb = (xb & EXP) == EXP ? QNAN : (uint16_t)(xb & 0x8000);
      xo[e] = lane * E + e < len ? xb : zb;
    }
    if (lane == 0) cm.lens[(long long)m * p.len_ld + g] = len;
  }
}

// max / sum over the four lanes n, n + 16, n + 32, n + 48
__device__ __forceinline__ float cf_max4(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float cf_sum4(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr int CF_WAVES = 4;

// The whole cutoff head of a prompt with D = 16 * NB <= 128 in one launch. Workgroup (x, group
// and matrix): W_g staged once in LDS in operand order, then each wave takes 16-row tiles
// grid-stride, the next tile's rows loading while one is worked on.
// MFMA operands: A = W rows (the logits), B = x rows, with the W rows permuted so that lane
// (row n = lane % 16, g = lane / 16) receives the D / 4 consecutive logits D / 4 * g .. of its
// row: A row i of block blk is logit D / 4 * (i / 4) + 4 * blk + i % 4. A row's maximum, sum
// and prefix sums then need two exchanges between four lanes instead of six steps across the
// wave for each, for 16 rows at once, and the masked copy is the B operand itself.
// Bound: VALU (softmax and counts, ~35 instructions per logit) and HBM. 8192 rows x 8 groups x
// 128, bf16: 31.2 us a call for 102 MB (two kernels, one a wave per row, 104.6; with the sums in
// the lanes' own order, whose counts fall otherwise on rounding ties, 29.0).
template <int DT, int NB>
__global__ __launch_bounds__(64 * CF_WAVES, 3) void cutoff_fused_kernel(CutoffParams p) {
  constexpr int D = 16 * NB, KS = D / 32, PL = D / 4;  // PL: logits per lane
  __shared__ __attribute__((aligned(16))) dkv_u32x4 sW[NB * KS][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int mat = blockIdx.y & 1, grp = blockIdx.y >> 1;
  const CutoffMat& cm = p.mat[mat];
  const int tiles = (p.M + 15) / 16, step = gridDim.x * CF_WAVES;
  int tile = blockIdx.x * CF_WAVES + wave;

  dkv_u32x4 xn[KS];
  auto load_x = [&](int t) {
    // rows past M (and tiles past the last) read the last row
    const uint16_t* xr = cm.x + (long long)min(16 * t + n, p.M - 1) * p.x_ld + grp * D + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) xn[s] = *(const dkv_u32x4*)(xr + 32 * s);
  };
  load_x(tile);
  for (int f = wave; f < NB * KS; f += CF_WAVES) {
    const int blk = f / KS, s = f % KS;
    sW[f][lane] = *(const dkv_u32x4*)(
        cm.wt + ((long long)grp * D + PL * (n >> 2) + 4 * blk + (n & 3)) * D + 32 * s + 8 * g);
  }
  uint32_t bias[PL / 2];  // packed pairs of this lane's logits
#pragma unroll
  for (int e = 0; e < PL / 2; ++e) {
    const uint16_t* b = cm.b + grp * D + PL * g + 2 * e;
    bias[e] = (uint32_t)b[0] | ((uint32_t)b[1] << 16);
  }
  __syncthreads();

  for (; tile < tiles; tile += step) {
    // keeps the W operands in LDS: hoisted out of the loop they would take 128 registers
    asm volatile("" ::: "memory");
    dkv_u32x4 x[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) x[s] = xn[s];
    load_x(tile + step);

    dkv_f32x4 acc[NB];
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
      acc[blk] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
        acc[blk] = mfma_16x16x32<DT>(sW[blk * KS + s][lane], x[s], acc[blk]);
    }
    // the rounded logits, packed (element e of the lane: logit PL * g + e)
    uint32_t lg[PL / 2];
#pragma unroll
    for (int e = 0; e < PL / 2; ++e) {
      const float v0 = acc[e / 2][2 * (e & 1)] + elt_f32<DT>((uint16_t)bias[e]);
      const float v1 = acc[e / 2][2 * (e & 1) + 1] + elt_f32<DT>((uint16_t)(bias[e] >> 16));
      lg[e] = (uint32_t)f32_elt<DT>(v0) | ((uint32_t)f32_elt<DT>(v1) << 16);
    }
    const int m = 16 * tile + n;
    const bool live = m < p.M;
    if (live) {
      uint16_t* lo = cm.logits + ((long long)m * p.G + grp) * D + PL * g;
      if (p.vec) {
#pragma unroll
        for (int v = 0; v < PL / 8; ++v)
          *(dkv_u32x4*)(lo + 8 * v) =
              dkv_u32x4{lg[4 * v], lg[4 * v + 1], lg[4 * v + 2], lg[4 * v + 3]};
      } else {
#pragma unroll
        for (int e = 0; e < PL; ++e) lo[e] = (uint16_t)(lg[e / 2] >> (16 * (e & 1)));
      }
    }
    auto logit = [&](int e) { return elt_f32<DT>((uint16_t)(lg[e / 2] >> (16 * (e & 1)))); };
    float mx = logit(0);
#pragma unroll
    for (int e = 1; e < PL; ++e) mx = fmaxf(mx, logit(e));
    mx = cf_max4(mx);
    // The sums below are taken in the order of cutoff_row_len (64 lanes of E consecutive positions:
    // a lane here holds 16 of those lanes' positions), so that a count on a rounding tie falls
    // the same way on every path.
    constexpr int E = PL / 16;
    float pr[PL], part[16];
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      part[l] = 0.f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        pr[E * l + e] = expf(logit(E * l + e) - mx);
        part[l] += pr[E * l + e];
      }
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1)  // the butterfly's tree
#pragma unroll
      for (int l = 0; l < 16; l += 2 * d) part[l] += part[l + d];
    const float sum = cf_sum4(part[0]);
    // probabilities in the compute dtype, their prefix sums in fp32
    const float rcp = 1.0f / sum;
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      float run = 0.f;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        run += dkv_round_to<DT>(cf_div(pr[E * l + e], sum, rcp));
        pr[E * l + e] = run;
      }
      part[l] = run;
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1)  // inclusive scan of the 16 totals
#pragma unroll
      for (int l = 15; l >= d; --l) part[l] += part[l - d];
    // the totals of the row's lanes before this one
    const float t16 = __shfl_xor(part[15], 16, 64);
    const float t32 = __shfl_xor(part[15] + t16, 32, 64);
    const float b1 = (g & 1) ? t16 : 0.f, b2 = (g & 2) ? t32 : 0.f;
    // a prefix sum counts when its rounding reaches the threshold, i.e. when it reaches the
    // smallest fp32 value that rounds to it
    int cnt = 0;
#pragma unroll
    for (int l = 0; l < 16; ++l) {
      const float excl = ((part[l] + b1) + b2) - pr[E * l + E - 1];
#pragma unroll
      for (int e = 0; e < E; ++e) cnt += excl + pr[E * l + e] >= p.count_min ? 1 : 0;
    }
    cnt += __shfl_xor(cnt, 16, 64);
    cnt += __shfl_xor(cnt, 32, 64);
    const int len = min(cnt, max(p.low_rank, 0));

    if (!live) continue;
    // x * 1 or x * 0 written bitwise, as row_task writes them
    constexpr uint32_t EXP = DT == DKV_BF16 ? 0x7f80u : 0x7c00u;
    constexpr uint32_t QNAN = DT == DKV_BF16 ? 0x7fc0u : 0x7e00u;
    uint16_t* xo = cm.out + (long long)m * p.out_ld + grp * D + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t w[4] = {x[s].x, x[s].y, x[s].z, x[s].w};
      const int keep = len - 32 * s - 8 * g;  // elements of this piece that stay
      uint32_t o[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t a = w[d] & 0xffffu, b = w[d] >> 16;
        const uint32_t za = (a & EXP) == EXP ? QNAN : (a & 0x8000u);
        const uint32_t zb = (b & EXP) == EXP ? QNAN : (b & 0x8000u);
        o[d] = (2 * d < keep ? a : za) | ((2 * d + 1 < keep ? b : zb) << 16);
      }
      if (p.vec) {
        *(dkv_u32x4*)(xo + 32 * s) = dkv_u32x4{o[0], o[1], o[2], o[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) xo[32 * s + e] = (uint16_t)(o[e / 2] >> (16 * (e & 1)));
      }
    }
    if (g == 0) cm.lens[(long long)m * p.len_ld + grp] = len;
  }
}

// Decode step of the per-head layout, after the logits: for each (batch b, group g, K|V) the
// count, then the decode append of that token to cache row b*G + g at position seq (the first
// len coefficients -- exactly what the masked copy followed by the append stores); waves past
// those tasks rotate the query rows (RoPE at position pos).
struct TailParams {
  CutoffParams cp;
  void* flat[2];
  long long flat_ld[2];
  int* lens[2];
  int* offs[2];
  long long tab_sb[2], tab_ss[2];
  int* ptr[2];
  int seq;
  uint16_t* q;
  long long q_sb;  // elements between batch rows of q (heads are contiguous 128-element rows)
  int q_rows, Hq;
  int pos;
  float log_theta;
};

// count, table entries and append of cache row rg = b*G + g of matrix mat (one wave). pre:
// the row's pointer (lane 0) and this lane's E coefficients when the caller loaded them
// ahead (have_pre), else they are loaded here.
template <int DT, int E>
__device__ __forceinline__ void append_row(const TailParams& t, int mat, long long rg, int lane,
                                           bool have_pre = false, int pre_off = 0,
                                           const uint16_t* pre_x = nullptr) {
  const CutoffParams& p = t.cp;
  const int m = (int)(rg / p.G), g = (int)(rg % p.G);
  const int len = cutoff_row_len<DT, E>(p, p.mat[mat].logits + rg * p.D, lane);
  int off = 0;
  if (lane == 0) {
    off = have_pre ? pre_off : t.ptr[mat][rg];
    t.ptr[mat][rg] = off + len;
    t.lens[mat][rg * t.tab_sb[mat] + (long long)t.seq * t.tab_ss[mat]] = len;
    t.offs[mat][rg * t.tab_sb[mat] + (long long)t.seq * t.tab_ss[mat]] = off;
  }
  off = __shfl(off, 0, 64);
  const uint16_t* xs = p.mat[mat].x + (long long)m * p.x_ld + (long long)g * p.D + lane * E;
  uint16_t* dst = (uint16_t*)t.flat[mat] + rg * t.flat_ld[mat] + off + lane * E;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (lane * E + e < len) dst[e] = have_pre ? pre_x[e] : xs[e];
}

// One launch for the whole tail of a decode step's cutoff head: workgroup 2g + mat computes the
// logits of group g of matrix mat (K or V) for 16 rows at a time (wave w: columns 16w + 64c, as
// logits_tile computes them), then its waves take those rows' counts and appends;
// the workgroups past 2G rotate the query rows (RoPE at position pos), one per wave.
template <int DT, int E>
__global__ __launch_bounds__(256) void cutoff_layer_kernel(TailParams t) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const CutoffParams& p = t.cp;
  const int n_cut = 2 * p.G;
  if ((int)blockIdx.x < n_cut) {
    const int mat = blockIdx.x & 1, g = blockIdx.x >> 1;
    // the first row of each wave: its pointer and coefficients loaded before the logits, so
    // that their latency overlaps the products
    int off0 = 0;
    uint16_t x0[E];
    if (wave < p.M) {
      const long long rg = (long long)wave * p.G + g;
      if (lane == 0) off0 = t.ptr[mat][rg];
      const uint16_t* xs = p.mat[mat].x + (long long)wave * p.x_ld + (long long)g * p.D + lane * E;
#pragma unroll
      for (int e = 0; e < E; ++e) x0[e] = xs[e];
    }
    for (int row0 = 0; row0 < p.M; row0 += CT_ROWS) {
      for (int c0 = 0; c0 < p.D; c0 += CT_COLS) logits_tile<DT>(p, mat, g, row0, c0 + 16 * wave, lane);
      __syncthreads();  // the rows' logits (global workspace) are visible to the workgroup
      for (int m = row0 + wave; m < min(row0 + CT_ROWS, p.M); m += 4)
        append_row<DT, E>(t, mat, (long long)m * p.G + g, lane, m == wave, off0, x0);
    }
    return;
  }
  const long long qr = (long long)(blockIdx.x - n_cut) * 4 + wave;
  if (qr < t.q_rows)
    dkv_rope_pair<DT>(t.q + (qr / t.Hq) * t.q_sb + (qr % t.Hq) * 128, lane, t.pos, t.log_theta);
}

// cutoff_layer_kernel for a decode step of the per-head layout (D <= 128), in one memory round
// trip before the stores: workgroup (16-row tile rt, 2g + mat) of 8 waves loads its rows' append
// pointers and inputs, computes the rows' logits into LDS as cutoff_small_kernel does, then wave
// w appends rows 16 rt + w and 16 rt + w + 8; the workgroups past the 2G x tiles rotate the
// query rows, one per wave.
template <int DT, int E>
__global__ __launch_bounds__(64 * CS_WAVES) void cutoff_layer_small_kernel(TailParams t) {
  __shared__ uint16_t sLog[CT_ROWS][128];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const CutoffParams& p = t.cp;
  const int n_cut = 2 * p.G * ((p.M + CT_ROWS - 1) / CT_ROWS);
  if ((int)blockIdx.x < n_cut) {
    const int rt = blockIdx.x / (2 * p.G), id = blockIdx.x % (2 * p.G);
    const int mat = id & 1, g = id >> 1;
    const int row0 = rt * CT_ROWS;
    const int D = p.D;
    int off[2];
    uint16_t xr[2][E];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int m = min(row0 + wave + CS_WAVES * r, p.M - 1);
      off[r] = t.ptr[mat][(long long)m * p.G + g];
      const uint16_t* xs = p.mat[mat].x + (long long)m * p.x_ld + (long long)g * D + lane * E;
#pragma unroll
      for (int e = 0; e < E; ++e) xr[r][e] = xs[e];
    }
    small_logits<DT>(p, mat, g, wave, lane, sLog, row0);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int m = row0 + wave + CS_WAVES * r;
      if (m >= p.M) break;
      const long long rg = (long long)m * p.G + g;
      const int len = cutoff_row_len<DT, E>(p, &sLog[m - row0][0], lane);
      if (lane == 0) {
        t.ptr[mat][rg] = off[r] + len;
        t.lens[mat][rg * t.tab_sb[mat] + (long long)t.seq * t.tab_ss[mat]] = len;
        t.offs[mat][rg * t.tab_sb[mat] + (long long)t.seq * t.tab_ss[mat]] = off[r];
      }
      uint16_t* dst = (uint16_t*)t.flat[mat] + rg * t.flat_ld[mat] + off[r] + lane * E;
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (lane * E + e < len) dst[e] = xr[r][e];
    }
    return;
  }
  const long long qr = (long long)(blockIdx.x - n_cut) * CS_WAVES + wave;
  if (qr < t.q_rows)
    dkv_rope_pair<DT>(t.q + (qr / t.Hq) * t.q_sb + (qr % t.Hq) * 128, lane, t.pos, t.log_theta);
}

template <int DT, int STEPS, int TM>
void launch_logits_tile(const CutoffParams& p, hipStream_t st) {
  const int nc = 128 * STEPS / CG_TN, rt = (p.M + TM - 1) / TM;
  const unsigned grid = (unsigned)(8LL * nc * ((rt + 3) / 4) * p.G);
  hipLaunchKernelGGL((cutoff_logits_tile_kernel<DT, STEPS, TM>), dim3(grid), dim3(256), 0, st, p);
}

// The logits of every (row, group, K|V) into the workspace, D of 256, 512 or 1024. Graph-replayed
// us of the whole call (bf16 / fp16, one group, D = 1024), split-K / 32-row / 64-row tiles: 64
// rows 9.5 / 11.0 / 12.3, 100 rows 13.0 / 11.2 / 12.4, 512 rows 35.8 / 12.6 / 13.7, 800 rows 52.9
// / 16.1 / 15.4, 3001 rows 122.6 / 42.4 / 32.7; D = 512: 150 rows 8.2 / 8.6 / 9.3, 512 rows
// 13.1 / 9.0 / 9.7, 1500 rows 30.0 / 12.5 / 12.0; D = 256: 301 rows 6.4 / 7.3, 800 rows 9.3 /
// 8.0. So the split-K kernel while its workgroups stay within three per CU (its 16 x 16 tiles
// read 64 KB of operands for 0.5 MFLOP, but all at once), then 32-row tiles while they leave CUs
// idle or about fill them, then 64-row ones. The tile kernels address x by 32-bit offsets
// from a tile's first row, so a larger row stride stays on split-K.
void launch_logits(const CutoffParams& p, int dtype, hipStream_t st) {
  const int D = p.D, M = p.M, G = p.G;
  const unsigned gy = (unsigned)((M + CT_ROWS - 1) / CT_ROWS), gz = (unsigned)(2 * G);
  if ((long long)(D / 16) * gy * gz > 3 * 256 && p.x_ld < (1LL << 23)) {
#define DKV_LT(STEPS_, TM_)                             \
  do {                                                  \
    if (dtype == DKV_BF16)                              \
      launch_logits_tile<DKV_BF16, STEPS_, TM_>(p, st); \
    else                                                \
      launch_logits_tile<DKV_F16, STEPS_, TM_>(p, st);  \
  } while (0)
    const bool small = (long long)(D / CG_TN) * ((M + 31) / 32) * gz <= 320;
    if (D == 1024) {
      if (small) DKV_LT(8, 32);
      else DKV_LT(8, 64);
    } else if (D == 512) {
      if (small) DKV_LT(4, 32);
      else DKV_LT(4, 64);
    } else {
      if (small) DKV_LT(2, 32);
      else DKV_LT(2, 64);
    }
#undef DKV_LT
    return;
  }
#define DKV_LKS(STEPS_)                                                                        \
  do {                                                                                         \
    if (dtype == DKV_BF16)                                                                     \
      hipLaunchKernelGGL((cutoff_logits_ks_kernel<DKV_BF16, STEPS_>), dim3(D / 16, gy, gz),    \
                         dim3(256), 0, st, p);                                                 \
    else                                                                                       \
      hipLaunchKernelGGL((cutoff_logits_ks_kernel<DKV_F16, STEPS_>), dim3(D / 16, gy, gz),     \
                         dim3(256), 0, st, p);                                                 \
  } while (0)
  if (D == 1024)
    DKV_LKS(8);
  else if (D == 512)
    DKV_LKS(4);
  else
    DKV_LKS(2);
#undef DKV_LKS
}

template <int DT, int E>
void launch_rows(const CutoffParams& p, hipStream_t st) {
  const long long tasks = 2LL * p.M * p.G;
  hipLaunchKernelGGL((cutoff_rows_kernel<DT, E>), dim3((unsigned)((tasks + 3) / 4)), dim3(256), 0,
                     st, p);
}

template <int DT, int NB>
void launch_fused(const CutoffParams& p, hipStream_t st) {
  // about three resident workgroups per CU (registers); every wave the same number of tiles
  const int tiles = (p.M + 15) / 16;
  const int most = max(1, 3 * 256 / (2 * p.G));
  const int per_wave = (tiles + most * CF_WAVES - 1) / (most * CF_WAVES);
  const int gx = (tiles + per_wave * CF_WAVES - 1) / (per_wave * CF_WAVES);
  hipLaunchKernelGGL((cutoff_fused_kernel<DT, NB>), dim3(gx, 2 * p.G), dim3(64 * CF_WAVES), 0, st,
                     p);
}

// The smallest fp32 value whose rounding to the compute dtype is >= thr (a value of that
// dtype): the midpoint between thr and its predecessor, or the next fp32 value when the tie
// goes to the predecessor.
float count_min_of(int dtype, float thr) {
  if (!(thr > 0.f) || !(thr <= 2.f)) return thr <= 0.f ? -INFINITY : thr;  // prefix sums are in [0, ~1]
  const uint16_t bits = dtype == DKV_BF16 ? __builtin_bit_cast(uint16_t, (__bf16)thr)
                                          : __builtin_bit_cast(uint16_t, (_Float16)thr);
  const uint16_t prev_bits = (uint16_t)(bits - 1);
  const float prev = dtype == DKV_BF16 ? (float)__builtin_bit_cast(__bf16, prev_bits)
                                       : (float)__builtin_bit_cast(_Float16, prev_bits);
  const float mid = prev + 0.5f * (thr - prev);  // exact: one more bit than the dtype holds
  return (bits & 1) == 0 ? mid : nextafterf(mid, INFINITY);
}

}  // namespace

extern "C" long long dkv_cutoff_workspace_bytes(int M, int G, int D) {
  if (M < 0 || G <= 0 || D <= 0) return -1;
  return 2LL * M * G * D * 2;
}

extern "C" int dkv_cutoff_kv(void* stream, int dtype, const void* xk, const void* xv,
                             long long x_ld, const void* wt_k, const void* wt_v, const void* b_k,
                             const void* b_v, float threshold, int low_rank, void* out_k,
                             void* out_v, long long out_ld, int* len_k, int* len_v,
                             long long len_ld, void* workspace, long long workspace_bytes, int M,
                             int G, int D) {
  if (dtype != DKV_F16 && dtype != DKV_BF16) return DKV_E_UNSUPPORTED;
  if (M < 0 || G <= 0 || D <= 0) return DKV_E_ARG;
  if (M == 0) return DKV_OK;
  if (!xk || !xv || !wt_k || !wt_v || !b_k || !b_v || !out_k || !out_v || !len_k || !len_v ||
      !workspace)
    return DKV_E_ARG;
  if (D % 64 != 0 || D > 1024) return DKV_E_UNSUPPORTED;
  if (x_ld < (long long)G * D || out_ld < (long long)G * D || len_ld < G) return DKV_E_ARG;
  if (x_ld % 8 != 0 || ((uintptr_t)xk | (uintptr_t)xv | (uintptr_t)wt_k | (uintptr_t)wt_v) % 16)
    return DKV_E_UNSUPPORTED;  // 16-byte operand loads
  if (workspace_bytes < dkv_cutoff_workspace_bytes(M, G, D)) return DKV_E_WORKSPACE;
  if ((long long)M * G * D >= (1LL << 31) / 2) return DKV_E_UNSUPPORTED;
  CutoffParams p;
  const void* xs[2] = {xk, xv};
  const void* ws[2] = {wt_k, wt_v};
  const void* bs[2] = {b_k, b_v};
  void* os[2] = {out_k, out_v};
  int* ls[2] = {len_k, len_v};
  for (int t = 0; t < 2; ++t) {
    p.mat[t].x = (const uint16_t*)xs[t];
    p.mat[t].wt = (const uint16_t*)ws[t];
    p.mat[t].b = (const uint16_t*)bs[t];
    p.mat[t].out = (uint16_t*)os[t];
    p.mat[t].lens = ls[t];
    p.mat[t].logits = (uint16_t*)workspace + (long long)t * M * G * D;
  }
  p.x_ld = x_ld;
  p.out_ld = out_ld;
  p.len_ld = len_ld;
  p.M = M;
  p.G = G;
  p.D = D;
  p.low_rank = low_rank < 0 ? D : min(low_rank, D);
  // the reference compares against 0.1 in the compute dtype
  p.count_min = count_min_of(
      dtype, dtype == DKV_BF16 ? (float)(__bf16)threshold : (float)(_Float16)threshold);
  p.vec = (((uintptr_t)out_k | (uintptr_t)out_v | (uintptr_t)workspace) % 16 == 0 &&
           out_ld % 8 == 0)
              ? 1
              : 0;
  const int E = D / 64;
  if (E != 1 && E != 2 && E != 4 && E != 8 && E != 16) return DKV_E_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  // D <= 128: the 8-wave kernel (a 16-row tile per workgroup) up to one workgroup per CU, the
  // wave-per-tile kernel past that. Graph-replayed us per call, 8-wave / wave per tile (bf16, fp16
  // within 2%): G = 8, D = 128: 33 rows (48 workgroups) 5.3 / 6.7, 250 (256) 5.6 / 7.1, 301 (304)
  // 7.5 / 7.3, 1024 rows 12.4 / 8.2, 8192 rows 66 / 31.6 (two kernels, a wave per row, before: 5.9
  // at 33 rows, 19.6 at 1024, 105 at 8192); G = 4: 500 rows (256) 5.6 / 7.1, 640 (320) 7.5 / 7.3;
  // G = 2: 1024 (256) 5.7 / 7.1, 1300 (328) 7.7 / 7.2; G = 32: 33 (192) 5.4 / 6.8, 100 (448) 7.8 /
  // 7.4; G = 8, D = 64: 250 4.4 / 4.5, 301 5.7 / 4.7.
  const long long row_tiles = (M + CT_ROWS - 1) / CT_ROWS;
  if (D <= 128 && (row_tiles == 1 || 2 * G * row_tiles <= 256)) {
    const dim3 sgrid((unsigned)(2 * G), (unsigned)row_tiles);
    if (dtype == DKV_BF16) {
      if (E == 1)
        hipLaunchKernelGGL((cutoff_small_kernel<DKV_BF16, 1>), sgrid, dim3(64 * CS_WAVES), 0, st, p);
      else
        hipLaunchKernelGGL((cutoff_small_kernel<DKV_BF16, 2>), sgrid, dim3(64 * CS_WAVES), 0, st, p);
    } else {
      if (E == 1)
        hipLaunchKernelGGL((cutoff_small_kernel<DKV_F16, 1>), sgrid, dim3(64 * CS_WAVES), 0, st, p);
      else
        hipLaunchKernelGGL((cutoff_small_kernel<DKV_F16, 2>), sgrid, dim3(64 * CS_WAVES), 0, st, p);
    }
    DKV_HIP_CHECK_LAUNCH();
    return DKV_OK;
  }
  if (D <= 128) {
    if (2 * G > 65535) return DKV_E_UNSUPPORTED;
    if (dtype == DKV_BF16) {
      if (E == 1)
        launch_fused<DKV_BF16, 4>(p, st);
      else
        launch_fused<DKV_BF16, 8>(p, st);
    } else {
      if (E == 1)
        launch_fused<DKV_F16, 4>(p, st);
      else
        launch_fused<DKV_F16, 8>(p, st);
    }
    DKV_HIP_CHECK_LAUNCH();
    return DKV_OK;
  }
  launch_logits(p, dtype, st);
  DKV_HIP_CHECK_LAUNCH();
#define DKV_ROWS_CASE(e)                                        \
  case e:                                                       \
    if (dtype == DKV_BF16)                                      \
      launch_rows<DKV_BF16, e>(p, st);                          \
    else                                                        \
      launch_rows<DKV_F16, e>(p, st);                           \
    break;
  switch (E) {
    DKV_ROWS_CASE(4)
    DKV_ROWS_CASE(8)
    DKV_ROWS_CASE(16)
    default:
      return DKV_E_UNSUPPORTED;
  }
#undef DKV_ROWS_CASE
  DKV_HIP_CHECK_LAUNCH();
  return DKV_OK;
}

// The decode step's cutoff head, K+V append and query RoPE in one launch
// (cutoff_layer_kernel). Used by dkv_decode_layer; same checks as
// dkv_cutoff_kv for the cutoff part. The per-row scratch (coef_k/v, len_k/v) of the layer's
// argument block is not used.
int dkv_layer_cutoff_append_rope(void* stream, const DkvDecodeLayer* L, const void* k_coef,
                                 const void* v_coef, void* q, int seq, int pos) {
  const int dtype = L->dtype, M = L->B, G = L->G, D = L->R;
  if (dtype != DKV_F16 && dtype != DKV_BF16) return DKV_E_UNSUPPORTED;
  if (M < 0 || G <= 0 || D <= 0 || L->Hq <= 0 || L->Dh != 128) return DKV_E_ARG;
  if (M == 0) return DKV_OK;
  if (!L->wt_k || !L->wt_v || !L->b_k || !L->b_v || !L->cut_ws || !L->flat_k || !L->flat_v ||
      !L->lens_k || !L->offs_k || !L->lens_v || !L->offs_v || !L->ptr_k || !L->ptr_v)
    return DKV_E_ARG;
  if (D % 64 != 0 || D > 1024) return DKV_E_UNSUPPORTED;
  const long long x_ld = L->coef_ld ? L->coef_ld : (long long)G * D;
  const long long q_sb = L->q_sb ? L->q_sb : (long long)L->Hq * 128;
  if (x_ld < (long long)G * D || q_sb < (long long)L->Hq * 128) return DKV_E_ARG;
  if (x_ld % 8 != 0 || ((uintptr_t)k_coef | (uintptr_t)v_coef | (uintptr_t)L->wt_k |
                        (uintptr_t)L->wt_v) % 16)
    return DKV_E_UNSUPPORTED;
  if (L->cut_ws_bytes < dkv_cutoff_workspace_bytes(M, G, D)) return DKV_E_WORKSPACE;
  if ((long long)M * G * D >= (1LL << 31) / 2) return DKV_E_UNSUPPORTED;
  const int E = D / 64;
  if (E != 1 && E != 2 && E != 4 && E != 8 && E != 16) return DKV_E_UNSUPPORTED;
  TailParams t;
  CutoffParams& p = t.cp;
  const void* xs[2] = {k_coef, v_coef};
  const void* ws[2] = {L->wt_k, L->wt_v};
  const void* bs[2] = {L->b_k, L->b_v};
  for (int m = 0; m < 2; ++m) {
    p.mat[m].x = (const uint16_t*)xs[m];
    p.mat[m].wt = (const uint16_t*)ws[m];
    p.mat[m].b = (const uint16_t*)bs[m];
    p.mat[m].out = nullptr;
    p.mat[m].lens = nullptr;
    p.mat[m].logits = (uint16_t*)L->cut_ws + (long long)m * M * G * D;
  }
  p.x_ld = x_ld;
  p.out_ld = x_ld;
  p.len_ld = G;
  p.M = M;
  p.G = G;
  p.D = D;
  p.low_rank = L->low_rank < 0 ? D : min(L->low_rank, D);
  p.count_min = count_min_of(
      dtype, dtype == DKV_BF16 ? (float)(__bf16)L->threshold : (float)(_Float16)L->threshold);
  p.vec = 0;
  t.flat[0] = L->flat_k;
  t.flat[1] = L->flat_v;
  t.flat_ld[0] = L->flat_k_ld;
  t.flat_ld[1] = L->flat_v_ld;
  t.lens[0] = L->lens_k;
  t.lens[1] = L->lens_v;
  t.offs[0] = L->offs_k;
  t.offs[1] = L->offs_v;
  t.tab_sb[0] = L->tab_k_sb;
  t.tab_sb[1] = L->tab_v_sb;
  t.tab_ss[0] = L->tab_k_ss;
  t.tab_ss[1] = L->tab_v_ss;
  t.ptr[0] = L->ptr_k;
  t.ptr[1] = L->ptr_v;
  t.seq = seq;
  t.q = (uint16_t*)q;
  t.q_sb = q_sb;
  t.q_rows = pos < 0 ? 0 : M * L->Hq;  // pos < 0: the caller rotated q already
  t.Hq = L->Hq;
  t.pos = pos;
  t.log_theta = L->log_theta;
  hipStream_t st = (hipStream_t)stream;
  if (D <= 128) {
    // every 16-row tile of every (group, K|V) in its own workgroup, then the query rows
    const long long tiles = (M + CT_ROWS - 1) / CT_ROWS;
    const dim3 sgrid((unsigned)(2 * G * tiles + (t.q_rows + CS_WAVES - 1) / CS_WAVES));
    if (E == 1) {
      if (dtype == DKV_BF16)
        hipLaunchKernelGGL((cutoff_layer_small_kernel<DKV_BF16, 1>), sgrid, dim3(64 * CS_WAVES),
                           0, st, t);
      else
        hipLaunchKernelGGL((cutoff_layer_small_kernel<DKV_F16, 1>), sgrid, dim3(64 * CS_WAVES),
                           0, st, t);
    } else {
      if (dtype == DKV_BF16)
        hipLaunchKernelGGL((cutoff_layer_small_kernel<DKV_BF16, 2>), sgrid, dim3(64 * CS_WAVES),
                           0, st, t);
      else
        hipLaunchKernelGGL((cutoff_layer_small_kernel<DKV_F16, 2>), sgrid, dim3(64 * CS_WAVES),
                           0, st, t);
    }
    DKV_HIP_CHECK_LAUNCH();
    return DKV_OK;
  }
  const dim3 grid((unsigned)(2 * G + (t.q_rows + 3) / 4));
#define DKV_TAIL_CASE(e)                                                                 \
  case e:                                                                                \
    if (dtype == DKV_BF16)                                                               \
      hipLaunchKernelGGL((cutoff_layer_kernel<DKV_BF16, e>), grid, dim3(256), 0, st, t);       \
    else                                                                                 \
      hipLaunchKernelGGL((cutoff_layer_kernel<DKV_F16, e>), grid, dim3(256), 0, st, t);        \
    break;
  switch (E) {
    DKV_TAIL_CASE(1)
    DKV_TAIL_CASE(2)
    DKV_TAIL_CASE(4)
    DKV_TAIL_CASE(8)
    DKV_TAIL_CASE(16)
    default:
      return DKV_E_UNSUPPORTED;
  }
#undef DKV_TAIL_CASE
  DKV_HIP_CHECK_LAUNCH();
  return DKV_OK;
}
