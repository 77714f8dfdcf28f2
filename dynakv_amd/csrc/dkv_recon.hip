// Dense K and V of a prompt from its masked coefficient rows, for the compressed prefill
// attention (reference compressed_attention.py:359-386 reconstructs the prompt's keys and
// values through the up-projection bases, get_origin_states in compressed_cache.py:36-56 returns
// the coefficients zero past each token's count, and the keys are rotated before the causal
// attention, :375-378). One launch reconstructs both: K[t] = R(t) (B_K^T c_K[t]) and
// V[t] = B_V^T c_V[t] per cache row (b, g), the products on 16x16x32 MFMA with fp32
// accumulation; the keys rounded to the dtype, rotated in fp32 and rounded again, as the
// reference rounds the projection and then the rotation. The rotation of position p = 16T + n
// is R(16T) R(n) composed in fp32 from the rows of the RoPE table (dkv_rope_table: cos and sin
// of the fp32 angles n * inv_freq and 16T * inv_freq), not a sine and cosine per element.
//
// recon_kv_kernel: workgroup = (RW * 16 * tiles tokens, cache row, K | V), four waves of 16 tokens
// at a time (recon_one_kernel, below: a single tile). The row's basis ([rank][dim], ranks past R
// zero) is staged in LDS, read transposed (ds_read_b64_tr_b16) once and kept in registers as the A
// operand (dims x ranks) of every tile; each lane loads its token's 8 coefficients of a 32-rank
// chunk as the B operand, a tile ahead. The dims are dealt to the A rows so that lane (token n, g)
// ends up with dims 16g .. 16g + 15 and 64 + 16g .. of its token: the rotate-half pairs (d, d + 64)
// in one lane, stored 16 bytes at a time. A lane's positions all have one offset in their
// 16-position tile, so R(n) stays in registers too. A transposed basis (BT) is staged and read as
// it lies (us with every wave loading its operands from the basis / staged, rank 128: 64 rows x 128
// tokens 8.1 / 6.6, 16 x 2048 15.7 / 11.5, 4096 x 64 158 / 88, where copying the bases first took
// 99).
// Bound: HBM. B = 4, 8 groups, S = 2048, rank 128 (67 MB): 21 us, 3.2 TB/s; with one 64-token tile
// per workgroup, the basis staged for each and 8-byte stores 32 us. Ranks of 96 and fewer skip the
// chunks past them (16 rows x 2048 tokens, us with all four chunks / skipping: rank 64 12.0 / 10.2,
// rank 8 11.7 / 9.0).
#include "dkv_common.h"
#include "dkv_mfma_ops.h"

namespace {

constexpr int DH = 128;
constexpr int RW = 4;  // waves per workgroup (16 tokens each)
constexpr int RT_FIXED = 17;  // RoPE table rows before the tile rows R(16T)

// One 64-token tile per workgroup (grids of up to 512 workgroups, where the latency of a single tile
// is what a call takes): the A operands read from LDS as each product needs them, chunks past the
// rank skipped, nothing kept for a further tile. Result lane (n, g): dims 16 blk + 4g + u. Graph-
// replayed us, this kernel / recon_kv_kernel with one tile (rows x tokens, rank): 8 x 17, 128
// 5.6 / 6.8; 64 x 128, 128 7.4 / 7.9; 32 x 333, 64 7.4 / 8.9; 16 x 100, 8 4.9 / 6.5; at 512
// workgroups (8 x 2048, 128) 9.9 / 10.1. Above, several tiles per workgroup are ahead (16 x 2048,
// 128 15.0 / 12.9).
template <int DT>
__global__ __launch_bounds__(RW * 64) void recon_one_kernel(
    const uint16_t* __restrict__ ck, const uint16_t* __restrict__ cv, long long c_sr,
    long long c_st, const uint16_t* __restrict__ kb, const uint16_t* __restrict__ vb,
    long long b_sg, long long b_sr, uint16_t* __restrict__ ko, uint16_t* __restrict__ vo,
    long long o_sr, long long o_st, int G, int S, int R, int pos0, const float* __restrict__ rope) {
  __shared__ __attribute__((aligned(16))) uint16_t sB[DH * DH];  // [rank][dim]
  const bool is_k = blockIdx.z == 0;
  const int row = blockIdx.y, grp = row % G;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  const uint16_t* c = is_k ? ck : cv;
  const uint16_t* bg = (is_k ? kb : vb) + (long long)grp * b_sg;
  uint16_t* o = is_k ? ko : vo;

  // this lane's token and its coefficient pieces (ranks 32 cc + 8g .. +8; R is a multiple of 8)
  const int t = (blockIdx.x * RW + wave) * 16 + n;
  const uint16_t* cr = c + (long long)row * c_sr + (long long)min(t, S - 1) * c_st;
  dkv_u32x4 xc[4];
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) {
    const int r0 = 32 * cc + 8 * g;
    xc[cc] = (t < S && r0 < R) ? *(const dkv_u32x4*)(cr + r0) : dkv_u32x4{0u, 0u, 0u, 0u};
  }
  // the basis, 16-byte pieces (rank r, dims d8 .. d8 + 7), ranks past R as zeros
  for (int pc = tid; pc < DH * DH / 8; pc += RW * 64) {
    const int r = pc >> 4, d8 = (pc & 15) * 8;
    *(dkv_u32x4*)(sB + r * DH + d8) =
        r < R ? *(const dkv_u32x4*)(bg + (long long)r * b_sr + d8) : dkv_u32x4{0u, 0u, 0u, 0u};
  }
  __syncthreads();

  dkv_f32x4 acc[8];
#pragma unroll
  for (int blk = 0; blk < 8; ++blk) acc[blk] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
  typedef __attribute__((address_space(3))) dkv_i16x4 lds_i16x4;
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) {
    if (32 * cc >= R) break;  // uniform: chunks wholly past the rank are zero
#pragma unroll
    for (int blk = 0; blk < 8; ++blk) {
      // lane (n, g) receives ranks 32 cc + 8g .. +3 and +4 .. +7 of dim 16 blk + n
      const uint16_t* src = sB + (32 * cc + 8 * g + (n >> 2)) * DH + 16 * blk + 4 * (n & 3);
      const dkv_u32x2 b0 = __builtin_bit_cast(
          dkv_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                         (lds_i16x4*)(__attribute__((address_space(3))) uint16_t*)src));
      const dkv_u32x2 b1 = __builtin_bit_cast(
          dkv_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                         (lds_i16x4*)(__attribute__((address_space(3))) uint16_t*)(src + 4 * DH)));
      acc[blk] = dkv_mfma32<DT>(dkv_u32x4{b0.x, b0.y, b1.x, b1.y}, xc[cc], acc[blk]);
    }
  }
  if (t >= S) return;
  // lane (n, g): dims 16 blk + 4g + u of token t in acc[blk][u]
  if (is_k) {
    const int pos = pos0 + t;
    // (cos, sin) of frequencies 16 blk + 4g .. +3: 32 contiguous bytes of a table row
    const float* rn = rope + (pos & 15) * 128 + 8 * g;
    const float* rt = rope + (RT_FIXED + (pos >> 4)) * 128 + 8 * g;
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      const dkv_f32x4 n0 = *(const dkv_f32x4*)(rn + 32 * blk), n1 = *(const dkv_f32x4*)(rn + 32 * blk + 4);
      const dkv_f32x4 t0 = *(const dkv_f32x4*)(rt + 32 * blk), t1 = *(const dkv_f32x4*)(rt + 32 * blk + 4);
      const float nc[4] = {n0.x, n0.z, n1.x, n1.z}, ns[4] = {n0.y, n0.w, n1.y, n1.w};
      const float tc[4] = {t0.x, t0.z, t1.x, t1.z}, ts[4] = {t0.y, t0.w, t1.y, t1.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float cs = tc[u] * nc[u] - ts[u] * ns[u], sn = ts[u] * nc[u] + tc[u] * ns[u];
        // the projection rounded to the dtype first, then rotated: the reference's two steps
        // (the up-projection's product in the dtype, then apply_rotary_pos_emb_)
        const float a = dkv_round_to<DT>(acc[blk][u]), bb = dkv_round_to<DT>(acc[blk + 4][u]);
        acc[blk][u] = a * cs - bb * sn;
        acc[blk + 4][u] = bb * cs + a * sn;
      }
    }
  }
  uint16_t* orow = o + (long long)row * o_sr + (long long)t * o_st;
#pragma unroll
  for (int blk = 0; blk < 8; ++blk) {
    uint32_t w[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float lo = acc[blk][2 * e], hi = acc[blk][2 * e + 1];
      if constexpr (DT == DKV_BF16)
        w[e] = dkv_f32_to_bf16_bits(lo) | (dkv_f32_to_bf16_bits(hi) << 16);
      else
        w[e] = dkv_f32_to_f16_bits(lo) | (dkv_f32_to_f16_bits(hi) << 16);
    }
    *(dkv_u32x2*)(orow + 16 * blk + 4 * g) = dkv_u32x2{w[0], w[1]};
  }
}

template <int DT, bool BT>
__global__ __launch_bounds__(RW * 64, 2) void recon_kv_kernel(
    const uint16_t* __restrict__ ck, const uint16_t* __restrict__ cv, long long c_sr,
    long long c_st, const uint16_t* __restrict__ kb, const uint16_t* __restrict__ vb,
    long long b_sg, long long b_sr, uint16_t* __restrict__ ko, uint16_t* __restrict__ vo,
    long long o_sr, long long o_st, int G, int S, int R, int pos0, const float* __restrict__ rope,
    int tiles) {
  __shared__ __attribute__((aligned(16))) uint16_t sB[DH * DH];  // [rank][dim]
  const bool is_k = blockIdx.z == 0;
  const int row = blockIdx.y, grp = row % G;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  const uint16_t* c = is_k ? ck : cv;
  const uint16_t* bg = (is_k ? kb : vb) + (long long)grp * b_sg;
  uint16_t* o = is_k ? ko : vo;

  // a lane's token of tile i and its coefficient pieces (ranks 32 cc + 8g .. +8; R is a multiple
  // of 8); tokens past S read as zeros
  const int tok0 = (blockIdx.x * tiles * RW + wave) * 16 + n;
  const uint16_t* cr = c + (long long)row * c_sr;
  dkv_u32x4 xn[4];
  auto load_x = [&](int t) {
    const uint16_t* cp = cr + (long long)min(t, S - 1) * c_st;
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      const int r0 = 32 * cc + 8 * g;
      xn[cc] = (t < S && r0 < R) ? *(const dkv_u32x4*)(cp + r0) : dkv_u32x4{0u, 0u, 0u, 0u};
    }
  };
  load_x(tok0);
  // R(n) of the lane's positions, frequencies 16g .. 16g + 15 as (cos, sin) pairs
  dkv_f32x4 rn[8];
  if (is_k) {
    const float* rp = rope + ((pos0 + n) & 15) * 128 + 32 * g;
#pragma unroll
    for (int e = 0; e < 8; ++e) rn[e] = *(const dkv_f32x4*)(rp + 4 * e);
  }
  // A operands: block blk = 4h + b, row i holds dim 64h + 16 (i / 4) + 4b + i % 4; lane (n, g)
  // receives ranks 32 cc + 8g .. +3 and +4 .. +7 of its row's dim
  typedef __attribute__((address_space(3))) dkv_i16x4 lds_i16x4;
  dkv_u32x4 a[4][8];
  if constexpr (BT) {
    // [dim][rank] as it comes, 16-byte pieces (dim d, ranks 8c .. 8c + 7; those past R as zeros; of
    // 32, 64 or 128 ranks) at position c ^ (d % 4 + 4 (d / 16 % 4)), so that the 16 rows of an
    // operand read lie apart
    const int sh = R > 64 ? 4 : (R > 32 ? 3 : 2);
    for (int pc = tid; pc < DH << sh; pc += RW * 64) {
      const int d = pc >> sh, c8 = pc & ((1 << sh) - 1);
      *(dkv_u32x4*)(sB + d * DH + 8 * (c8 ^ ((d & 3) | ((d >> 2) & 12)))) =
          8 * c8 < R ? *(const dkv_u32x4*)(bg + (long long)d * b_sr + 8 * c8)
                     : dkv_u32x4{0u, 0u, 0u, 0u};
    }
  } else {
    // the basis up to its last 32-rank chunk, 16-byte pieces (rank r, dims d8 .. d8 + 7), ranks past
    // R as zeros
    for (int pc = tid; pc < (R + 31) / 32 * 32 * (DH / 8); pc += RW * 64) {
      const int r = pc >> 4, d8 = (pc & 15) * 8;
      *(dkv_u32x4*)(sB + r * DH + d8) =
          r < R ? *(const dkv_u32x4*)(bg + (long long)r * b_sr + d8) : dkv_u32x4{0u, 0u, 0u, 0u};
    }
  }
  __syncthreads();
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) {
    if (32 * cc >= R) break;  // uniform: chunks wholly past the rank take no part
#pragma unroll
    for (int blk = 0; blk < 8; ++blk) {
      if constexpr (BT) {
        const int d = 64 * (blk >> 2) + 16 * (n >> 2) + 4 * (blk & 3) + (n & 3);
        a[cc][blk] = *(const dkv_u32x4*)(sB + d * DH + 8 * ((4 * cc + g) ^ n));
      } else {
        const uint16_t* src = sB + (32 * cc + 8 * g + (n >> 2)) * DH + 64 * (blk >> 2) +
                              16 * (n & 3) + 4 * (blk & 3);
        const dkv_u32x2 b0 = __builtin_bit_cast(
            dkv_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                           (lds_i16x4*)(__attribute__((address_space(3))) uint16_t*)src));
        const dkv_u32x2 b1 = __builtin_bit_cast(
            dkv_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                           (lds_i16x4*)(__attribute__((address_space(3))) uint16_t*)(src + 4 * DH)));
        a[cc][blk] = dkv_u32x4{b0.x, b0.y, b1.x, b1.y};
      }
    }
  }

  for (int i = 0; i < tiles; ++i) {
    const int t = tok0 + i * RW * 16;
    if (t - n >= S) break;  // the wave's tokens are all past the end (uniform)
    dkv_f32x4 acc[8];
#pragma unroll
    for (int blk = 0; blk < 8; ++blk) acc[blk] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      if (32 * cc >= R) break;
#pragma unroll
      for (int blk = 0; blk < 8; ++blk) acc[blk] = dkv_mfma32<DT>(a[cc][blk], xn[cc], acc[blk]);
    }
    if (i + 1 < tiles) load_x(t + RW * 16);
    if (t >= S) continue;
    // lane (n, g): dims 64h + 16g + 4b + u of token t in acc[4h + b][u]
    if (is_k) {
      const float* rt = rope + (RT_FIXED + ((pos0 + t) >> 4)) * 128 + 32 * g;
#pragma unroll
      for (int e = 0; e < 8; ++e) {  // frequencies 16g + 2e, + 1
        const dkv_f32x4 tt = *(const dkv_f32x4*)(rt + 4 * e);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          const int b = e >> 1, u = 2 * (e & 1) + f;
          const float tc = tt[2 * f], ts = tt[2 * f + 1], nc = rn[e][2 * f], ns = rn[e][2 * f + 1];
          const float cs = tc * nc - ts * ns, sn = ts * nc + tc * ns;
          // the projection rounded to the dtype first, then rotated: the reference's two steps
          // (the up-projection's product in the dtype, then apply_rotary_pos_emb_)
          const float x = dkv_round_to<DT>(acc[b][u]), y = dkv_round_to<DT>(acc[4 + b][u]);
          acc[b][u] = x * cs - y * sn;
          acc[4 + b][u] = y * cs + x * sn;
        }
      }
    }
    uint16_t* orow = o + (long long)row * o_sr + (long long)t * o_st + 16 * g;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float lo = acc[4 * h + (e >> 1)][2 * (e & 1)];
        const float hi = acc[4 * h + (e >> 1)][2 * (e & 1) + 1];
        if constexpr (DT == DKV_BF16)
          w[e] = dkv_f32_to_bf16_bits(lo) | (dkv_f32_to_bf16_bits(hi) << 16);
        else
          w[e] = dkv_f32_to_f16_bits(lo) | (dkv_f32_to_f16_bits(hi) << 16);
      }
      uint16_t* od = orow + 64 * h;
      if (((uintptr_t)od & 15) == 0) {
        *(dkv_u32x4*)od = dkv_u32x4{w[0], w[1], w[2], w[3]};
        *(dkv_u32x4*)(od + 8) = dkv_u32x4{w[4], w[5], w[6], w[7]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) *(dkv_u32x2*)(od + 4 * e) = dkv_u32x2{w[2 * e], w[2 * e + 1]};
      }
    }
  }
}

}  // namespace

static int recon_kv(int bt, void* stream, int dtype, const void* ck, const void* cv,
                            long long c_sr, long long c_st, const void* k_basis,
                            const void* v_basis, long long b_sg, long long b_sr, void* k_out,
                            void* v_out, long long o_sr, long long o_st, int rows, int G, int S,
                            int R, int pos0, const float* rope, int rope_tiles) {
  if (dtype != DKV_F16 && dtype != DKV_BF16) return DKV_E_UNSUPPORTED;
  if (rows < 0 || G <= 0 || S < 0 || R <= 0 || pos0 < 0) return DKV_E_ARG;
  if (rows == 0 || S == 0) return DKV_OK;
  if (!ck || !cv || !k_basis || !v_basis || !k_out || !v_out || !rope) return DKV_E_ARG;
  if ((long long)rope_tiles * 16 < (long long)pos0 + S) return DKV_E_ARG;
  if ((uintptr_t)rope & 15) return DKV_E_UNSUPPORTED;
  if (R > DH || R % 8 != 0 || rows % G != 0) return DKV_E_UNSUPPORTED;
  // 16-byte coefficient pieces and basis rows, 8-byte output pieces
  auto a16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  if (!a16(ck) || !a16(cv) || !a16(k_basis) || !a16(v_basis) || (c_sr & 7) || (c_st & 7) ||
      (b_sg & 7) || (b_sr & 7) || ((uintptr_t)k_out & 7) || ((uintptr_t)v_out & 7) ||
      (o_sr & 3) || (o_st & 3))
    return DKV_E_UNSUPPORTED;
  if (S > 65535 * 64 || rows > 65535) return DKV_E_UNSUPPORTED;
  // 64-token tiles per workgroup: the grid within the 512 workgroups that run at once (two per
  // CU). Graph-replayed us, rank 128, one tile each in recon_one_kernel / the chosen count: 512 tiles
  // in all (8 rows x 2048 tokens) 9.9; 768 12.8 / 11.9 (two); 1024 14.9 / 12.7 (two); 2048 28.6 / 20.1
  // (four; 1 / 2 / 4 tiles of recon_kv_kernel when it was written: 36.6 / 27.6 / 21.0).
  const long long t64 = (S + 63) / 64, per = (t64 * rows * 2 + 511) / 512;
  const int tiles = (int)(per < t64 ? per : t64);
  const dim3 grid((unsigned)((t64 + tiles - 1) / tiles), (unsigned)rows, 2);
  hipStream_t st = (hipStream_t)stream;
#define DKV_RECON(KERNEL, ...)                                                                  \
  hipLaunchKernelGGL((KERNEL), grid, dim3(RW * 64), 0, st, (const uint16_t*)ck,                 \
                     (const uint16_t*)cv, c_sr, c_st, (const uint16_t*)k_basis,                 \
                     (const uint16_t*)v_basis, b_sg, b_sr, (uint16_t*)k_out, (uint16_t*)v_out,  \
                     o_sr, o_st, G, S, R, pos0, rope __VA_OPT__(, ) __VA_ARGS__)
  if (tiles == 1 && !bt) {
    if (dtype == DKV_BF16)
      DKV_RECON(recon_one_kernel<DKV_BF16>);
    else
      DKV_RECON(recon_one_kernel<DKV_F16>);
  } else if (bt) {
    if (dtype == DKV_BF16)
      DKV_RECON((recon_kv_kernel<DKV_BF16, true>), tiles);
    else
      DKV_RECON((recon_kv_kernel<DKV_F16, true>), tiles);
  } else {
    if (dtype == DKV_BF16)
      DKV_RECON((recon_kv_kernel<DKV_BF16, false>), tiles);
    else
      DKV_RECON((recon_kv_kernel<DKV_F16, false>), tiles);
  }
#undef DKV_RECON
  DKV_HIP_CHECK_LAUNCH();
  return DKV_OK;
}

extern "C" int dkv_recon_kv(void* stream, int dtype, const void* ck, const void* cv,
                            long long c_sr, long long c_st, const void* k_basis,
                            const void* v_basis, long long b_sg, long long b_sr, void* k_out,
                            void* v_out, long long o_sr, long long o_st, int rows, int G, int S,
                            int R, int pos0, const float* rope, int rope_tiles) {
  return recon_kv(0, stream, dtype, ck, cv, c_sr, c_st, k_basis, v_basis, b_sg, b_sr, k_out, v_out,
                  o_sr, o_st, rows, G, S, R, pos0, rope, rope_tiles);
}

extern "C" int dkv_recon_kv_bt(void* stream, int dtype, const void* ck, const void* cv,
                               long long c_sr, long long c_st, const void* k_basis,
                               const void* v_basis, long long b_sg, long long b_sd, void* k_out,
                               void* v_out, long long o_sr, long long o_st, int rows, int G, int S,
                               int R, int pos0, const float* rope, int rope_tiles) {
  return recon_kv(1, stream, dtype, ck, cv, c_sr, c_st, k_basis, v_basis, b_sg, b_sd, k_out, v_out,
                  o_sr, o_st, rows, G, S, R, pos0, rope, rope_tiles);
}
