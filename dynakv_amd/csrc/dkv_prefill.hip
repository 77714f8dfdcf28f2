// Prefill attention over the reconstructed cache.
//
// Reference behaviour: the prefill branch of CustomAttention.forward
// (src/dynakv/kernels/compressed_attention.py:359-386) packs the prompt's coefficients into the
// cache (update_sp), re-expands the whole cache (get_origin_states, compressed_cache.py:70-81),
// projects it through k_up / v_up (:160-165), applies RoPE at positions 0..S-1 to K
// (calc_cos_sin, :193-200, then apply_rotary_pos_emb_) and runs causal attention of the
// prompt's (RoPE'd) queries over it (eager / SDPA, :373-383).
//
// Here: dkv_rope_dense rotates dense K in place (rotate-half RoPE, fp32 angles
// float(pos) * inv_freq as the decode kernels form them, result rounded to the cache dtype);
// dkv_prefill_attention is a causal GQA flash-attention forward on MFMA:
//   one workgroup = 64 or 128 queries of one query head (4 waves x 2 blocks of 16 queries for a
//   grid that fills the chip several times, so every K and V operand read from LDS serves two
//   products; smaller grids 8 or 4 waves of one block), the work items handed out longest
//   first and evenly over the 8 XCDs, a KV head's query heads on one XCD (the grid's own
//   order gave XCD k only the query blocks k, k+8, ...: 0.40 ms against 0.25 at B=4,
//   S=2048); key tiles of 64
//   are staged in LDS (double-buffered, direct-to-LDS loads, 16-byte chunks XOR-swizzled by
//   key so that both the row reads of K and the transposed reads of V avoid bank conflicts);
//   S^T = K Q^T on 16x16x32 MFMA (each lane then holds one query's scores for 16 keys), online
//   softmax in fp32 with lane maxima by permlane swaps (the running maximum raised only when a
//   tile's exceeds it by more than 2^8, so most tiles skip the rescale), P kept as a bf16/fp16
//   hi + lo pair and P.V on 16x16x32 MFMA over 32 keys at a time, one product with the hi parts
//   and one with the lo parts against the same V operand (read transposed from LDS ahead of the
//   softmax).
#include "dkv_common.h"

namespace {

constexpr int FA_DH = 128;
constexpr float FA_RESCALE = 8.f;  // log2 units a tile's maximum may exceed the running one
constexpr int FA_BK = 64;     // keys per tile
constexpr int FA_TILE_BYTES = FA_BK * FA_DH * 2;  // 16 KB

struct PrefillParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  void* out;
  long long q_sb, q_sh, q_ss;
  long long k_sb, k_sh, k_ss;
  long long v_sb, v_sh, v_ss;
  long long o_sb, o_sh, o_ss;
  int B, Hq, Hkv, Sq, Sk, q_offset, causal;
  float scale_log2;  // softmax scale * log2(e)
  uint32_t k_bytes, v_bytes;
  const int* kstart;  // per batch row: keys before it are masked (left padding); may be null
};

template <int DT>
__device__ __forceinline__ dkv_f32x4 mfma32(const dkv_u32x4& a, const dkv_u32x4& b, dkv_f32x4 c) {
  if constexpr (DT == DKV_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dkv_bf16x8, a),
                                                   __builtin_bit_cast(dkv_bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(dkv_f16x8, a),
                                                  __builtin_bit_cast(dkv_f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ void fa_lds_load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds_base,
                                              uint32_t byte_off, uint32_t tile_off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               ::"s"(lds_base), "v"(byte_off), "s"(rsrc), "s"(tile_off)
               : "memory", "m0");
}

__device__ __forceinline__ uint32_t fa_lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

__device__ __forceinline__ float fa_max(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

__device__ __forceinline__ float fa_max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// max over the four lanes n, n+16, n+32, n+48
__device__ __forceinline__ float fa_max4(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fa_max(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fa_max(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <int DT>
__device__ __forceinline__ void split_hi_lo(const float (&p)[4], dkv_u32x2& hi, dkv_u32x2& lo) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  if constexpr (DT == DKV_BF16) {
    const dkv_bf16x2 h01 = __builtin_convertvector(f32x2{p[0], p[1]}, dkv_bf16x2);
    const dkv_bf16x2 h23 = __builtin_convertvector(f32x2{p[2], p[3]}, dkv_bf16x2);
    const dkv_bf16x2 l01 =
        __builtin_convertvector(f32x2{p[0] - (float)h01[0], p[1] - (float)h01[1]}, dkv_bf16x2);
    const dkv_bf16x2 l23 =
        __builtin_convertvector(f32x2{p[2] - (float)h23[0], p[3] - (float)h23[1]}, dkv_bf16x2);
    hi = dkv_u32x2{__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23)};
    lo = dkv_u32x2{__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23)};
  } else {
    const dkv_f16x2 h01 = __builtin_convertvector(f32x2{p[0], p[1]}, dkv_f16x2);
    const dkv_f16x2 h23 = __builtin_convertvector(f32x2{p[2], p[3]}, dkv_f16x2);
    const dkv_f16x2 l01 =
        __builtin_convertvector(f32x2{p[0] - (float)h01[0], p[1] - (float)h01[1]}, dkv_f16x2);
    const dkv_f16x2 l23 =
        __builtin_convertvector(f32x2{p[2] - (float)h23[0], p[3] - (float)h23[1]}, dkv_f16x2);
    hi = dkv_u32x2{__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23)};
    lo = dkv_u32x2{__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23)};
  }
}

// grid: (ceil(Sq / (16 QB NW)), Hq, B); NW waves of QB blocks of 16 queries (the workgroup's item
// is remapped from its linear id, see below). ODT: output dtype (DT or fp32).
// Bound: issue slots. Per wave and tile (QB = 2) 96 products of 16 cycles against ~235 vector
// instructions, which measure 6.6 cycles each beside a full product stream (10.5 for exp2): the
// vector work of one wave has to fit beside the products of the others. B = 4, S = 2048, 32/8
// heads: 187 us, 1.1 PFLOP/s of products (203 us with each P.V operand pair built by two moves, a
// serial maximum chain and per-lane load offsets for every tile).
template <int DT, int ODT, int FA_QB, int FA_NW>
__global__ __launch_bounds__(64 * FA_NW, FA_NW == 8 ? 4 : 2) void fa_prefill_kernel(PrefillParams p) {
  constexpr int FA_QW = 16 * FA_QB;     // queries per wave
  constexpr int FA_BQ = FA_NW * FA_QW;  // queries per workgroup
  constexpr int FA_LW = FA_BK / 4 / FA_NW;  // K (or V) loads per wave and tile
  // 1 KB aligned: the operand reads form their addresses by exclusive-or
  __shared__ __attribute__((aligned(1024))) uint8_t sK[2][FA_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t sV[2][FA_TILE_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, g = lane >> 4;
  // Work item of this workgroup. Workgroups go to the 8 XCDs round-robin by linear id L (XCD
  // L % 8, in order of L on each), so items are handed out by L in longest-first order of
  // causal work: units (query block, b, KV head) from the last query block down, unit
  // c + 8j to XCD c, each unit's query heads consecutive on it (they read the same K and V
  // tiles, from that XCD's L2). Every XCD then gets the same mix of query blocks, each
  // longest first. (The grid's own order gave XCD k the query blocks k, k+8, ... only: 2.4x
  // the work on XCD 7 as on XCD 0 at 16 blocks.) When the units do not divide among the
  // XCDs the items go out by L in the same longest-first order, query heads spread.
  int b, h, qblk;
  {
    const int nx = gridDim.x, ny = gridDim.y, nz = gridDim.z;
    const int L = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
    const int grp = p.Hq / p.Hkv;       // query heads per KV head
    const int units = nx * nz * p.Hkv;  // (query block, b, KV head)
    if (units % 8 == 0) {
      const int xcd = L & 7, rank = L >> 3;
      const int u = xcd + 8 * (rank / grp);
      const int per = nz * p.Hkv;  // units per query block
      qblk = nx - 1 - u / per;
      b = (u % per) / p.Hkv;
      h = ((u % per) % p.Hkv) * grp + rank % grp;
    } else {
      const int per = ny * nz;  // items per query block
      qblk = nx - 1 - L / per;
      h = (L % per) % ny;
      b = (L % per) / ny;
    }
  }
  const int kvh = h / (p.Hq / p.Hkv);
  const int q0 = qblk * FA_BQ;
  const int wq0 = q0 + FA_QW * wave;  // the wave's first query
  // this lane's query in block qb (B operand column, output row)
  auto qrow = [&](int qb) { return wq0 + 16 * qb + n; };

  // Q^T operands: lane (query n of block qb, k-group g) holds dims 32s + 8g .. +8
  dkv_u32x4 qop[FA_QB][4];
#pragma unroll
  for (int qb = 0; qb < FA_QB; ++qb) {
    const uint16_t* qp = p.q + (long long)b * p.q_sb + (long long)h * p.q_sh +
                         (long long)min(qrow(qb), p.Sq - 1) * p.q_ss + 8 * g;
#pragma unroll
    for (int s = 0; s < 4; ++s) qop[qb][s] = *(const dkv_u32x4*)(qp + 32 * s);
  }

  // keys this workgroup needs: causal limit of its last query; the wave's own limit
  const int q_last_pos = p.q_offset + min(q0 + FA_BQ, p.Sq) - 1;
  const int k_end = p.causal ? min(p.Sk, q_last_pos + 1) : p.Sk;
  const int n_tiles = (k_end + FA_BK - 1) / FA_BK;
  // keys before ks are masked (a left-padded row's padding); tiles wholly before it are skipped
  const int ks = p.kstart ? min(max(p.kstart[b], 0), p.Sk) : 0;
  const int t0 = ks / FA_BK;
  const int wave_k_end =
      p.causal ? min(k_end, p.q_offset + min(wq0 + FA_QW, p.Sq)) : k_end;  // <= k_end

  const __amdgpu_buffer_rsrc_t rk = dkv_make_rsrc(p.k, p.k_bytes);
  const __amdgpu_buffer_rsrc_t rv = dkv_make_rsrc(p.v, p.v_bytes);
  const long long kbase = (long long)b * p.k_sb + (long long)kvh * p.k_sh;
  const long long vbase = (long long)b * p.v_sb + (long long)kvh * p.v_sh;
  // tile loads: wave w, instruction c stores keys 64 / NW * w + 4c + l/16, LDS chunk position
  // l%16, which holds the key's 16-byte dims chunk (l%16) ^ (key % 16). A tile inside the key range
  // moves the lanes' offsets by a scalar; in the last one each lane's key is checked.
  // (Key 4c + l/16's chunk is key l/16's with 4c added to the exclusive-or.)
  const int kk0 = FA_BK / FA_NW * wave + (lane >> 4);
  const uint32_t chunk0 = 16u * ((lane & 15) ^ (kk0 & 15));
  const uint32_t ko = (uint32_t)((kbase + (long long)kk0 * p.k_ss) * 2);
  const uint32_t vo = (uint32_t)((vbase + (long long)kk0 * p.v_ss) * 2);
  auto issue = [&](const __amdgpu_buffer_rsrc_t& rs, uint32_t row, long long ss, uint8_t* buf,
                   int t) {
    const uint32_t step = (uint32_t)ss * 2;  // bytes per key
    const uint32_t dst = fa_lds_addr(buf) + FA_BK / FA_NW * wave * 256;
    const uint32_t toff = (uint32_t)t * FA_BK * step;
    if ((t + 1) * FA_BK <= k_end) {
#pragma unroll
      for (int c = 0; c < FA_LW; ++c)
        fa_lds_load16(rs, dst + 4 * c * 256, row + (chunk0 ^ (64u * c)), toff + 4 * c * step);
    } else {
#pragma unroll
      for (int c = 0; c < FA_LW; ++c) {
        const int key = t * FA_BK + kk0 + 4 * c;
        fa_lds_load16(rs, dst + 4 * c * 256,
                      key < k_end ? row + (chunk0 ^ (64u * c)) + toff + 4 * c * step : 0x7ffffff0u,
                      0u);
      }
    }
  };

  dkv_f32x4 acc[FA_QB][8];
#pragma unroll
  for (int qb = 0; qb < FA_QB; ++qb)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[qb][i] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
  // running maxima (log2 units) and sums per query block; a maximum is only raised when the
  // tile's exceeds it by more than FA_RESCALE, so P may reach 2^FA_RESCALE
  float m_run[FA_QB], l_run[FA_QB];
#pragma unroll
  for (int qb = 0; qb < FA_QB; ++qb) {
    m_run[qb] = -1.0e30f;
    l_run[qb] = 0.f;
  }

  // S^T = K Q^T of key block kb: A = K rows (lane: key 16kb + n, dims 32s + 8g .. +8), B = Q^T of
  // block qb; lane (query n, g) then holds keys 16kb + 4g + u, unscaled (see the maxima below)
  const uint32_t krd = n * 256 + 16 * (g ^ n);  // + 4096 * kb, dims chunk 4s + g: ^ 64 * s
  typedef __attribute__((address_space(3))) dkv_u32x4 lds_u32x4;
  auto qk = [&](uint32_t kt, int kb, dkv_f32x4(&z)[FA_QB][4]) {
#pragma unroll
    for (int qb = 0; qb < FA_QB; ++qb) z[qb][kb] = dkv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const dkv_u32x4 a = *(const lds_u32x4*)(((kt + krd) ^ (64 * s)) + 4096 * kb);
#pragma unroll
      for (int qb = 0; qb < FA_QB; ++qb) z[qb][kb] = mfma32<DT>(a, qop[qb][s], z[qb][kb]);
    }
  };

  // transposed V reads: lane L = 4i + q of each 16-lane group reads key 16kb + 4g + i, dims
  // 16db + 4q .. +3 (8 bytes; ^ 32 * db, + 4096 * kb); lane i then holds dim 16db + i of keys
  // 4g .. 4g+3
  const uint32_t vrd = (4 * g + (n >> 2)) * 256 + 16 * (((n & 3) >> 1) ^ (4 * g + (n >> 2))) + 8 * (n & 1);
  typedef __attribute__((address_space(3))) dkv_i16x4 lds_i16x4;

  if (t0 < n_tiles) {
    issue(rk, ko, p.k_ss, sK[t0 & 1], t0);
    issue(rv, vo, p.v_ss, sV[t0 & 1], t0);
  }
  for (int t = t0; t < n_tiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // tile t is in LDS for every wave; tile t-1's buffer is free
    if (t + 1 < n_tiles) {
      issue(rk, ko, p.k_ss, sK[(t + 1) & 1], t + 1);
      issue(rv, vo, p.v_ss, sV[(t + 1) & 1], t + 1);
    }
    const int key0 = t * FA_BK;
    if (key0 >= wave_k_end) continue;  // every key of the tile is past the wave's queries
    const uint32_t kt = fa_lds_addr(sK[t & 1]);
    const uint32_t vt = fa_lds_addr(sV[t & 1]) + vrd;
    dkv_f32x4 z[FA_QB][4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) qk(kt, kb, z);
    if (key0 + FA_BK > k_end || key0 < ks || (p.causal && key0 + FA_BK - 1 > p.q_offset + wq0)) {
#pragma unroll
      for (int qb = 0; qb < FA_QB; ++qb) {
        const int my_pos = p.q_offset + qrow(qb);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int key = key0 + 16 * kb + 4 * g + u;
            if (key >= k_end || key < ks || (p.causal && key > my_pos)) z[qb][kb][u] = -INFINITY;
          }
      }
    }
    // V operands of key blocks 0 and 1: read ahead of the softmax
    dkv_u32x2 vx[8][2];
    auto vread = [&](int j, int db) {
      const uint32_t src = (vt ^ (32 * db)) + 8192 * j;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        vx[db][kk] = __builtin_bit_cast(
            dkv_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(src + 4096 * kk)));
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int db = 0; db < 8; ++db) vread(0, db);
    __builtin_amdgcn_sched_barrier(0);
    float tmax[FA_QB];
#pragma unroll
    for (int qb = 0; qb < FA_QB; ++qb) {
      float m[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        m[kb] = fa_max3(fa_max3(z[qb][kb][0], z[qb][kb][1], z[qb][kb][2]), z[qb][kb][3],
                        z[qb][kb][3]);
      // the scale is applied to the tile's maximum and inside the exponent's fma (one VALU
      // per score less than scaling every score: 2-3% of the launch); it is positive (the
      // entry point checks), so the maximum commutes with it
      tmax[qb] = fa_max4(fa_max3(fa_max3(m[0], m[1], m[2]), m[3], m[3])) * p.scale_log2;
    }
    if (__ballot(tmax[0] > m_run[0] + FA_RESCALE || tmax[FA_QB - 1] > m_run[FA_QB - 1] + FA_RESCALE)) {
#pragma unroll
      for (int qb = 0; qb < FA_QB; ++qb) {
        const float m_new = fa_max(m_run[qb], tmax[qb]);
        const float alpha = __builtin_amdgcn_exp2f(m_run[qb] - m_new);
        m_run[qb] = m_new;
        l_run[qb] *= alpha;
        // acc rows are dims, columns queries: lane (query n, g) holds dims 16db + 4g + u of
        // query n, so its rescale factor is its own alpha
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[qb][i][u] *= alpha;
      }
    }

    // P of key blocks 2j and 2j + 1, hi and lo parts: the B operands of P.V pair key block 2j's
    // keys 4g .. 4g+3 in k = 8g .. 8g+3 with key block 2j + 1's in k = 8g+4 .. 8g+7
    dkv_u32x4 bh[2][FA_QB], bl[2][FA_QB];
    auto probs = [&](int j, int kk, int qb) {
      float pu[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        pu[u] = __builtin_amdgcn_exp2f(
            __builtin_fmaf(z[qb][2 * j + kk][u], p.scale_log2, -m_run[qb]));
        l_run[qb] += pu[u];
      }
      dkv_u32x2 ph, pl;
      split_hi_lo<DT>(pu, ph, pl);
      bh[j][qb][2 * kk] = ph.x;
      bh[j][qb][2 * kk + 1] = ph.y;
      bl[j][qb][2 * kk] = pl.x;
      bl[j][qb][2 * kk + 1] = pl.y;
    };
#pragma unroll
    for (int i = 0; i < 2 * FA_QB; ++i) probs(0, i & 1, i >> 1);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int db = 0; db < 8; ++db) {
        __builtin_amdgcn_sched_barrier(0);
        const dkv_u32x4 aop = {vx[db][0].x, vx[db][0].y, vx[db][1].x, vx[db][1].y};
        if (j == 0) vread(1, db);
#pragma unroll
        for (int qb = 0; qb < FA_QB; ++qb) acc[qb][db] = mfma32<DT>(aop, bh[j][qb], acc[qb][db]);
#pragma unroll
        for (int qb = 0; qb < FA_QB; ++qb) acc[qb][db] = mfma32<DT>(aop, bl[j][qb], acc[qb][db]);
        if (j == 0 && db % (4 / FA_QB) == 4 / FA_QB - 1) probs(1, db / (4 / FA_QB) % 2, db / (8 / FA_QB));
      }
    }
  }

#pragma unroll
  for (int qb = 0; qb < FA_QB; ++qb) {
    // l over each tile's 64 keys sits in the lane's 16 keys x 4 lanes of the query
    float l = l_run[qb];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const int qr = qrow(qb);
    if (qr < p.Sq) {
      // a query with no key to attend (a padding position before the row's first key) gets 0
      const float inv = l > 0.f ? 1.f / l : 0.f;
      const long long ob = (long long)b * p.o_sb + (long long)h * p.o_sh + (long long)qr * p.o_ss;
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          dkv_store_f32<ODT>(p.out, ob + 16 * db + 4 * g + u, acc[qb][db][u] * inv);
    }
  }
}

template <int DT, int ODT, int QB, int NW>
void launch_prefill_shape(const PrefillParams& p, hipStream_t st) {
  constexpr int BQ = 16 * QB * NW;
  hipLaunchKernelGGL((fa_prefill_kernel<DT, ODT, QB, NW>),
                     dim3((unsigned)((p.Sq + BQ - 1) / BQ), (unsigned)p.Hq, (unsigned)p.B),
                     dim3(64 * NW), 0, st, p);
}
// The shape by the number of 128-query workgroups: more than two rounds of the 512 that fit the
// chip take two query blocks per wave (each K and V operand read from LDS serves two products);
// up to that, one block per wave and 8 waves (four waves per SIMD instead of two, while the LDS
// reads have room); one workgroup per CU or fewer take 64 queries, for twice the workgroups.
// Graph-replayed us, 2 blocks x 4 waves / 1 x 8 / 1 x 4 (32 query heads, 8 KV heads): 128
// workgroups (B = 1, S = 512) 19.4 / 17.2 / 14.2; 256 (B = 1, S = 1024) 33.4 / 29.6 / 26.7; 384
// (B = 3, S = 512) 23.5 / 21.4 / 21.8; 576 (B = 2, S = 1111) 44.0 / 42.0 / 46.9; 1024 (B = 4, S =
// 1024) 60.2 / 58.6 / 70.0; 1536 (B = 3, S = 2048) 142 / 146 / 171; 2048 (B = 4) 184 / 193 / 222.
template <int DT, int ODT>
void launch_prefill(const PrefillParams& p, hipStream_t st) {
  const long long wg = (long long)((p.Sq + 127) / 128) * p.Hq * p.B;
  if (wg > 1024)
    launch_prefill_shape<DT, ODT, 2, 4>(p, st);
  else if (wg > 256)
    launch_prefill_shape<DT, ODT, 1, 8>(p, st);
  else
    launch_prefill_shape<DT, ODT, 1, 4>(p, st);
}

// In-place rotate-half RoPE on dense rows x[r][s][d] (d < 128): position pos0 + s, angle
// float(pos) * inv_freq_i in fp32, the rotation in fp32, the result rounded to the dtype.
template <int DT>
__global__ __launch_bounds__(256) void rope_dense_kernel(uint16_t* __restrict__ x, long long r_ld,
                                                         long long s_ld, int rows, int S, int pos0,
                                                         float log_theta) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long total = (long long)rows * S * 64;
  if (idx >= total) return;
  const int i = (int)(idx % 64);
  const long long rs = idx / 64;
  const int s = (int)(rs % S);
  const long long r = rs / S;
  dkv_rope_pair<DT>(x + r * r_ld + (long long)s * s_ld, i, pos0 + s, log_theta);
}

// In-place rotate-half RoPE of x (B, H, S, 128) with given cos / sin tables (B, S, 128) in the
// dtype, rounded as the reference's apply_rotary_pos_emb_ computes (x * cos) + (rotate_half(x)
// * sin) in the dtype (compressed_attention.py:18-22): each product rounded, then their sum.
template <int DT>
__global__ __launch_bounds__(256) void rope_apply_kernel(uint16_t* __restrict__ x, long long x_sb,
                                                         long long x_sh, long long x_ss,
                                                         const uint16_t* __restrict__ cs,
                                                         const uint16_t* __restrict__ sn,
                                                         long long c_sb, long long c_ss, int B,
                                                         int H, int S) {
  // no contraction: for fp16 the compiler narrows the products and the sum to half arithmetic
  // and would fuse them into one fma, skipping the product's rounding
#pragma clang fp contract(off)
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long total = (long long)B * H * S * 64;
  if (idx >= total) return;
  const int i = (int)(idx % 64);
  long long r = idx / 64;
  const int s = (int)(r % S);
  r /= S;
  const int h = (int)(r % H);
  const int b = (int)(r / H);
  uint16_t* xr = x + (long long)b * x_sb + (long long)h * x_sh + (long long)s * x_ss;
  const long long co = (long long)b * c_sb + (long long)s * c_ss;
  const float x1 = dkv_load_f32<DT>(xr, i), x2 = dkv_load_f32<DT>(xr, i + 64);
  const float c1 = dkv_load_f32<DT>(cs, co + i), c2 = dkv_load_f32<DT>(cs, co + i + 64);
  const float s1 = dkv_load_f32<DT>(sn, co + i), s2 = dkv_load_f32<DT>(sn, co + i + 64);
  const float o1 = dkv_round_to<DT>(x1 * c1) + dkv_round_to<DT>(-x2 * s1);
  const float o2 = dkv_round_to<DT>(x2 * c2) + dkv_round_to<DT>(x1 * s2);
  dkv_store_f32<DT>(xr, i, o1);
  dkv_store_f32<DT>(xr, i + 64, o2);
}

}  // namespace

extern "C" int dkv_rope_dense(void* stream, int dtype, void* x, long long row_ld, long long tok_ld,
                              int rows, int S, int pos0, float log_theta) {
  if (dtype != DKV_F16 && dtype != DKV_BF16) return DKV_E_UNSUPPORTED;
  if (rows < 0 || S < 0) return DKV_E_ARG;
  if (rows == 0 || S == 0) return DKV_OK;
  if (!x) return DKV_E_ARG;
  const long long total = (long long)rows * S * 64;
  const dim3 grid((unsigned)((total + 255) / 256));
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DKV_BF16)
    hipLaunchKernelGGL(rope_dense_kernel<DKV_BF16>, grid, dim3(256), 0, st, (uint16_t*)x, row_ld,
                       tok_ld, rows, S, pos0, log_theta);
  else
    hipLaunchKernelGGL(rope_dense_kernel<DKV_F16>, grid, dim3(256), 0, st, (uint16_t*)x, row_ld,
                       tok_ld, rows, S, pos0, log_theta);
  DKV_HIP_CHECK_LAUNCH();
  return DKV_OK;
}

extern "C" int dkv_rope_apply(void* stream, int dtype, void* x, long long x_sb, long long x_sh,
                              long long x_ss, const void* cos, const void* sin, long long cs_sb,
                              long long cs_ss, int B, int H, int S) {
  if (dtype != DKV_F16 && dtype != DKV_BF16) return DKV_E_UNSUPPORTED;
  if (B < 0 || H < 0 || S < 0 || cs_sb < 0 || cs_ss < 0) return DKV_E_ARG;
  const long long total = (long long)B * H * S * 64;
  if (total == 0) return DKV_OK;
  if (!x || !cos || !sin) return DKV_E_ARG;
  const dim3 grid((unsigned)((total + 255) / 256));
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DKV_BF16)
    hipLaunchKernelGGL(rope_apply_kernel<DKV_BF16>, grid, dim3(256), 0, st, (uint16_t*)x, x_sb,
                       x_sh, x_ss, (const uint16_t*)cos, (const uint16_t*)sin, cs_sb, cs_ss, B, H,
                       S);
  else
    hipLaunchKernelGGL(rope_apply_kernel<DKV_F16>, grid, dim3(256), 0, st, (uint16_t*)x, x_sb,
                       x_sh, x_ss, (const uint16_t*)cos, (const uint16_t*)sin, cs_sb, cs_ss, B, H,
                       S);
  DKV_HIP_CHECK_LAUNCH();
  return DKV_OK;
}

extern "C" int dkv_prefill_attention(void* stream, int dtype, const void* q, long long q_sb,
                                     long long q_sh, long long q_ss, const void* k, long long k_sb,
                                     long long k_sh, long long k_ss, long long k_elems,
                                     const void* v, long long v_sb, long long v_sh, long long v_ss,
                                     long long v_elems, void* out, int out_dtype, long long o_sb,
                                     long long o_sh, long long o_ss, int B, int Hq, int Hkv,
                                     int Sq, int Sk, int Dh, int causal, float scale,
                                     const int* kstart) {
  // the kernel takes each tile's maximum before scaling: a positive, finite scale only
  if (!(scale > 0.f) || !(scale < INFINITY)) return DKV_E_UNSUPPORTED;
  if (dtype != DKV_F16 && dtype != DKV_BF16) return DKV_E_UNSUPPORTED;
  if (out_dtype != dtype && out_dtype != DKV_F32) return DKV_E_ARG;
  if (B < 0 || Hq <= 0 || Hkv <= 0 || Sq < 0 || Sk < 0) return DKV_E_ARG;
  if (Dh != FA_DH || Hq % Hkv != 0) return DKV_E_UNSUPPORTED;
  if (B == 0 || Sq == 0) return DKV_OK;
  if (!q || !k || !v || !out) return DKV_E_ARG;
  if (causal && Sk < Sq) return DKV_E_ARG;  // queries are the last Sq positions of the keys
  // 16-byte operand loads: unit dim stride, row strides in whole 16-byte units
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % 16 || q_ss % 8 || k_ss % 8 || v_ss % 8 ||
      k_sh % 8 || v_sh % 8 || k_sb % 8 || v_sb % 8 || q_sh % 8 || q_sb % 8)
    return DKV_E_UNSUPPORTED;
  if (k_elems * 2 >= (1LL << 31) || v_elems * 2 >= (1LL << 31)) return DKV_E_UNSUPPORTED;
  PrefillParams p;
  p.q = (const uint16_t*)q;
  p.k = (const uint16_t*)k;
  p.v = (const uint16_t*)v;
  p.out = out;
  p.q_sb = q_sb; p.q_sh = q_sh; p.q_ss = q_ss;
  p.k_sb = k_sb; p.k_sh = k_sh; p.k_ss = k_ss;
  p.v_sb = v_sb; p.v_sh = v_sh; p.v_ss = v_ss;
  p.o_sb = o_sb; p.o_sh = o_sh; p.o_ss = o_ss;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.Sq = Sq; p.Sk = Sk;
  p.q_offset = causal ? Sk - Sq : 0;
  p.causal = causal ? 1 : 0;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.k_bytes = (uint32_t)(k_elems * 2);
  p.v_bytes = (uint32_t)(v_elems * 2);
  p.kstart = kstart;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == DKV_BF16) {
    if (out_dtype == DKV_F32)
      launch_prefill<DKV_BF16, DKV_F32>(p, st);
    else
      launch_prefill<DKV_BF16, DKV_BF16>(p, st);
  } else {
    if (out_dtype == DKV_F32)
      launch_prefill<DKV_F16, DKV_F32>(p, st);
    else
      launch_prefill<DKV_F16, DKV_F16>(p, st);
  }
  DKV_HIP_CHECK_LAUNCH();
  return DKV_OK;
}
