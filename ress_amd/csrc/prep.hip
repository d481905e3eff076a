// Block preparation: mean pooling, per-block INT8 quantisation of Q and K, and
// packing of V into the attention kernel's MFMA-ready layout.
//
// Replaces, for the block-sparse path:
//   * predict_attention's avg_pool1d of Q (128) and K (64), ceil mode, a partial
//     block divided by its valid count  (reference src/ress/models/attention.py:82-100)
//   * block_mean_value's pool of V (64)                     (attention.py:103-109)
//   * km = key.mean(dim=-2) and per_block_int8(q, k - km)   (attention.py:231-233,
//     SpargeAttn quant_per_block with external/patches/spargeattn.patch:38-41:
//     Q is quantised with sm_scale = 1)
//
// One workgroup of four waves per (block, batch*head). Lane l owns dims 8*(l&7)..+7 of its
// wave's token lane l>>3; a wave reads eight tokens, 1 KiB, at a time.
#include "common.h"

// hi (and, if lo_dst is set, lo) codes of 8 values -> two 8-byte stores. Two terms ("split" INT8):
// x ~ scale*hi + (scale/254)*lo. hi is the per-block code; lo quantises the exact residual
// fmaf(-scale, hi, x) (|r| <= scale/2) with the scale scale/254, so |lo| <= 127. The codes are
// quant_i8's through the division-free quant_i8x8_rcp, with one branch for the eight: one per
// element made the code passes VALU-bound (k_quant_k, then one wave a block, 38.7 -> 28.9 us with
// both terms over 32 heads of 9,618 tokens, 26.7 -> 22.2 us with one over 16 heads of 21,984)
__device__ __forceinline__ void store_codes(const float (&x)[8], float scale, int8_t* hi_dst, int8_t* lo_dst) {
  int hi[8], lo[8];
  const float rc = scale != 0.0f ? 1.0f / scale : 0.0f;
  quant_i8x8_rcp(x, scale, rc, hi);
  *reinterpret_cast<uint2*>(hi_dst) = pack_i8x8(hi);
  if (lo_dst) {
    const float s2 = scale / 254.0f;
    const float rc2 = s2 != 0.0f ? 1.0f / s2 : 0.0f;
    float r[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) r[c] = fmaf(-scale, (float)hi[c], x[c]);
    quant_i8x8_rcp(r, s2, rc2, lo);
    *reinterpret_cast<uint2*>(lo_dst) = pack_i8x8(lo);
  }
}

// ----------------------------------------------------------------------------
// The Q and K/V passes: one workgroup of four waves per block. Lane group j of wave w reads rows
// 32 i + 8 w + j, every row of the block in flight at once, and keeps them in registers for what is
// done row by row (codes, fp16 rows, norms); copies in LDS serve what crosses rows. There thread
// (j, p), j = tid / 32, adds dims 2p and 2p+1 of rows 8 i + j in the order of i, and the eight j meet in
// the tree of SUM8x, so the sums are those of one wave whose lane group j walks rows 8 i + j.
// The order of that one wave is kept because the codes, maps and counts hang on its bits; as that
// one wave per block, which waits for a row's load before it takes the next and has all of a
// block's code arithmetic in line, the pass was bound by latency on small layers and by
// instruction issue with codes. Now HBM-bound from some 10,000 tokens (5.8 TB/s over what it reads
// and writes at 16 heads of 21,984 tokens). Times before and after, us:
//   k_prep_qkv, 16-bit operands: 16 heads of 1,374 tokens 14.7 -> 8.8, of 21,984 46.0 -> 38.9, of
//   43,968 91.0 -> 79.5; 24 heads of 21,861 82.0 -> 58.8;
//   k_prep_qkv, split codes, 32 heads of 9,618: 63.7 -> 41.1; k_prep_q, 16 heads of 21,984: 31.5 -> 20.6.
struct PrepLds {
  union {
    uint16_t q[128 * 64];  // Q: the block
    struct {
      uint16_t v[64 * 64];  // K/V: V rows, then the parts
      union {
        uint16_t k[64 * 64];  // K rows
        uint16_t vt[64 * VT_ROW];  // then V^T
      };
    };
    float part[3][8][64];  // SUM8x partial sums [quantity][j][dim]
  };
  float red[4];
};
static_assert(sizeof(float) * 3 * 8 * 64 <= 64 * 64 * 2, "the parts must fit over the V rows");

// this thread's two chains (dims 2p, 2p+1) over rows 8 i + j < cnt of a tile of 8 N rows
template <int N>
__device__ __forceinline__ void tile_sums(const uint16_t* tile, int j, int p, int cnt, float& a0, float& a1) {
  a0 = a1 = 0.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(tile + (8 * i + j) * 64 + 2 * p);
    const float s0 = a0 + bf16_lo(w), s1 = a1 + bf16_hi(w);
    a0 = 8 * i + j < cnt ? s0 : a0;
    a1 = 8 * i + j < cnt ? s1 : a1;
  }
}
// sum8_tree over the stored parts of one dim
__device__ __forceinline__ float part_tree(const float (&part)[8][64], int d) {
  return ((part[0][d] + part[1][d]) + (part[2][d] + part[3][d])) +
         ((part[4][d] + part[5][d]) + (part[6][d] + part[7][d]));
}

// Q blocks: kernel q-blocks 0..q_blk_p-1 hold patch queries, q_blk_p.. the
// special queries. Writes q_i8 [BH][q_blk_total][128][64], q_scale [BH][q_blk_total]
// and, for patch blocks, pooled_q [BH][q_blk_p][64].
__device__ __forceinline__ void prep_q_block(int qb, int bh, const uint16_t* __restrict__ q, const Strides& sq,
                                             const TokenMap& m, int q_blk_p, int q_blk_total,
                                             int8_t* __restrict__ q_i8, int8_t* __restrict__ q_lo,
                                             float* __restrict__ q_scale, float* __restrict__ pooled_q, PrepLds& lds) {
  const int tid = threadIdx.x, row0 = tid >> 3, dg = tid & 7;
  const bool special = qb >= q_blk_p;
  const int base = special ? (qb - q_blk_p) * 128 : qb * 128;
  const int cnt = min(128, (special ? m.T_s : m.T_p) - base);
  const uint16_t* src = q + bh_offset(bh, sq) + dg * 8;

  uint4 raw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // rows past the end: the block's first, then zero
    const int t = base + (32 * i + row0 < cnt ? 32 * i + row0 : 0);
    const int tok = special ? special_to_storage(t, m) : patch_to_storage(t, m);
    raw[i] = *reinterpret_cast<const uint4*>(src + (long long)tok * sq.t);
  }
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (32 * i + row0 >= cnt) raw[i] = make_uint4(0u, 0u, 0u, 0u);
    if (!special) *reinterpret_cast<uint4*>(lds.q + (32 * i + row0) * 64 + dg * 8) = raw[i];
    if (q_i8) {
      float x[8];
      unpack_bf16x8(raw[i], x);
#pragma unroll
      for (int c = 0; c < 8; ++c) amax = fmaxf(amax, fabsf(x[c]));
    }
  }
  if (q_i8) {
    amax = wave_max(amax);
    if ((tid & 63) == 0) lds.red[tid >> 6] = amax;
  }
  __syncthreads();
  if (q_i8) {  // null: pooling only (the 16-bit attention operands read Q directly)
    const float scale = fmaxf(fmaxf(lds.red[0], lds.red[1]), fmaxf(lds.red[2], lds.red[3])) / 127.0f;
    if (tid == 0) q_scale[(long long)bh * q_blk_total + qb] = scale;
    const long long off = (((long long)bh * q_blk_total + qb) * 128) * 64 + dg * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x[8];
      unpack_bf16x8(raw[i], x);
      const int r = (32 * i + row0) * 64;
      store_codes(x, scale, q_i8 + off + r, q_lo ? q_lo + off + r : nullptr);
    }
  }
  if (special) return;
  const int j = tid >> 5, p = tid & 31;
  float a0, a1;
  tile_sums<16>(lds.q, j, p, cnt, a0, a1);
  __syncthreads();  // the tile has been read
  *reinterpret_cast<float2*>(&lds.part[0][j][2 * p]) = make_float2(a0, a1);
  __syncthreads();
  if (tid < 64) pooled_q[((long long)bh * q_blk_p + qb) * 64 + tid] = part_tree(lds.part[0], tid) / (float)cnt;
}
__global__ __launch_bounds__(256) void k_prep_q(const uint16_t* __restrict__ q, Strides sq, TokenMap m,
                                                int q_blk_p, int q_blk_total, int8_t* __restrict__ q_i8,
                                                int8_t* __restrict__ q_lo, float* __restrict__ q_scale,
                                                float* __restrict__ pooled_q) {
  __shared__ __attribute__((aligned(16))) PrepLds lds;
  prep_q_block(blockIdx.x, blockIdx.y, q, sq, m, q_blk_p, q_blk_total, q_i8, q_lo, q_scale, pooled_q, lds);
}

// ----------------------------------------------------------------------------
// K/V blocks over the kernel key grid (patch keys then special keys).
//  ksum   [BH][kb_tot][64]  full-block K sums (SUM8x), for the key mean (or null)
//  k_pack [BH][kb_tot][64 keys][64] fp16 row-major K blocks (or null); a bf16 value is
//         exact in fp16 unless below 2^-14 in magnitude (the subnormal range) or above 65504
//  k_norm [BH][kb_tot]  the block's largest key norm sqrt(sum_d k_d^2) (or null): per key
//         an fmaf chain over each lane's 8 dims, the tree of the 8 lanes, sqrtf; then the max
//  pooled_k [BH][kb_pool][64]  K means of the scoring grid: the patch keys only (kb_pool =
//                              kb_p), or every key in kernel order (kb_pool = kb_tot; the
//                              sink-mass map, attention.py:78, 451-452)
//  pooled_v [BH][kb_pool][64]  V means over the same grid (ReSS's v_bar)
//  v_pack [BH][kb_tot][64 dims][64 keys]  bf16, keys permuted inside every group of
//         16 as 0-3,8-11,4-7,12-15 so that one 16-byte read per lane is an MFMA
//         operand; keys past the sequence end are zero.
__device__ __forceinline__ void prep_kv_block(int kb, int bh, const uint16_t* __restrict__ k,
                                              const uint16_t* __restrict__ v, const Strides& sk, const Strides& sv,
                                              const TokenMap& m, int Tk, int kb_tot, int kb_p,
                                              float* __restrict__ ksum, float* __restrict__ pooled_k,
                                              float* __restrict__ pooled_v, uint16_t* __restrict__ v_pack,
                                              uint16_t* __restrict__ k_pack, float* __restrict__ k_norm, int T_pool,
                                              PrepLds& lds) {
  const int tid = threadIdx.x, row0 = tid >> 3, dg = tid & 7;
  const int base = kb * 64;
  const int cnt = min(64, Tk - base);
  const int cnt_p = min(64, T_pool - base);  // <= 0 past the pooled keys
  const uint16_t* ksrc = k + bh_offset(bh, sk) + dg * 8;
  const uint16_t* vsrc = v + bh_offset(bh, sv) + dg * 8;
  const bool pools = kb < kb_p;

  uint4 rk[2], rv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // rows past the end: the block's first, then zero
    const int tok = key_to_storage(base + (32 * i + row0 < cnt ? 32 * i + row0 : 0), m);
    rk[i] = *reinterpret_cast<const uint4*>(ksrc + (long long)tok * sk.t);
    rv[i] = *reinterpret_cast<const uint4*>(vsrc + (long long)tok * sv.t);
  }
  float nmax = 0.0f;  // largest norm of the keys of this lane group
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int t = 32 * i + row0;
    if (t >= cnt) rk[i] = rv[i] = make_uint4(0u, 0u, 0u, 0u);
    *reinterpret_cast<uint4*>(lds.k + t * 64 + dg * 8) = rk[i];
    *reinterpret_cast<uint4*>(lds.v + t * 64 + dg * 8) = rv[i];
    float x[8];
    unpack_bf16x8(rk[i], x);
    if (k_pack) {  // row-major fp16 K block, zero past the sequence end
      uint4 h;
      h.x = f32x2_to_f16_bits(x[0], x[1]);
      h.y = f32x2_to_f16_bits(x[2], x[3]);
      h.z = f32x2_to_f16_bits(x[4], x[5]);
      h.w = f32x2_to_f16_bits(x[6], x[7]);
      *reinterpret_cast<uint4*>(k_pack + (((long long)bh * kb_tot + kb) * 64 + t) * 64 + dg * 8) = h;
    }
    if (k_norm) {  // key t's squared norm: the tree of the 8 dim-group lanes of its group
      float ss = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c) ss = fmaf(x[c], x[c], ss);
      // an element fp16 cannot hold (|x| >= 65520 rounds to inf): the key's norm is inf
      bool over = false;
#pragma unroll
      for (int c = 0; c < 8; ++c) over |= !(fabsf(x[c]) < 65520.0f);
      if (over) ss = __builtin_huge_valf();
      ss = ss + xor_lane_f<1>(ss);
      ss = ss + xor_lane_f<2>(ss);
      ss = ss + xor_lane_f<4>(ss);
      nmax = fmaxf(nmax, sqrtf(ss));
    }
  }
  if (k_norm) {
    nmax = fmaxf(nmax, xor_lane_f<8>(nmax));
    nmax = fmaxf(nmax, xor_lane_f<16>(nmax));
    nmax = fmaxf(nmax, xor_lane_f<32>(nmax));
    if ((tid & 63) == 0) lds.red[tid >> 6] = nmax;
  }
  __syncthreads();
  const int j = tid >> 5, p = tid & 31;
  float ka0 = 0.0f, ka1 = 0.0f, kp0 = 0.0f, kp1 = 0.0f, vp0 = 0.0f, vp1 = 0.0f;
  if (ksum) tile_sums<8>(lds.k, j, p, cnt, ka0, ka1);
  if (pools) {
    tile_sums<8>(lds.k, j, p, cnt_p, kp0, kp1);
    tile_sums<8>(lds.v, j, p, cnt_p, vp0, vp1);
  }
  uint32_t w[8];
  vt_read(lds.v, j, p, w);
  __syncthreads();  // the tiles have been read
  vt_write(lds.vt, j, p, w);
  if (ksum) *reinterpret_cast<float2*>(&lds.part[0][j][2 * p]) = make_float2(ka0, ka1);
  if (pools) {
    *reinterpret_cast<float2*>(&lds.part[1][j][2 * p]) = make_float2(kp0, kp1);
    *reinterpret_cast<float2*>(&lds.part[2][j][2 * p]) = make_float2(vp0, vp1);
  }
  __syncthreads();
  uint4* dst = reinterpret_cast<uint4*>(v_pack + ((long long)bh * kb_tot + kb) * 4096);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    dst[i * 256 + tid] = *reinterpret_cast<const uint4*>(lds.vt + (32 * i + row0) * VT_ROW + 8 * dg);
  const int d = tid & 63, part = tid >> 6;  // one wave per quantity
  if (part == 0 && ksum) ksum[((long long)bh * kb_tot + kb) * 64 + d] = part_tree(lds.part[0], d);
  if (part == 1 && pools) pooled_k[((long long)bh * kb_p + kb) * 64 + d] = part_tree(lds.part[1], d) / (float)cnt_p;
  if (part == 2 && pools) pooled_v[((long long)bh * kb_p + kb) * 64 + d] = part_tree(lds.part[2], d) / (float)cnt_p;
  if (part == 3 && k_norm && d == 0)
    k_norm[(long long)bh * kb_tot + kb] = fmaxf(fmaxf(lds.red[0], lds.red[1]), fmaxf(lds.red[2], lds.red[3]));
}
__global__ __launch_bounds__(256) void k_prep_kv(const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                                 Strides sk, Strides sv, TokenMap m, int Tk, int kb_tot, int kb_p,
                                                 float* __restrict__ ksum, float* __restrict__ pooled_k,
                                                 float* __restrict__ pooled_v, uint16_t* __restrict__ v_pack,
                                                 uint16_t* __restrict__ k_pack, float* __restrict__ k_norm) {
  __shared__ __attribute__((aligned(16))) PrepLds lds;
  prep_kv_block(blockIdx.x, blockIdx.y, k, v, sk, sv, m, Tk, kb_tot, kb_p, ksum, pooled_k, pooled_v, v_pack, k_pack,
                k_norm, m.T_p, lds);
}

// The layer's Q blocks and K/V blocks in one launch (they are independent): x < nqb is Q
// block x, the rest K/V block x - nqb. The K/V pools cover the first T_pool keys in kernel
// order (T_p: the patch keys; Tk: every key) in kb_pool blocks.
__global__ __launch_bounds__(256) void k_prep_qkv(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                  const uint16_t* __restrict__ v, Strides sq, Strides sk, Strides sv,
                                                  TokenMap m, int nqb, int q_blk_p, int q_blk_total, int Tk, int kb_tot,
                                                  int kb_p, int8_t* __restrict__ q_i8, int8_t* __restrict__ q_lo,
                                                  float* __restrict__ q_scale, float* __restrict__ pooled_q,
                                                  float* __restrict__ ksum, float* __restrict__ pooled_k,
                                                  float* __restrict__ pooled_v, uint16_t* __restrict__ v_pack,
                                                  uint16_t* __restrict__ k_pack, float* __restrict__ k_norm,
                                                  int T_pool) {
  __shared__ __attribute__((aligned(16))) PrepLds lds;
  if ((int)blockIdx.x < nqb)
    prep_q_block(blockIdx.x, blockIdx.y, q, sq, m, q_blk_p, q_blk_total, q_i8, q_lo, q_scale, pooled_q, lds);
  else
    prep_kv_block(blockIdx.x - nqb, blockIdx.y, k, v, sk, sv, m, Tk, kb_tot, kb_p, ksum, pooled_k, pooled_v, v_pack,
                  k_pack, k_norm, T_pool, lds);
}

// The block sums alone (ksum of prep_kv_block, the same SUM8x order): one wave per 64-key block,
// four per workgroup, every row of the block loaded before the sums. HBM-bound: 45 MB in 10.4 us.
__global__ __launch_bounds__(256) void k_key_sums(const uint16_t* __restrict__ k, Strides sk, int Tk, int nk,
                                                  float* __restrict__ ksum) {
  const int lane = threadIdx.x & 63, kb = blockIdx.x * 4 + (threadIdx.x >> 6), bh = blockIdx.y;
  if (kb >= nk) return;
  const int j = lane >> 3, dg = lane & 7, cnt = min(64, Tk - kb * 64);
  const uint16_t* src = k + bh_offset(bh, sk) + (long long)(kb * 64) * sk.t + dg * 8;
  uint4 r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    r[i] = make_uint4(0u, 0u, 0u, 0u);
    if (8 * i + j < cnt) r[i] = *reinterpret_cast<const uint4*>(src + (long long)(8 * i + j) * sk.t);
  }
  float a[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) a[c] = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float x[8];
    unpack_bf16x8(r[i], x);
    if (8 * i + j < cnt) {
#pragma unroll
      for (int c = 0; c < 8; ++c) a[c] = a[c] + x[c];
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) a[c] = sum8_tree(a[c]);
  if (j == 0) {
    float4* dst = reinterpret_cast<float4*>(ksum + ((long long)bh * nk + kb) * 64 + dg * 8);
    dst[0] = make_float4(a[0], a[1], a[2], a[3]);
    dst[1] = make_float4(a[4], a[5], a[6], a[7]);
  }
}

// key mean over all Tk keys: km[d] = SEQ-sum of the block sums / Tk, one workgroup a head. The
// sum is one chain of adds per dim, so what there is to gain is the loads' round trips: eight
// waves bring KM_CHUNK blocks at a time into LDS, the next chunk in flight while wave 0 adds one
// (151 blocks: 6.4 us with one wave loading 16 blocks at a time, 4.7 us so).
constexpr int KM_CHUNK = 128;
__global__ __launch_bounds__(512) void k_key_mean(const float* __restrict__ ksum, int kb_tot, int Tk,
                                                  float* __restrict__ km) {
  __shared__ float buf[2][KM_CHUNK * 64];
  const int bh = blockIdx.x, tid = threadIdx.x, d = tid & 63;
  const float* src = ksum + (long long)bh * kb_tot * 64;
  float nxt[KM_CHUNK / 8];  // this thread's dim of every eighth block (blocks past the end: the last)
  auto load = [&](int b0) {
#pragma unroll
    for (int i = 0; i < KM_CHUNK / 8; ++i) nxt[i] = src[min(b0 + (tid >> 6) + 8 * i, kb_tot - 1) * 64 + d];
  };
  load(0);
  float acc = 0.0f;
  for (int b0 = 0, p = 0; b0 < kb_tot; b0 += KM_CHUNK, p ^= 1) {
#pragma unroll
    for (int i = 0; i < KM_CHUNK / 8; ++i) buf[p][tid + 512 * i] = nxt[i];
    __syncthreads();  // also: wave 0 has added the chunk this buffer held before
    if (b0 + KM_CHUNK < kb_tot) load(b0 + KM_CHUNK);
    if (tid < 64) {
      const int n = min(KM_CHUNK, kb_tot - b0);
      int b = 0;
      for (; b + 16 <= n; b += 16) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = buf[p][(b + j) * 64 + d];
#pragma unroll
        for (int j = 0; j < 16; ++j) acc = acc + v[j];
      }
      for (; b < n; ++b) acc = acc + buf[p][b * 64 + d];
    }
  }
  if (tid < 64) km[(long long)bh * 64 + d] = acc / (float)Tk;
}

// K quantisation after smoothing: x = k - km (fp32), per 64-key block.
// k_i8 [BH][kb_tot][64 keys][64], k_scale [BH][kb_tot]. km may be null (no smoothing).
// Four waves a block, two rows a lane, both loads ahead (one wave a block: 28.6 us with both
// terms over 32 heads of 9,618 tokens and 22.9 us with one over 16 heads of 21,984; so 22.2 and 18.1).
__global__ __launch_bounds__(256) void k_quant_k(const uint16_t* __restrict__ k, Strides sk, TokenMap m, int Tk,
                                                 int kb_tot, const float* __restrict__ km, int8_t* __restrict__ k_i8,
                                                 int8_t* __restrict__ k_lo, float* __restrict__ k_scale) {
  __shared__ float red[4];
  const int kb = blockIdx.x, bh = blockIdx.y, tid = threadIdx.x;
  const int row0 = tid >> 3, dg = tid & 7;
  const int base = kb * 64;
  const int cnt = min(64, Tk - base);
  const uint16_t* src = k + bh_offset(bh, sk) + dg * 8;
  uint4 r[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)  // rows past the end: the block's first, masked below
    r[i] = *reinterpret_cast<const uint4*>(
        src + (long long)key_to_storage(base + (32 * i + row0 < cnt ? 32 * i + row0 : 0), m) * sk.t);
  float mean[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) mean[c] = km ? km[(long long)bh * 64 + dg * 8 + c] : 0.0f;
  float x[2][8];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    unpack_bf16x8(r[i], x[i]);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      x[i][c] = (32 * i + row0 < cnt) ? x[i][c] - mean[c] : 0.0f;
      amax = fmaxf(amax, fabsf(x[i][c]));
    }
  }
  amax = wave_max(amax);
  if ((tid & 63) == 0) red[tid >> 6] = amax;
  __syncthreads();
  const float scale = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])) / 127.0f;
  if (tid == 0) k_scale[(long long)bh * kb_tot + kb] = scale;
  const long long off = ((long long)bh * kb_tot + kb) * 4096 + dg * 8;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int at = (32 * i + row0) * 64;
    store_codes(x[i], scale, k_i8 + off + at, k_lo ? k_lo + off + at : nullptr);
  }
}

// ============================================================================
// C ABI
// ============================================================================
static bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

static TokenMap make_map(int frames, int P, int S, const int* perm = nullptr) {
  TokenMap m;
  m.P = P;
  m.S = S;
  m.HW = P - S;
  m.T_p = frames * (P - S);
  m.T_s = frames * S;
  m.perm = perm;
  return m;
}

// Fused preparation of one layer's Q/K/V for the ReSS forward (reference
// attention.py:398-491 + 226-233). Inputs are the backbone's bf16 Q/K/V in storage
// order with element strides (sB, sH, sT); D = 64 with unit stride.
//  * INT8 operands (q_i8 and k_i8 set): codes, scales, key mean; q_lo/k_lo (same
//    layouts as q_i8/k_i8) receive the split-INT8 residual codes, or are null.
//  * 16-bit operands (q_i8 and k_i8 null): the pools, v_pack, k_pack and, in k_scale,
//    each key block's largest key norm (k_norm of k_prep_kv) are written; q_lo,
//    q_scale, k_lo, ksum and km are unused (may be null).
// k_pack [BH][kb_tot][64 keys][64] fp16 (keys in kernel order, zero-padded) is
// written whenever it is non-null. patch_order: null, or HW = P-S int32 in device memory,
// the frame's patch tokens in the order blocks are formed (the Hilbert order of
// hilbert_permute), read in place; the same table must go to the attention call.
// pool_all: 0 pools K and V over the patch keys (kb_p blocks), 1 over every key in kernel
// order (kb_tot blocks: the sink-mass map of attention.py:78, 451-452 and its v_bar).
RESS_API int ress_prep_qkv(const void* q, const void* k, const void* v, int B, int H, int frames, int P, int S,
                           const int* patch_order, long long sqB, long long sqH, long long sqT, long long skB, long long skH, long long skT,
                           long long svB, long long svH, long long svT, void* q_i8, void* q_lo, void* q_scale,
                           void* pooled_q, void* k_i8, void* k_lo, void* k_scale, void* pooled_k, void* pooled_v,
                           void* v_pack, void* k_pack, void* ksum, void* km, int pool_all, hipStream_t stream) {
  RESS_REQUIRE(B > 0 && H > 0 && frames > 0 && P > S && S >= 0, "ress_prep_qkv: bad geometry B=%d H=%d F=%d P=%d S=%d",
               B, H, frames, P, S);
  RESS_REQUIRE(pool_all == 0 || pool_all == 1, "ress_prep_qkv: pool_all must be 0 or 1");
  RESS_REQUIRE(q && k && v && pooled_q && pooled_k && pooled_v && v_pack, "ress_prep_qkv: null pointer");
  const bool quant = q_i8 != nullptr;
  RESS_REQUIRE((q_i8 == nullptr) == (k_i8 == nullptr), "ress_prep_qkv: give both q_i8 and k_i8, or neither");
  RESS_REQUIRE(!quant || (q_scale && k_scale && ksum && km), "ress_prep_qkv: INT8 operands need q_scale, k_scale, ksum, km");
  RESS_REQUIRE(quant || (k_pack && k_scale), "ress_prep_qkv: 16-bit operands need k_pack and k_scale");
  RESS_REQUIRE(quant || (!q_lo && !k_lo), "ress_prep_qkv: q_lo/k_lo need the INT8 operands");
  RESS_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(v_pack) && aligned16(q_i8) && aligned16(k_i8) &&
                   aligned16(q_lo) && aligned16(k_lo) && aligned16(k_pack),
               "ress_prep_qkv: tensors must be 16-byte aligned");
  RESS_REQUIRE(sqT % 8 == 0 && skT % 8 == 0 && svT % 8 == 0 && sqH % 8 == 0 && skH % 8 == 0 && svH % 8 == 0 &&
                   sqB % 8 == 0 && skB % 8 == 0 && svB % 8 == 0,
               "ress_prep_qkv: strides must be multiples of 8 elements");
  TokenMap m = make_map(frames, P, S, patch_order);
  const int Tk = frames * P;
  const int BH = B * H;
  const int q_blk_p = cdiv(m.T_p, 128), q_blk_s = cdiv(m.T_s, 128);
  const int kb_tot = cdiv(Tk, 64), kb_p = cdiv(m.T_p, 64);
  Strides sq{sqB, sqH, sqT, H}, sk{skB, skH, skT, H}, sv{svB, svH, svT, H};
  // without codes only the patch blocks (the pooled ones) have Q work
  const int nqb = quant ? q_blk_p + q_blk_s : q_blk_p;
  hipLaunchKernelGGL(k_prep_qkv, dim3(nqb + kb_tot, BH), dim3(256), 0, stream, (const uint16_t*)q, (const uint16_t*)k,
                     (const uint16_t*)v, sq, sk, sv, m, nqb, q_blk_p, q_blk_p + q_blk_s, Tk, kb_tot,
                     pool_all ? kb_tot : kb_p,
                     (int8_t*)q_i8, (int8_t*)q_lo, (float*)q_scale, (float*)pooled_q,
                     (float*)(quant ? ksum : nullptr), (float*)pooled_k, (float*)pooled_v, (uint16_t*)v_pack,
                     (uint16_t*)k_pack, (float*)(quant ? nullptr : k_scale), pool_all ? Tk : m.T_p);
  RESS_LAUNCHED("k_prep_qkv");
  if (!quant) return 0;
  hipLaunchKernelGGL(k_key_mean, dim3(BH), dim3(512), 0, stream, (const float*)ksum, kb_tot, Tk, (float*)km);
  RESS_LAUNCHED("k_key_mean");
  hipLaunchKernelGGL(k_quant_k, dim3(kb_tot, BH), dim3(256), 0, stream, (const uint16_t*)k, sk, m, Tk, kb_tot,
                     (const float*)km, (int8_t*)k_i8, (int8_t*)k_lo, (float*)k_scale);
  RESS_LAUNCHED("k_quant_k");
  return 0;
}

// Mirror of SpargeAttn's per_block_int8(q, k) as the reference calls it
// (attention.py:232, with the patched Q scale of spargeattn.patch:38-41): plain
// sequences of Tq / Tk tokens, Q blocks of 128, K blocks of 64, optional key mean
// km [B*H][64] subtracted from K first (null = none). Outputs use the attention
// kernel's blocked layout: q_i8 [BH][ceil(Tq/128)][128][64],
// k_i8 [BH][ceil(Tk/64)][64][64], scales [BH][nblk].
RESS_API int ress_per_block_int8(const void* q, const void* k, const void* km, int B, int H, int Tq, int Tk,
                                 long long sqB, long long sqH, long long sqT, long long skB, long long skH,
                                 long long skT, void* q_i8, void* q_scale, void* k_i8, void* k_scale, void* pooled_q,
                                 hipStream_t stream) {
  RESS_REQUIRE(B > 0 && H > 0 && Tq > 0 && Tk > 0, "ress_per_block_int8: bad geometry");
  RESS_REQUIRE(q && k && q_i8 && q_scale && k_i8 && k_scale && pooled_q, "ress_per_block_int8: null pointer");
  RESS_REQUIRE(aligned16(q) && aligned16(k) && aligned16(q_i8) && aligned16(k_i8),
               "ress_per_block_int8: tensors must be 16-byte aligned");
  RESS_REQUIRE(sqT % 8 == 0 && skT % 8 == 0 && sqH % 8 == 0 && skH % 8 == 0 && sqB % 8 == 0 && skB % 8 == 0,
               "ress_per_block_int8: strides must be multiples of 8 elements");
  const int BH = B * H;
  TokenMap mq = make_map(1, Tq, 0), mk = make_map(1, Tk, 0);
  Strides sq{sqB, sqH, sqT, H}, sk{skB, skH, skT, H};
  const int nq = cdiv(Tq, 128), nk = cdiv(Tk, 64);
  hipLaunchKernelGGL(k_prep_q, dim3(nq, BH), dim3(256), 0, stream, (const uint16_t*)q, sq, mq, nq, nq, (int8_t*)q_i8,
                     (int8_t*)nullptr, (float*)q_scale, (float*)pooled_q);
  RESS_LAUNCHED("k_prep_q");
  hipLaunchKernelGGL(k_quant_k, dim3(nk, BH), dim3(256), 0, stream, (const uint16_t*)k, sk, mk, Tk, nk,
                     (const float*)km, (int8_t*)k_i8, (int8_t*)nullptr, (float*)k_scale);
  RESS_LAUNCHED("k_quant_k");
  return 0;
}

// Key mean of a plain (B,H,Tk,64) bf16 tensor (reference attention.py:231): km [B*H][64] fp32,
// with ksum [B*H][ceil(Tk/64)][64] fp32 as workspace; the orders of ress_prep_kv_plain, without
// its other outputs (31 us of packing for 16 heads of 21,984 keys, 10.4 us the sums alone).
RESS_API int ress_key_mean(const void* k, int B, int H, int Tk, long long skB, long long skH, long long skT, void* ksum,
                           void* km, hipStream_t stream) {
  RESS_REQUIRE(B > 0 && H > 0 && Tk > 0, "ress_key_mean: bad geometry");
  RESS_REQUIRE(k && ksum && km, "ress_key_mean: null pointer");
  RESS_REQUIRE(aligned16(k) && aligned16(ksum), "ress_key_mean: k and ksum must be 16-byte aligned");
  RESS_REQUIRE(skT % 8 == 0 && skH % 8 == 0 && skB % 8 == 0, "ress_key_mean: strides must be multiples of 8 elements");
  const int BH = B * H, nk = cdiv(Tk, 64);
  hipLaunchKernelGGL(k_key_sums, dim3(cdiv(nk, 4), BH), dim3(256), 0, stream, (const uint16_t*)k,
                     Strides{skB, skH, skT, H}, Tk, nk, (float*)ksum);
  RESS_LAUNCHED("k_key_sums");
  hipLaunchKernelGGL(k_key_mean, dim3(BH), dim3(512), 0, stream, (const float*)ksum, nk, Tk, (float*)km);
  RESS_LAUNCHED("k_key_mean");
  return 0;
}

// Key mean of a plain (B,H,Tk,64) bf16 tensor (reference attention.py:231), via the
// same SUM8x block sums and SEQ block order as the fused path. ksum is workspace
// [BH][ceil(Tk/64)][64] fp32; the pooled/packed outputs of the block pass go to
// pooled_k [BH][ceil(Tk/64)][64], pooled_v (same) and v_pack [BH][ceil(Tk/64)][4096] bf16.
RESS_API int ress_prep_kv_plain(const void* k, const void* v, int B, int H, int Tk, long long skB, long long skH,
                                long long skT, long long svB, long long svH, long long svT, void* ksum, void* km,
                                void* pooled_k, void* pooled_v, void* v_pack, hipStream_t stream) {
  RESS_REQUIRE(B > 0 && H > 0 && Tk > 0, "ress_prep_kv_plain: bad geometry");
  RESS_REQUIRE(k && v && ksum && km && pooled_k && pooled_v && v_pack, "ress_prep_kv_plain: null pointer");
  RESS_REQUIRE(aligned16(k) && aligned16(v) && aligned16(v_pack), "ress_prep_kv_plain: tensors must be 16-byte aligned");
  RESS_REQUIRE(skT % 8 == 0 && svT % 8 == 0 && skH % 8 == 0 && svH % 8 == 0 && skB % 8 == 0 && svB % 8 == 0,
               "ress_prep_kv_plain: strides must be multiples of 8 elements");
  const int BH = B * H, nk = cdiv(Tk, 64);
  TokenMap mk = make_map(1, Tk, 0);
  Strides sk{skB, skH, skT, H}, sv{svB, svH, svT, H};
  hipLaunchKernelGGL(k_prep_kv, dim3(nk, BH), dim3(256), 0, stream, (const uint16_t*)k, (const uint16_t*)v, sk, sv, mk,
                     Tk, nk, nk, (float*)ksum, (float*)pooled_k, (float*)pooled_v, (uint16_t*)v_pack,
                     (uint16_t*)nullptr, (float*)nullptr);
  RESS_LAUNCHED("k_prep_kv");
  hipLaunchKernelGGL(k_key_mean, dim3(BH), dim3(512), 0, stream, (const float*)ksum, nk, Tk, (float*)km);
  RESS_LAUNCHED("k_key_mean");
  return 0;
}
