// Fused q/k normalisation and 2D rotary embedding of a QKV projection, writing q, k, v in
// the head-major layout the attention path reads.
//
// Replaces, for a VGGT-family attention module (reference src/ress/models/qkv.py:60-68,
// compute_patch_qkv before its patch/special split): qkv.reshape(B, N, 3, nh, hd)
// .permute(2, 0, 3, 1, 4), q_norm / k_norm (LayerNorm over the 64 head dims, affine), and
// the 2D RoPE of q and k (the first 32 head dims rotate with the row position, the last
// 32 with the column, rotate-half pairs (j, j+16) at frequencies base^(-2i/32)), with the
// same rounding points as the torch modules: LayerNorm output rounded to the activation
// dtype (bf16), the rotation in fp32 (x*cos + rot(x)*sin, no contraction), rounded again.
// cos/sin are the hardware functions (not the library's), so a small fraction of q/k
// values differ from the modules' by one bf16 rounding.
//
// One 256-thread workgroup per QKN_TOKENS consecutive tokens of a batch entry. The rotation's
// angles depend on the token and the dim alone, so the workgroup first puts the cosines and
// sines of its tokens (32 angles each, two halves of 16 frequencies) in LDS, one angle a thread.
// Then eight lanes take a head of a token (lane owns dims 8(t%8)..+7 of q, k and v, one 16-byte
// access each), the workgroup walking its tokens' heads 32 at a time with the next ones' loads
// in flight. LayerNorm statistics reduce over the eight lanes: pairs of dims in the lane, then
// xor 1, 2, 4; the rotation partner dims j +- 16 sit two lanes away (xor 2).
// HBM-bound (6 KiB read and written per 16-head token). Sixteen tokens per workgroup with every
// thread computing its own angles and loading 8 bytes when it needed them took 52.9 us for
// 13,740 tokens of 16 heads (48.8 alone, 3.5 TB/s) and 37.1 for 8,244; this form 30.5 (5.5 TB/s)
// and 21.6, the same bits.
#include "common.h"

namespace {

constexpr int QKN_TOKENS = 8;
constexpr int QKN_THREADS = 256;

// 16 bytes in one access, or in two of 8 where the buffers are only 8-byte aligned
template <bool A16>
__device__ __forceinline__ uint4 ld16(const uint16_t* p) {
  if constexpr (A16) {
    return *reinterpret_cast<const uint4*>(p);
  } else {
    const uint2 a = reinterpret_cast<const uint2*>(p)[0], b = reinterpret_cast<const uint2*>(p)[1];
    return make_uint4(a.x, a.y, b.x, b.y);
  }
}
template <bool A16>
__device__ __forceinline__ void st16(uint16_t* p, const uint4& v) {
  if constexpr (A16) {
    *reinterpret_cast<uint4*>(p) = v;
  } else {
    reinterpret_cast<uint2*>(p)[0] = make_uint2(v.x, v.y);
    reinterpret_cast<uint2*>(p)[1] = make_uint2(v.z, v.w);
  }
}
__device__ __forceinline__ uint4 pack_bf16x8(const float (&x)[8]) {
  return make_uint4(f32_to_bf16_bits(x[0]) | (f32_to_bf16_bits(x[1]) << 16),
                    f32_to_bf16_bits(x[2]) | (f32_to_bf16_bits(x[3]) << 16),
                    f32_to_bf16_bits(x[4]) | (f32_to_bf16_bits(x[5]) << 16),
                    f32_to_bf16_bits(x[6]) | (f32_to_bf16_bits(x[7]) << 16));
}
// the sum over a head's 64 values, 8 per lane: ((x0 + x1) + (x2 + x3)) per four, then pairs
__device__ __forceinline__ float sum64_of8(const float (&x)[8]) {
  float v = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
  v = v + xor_lane_f<1>(v);
  v = v + xor_lane_f<2>(v);
  v = v + xor_lane_f<4>(v);
  return v;
}

// LayerNorm of one head's 64 values (8 per lane) -> bf16-rounded fp32, in place
__device__ __forceinline__ void head_norm(float (&x)[8], const uint4& w, const uint4& b, float eps) {
  const float mean = sum64_of8(x) * (1.0f / 64.0f);
  float c2[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    x[u] = x[u] - mean;
    c2[u] = x[u] * x[u];
  }
  const float var = sum64_of8(c2) * (1.0f / 64.0f);
  const float rstd = 1.0f / sqrtf(var + eps);
  float gw[8], gb[8];
  unpack_bf16x8(w, gw);
  unpack_bf16x8(b, gb);
#pragma unroll
  for (int u = 0; u < 8; ++u) x[u] = round_bf16(x[u] * rstd * gw[u] + gb[u]);
}

// rotate-half RoPE of the lane's dims within their 32-dim half, given cos/sin of their angles;
// lo: dims below 16 of the half
__device__ __forceinline__ void rope8(float (&y)[8], bool lo, const float (&cs)[8], const float (&sn)[8]) {
  float o[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) o[u] = xor_lane_f<2>(y[u]);  // dims +- 16
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const float rot = lo ? -o[u] : o[u];
    const float a = y[u] * cs[u], bb = rot * sn[u];
    y[u] = round_bf16(a + bb);
  }
}

template <bool A16>
__global__ __launch_bounds__(QKN_THREADS) void k_qk_norm_rope(
    const uint16_t* __restrict__ qkv, int T, int nh, const uint16_t* __restrict__ qw, const uint16_t* __restrict__ qb,
    const uint16_t* __restrict__ kw, const uint16_t* __restrict__ kb, float eps, const long long* __restrict__ pos,
    float base, uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out) {
  __shared__ __align__(16) float cs_l[QKN_TOKENS][32], sn_l[QKN_TOKENS][32];  // [token][half * 16 + frequency]
  const int b = blockIdx.y, t = threadIdx.x, d0 = (t & 7) * 8;
  const int tok0 = blockIdx.x * QKN_TOKENS, ntok = min(QKN_TOKENS, T - tok0);
  const int C = nh * 64, items = ntok * nh;  // (token, head) pairs, eight lanes each
  const uint16_t* src = qkv + ((long long)b * T + tok0) * 3 * C + d0;
  uint4 rq, rk, rv;
  auto load = [&](int i) {
    const int tk = i / nh, h = i - tk * nh;
    const uint16_t* p = src + (long long)tk * 3 * C + h * 64;
    rq = ld16<A16>(p);
    rk = ld16<A16>(p + C);
    rv = ld16<A16>(p + 2 * C);
  };
  int i = t >> 3;
  if (i < items) load(i);
  const uint4 qw8 = ld16<false>(qw + d0), qb8 = ld16<false>(qb + d0), kw8 = ld16<false>(kw + d0),
              kb8 = ld16<false>(kb + d0);
  if (pos) {
    static_assert(QKN_TOKENS * 32 == QKN_THREADS, "one angle a thread");
    const int tk = t >> 5, half = (t >> 4) & 1;
    // frequency base^(-2i/32) of dim i of the half
    const float inv = 1.0f / powf(base, (float)(2 * (t & 15)) / 32.0f);
    if (tk < ntok) {
      const float p = (float)pos[((long long)b * T + tok0 + tk) * 2 + half];
      const float ang = p * inv;
      // the hardware sine/cosine for patch-grid positions (|angle| <= |p| <= 256 rad): their
      // absolute error (~1e-6 at a few tens of radians) moves about one output in a thousand
      // by one bf16 rounding against the library's cosf/sinf, at a fraction of the cost;
      // larger positions take the library functions
      const bool hw = fabsf(p) <= 256.0f;
      cs_l[tk][t & 31] = hw ? __cosf(ang) : cosf(ang);
      sn_l[tk][t & 31] = hw ? __sinf(ang) : sinf(ang);
    }
    __syncthreads();
  }
  const bool lo = (d0 & 31) < 16;
  const int f0 = (d0 >> 5) * 16 + (d0 & 15);  // the lane's first angle
  while (i < items) {
    const int tk = i / nh, h = i - tk * nh;
    float q[8], k[8];
    unpack_bf16x8(rq, q);
    unpack_bf16x8(rk, k);
    const uint4 v = rv;
    const int nxt = i + QKN_THREADS / 8;
    if (nxt < items) load(nxt);
    head_norm(q, qw8, qb8, eps);
    head_norm(k, kw8, kb8, eps);
    if (pos) {
      float cs[8], sn[8];
#pragma unroll
      for (int u = 0; u < 8; u += 4) {
        const float4 c4 = *reinterpret_cast<const float4*>(&cs_l[tk][f0 + u]);
        const float4 s4 = *reinterpret_cast<const float4*>(&sn_l[tk][f0 + u]);
        cs[u] = c4.x, cs[u + 1] = c4.y, cs[u + 2] = c4.z, cs[u + 3] = c4.w;
        sn[u] = s4.x, sn[u + 1] = s4.y, sn[u + 2] = s4.z, sn[u + 3] = s4.w;
      }
      rope8(q, lo, cs, sn);
      rope8(k, lo, cs, sn);
    }
    const long long o = (((long long)b * nh + h) * T + tok0 + tk) * 64 + d0;
    st16<A16>(q_out + o, pack_bf16x8(q));
    st16<A16>(k_out + o, pack_bf16x8(k));
    st16<A16>(v_out + o, v);
    i = nxt;
  }
}

}  // namespace

// qkv (B, T, 3*nh*64) bf16 contiguous (the qkv Linear's output); q_norm / k_norm affine
// weights and biases [64] bf16; pos (B, T, 2) int64 (row, column) or NULL (no rotation);
// outputs q, k, v (B, nh, T, 64) bf16 contiguous.
RESS_API int ress_qk_norm_rope(const void* qkv, int B, int T, int nh, const void* q_weight, const void* q_bias,
                               const void* k_weight, const void* k_bias, float eps, const void* pos, float rope_base,
                               void* q_out, void* k_out, void* v_out, hipStream_t stream) {
  RESS_REQUIRE(B > 0 && T >= 0 && nh > 0 && nh <= 64, "ress_qk_norm_rope: bad geometry B=%d T=%d nh=%d", B, T, nh);
  RESS_REQUIRE(qkv && q_weight && q_bias && k_weight && k_bias && q_out && k_out && v_out,
               "ress_qk_norm_rope: null pointer");
  RESS_REQUIRE(((uintptr_t)qkv & 7u) == 0 && ((uintptr_t)q_out & 7u) == 0 && ((uintptr_t)k_out & 7u) == 0 &&
                   ((uintptr_t)v_out & 7u) == 0 && ((uintptr_t)q_weight & 7u) == 0 && ((uintptr_t)q_bias & 7u) == 0 &&
                   ((uintptr_t)k_weight & 7u) == 0 && ((uintptr_t)k_bias & 7u) == 0,
               "ress_qk_norm_rope: buffers must be 8-byte aligned");
  if (T == 0) return 0;
  const bool a16 = (((uintptr_t)qkv | (uintptr_t)q_out | (uintptr_t)k_out | (uintptr_t)v_out) & 15u) == 0;
  hipLaunchKernelGGL(a16 ? k_qk_norm_rope<true> : k_qk_norm_rope<false>, dim3(cdiv(T, QKN_TOKENS), B),
                     dim3(QKN_THREADS), 0, stream, (const uint16_t*)qkv, T, nh, (const uint16_t*)q_weight, (const uint16_t*)q_bias, (const uint16_t*)k_weight,
                     (const uint16_t*)k_bias, eps, (const long long*)pos, rope_base, (uint16_t*)q_out,
                     (uint16_t*)k_out, (uint16_t*)v_out);
  RESS_LAUNCHED("k_qk_norm_rope");
  return 0;
}
