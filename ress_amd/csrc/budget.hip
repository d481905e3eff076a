// Per-(head, query-block) key-block budgets.
//
// Replaces:
//   compute_baseline_num_to_select  (reference src/ress/models/attention.py:268-293)
//     cdf:  sort desc, cumsum, searchsorted(cdf, fp32(tau) + 1e-5, right=True)
//     sr:   topk = int(k_blk * (1 - sr)) (host double arithmetic), max(cdf_count, topk)
//   adjust_attention_selection      (reference src/ress/budget/_proportional.py:49-115)
//     HeSS cap-and-redistribute across heads per query-block column, fp32
//   the MIN_NUM_TO_SELECT floor     (attention.py:525)
//
// The CDF prefix sum is sequential (SEQ) over the descending-sorted row, so it
// does not depend on how ties are ordered.
#include "common.h"

// The CDF count of a row: the number of leading prefix sums (SEQ, over the descending row) up to
// the first one past thr, n if none is.
//
// Rows of up to 2,048 entries (k_cdf_count_wave): one wave per row, E entries a lane in
// registers as order keys. A bitonic sort with entry i in lane i / E, register i % E: strides
// below E stay in the lane, the others exchange keys across lanes (xor_lane). Then the one
// chain of adds, E values read from a lane at a time, which looks for the crossing inside the
// batch that has one. VALU-bound. In the LDS form below, whose every stage pays its index
// arithmetic and LDS round trip, 4,104 score rows of 340 took 62 us and 688 rows of 85 11.0 us;
// this form takes 21.4 and 6.0; 4,096 probability rows of 2,048 197 -> 60 us. The limit of 2,048
// is the 32 keys a lane that the chain's batch still holds in scalar registers.
// A positive NaN sorts above +inf and makes every prefix sum NaN: the row keeps all its entries.
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? k ^ 0x80000000u : ~k);
}
// the larger key first
__device__ __forceinline__ void key_order(uint32_t& a, uint32_t& b) {
  const uint32_t hi = max(a, b), lo = min(a, b);
  a = hi;
  b = lo;
}
template <int J, int E>
__device__ __forceinline__ void key_order_lanes(uint32_t (&key)[E], int lane) {
  const bool lower = (lane & J) == 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const uint32_t p = xor_lane<J>(key[e]);
    key[e] = lower ? max(key[e], p) : min(key[e], p);
  }
}
template <int E>
__global__ __launch_bounds__(256) void k_cdf_count_wave(const float* __restrict__ attn_cond, long long rows, int n,
                                                        float thr, int topk, int* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= rows) return;  // wave-uniform
  const float* src = attn_cond + row * n;
  uint32_t key[E];
#pragma unroll
  for (int e = 0; e < E; ++e)  // the order before the sort is of no account: coalesced loads
    key[e] = order_key(64 * e + lane < n ? src[64 * e + lane] : -__builtin_huge_valf());
  // sizes below E, directions alternating by the entry's bits
#pragma unroll
  for (int size = 2; size < E; size <<= 1)
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1)
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((e & stride) == 0) {
          if ((e & size) == 0) key_order(key[e], key[e | stride]);
          else key_order(key[e | stride], key[e]);
        }
  // size s * E: lanes with bit s sort the other way round, as complemented keys the same way
  uint32_t flip = 0u;
#pragma unroll 1
  for (int s = E == 1 ? 2 : 1; s <= 64; s <<= 1) {
    const uint32_t f = (lane & s) ? ~0u : 0u;
#pragma unroll
    for (int e = 0; e < E; ++e) key[e] ^= flip ^ f;
    flip = f;
    if (s >= 64) key_order_lanes<32>(key, lane);
    if (s >= 32) key_order_lanes<16>(key, lane);
    if (s >= 16) key_order_lanes<8>(key, lane);
    if (s >= 8) key_order_lanes<4>(key, lane);
    if (s >= 4) key_order_lanes<2>(key, lane);
    if (s >= 2) key_order_lanes<1>(key, lane);
#pragma unroll
    for (int stride = E >> 1; stride > 0; stride >>= 1)
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((e & stride) == 0) key_order(key[e], key[e | stride]);
  }
  // (at s = 64 no lane has the bit: flip is 0, the keys are the row's)
  float x[E];
#pragma unroll
  for (int e = 0; e < E; ++e) x[e] = key_value(key[e]);
  float c = 0.0f;
  int count = n;
  for (int l = 0; l * E < n; ++l) {  // padding past the row is -inf, which crosses nothing
    const float c0 = c;
    float top = -__builtin_huge_valf(), y[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      y[e] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[e]), l));
      c = c + y[e];
      top = fmaxf(top, c);
    }
    if (top > thr) {  // uniform: the batch's first prefix sum past thr
      c = c0;
      count = l * E;
      bool on = true;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        c = c + y[e];
        on = on && !(c > thr);
        count += on ? 1 : 0;
      }
      break;
    }
  }
  if (lane == 0) out[row] = count > topk ? count : topk;
}

// Longer rows: one workgroup of 256 threads per row, the sort in LDS. In a stage of stride <= 64
// a wave's 64 pairs lie in its own 128 entries, so between two such stages a wave's own LDS
// order is enough. Wave 0 runs the chain sixteen values at a time. 4,096 rows of 4,293: 885 us
// (1,126 with a barrier after every stage and one lane adding a value at a time).
__global__ __launch_bounds__(256) void k_cdf_count(const float* __restrict__ attn_cond, int n, int npow2,
                                                   float thr, int topk, int* __restrict__ out) {
  extern __shared__ float v[];  // npow2
  const long long row = blockIdx.x;
  const float* src = attn_cond + row * n;
  for (int i = threadIdx.x; i < npow2; i += 256) v[i] = i < n ? src[i] : -__builtin_huge_valf();
  __syncthreads();
  for (int size = 2; size <= npow2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < (npow2 >> 1); t += 256) {
        const int lo = 2 * t - (t & (stride - 1));
        const int hi = lo + stride;
        const bool desc = (lo & size) == 0;
        const float a = v[lo], b = v[hi];
        // descending sub-sequence when desc: larger first
        if ((a < b) == desc) {
          v[lo] = b;
          v[hi] = a;
        }
      }
      const int next = stride > 1 ? stride >> 1 : size;  // the next stage's stride
      if (stride > 64 || next > 64) {
        __syncthreads();
      } else {  // this wave's LDS accesses stay in program order
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    float c = 0.0f;
    int count = n;
    for (int i0 = 0; i0 < n; i0 += 16) {
      float x[16];  // past the row the padding's -inf, which crosses nothing
#pragma unroll
      for (int j = 0; j < 16; ++j) x[j] = v[min(i0 + j, npow2 - 1)];
      const float c0 = c;
      float top = -__builtin_huge_valf();
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        c = c + x[j];
        top = fmaxf(top, c);
      }
      if (top > thr) {  // uniform: the batch's first prefix sum past thr
        c = c0;
        count = n;
        for (int j = 0; j < 16 && i0 + j < n; ++j) {
          c = c + v[i0 + j];
          if (c > thr) {
            count = i0 + j;
            break;
          }
        }
        break;
      }
    }
    if (threadIdx.x == 0) out[row] = count > topk ? count : topk;
  }
}

__global__ __launch_bounds__(64) void k_fill_int(int* __restrict__ out, long long n, int value) {
  const long long i = (long long)blockIdx.x * 64 + threadIdx.x;
  if (i < n) out[i] = value;
}

#define RESS_MAX_HEADS 64

// SEQ sum of lanes 0..HB-1 (x is +0 on lanes past the heads, which leaves the sum unchanged)
template <int HB>
__device__ __forceinline__ float seq_sum_lanes(float x) {
  float acc = 0.0f;
#pragma unroll
  for (int h = 0; h < HB; ++h) acc = acc + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), h));
  return acc;
}

// One wave per (batch, q-block) column, lane h = head h. baseline/out are
// [B][H][q_blk] int32 (out may alias baseline). scores_norm [H] fp32 (already
// normalised, or null for the uniform budget). iters_out [B][q_blk] receives the
// number of cap-redistribute iterations, or -1 if max_iters was reached.
// HB >= H is a compile-time bound: the head sums are chains over lanes 0..HB-1 in order.
// Bound by the latency of those two chains and one division per iteration; with one thread
// per column every head's division was in the chain too (172 columns of 16 heads 9.3 us,
// 171 of 24 heads 25.3 us; this form 4.8 and 6.6).
template <int HB>
__global__ __launch_bounds__(256) void k_head_budget(const int* baseline, int B, int H, int q_blk,
                                                     const float* __restrict__ scores_norm, float one_minus_beta,
                                                     float beta, int max_val, int max_iters, int min_select,
                                                     int* out, int* __restrict__ iters_out) {
  const int col = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = threadIdx.x & 63;
  if (col >= B * q_blk) return;  // wave-uniform
  const int b = col / q_blk, qb = col - b * q_blk;
  const bool head = h < H;
  const long long at = ((long long)b * H + (head ? h : 0)) * q_blk + qb;
  const int bv = head ? baseline[at] : 0;
  if (scores_norm == nullptr) {
    if (head) out[at] = bv < min_select ? min_select : bv;
    if (iters_out && h == 0) iters_out[col] = 0;
    return;
  }
  const long long total = (long long)lane63_u64(wave_scan_sum_u64((unsigned long long)(long long)bv));
  const float total_f = (float)total;
  const float ideal = head ? scores_norm[h] * total_f : 0.0f;
  float adj = one_minus_beta * (float)bv + beta * ideal;
  const float maxv = (float)max_val;
  int it = 0;
  for (; it < max_iters; ++it) {
    const float d = adj - maxv;
    const float ex = head ? (d < 0.0f ? 0.0f : d) : 0.0f;  // clamp(min=0), NaN kept
    const float esum = seq_sum_lanes<HB>(ex);
    if (!__all(ex - ex == 0.0f) || !(esum > 0.0f)) break;  // uniform
    adj = adj > maxv ? maxv : adj;
    const float w = head ? adj * (adj < maxv ? 1.0f : 0.0f) : 0.0f;
    const float den = seq_sum_lanes<HB>(w) + 0x1.12e0bep-30f;  // + 1e-9
    adj = adj + (w / den) * esum;
  }
  if (iters_out && h == 0) iters_out[col] = it < max_iters ? it : -1;
  if (head) {
    const float a = adj > maxv ? maxv : adj;
    const int c = (int)floorf(a);
    out[at] = c < min_select ? min_select : c;
  }
}

// Baseline budget for rows [rows][n]: cdf_threshold < 0 disables the CDF cut;
// topk < 0 disables the sparse-ratio floor (at least one must be enabled).
RESS_API int ress_baseline_budget(const void* attn_cond, long long rows, int n, float cdf_threshold, int topk,
                                  void* out_counts, hipStream_t stream) {
  RESS_REQUIRE(rows >= 0 && n > 0, "ress_baseline_budget: bad geometry rows=%lld n=%d", rows, n);
  RESS_REQUIRE(cdf_threshold >= 0.0f || topk >= 0,
               "ress_baseline_budget: at least one of sparse_ratio/cdf_threshold required");
  RESS_REQUIRE(attn_cond && out_counts, "ress_baseline_budget: null pointer");
  if (rows == 0) return 0;
  if (cdf_threshold < 0.0f) {
    hipLaunchKernelGGL(k_fill_int, dim3((unsigned)((rows + 63) / 64)), dim3(64), 0, stream, (int*)out_counts, rows,
                       topk);
    RESS_LAUNCHED("k_fill_int");
    return 0;
  }
  int npow2 = 1;
  while (npow2 < n) npow2 <<= 1;
  RESS_REQUIRE(npow2 <= 16384, "ress_baseline_budget: row length %d exceeds 16384", n);
  const float thr = cdf_threshold + 0x1.4f8b58p-17f;  // fp32(tau) + 1e-5
  if (npow2 <= 64 * 32) {
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, (const float*)attn_cond, rows, n,
                         thr, topk, (int*)out_counts);
    };
    if (npow2 <= 64) go(k_cdf_count_wave<1>);
    else if (npow2 <= 128) go(k_cdf_count_wave<2>);
    else if (npow2 <= 256) go(k_cdf_count_wave<4>);
    else if (npow2 <= 512) go(k_cdf_count_wave<8>);
    else if (npow2 <= 1024) go(k_cdf_count_wave<16>);
    else go(k_cdf_count_wave<32>);
    RESS_LAUNCHED("k_cdf_count_wave");
    return 0;
  }
  hipLaunchKernelGGL(k_cdf_count, dim3((unsigned)rows), dim3(256), npow2 * sizeof(float), stream,
                     (const float*)attn_cond, n, npow2, thr, topk, (int*)out_counts);
  RESS_LAUNCHED("k_cdf_count");
  return 0;
}

// HeSS head reallocation + floor. scores_norm null = uniform budget (floor only).
RESS_API int ress_head_budget(const void* baseline, int B, int H, int q_blk, const void* scores_norm, double beta,
                              int max_val, int max_iters, int min_select, void* out_counts, void* iters_out,
                              hipStream_t stream) {
  RESS_REQUIRE(B > 0 && H > 0 && q_blk > 0, "ress_head_budget: bad geometry");
  RESS_REQUIRE(H <= RESS_MAX_HEADS, "ress_head_budget: H=%d exceeds %d", H, RESS_MAX_HEADS);
  RESS_REQUIRE(baseline && out_counts, "ress_head_budget: null pointer");
  RESS_REQUIRE(max_iters > 0, "ress_head_budget: max_iters must be positive");
  const int cols = B * q_blk;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((cols + 3) / 4), dim3(256), 0, stream, (const int*)baseline, B, H, q_blk,
                       (const float*)scores_norm, (float)(1.0 - beta), (float)beta, max_val, max_iters, min_select,
                       (int*)out_counts, (int*)iters_out);
  };
  if (H <= 8) go(k_head_budget<8>);
  else if (H <= 16) go(k_head_budget<16>);
  else if (H <= 32) go(k_head_budget<32>);
  else go(k_head_budget<RESS_MAX_HEADS>);
  RESS_LAUNCHED("k_head_budget");
  return 0;
}
