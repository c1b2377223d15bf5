// Shared by the attention kernels (attention.hip, attention_f32.hip): arguments, mask reads, the
// transposing LDS read and the merge of key splits.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "wave_ops.h"

namespace mthip {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;

struct FlashArgs {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  int64_t qs[3], ks[3], vs[3], os[3];  // element strides: batch, head, sequence (last dim contiguous)
  int64_t H, Hk, Lq, Lk, E, Ev;
  int mask_kind, mask_dtype;
  const void* mask;
  int64_t ms[4];  // mask strides: b, h, q, k
  int causal;
  float scale;  // as given: zero and negative values multiply the scores like any other
  int cus;  // compute units of the device (launch-shape choices)
  // Key splits (flash kernel): workgroup z of gridDim.z takes keys [z * kv_chunk, (z+1) *
  // kv_chunk) and, when gridDim.z > 1, writes its unnormalised accumulator and (max, sum) to
  // part[z][b*H + h][q][pitch] (dims 0 .. DVB*32-1, then max at DVB*32 and sum at DVB*32 + 1,
  // fp16: log2 units) for flash_combine_kernel instead of the output.
  int kv_chunk;
  float* part;
  int part_pitch;
};

__device__ __forceinline__ float mask_value(const FlashArgs& a, int64_t b, int64_t h, int64_t q, int64_t k,
                                            float score) {
  if (a.mask_kind == MTHIP_MASK_NONE) return score;
  const int64_t off = b * a.ms[0] + h * a.ms[1] + q * a.ms[2] + k * a.ms[3];
  if (a.mask_kind == MTHIP_MASK_BOOL) return reinterpret_cast<const uint8_t*>(a.mask)[off] ? score : -INFINITY;
  if (a.mask_dtype == MTHIP_F16) return score + h2f_bits(reinterpret_cast<const uint16_t*>(a.mask)[off]);
  return score + reinterpret_cast<const float*>(a.mask)[off];
}

typedef short shortx4 __attribute__((ext_vector_type(4)));

// ds_read_b64_tr_b16: lane j of each 16-lane group receives halves [j%4] of the 8-byte rows read
// by lanes j/4, j/4+4, j/4+8 and j/4+12 of the group (p points into LDS).
__device__ __forceinline__ halfx4 tr_read16(const uint16_t* p) {
  return __builtin_bit_cast(halfx4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                        (__attribute__((address_space(3))) shortx4*)(const_cast<uint16_t*>(p))));
}

// Merges the key splits of the flash kernel: per query, m = max_z m_z, l = sum_z l_z 2^(m_z - m),
// o = (sum_z acc_z 2^(m_z - m)) / l (fp32: powers of e), narrowed once (a split that saw only masked keys has
// m_z = -inf and weight 0; with none left, l = 0 and 0/0 gives the reference's NaN).  One thread
// per 4 consecutive output dims of one query.
template <typename T>
__global__ __launch_bounds__(256) void flash_combine_kernel(const FlashArgs a, int splits, int dvb32) {
  const int groups = (int)((a.Ev + 3) / 4);
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (query, 4-dim group) of head blockIdx.y
  if (t >= a.Lq * groups) return;
  const int64_t bh = blockIdx.y, BH = gridDim.y;
  const int64_t q = t / groups;
  const int d0 = (int)(t - q * groups) * 4;
  float m = -INFINITY;
  for (int z = 0; z < splits; ++z) m = fmaxf(m, a.part[((z * BH + bh) * a.Lq + q) * a.part_pitch + dvb32]);
  float l = 0.0f, o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int z = 0; z < splits; ++z) {
    const float* row = a.part + ((z * BH + bh) * a.Lq + q) * a.part_pitch;
    const float2 ml = *reinterpret_cast<const float2*>(row + dvb32);
    // (fp32: maxima in natural units)
    const float d = sizeof(T) == 4 ? (ml.x - m) * kLog2e : ml.x - m;
    const float w = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(d);
    const float4 v = *reinterpret_cast<const float4*>(row + d0);
    l += ml.y * w;
    o[0] += v.x * w;
    o[1] += v.y * w;
    o[2] += v.z * w;
    o[3] += v.w * w;
  }
  const float inv_l = 1.0f / l;
  const int64_t b = bh / a.H, h = bh - b * a.H;
  T* O = reinterpret_cast<T*>(a.o) + b * a.os[0] + h * a.os[1] + q * a.os[2];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (d0 + j < a.Ev) Elem<T>::store(O, d0 + j, sizeof(T) == 4 ? o[j] / l : o[j] * inv_l);
}

// fp32 attention with head dims up to 160 (attention_f32.hip).
int launch_flash_f32(int device, FlashArgs& a, int64_t bh, hipStream_t s);

}  // namespace mthip
