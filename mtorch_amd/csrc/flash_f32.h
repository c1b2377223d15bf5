// Flash attention for fp32 operands on the bf16 matrix cores, head dims up to 160.
//
// The layout is the fp16 kernel's (attention.hip): a wave owns 32 queries and computes S^T = K . Q^T
// per 32-key tile, so a lane holds one query's scores against 16 keys, softmax runs in registers, and the probabilities are the B operand of O^T += V^T . P^T as they stand (register r
// <-> key 8 (r / 4) + 4 (lane / 32) + r % 4).  Q, K, V and P are each cut into three bf16 parts
// (gemm_split.h) and both products are the six part products that matter: nothing is held in fewer
// than 24 significand bits (down to 2^-110, where bf16 runs out of exponent; see below).  Q's parts stay in registers; K and V are cut while they are staged in
// LDS, K as rows of three part blocks (an odd number of 16-byte chunks: a fragment read covers every
// bank), V as three row-major tiles read through the transposing LDS read.
//
// A workgroup is 4 waves: KG = 1 gives them 128 queries and one key tile per step, KG = 2 64 queries
// and two key tiles, each pair of waves with its own running softmax, merged through LDS at the end
// -- for grids that would leave SIMDs without a wave.
//
// 2x8 heads, 1024x1024, head dim 80: 56 us (5.4 GFLOP as 32 GFLOP of bf16 products, 580 TFLOP/s)
// against 2709 us of a wave per query; what bounds it is the alternation of the MFMA chains with the
// softmax and cutting VALU work at two waves per SIMD.
//
// Scores, masks and maxima stay in natural units and exp(s - m) is taken of their difference, as the
// row-wise kernel does: a score scaled by log2 e would be rounded once more and overflow earlier.  A
// score's a1b1 products are added last, on top of all its small ones, so that its error is that of one
// rounding per 16 dims.
//
// A query is computed again by its wave in plain fp32 (flash_row) where the parts do not do: its sums
// or outputs non-finite (infinities, NaNs, operands next to the fp32 maximum); Q with elements that
// lose bits (below 2^-110) or of 2^60 and more (K may then have lost bits that matter); an output that
// is not zero and below 2^-70 or 2^-106 of the largest |V| (bits that small probabilities lose), or zero
// while some V lost bits.  A fully masked row stays 0 / 0 = NaN.  One NaN key thus sends every query
// through flash_row, which is some 50 times slower.
#pragma once

#include "attention.h"
#include "gemm_split.h"

namespace mthip {
namespace {

// One query in plain fp32 over keys [kb, ke), the row-wise kernel's steps: the max, the sum and this lane's output dims lane + 64 j.
template <int VPL>
__device__ void flash_row(const FlashArgs& a, int64_t b, int64_t head, int64_t q, int kb, int ke,
                                                    float& m_out, float& l_out, float (&o)[VPL]) {
  const int lane = threadIdx.x & 63;
  const int64_t kvh = head / (a.H / a.Hk);
  const float* Q = reinterpret_cast<const float*>(a.q) + b * a.qs[0] + head * a.qs[1] + q * a.qs[2];
  const float* K = reinterpret_cast<const float*>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const float* V = reinterpret_cast<const float*>(a.v) + b * a.vs[0] + kvh * a.vs[1];
  float qv[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int d = lane + 64 * j;
    qv[j] = d < a.E ? Q[d] : 0.0f;
    o[j] = 0.0f;
  }
  float m = -INFINITY, l = 0.0f;
  for (int64_t key = kb; key < ke; ++key) {
    float part = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int d = lane + 64 * j;
      if (d < a.E) part += qv[j] * K[key * a.ks[2] + d];
    }
    part = wave_sum(part);
    float sc = part * a.scale;
    if (a.causal && key > q) sc = -INFINITY;
    sc = mask_value(a, b, head, q, key, sc);
    const float mn = fmaxf(m, sc), mu = mn == -INFINITY ? 0.0f : mn;
    const float alpha = expf(m - mu), p = expf(sc - mu);
    l = l * alpha + p;
    m = mn;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int d = lane + 64 * j;
      o[j] = o[j] * alpha + (d < a.Ev ? p * V[key * a.vs[2] + d] : 0.0f);
    }
  }
  m_out = m;
  l_out = l;
}

// DK: head dim padded to a multiple of 16; MASKED: a mask or causal masking may apply.
template <int DK, int KG, bool MASKED>
__global__ __launch_bounds__(256, DK <= 80 ? 2 : 1) void flash_fwd_f32_kernel(const FlashArgs a) {
  constexpr int NSTEP = DK / 16, DVB = (DK + 31) / 32;
  constexpr int QB = 4 / KG;                // query blocks (waves per key group)
  constexpr int BKV = 32 * KG;              // keys staged per step
  constexpr int KPITCH = 6 * DK + 16;       // bytes of a K row: three part blocks and a pad
  constexpr int VRP = DVB * 32 + 8;         // halves of a V row of one part
  constexpr int KT = 32 * KPITCH, VT = 3 * 32 * VRP * 2;  // bytes of one key tile
  constexpr int KCHR = DK / 8, VCHR = DVB * 4;            // 8-element chunks per row
  constexpr int KCH = (BKV * KCHR + 255) / 256, VCH = (BKV * VCHR + 255) / 256;
  constexpr int XCH = KG > 1 ? QB * 64 * 17 * 4 : 0;      // bytes of the merge buffer
  constexpr uint32_t kOob = 0x80000000u;
  __shared__ __align__(16) unsigned char smem[KG * (KT + VT) > XCH ? KG * (KT + VT) : XCH];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / QB, hh = lane >> 5, col = lane & 31;
  const int64_t bh = blockIdx.y;
  const int64_t b = bh / a.H, head = bh - b * a.H;
  const int64_t kvh = head / (a.H / a.Hk);
  const int64_t q = (int64_t)blockIdx.x * (32 * QB) + (wave % QB) * 32 + col;
  const bool qok = q < a.Lq;
  const int kb = (int)blockIdx.z * a.kv_chunk;
  const int Lk = min((int)a.Lk, kb + a.kv_chunk), E = (int)a.E, Ev = (int)a.Ev;
  const float* Q = reinterpret_cast<const float*>(a.q) + b * a.qs[0] + head * a.qs[1];
  const float* K = reinterpret_cast<const float*>(a.k) + b * a.ks[0] + kvh * a.ks[1];
  const float* V = reinterpret_cast<const float*>(a.v) + b * a.vs[0] + kvh * a.vs[1];

  // Q^T fragments (B operand of S^T): query q, dims 16 st + 8 hh + [0, 8).
  bf16x8 qf[NSTEP][3];
  uint32_t q_rest = 0;
  float q_max = 0.0f;
#pragma unroll
  for (int st = 0; st < NSTEP; ++st) {
    const int d0 = st * 16 + hh * 8;
    uint32_t p[4][3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = qok && d0 + 2 * e < E ? Q[q * a.qs[2] + d0 + 2 * e] : 0.0f;
      const float y = qok && d0 + 2 * e + 1 < E ? Q[q * a.qs[2] + d0 + 2 * e + 1] : 0.0f;
      split_pair(x, y, p[e], q_rest);
      q_max = fmaxf(q_max, fmaxf(fabsf(x), fabsf(y)));
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) qf[st][t] = __builtin_bit_cast(bf16x8, make_uint4(p[0][t], p[1][t], p[2][t], p[3][t]));
  }

  // (a mask of lanes at once: left to its use, the compiler holds Q's elements through the loop)
  const uint64_t q_bad = __builtin_amdgcn_ballot_w64((q_rest & 0xffffu) != 0 || q_max >= 0x1p60f);

  // Staging: thread chunk c covers key c / CHR and dims 8 (c % CHR) of the step.  Loads need only
  // 4-byte alignment; a chunk that crosses E (Ev) is cleared past it.
  const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)K, (short)0, (int)(((int64_t)(Lk > 0 ? Lk - 1 : 0) * a.ks[2] + E) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)V, (short)0, (int)(((int64_t)(Lk > 0 ? Lk - 1 : 0) * a.vs[2] + Ev) * 4), 0x00020000);
  float kr[KCH][8], vr[VCH][8];
  auto load8 = [&](const __amdgpu_buffer_rsrc_t& r, bool row_ok, uint32_t elem, int d0, int D, float (&x)[8]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint4 u = __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(row_ok && d0 + 4 * h < D ? (elem + 4 * h) * 4u : kOob), 0, 0));
      x[4 * h] = __uint_as_float(u.x);
      x[4 * h + 1] = __uint_as_float(u.y);
      x[4 * h + 2] = __uint_as_float(u.z);
      x[4 * h + 3] = __uint_as_float(u.w);
    }
  };
  auto fetch = [&](int kv0) {
#pragma unroll
    for (int i = 0; i < KCH; ++i) {
      const int c = tid + i * 256, key = kv0 + c / KCHR, d0 = (c % KCHR) * 8;
      load8(k_rsrc, c < BKV * KCHR && key < Lk, (uint32_t)(key * (int)a.ks[2] + d0), d0, E, kr[i]);
    }
#pragma unroll
    for (int i = 0; i < VCH; ++i) {
      const int c = tid + i * 256, key = kv0 + c / VCHR, d0 = (c % VCHR) * 8;
      load8(v_rsrc, c < BKV * VCHR && key < Lk, (uint32_t)(key * (int)a.vs[2] + d0), d0, Ev, vr[i]);
    }
  };
  uint32_t v_rest = 0;  // of the V elements this thread has cut: bits they lost, and the largest
  float v_max = 0.0f;
  auto cut8 = [&](auto is_v, float (&x)[8], int d0, int D, unsigned char* dst, int part_bytes) {
    if (D & 3) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = d0 + e < D ? x[e] : 0.0f;
    }
    uint32_t p[4][3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (decltype(is_v)::value) {
        v_max = abs_max_nan(abs_max_nan(v_max, x[2 * e]), x[2 * e + 1]);
        split_pair(x[2 * e], x[2 * e + 1], p[e], v_rest);
      } else {
        split_pair(x[2 * e], x[2 * e + 1], p[e]);
      }
    }
#pragma unroll
    for (int t = 0; t < 3; ++t)
      *reinterpret_cast<uint4*>(dst + t * part_bytes) = make_uint4(p[0][t], p[1][t], p[2][t], p[3][t]);
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < KCH; ++i) {
      const int c = tid + i * 256, key = c / KCHR, d0 = (c % KCHR) * 8;
      if (c < BKV * KCHR) cut8(std::false_type{}, kr[i], d0, E, smem + (key >> 5) * (KT + VT) + (key & 31) * KPITCH + d0 * 2, DK * 2);
    }
#pragma unroll
    for (int i = 0; i < VCH; ++i) {
      const int c = tid + i * 256, key = c / VCHR, d0 = (c % VCHR) * 8;
      if (c < BKV * VCHR)
        cut8(std::true_type{}, vr[i], d0, Ev, smem + (key >> 5) * (KT + VT) + KT + ((key & 31) * VRP + d0) * 2, 32 * VRP * 2);
    }
  };

  floatx16 acc[DVB];
#pragma unroll
  for (int i = 0; i < DVB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;
  constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
  const unsigned char* kt = smem + grp * (KT + VT) + col * KPITCH + hh * 16;
  // the lane's first half of the transposing read (see the fp16 kernel)
  const uint16_t* vt = reinterpret_cast<const uint16_t*>(smem + grp * (KT + VT) + KT) +
                       (hh * 4 + ((lane & 15) >> 2)) * VRP + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);

  fetch(kb);
  for (int kv = kb; kv < Lk; kv += BKV) {
    __syncthreads();  // every wave is done with the previous step
    stage();
    __syncthreads();
    if (kv + BKV < Lk) fetch(kv + BKV);
    const int kv0 = kv + 32 * grp;
    if (KG > 1 && kv0 >= Lk) continue;  // a key group past the last tile only keeps the barriers

    // the small part products of every step first, then the a1b1 on top of them
    floatx16 t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 0.0f;
#pragma unroll
    for (int st = 0; st < NSTEP; ++st) {
      bf16x8 kf[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) kf[p] = *reinterpret_cast<const bf16x8*>(kt + p * DK * 2 + st * 32);
#pragma unroll
      for (int p = 0; p < 5; ++p) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[PA[p]], qf[st][PB[p]], t, 0, 0, 0);
    }
    // (above five steps in two chains: no more roundings in a row than at head dim 80)
    constexpr int HALF = NSTEP > 5 ? NSTEP / 2 : NSTEP;
    floatx16 t2;
#pragma unroll
    for (int r = 0; r < 16; ++r) t2[r] = 0.0f;
#pragma unroll
    for (int st = 0; st < HALF; ++st) {
      t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(kt + st * 32), qf[st][0], t, 0, 0, 0);
      if constexpr (HALF < NSTEP)
        t2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(kt + (st + HALF) * 32),
                                                     qf[st + HALF][0], t2, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = (HALF < NSTEP ? t[r] + t2[r] : t[r]) * a.scale;
    float s[16], mx = -INFINITY;
    if (!MASKED && kv0 + 32 <= Lk) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = t[r];
        mx = fmaxf(mx, s[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = kv0 + 8 * (r >> 2) + 4 * hh + (r & 3);
        float v = t[r];
        if (key >= Lk) {
          v = -INFINITY;
        } else if constexpr (MASKED) {
          if (a.causal && key > q) v = -INFINITY;
          if (a.mask_kind != MTHIP_MASK_NONE && qok) {
            const int64_t off = b * a.ms[0] + head * a.ms[1] + q * a.ms[2] + key * a.ms[3];
            if (a.mask_kind == MTHIP_MASK_BOOL) {
              if (!reinterpret_cast<const uint8_t*>(a.mask)[off]) v = -INFINITY;
            } else {
              const float mv = a.mask_dtype == MTHIP_F16 ? h2f_bits(reinterpret_cast<const uint16_t*>(a.mask)[off])
                                                         : reinterpret_cast<const float*>(a.mask)[off];
              v += mv;
            }
          }
        }
        s[r] = v;
        mx = fmaxf(mx, v);
      }
    }
    mx = halves_max(mx);
    // lazy rescaling: the running max moves only when a score exceeds it by more than 5.5 (P <= 245)
    if (mx > m_run + 5.5f) {
      const float alpha = __builtin_amdgcn_exp2f((m_run - mx) * kLog2e);  // 0 when m_run = -inf
      l_run *= alpha;
#pragma unroll
      for (int i = 0; i < DVB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] *= alpha;
      m_run = mx;
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    float psum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f((s[r] - m_use) * kLog2e);
      psum += s[r];
    }
    l_run += halves_sum(psum);

    // O^T += V^T . P^T, two 16-key steps
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      uint32_t p[4][3];
#pragma unroll
      for (int e = 0; e < 4; ++e) split_pair(s[st * 8 + 2 * e], s[st * 8 + 2 * e + 1], p[e]);
      bf16x8 pf[3];
#pragma unroll
      for (int t3 = 0; t3 < 3; ++t3)
        pf[t3] = __builtin_bit_cast(bf16x8, make_uint4(p[0][t3], p[1][t3], p[2][t3], p[3][t3]));
#pragma unroll
      for (int i = 0; i < DVB; ++i) {
        bf16x8 vf[3];
#pragma unroll
        for (int t3 = 0; t3 < 3; ++t3) {
          const uint16_t* v0 = vt + t3 * 32 * VRP + st * 16 * VRP + i * 32;
          const halfx4 lo = tr_read16(v0), hi = tr_read16(v0 + 8 * VRP);
          const halfx8 v8 = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          vf[t3] = __builtin_bit_cast(bf16x8, v8);
        }
#pragma unroll
        for (int u = 0; u < 6; ++u) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[PA[u]], pf[PB[u]], acc[i], 0, 0, 0);
      }
    }
  }

  // what the V tiles of this workgroup held
  __shared__ float v_flags[4][2];
  {
    const float m = wave_reduce(v_max, [](float x, float y) { return abs_max_nan(x, y); });
    const bool r = __builtin_amdgcn_ballot_w64((v_rest & 0xffffu) != 0) != 0;
    if (lane == 0) {
      v_flags[wave][0] = m;
      v_flags[wave][1] = r ? 1.0f : 0.0f;
    }
    __syncthreads();
    v_max = abs_max_nan(abs_max_nan(v_flags[0][0], v_flags[1][0]), abs_max_nan(v_flags[2][0], v_flags[3][0]));
  }
  const bool v_lost = v_flags[0][1] + v_flags[1][1] + v_flags[2][1] + v_flags[3][1] != 0.0f;

  if constexpr (KG > 1) {
    // Fold group 1's (max, sum, accumulator) into group 0: the same lane of both groups holds the
    // same query and output dims.  A group without an unmasked key has max -inf and weight 0.
    float* xl = reinterpret_cast<float*>(smem) + ((wave % QB) * 64 + lane) * 17;
    __syncthreads();
    if (grp == 1) {
      xl[0] = m_run;
      xl[1] = l_run;
    }
    __syncthreads();
    float a0 = 1.0f, a1 = 0.0f;
    if (grp == 0) {
      const float m1 = xl[0], l1 = xl[1], m = fmaxf(m_run, m1);
      a0 = m == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m_run - m) * kLog2e);
      a1 = m == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m1 - m) * kLog2e);
      l_run = l_run * a0 + l1 * a1;
      m_run = m;
    }
#pragma unroll
    for (int i = 0; i < DVB; ++i) {
      __syncthreads();
      if (grp == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) xl[r] = acc[i][r];
      }
      __syncthreads();
      if (grp == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = acc[i][r] * a0 + xl[r] * a1;
      }
    }
    if (grp != 0) return;
  }

  const bool split = gridDim.z > 1;
  float* const part = split ? a.part + ((int64_t)blockIdx.z * gridDim.y + bh) * a.Lq * a.part_pitch : nullptr;
  float* const O = reinterpret_cast<float*>(a.o) + b * a.os[0] + head * a.os[1];

  // Queries to compute again (see the head of this file).  l = 0 is a fully masked row.
  const float low = fmaxf(0x1p-70f, 0x1p-106f * v_max);
  const uint32_t lowb = 2u * __float_as_uint(low) - 1u;
  float z = l_run * 0.0f;
  uint32_t lo = ~0u;
#pragma unroll
  for (int i = 0; i < DVB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      z = fmaf(acc[i][r], 0.0f, z);
      lo = min(lo, 2u * __float_as_uint(acc[i][r]) - 1u);
    }
  bool again = z != z || lo < lowb;
  if (v_lost) {
#pragma unroll
    for (int i = 0; i < DVB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) again |= acc[i][r] == 0.0f && i * 32 + 8 * (r >> 2) + 4 * hh + (r & 3) < Ev;
  }
  uint64_t bad = __builtin_amdgcn_ballot_w64(qok && again) | (q_bad & __builtin_amdgcn_ballot_w64(qok));
  bad = (bad | (bad >> 32)) & 0xffffffffu;
  bool mine = (bad >> col) & 1u;  // this lane's query is written by the loop below
  while (bad) {
    const int c = __builtin_ctzll(bad);
    bad &= bad - 1;
    const int64_t qq = q - col + c;
    constexpr int VPL = (DK + 63) / 64;
    float m, l, o[VPL];
    flash_row<VPL>(a, b, head, qq, kb, Lk, m, l, o);
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int d = lane + 64 * j;
      if (split) {
        if (d < DVB * 32) part[qq * a.part_pitch + d] = o[j];
      } else if (d < Ev) {
        O[qq * a.os[2] + d] = o[j] / l;
      }
    }
    if (split && lane == 0) *reinterpret_cast<float2*>(part + qq * a.part_pitch + DVB * 32) = make_float2(m, l);
  }
  if (!qok || mine) return;
  // acc / l in two steps: the quotient and one correction of it
  const float inv_l = 1.0f / l_run;
  auto out = [&](float x) {
    const float y = x * inv_l;
    return split ? x : fmaf(fmaf(-y, l_run, x), inv_l, y);
  };
  float* row = split ? part + q * a.part_pitch : O + q * a.os[2];
  const int D = split ? DVB * 32 : Ev;
  const bool vec = split || (((uintptr_t)row & 15) == 0 && (Ev & 3) == 0);
#pragma unroll
  for (int i = 0; i < DVB; ++i)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = i * 32 + 8 * g + 4 * hh;
      const float4 v = make_float4(out(acc[i][4 * g]), out(acc[i][4 * g + 1]), out(acc[i][4 * g + 2]), out(acc[i][4 * g + 3]));
      if (vec) {
        if (d0 < D) *reinterpret_cast<float4*>(row + d0) = v;
      } else {
        if (d0 < D) row[d0] = v.x;
        if (d0 + 1 < D) row[d0 + 1] = v.y;
        if (d0 + 2 < D) row[d0 + 2] = v.z;
        if (d0 + 3 < D) row[d0 + 3] = v.w;
      }
    }
  if (split && hh == 0) *reinterpret_cast<float2*>(row + DVB * 32) = make_float2(m_run, l_run);
}

}  // namespace
}  // namespace mthip
