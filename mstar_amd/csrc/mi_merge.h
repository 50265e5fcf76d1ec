// The merge of split-KV partials, shared by the decode and prefill translation
// units: a launch that follows both kinds of attention merges both.
#pragma once

#include "mi_plan.h"

namespace mi {

// One 256-thread workgroup per (request, kv-head); its 4 wavefronts split the output
// elements as the decode kernel's did: lane l of wavefront w merges row l%16,
// elements d = VW*(4*(l/16) + w) + j, read from the register-order partial
// layout with 64-lane contiguous (cache-line) loads.
template <typename MT, int D, int RUN, bool PAIR = false>
MI_DEVICE void merge_body(const DecodeParams& p, int32_t batch, int pair) {
  static_assert(!PAIR || D == 256, "paired kv-heads form 256-element rows");
  constexpr int VW = D / 16;
  constexpr int NS = VW / 4;  // float4 groups per lane per partial
  constexpr float kNegInf = -__builtin_inff();
  const int nkv = p.num_kv_heads;
  if (pair >= batch * nkv) return;
  const int b = pair / nkv;
  const int h = pair - b * nkv;
  const int c0 = p.chunk_indptr[b];
  const int nb = p.chunk_indptr[b + 1] - c0;
  if (nb == 1) return;  // written directly by the decode kernel
  int qo_start = b, qo_len = 1;
  if (p.qo_indptr) {
    qo_start = p.qo_indptr[b];
    qo_len = p.qo_indptr[b + 1] - qo_start;
  }
  const int G = p.group;
  const int rows = (PAIR ? 2 : 1) * qo_len * G;
  if (qo_len * G > p.short_rows) return;  // long-query request: written by the prefill kernel
  const int lane = lane_id();
  const int wave = (int)threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  if (col >= rows) return;
  const int half = PAIR && col >= qo_len * G ? 1 : 0;
  const int rcol = col - half * qo_len * G;
  const int hq = PAIR ? 2 * h + half : h;
  const int qtok = rcol / G, g = rcol - qtok * G;
  float4 acc[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  const int64_t u0 = (int64_t)c0 * nkv + h;  // unit of chunk c: u0 + c * nkv
  // One pass: each group of U partials is loaded with its lse values at
  // once (no separate max pass ahead of the loads), and the running sum is
  // rescaled when a partial raises the running max.
  float M = kNegInf, wsum = 0.f;
  constexpr int U = D > 128 ? 4 : 8;  // partials in flight per step
  for (int c = 0; c < nb; c += U) {
    float w[U];
    float4 o[U][NS];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      w[u] = kNegInf;
      if (c + u < nb) {
        const int64_t unit = u0 + (int64_t)(c + u) * nkv;
        w[u] = p.lse_part[unit * kRows + col];
        const float* src = p.o_part + unit * kRows * D + 4 * lane + 256 * wave * NS;
#pragma unroll
        for (int i = 0; i < NS; ++i) o[u][i] = *(const float4*)(src + 256 * i);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (w[u] == kNegInf) continue;  // past the end, or an empty partial (a NaN lse makes the row NaN)
      if (w[u] > M) {
        const float sc = fast_exp2(M - w[u]);  // 0 while M is -inf
        wsum *= sc;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
          acc[i].x *= sc;
          acc[i].y *= sc;
          acc[i].z *= sc;
          acc[i].w *= sc;
        }
        M = w[u];
      }
      const float wgt = fast_exp2(w[u] - M);
      wsum += wgt;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        acc[i].x += wgt * o[u][i].x;
        acc[i].y += wgt * o[u][i].y;
        acc[i].z += wgt * o[u][i].z;
        acc[i].w += wgt * o[u][i].w;
      }
    }
  }
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  const int64_t orow_off = (int64_t)(qo_start + qtok) * p.out_stride_tok + (int64_t)(hq * G + g) * p.out_stride_head;
  // this wave's elements of the row: group i holds d = dim_of(RUN, 4*grp + wave, 4*i) .. +3
  if constexpr (MT::kDtype == MI_F32) {
    float* orow = (float*)p.out + orow_off;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const float4 a = acc[i];
      *(float4*)(orow + dim_of(RUN, 4 * grp + wave, 4 * i)) = make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
    }
  } else {
    uint16_t* orow = (uint16_t*)p.out + orow_off;
    uint32_t w[VW / 2];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      w[2 * i] = MT::pack2(acc[i].x * inv, acc[i].y * inv);
      w[2 * i + 1] = MT::pack2(acc[i].z * inv, acc[i].w * inv);
    }
    if constexpr (VW == 4) {
      *(uint2*)(orow + dim_of(RUN, 4 * grp + wave, 0)) = make_uint2(w[0], w[1]);
    } else {
#pragma unroll
      for (int i = 0; i < VW / 2; i += 4) {
        const int d0 = dim_of(RUN, 4 * grp + wave, 2 * i);  // 8 consecutive elements
        if (PAIR && (d0 >= D / 2) != (half == 1)) continue;  // the other head's half
        *(uint4*)(orow + d0 - (PAIR ? (D / 2) * half : 0)) = make_uint4(w[i], w[i + 1], w[i + 2], w[i + 3]);
      }
    }
  }
}

}  // namespace mi
