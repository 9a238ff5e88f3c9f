// The activation backward of the expert FFN, element-wise (shared by the MFMA
// epilogue that applies it to dH and by the fp32 backward's kernels).
#pragma once

#include "mxm_kernels.h"

__device__ __forceinline__ float gelu_t(float v, float& deriv) {
  const float c = 0.7978845608f, k = 0.044715f;
  const float in = c * (v + k * v * v * v);
  const float t = tanhf(in);
  deriv = 0.5f * (1.0f + t) + 0.5f * v * (1.0f - t * t) * c * (1.0f + 3.0f * k * v * v);
  return 0.5f * v * (1.0f + t);
}

// dG and dU of one hidden unit from its gate and up projections g, u and dH
// (fp32; GLU: dG and dU, MLP: dU only).
__device__ __forceinline__ void act_bw_one(int etype, int act, float slope, float g, float u,
                                           float dh, float& dg, float& du) {
  if (etype == MXM_EXPERT_MLP) {
    float d;
    switch (act) {
      case MXM_ACT_SILU: {
        const float sg = 1.0f / (1.0f + expf(-u));
        d = sg * (1.0f + u * (1.0f - sg));
        break;
      }
      case MXM_ACT_GELU:
        (void)gelu_t(u, d);
        break;
      case MXM_ACT_RELU:
        d = u > 0.0f ? 1.0f : 0.0f;
        break;
      default: {
        const float y = u > 0.0f ? u : u * slope;
        d = 2.0f * y * (u > 0.0f ? 1.0f : slope);
        break;
      }
    }
    dg = 0.0f;
    du = dh * d;
  } else {
    float a, d;
    if (etype == MXM_EXPERT_SWIGLU) {
      a = 1.0f / (1.0f + expf(-g));
      d = a * (1.0f - a);
    } else {
      a = gelu_t(g, d);
    }
    dg = dh * u * d;
    du = dh * a;
  }
}

// 8 hidden units of one routed row of the bf16 flow: r = (dD W_down^T) ungated,
// gv / uv the raw bf16 gate and up projections (gv unused for a plain mlp).
//   h    as the up epilogue computes it (mxm_hidden_fast of the projections);
//        dot += <r, h as the forward stores it> (hi + lo for a split hidden)
//   hw   gate * h in bf16, hl = bf16(gate * h - that) for a split hidden
//   og, ou  dG and dU in bf16, from dH = gate * r
// KIND: the up projection's epilogue kind (sigmoid-GLU: the one fast sigmoid
// serves h and the derivative).
template <int KIND>
__device__ __forceinline__ void act_bw8(float slope, const float (&r)[8], uint4 gv, uint4 uv,
                                        float gate, uint4& og, uint4& ou, uint4& hw, uint4& hl,
                                        float& dot) {
  using EK = Epi<KIND>;
  const uint32_t uw[4] = {uv.x, uv.y, uv.z, uv.w}, gw[4] = {gv.x, gv.y, gv.z, gv.w};
  uint32_t o1[4], o2[4], xw[4], lw[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float dg[2], du[2], v[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const float gg = mxm_u2f(t ? gw[q] & 0xffff0000u : gw[q] << 16);
      const float uu = mxm_u2f(t ? uw[q] & 0xffff0000u : uw[q] << 16);
      const float rr = r[2 * q + t], d = gate * rr;
      float h;
      if constexpr (KIND == EPI_SWIGLU) {
        const float sg = mxm_sigmoid_fast(gg);
        h = mxm_rbf_fast(mxm_rbf_fast(sg) * uu);  // as mxm_hidden_fast
        dg[t] = d * uu * (sg * (1.0f - sg));
        du[t] = d * sg;
      } else {
        h = mxm_hidden_fast<true>(EK::ETYPE, EK::ACT, slope, gg, uu);
        act_bw_one(EK::ETYPE, EK::ACT, slope, gg, uu, d, dg[t], du[t]);
      }
      float hs = mxm_rbf_fast(h);
      if constexpr (EK::H_SPLIT) hs = hs + mxm_rbf_fast(h - hs);
      dot = __builtin_fmaf(rr, hs, dot);
      v[t] = gate * h;
    }
    xw[q] = mxm_pack_bf2_fast(v[0], v[1]);
    lw[q] = mxm_pack_bf2_fast(v[0] - mxm_u2f(xw[q] << 16), v[1] - mxm_u2f(xw[q] & 0xffff0000u));
    o1[q] = mxm_pack_bf2_fast(dg[0], dg[1]);
    o2[q] = mxm_pack_bf2_fast(du[0], du[1]);
  }
  og = make_uint4(o1[0], o1[1], o1[2], o1[3]);
  ou = make_uint4(o2[0], o2[1], o2[2], o2[3]);
  hw = make_uint4(xw[0], xw[1], xw[2], xw[3]);
  hl = make_uint4(lw[0], lw[1], lw[2], lw[3]);
}
