// Dispatch (per-expert counts, offsets, stable token permutation) and the
// deterministic combine.
//
// The reference has no dispatch: it runs every expert densely and masks with
// `top_idx == e` (gpu/ir.cpp:1118-1148).  The grouping defined here is the
// one that mask implies: expert e's rows are the tokens n with e among
// top_idx[n, :], in ascending n, and experts follow in ascending e.
//   counts[e]      = #{n : e in top_idx[n, :]}
//   offsets        = exclusive scan of counts (offsets[E] = N*K)
//   perm[offsets[e] + r] = the r-th such token
// The router leaves per-tile counts and per-slot in-tile ranks; the dispatch
// kernel below turns the counts into offsets and per-(tile, expert) bases and
// places every slot.  The result does not depend on scheduling.
//
// The combine sums, per token, gate * y over its K slots in ascending expert
// id, multiply then add in fp32, starting from 0 -- the accumulation order of
// `out = out + expert_out * gate` over e = 0..E-1 in gpu/ir.cpp:1148
// (unselected experts add +0 there).  Y is read once and delta written once,
// so the vector paths use nontemporal loads and stores (at 65,536 tokens the
// two are 2.7 GB, ten times the last-level cache; 0.52 -> 0.47 ms).
#include "mxm_kernels.h"

#include <type_traits>

namespace {
// 16-byte vectors for the nontemporal builtins (which take clang vector
// types, not HIP's float4 / uint4 structs).
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef unsigned int vu4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float wave_sum_fixed(float v) {
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) v = v + __shfl_xor(v, s, 64);
  return v;
}

// Sums of the tiles' histograms and partial sums over groups of
// MXM_DISPATCH_GROUP tiles, one workgroup per group (large batches: every
// workgroup of the dispatch reads this table, so it is kept short).
__global__ __launch_bounds__(256) void dispatch_group_kernel(DispatchArgs a) {
  const int g = blockIdx.x, t0 = g * MXM_DISPATCH_GROUP;
  const int t1 = min(a.ntiles, t0 + MXM_DISPATCH_GROUP);
  const int e = threadIdx.x;
  if (e < a.E) {
    int c = 0;
    float p = 0.0f;
    for (int t = t0; t < t1; ++t) {
      c += a.tile_counts[(size_t)t * a.E + e];
      p = p + a.tile_psum[(size_t)t * a.E + e];
    }
    a.group_counts[(size_t)g * a.E + e] = c;
    a.group_psum[(size_t)g * a.E + e] = p;
  }
  if (e < 64) {
    float s = t0 + e < t1 && e < MXM_DISPATCH_GROUP ? a.tile_ent[t0 + e] : 0.0f;
    s = wave_sum_fixed(s);
    if (e == 0) a.group_ent[g] = s;
  }
}

// Dispatch in one launch: every workgroup adds up the table of histograms
// (tiles' or groups') for itself -- all of it for the experts' totals, hence
// the offsets, and the rows before its own tiles for those tiles' bases --
// and places its tiles' slots.  Nothing is exchanged between workgroups: the
// table is a few to a few hundred KB, read from L2 by 1024 threads with
// several loads in flight, where a scan of its own with a ticket's release
// and acquire, and a launch for the slots after it, took 12-30 us (16384
// tokens of E 8: 7.7 + 4.0 us, 4096 of E 64: 23 + 5).  The last workgroup
// computes aux and entropy instead.  Sums of floats keep a fixed order:
// thread (group, e) adds the rows group, group + groups, ... ascending, the
// groups of a wave and the experts meet in butterflies, the waves in order.
constexpr int DP_NT = 1024;
constexpr int DP_TPW = 16;  // most tiles per workgroup

template <bool BF16>
__global__ __launch_bounds__(DP_NT) void dispatch_kernel(DispatchArgs a, int table_rows, int rows_per,
                                                         int tpw) {
  __shared__ int tot[MXM_MAX_EXPERTS], bef[MXM_MAX_EXPERTS];
  __shared__ int wsum[3][MXM_MAX_EXPERTS / 64];
  __shared__ int base[DP_TPW][MXM_MAX_EXPERTS];
  __shared__ float fpart[DP_NT], wterm[MXM_MAX_EXPERTS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int E = a.E, K = a.K;
  // table rows: tiles, or groups of rows_per tiles
  const int32_t* __restrict__ tab = rows_per > 1 ? a.group_counts : a.tile_counts;
  int lg = 2;  // experts padded to a power of two, one per thread of a group
  while ((1 << lg) < E) ++lg;
  const int Ep = 1 << lg, NG = DP_NT >> lg, e = tid & (Ep - 1), grp = tid >> lg;
  const bool aux_wg = blockIdx.x == gridDim.x - 1;
  const int t0 = blockIdx.x * tpw;                     // this workgroup's first tile
  const int r0 = aux_wg ? 0 : t0 / rows_per;           // table rows before it
  if (tid < MXM_MAX_EXPERTS) tot[tid] = bef[tid] = 0;
  __syncthreads();
  int vt = 0, vb = 0;
  constexpr int U = 8;
  for (int r = grp; r < table_rows; r += NG * U) {
    int v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = r + u * NG;
      v[u] = q < table_rows && e < E ? tab[(size_t)q * E + e] : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      vt += v[u];
      if (r + u * NG < r0) vb += v[u];
    }
  }
  // rows of the same expert within a wave, then over the waves (integers:
  // any order)
  for (int o = Ep; o < 64; o <<= 1) {
    vt += __shfl_xor(vt, o, 64);
    vb += __shfl_xor(vb, o, 64);
  }
  if (e < E && (Ep >= 64 || lane < Ep)) {
    atomicAdd(&tot[e], vt);
    atomicAdd(&bef[e], vb);
  }
  __syncthreads();
  // exclusive prefixes over the experts: rows, and the row tiles of both GEMMs
  int c = 0, u1 = 0, u2 = 0, i0 = 0, i1 = 0, i2 = 0;
  if (tid < MXM_MAX_EXPERTS) {
    c = tid < E ? tot[tid] : 0;
    u1 = (c + a.bm1 - 1) / a.bm1;
    u2 = (c + a.bm2 - 1) / a.bm2;
    i0 = c;
    i1 = u1;
    i2 = u2;
#pragma unroll
    for (int sh = 1; sh < 64; sh <<= 1) {
      const int v0 = __shfl_up(i0, sh, 64), v1 = __shfl_up(i1, sh, 64), v2 = __shfl_up(i2, sh, 64);
      if (lane >= sh) {
        i0 += v0;
        i1 += v1;
        i2 += v2;
      }
    }
    if (lane == 63) {
      wsum[0][wave] = i0;
      wsum[1][wave] = i1;
      wsum[2][wave] = i2;
    }
  }
  __syncthreads();
  int off = 0;
  if (tid < MXM_MAX_EXPERTS) {
    for (int w = 0; w < wave; ++w) {
      i0 += wsum[0][w];
      i1 += wsum[1][w];
      i2 += wsum[2][w];
    }
    off = i0 - c;
    if (blockIdx.x == 0 && tid < E) {
      a.counts[tid] = c;
      a.offsets[tid] = off;
      a.mstart1[tid] = i1 - u1;
      a.mstart2[tid] = i2 - u2;
      if (tid == E - 1) {
        a.offsets[E] = i0;
        a.mstart1[E] = i1;
        a.mstart2[E] = i2;
      }
    }
  }
  if (aux_wg) {
    const float* __restrict__ ps = rows_per > 1 ? a.group_psum : a.tile_psum;
    float s = 0.0f;
    for (int r = grp; r < table_rows; r += NG * U) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = r + u * NG;
        v[u] = q < table_rows && e < E ? ps[(size_t)q * E + e] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) s = s + v[u];
    }
    // the groups of a wave by a butterfly, then the waves in order
    for (int o = Ep; o < 64; o <<= 1) s = s + __shfl_xor(s, o, 64);
    const int ways = Ep < 64 ? DP_NT / 64 : NG, wd = Ep < 64 ? 64 : Ep;
    fpart[tid] = s;
    __syncthreads();
    if (tid < MXM_MAX_EXPERTS) {
      float term = 0.0f;
      if (tid < E) {
        s = fpart[tid];
        for (int g = 1; g < ways; ++g) s = s + fpart[g * wd + tid];
        const float mean = s / (float)a.N;
        const float frac = ((float)c / (float)K) / (float)a.N;
        term = (BF16 ? mxm_rbf(mean) : mean) * frac;
      }
      term = wave_sum_fixed(term);
      if (lane == 0) wterm[wave] = term;
    }
    __syncthreads();
    if (tid == 0) {
      float aux = wterm[0];
#pragma unroll
      for (int w = 1; w < MXM_MAX_EXPERTS / 64; ++w) aux = aux + wterm[w];
      const float raw = aux * (float)E;
      a.aux[0] = raw;
      if (a.aux_scaled) a.aux_scaled[0] = raw * a.aux_weight;
    }
    if (wave == 1) {
      const float* __restrict__ en = rows_per > 1 ? a.group_ent : a.tile_ent;
      float sum = 0.0f;
      for (int r = lane; r < table_rows; r += 64 * U) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = r + 64 * u < table_rows ? en[r + 64 * u] : 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u) sum = sum + v[u];
      }
      sum = wave_sum_fixed(sum);
      if (lane == 0) a.entropy[0] = -(sum / (float)a.N);
    }
    return;
  }
  // the bases of this workgroup's tiles
  if (tid < E) {
    int b = off + bef[tid];
    for (int t = r0 * rows_per; t < t0; ++t) b += a.tile_counts[(size_t)t * E + tid];
    const int nt = min(tpw, a.ntiles - t0);
    for (int j = 0; j < nt; ++j) {
      base[j][tid] = b;
      if (j + 1 < nt) b += a.tile_counts[(size_t)(t0 + j) * E + tid];
    }
  }
  __syncthreads();
  const int n0 = t0 * a.tile_tokens;
  const int nn = min(a.N - n0, tpw * a.tile_tokens);
  const size_t s0 = (size_t)n0 * K;
  const int shift = a.tile_tokens == 16 ? 4 : 6;
  for (int i = tid; i < nn * K; i += DP_NT) {
    const int ln = i / K;
    const int pos = base[ln >> shift][a.top_idx[s0 + i]] + a.slot_rank[s0 + i];
    a.perm[pos] = n0 + ln;
    a.slot_pos[s0 + i] = pos;
  }
}

// The combine for K <= 64 on narrow rows of whole 16-byte pieces: WPT waves per
// token, one for rows of 64 pieces, two up to 128, each sorting the token's
// picks for itself -- lane k's pick goes to its place in ascending expert order
// by a lane permute -- so there is no barrier and no LDS, and no thread of a
// workgroup is idle (a workgroup per token leaves three of four on a row of 512
// bf16).  Bound by memory in large batches, by the chain picks -> rows -> store
// in small ones: 16384 tokens of D 512 / K 2 18.6 -> 15.4 us, 8192 of D 640 / K 4
// 17.7 -> 14.9, 65536 of D 1024 / K 2 98 -> 94.  Wider rows fill the workgroup
// and keep the kernel below (65536 of D 2048 / K 8: 460 us, 472 with four waves
// of this one).
template <typename TY, int WPT>
__global__ __launch_bounds__(256) void combine_wave_kernel(CombineArgs a, int resid_vec) {
  constexpr int VEC = 16 / (int)sizeof(TY);
  typedef typename std::conditional<sizeof(TY) == 2, vu4, vf4>::type raw_t;
  constexpr int KC = 8;  // rows requested together
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = blockIdx.x * (4 / WPT) + wave / WPT;
  if (n >= a.N) return;  // (the whole wave)
  const int K = a.K, D = a.D;
  const size_t s0 = (size_t)n * K;
  int e = 0x7fffffff, p = 0;
  float g = 0.0f;
  if (lane < K) {
    e = a.top_idx[s0 + lane];
    g = a.gates[s0 + lane];
    p = a.slot_pos[s0 + lane];
  }
  // a token's K experts are distinct, so the number of smaller ones is the
  // slot's place; lanes past K keep theirs
  int r = 0;
  for (int j = 0; j < K; ++j) r += __builtin_amdgcn_readlane(e, j) < e;
  if (lane >= K) r = lane;
  const int sp = __builtin_amdgcn_ds_permute(r << 2, p);
  const float sg = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(r << 2, __builtin_bit_cast(int, g)));
  const TY* __restrict__ y = static_cast<const TY*>(a.y);
  const size_t ldy = a.ldy > 0 ? (size_t)a.ldy : (size_t)D;
  // D <= WPT * 64 * VEC: each lane has one piece of the row.  Lanes past D take
  // its last piece again and only leave out the store: the picks are read from
  // other lanes' registers, which is defined while every lane is active.
  const int dw = ((wave % WPT) * 64 + lane) * VEC;
  const int d = min(dw, D - VEC);
  float acc[VEC];
#pragma unroll
  for (int q = 0; q < VEC; ++q) acc[q] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += KC) {
    const int kn = min(KC, K - k0);
    raw_t row[KC];
#pragma unroll
    for (int u = 0; u < KC; ++u)
      if (u < kn)
        row[u] = __builtin_nontemporal_load(reinterpret_cast<const raw_t*>(
            y + (size_t)__builtin_amdgcn_readlane(sp, k0 + u) * ldy + d));
#pragma unroll
    for (int u = 0; u < KC; ++u) {
      if (u < kn) {
        float f[VEC];
        if constexpr (sizeof(TY) == 2) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            f[2 * q] = mxm_u2f(row[u][q] << 16);
            f[2 * q + 1] = mxm_u2f(row[u][q] & 0xffff0000u);
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) f[q] = row[u][q];
        }
        const float gk = mxm_u2f(__builtin_amdgcn_readlane(mxm_f2u(sg), k0 + u));
#pragma unroll
        for (int q = 0; q < VEC; ++q) acc[q] = __fadd_rn(acc[q], __fmul_rn(f[q], gk));
      }
    }
  }
  if (a.resid) {
    // block level: x + delta (* moe_scale), fp32
    const size_t i0 = (size_t)n * D + d;
    float xr[VEC];
    if (resid_vec && !a.resid_bf16) {
#pragma unroll
      for (int q = 0; q < VEC; q += 4) {
        const vf4 t = *reinterpret_cast<const vf4*>(static_cast<const float*>(a.resid) + i0 + q);
#pragma unroll
        for (int w = 0; w < 4; ++w) xr[q + w] = t[w];
      }
    } else {
#pragma unroll
      for (int q = 0; q < VEC; ++q)
        xr[q] = a.resid_bf16 ? mxm_bf2f(static_cast<const uint16_t*>(a.resid)[i0 + q])
                             : static_cast<const float*>(a.resid)[i0 + q];
    }
#pragma unroll
    for (int q = 0; q < VEC; ++q) {
      float v = acc[q];
      if (a.rscale) {
        const float sc = a.rscale_bf16 ? mxm_bf2f(static_cast<const uint16_t*>(a.rscale)[d + q])
                                       : static_cast<const float*>(a.rscale)[d + q];
        v = __fmul_rn(v, sc);
      }
      acc[q] = __fadd_rn(xr[q], v);
    }
  }
  if (dw >= D) return;
  float* dst = a.delta + (size_t)n * D + d;
#pragma unroll
  for (int q = 0; q < VEC; q += 4)
    __builtin_nontemporal_store(vf4{acc[q], acc[q + 1], acc[q + 2], acc[q + 3]},
                                reinterpret_cast<vf4*>(dst + q));
}

template <typename TY, int VEC>
__global__ __launch_bounds__(256) void combine_kernel(CombineArgs a) {
  __shared__ int sk[MXM_MAX_EXPERTS];  // the token's experts in top-k order
  __shared__ int sp[MXM_MAX_EXPERTS];  // slot positions, ascending expert id
  __shared__ float sg[MXM_MAX_EXPERTS];
  const int n = blockIdx.x;
  const int tid = threadIdx.x;
  const int K = a.K;  // K <= E <= 256 = blockDim.x
  int e = 0, p = 0;
  float g = 0.0f;
  if (tid < K) {
    e = a.top_idx[(size_t)n * K + tid];
    g = a.gates[(size_t)n * K + tid];
    p = a.slot_pos[(size_t)n * K + tid];
    sk[tid] = e;
  }
  __syncthreads();
  // a token's K experts are distinct, so the number of smaller ones is the
  // slot's place in ascending expert order
  if (tid < K) {
    int r = 0;
    for (int j = 0; j < K; ++j) r += sk[j] < e;
    sp[r] = p;
    sg[r] = g;
  }
  __syncthreads();
  const TY* y = static_cast<const TY*>(a.y);
  const size_t ldy = a.ldy > 0 ? (size_t)a.ldy : (size_t)a.D;
  for (int d = tid * VEC; d < a.D; d += 256 * VEC) {
    float acc[VEC];
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[q] = 0.0f;
    if constexpr ((sizeof(TY) == 2 && VEC == 8) || (sizeof(TY) == 4 && VEC == 4)) {
      // the rows of up to KC slots are requested together, then accumulated
      // in ascending expert order
      constexpr int KC = 8;
      typedef typename std::conditional<sizeof(TY) == 2, vu4, vf4>::type raw_t;
      for (int k0 = 0; k0 < K; k0 += KC) {
        const int kn = min(KC, K - k0);
        raw_t r[KC];
#pragma unroll
        for (int u = 0; u < KC; ++u)
          if (u < kn)
            r[u] = __builtin_nontemporal_load(
                reinterpret_cast<const raw_t*>(y + (size_t)sp[k0 + u] * ldy + d));
#pragma unroll
        for (int u = 0; u < KC; ++u) {
          if (u < kn) {
            float f[VEC];
            if constexpr (sizeof(TY) == 2) {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                f[2 * q] = mxm_u2f(r[u][q] << 16);
                f[2 * q + 1] = mxm_u2f(r[u][q] & 0xffff0000u);
              }
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q) f[q] = r[u][q];
            }
            const float g = sg[k0 + u];
#pragma unroll
            for (int q = 0; q < VEC; ++q) acc[q] = __fadd_rn(acc[q], __fmul_rn(f[q], g));
          }
        }
      }
    } else {
      for (int k = 0; k < K; ++k) {
        const TY* src = y + (size_t)sp[k] * ldy + d;
        float f[VEC];
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
          if constexpr (sizeof(TY) == 2)
            f[q] = mxm_bf2f(reinterpret_cast<const uint16_t*>(src)[q]);
          else
            f[q] = reinterpret_cast<const float*>(src)[q];
        }
        const float g = sg[k];
#pragma unroll
        for (int q = 0; q < VEC; ++q) acc[q] = __fadd_rn(acc[q], __fmul_rn(f[q], g));
      }
    }
    if (a.resid) {
      // block level: x + delta (* moe_scale), fp32
#pragma unroll
      for (int q = 0; q < VEC; ++q) {
        const size_t i = (size_t)n * a.D + d + q;
        const float xr = a.resid_bf16 ? mxm_bf2f(static_cast<const uint16_t*>(a.resid)[i])
                                      : static_cast<const float*>(a.resid)[i];
        float v = acc[q];
        if (a.rscale) {
          const float sc = a.rscale_bf16 ? mxm_bf2f(static_cast<const uint16_t*>(a.rscale)[d + q])
                                         : static_cast<const float*>(a.rscale)[d + q];
          v = __fmul_rn(v, sc);
        }
        acc[q] = __fadd_rn(xr, v);
      }
    }
    float* dst = a.delta + (size_t)n * a.D + d;
    if constexpr (VEC == 4 || VEC == 8) {
#pragma unroll
      for (int q = 0; q < VEC; q += 4)
        __builtin_nontemporal_store(vf4{acc[q], acc[q + 1], acc[q + 2], acc[q + 3]},
                                    reinterpret_cast<vf4*>(dst + q));
    } else {
#pragma unroll
      for (int q = 0; q < VEC; ++q) dst[q] = acc[q];
    }
  }
}


// The int8 decode flow's combine: y token-major, so a token's rows are known
// before its picks are read -- the first KC rows of each thread's first
// columns are requested first, then the gates are sorted into ascending
// expert order, then the sum runs multiply then add in fp32 in that order
// (the reference's e-loop, as combine_kernel).
template <typename TY, int VEC>
__global__ __launch_bounds__(256) void combine_tm_kernel(CombineArgs a) {
  __shared__ int sk[MXM_MAX_EXPERTS];
  __shared__ float sg[MXM_MAX_EXPERTS];
  const int n = blockIdx.x;
  const int tid = threadIdx.x;
  const int K = a.K;
  const TY* y = static_cast<const TY*>(a.y);
  const size_t ldy = a.ldy > 0 ? (size_t)a.ldy : (size_t)a.D;
  const size_t row0 = (size_t)n * K;
  constexpr bool WIDE = (sizeof(TY) == 2 && VEC == 8) || (sizeof(TY) == 4 && VEC == 4);
  typedef typename std::conditional<sizeof(TY) == 2, vu4, vf4>::type raw_t;
  constexpr int KC = 8;
  const int d0 = tid * VEC;
  raw_t pre[KC];
  if constexpr (WIDE) {
    if (d0 < a.D) {
#pragma unroll
      for (int u = 0; u < KC; ++u)
        if (u < K) pre[u] = __builtin_nontemporal_load(
                       reinterpret_cast<const raw_t*>(y + (row0 + u) * ldy + d0));
    }
  }
  int e = 0;
  float g = 0.0f;
  if (tid < K) {
    e = a.top_idx[row0 + tid];
    g = a.gates[row0 + tid];
    sk[tid] = e;
  }
  __syncthreads();
  if (tid < K) {
    int r = 0;
    for (int j = 0; j < K; ++j) r += sk[j] < e;
    sg[r] = g;
  }
  __syncthreads();
  auto add_raw = [&](float (&acc)[VEC], const raw_t& v, float gg) {
    float f[VEC];
    if constexpr (sizeof(TY) == 2) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f[2 * q] = mxm_u2f(v[q] << 16);
        f[2 * q + 1] = mxm_u2f(v[q] & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) f[q] = v[q];
    }
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[q] = __fadd_rn(acc[q], __fmul_rn(f[q], gg));
  };
  for (int d = d0; d < a.D; d += 256 * VEC) {
    float acc[VEC];
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[q] = 0.0f;
    if constexpr (WIDE) {
      for (int k0 = 0; k0 < K; k0 += KC) {
        const int kn = min(KC, K - k0);
        raw_t r[KC];
        if (d == d0 && k0 == 0) {
#pragma unroll
          for (int u = 0; u < KC; ++u) r[u] = pre[u];
        } else {
#pragma unroll
          for (int u = 0; u < KC; ++u)
            if (u < kn) r[u] = __builtin_nontemporal_load(
                            reinterpret_cast<const raw_t*>(y + (row0 + k0 + u) * ldy + d));
        }
#pragma unroll
        for (int u = 0; u < KC; ++u)
          if (u < kn) add_raw(acc, r[u], sg[k0 + u]);
      }
    } else {
      for (int k = 0; k < K; ++k) {
        const TY* src = y + (row0 + k) * ldy + d;
        float f[VEC];
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
          if constexpr (sizeof(TY) == 2)
            f[q] = mxm_bf2f(reinterpret_cast<const uint16_t*>(src)[q]);
          else
            f[q] = reinterpret_cast<const float*>(src)[q];
        }
#pragma unroll
        for (int q = 0; q < VEC; ++q) acc[q] = __fadd_rn(acc[q], __fmul_rn(f[q], sg[k]));
      }
    }
    if (a.resid) {
      // block level: x + delta (* moe_scale), fp32
#pragma unroll
      for (int q = 0; q < VEC; ++q) {
        const size_t i = (size_t)n * a.D + d + q;
        const float xr = a.resid_bf16 ? mxm_bf2f(static_cast<const uint16_t*>(a.resid)[i])
                                      : static_cast<const float*>(a.resid)[i];
        float v = acc[q];
        if (a.rscale) {
          const float sc = a.rscale_bf16 ? mxm_bf2f(static_cast<const uint16_t*>(a.rscale)[d + q])
                                         : static_cast<const float*>(a.rscale)[d + q];
          v = __fmul_rn(v, sc);
        }
        acc[q] = __fadd_rn(xr, v);
      }
    }
    float* dst = a.delta + (size_t)n * a.D + d;
    if constexpr (VEC == 4 || VEC == 8) {
#pragma unroll
      for (int q = 0; q < VEC; q += 4)
        __builtin_nontemporal_store(vf4{acc[q], acc[q + 1], acc[q + 2], acc[q + 3]},
                                    reinterpret_cast<vf4*>(dst + q));
    } else {
#pragma unroll
      for (int q = 0; q < VEC; ++q) dst[q] = acc[q];
    }
  }
}

}  // namespace

int mxm_dispatch_groups(int ntiles, int E) {
  return (int64_t)ntiles * E > MXM_DISPATCH_TABLE
             ? (ntiles + MXM_DISPATCH_GROUP - 1) / MXM_DISPATCH_GROUP
             : 0;
}

void mxm_launch_dispatch(const DispatchArgs& a, bool bf16, hipStream_t s) {
  const int groups = a.group_counts ? mxm_dispatch_groups(a.ntiles, a.E) : 0;
  if (groups > 0) hipLaunchKernelGGL(dispatch_group_kernel, dim3(groups), dim3(256), 0, s, a);
  // up to 256 workgroups of whole tiles (more past DP_TPW tiles each); tiles
  // per workgroup a power of two, so that one lies within a group
  int tpw = 1;
  while (tpw < DP_TPW && (a.ntiles + tpw - 1) / tpw > 256) tpw *= 2;
  const dim3 grid((a.ntiles + tpw - 1) / tpw + 1);
  const int rows = groups > 0 ? groups : a.ntiles, per = groups > 0 ? MXM_DISPATCH_GROUP : 1;
  if (bf16)
    hipLaunchKernelGGL(dispatch_kernel<true>, grid, dim3(DP_NT), 0, s, a, rows, per, tpw);
  else
    hipLaunchKernelGGL(dispatch_kernel<false>, grid, dim3(DP_NT), 0, s, a, rows, per, tpw);
}

void mxm_launch_combine(const CombineArgs& a, bool y_bf16, hipStream_t s) {
  if (a.N <= 0) return;
  const int ldy = a.ldy > 0 ? a.ldy : a.D;
  const bool aligned = (reinterpret_cast<uintptr_t>(a.y) % 16 == 0) &&
                       (reinterpret_cast<uintptr_t>(a.delta) % 16 == 0) && ldy % 8 == 0;
  const int span = y_bf16 ? 512 : 256;
  if (aligned && a.K <= 64 && a.D % (y_bf16 ? 8 : 4) == 0 && a.D <= 2 * span) {
    const int rv = a.resid && reinterpret_cast<uintptr_t>(a.resid) % 16 == 0;
    auto go = [&](auto wpt) {
      constexpr int W = decltype(wpt)::value;
      const dim3 grid((a.N + 4 / W - 1) / (4 / W));
      if (y_bf16)
        hipLaunchKernelGGL((combine_wave_kernel<uint16_t, W>), grid, dim3(256), 0, s, a, rv);
      else
        hipLaunchKernelGGL((combine_wave_kernel<float, W>), grid, dim3(256), 0, s, a, rv);
    };
    if (a.D <= span) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, 2>{});
    return;
  }
  if (y_bf16) {
    if (aligned && a.D % 8 == 0)
      hipLaunchKernelGGL((combine_kernel<uint16_t, 8>), dim3(a.N), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((combine_kernel<uint16_t, 1>), dim3(a.N), dim3(256), 0, s, a);
  } else {
    if (aligned && a.D % 4 == 0)
      hipLaunchKernelGGL((combine_kernel<float, 4>), dim3(a.N), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((combine_kernel<float, 1>), dim3(a.N), dim3(256), 0, s, a);
  }
}

void mxm_launch_combine_tm(const CombineArgs& a, bool y_bf16, hipStream_t s) {
  if (a.N <= 0) return;
  const int ldy = a.ldy > 0 ? a.ldy : a.D;
  const bool aligned = (reinterpret_cast<uintptr_t>(a.y) % 16 == 0) &&
                       (reinterpret_cast<uintptr_t>(a.delta) % 16 == 0) && ldy % 8 == 0;
  const dim3 grid(a.N);
  if (y_bf16) {
    if (aligned && a.D % 8 == 0)
      hipLaunchKernelGGL((combine_tm_kernel<uint16_t, 8>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((combine_tm_kernel<uint16_t, 1>), grid, dim3(256), 0, s, a);
  } else {
    if (aligned && a.D % 4 == 0)
      hipLaunchKernelGGL((combine_tm_kernel<float, 4>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((combine_tm_kernel<float, 1>), grid, dim3(256), 0, s, a);
  }
}
