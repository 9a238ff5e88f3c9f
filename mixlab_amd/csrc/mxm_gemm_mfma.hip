// Grouped expert FFN on bf16 MFMA (gfx950, v_mfma_f32_32x32x16_bf16).
//
// One workgroup computes a BM x BN tile of one expert's output.  A rows are
// the expert's permuted slots: for the up projections they are gathered from
// x through `perm` (each row is D contiguous bf16), for the down projection
// they are the contiguous rows of H.  B is the expert's weight stored
// transposed ([out, in], k contiguous) so both operands stream k-contiguous
// 16-byte chunks.
//
// Operand tiles move global -> LDS with global_load_lds_dwordx4 (no VGPR
// round trip) into a ring of NS stages of BK k each; each lane's 16-byte
// chunk lands at a swizzled position so the 16-lane phases of ds_read_b128
// hit distinct banks.  Waves wait for their own loads with explicit vmcnt
// counts and meet at s_barrier; the loads of the next stage are spread over
// the first k steps of the current one so the vector memory path fills in
// the background.  With three or more stages the barrier of stage kt+1 is
// taken before the last k step of stage kt, so it overlaps MFMA work.
//
// Tile shapes: 256 x 256 x 64 (8 waves as 2 x 4, each 128 x 64 = 4 x 2 MFMA
// tiles, 2 stages, one workgroup per CU), 256 x 128 x 32 (4 waves, 3 stages)
// and 128 x 128 x 64 (4 waves, 2 stages; two workgroups per CU), and 128 x
// 128 x 64 with four more waves that do the loading (4 stages).  By default a
// launch mixes 256 x 256 and 128 x 128 tiles (gemm_sched_kernel) or takes 128
// x 128 ones in pairs (mxm_launch_gemm_mfma); flags select one shape.  The
// GLU weight rows are interleaved in groups of 32 (gate cols f..f+31, then up
// cols f..f+31), so a wave's two column MFMA tiles hold gate and up for the
// same 32 hidden units and the activation is applied straight from the
// accumulators.
//
// Ragged experts: every workgroup computes the tiles of the launch from the
// experts' offsets (prefixes of their row tiles in LDS), so a tile's expert
// and rows are resolved without a launch or a memory lookup for it.
//
// The grid is persistent: as many workgroups as fit on the device at once,
// each walking its places of the tile list; a CU goes from one tile's
// epilogue straight to the next tile while the stores drain, instead of
// waiting for the workgroup to retire and a new one to be dispatched.
//
// Tile order: row tiles are grouped GM at a time with the column tiles of a
// group adjacent, and each XCD (the hardware hands workgroup L to XCD L % 8)
// takes an eighth of that list in whole groups (XcdPart), so its L2 sees a GM x
// (N/BN) block of tiles sharing A rows and B columns and every CU gets the same
// number of tiles to within one.  The epilogue applies the activation (hardware exp2 /
// rcp and bf16 conversion), stages each wave's bf16 tile through LDS
// (chunk-swizzled) and writes 16-byte row segments.
#include <algorithm>
#include <type_traits>

#include "mxm_act_bw.h"
#include "mxm_kernels.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
// Native vector type for 16-byte moves (HIP's uint4 wrapper class defeats
// scalar replacement of the prefetch registers).
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

#ifndef MXM_DMA_STEPS
#define MXM_DMA_STEPS 2
#endif

#ifndef MXM_GM
#define MXM_GM 6
#endif
constexpr int GM = MXM_GM;        // row tiles per scheduling group

// Physical 16-byte chunk of logical chunk kc in tile row `row` (CH chunks per
// row).  ds_read_b128 is serviced 16 lanes (16 consecutive rows, one chunk)
// at a time over 64 four-byte banks = 16 groups of 16 bytes; rows r and
// r + 16/CH fall in the same groups, so the CH rows of a phase that share
// them get distinct chunks.
template <int CH>
__device__ __forceinline__ int swz_phys(int row, int kc) {
  return kc ^ ((row / (16 / CH)) % CH);
}
template <int CH>
__device__ __forceinline__ int swz(int row, int kc) {
  return row * CH + swz_phys<CH>(row, kc);
}

// Direct global->LDS load of 16 bytes per lane (global_load_lds_dwordx4):
// lane l's data lands at LDS address `lds` + 16*l.  Issued as inline asm so
// the compiler does not track it: its conservative tracking of LDS DMA would
// otherwise drain every in-flight stage before the next LDS read.  The caller
// waits with explicit vmcnt counts (stage_barrier) before reading.  M0 holds
// the LDS base; nothing else in these kernels uses M0.
__device__ __forceinline__ void dma16(const void* g, const void* lds) {
  const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(g), "s"(base)
               : "memory", "m0");
}

// The same load from a uniform 64-bit base in SGPRs plus the lane's 32-bit
// byte offset (the SGPR-base form: no 64-bit address arithmetic per load).
__device__ __forceinline__ void dma16s(const void* base, unsigned off_bytes, const void* lds) {
  const unsigned lb = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)lds);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off_bytes), "s"(base), "s"(lb)
               : "memory", "m0");
}

// Wait until at most N of this thread's direct-to-LDS loads are in flight and
// its LDS reads are done, then the workgroup barrier.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

// The barrier of a wave with no loads in flight: its LDS reads are done.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

// Tile family: BM x BN workgroup tile, WM x WN waves, each wave
// (BM/WM) x (BN/WN) = TM x TN MFMA 32x32 tiles.  With LOADERS, that many
// more waves issue all the loads and the computing waves none.
template <int BM, int BN, int WM, int WN, int WAVES_PER_SIMD, int NSTAGE, int BKK, int LOADERS = 0>
struct Tile {
  static constexpr int NS = NSTAGE;
  static constexpr int BK = BKK;      // k per LDS stage
  static constexpr int CH = BKK / 8;  // 16-byte chunks per tile row
  static constexpr int CW = WM * WN;  // computing waves
  static constexpr int LW = LOADERS > 0 ? LOADERS : CW;  // waves that load
  static constexpr int NT = 64 * (CW + LOADERS);
  static constexpr int TM = BM / WM / 32;
  static constexpr int TN = BN / WN / 32;
  static constexpr int A_CH = BM * CH;
  static constexpr int B_CH = BN * CH;
  static constexpr int BUF = A_CH + B_CH;
  static constexpr int WPS = WAVES_PER_SIMD;
  static_assert(TN % 2 == 0, "GLU epilogue pairs gate and up column tiles");
  static_assert(A_CH % (64 * LW) == 0 && B_CH % (64 * LW) == 0, "whole chunks per thread");
};

// One BM x BN tile: rows row0 .. row0 + rows - 1 of expert e (rows <= BM) by
// columns n0 .. n0 + BN - 1, with the LDS ring (NS * BUF chunks) at lds.
template <class TL, int BM, int BN, int WM, int WN, int EPI>
__device__ __forceinline__ void gemm_tile(const GemmArgs& a, u32x4_t* lds, int e, int row0,
                                          int rows, int n0) {
  constexpr int MODE = Epi<EPI>::MODE;
  constexpr bool DOWN_SPLIT = Epi<EPI>::DOWN_SPLIT;  // A = [hi | lo] planes, y in fp32
  // 32-bit A offsets (when A fits) for the forward's up projections only:
  // measured faster there, slower for the down projection and no faster
  // for the raw-keeping variant
  constexpr bool A_OFF32 = MODE != MXM_GEMM_DOWN && !Epi<EPI>::KEEP_RAW;
  constexpr bool H_SPLIT = Epi<EPI>::H_SPLIT;        // H stored as [hi | lo] planes
  constexpr int NT = TL::NT, TM = TL::TM, TN = TL::TN;
  constexpr int A_CH = TL::A_CH, BUF = TL::BUF;
  constexpr int NW = NT / 64, LW = TL::LW;
  constexpr int NS = TL::NS;  // LDS stages in the ring (NS-1 in flight)
  constexpr int BK = TL::BK, CH = TL::CH;
  const int Kd = a.Kd;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  // int8 weights (the bf16 B holds the integers q): this lane's output
  // columns' scales, read before the k loop so their latency is hidden.
  // Lane l's accumulators of column tile j are column j*32 + l%32 of the
  // wave's; GLU tiles alternate gate (scale0) and up (scale1) over the same
  // 32 hidden units.
  float scv[TN];
  if constexpr (Epi<EPI>::SCALED) {
    const int wc0 = n0 + wn * TN * 32;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (MODE == MXM_GEMM_GLU) {
        const int hc = a.Ncols / 2;
        const float* sp = (j & 1) ? a.scale1 : a.scale0;
        scv[j] = sp[(size_t)e * hc + wc0 / 2 + (j >> 1) * 32 + (lane & 31)];
      } else {
        scv[j] = a.scale0[(size_t)e * a.Ncols + wc0 + j * 32 + (lane & 31)];
      }
    }
  }

  const uint16_t* __restrict__ A = static_cast<const uint16_t*>(a.a);
  // B rows hold Kb k values; the split down projection reads W_down [D][F]
  // twice along its reduction over the hi and lo planes (k wraps at F)
  const int Kb = DOWN_SPLIT ? Kd / 2 : Kd;
  // pairs of operand planes along k (GemmArgs::f32_out)
  constexpr bool PAIRS = Epi<EPI>::PLANE_PAIRS;
  const int Kp = PAIRS ? Kd / a.planes : Kd;
  const int lda = PAIRS ? a.lda : Kd, ldb = PAIRS ? a.ldb : Kb;
  // first element of stage k0 within A's and B's rows
  auto ka = [&](int k0) {
    if constexpr (!PAIRS) return k0;
    const int p = (k0 >= Kp) + (k0 >= 2 * Kp);
    return k0 - p * Kp + ((a.amap >> p) & 1) * Kp;
  };
  auto kb = [&](int k0) {
    if constexpr (DOWN_SPLIT) return k0 >= Kb ? k0 - Kb : k0;
    if constexpr (!PAIRS) return k0;
    const int p = (k0 >= Kp) + (k0 >= 2 * Kp);
    return k0 - p * Kp + ((a.bmap >> p) & 1) * Kp;
  };
  const uint16_t* __restrict__ B =
      static_cast<const uint16_t*>(a.b0) + (size_t)e * a.Ncols * ldb;

  // Global->LDS: global_load_lds_dwordx4 writes lane l's 16 bytes to
  // LDS base + 16*l, so one wave-load fills 1 KB = 64/CH consecutive tile
  // rows.  Lane l lands in row (l/CH) of its group at physical chunk l%CH and
  // fetches the logical k-chunk stored there -- the swizzle is applied on the
  // global address.
  constexpr int RPW = 64 / CH;     // tile rows per wave-load
  constexpr int QA = BM / RPW / LW;  // A wave-loads per wave per stage
  constexpr int QB = BN / RPW / LW;
  constexpr int LDPS = QA + QB;      // direct-to-LDS loads per thread per stage
  static_assert(QA * RPW * LW == BM && QB * RPW * LW == BN, "whole wave-loads");
  constexpr bool LOADERS = LW != NW;
  // this wave's place among the loading waves (a computing wave of a tile
  // with loaders: any)
  const int lwave = LOADERS ? (wave >= TL::CW ? wave - TL::CW : 0) : wave;
  const int lrow = lane / CH;  // row within the wave-load group
  // Logical chunk of this lane's physical slot (the swizzle is an involution).
  // It depends on the tile row modulo 16; the row of load i is
  // (lwave + LW*i)*RPW + lrow, which is the same modulo 16 for every i because
  // LW*RPW is a multiple of 16.
  static_assert((LW * RPW) % 16 == 0, "swizzle phase is the same for every wave-load of a lane");
  const int lkc = swz_phys<CH>(lwave * RPW + lrow, lane % CH);
  size_t aoff[QA];
#pragma unroll
  for (int i = 0; i < QA; ++i) {
    const int r = (lwave + LW * i) * RPW + lrow;
    const int p = row0 + min(r, rows - 1);  // rows past the segment reload a valid row
    const int src = (MODE == MXM_GEMM_DOWN && !a.gather_a) ? p : a.perm[p];
    aoff[i] = 2 * ((size_t)src * lda + lkc * 8);  // bytes
  }
  const size_t bstep = (size_t)(LW * RPW) * ldb;
  // the B loads as 32-bit byte offsets from the expert's matrix (one expert's
  // Ncols x Kb bf16 stays far below 4 GiB); the wave index in an SGPR keeps
  // every load's LDS destination scalar
  const int wv = __builtin_amdgcn_readfirstlane(lwave);
  const unsigned boff = (unsigned)(2 * ((size_t)(n0 + wv * RPW + lrow) * ldb + lkc * 8));
  const unsigned bstep_b = (unsigned)(2 * bstep);

// Direct-to-LDS loads Q0 .. Q1-1 of one stage (load q < QA fills A rows,
// the rest B rows).
#define MXM_DMA_LOOP(STAGE, K0, Q0, Q1, ALOAD)                                                \
  _Pragma("unroll") for (int q_ = (Q0); q_ < (Q1); ++q_) {                                    \
    if (q_ < QA) {                                                                            \
      ALOAD;                                                                                  \
    } else {                                                                                  \
      dma16s(B + kb(K0), boff + (q_ - QA) * bstep_b,                                          \
             STAGE + A_CH + (wv + LW * (q_ - QA)) * 64);                                      \
    }                                                                                         \
  }
#define MXM_DMA_PART(STAGE, K0, Q0, Q1)                                                       \
  do {                                                                                        \
    if (A_OFF32 && a.a_off32) {                                                               \
      MXM_DMA_LOOP(STAGE, K0, Q0, Q1,                                                         \
                   dma16s(A + ka(K0), (unsigned)aoff[q_], STAGE + (wv + LW * q_) * 64))       \
    } else {                                                                                  \
      MXM_DMA_LOOP(STAGE, K0, Q0, Q1,                                                         \
                   dma16(reinterpret_cast<const char*>(A + ka(K0)) + aoff[q_],                \
                         STAGE + (wv + LW * q_) * 64))                                        \
    }                                                                                         \
  } while (0)
#define MXM_DMA(STAGE, K0) MXM_DMA_PART(STAGE, K0, 0, LDPS)
  // Stage barrier: this thread's loads of the current stage have landed (at
  // most AHEAD later stages still in flight), then the workgroup barrier --
  // the stage is complete for every wave and the stage consumed in the
  // previous step is free.
#define MXM_STAGE_BARRIER(AHEAD)              \
  do {                                        \
    if ((AHEAD) >= 3)                         \
      stage_barrier<3 * LDPS>();              \
    else if ((AHEAD) == 2)                    \
      stage_barrier<2 * LDPS>();              \
    else if ((AHEAD) == 1)                    \
      stage_barrier<LDPS>();                  \
    else                                      \
      stage_barrier<0>();                     \
  } while (0)
  static_assert(NS >= 2 && NS <= 5, "stage barrier counts cover up to three stages ahead");
  static_assert(3 * LDPS <= 63, "vmcnt holds at most 63 outstanding loads");

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // Fragment registers are double-buffered across the 16-wide k steps: the
  // reads for step ks+1 are issued before the MFMAs of step ks.
  const int arow = wm * TM * 32 + (lane & 31);
  const int brow = wn * TN * 32 + (lane & 31);
  bf16x8_t af[2][TM], bfm[2][TN];

#define MXM_FRAGS(STAGE, P, KS)                                                               \
  do {                                                                                        \
    const int kc_ = (KS) * 2 + (lane >> 5);                                                   \
    /* B first: the first MFMA needs b0 and a0, so it waits for TN + 1 reads */               \
    _Pragma("unroll") for (int j = 0; j < TN; ++j) bfm[P][j] =                                \
        __builtin_bit_cast(bf16x8_t, (STAGE)[A_CH + swz<CH>(brow + j * 32, kc_)]);            \
    _Pragma("unroll") for (int i = 0; i < TM; ++i) af[P][i] =                                 \
        __builtin_bit_cast(bf16x8_t, (STAGE)[swz<CH>(arow + i * 32, kc_)]);                   \
  } while (0)
// Per 16-wide k step: the fragment reads of the next step are interleaved
// one by one between the MFMAs of this step (sched_group_barrier pins the
// order: 1 MFMA, 1 LDS read, ...), so LDS latency hides behind MFMAs.  After
// the stage barrier the first step's TM + TN reads are all issued before its
// first MFMA, so the stage start costs one LDS latency rather than a read,
// wait, MFMA chain.  After
// each step, a share of the direct-to-LDS loads of stage DSTAGE (k offset
// DK0) is issued, so the vector memory path fills in the background instead
// of stalling every wave right after the stage barrier.
#define MXM_COMPUTE(STAGE, DO_DMA, DSTAGE, DK0)                                               \
  do {                                                                                        \
    MXM_FRAGS(STAGE, 0, 0);                                                                   \
    _Pragma("unroll") for (int ks = 0; ks < BK / 16; ++ks) {                                  \
      if (ks + 1 < BK / 16) MXM_FRAGS(STAGE, (ks + 1) & 1, ks + 1);                           \
      _Pragma("unroll") for (int i = 0; i < TM; ++i)                                          \
          _Pragma("unroll") for (int j = 0; j < TN; ++j) acc[i][j] =                          \
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][i], bfm[ks & 1][j],          \
                                                      acc[i][j], 0, 0, 0);                    \
      if (ks + 1 < BK / 16) {                                                                 \
        if (ks == 0) /* the first step's fragments all go out before its MFMAs */             \
          __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);                            \
        _Pragma("unroll") for (int q = 0; q < TM * TN; ++q) {                                 \
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                  \
          if (q < TM + TN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                 \
        }                                                                                     \
      }                                                                                       \
      if ((DO_DMA) && ks < DSTEPS)                                                            \
        MXM_DMA_PART(DSTAGE, DK0, ks * LDPS / DSTEPS, (ks + 1) * LDPS / DSTEPS);              \
    }                                                                                         \
  } while (0)

// One 16-wide k step on fragment set P; if DOFRAG, the fragments of k step
// FKS of stage FSTAGE are read into set P^1 in between the MFMAs.
#define MXM_KSTEP(P, FSTAGE, FKS, DOFRAG)                                                     \
  do {                                                                                        \
    if (DOFRAG) MXM_FRAGS(FSTAGE, (P) ^ 1, FKS);                                              \
    _Pragma("unroll") for (int i = 0; i < TM; ++i)                                            \
        _Pragma("unroll") for (int j = 0; j < TN; ++j) acc[i][j] =                            \
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[P][i], bfm[P][j], acc[i][j], 0, 0, 0); \
    if (DOFRAG) {                                                                             \
      _Pragma("unroll") for (int q = 0; q < TM * TN; ++q) {                                   \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                    \
        if (q < TM + TN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                   \
      }                                                                                       \
    }                                                                                         \
  } while (0)

  // k steps over which the next stage's loads are spread
  constexpr int DSTEPS = (MXM_DMA_STEPS > 0 && MXM_DMA_STEPS < BK / 16) ? MXM_DMA_STEPS : BK / 16;
  constexpr int KS = BK / 16;
  const int nk = Kd / BK;
  if constexpr (LOADERS) {
    // Loading waves keep NS - 1 stages in flight; the computing waves only
    // meet them at the stage barriers.  (With all waves loading, the loads of
    // a stage queue up in every wave's way: a 128 x 128 x 64 stage takes the
    // CU's load path about as long to accept as its MFMAs run.)  The barrier
    // before a stage's last k step, as in the deep ring below.
    static_assert(NS >= 3 && KS % 2 == 0, "a deep ring");
    if (__builtin_amdgcn_readfirstlane(wave) >= TL::CW) {
#pragma unroll
      for (int st = 0; st < NS - 1; ++st)
        if (st < nk) MXM_DMA(lds + st * BUF, st * BK);
      MXM_STAGE_BARRIER(min(NS - 2, nk - 1));
      for (int kt = 0; kt < nk - 1; ++kt) {
        MXM_STAGE_BARRIER(min(NS - 3, nk - 2 - kt));
        if (kt + NS - 1 < nk) MXM_DMA(lds + ((kt + NS - 1) % NS) * BUF, (kt + NS - 1) * BK);
      }
      MXM_STAGE_BARRIER(0);
      return;
    }
    lds_barrier();
    MXM_FRAGS(lds, 0, 0);
    for (int kt = 0; kt < nk - 1; ++kt) {
      const u32x4_t* cur = lds + (kt % NS) * BUF;
#pragma unroll
      for (int ks = 0; ks < KS - 1; ++ks) MXM_KSTEP(ks & 1, cur, ks + 1, true);
      lds_barrier();
      MXM_KSTEP((KS - 1) & 1, lds + ((kt + 1) % NS) * BUF, 0, true);
    }
    const u32x4_t* cur = lds + ((nk - 1) % NS) * BUF;
#pragma unroll
    for (int ks = 0; ks < KS - 1; ++ks) MXM_KSTEP(ks & 1, cur, ks + 1, true);
    MXM_KSTEP((KS - 1) & 1, cur, 0, false);
    lds_barrier();
  } else {
  // first stage: the weight rows go out first, they do not wait for perm
  if (nk > 0) {
    MXM_DMA_PART(lds, 0, QA, LDPS);
    MXM_DMA_PART(lds, 0, 0, QA);
  }
#pragma unroll
  for (int st = 1; st < NS - 1; ++st)
    if (st < nk) MXM_DMA(lds + st * BUF, st * BK);
  if constexpr (NS >= 3) {
    // Deep ring: the barrier of stage kt+1 is taken before the last k step
    // of stage kt, while that step's fragments are already in registers and
    // the MFMAs issued just before it are still executing, so the barrier
    // and the first fragment reads of the next stage overlap MFMA work.  At
    // that barrier stage kt+1 has landed and stage kt-1 is free; it receives
    // stage kt+NS-1.
    static_assert(KS % 2 == 0, "fragment set parity repeats every stage");
    MXM_STAGE_BARRIER(min(NS - 2, nk - 1));
    MXM_FRAGS(lds, 0, 0);
    // (the last stage is peeled so the accumulators flow through one path)
    for (int kt = 0; kt < nk - 1; ++kt) {
      const u32x4_t* cur = lds + (kt % NS) * BUF;
#pragma unroll
      for (int ks = 0; ks < KS - 1; ++ks) MXM_KSTEP(ks & 1, cur, ks + 1, true);
      MXM_STAGE_BARRIER(min(NS - 3, nk - 2 - kt));
      if (kt + NS - 1 < nk) MXM_DMA(lds + ((kt + NS - 1) % NS) * BUF, (kt + NS - 1) * BK);
      MXM_KSTEP((KS - 1) & 1, lds + ((kt + 1) % NS) * BUF, 0, true);
    }
    {
      const u32x4_t* cur = lds + ((nk - 1) % NS) * BUF;
#pragma unroll
      for (int ks = 0; ks < KS - 1; ++ks) MXM_KSTEP(ks & 1, cur, ks + 1, true);
      MXM_KSTEP((KS - 1) & 1, cur, 0, false);
    }
  } else {
    for (int kt = 0; kt < nk; ++kt) {
      // stage kt is complete and the stage consumed at kt-1 is free; it
      // receives stage kt+NS-1 while the MFMAs of stage kt run
      MXM_STAGE_BARRIER(min(NS - 2, nk - 1 - kt));
      const u32x4_t* cur = lds + (kt % NS) * BUF;
      const bool more = kt + NS - 1 < nk;
      MXM_COMPUTE(cur, more, lds + ((kt + NS - 1) % NS) * BUF, (kt + NS - 1) * BK);
    }
  }
  MXM_STAGE_BARRIER(0);  // every wave is done reading before the staging reuse
  }
#undef MXM_DMA
#undef MXM_DMA_PART
#undef MXM_STAGE_BARRIER
#undef MXM_FRAGS
#undef MXM_COMPUTE
#undef MXM_KSTEP

  if constexpr (Epi<EPI>::SCALED) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] *= scv[j];
  }
  if constexpr (Epi<EPI>::ACT_BW) {
    // The activation backward on dH in the accumulators, 32 rows at a time: each
    // wave stages its 32 x 64 block in LDS and takes 8 hidden units of a row per
    // lane, whose raw projections are loaded before.  (As a pass of its own over
    // a stored bf16 dH it read and wrote 0.8 GB: the product and it took 229 us
    // at 32768 rows of ffn 2048, the product with this epilogue 187.)  Each
    // kind has its code, and a block's projections are requested together: with
    // the kind looked up at run time and one request after the other, 18000
    // rows of ffn 512 took 66.5 us for a plain silu, 59.2 for geglu; 29.0 and
    // 42.2 like this.
    constexpr int KIND = Epi<EPI>::BW_KIND;
    constexpr bool glu = Epi<KIND>::MODE == MXM_GEMM_GLU, split = Epi<KIND>::H_SPLIT;
    // kinds with a tanh: the code of 8 rows once per block (four copies keep
    // the block loop, and so the accumulators' indexes, from being unrolled)
    constexpr bool ONCE = Epi<KIND>::ACT == MXM_ACT_GELU;
    constexpr int SR = 72;  // floats per staged row: the two half-waves' writes in other banks
    static_assert(TN == 2 && TL::CW * 32 * SR * 4 <= (int)sizeof(u32x4_t) * NS * BUF, "staging");
    float* st = reinterpret_cast<float*>(lds) + wave * (32 * SR);
    const int F = a.Ncols, NC = glu ? 2 * F : F;
    const int wc = n0 + wn * 64, f = wc + (lane & 7) * 8;
    const int cu = glu ? (f >> 5) * 64 + 32 + (f & 31) : f;
    const size_t hstride = split ? 2 * (size_t)F : (size_t)F;
    const int dgs = mxm_dgp_stride(F);
    float* __restrict__ dgp = a.abw.dgp + (wc >> 6);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int lr0 = wm * TM * 32 + i * 32 + (lane >> 3);
      auto load = [&](int s, uint4& gv, uint4& uv, float& gate) {
        const int p = row0 + min(lr0 + 8 * s, rows - 1);  // (rows past the segment: its last)
        const uint16_t* g = a.abw.gu + (size_t)p * NC + cu;
        uv = *reinterpret_cast<const uint4*>(g);
        gv = glu ? *reinterpret_cast<const uint4*>(g - 32) : make_uint4(0u, 0u, 0u, 0u);
        gate = a.abw.gp[p];
      };
      auto apply = [&](int s, uint4 gv, uint4 uv, float gate) {
        const float4* q = reinterpret_cast<const float4*>(st + (8 * s + (lane >> 3)) * SR +
                                                          (lane & 7) * 8);
        const float4 r0 = q[0], r1 = q[1];
        const float rr[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
        uint4 og, ou, hw, hl;
        float dot = 0.0f;
        act_bw8<KIND>(a.slope, rr, gv, uv, gate, og, ou, hw, hl, dot);
        dot = dot + mxm_xor_lane_f(dot, 1);
        dot = dot + mxm_xor_lane_f(dot, 2);
        dot = dot + mxm_xor_lane_f(dot, 4);
        const int lr = lr0 + 8 * s;
        if (lr < rows) {
          const size_t p = (size_t)(row0 + lr);
          uint16_t* o = a.abw.dgu + p * NC + cu;
          *reinterpret_cast<uint4*>(o) = ou;
          if (glu) *reinterpret_cast<uint4*>(o - 32) = og;
          uint16_t* h = a.abw.Hg + p * hstride + f;
          *reinterpret_cast<uint4*>(h) = hw;
          if (split) *reinterpret_cast<uint4*>(h + F) = hl;
          if ((lane & 7) == 0) dgp[p * dgs] = dot;
        }
      };
      uint4 gv[4], uv[4];
      float gate[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) load(s, gv[s], uv[s], gate[s]);
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          st[((r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * SR + j * 32 + (lane & 31)] = acc[i][j][r];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if constexpr (!ONCE) {
#pragma unroll
        for (int s = 0; s < 4; ++s) apply(s, gv[s], uv[s], gate[s]);
      } else {
#pragma unroll 1
        for (int s = 0; s < 4; ++s) {
          apply(s, gv[0], uv[0], gate[0]);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            gv[q] = gv[q + 1];
            uv[q] = uv[q + 1];
            gate[q] = gate[q + 1];
          }
        }
      }
      // this wave's reads are complete before the next block is staged
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
  if constexpr (Epi<EPI>::Y_F32) {
    // y in fp32, straight from the accumulators: register r of lane l holds
    // C[(r/4)*8 + (l/32)*4 + r%4][l%32], so each store instruction writes
    // 32 consecutive floats of two rows
    float* __restrict__ yo = static_cast<float*>(a.out);
    const int ycol = n0 + wn * TN * 32 + (lane & 31);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int lr = wm * TM * 32 + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
        if (lr < rows) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            __builtin_nontemporal_store(acc[i][j][r],
                                        yo + (size_t)(row0 + lr) * a.Ncols + ycol + j * 32);
        }
      }
    return;
  }
  // ---- epilogue: activation, bf16, per-wave LDS staging, 16-byte stores ----
  // 32x32 accumulator layout: register r of lane l holds
  // C[(r/4)*8 + (l/32)*4 + r%4][l%32].  Registers r and r+1 (r even) hold two
  // consecutive rows of one column; they are converted together and staged
  // as one 32-bit word (low half the even row) of a row-pair line, so a wave
  // writes half as many LDS words as it has outputs.  Lines hold C words (the
  // wave's output columns).  Staging swizzle, with kp the row pair:
  //   C = 64: line kp, 16-byte chunk ch -> ch ^ (kp & 1) ^ ((kp >> 1 & 1) << 3)
  //   C = 32: line kp ^ (kp >> 1 & 1), chunk ch -> ch ^ (kp >> 1 & 1)
  // A write instruction covers 32 columns of row pairs kp and kp + 2 (the two
  // half-waves), which land in disjoint banks; a read instruction's 16-lane
  // phases take two 16-byte chunks of four (C = 32) or two (C = 64) row
  // pairs, also in disjoint banks.
  constexpr int WROWS = TM * 32;
  constexpr int C = (MODE == MXM_GEMM_GLU) ? TN * 16 : TN * 32;  // output columns per wave
  static_assert(C == 32 || C == 64, "staging swizzle covers 32 or 64 columns per wave");
  // words of staging per row pair and wave: the widest of the tile's stores
  constexpr int CS = Epi<EPI>::KEEP_RAW && TN * 32 > C ? TN * 32 : C;
  static_assert(NW * WROWS * CS * 2 <= (int)sizeof(u32x4_t) * NS * BUF, "staging fits in LDS");
  uint32_t* stage = reinterpret_cast<uint32_t*>(lds) + (size_t)wave * (WROWS / 2) * CS;
  auto word_at = [](int kp, int c) -> int {
    const int b1 = (kp >> 1) & 1;
    if constexpr (C == 64) {
      const int ch = (c >> 2) ^ (kp & 1) ^ (b1 << 3);
      return kp * C + ch * 4 + (c & 3);
    } else {
      const int ch = (c >> 2) ^ b1;
      return (kp ^ b1) * C + ch * 4 + (c & 3);
    }
  };
  const int col = lane & 31;
  if constexpr (Epi<EPI>::KEEP_RAW) {
    // the raw bf16 projections (all TN column tiles: gate and up interleaved
    // as W1's rows) to out2, through the same staging with 64 columns per
    // wave, before the activation overwrites the accumulators.  The kept
    // forwards go on to the hidden from the same accumulators: 188 us at
    // 32768 rows of ffn 2048, where the projections alone took 172 and a
    // hidden pass that read them back another 76.
    constexpr int CR = TN * 32;
    static_assert(CR == 64 && CR == CS, "raw staging of 64 columns per wave");
    uint32_t* rst = stage;
    auto rword = [](int kp, int c) -> int {
      const int b1 = (kp >> 1) & 1;
      const int ch = (c >> 2) ^ (kp & 1) ^ (b1 << 3);
      return kp * CR + ch * 4 + (c & 3);
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const int kp = i * 16 + (r >> 2) * 4 + (lane >> 5) * 2 + ((r & 3) >> 1);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          rst[rword(kp, j * 32 + col)] = mxm_pack_bf2_fast(acc[i][j][r], acc[i][j][r + 1]);
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint16_t* __restrict__ rout = static_cast<uint16_t*>(a.out2);
    constexpr int RSEGS = CR / 8;
#pragma unroll
    for (int it = 0; it < (WROWS / 2) * RSEGS / 64; ++it) {
      const int q = lane + 64 * it;
      const int kp = q / RSEGS, sg = q % RSEGS;
      const u32x4_t w0 = *reinterpret_cast<const u32x4_t*>(rst + rword(kp, sg * 8));
      const u32x4_t w1 = *reinterpret_cast<const u32x4_t*>(rst + rword(kp, sg * 8 + 4));
      const uint32_t wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
      u32x4_t lo, hi;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        lo[m] = __builtin_amdgcn_perm(wv[2 * m + 1], wv[2 * m], 0x05040100u);
        hi[m] = __builtin_amdgcn_perm(wv[2 * m + 1], wv[2 * m], 0x07060302u);
      }
      const int grow = wm * WROWS + 2 * kp;
      const int c0r = n0 + wn * CR + sg * 8;
      if (grow < rows)
        *reinterpret_cast<u32x4_t*>(rout + (size_t)(row0 + grow) * a.Ncols + c0r) = lo;
      if (grow + 1 < rows)
        *reinterpret_cast<u32x4_t*>(rout + (size_t)(row0 + grow + 1) * a.Ncols + c0r) = hi;
    }
    if constexpr (Epi<EPI>::RAW_ONLY) return;  // the backward's hidden-gradient product derives H
    // this wave's reads of the raw staging are complete
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
  // kinds whose hidden is fp32 store it as two bf16 planes (hi, then lo =
  // bf16(h - hi)) through the same staging, one plane after the other
  constexpr int NPLANE = H_SPLIT ? 2 : 1;
  if constexpr (H_SPLIT) {
    // the fp32 hidden, computed once in place: h overwrites the gate
    // accumulator (GLU) or the projection's (MLP), which are dead after it
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if constexpr (MODE == MXM_GEMM_GLU) {
#pragma unroll
          for (int pj = 0; pj < TN / 2; ++pj)
            acc[i][2 * pj][r] = mxm_hidden_fast<true>(
                Epi<EPI>::ETYPE, Epi<EPI>::ACT, a.slope, mxm_rbf_fast(acc[i][2 * pj][r]),
                mxm_rbf_fast(acc[i][2 * pj + 1][r]));
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j][r] = mxm_hidden_fast<true>(MXM_EXPERT_MLP, Epi<EPI>::ACT, a.slope, 0.0f,
                                                 mxm_rbf_fast(acc[i][j][r]));
        }
      }
  }
#pragma unroll
  for (int plane = 0; plane < NPLANE; ++plane) {
  if (plane > 0) {
    // this wave's reads of the previous plane's staging are complete
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const int kp = i * 16 + (r >> 2) * 4 + (lane >> 5) * 2 + ((r & 3) >> 1);
      if (MODE == MXM_GEMM_GLU) {
#pragma unroll
        for (int pj = 0; pj < TN / 2; ++pj) {
          float h[2];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            if constexpr (H_SPLIT) {  // h computed above; plane 1 holds h - bf16(h)
              h[q] = acc[i][2 * pj][r + q];
              if (plane == 1) h[q] = h[q] - mxm_rbf_fast(h[q]);
            } else {
              const float gg = mxm_rbf_fast(acc[i][2 * pj][r + q]);
              const float u = mxm_rbf_fast(acc[i][2 * pj + 1][r + q]);
              h[q] = mxm_hidden_fast<true>(Epi<EPI>::ETYPE, Epi<EPI>::ACT, a.slope, gg, u);
            }
          }
          stage[word_at(kp, pj * 32 + col)] = mxm_pack_bf2_fast(h[0], h[1]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float v[2];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            v[q] = acc[i][j][r + q];
            if constexpr (H_SPLIT) {  // h computed above
              if (plane == 1) v[q] = v[q] - mxm_rbf_fast(v[q]);
            } else if (MODE == MXM_GEMM_MLP) {
              v[q] = mxm_hidden_fast<true>(MXM_EXPERT_MLP, Epi<EPI>::ACT, a.slope, 0.0f,
                                           mxm_rbf_fast(v[q]));
            }
          }
          stage[word_at(kp, j * 32 + col)] = mxm_pack_bf2_fast(v[0], v[1]);
        }
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // each lane takes 8 columns of one row pair: two 16-byte chunks, split by
  // byte permutes into the even row's and the odd row's 16-byte segments
  const int hcols = (MODE == MXM_GEMM_GLU) ? a.Ncols / 2 : a.Ncols;  // F (up) or D (down)
  const int ldo = H_SPLIT ? 2 * hcols : hcols;
  const int c0 = n0 / (MODE == MXM_GEMM_GLU ? 2 : 1) + wn * C + plane * hcols;
  uint16_t* __restrict__ out = static_cast<uint16_t*>(a.out);
  constexpr int SEGS = C / 8;  // 8-column segments per row pair
  // (each plane computes its own addresses: kept from one to the next they
  // would spill)
  int ln = lane;
  if constexpr (H_SPLIT) asm volatile("" : "+v"(ln));
#pragma unroll
  for (int it = 0; it < (WROWS / 2) * SEGS / 64; ++it) {
    const int q = ln + 64 * it;
    const int kp = q / SEGS, sg = q % SEGS;
    const u32x4_t w0 = *reinterpret_cast<const u32x4_t*>(stage + word_at(kp, sg * 8));
    const u32x4_t w1 = *reinterpret_cast<const u32x4_t*>(stage + word_at(kp, sg * 8 + 4));
    const uint32_t wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
    u32x4_t lo, hi;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      lo[m] = __builtin_amdgcn_perm(wv[2 * m + 1], wv[2 * m], 0x05040100u);  // low halves
      hi[m] = __builtin_amdgcn_perm(wv[2 * m + 1], wv[2 * m], 0x07060302u);  // high halves
    }
    const int grow = wm * WROWS + 2 * kp;
    // Y (down projection) is read once, by the combine, and is several times
    // the last-level cache: stored nontemporal.  H stays cached for the down
    // GEMM's re-reads.
    u32x4_t* d0 = reinterpret_cast<u32x4_t*>(out + (size_t)(row0 + grow) * ldo + c0 + sg * 8);
    u32x4_t* d1 = reinterpret_cast<u32x4_t*>(out + (size_t)(row0 + grow + 1) * ldo + c0 + sg * 8);
    if constexpr (MODE == MXM_GEMM_DOWN) {
      if (grow < rows) __builtin_nontemporal_store(lo, d0);
      if (grow + 1 < rows) __builtin_nontemporal_store(hi, d1);
    } else {
      if (grow < rows) *d0 = lo;
      if (grow + 1 < rows) *d1 = hi;
    }
  }
  }  // plane loop
}

// ---- the scheduled kernel: 256 x 256 tiles, what is left in 128 x 128 ------
//
// A CU holds one 256 x 256 tile at a time, so a launch of T such tiles takes
// ceil(T / 256) rounds however few tiles the last one has, and an expert's
// last row tile costs a whole tile however few rows it has.  This kernel
// plans its own work from the experts' row counts: 256-row tiles where they
// are full or more than half full, 128 x 128 tiles (8 waves, four LDS stages
// of 64 k: the same 128 KB of LDS with three stages in flight instead of
// one) for an expert's last 128 rows or fewer, for the columns past a
// multiple of 256, and for the big tiles of a last round that would leave
// most CUs idle.  Every output is one tile's sum over k in ascending order
// whichever shape it falls in, so the plan changes no result.
//
// The plan is a function of the counts only, computed by every workgroup in
// LDS (prefixes over the experts of the big and the small row tiles), so it
// needs neither a launch before it nor a lookup in memory per tile.  Each XCD
// (workgroup L runs on XCD L % 8) takes an eighth of the big tiles (XcdPart),
// in groups of GM row tiles by all column tiles, then of the small ones; the
// workgroups that have one big tile fewer start the small ones.
//
// Measured against one tile shape per launch (16384 tokens of D 512 / E 8 / K
// 2 / ffn 2048): gate+up 163 -> 147 us, down (272 tiles of 256 x 256, or 1056
// of 128 x 128) 89 -> 72 us, 0.95 PFLOP/s of the 1.2 that this card reaches
// on a large dense product; 4096 tokens of D 2048 / E 64 / K 8 / ffn 1408
// gate+up 502 -> 455 us.
using BigTile = Tile<256, 256, 2, 4, 2, 2, 64>;
using SmallTile = Tile<128, 128, 2, 2, 2, 4, 64, 4>;
constexpr int SMALL_PER_BIG = 3;  // small tiles in the time of a big one

struct SchedLds {
  int big[MXM_MAX_EXPERTS + 1];    // first big row tile of expert e
  int small[MXM_MAX_EXPERTS + 1];  // first small row tile (an expert has one or none)
  int off[MXM_MAX_EXPERTS + 1];    // offsets
  int wsum[2][MXM_MAX_EXPERTS / 64];
};

// Inclusive prefix sum over the wave (lanes past a row's or the wave's start
// add 0): row shifts, then the rows' last lanes broadcast on.
__device__ __forceinline__ int wave_prefix(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return v;
}

// Prefixes of the experts' row tiles of BM rows: (count + rnd) / BM big ones,
// and a small one for rows left over (rnd = BM - 1 leaves none).
template <int BM>
__device__ __forceinline__ void sched_build(SchedLds& S, const int32_t* offsets, int E, int rnd) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  static_assert(MXM_MAX_EXPERTS % 64 == 0 && MXM_MAX_EXPERTS <= 256, "one expert per thread");
  const int o0 = tid < E ? offsets[tid] : 0;
  const int o1 = tid < E ? offsets[tid + 1] : 0;
  const int nb = (o1 - o0 + rnd) / BM, ns = o1 - o0 > nb * BM ? 1 : 0;
  int ib = wave_prefix(nb), is = wave_prefix(ns);
  if (lane == 63 && wave < MXM_MAX_EXPERTS / 64) {
    S.wsum[0][wave] = ib;
    S.wsum[1][wave] = is;
  }
  __syncthreads();
  if (tid < MXM_MAX_EXPERTS) {
    for (int w = 0; w < wave; ++w) {
      ib += S.wsum[0][w];
      is += S.wsum[1][w];
    }
    if (tid < E) {
      S.big[tid + 1] = ib;
      S.small[tid + 1] = is;
      S.off[tid + 1] = o1;
      if (tid == 0) S.big[0] = S.small[0] = S.off[0] = 0;
    }
  }
  __syncthreads();
}

// The expert of row tile t: the number of e in 1 .. E-1 with pre[e] <= t.
__device__ __forceinline__ int sched_find(const int* pre, int E, int t) {
  const int lane = threadIdx.x & 63;
  int e = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int i = e0 + lane + 1;
    e += __popcll(__ballot(i < E && pre[i] <= t));
  }
  return e;
}

// Row tile and column tile of place q in the list of a launch's tiles: groups
// of GM row tiles (of `nrow`), a group's `ncol` column tiles one after the
// other.
__device__ __forceinline__ void sched_place(int q, int nrow, int ncol, int& mt, int& nt) {
  const int g = q / (GM * ncol), rr = q - g * (GM * ncol);
  const int rig = min(GM, nrow - g * GM);
  mt = g * GM + rr % rig;
  nt = rr / rig;
}

// An XCD's part of a list of n tiles in groups of `chunk` (GM row tiles by all
// column tiles): every eighth group, so that at any time all XCDs work on the
// same few experts, whose weights then come from the last-level cache the second
// time; what is left past whole eights of groups in contiguous eighths, so that
// all CUs get the same number of tiles to within one.  (Contiguous eighths of
// the whole list keep eight experts' weights in use at once: forwards of 65536
// tokens of D 2048 / E 64 / K 8 / ffn 5468, 360 MB of them, 33.0 ms, 31.6 like
// this; 32768 of D 2048 / E 8 / K 2 / ffn 8192 6.14 -> 5.95.)
struct XcdPart {
  int xcd, chunk, whole, base, size;  // whole: tiles of this XCD in whole groups
  __device__ __forceinline__ XcdPart(int64_t n, int chunk_, int xcd_) : xcd(xcd_), chunk(chunk_) {
    const int eights = (int)(n / (8 * (int64_t)chunk));
    const int64_t rest = n - (int64_t)eights * 8 * chunk;
    const int lo = (int)(rest * xcd / 8);
    whole = eights * chunk;
    base = (int)(n - rest) + lo;
    size = whole + (int)(rest * (xcd + 1) / 8) - lo;
  }
  // place in the list of this XCD's tile p (< size)
  __device__ __forceinline__ int operator()(int p) const {
    if (p >= whole) return base + p - whole;
    const int g = p / chunk;
    return (g * 8 + xcd) * chunk + p - g * chunk;
  }
};

template <int EPI>
__global__ __launch_bounds__(512, 1) void gemm_sched_kernel(GemmArgs a, int whole) {
  static_assert(BigTile::NS * BigTile::BUF == SmallTile::NS * SmallTile::BUF &&
                    BigTile::NT == 512 && SmallTile::NT == 512,
                "both shapes share the ring and the workgroup");
  __shared__ u32x4_t lds[BigTile::NS * BigTile::BUF];
  __shared__ SchedLds S;
  const int E = a.E;
  // whole: 256 x 256 tiles only (Ncols a multiple of 256)
  sched_build<256>(S, a.offsets, E, whole ? 255 : 127);
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int BR = uni(S.big[E]), SR = uni(S.small[E]);
  const int ncb = a.Ncols / 256, ncs = a.Ncols / 128;  // column tiles
  const int G = gridDim.x;
  // big tiles B, small tiles S0 whatever becomes of the last round; that
  // round's `rem` big tiles are cut in four each where all the small tiles
  // then take fewer rounds of CUs than the two kinds apart
  const int B = BR * ncb;
  const int S0 = SR * ncs + (ncs & 1) * 2 * BR;
  const int rem = B % G;
  int Bm = B;
  if (!whole && rem > 0) {
    const int cut = (4 * rem + S0 + G - 1) / G;
    const int left = max(0, S0 - (G - rem) * SMALL_PER_BIG);
    const int keep = SMALL_PER_BIG + (left + G - 1) / G;
    if (cut < keep) Bm = B - rem;
  }
  const int Ns = S0 + 4 * (B - Bm);
  // this XCD's part of both lists, and this workgroup's place in it
  const int xcd = blockIdx.x & 7, s = blockIdx.x >> 3, W = G >> 3;
  const XcdPart part(Bm, GM * max(ncb, 1), xcd);
  const int slo = (int)((int64_t)Ns * xcd / 8), sn = (int)((int64_t)Ns * (xcd + 1) / 8) - slo;
  bool first = true;
  for (int p = s; p < part.size; p += W) {
    // every wave has read the previous tile's epilogue staging out of LDS
    // (plain s_barrier: no wait for that epilogue's stores)
    if (!first) asm volatile("s_barrier" ::: "memory");
    first = false;
    int mt, nt;
    sched_place(part(p), BR, ncb, mt, nt);
    const int e = uni(sched_find(S.big, E, mt));
    const int row0 = uni(S.off[e] + (mt - S.big[e]) * 256);
    const int rows = min(256, uni(S.off[e + 1]) - row0);
    gemm_tile<BigTile, 256, 256, 2, 4, EPI>(a, lds, e, row0, rows, nt * 256);
  }
  if (whole) return;
  const int odd = part.size % W;              // workgroups with one big tile more
  const int idle = odd > 0 ? W - odd : 0;     // ... and the rest, which start
  const int ahead = SMALL_PER_BIG * idle;
  for (int k = (idle > 0 && s >= odd) ? 0 : SMALL_PER_BIG;; ++k) {
    const int i = k < SMALL_PER_BIG ? s - odd + k * idle : ahead + s + (k - SMALL_PER_BIG) * W;
    if (i >= sn) {
      if (k < SMALL_PER_BIG) continue;
      break;
    }
    if (!first) asm volatile("s_barrier" ::: "memory");
    first = false;
    int t = slo + i, e, row0, rows, n0;
    if (t < SR * ncs) {
      // an expert's last rows
      const int sr = t / ncs;
      e = uni(sched_find(S.small, E, sr));
      row0 = uni(S.off[e] + (S.big[e + 1] - S.big[e]) * 256);
      rows = uni(S.off[e + 1]) - row0;
      n0 = (t - sr * ncs) * 128;
    } else {
      int mt, half;
      if (t < S0) {
        // the last 128 columns of the big row tiles
        t -= SR * ncs;
        mt = t >> 1;
        half = t & 1;
        n0 = ncb * 256;
      } else {
        // a quarter of a big tile of the last round
        t -= S0;
        int nt;
        sched_place(Bm + (t >> 2), BR, ncb, mt, nt);
        half = (t >> 1) & 1;
        n0 = nt * 256 + (t & 1) * 128;
      }
      e = uni(sched_find(S.big, E, mt));
      row0 = uni(S.off[e] + (mt - S.big[e]) * 256) + half * 128;
      rows = min(128, uni(S.off[e + 1]) - row0);
    }
    gemm_tile<SmallTile, 128, 128, 2, 2, EPI>(a, lds, e, row0, rows, n0);
  }
}

// Tiles of one shape, two workgroups of 4 waves on a CU: the requested
// families, and launches of up to two 128 x 128 tiles per CU, whose second
// round of single tiles would leave most CUs idle on the kernel above.
template <class TL, int BM, int BN, int WM, int WN, int EPI>
__global__ __launch_bounds__(TL::NT, TL::WPS * 256 / TL::NT) void gemm_kernel(GemmArgs a) {
  __shared__ u32x4_t lds[TL::NS * TL::BUF];
  __shared__ SchedLds S;
  const int E = a.E, lane = threadIdx.x & 63;
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  // up to 64 experts: their row tiles in each wave's lanes (lane e: expert e),
  // so that a tile's rows are known without LDS or a barrier.  These launches
  // are often short, and what stands before the first load is part of each:
  // 200 tokens of D 192 / E 4 / K 2 / ffn 256, 6.4 and 7.1 us for the two
  // products from LDS prefixes with the whole device's workgroups launched,
  // 5.7 and 5.7 like this with tile_grid's.
  const bool lanes = E <= 64;
  int o0 = 0, o1 = 0, pre = 0;
  if (lanes) {
    if (lane < E) {
      o0 = a.offsets[lane];
      o1 = a.offsets[lane + 1];
    }
    pre = wave_prefix((o1 - o0 + BM - 1) / BM);
  } else {
    sched_build<BM>(S, a.offsets, E, BM - 1);
  }
  const int BR = lanes ? __builtin_amdgcn_readlane(pre, 63) : uni(S.big[E]);
  const int ncol = a.Ncols / BN;
  const int64_t T = (int64_t)BR * ncol;
  const int xcd = blockIdx.x & 7, s = blockIdx.x >> 3, W = gridDim.x >> 3;
  const XcdPart part(T, GM * ncol, xcd);
  for (int p = s; p < part.size; p += W) {
    if (p != s) asm volatile("s_barrier" ::: "memory");  // as above
    int mt, nt;
    sched_place(part(p), BR, ncol, mt, nt);
    int e, row0, rend;
    if (lanes) {
      e = __popcll(__ballot(pre <= mt));  // (lanes past E hold BR > mt)
      row0 = __builtin_amdgcn_readlane(o0, e) +
             (mt - (e > 0 ? __builtin_amdgcn_readlane(pre, e - 1) : 0)) * BM;
      rend = __builtin_amdgcn_readlane(o1, e);
    } else {
      e = uni(sched_find(S.big, E, mt));
      row0 = uni(S.off[e] + (mt - S.big[e]) * BM);
      rend = uni(S.off[e + 1]);
    }
    gemm_tile<TL, BM, BN, WM, WN, EPI>(a, lds, e, row0, min(BM, rend - row0), nt * BN);
  }
}

// Workgroups resident at once on the current device: CUs x workgroups per
// CU, rounded down to a multiple of 8 so a workgroup's tiles all map to the
// XCD it runs on.
static int persistent_grid(int per_cu) {
  static int ncu[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (ncu[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    ncu[dev] = n;
  }
  return std::max(8, ncu[dev] * per_cu / 8 * 8);
}

// ... but no more workgroups than the launch can have tiles (an expert's last
// tile may be partial), in eights for the XCDs.
static int tile_grid(const GemmArgs& a, int per_cu, int bm, int bn) {
  const int64_t row_tiles = a.rows_total / bm + std::min(a.E, a.rows_total);
  const int64_t tiles = row_tiles * ((a.Ncols + bn - 1) / bn);
  return (int)std::min<int64_t>(persistent_grid(per_cu), (tiles + 7) / 8 * 8);
}

// Calls f with the hidden activation's kind of these arguments as a constant.
template <class F>
void with_kind(const GemmArgs& a, F&& f) {
  switch (mxm_epi_kind(a.expert_type, a.activation)) {
    case EPI_GEGLU:
      return f(std::integral_constant<int, EPI_GEGLU>{});
    case EPI_MLP_SILU:
      return f(std::integral_constant<int, EPI_MLP_SILU>{});
    case EPI_MLP_GELU:
      return f(std::integral_constant<int, EPI_MLP_GELU>{});
    case EPI_MLP_RELU:
      return f(std::integral_constant<int, EPI_MLP_RELU>{});
    case EPI_MLP_LEAKY:
      return f(std::integral_constant<int, EPI_MLP_LEAKY>{});
    default:
      return f(std::integral_constant<int, EPI_SWIGLU>{});
  }
}

// Calls f with the epilogue kind of these arguments as a constant: an up
// projection may keep its raw projections (GemmArgs::out2), and weights may
// be int8 integers with per-column scales (scale0).
template <class F>
void with_epi(const GemmArgs& a, F&& f) {
  auto up = [&](auto kind) {
    constexpr int K = decltype(kind)::value;
    if (a.out2 && a.out)
      f(std::integral_constant<int, EPI_KEEP_H + K>{});
    else if (a.out2)
      f(std::integral_constant<int, EPI_KEEP + K>{});
    else if (a.scale0)
      f(std::integral_constant<int, EPI_SCALE + K>{});
    else
      f(kind);
  };
  if (a.mode == MXM_GEMM_DOWN) {
    if (a.scale0 && a.h_split)
      f(std::integral_constant<int, EPI_SCALE + EPI_DOWN_F32>{});
    else if (a.scale0)
      f(std::integral_constant<int, EPI_SCALE + EPI_DOWN>{});
    else if (a.h_split)
      f(std::integral_constant<int, EPI_DOWN_F32>{});
    else if (a.f32_out)
      f(std::integral_constant<int, EPI_F32>{});
    else if (a.abw.dgu)
      with_kind(a, [&](auto kind) {
        f(std::integral_constant<int, EPI_ACT_BW + decltype(kind)::value>{});
      });
    else
      f(std::integral_constant<int, EPI_DOWN>{});
    return;
  }
  with_kind(a, up);
}

template <int BM, int BN, int WM, int WN, int WPS, int NSTG, int BKK>
void launch_family(const GemmArgs& a, hipStream_t s) {
  using TL = Tile<BM, BN, WM, WN, WPS, NSTG, BKK>;
  // workgroups per CU: what the launch bounds allow, capped by LDS
  constexpr int lds_bytes = NSTG * TL::BUF * 16 + (int)sizeof(SchedLds);
  constexpr int per_cu = std::min(TL::WPS * 256 / TL::NT, 160 * 1024 / lds_bytes);
  static_assert(per_cu == 2, "two workgroups per CU");
  with_epi(a, [&](auto epi) {
    hipLaunchKernelGGL((gemm_kernel<TL, BM, BN, WM, WN, decltype(epi)::value>),
                       dim3(tile_grid(a, per_cu, BM, BN)), dim3(TL::NT), 0, s, a);
  });
}

// The scheduled kernel: one workgroup per CU, or per 128 x 128 tile (its list
// is no longer than theirs).  whole: 256 x 256 tiles only.
void launch_sched(const GemmArgs& a, hipStream_t s, int whole) {
  with_epi(a, [&](auto epi) {
    hipLaunchKernelGGL((gemm_sched_kernel<decltype(epi)::value>),
                       dim3(tile_grid(a, 1, 128, 128)), dim3(512), 0, s, a, whole);
  });
}

}  // namespace

int mxm_mfma_tile_rows(int Ncols, int Kd, int family) {
  if (Kd % 64 != 0) return 0;
  // B loads address one expert's matrix with 32-bit byte offsets
  if ((size_t)Ncols * Kd * 2 >= ((size_t)1 << 32)) return 0;
  const bool f256 = Ncols % 256 == 0, f128 = Ncols % 128 == 0;
  switch (family) {
    case MXM_TILE_256x128:
      return f128 ? 256 : 0;
    case MXM_TILE_128x128:
      return f128 ? 128 : 0;
    case MXM_TILE_256x256:
      return f256 ? 256 : 0;
    default:  // auto and the scheduled kernel
      return f256 ? 256 : f128 ? 128 : 0;
  }
}

int mxm_mfma_family(int rows, int E, int Ncols, int Kd, int family) {
  if (family != MXM_TILE_AUTO) return family;
  // 128 x 128 tiles of a launch with evenly loaded experts, the last tile
  // of each half full.  Between one and two of them per CU the pairs run
  // them in one round (2000 tokens of D 1024 / E 16 / K 2 / ffn 2734, down:
  // 312 tiles 43 us, 48 on the scheduled kernel; 6000 of D 512 / E 16 / ffn
  // 1024: 407 tiles 17.2 / 20.2 us); below, the scheduled kernel's deeper
  // ring is faster (219 tiles of 64 stages: 48 / 34 us), above, its big
  // tiles (527: 29.7 / 26.8, 1040: 85 / 71).  A pair also overlaps one
  // tile's epilogue with the other's products, which counts where tiles
  // have few stages (6 and fewer: 20000 tokens of D 256, up 36.0 / 38.3 us,
  // 12000 of D 384 52.4 / 54.9; at 8 stages 161 / 147), and 128 columns
  // hold no big tile (23433 tokens, D 128: 15.7 / 18.5 us).
  const int64_t tiles = ((int64_t)rows + 64 * (int64_t)E) / 128 * (Ncols / 128);
  const int n_cu = persistent_grid(1);
  return Ncols < 256 || Kd <= 384 || (tiles > n_cu && tiles <= 2 * n_cu) ? MXM_TILE_128x128
                                                                        : MXM_TILE_AUTO;
}

void mxm_launch_gemm_mfma(const GemmArgs& args, hipStream_t s) {
  if (args.rows_total <= 0) return;
  GemmArgs a = args;
  a.a_off32 = !a.no_off32 && (size_t)a.rows_total * a.Kd * 2 < ((size_t)1 << 32);
  switch (mxm_mfma_family(a.rows_total, a.E, a.Ncols, a.Kd, a.family)) {
    case MXM_TILE_256x128:
      launch_family<256, 128, 2, 2, 2, 3, 32>(a, s);
      break;
    case MXM_TILE_128x128:
      launch_family<128, 128, 2, 2, 2, 2, 64>(a, s);
      break;
    case MXM_TILE_256x256:
      launch_sched(a, s, 1);
      break;
    default:
      launch_sched(a, s, 0);
      break;
  }
}
