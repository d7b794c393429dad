// dsv_lmhead.hip — lm_head fused with the acceptance statistics, on gfx950.
//
// The target's logits for the tree nodes are lm_head(hidden) = hidden . W^T
// ([R, Dm] x [V, Dm]^T, bf16 in, fp32 accumulate, bf16 out: the reference's
// self.base_model.lm_head, draft/diffspec_model.py:229-231, whose [M, V]
// output verify_new reduces with argmax, draft/tree_verification.py:100-102).
// Here the logits never reach HBM unless asked for: each workgroup computes a
// 256-row slice of the vocabulary for all (up to 256) hidden rows, rounds every
// logit to bf16 exactly as the reference's bf16 logits are, and reduces its
// slice to the acceptance statistics of kernel 4 (argmax with the lowest index
// on ties; softmax (m, l, s) for typical acceptance) per hidden row.  A
// combine kernel and the tree walk of kernel 4 follow.
//
// The operation streams W (V * Dm * 2 bytes, 1.05 GB for Llama-3.1-8B) once
// per pass of up to 256 hidden rows and is HBM-bound: 64 flop per byte at 64
// rows, a fifth of the MFMA ridge.  A pass per 64 rows read W three times for
// three trees of 64 nodes: 590 us against 304 us in one pass (128256 x 4096,
// whole call); 256 rows 780 -> 338 us.  Layout per workgroup:
//   * up to 64 hidden rows: 4 waves of two 32-row vocabulary blocks each, two
//     workgroups per CU (215 us at 64 rows, 5 TB/s).  More rows: 8 waves of
//     one block each, so that the accumulators (16 registers per 32 rows) leave
//     two waves per SIMD; with 4 waves at one per SIMD the loads' issue, the
//     LDS reads and the MFMAs of a step do not overlap (374 against 344 us at
//     256 rows).  The A operand comes straight from HBM into registers, up to
//     three steps of 64 elements of Dm in flight ahead of the MFMAs;
//   * the hidden rows (B operand, 64 elements per step) are staged once per
//     workgroup through a double-buffered LDS tile;
//   * v_mfma_f32_32x32x16_bf16.  MFMA sub-step j of a step covers elements
//     [16j, 16j + 16) of the step's 64: lanes 0-31 hold the first 8, lanes
//     32-63 the next 8, the same on A and B, so one load instruction reads 32
//     contiguous bytes of each of 32 W rows (the four sub-steps of a row
//     share its cache line, so these loads must not be non-temporal: 315 ->
//     406 us at 192 rows);
//   * workgroups start their sweep over Dm at different steps (a rotation),
//     which spreads their concurrent W reads over the memory channels.
// Hidden rows beyond R are zero; vocabulary rows beyond V are clamped loads
// whose results are dropped.

#include <algorithm>

#include "dsv_internal.h"
#include "dsv_stats.h"

namespace dsv {

namespace {

constexpr int kKB = 2 * kLmK;                        // bytes of one row per step
constexpr int kHStride = kKB + 16;                   // LDS step tile: bytes per hidden row
constexpr int kTStride = 2 * kLmVocab + 16;          // LDS logits tile: bytes per hidden row
constexpr int kHChunks = kKB / 64;                   // 16-byte chunks a thread stages per step and row group
constexpr int kQ = kLmVocab / 4;                     // vocabulary rows per statistics thread
constexpr float kNegInfL = -__builtin_huge_valf();
constexpr float kLog2eL = 1.4426950408889634074f;
static_assert(kQ % 8 == 0, "statistics read 16-byte chunks");

template <int V>
struct IC {
  static constexpr int value = V;
};

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                 0, 0, 0);
}

__device__ __forceinline__ uint32_t bf16_rne(float x) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x);
}

// Threads of a workgroup: four waves of two vocabulary blocks each for up to 64
// hidden rows (two workgroups per CU), eight waves of one block each beyond.
constexpr int lm_threads(int cb) { return cb <= 2 ? 256 : 512; }

// CB: 32-row blocks of hidden rows per workgroup (its rows: 32 * CB).
template <bool TYPICAL, int CB>
__global__ void __launch_bounds__(lm_threads(CB), 2) lmhead_stats_kernel(const LmArgs a) {
  constexpr int KS = kLmKS, NT = lm_threads(CB);
  constexpr int RB = kLmVocab / 32 / (NT / 64);        // 32-row vocabulary blocks per wave
  constexpr int kRows = 32 * CB;
  constexpr int RG = NT / 4;                           // hidden rows of a group (four threads each)
  constexpr int HG = (kRows + RG - 1) / RG;            // groups (staging, statistics)
  constexpr int NB = CB <= 2 ? 3 : 4;                  // W register buffers
  constexpr int HD = CB <= 2 ? 1 : 2;                  // steps from a hidden row's load to its use
  constexpr int kHBytes = kRows * kHStride;            // one step tile
  constexpr int kSmem = (2 * kHBytes > kRows * kTStride) ? 2 * kHBytes : kRows * kTStride;
  static_assert(kSmem <= 160 * 1024, "LDS of a CU");
  __shared__ __align__(16) uint8_t smem[kSmem];
  uint8_t* const hb0 = smem;
  uint8_t* const hb1 = smem + kHBytes;

  const int tid = threadIdx.x, wid = tid >> 6, lane = tid & 63, lj = lane & 31, lg = lane >> 5;
  const int blk = blockIdx.x;
  const int64_t v0 = (int64_t)blk * kLmVocab;
  const int r0 = blockIdx.y * kRows;
  const int S = a.Dm / kLmK;

  // This lane's W rows (clamped into the vocabulary).  MFMA sub-step j of a
  // step covers elements [16j, 16j + 16): lanes 0-31 the first 8, lanes
  // 32-63 the next 8 (the operand layout of v_mfma_f32_32x32x16), so a load
  // instruction reads 32 contiguous bytes of each of 32 rows.
  const uint16_t* wrow[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    int64_t v = v0 + (wid * RB + rb) * 32 + lj;
    v = v < a.V ? v : a.V - 1;
    wrow[rb] = a.w + v * a.ldw + lg * 8;
  }
  // Hidden-row staging: thread -> (row hr, part hc) of a step.
  // (of row group g: row RG g + hr)
  const int hr = tid >> 2, hc = tid & 3;
  bool hin[HG], hvalid[HG];  // row in the tile; row below R
  const uint16_t* hrow[HG];
#pragma unroll
  for (int g = 0; g < HG; ++g) {
    hin[g] = RG * g + hr < kRows;
    hvalid[g] = hin[g] && r0 + RG * g + hr < a.R;
    hrow[g] = a.h + (int64_t)min(r0 + RG * g + hr, a.R - 1) * a.ldh + hc * (kLmK / 4);
  }

  u32x4 wb[NB][RB][KS];
  u32x4 hreg[HD][HG][kHChunks];
  f32x16 acc[RB][CB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = f32x16{};

  // Workgroups start the reduction at different steps (the sum is taken in a
  // rotated order): at any moment they read different columns of W, whose
  // rows are 2*Dm bytes apart, so the reads spread over the memory channels
  // instead of all landing on the same address bits.
  const int rot = (int)(((int64_t)blk * 7) % S);
  auto col = [&](int s) -> int64_t {
    int x = min(s, S - 1) + rot;
    if (x >= S) x -= S;
    return (int64_t)x * kLmK;
  };
  // Loads past the last step re-read the last one (an L2 hit), so every step
  // issues the same loads and the compiler's wait counts stay exact.
  auto load_w = [&](auto buf_c, int s) {
    constexpr int b = decltype(buf_c)::value;
    const int64_t off = col(s);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int j = 0; j < KS; ++j) wb[b][rb][j] = *reinterpret_cast<const u32x4*>(wrow[rb] + off + 16 * j);
  };
  auto load_h = [&](auto buf_c, int s) {
    constexpr int b = decltype(buf_c)::value;
    const int64_t off = col(s);
#pragma unroll
    for (int g = 0; g < HG; ++g)
#pragma unroll
      for (int c = 0; c < kHChunks; ++c) hreg[b][g][c] = *reinterpret_cast<const u32x4*>(hrow[g] + off + 8 * c);
  };
  // Rows beyond R stay zero in both buffers (written once below).
  auto store_h = [&](auto buf_c, int s) {
    constexpr int b = decltype(buf_c)::value;
    uint8_t* dst = ((s & 1) ? hb1 : hb0) + hr * kHStride + hc * (kKB / 4);
#pragma unroll
    for (int g = 0; g < HG; ++g)
      if (hvalid[g]) {
#pragma unroll
        for (int c = 0; c < kHChunks; ++c) *reinterpret_cast<u32x4*>(dst + g * RG * kHStride + 16 * c) = hreg[b][g][c];
      }
  };

  // Step s (W buffer b = s mod NB): the loads of h(s+HD) and W(s+NB-1) issued,
  // MFMAs on W(s) and h(s) (its B operands read from LDS ahead of them), h(s+1)
  // into the other LDS buffer, one barrier.  Loads complete in order: with HD =
  // 2, h(s+1) was issued a step earlier, so the wait for it leaves W(s+2),
  // h(s+2) and W(s+3) in flight; with HD = 1 it drains all W but the newest
  // step, which two workgroups per CU hide (64 rows: 3% faster than HD = 2 and
  // four W buffers).
  auto step = [&](auto buf_c, int s) {
    constexpr int b = decltype(buf_c)::value;
    const uint8_t* hb = (s & 1) ? hb1 : hb0;
    if constexpr (CB <= 2) {
      // All of the step's B operands at once, a row block's sub-steps together;
      // products of one vocabulary block after the other.  Sub-steps read one by
      // one and hidden rows outside vocabulary blocks, as for larger CB, moves a
      // wait for the hidden rows out of the branch that waves of rows beyond R
      // skip: 16 rows, 50257 x 4096, 99.6 against 91.7 us a call, 32000 x 4096
      // 87.1 against 81.6; 64 rows 1%.
      u32x4 bf[CB][KS];
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int j = 0; j < KS; ++j)
          bf[cb][j] = *reinterpret_cast<const u32x4*>(hb + (cb * 32 + lj) * kHStride + lg * 16 + 32 * j);
      load_h(IC<b % HD>{}, s + HD);
      load_w(IC<(b + NB - 1) % NB>{}, s + NB - 1);
#pragma unroll
      for (int j = 0; j < KS; ++j)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mfma_bf16(wb[b][rb][j], bf[cb][j], acc[rb][cb]);
    } else {
      // B operands read one sub-step ahead up to CB = 6; the registers of
      // larger CB do not hold two sub-steps'.
      constexpr int PF = CB <= 6 ? 1 : 0;
      u32x4 bf[PF + 1][CB];
      auto read_b = [&](int j) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
          bf[j & PF][cb] = *reinterpret_cast<const u32x4*>(hb + (cb * 32 + lj) * kHStride + lg * 16 + 32 * j);
      };
#pragma unroll
      for (int j = 0; j < PF; ++j) read_b(j);
      load_h(IC<b % HD>{}, s + HD);
      load_w(IC<(b + NB - 1) % NB>{}, s + NB - 1);
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        if (j + PF < KS) read_b(j + PF);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb) acc[rb][cb] = mfma_bf16(wb[b][rb][j], bf[j & PF][cb], acc[rb][cb]);
      }
    }
    // The wait for h(s+1) stays behind the MFMAs.
    __builtin_amdgcn_sched_barrier(0);
    store_h(IC<(b + 1) % HD>{}, s + 1);
    __syncthreads();
  };

  load_h(IC<0>{}, 0);
  load_w(IC<0>{}, 0);
  if constexpr (HD == 2) load_h(IC<1>{}, 1);
  load_w(IC<1>{}, 1);
  if constexpr (NB == 4) load_w(IC<2>{}, 2);
#pragma unroll
  for (int g = 0; g < HG; ++g)
    if (hin[g] && !hvalid[g]) {
      const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        uint8_t* dst = (x ? hb1 : hb0) + (RG * g + hr) * kHStride + hc * (kKB / 4);
#pragma unroll
        for (int c = 0; c < kHChunks; ++c) *reinterpret_cast<u32x4*>(dst + 16 * c) = z;
      }
    }
  store_h(IC<0>{}, 0);
  __syncthreads();
  // NB steps per iteration (one per W register buffer), no conditions in
  // the body; the last S % NB steps follow.
  int s = 0;
  for (; s + NB <= S; s += NB) {
    step(IC<0>{}, s);
    step(IC<1>{}, s + 1);
    step(IC<2>{}, s + 2);
    if constexpr (NB == 4) step(IC<3>{}, s + 3);
  }
  if (s < S) step(IC<0>{}, s);
  if (s + 1 < S) step(IC<1>{}, s + 1);
  if (NB == 4 && s + 2 < S) step(IC<2>{}, s + 2);

  // ---- logits tile in LDS: [hidden row][vocab] bf16 (RNE, as the reference's
  // bf16 logits) ---------------------------------------------------------------------
  // Accumulator value e of block (rb, cb) holds vocab row
  // 32*(wid*RB + rb) + 8*(e/4) + 4*lg + e%4 and hidden row cb*32 + lj.
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x16 x = acc[rb][cb];
        const u32x2 val = {bf16_rne(x[4 * q4]) | (bf16_rne(x[4 * q4 + 1]) << 16),
                           bf16_rne(x[4 * q4 + 2]) | (bf16_rne(x[4 * q4 + 3]) << 16)};
        const int vv = (wid * RB + rb) * 32 + 8 * q4 + 4 * lg;
        *reinterpret_cast<u32x2*>(smem + (cb * 32 + lj) * kTStride + vv * 2) = val;
      }
  __syncthreads();

  // ---- statistics: thread (hidden row j of a row group, quarter q) over kQ vocab rows
#pragma unroll 1
  for (int jg = 0; jg < HG; ++jg) {
    const int j = RG * jg + (tid >> 2), q = tid & 3;
    if (kRows % RG != 0 && j >= kRows) break;  // (whole waves: kRows is a multiple of 32)
    const int row = r0 + j;
    const int64_t vq = v0 + q * kQ;
    const uint8_t* tr = smem + j * kTStride + q * (2 * kQ);
    ArgMax best{kNegInfL, 0x7fffffff};
    bool have = false;
    Soft sm{kNegInfL, 0.f, 0.f};
    const float zs = a.inv_temp * kLog2eL;
    float xs[kQ];
#pragma unroll
    for (int c = 0; c < kQ / 8; ++c) {
      const u32x4 w4 = *reinterpret_cast<const u32x4*>(tr + 16 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        xs[8 * c + 2 * e] = __uint_as_float(w4[e] << 16);
        xs[8 * c + 2 * e + 1] = __uint_as_float(w4[e] & 0xffff0000u);
      }
    }
    const int nv = (int)min<int64_t>(kQ, a.V - vq);  // valid vocab rows of this quarter (may be <= 0)
    float vmax = kNegInfL;
#pragma unroll
    for (int e = 0; e < kQ; ++e) {
      if (e < nv) {
        if (!have || am_better(xs[e], (int)(vq + e), best.v, best.i)) {
          best.v = xs[e];
          best.i = (int)(vq + e);
          have = true;
        }
        if constexpr (TYPICAL) vmax = fmaxf(vmax, xs[e] * zs);
      }
    }
    if constexpr (TYPICAL) {
      if (vmax != kNegInfL) {
        sm.m = vmax;
#pragma unroll
        for (int e = 0; e < kQ; ++e) {
          if (e < nv) {
            const float p = __builtin_amdgcn_exp2f(fmaf(xs[e], zs, -sm.m));
            sm.l += p;
            // 0 log 0 = 0: a -inf logit (p = 0) adds nothing to s.
            if (p > 0.f) sm.s = fmaf(xs[e] * a.inv_temp, p, sm.s);
          }
        }
      }
    }
    // The four quarters of a row are adjacent lanes.
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) {
      const float ov = __shfl_xor(best.v, o);
      const int oi = __shfl_xor(best.i, o);
      const int oh = __shfl_xor((int)have, o);
      if (oh && (!have || am_better(ov, oi, best.v, best.i))) {
        best.v = ov;
        best.i = oi;
        have = true;
      }
      if constexpr (TYPICAL) {
        Soft other{__shfl_xor(sm.m, o), __shfl_xor(sm.l, o), __shfl_xor(sm.s, o)};
        sm = soft_merge(sm, other);
      }
    }
    if (q == 0 && row < a.R) {
      const int64_t o = (int64_t)row * a.nblk + blk;
      a.rstat[o] = make_float4(best.v, __int_as_float(have ? best.i : -1), sm.m, sm.l);
      if constexpr (TYPICAL) a.rstat2[o] = sm.s;
    }

    // ---- optional logits output [R, V] ------------------------------------------------
    if (a.lout != nullptr && row < a.R && nv > 0) {
      uint16_t* dst = a.lout + (int64_t)row * a.lo_sr + vq;
      const uint16_t* src = reinterpret_cast<const uint16_t*>(tr);
      if (nv == kQ && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
#pragma unroll
        for (int c = 0; c < kQ / 8; ++c) reinterpret_cast<u32x4*>(dst)[c] = reinterpret_cast<const u32x4*>(src)[c];
      } else {
        for (int e = 0; e < nv; ++e) dst[e] = src[e];
      }
    }
  }

  // ---- typical: each node's draft-token logit under its parent --------------------
  // Node i of tree t (hidden row t*M + i) needs logit[t*M + parent(i)][draft(i)];
  // the workgroup that holds both that hidden row and that vocabulary row
  // writes it.  parent(i) follows the walk: verify_new's parent_ext
  // (draft/tree_verification.py:120-125), malformed entries mapped to the
  // root (the walk flags them itself).
  if constexpr (TYPICAL) {
    for (int rho = tid; rho < a.R; rho += NT) {
      const int t = rho / a.M, i = rho - t * a.M;
      if (i == 0) continue;
      int64_t p = a.parent[(int64_t)t * a.p_st + (int64_t)(i - 1) * a.p_sm];
      if (p == i - 1) p = -1;
      if (p < -1 || p >= a.M - 1) p = -1;
      const int prow = t * a.M + (int)p + 1 - r0;
      const int64_t tok = a.draft[(int64_t)t * a.d_st + (int64_t)i * a.d_sm];
      if (prow >= 0 && prow < kRows && tok >= v0 && tok < v0 + kLmVocab && tok < a.V) {
        const uint16_t bits = *reinterpret_cast<const uint16_t*>(smem + prow * kTStride + (tok - v0) * 2);
        a.xtok[rho] = __uint_as_float((uint32_t)bits << 16);
      }
    }
  }
}

template <int CB>
hipError_t launch_stats(const LmArgs& lm, hipStream_t s) {
  const dim3 grid((unsigned)lm.nblk, (unsigned)((lm.R + 32 * CB - 1) / (32 * CB))), block(lm_threads(CB));
  if (lm.mode == 1)
    hipLaunchKernelGGL((lmhead_stats_kernel<true, CB>), grid, block, 0, s, lm);
  else
    hipLaunchKernelGGL((lmhead_stats_kernel<false, CB>), grid, block, 0, s, lm);
  return hipGetLastError();
}

}  // namespace

int lmhead_blocks(int64_t V) { return (int)((V + kLmVocab - 1) / kLmVocab); }

hipError_t launch_lmhead_accept(const AcceptArgs& acc, const LmArgs& lm, hipStream_t s) {
  if (lm.R <= 0) return hipSuccess;
  // Passes over W: as few as 256 rows each allow, but where the vocabulary
  // slices leave half of the CUs idle, as many as fill them (they run at the same
  // time and share W through the caches): 125 slices (32000 x 4096), 256 rows,
  // one pass 142 us, two 124 us; 197 slices, 192 rows, one pass 151 us, two
  // 227 us.  Rows of a pass: the next of 64, 128, 192, 256.
  const int nrb = (lm.R + 31) / 32, cus = acc.cus > 0 ? acc.cus : 256;
  int passes = (nrb + 7) / 8;
  if (2 * lm.nblk <= cus) passes = std::max(passes, std::min(cus / lm.nblk, (nrb + 1) / 2));
  const int cb = (nrb + passes - 1) / passes;
  hipError_t e = cb <= 2   ? launch_stats<2>(lm, s)
                 : cb <= 4 ? launch_stats<4>(lm, s)
                 : cb <= 6 ? launch_stats<6>(lm, s)
                           : launch_stats<8>(lm, s);
  if (e != hipSuccess) return e;
  return launch_accept_from_parts(acc, lm.rstat, lm.rstat2, lm.nblk, s);
}

}  // namespace dsv
