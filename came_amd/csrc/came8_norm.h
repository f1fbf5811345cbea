// The clip's update norm in the reference's own summation order, computed in parallel.
//
// The reference clips the update by its RMS, u.norm(2) / sqrt(N) (came_pytorch/CAME8bitFull.py:121-122,
// 1032).  On CPU, torch sums a contiguous fp32 tensor's squares for norm(2) in one thread as eight
// interleaved accumulators, acc[i % 8] = fma(u_i, u_i, acc[i % 8]) over the first N - N % 8 elements,
// then acc[0] + acc[1] + ... + acc[7] left to right, then the N % 8 remaining elements: when four or
// more remain, the next four as rounded squares added one at a time, b = (b + RN(u*u)), then the last
// N % 4 as fused multiply-adds, b = fma(u, u, b); then a correctly rounded sqrt.  Each accumulator is a serial chain of up to
// N / 8 dependent fused multiply-adds (16.4 M for a 32000 x 4096 matrix); its rounding errors are
// part of the result (about 1.5% of the norm at that size), so the exact chain has to be replayed.
//
// Replay without the serial dependence.  While a chain's value s stays inside one binade
// [2^E, 2^(E+1)) (E = -126 also covers the subnormals) it is m * 2^(E-23) with an integer m < 2^24,
// and fma(x, x, s) = (m + n) * 2^(E-23) with n = round(x^2 * 2^(23-E)), provided m + n < 2^24 and
// x^2 * 2^(23-E) is not a half-integer: the exact sum then lies strictly inside the binade, whose
// floats are exactly the multiples of 2^(E-23).  So inside a binade the chain is an integer sum of
// per-element increments that do not depend on s.  An element whose increment is not determined this
// way is "special": its square is a half-integer after scaling (a tie, whose rounding depends on m's
// parity), or infinite or NaN; an element whose increment takes the chain out of the binade ends the
// run of known increments.  The increments are formed by the same fused multiply-add, into two sums
// one unit apart (norm_base's comment says how they show a special element).
//
//   k_norm_est               an estimate of each chain's value along the tensor, from sums the step
//                            has already formed (per row band: rm * sum_j c_j^2 * sum_i g_ij^2 / R_i;
//                            per 1-D tile: the tile's sum of u^2); the records kernels add the units
//                            before a segment themselves (norm_unit_prefix).
//   k_norm_seg               one workgroup per segment of kNormSegElems elements (512 per chain):
//                            per chain, the candidate binade Ea of the estimate (and Ea + 1 near a
//                            binade edge), the integer sums of the increments under each, or that
//                            the segment holds special elements or leaves the binade; and
//                            the chain's fp32 sum of the segment's rounded squares.
//   k_norm_bsum, k_norm_fix  each chain's own estimate (the prefix of its segment sums), and records
//                            rebuilt under that estimate's binades where the tensor-wide estimate
//                            (an eighth of the prefix) named others.  The chains of heavy-tailed
//                            updates drift far apart; without the rebuild most of their segments
//                            would miss and be replayed.
//   k_norm_walk              one wavefront per chain: applies the first segment from s = 0 element by
//                            element (no record of it is read: a tensor of one segment forms none),
//                            then skips every run of segments whose record covers the chain's current
//                            binade without specials and without leaving the binade (a wavefront scan
//                            of the integer sums), and replays the segment where that fails: binade
//                            crossings, specials, and estimates that missed.  A replay holds the
//                            segment's 512 elements in the wavefront and applies the increments of the
//                            chain's binade with a saturating prefix sum up to the first element that
//                            leaves the binade or is special, that element with fmaf, and so on: one
//                            round per crossing or special element.
//   k_norm_final             the eight accumulators and the tail in the reference's order, sqrt,
//                            and the clip divisor.
//
// Only the replay's fmaf of an element that leaves the binade (or is special) uses floating-point
// addition on the chain; everything else is exact integer arithmetic, so the result equals the
// serial chain bit for bit whatever the estimates were (they only decide how many segments are
// replayed).
#pragma once

#include "came8_kernels.h"

namespace came8 {

constexpr int kNormSegElems = 4096;                    // flat elements per segment (a multiple of 8)
constexpr int kNormChainSeg = kNormSegElems / 8;       // elements per chain per segment
constexpr int kNormChunks = kNormSegElems / (8 * 64);  // 8-element chunks per lane of a segment's wavefront
// segments per thread per batch of the walk: after each replay the walk scans its lanes' records again,
// so a batch of fewer records per lane makes each scan shorter, at one batch load more per 64 * this
// many segments (with the replays' loads issued together: C1 0.2058 / 0.1997 ms and C2 2.131 / 2.115
// ms with 8 / 4, C4 the same; 16 and 32 slower)
constexpr int kNormWalkSegs = 4;
static_assert(kNormWalkSegs % 4 == 0, "the walk loads each lane's records four at a time");
constexpr int kNormGroup = 2;                          // chunks per lane loaded together
constexpr int64_t kNormMaxUnits = 4096;                // estimate units per tensor of single-band matrices
                                                       // or tiles (more are grouped)

// binade of a finite s >= 0: E with s in [2^E, 2^(E+1)), or -126 below 2^-125
__device__ __forceinline__ int norm_binade(float s) {
  const int e = int(__float_as_uint(s) >> 23);
  return e == 0 ? -126 : e - 127;
}
// s = m * 2^(E-23) for E = norm_binade(s): the integer m < 2^24, and back
__device__ __forceinline__ uint32_t norm_mant(float s, int E) { return __float_as_uint(s) - (uint32_t(E + 126) << 23); }
__device__ __forceinline__ float norm_value(uint32_t m, int E) { return __uint_as_float((uint32_t(E + 126) << 23) + m); }

// binade of an estimate (any float): -126 for values <= 2^-125 (and NaN), 127 for +inf
__device__ __forceinline__ int norm_est_binade(float v) {
  if (!(v > 0x1p-125f)) return -126;
  if (!(v <= 0x1.fffffep127f)) return 127;
  return norm_binade(v);
}

// The increments of a run of elements under binade E, per lane and chain, without knowing the chain's value: two
// running sums started inside the binade, at 2^E (even mantissa) and one unit 2^(E-23) above it (odd), each element
// one fused multiply-add into both.  A fused multiply-add that stays in the binade adds the element's increment,
// rounded as the chain would round it, so the first sum less its start is the increments' integer sum, exactly; the
// two sums stay one unit apart unless an element is a tie, which rounds to the even side: then they come out two
// units or none apart and stay so.  Read off once per lane (norm_lane_value), an exception makes the walk replay
// the segment:
//   * a tie: the rounding of that element depends on the chain's parity;
//   * a sum that left the binade (it only grows; so does one that met a NaN or an infinity): the increments reach
//     2^23 units, and a chain of a normal binade, whose mantissa is at least 2^23, leaves it too (in the subnormal
//     binade the replay decides).
// Squares are exact inside the multiply-add, so the subnormal binade needs no rule of its own.  Five instructions an
// element with the conversion aside (three products of u, the sum of squares, the two sums; two more per further
// binade); scaling, rounding and comparing each square took nine, and five more, and bound the records kernel by
// issue rate (1.07 G bf16 elements: 446 -> 395 us, 5.5 TB/s; one 2048x2048 fp32 matrix: 20.2 -> 13.6 us).
__device__ __forceinline__ float norm_base(int E) { return __uint_as_float(uint32_t(E + 127) << 23); }
// the lane's increments for one chain under E as the record's integer, or kNormFull for an exception (E = 128, the
// binade above the largest, holds no chain)
__device__ __forceinline__ uint32_t norm_lane_value(float even, float odd, int E) {
  const uint32_t base = uint32_t(E + 127) << 23;
  const uint32_t n = __float_as_uint(even) - base;
  return (n < (1u << 23) && __float_as_uint(odd) - base == n + 1u && E < 128) ? n : (1u << 24);
}

// Record word 0: Ea + 256 (9 bits) | kRecTwo when word 2 holds the sum under Ea + 1.  Words 1 and 2:
// the integer sums of the increments under Ea and Ea + 1, at most 2^24 (2^24: the segment leaves
// the binade or holds a special element).
constexpr uint32_t kRecTwo = 1u << 9;
constexpr uint32_t kNormFull = 1u << 24;

// ---------------------------------------------------------------------------
// estimates
// ---------------------------------------------------------------------------
// Units: row band b of matrix m (unit m * nbands + b; for matrices of the thread-per-matrix passes the
// matrix is its band) or 2048-element tile u of a 1-D tensor.  The sum of u_ij^2 over a band is
// rm * sum_i (1 / R_i) * sum_j c_j^2 * g_ij^2 without the roundings.  The thread-per-matrix passes form u
// themselves and write their groups' sums of u^2 (k_tiny_pass1).  The band
// passes of the default clip mode keep no W (k_fact_pass1n); their estimate gives every row of the band
// the band's column profile of g^2 (the partials U_j):
//   rm * (sum_i e_i / R_i) * (sum_j c_j^2 U_j) / (sum_j U_j),   e_i = sum_j g_ij^2,
// exact when the rows' profiles agree (Gaussian rows: ~1e-5 relative per band) and a few percent off
// on heavy-tailed rows; k_norm_fix rebuilds the records of a chain that the estimate misleads.
// WIDE: a workgroup per unit (matrices of at least 256 columns); otherwise kEstLanes lanes per unit: a thread per unit
// read its row of partials serially, four workgroups a launch for a thousand bands, bound by one load after the other
// (bands of four matrices of 24 to 200 columns among 30 tensors: 39 -> 11 us).
constexpr int kEstLanes = 16, kEstUnits = kThreads / kEstLanes;  // lanes of a unit, units of a workgroup
template <typename T>
__device__ __forceinline__ T est_lanes_sum(T v) {
#pragma unroll
  for (int o = kEstLanes / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kEstLanes);
  return v;
}
template <bool WIDE>
__global__ __launch_bounds__(kThreads) void k_norm_est(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                       const int64_t* __restrict__ wstart, int ntens, Hp hp) {
  __shared__ float ssum[4], usum[4];
  __shared__ double rsm[4];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t total = wstart[ntens];
  for (int64_t w = blockIdx.x; w < total; w += gridDim.x) {
    const int slot = find_slot(wstart, ntens, w);
    const DevTensor& t = T[tids[slot]];
    if constexpr (WIDE) {  // band passes (never the thread-per-matrix ones)
      const int64_t u = w - wstart[slot];
      const int64_t m = u / t.nbands;
      const float* __restrict__ Up = t.partU + u * t.C;
      const float* __restrict__ cf = t.cfac + m * t.C;
      // kEstBatch columns per thread loaded before the first is added (an estimate: the order is free)
      constexpr int kEstBatch = 8;
      float acc[kEstBatch] = {}, accu[kEstBatch] = {};
      int64_t j = tid;
      for (; j + (kEstBatch - 1) * kThreads < t.C; j += kEstBatch * kThreads) {
        float c[kEstBatch], uv[kEstBatch];
#pragma unroll
        for (int q = 0; q < kEstBatch; ++q) {
          c[q] = cf[j + q * kThreads];
          uv[q] = Up[j + q * kThreads];
        }
#pragma unroll
        for (int q = 0; q < kEstBatch; ++q) {
          acc[q] = fmaf(c[q] * c[q], uv[q], acc[q]);
          accu[q] += uv[q];
        }
      }
      for (; j < t.C; j += kThreads) {
        acc[0] = fmaf(cf[j] * cf[j], Up[j], acc[0]);
        accu[0] += Up[j];
      }
      // the matrix's mean row state: the workgroup sums the band sums, thread k over
      // sums k, k + 256, ... (one round of loads, not one thread's chain after the reductions)
      double rp = 0.0;
      for (int64_t k = tid; k < t.nbands; k += kThreads) rp += double(t.rsum[m * t.nbands + k]);
      float s = 0.0f, su = 0.0f;
#pragma unroll
      for (int q = 0; q < kEstBatch; ++q) {
        s += acc[q];
        su += accu[q];
      }
      s = wave_sum(s);
      su = wave_sum(su);
      rp = wave_sum(rp);
      if (lane == 0) {
        ssum[wid] = s;
        usum[wid] = su;
        rsm[wid] = rp;
      }
      __syncthreads();
      if (tid == 0) {
        const float cs = ((ssum[0] + ssum[1]) + ssum[2]) + ssum[3];
        const float us = ((usum[0] + usum[1]) + usum[2]) + usum[3];
        const float rm = row_mean_of_sum(t, ((rsm[0] + rsm[1]) + rsm[2]) + rsm[3]);
        t.nest[u] = us > 0.0f ? rm * t.esum[u] * (cs / us) : 0.0f;
      }
      __syncthreads();
    } else {
      const int64_t u = (w - wstart[slot]) * kEstUnits + tid / kEstLanes;
      const int l = tid % kEstLanes;
      if (u >= t.nunit) continue;
      // the unit's ngrp base units: row bands, or (ngrp > 1) whole single-band matrices, or tiles
      const int64_t nbase = t.factored ? t.P * t.nbands : t.nclip;
      const int64_t b0 = u * t.ngrp, b1 = min(nbase, b0 + t.ngrp);
      float e = 0.0f;
      if (t.factored) {  // a band pass of the default mode: the band's profile of g^2
        for (int64_t b = b0; b < b1; ++b) {
          const int64_t m = b / t.nbands;
          const float* __restrict__ Up = t.partU + b * t.C;
          const float* __restrict__ cf = t.cfac + m * t.C;
          float s = 0.0f, su = 0.0f;
#pragma unroll 4
          for (int64_t j = l; j < t.C; j += kEstLanes) {
            s = fmaf(cf[j] * cf[j], Up[j], s);
            su += Up[j];
          }
          double rp = 0.0;  // the matrix's mean row state
          for (int64_t k = l; k < t.nbands; k += kEstLanes) rp += double(t.rsum[m * t.nbands + k]);
          s = est_lanes_sum(s);
          su = est_lanes_sum(su);
          rp = est_lanes_sum(rp);
          e += su > 0.0f ? row_mean_of_sum(t, rp) * t.esum[b] * (s / su) : 0.0f;
        }
      } else {
        for (int64_t b = b0 + l; b < b1; b += kEstLanes) e += float(t.clip_part[b]);
        e = est_lanes_sum(e);
      }
      if (l == 0) t.nest[u] = e;
    }
  }
}

// The estimated sum of u^2 over the units before unit u (0 <= u <= nunit), from the units' own
// estimates: the wavefront adds them, lane l over units l, l + 64, ..., eight loads in flight.  Every
// lane of the wavefront calls it with the same u and gets the same value.  (The order of the sum is
// free: an estimate decides only which segments are replayed, never the result.)
__device__ __forceinline__ float norm_unit_prefix(const DevTensor& t, int64_t u) {
  const int lane = threadIdx.x & (kWave - 1);
  const CAME8_GLOBAL float* __restrict__ e = gbl(t.nest);
  float s = 0.0f;
  int64_t k = lane;
  for (; k + 7 * kWave < u; k += 8 * kWave) {
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = e[k + q * kWave];
#pragma unroll
    for (int q = 0; q < 8; ++q) s += v[q];
  }
  for (; k < u; k += kWave) s += e[k];
  return wave_sum(s);
}

// Estimated sum of u^2 over the flat elements before f (0 <= f <= N), linear inside a unit.
__device__ __forceinline__ float norm_est_at(const DevTensor& t, int64_t f) {
  int64_t u, us, ue;
  if (t.factored) {
    const int64_t row = t.idx32 ? int64_t(udiv_magic(uint32_t(f), t.mC, t.sC)) : f / t.C;
    const int64_t m = t.idx32 ? int64_t(udiv_magic(uint32_t(row), t.mR, t.sR)) : row / t.R;
    if (m >= t.P) return norm_unit_prefix(t, t.nunit);
    const int64_t i = row - m * t.R;
    if (t.ngrp > 1) {  // groups of ngrp single-band matrices
      u = m / t.ngrp;
      us = u * t.ngrp * t.R * t.C;
      ue = min(t.P, (u + 1) * t.ngrp) * t.R * t.C;
    } else {
      const int64_t b = int64_t(uint32_t(i) / uint32_t(t.rb));  // rows per band <= 256
      u = m * t.nbands + b;
      us = (m * t.R + b * t.rb) * t.C;
      ue = (m * t.R + min((b + 1) * t.rb, t.R)) * t.C;
    }
  } else {
    u = f / (kTile * t.ngrp);
    if (u >= t.nunit) return norm_unit_prefix(t, t.nunit);
    us = u * kTile * t.ngrp;
    ue = min(us + kTile * t.ngrp, t.N);
  }
  return norm_unit_prefix(t, u) + gbl(t.nest)[u] * (float(f - us) / float(ue - us));
}

// ---------------------------------------------------------------------------
// segment records
// ---------------------------------------------------------------------------
// One halving step of norm_group_sums: lanes with bit O set keep values [H, 2H) and send [0, H) to their
// partner lane ^ O, which keeps [0, H); each adds what it receives (H, O compile-time constants).
template <int H, int O, typename T, int L>
__device__ __forceinline__ void norm_halve(T (&v)[L], int lane) {
  const bool up = (lane & O) != 0;
#pragma unroll
  for (int k = 0; k < H; ++k) {
    const T mine = up ? v[H + k] : v[k];
    const T other = up ? v[k] : v[H + k];
    v[k] = mine + __shfl_xor(other, O, kWave);
  }
}

// Per-value sums over groups of G lanes (G a power of two up to 64) of NV values per lane (NV = 8 or
// 16).  Halving steps with the partners lane ^ G/2, ^ G/4, ... leave each lane NV / G values (NV > G)
// or one, summed over the lanes that share the lane bits halved so far; butterfly sums over the
// remaining low lane bits complete it (NV < G).  On return, lane i of a group (i = lane % G) holds
// the totals of values i * NV / G + k in v[k], k < NV / G (NV >= G), or of value i / (G / NV) in v[0]
// (NV < G).
template <int O, int H, typename T, int L>
__device__ __forceinline__ void norm_group_steps(T (&v)[L], int lane) {
  if constexpr (O >= 1) {
    if constexpr (H >= 1) {
      norm_halve<H, O>(v, lane);
    } else {
      v[0] += __shfl_xor(v[0], O, kWave);
    }
    norm_group_steps<O / 2, H / 2>(v, lane);
  }
}
template <int G, int NV, typename T, int L>
__device__ __forceinline__ void norm_group_sums(T (&v)[L], int lane) {
  static_assert(L >= NV && G >= 2 && G <= kWave && (G & (G - 1)) == 0, "bad group");
  norm_group_steps<G / 2, NV / 2>(v, lane);
}
// The same over the whole wavefront: v[0] of lane l holds the total of value l >> 3 (NV = 8) or l >> 2
// (NV = 16).
template <int NV, typename T, int L>
__device__ __forceinline__ void norm_lane_sums(T (&v)[L], int lane) {
  norm_group_sums<kWave, NV>(v, lane);
}

// u_at of the 8 elements e[v] (in bounds) of any tensor, every operand loaded before the first is
// used: the tensor's kind is tested once for the 8, so that no branch between the elements makes the
// wavefront wait out each element's loads in turn.
template <typename TG>
__device__ __forceinline__ void norm_x_any8(const DevTensor& t, const int64_t (&e)[8], const Hp& hp, float (&x)[8]) {
  using GS = typename TG::storage;
  const CAME8_GLOBAL GS* __restrict__ gp = gbl(static_cast<const GS*>(t.g));
  float gv[8], a[8], b[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) gv[v] = TG::load(gp[e[v]]);
  if (t.factored) {
    const CAME8_GLOBAL float* __restrict__ rf = gbl(t.rfac);
    const CAME8_GLOBAL float* __restrict__ cf = gbl(t.cfac);
    if (t.idx32) {
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const uint32_t row = udiv_magic(uint32_t(e[v]), t.mC, t.sC);
        const uint32_t j = uint32_t(e[v]) - row * uint32_t(t.C);
        const uint32_t m = udiv_magic(row, t.mR, t.sR);
        a[v] = rf[row];
        b[v] = cf[int64_t(m) * t.C + j];
      }
    } else {
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const int64_t row = e[v] / t.C;
        const int64_t j = e[v] - row * t.C;
        a[v] = rf[row];
        b[v] = cf[(row / t.R) * t.C + j];
      }
    }
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = (a[v] * b[v]) * gv[v];
  } else {
    if (t.fp32st) {
#pragma unroll
      for (int v = 0; v < 8; ++v) a[v] = gbl(st_sq_row(t))[e[v]];
    } else {
#pragma unroll
      for (int v = 0; v < 8; ++v) a[v] = deq_u8(gbl(t.rq)[e[v]], gbl(t.ra)[blk_of(e[v], hp)]);
    }
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = rsqrt_ref(vec_v_from(gv[v], a[v], hp)) * gv[v];
  }
}

// The x = u of the 8 elements at flat index f (a multiple of 8) of a factored tensor whose rows hold
// whole 8-element chunks, 16-byte aligned, with flat indices below 2^31.
template <typename TG>
struct NormChunk {
  float g[8], cf[8], r;
  __device__ __forceinline__ void load(const DevTensor& t, uint32_t f) {
    using GS = typename TG::storage;
    const uint32_t row = udiv_magic(f, t.mC, t.sC);
    const uint32_t j = f - row * uint32_t(t.C);
    const uint32_t m = udiv_magic(row, t.mR, t.sR);
    r = gbl(t.rfac)[row];
    load8<TG>(gbl(static_cast<const GS*>(t.g) + f), g);
    load8<F32>(gbl(t.cfac + int64_t(m) * t.C + j), cf);
  }
};

// The same for a factored tensor of at least 8 columns whose rows do not hold whole chunks: the chunk
// may end in the next row (and the next matrix); its gradient is still 16-byte aligned.
template <typename TG>
__device__ __forceinline__ void norm_chunk_rows(const DevTensor& t, uint32_t f, float (&x)[8]) {
  using GS = typename TG::storage;
  const uint32_t C = uint32_t(t.C);
  const uint32_t row = udiv_magic(f, t.mC, t.sC);
  const uint32_t j = f - row * C;
  const uint32_t m0 = udiv_magic(row, t.mR, t.sR);
  float gv[8];
  load8<TG>(gbl(static_cast<const GS*>(t.g) + f), gv);
  const bool cross = j + 8 > C;  // the elements from C - j on are the next row's
  const uint32_t m1 = cross ? udiv_magic(row + 1, t.mR, t.sR) : m0;
  const float r0 = gbl(t.rfac)[row];
  const float r1 = cross ? gbl(t.rfac)[row + 1] : r0;
  const CAME8_GLOBAL float* __restrict__ cf = gbl(t.cfac);
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const bool nx = j + v >= C;
    const uint32_t col = nx ? j + v - C : j + v;
    const float c = cf[int64_t(nx ? m1 : m0) * C + col];
    x[v] = ((nx ? r1 : r0) * c) * gv[v];
  }
}

// How a norm kernel loads the x of a tensor's 8-element chunks: kNormVec for factored tensors whose rows
// hold whole chunks, kNormRows for other factored tensors of at least 8 columns (both: gradient 16-byte
// aligned, N < 2^31; the host checks), kNormAny (u_at of each element) for the rest.
constexpr int kNormAny = 0, kNormRows = 1, kNormVec = 2;

// Per-lane, per-chain accumulators of one segment: the pair of sums under the candidate binade Ea (ae, ao) and
// under Ea + 1 (be, bo), and the fp32 sum of the squares (hs).
struct NormAcc {
  float ae[8], ao[8], be[8], bo[8], hs[8];
  __device__ __forceinline__ void init(int v, int Ea) {
    ae[v] = norm_base(Ea);
    ao[v] = __uint_as_float(__float_as_uint(ae[v]) + 1u);
    be[v] = norm_base(Ea + 1);
    bo[v] = __uint_as_float(__float_as_uint(be[v]) + 1u);
    hs[v] = 0.0f;
  }
  __device__ __forceinline__ void init(int Ea) {
#pragma unroll
    for (int v = 0; v < 8; ++v) init(v, Ea);
  }
  // element x of chain v (TWO: under Ea + 1 too)
  template <bool TWO>
  __device__ __forceinline__ void add(int v, float x) {
    hs[v] = fmaf(x, x, hs[v]);
    ae[v] = fmaf(x, x, ae[v]);
    ao[v] = fmaf(x, x, ao[v]);
    if constexpr (TWO) {
      be[v] = fmaf(x, x, be[v]);
      bo[v] = fmaf(x, x, bo[v]);
    }
  }
  // An empty asm that reads and writes the sums: in a fully unrolled segment the code generator would
  // otherwise interleave chunks and hold their elements longer.
  template <bool TWO>
  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      asm volatile("" : "+v"(ae[v]), "+v"(ao[v]), "+v"(hs[v]));
      if constexpr (TWO) asm volatile("" : "+v"(be[v]), "+v"(bo[v]));
    }
  }
  __device__ __forceinline__ uint32_t val_a(int v, int Ea) const { return norm_lane_value(ae[v], ao[v], Ea); }
  __device__ __forceinline__ uint32_t val_b(int v, int Ea) const { return norm_lane_value(be[v], bo[v], Ea + 1); }
};

// The x of the 8 elements at flat index f (a multiple of 8): element v belongs to chain v.  Elements
// at or past f1 (a multiple of 8) are 0.
template <typename TG, int FORM>
__device__ __forceinline__ void norm_chunk_x(const DevTensor& t, int64_t f, int64_t f1, const Hp& hp,
                                             float (&x)[8]) {
  const bool in = f < f1;
  if constexpr (FORM == kNormVec) {
    NormChunk<TG> ch;
    ch.load(t, uint32_t(in ? f : f1 - 8));
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = in ? (ch.r * ch.cf[v]) * ch.g[v] : 0.0f;
  } else if constexpr (FORM == kNormRows) {
    norm_chunk_rows<TG>(t, uint32_t(in ? f : f1 - 8), x);
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = in ? x[v] : 0.0f;
  } else {  // a chunk past f1 reads the last chunk before it (f1 >= 8)
    int64_t e[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) e[v] = (in ? f : f1 - 8) + v;
    norm_x_any8<TG>(t, e, hp, x);
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = in ? x[v] : 0.0f;
  }
}

// Adds chunk steps [h0, h1) of one segment to a lane's sums (TWO: under Ea + 1 too).
// FULL: the segment holds all kNormSegElems elements.
template <typename TG, int FORM, bool TWO, bool FULL>
__device__ __forceinline__ void norm_seg_sums(const DevTensor& t, int64_t f0, int64_t f1, int lane,
                                              const Hp& hp, NormAcc& a, int h0 = 0, int h1 = kNormChunks) {
  auto account = [&](const float (&x)[8]) {
#pragma unroll
    for (int v = 0; v < 8; ++v) a.add<TWO>(v, x[v]);
  };
  if constexpr (FORM == kNormRows) {
#pragma unroll 1
    for (int h = h0; h < h1; h += kNormGroup) {
      float x[kNormGroup][8];
#pragma unroll
      for (int q = 0; q < kNormGroup; ++q)
        norm_chunk_x<TG, kNormRows>(t, f0 + (h + q) * 512 + lane * 8, FULL ? f0 + kNormSegElems : f1, hp, x[q]);
#pragma unroll
      for (int q = 0; q < kNormGroup; ++q) account(x[q]);
    }
  } else if constexpr (FORM == kNormVec) {
    // in a partial segment, chunks past its end load its last chunk and count for nothing
#pragma unroll 1
    for (int h = h0; h < h1; h += kNormGroup) {
      NormChunk<TG> ch[kNormGroup];
#pragma unroll
      for (int q = 0; q < kNormGroup; ++q) {
        const int64_t f = f0 + (h + q) * 512 + lane * 8;
        ch[q].load(t, uint32_t(FULL ? f : min(f, f1 - 8)));
      }
#pragma unroll
      for (int q = 0; q < kNormGroup; ++q) {
        const bool in = FULL || f0 + (h + q) * 512 + lane * 8 < f1;
        float x[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) x[v] = in ? (ch[q].r * ch[q].cf[v]) * ch[q].g[v] : 0.0f;
        account(x);
      }
    }
  } else {  // chunks past the segment's end count for nothing
#pragma unroll 1
    for (int h = h0; h < h1; h += kNormGroup) {
      float x[kNormGroup][8];
#pragma unroll
      for (int q = 0; q < kNormGroup; ++q)
        norm_chunk_x<TG, kNormAny>(t, f0 + (h + q) * 512 + lane * 8, FULL ? f0 + kNormSegElems : f1, hp, x[q]);
#pragma unroll
      for (int q = 0; q < kNormGroup; ++q) account(x[q]);
    }
  }
}

// Writes the records of one segment from the per-lane, per-chain sums of the workgroup's wavefronts
// (each took a part of the segment's chunks), and the chains' sums of squares.  Each wavefront sums its
// lanes' integer records (a lane's sum is an exact integer below 2^24, or 2^24 when it holds a tie or
// leaves the binade) and caps the total at 2^24; wavefront 0 adds the four totals in order, caps again
// and writes the records.  xacc and xhs are LDS of the workgroup; every thread of it calls this.
__device__ __forceinline__ void norm_write_records(const DevTensor& t, int64_t seg, int Ea, bool two, int lane,
                                                   int wid, const NormAcc& a, uint32_t (*xacc)[16], float (*xhs)[8]) {
  uint32_t acc[16];
  float hs[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    acc[v] = a.val_a(v, Ea);
    acc[8 + v] = two ? a.val_b(v, Ea) : 0u;
    hs[v] = a.hs[v];
  }
  norm_lane_sums<8>(hs, lane);    // lane 8c: chain c
  norm_lane_sums<16>(acc, lane);  // lane 4c: chain c under Ea; lane 32 + 4c: under Ea + 1
  if ((lane & 7) == 0) xhs[wid][lane >> 3] = hs[0];
  if ((lane & 3) == 0) xacc[wid][lane >> 2] = min(acc[0], kNormFull);
  __syncthreads();
  if (wid == 0) {
    const int64_t nseg = t.nseg;
    const int c = lane & 7;
    if (lane < 16) {
      uint32_t sum = 0;
#pragma unroll
      for (int k = 0; k < kThreads / kWave; ++k) sum += xacc[k][lane];
      sum = min(sum, kNormFull);
      if (lane < 8) {
        t.nrec[c * nseg + seg] = uint32_t(Ea + 256) | (two ? kRecTwo : 0u);
        t.nrec[(8 + c) * nseg + seg] = sum;
      } else {
        t.nrec[(16 + c) * nseg + seg] = two ? sum : kNormFull;
      }
    }
    if (lane < 8) {
      float h = xhs[0][lane];
#pragma unroll
      for (int k = 1; k < kThreads / kWave; ++k) h += xhs[k][lane];
      t.nsum[lane * nseg + seg] = h;
    }
  }
  __syncthreads();  // xacc and xhs are written again by the next segment
}

// Candidate binades of a chain whose estimated value is est: Ea, and whether Ea + 1 is one too.
__device__ __forceinline__ void norm_candidates(float est, int& Ea, bool& two) {
  Ea = norm_est_binade(est * 0.875f);
  two = norm_est_binade(est * 1.015625f) > Ea;
}

constexpr int kNormRunSegs = 64;       // segments per work item of k_norm_seg2d (at most; 16 for small tensors)
constexpr int kNormLdsCols = 16384;    // column factors k_norm_seg2d stages in LDS (64 KB; rows of whole chunks
                                       // up to this wide, other rows 8 less)
constexpr int kNormSegLanes = 16;      // lanes per segment in k_norm_seg2d (narrowest rows: 8 * this)
constexpr int kNormSegAhead = 8;       // chunks per lane in flight there

// The per-lane, per-chain sums of one whole segment per group of G lanes (lane i = lane % G of the
// group takes the 8-element chunks at f0 + 8 * G * q + 8 * i) of a matrix (prefix 1) whose column
// factors are staged in LDS (cl), rows at least 8 * G wide, gradient 16-byte aligned, 32-bit flat
// indices.  A chunk's row and column follow from the previous chunk's by one wrap, as the rows are at
// least 8 * G wide.  ROWS: rows that are not whole chunks; a chunk may end in the next row, whose
// column factors continue in cl past C (the staging repeats the first 8 there) and whose row factor
// the elements from C - col on take (a select per element: a branch around it would double the
// unrolled loop, which then no longer unrolls).  The schedule is fixed by hand, a step per chunk: the column factors
// of the next chunk are read from LDS, this chunk is accounted, and the gradient and row factor of
// the chunk kNormSegAhead on are loaded into the registers this one frees.  Scheduling barriers keep
// the compiler from hoisting the loads further, and NormAcc::pin keeps each chunk's roundings in its
// step (either would cost registers, not time).
template <typename TG, int G, bool TWO, bool ROWS>
__device__ __forceinline__ void norm_seg_lds(const DevTensor& t, const float* cl, uint32_t f0, int li, NormAcc& a) {
  using GS = typename TG::storage;
  constexpr int Q = kNormSegElems / (8 * G), D = kNormSegAhead, NW = int(sizeof(GS)) * 2;
  static_assert(Q >= D, "segment chunks");
  const CAME8_GLOBAL GS* __restrict__ g = gbl(static_cast<const GS*>(t.g));
  const CAME8_GLOBAL float* __restrict__ rf = gbl(t.rfac);
  const uint32_t C = uint32_t(t.C), rlast = uint32_t(t.R) - 1u;
  uint32_t f = f0 + uint32_t(li * 8);
  uint32_t row = udiv_magic(f, t.mC, t.sC);
  uint32_t col = f - row * C;
  uint32_t gw[D][NW];  // 16 or 32 bytes of gradient per chunk
  float r[D], r1[ROWS ? D : 1];
  uint32_t cc[D];
  auto issue = [&](int s) __attribute__((always_inline)) {
    cc[s] = col;
    r[s] = rf[row];
    if constexpr (ROWS) r1[s] = rf[min(row + 1u, rlast)];  // the next row's, for a chunk that ends there
    if constexpr (sizeof(GS) == 2) {
      const u32x4 v = ld_nt((const CAME8_GLOBAL u32x4*)(g + f));
      gw[s][0] = v.x; gw[s][1] = v.y; gw[s][2] = v.z; gw[s][3] = v.w;
    } else {
      const u32x4 b0 = *(const CAME8_GLOBAL u32x4*)(g + f);  // two per lane: no hint
      const u32x4 b1 = *(const CAME8_GLOBAL u32x4*)(g + f + 4);
      gw[s][0] = b0.x; gw[s][1] = b0.y; gw[s][2] = b0.z; gw[s][3] = b0.w;
      gw[s][4] = b1.x; gw[s][5] = b1.y; gw[s][6] = b1.z; gw[s][7] = b1.w;
    }
    f += 8 * G;
    col += 8 * G;
    const bool wrap = col >= C;
    col = wrap ? col - C : col;
    row += wrap ? 1u : 0u;
  };
  // the column factors of a chunk at column col (ROWS: 4-byte aligned, read in pairs)
  auto read_c = [&](uint32_t col, float (&cv)[8]) __attribute__((always_inline)) {
    if constexpr (ROWS) {
#pragma unroll
      for (int v = 0; v < 8; ++v) cv[v] = cl[col + v];
    } else {
      const f32x4 c0 = *reinterpret_cast<const f32x4*>(cl + col);
      const f32x4 c1 = *reinterpret_cast<const f32x4*>(cl + col + 4);
      cv[0] = c0.x; cv[1] = c0.y; cv[2] = c0.z; cv[3] = c0.w;
      cv[4] = c1.x; cv[5] = c1.y; cv[6] = c1.z; cv[7] = c1.w;
    }
  };
#pragma unroll
  for (int q = 0; q < D; ++q) issue(q);
  float cn[8];
  read_c(cc[0], cn);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    __builtin_amdgcn_sched_barrier(0);
    const int s = q % D;
    float cv[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) cv[v] = cn[v];
    if (q + 1 < Q) read_c(cc[(q + 1) % D], cn);
    if constexpr (ROWS) {
      const uint32_t b = C - cc[s];  // the chunk's elements in its first row
#pragma unroll
      for (int v = 0; v < 8; ++v)
        a.add<TWO>(v, ((uint32_t(v) < b ? r[s] : r1[s]) * cv[v]) * TG::elem(gw[s], v));
      a.template pin<TWO>();
    } else {
#pragma unroll
      for (int v = 0; v < 8; ++v) a.add<TWO>(v, (r[s] * cv[v]) * TG::elem(gw[s], v));
      a.template pin<TWO>();
    }
    if (q + D < Q) issue(s);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// Writes the records of the segment of each active group of G lanes (li = lane % G) from the lanes'
// per-chain sums, and the chains' sums of squares.  Ea: the group's binade; two: sums under Ea + 1
// were formed (uniform over the wavefront).
template <int G>
__device__ __forceinline__ void norm_write_records_g(const DevTensor& t, int64_t seg, int Ea, bool two, bool act,
                                                     int lane, const NormAcc& a) {
  const int li = lane & (G - 1);
  uint32_t acc[16];
  float hs[8];
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    acc[v] = a.val_a(v, Ea);
    acc[8 + v] = two ? a.val_b(v, Ea) : 0u;
    hs[v] = a.hs[v];
  }
  const int64_t nseg = t.nseg;
  uint32_t* __restrict__ W0 = t.nrec;
  uint32_t* __restrict__ WA = t.nrec + 8 * nseg;
  uint32_t* __restrict__ WB = t.nrec + 16 * nseg;
  // value index i / (G / NV) (NV < G) or i * NV / G + k (NV >= G) after norm_group_sums
  norm_group_sums<G, 8>(hs, lane);
  constexpr int H8 = G > 8 ? G / 8 : 1, K8 = G < 8 ? 8 / G : 1;
#pragma unroll
  for (int k = 0; k < K8; ++k) {
    const int c = G >= 8 ? li / H8 : li * K8 + k;
    if (act && li % H8 == 0) t.nsum[c * nseg + seg] = hs[k];
  }
  if (two) {
    norm_group_sums<G, 16>(acc, lane);
    constexpr int H16 = G > 16 ? G / 16 : 1, K16 = G < 16 ? 16 / G : 1;
#pragma unroll
    for (int k = 0; k < K16; ++k) {
      const int i = G >= 16 ? li / H16 : li * K16 + k;  // i < 8: chain i under Ea; else chain i - 8 under Ea + 1
      if (act && li % H16 == 0) {
        const uint32_t sum = min(acc[k], kNormFull);
        if (i < 8) {
          W0[i * nseg + seg] = uint32_t(Ea + 256) | kRecTwo;
          WA[i * nseg + seg] = sum;
        } else {
          WB[(i - 8) * nseg + seg] = sum;
        }
      }
    }
  } else {
    norm_group_sums<G, 8>(acc, lane);
#pragma unroll
    for (int k = 0; k < K8; ++k) {
      const int c = G >= 8 ? li / H8 : li * K8 + k;
      if (act && li % H8 == 0) {
        W0[c * nseg + seg] = uint32_t(Ea + 256);
        WA[c * nseg + seg] = min(acc[k], kNormFull);
        WB[c * nseg + seg] = kNormFull;
      }
    }
  }
}

// The segments of one wavefront in a run of k_norm_seg2d: segments k0 + sub for k0 = wid * SPW,
// wid * SPW + 4 * SPW, ... below nrun, sub = lane / G.  TWO holds for all of them.
template <typename TG, int G, bool TWO, bool ROWS>
__device__ __forceinline__ void norm_seg2d_wave(const DevTensor& t, const float* cl, int64_t run0, int64_t nrun,
                                                float e0, float e1, int wid, int lane) {
  constexpr int SPW = kWave / G;
  const int li = lane & (G - 1), sub = lane / G;
#pragma unroll 1
  for (int64_t k0 = int64_t(wid) * SPW; k0 < nrun; k0 += (kThreads / kWave) * SPW) {
    // a group past the run's end takes its last segment again and writes nothing
    const bool act = k0 + sub < nrun;
    const int64_t k = act ? k0 + sub : nrun - 1;
    const int64_t seg = run0 + k;
    int Ea;
    bool two;
    norm_candidates(e0 + (e1 - e0) * (float(k) / float(nrun)), Ea, two);
    NormAcc a;
    a.init(Ea);
    wait_vm_all();  // the previous records' stores: the chunk loads' waits then count only loads
    norm_seg_lds<TG, G, TWO, ROWS>(t, cl, uint32_t(seg * kNormSegElems), li, a);
    norm_write_records_g<G>(t, seg, Ea, TWO, act, lane, a);
  }
}

// Records of the whole segments [0, nseg0) of 2-D factored tensors whose rows are at least
// 8 * kNormSegLanes and at most kNormLdsCols wide, gradient 16-byte aligned, with 32-bit flat indices
// (the host checks); FORM kNormVec when the rows hold whole 8-element chunks, else kNormRows.  The last,
// partial segment is k_norm_seg's.  A work item is a run of nrun (16 to kNormRunSegs)
// segments: the workgroup stages the matrix's column factors in LDS once, and each wavefront takes
// kWave / kNormSegLanes consecutive segments at a time, a group of kNormSegLanes lanes per segment.
// A wavefront forms the sums under Ea + 1 for all its segments of the run when one of them needs them
// (a record with both sums is never wrong); the choice is made once per run, so that no code is shared between the forms' segment loops (the
// compiler would hoist a shared start, and the registers it holds, above the branch).
template <typename TG, int FORM>
__global__ __launch_bounds__(kThreads) void k_norm_seg2d(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                         const int64_t* __restrict__ wstart, int ntens, Hp hp) {
  static_assert(FORM == kNormVec || FORM == kNormRows, "k_norm_seg2d forms");
  constexpr bool ROWS = FORM == kNormRows;
  constexpr int G = kNormSegLanes, SPW = kWave / G;  // lanes per segment, segments per wavefront
  extern __shared__ float cl[];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t total = wstart[ntens];
  int32_t staged = -1;
  for (int64_t w = blockIdx.x; w < total; w += gridDim.x) {
    const int slot = find_slot(wstart, ntens, w);
    const int32_t ti = tids[slot];
    const DevTensor& t = T[ti];
    if (ti != staged) {  // uniform over the workgroup
      __syncthreads();
      if constexpr (ROWS) {  // C + 8 factors: the row's, then its first 8 again (for chunks that wrap)
        for (int64_t j = tid; j < t.C + 8; j += kThreads) cl[j] = gbl(t.cfac)[j < t.C ? j : j - t.C];
      } else {
        for (int64_t j = tid * 4; j < t.C; j += kThreads * 4)
          *reinterpret_cast<f32x4*>(cl + j) = *reinterpret_cast<const CAME8_GLOBAL f32x4*>(gbl(t.cfac) + j);
      }
      __syncthreads();
      staged = ti;
    }
    const int64_t run0 = (w - wstart[slot]) * t.nrun;
    const int64_t nrun = min(t.nrun, t.nseg0 - run0);
    const int64_t main = t.N - (t.N & 7);
    // the estimate at both ends of the run, linear in between (a chain holds about 1/8 of it)
    const float e0 = uniform_f32(norm_est_at(t, run0 * kNormSegElems)) * 0.125f;
    const float e1 = uniform_f32(norm_est_at(t, min((run0 + nrun) * kNormSegElems, main))) * 0.125f;
    bool any_two = false;
    for (int64_t k0 = int64_t(wid) * SPW; k0 < nrun; k0 += (kThreads / kWave) * SPW) {
      const int64_t k = min(k0 + lane / G, nrun - 1);
      int Ea;
      bool two;
      norm_candidates(e0 + (e1 - e0) * (float(k) / float(nrun)), Ea, two);
      any_two |= two;
    }
    if (__any(any_two)) norm_seg2d_wave<TG, G, true, ROWS>(t, cl, run0, nrun, e0, e1, wid, lane);
    else norm_seg2d_wave<TG, G, false, ROWS>(t, cl, run0, nrun, e0, e1, wid, lane);
  }
}

// Records of the segments [nseg0, nseg).  One workgroup per segment: lane l of wavefront w takes the
// 8-element chunks at 512q + 8l of the segment for q in [w, w + 1) * kNormGroup (element v of a chunk
// belongs to chain v), and norm_write_records adds the wavefronts' sums.  FORM: how the chunks are
// loaded (norm_chunk_x).
template <typename TG, int FORM>
__global__ __launch_bounds__(kThreads, 4) void k_norm_seg(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                          const int64_t* __restrict__ wstart, int ntens, Hp hp) {
  static_assert(kNormChunks == (kThreads / kWave) * kNormGroup, "a wavefront per kNormGroup chunk steps");
  __shared__ uint32_t xacc[kThreads / kWave][16];
  __shared__ float xhs[kThreads / kWave][8];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t total = wstart[ntens];
  for (int64_t w = blockIdx.x; w < total; w += gridDim.x) {
    const int slot = find_slot(wstart, ntens, w);
    const DevTensor& t = T[tids[slot]];
    // one segment per work item; wavefront wid takes its chunk steps [wid, wid + 1) * kNormGroup
    const int64_t seg = t.nseg0 + (w - wstart[slot]);
    const int h0 = wid * kNormGroup, h1 = h0 + kNormGroup;
    const int64_t main = t.N - (t.N & 7);
    const int64_t f0 = seg * kNormSegElems;
    const int64_t f1 = min(f0 + kNormSegElems, main);
    // candidate binades from the estimate at the segment's start (a chain holds about 1/8 of it)
    int Ea;
    bool two;
    norm_candidates(uniform_f32(norm_est_at(t, f0)) * 0.125f, Ea, two);
    NormAcc a;
    a.init(Ea);
    const bool full = f1 - f0 == kNormSegElems;
    if (two) {
      if (full) norm_seg_sums<TG, FORM, true, true>(t, f0, f1, lane, hp, a, h0, h1);
      else norm_seg_sums<TG, FORM, true, false>(t, f0, f1, lane, hp, a, h0, h1);
    } else {
      if (full) norm_seg_sums<TG, FORM, false, true>(t, f0, f1, lane, hp, a, h0, h1);
      else norm_seg_sums<TG, FORM, false, false>(t, f0, f1, lane, hp, a, h0, h1);
    }
    norm_write_records(t, seg, Ea, two, lane, wid, a, xacc, xhs);
  }
}

// The x of the 8 elements of the chunk at flat index f (a multiple of 8, in a whole segment) of a tensor
// that k_norm_seg2d takes, with the column factors staged in LDS (cl) as it stages them.  ROWS: the
// chunk may end in the next row (kNormRows).
template <typename TG, bool ROWS>
__device__ __forceinline__ void norm_chunk_lds(const DevTensor& t, const float* cl, uint32_t f, float (&x)[8]) {
  using GS = typename TG::storage;
  const uint32_t C = uint32_t(t.C);
  const uint32_t row = udiv_magic(f, t.mC, t.sC);
  const uint32_t col = f - row * C;
  float gv[8];
  load8<TG>(gbl(static_cast<const GS*>(t.g) + f), gv);
  const float r0 = gbl(t.rfac)[row];
  if constexpr (ROWS) {
    const float r1 = gbl(t.rfac)[min(row + 1u, uint32_t(t.R) - 1u)];
    const uint32_t b = C - col;  // the chunk's elements in its first row
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = ((uint32_t(v) < b ? r0 : r1) * cl[col + v]) * gv[v];
  } else {
    const f32x4 c0 = *reinterpret_cast<const f32x4*>(cl + col);
    const f32x4 c1 = *reinterpret_cast<const f32x4*>(cl + col + 4);
    const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
    for (int v = 0; v < 8; ++v) x[v] = (r0 * cv[v]) * gv[v];
  }
}

// Stages the column factors of a tensor that k_norm_seg2d takes in LDS (cl) as k_norm_seg2d does: ROWS,
// C + 8 factors (the row's, then its first 8 again).  Every thread of the workgroup calls it.
template <bool ROWS>
__device__ __forceinline__ void norm_stage_cols(const DevTensor& t, float* cl) {
  const int tid = threadIdx.x;
  if constexpr (ROWS) {
    for (int64_t j = tid; j < t.C + 8; j += kThreads) cl[j] = gbl(t.cfac)[j < t.C ? j : j - t.C];
  } else {
    for (int64_t j = tid * 4; j < t.C; j += kThreads * 4)
      *reinterpret_cast<f32x4*>(cl + j) = *reinterpret_cast<const CAME8_GLOBAL f32x4*>(gbl(t.cfac) + j);
  }
}

// ---------------------------------------------------------------------------
// each chain's own estimate, and records rebuilt under it
// ---------------------------------------------------------------------------
constexpr int kNormFixSegs = kThreads;  // segments per block of the chains' estimates, and at most per work item of k_norm_fix
// Segments whose records need rebuilding come in runs (where the tensor-wide estimate passes a binade boundary), and a
// work item rebuilds its own, so a launch of few items had one workgroup do hundreds: items are halved, down to
// kNormFixMinSegs segments, until the launch has kNormFixMinItems (came8.hip).  22.9 M elements of 3x3 and 1x1
// matrices: 721 us in items of 256 segments, 67 in items of 16; heavy-tailed ragged matrices 410 + 390 -> 81 + 63 us.
constexpr int64_t kNormFixMinSegs = 16, kNormFixMinItems = 1024;
constexpr int64_t kNormFixDirect = 4;   // tensors of at most this many blocks: k_norm_fix adds the segments' sums itself

// Each chain's sum of squares over a block of kNormFixSegs segments (nbsum[c][block]), for the prefix
// k_norm_fix forms.  One work item per block; thread i takes segment i of the block.
template <int = 0>
__global__ __launch_bounds__(kThreads) void k_norm_bsum(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                        const int64_t* __restrict__ wstart, int ntens) {
  __shared__ float part[kThreads / kWave][8];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t total = wstart[ntens];
  for (int64_t w = blockIdx.x; w < total; w += gridDim.x) {
    const int slot = find_slot(wstart, ntens, w);
    const DevTensor& t = T[tids[slot]];
    const int64_t nseg = t.nseg;
    const int64_t blk = w - wstart[slot];
    const int64_t seg = blk * kNormFixSegs + tid;
    float v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = seg < nseg ? t.nsum[c * nseg + seg] : 0.0f;
    norm_lane_sums<8>(v, lane);  // lane 8c: chain c over the wavefront
    if ((lane & 7) == 0) part[wid][lane >> 3] = v[0];
    __syncthreads();
    if (tid < 8) t.nbsum[tid * t.nblk + blk] = (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
    __syncthreads();
  }
}

// The chains' estimates at the segments [base, base + fseg) of one work item of k_norm_fix, into est[c][thread]: the
// sums of the segments before it plus an exclusive scan of the item's own (v: thread i's segment's, 0 past the item).
__device__ __forceinline__ void norm_item_estimates(const DevTensor& t, int64_t base, const float (&v)[8],
                                                    float (&est)[8][kNormFixSegs], float (&part)[kThreads / kWave][8],
                                                    float (&base_l)[8]) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  // thread i adds chain i % 8's sums i / 8, i / 8 + 32, ... in that order, four loads in flight at a time: the whole
  // blocks before the item (k_norm_bsum; a tensor of at most kNormFixDirect blocks has none) and then the segments
  // left before it.
  {
    float acc = 0.0f;
    const int c = tid & 7;
    constexpr int kStep = kThreads / 8;
    auto add = [&](const float* __restrict__ nb, int64_t nend) __attribute__((always_inline)) {
      int64_t b = tid >> 3;
      for (; b + 3 * kStep < nend; b += 4 * kStep) {
        float y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = nb[b + u * kStep];
#pragma unroll
        for (int u = 0; u < 4; ++u) acc += y[u];
      }
      for (; b < nend; b += kStep) acc += nb[b];
    };
    const int64_t nblk = t.nblk <= kNormFixDirect ? 0 : base / kNormFixSegs;  // uniform
    add(t.nbsum + c * t.nblk, nblk);
    add(t.nsum + c * t.nseg + nblk * kNormFixSegs, base - nblk * kNormFixSegs);
    est[c][tid >> 3] = acc;  // scratch: 32 partials per chain
  }
  __syncthreads();
  if (tid < 8) {
    float acc = 0.0f;
    for (int k = 0; k < kThreads / 8; ++k) acc += est[tid][k];
    base_l[tid] = acc;
  }
  __syncthreads();
  // this item's segments (v: this thread's segment's sums of squares, 0 past the tensor's segments):
  // an exclusive scan over the threads, per chain
  float incl[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) incl[c] = v[c];
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float y = __shfl_up(incl[c], o, kWave);
      incl[c] += lane >= o ? y : 0.0f;
    }
  }
  if (lane == kWave - 1) {
#pragma unroll
    for (int c = 0; c < 8; ++c) part[wid][c] = incl[c];
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float off = base_l[c];
    for (int k = 0; k < kThreads / kWave; ++k) off += k < wid ? part[k][c] : 0.0f;
    est[c][tid] = off + (incl[c] - v[c]);
  }
  __syncthreads();
}


// Writes the records of the chains in mask from a rebuild under a binade pair per chain (Ea[c], Ea[c] + 1).
__device__ __forceinline__ void norm_write_records_pc(const DevTensor& t, int64_t seg, const int (&Ea)[8],
                                                      uint32_t mask, int lane, const NormAcc& a) {
  uint32_t acc[16];
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    acc[v] = a.val_a(v, Ea[v]);
    acc[8 + v] = a.val_b(v, Ea[v]);
  }
  norm_lane_sums<16>(acc, lane);  // lane 4c: chain c under Ea[c]; lane 32 + 4c: under Ea[c] + 1
  const int c = (lane >> 2) & 7;
  int Ec = Ea[0];
#pragma unroll
  for (int v = 1; v < 8; ++v) Ec = c == v ? Ea[v] : Ec;
  if ((lane & 3) == 0 && ((mask >> c) & 1u)) {
    const int64_t nseg = t.nseg;
    const uint32_t sum = min(acc[0], kNormFull);
    if (lane < 32) {
      t.nrec[c * nseg + seg] = uint32_t(Ec + 256) | kRecTwo;
      t.nrec[(8 + c) * nseg + seg] = sum;
    } else {
      t.nrec[(16 + c) * nseg + seg] = sum;
    }
  }
}

// Records rebuilt under each chain's own estimate.  A work item is t.nfseg consecutive segments
// of one tensor, one per thread: the chains' estimates at each segment (norm_item_estimates, taken as
// within [-2%, +0.5%] of the chain) are checked against the segment's eight records, and the segments
// where a record's binades do not cover a chain's are listed in LDS and shared out to the wavefronts,
// which rebuild them a segment at a time under each chain's own candidates Ea and Ea + 1 (both sums
// always).  FORM as for k_norm_seg.  The whole segments of a tensor that k_norm_seg2d takes (nseg0 > 0)
// read their column factors from LDS, staged once per tensor as k_norm_seg2d stages them.
template <typename TG, int FORM>
__global__ __launch_bounds__(kThreads) void k_norm_fix(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                       const int64_t* __restrict__ wstart, int ntens, Hp hp) {
  extern __shared__ float cl[];            // column factors (launches with tensors that k_norm_seg2d takes)
  __shared__ uint32_t list[kNormFixSegs];  // (thread << 8) | mask of the chains to rebuild
  __shared__ int nlist;
  __shared__ float est_l[8][kNormFixSegs];
  __shared__ float part[kThreads / kWave][8];
  __shared__ float base_l[8];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int64_t total = wstart[ntens];
  int32_t staged = -1;
  for (int64_t w = blockIdx.x; w < total; w += gridDim.x) {
    const int slot = find_slot(wstart, ntens, w);
    const int32_t ti = tids[slot];
    const DevTensor& t = T[ti];
    const int64_t nseg = t.nseg;
    const int64_t base = (w - wstart[slot]) * t.nfseg;
    const int64_t seg = base + tid, end = min(nseg, base + t.nfseg);  // of this item
    if (tid == 0) nlist = 0;
    // this thread's segment's sums of squares and record words, loaded before the estimates' sums
    float v[8];
    uint32_t w0s[8];
    {
      const int64_t sc = seg < end ? seg : end - 1;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        v[c] = t.nsum[c * nseg + sc];
        w0s[c] = t.nrec[c * nseg + sc];
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = seg < end ? v[c] : 0.0f;
    }
    norm_item_estimates(t, base, v, est_l, part, base_l);  // synchronises the workgroup
    uint32_t need = 0;
    if (seg < end) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float est = est_l[c][tid];
        const uint32_t w0 = w0s[c];
        const int Ea = int(w0 & 511u) - 256;
        const bool two = (w0 & kRecTwo) != 0;
        const int lo = norm_est_binade(est * 0.98f), hi = norm_est_binade(est * 1.005f);
        const bool ok = (lo == Ea || (two && lo == Ea + 1)) && (hi == Ea || (two && hi == Ea + 1));
        need |= ok ? 0u : (1u << c);
      }
    }
    if (need != 0) list[atomicAdd(&nlist, 1)] = (uint32_t(tid) << 8) | need;
    __syncthreads();
    const int n = nlist;
    const int64_t main = t.N - (t.N & 7);
    constexpr bool kLds = FORM != kNormAny;
    if (kLds && n > 0 && t.nseg0 > 0 && ti != staged) {  // uniform over the workgroup
      norm_stage_cols<FORM == kNormRows>(t, cl);
      __syncthreads();
      staged = ti;
    }
    for (int k = wid; k < n; k += kThreads / kWave) {  // uniform over the wavefront
      const uint32_t e = list[k];
      const int64_t sf = base + (e >> 8);
      int Ea[8];
      NormAcc a;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        bool two;
        norm_candidates(est_l[c][e >> 8], Ea[c], two);
        a.init(c, Ea[c]);
      }
      const int64_t f0 = sf * kNormSegElems, f1 = min(f0 + kNormSegElems, main);
      if (kLds && sf < t.nseg0) {  // uniform over the wavefront
#pragma unroll 1
        for (int h = 0; h < kNormChunks; h += kNormGroup) {
          float x[kNormGroup][8];
#pragma unroll
          for (int q = 0; q < kNormGroup; ++q)
            norm_chunk_lds<TG, FORM == kNormRows>(t, cl, uint32_t(f0 + (h + q) * 512 + lane * 8), x[q]);
#pragma unroll
          for (int q = 0; q < kNormGroup; ++q)
#pragma unroll
            for (int v = 0; v < 8; ++v) a.add<true>(v, x[q][v]);
        }
      } else {
#pragma unroll 1
        for (int h = 0; h < kNormChunks; h += kNormGroup) {
          float x[kNormGroup][8];
#pragma unroll
          for (int q = 0; q < kNormGroup; ++q) norm_chunk_x<TG, FORM>(t, f0 + (h + q) * 512 + lane * 8, f1, hp, x[q]);
#pragma unroll
          for (int q = 0; q < kNormGroup; ++q)
#pragma unroll
            for (int v = 0; v < 8; ++v) a.add<true>(v, x[q][v]);
        }
      }
      norm_write_records_pc(t, sf, Ea, e & 255u, lane, a);
    }
    __syncthreads();  // the list is reused by the next item
  }
}

// ---------------------------------------------------------------------------
// walk
// ---------------------------------------------------------------------------
constexpr uint32_t kNormSat = 1u << 25;  // saturating integer sums: anything >= 2^24 leaves the binade
__device__ __forceinline__ uint32_t sat_add(uint32_t a, uint32_t b) { return min(a + b, kNormSat); }

// Cross-lane steps of the walk, all 64 lanes active.  DPP: row_shr:n (0x110 + n; lanes shifted in from
// before their row's start read 0), row_bcast:15 (0x142) and row_bcast:31 (0x143) with row masks
// (rows outside them add 0), wave_shr:1 (0x138).
template <int CTRL, int ROWS, bool BOUND>
__device__ __forceinline__ uint32_t norm_dpp(uint32_t v) {
  return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, ROWS, 0xf, BOUND));
}
// inclusive scan of saturating sums over the wavefront, in lane order
__device__ __forceinline__ uint32_t norm_wave_scan(uint32_t v) {
  v = sat_add(v, norm_dpp<0x111, 0xf, true>(v));
  v = sat_add(v, norm_dpp<0x112, 0xf, true>(v));
  v = sat_add(v, norm_dpp<0x114, 0xf, true>(v));
  v = sat_add(v, norm_dpp<0x118, 0xf, true>(v));  // each row of 16 scanned
  v = sat_add(v, norm_dpp<0x142, 0xa, false>(v));  // rows 1 and 3 add the totals of rows 0 and 2
  v = sat_add(v, norm_dpp<0x143, 0xc, false>(v));  // rows 2 and 3 add the total of rows 0 and 1
  return v;
}
// the inclusive value of the previous lane (0 for lane 0)
__device__ __forceinline__ uint32_t norm_wave_prev(uint32_t incl) { return norm_dpp<0x138, 0xf, true>(incl); }
// lane `src`'s value (src uniform)
__device__ __forceinline__ uint32_t norm_lane(uint32_t v, int src) { return uint32_t(__builtin_amdgcn_readlane(int(v), src)); }
__device__ __forceinline__ float norm_lane(float v, int src) { return __uint_as_float(norm_lane(__float_as_uint(v), src)); }

// The x of the 8 elements of a chain at flat indices e0, e0 + 8, ..., e0 + 56 (the first n of them, n <= 8, lie in
// the segment; the others are 0).  A matrix's rows and columns follow from the first element's by one wrap each
// (rows of at least 8 elements); other tensors divide for every element.
template <typename TG>
__device__ __forceinline__ void norm_x_chain8(const DevTensor& t, int64_t e0, int n, const Hp& hp, float (&x)[8]) {
  if (t.factored && t.P == 1 && t.idx32 && t.C >= 8) {  // uniform
    using GS = typename TG::storage;
    const CAME8_GLOBAL GS* __restrict__ g = gbl(static_cast<const GS*>(t.g));
    const CAME8_GLOBAL float* __restrict__ rf = gbl(t.rfac);
    const CAME8_GLOBAL float* __restrict__ cf = gbl(t.cfac);
    const uint32_t C = uint32_t(t.C), f = uint32_t(e0);
    uint32_t row = udiv_magic(f, t.mC, t.sC), col = f - row * C;
    const uint32_t row0 = row, col0 = col;
    float gv[8], a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {  // an element past the segment reads the first one
      const bool in = j < n;
      gv[j] = TG::load(g[in ? f + 8u * uint32_t(j) : f]);
      a[j] = rf[in ? row : row0];
      b[j] = cf[in ? col : col0];
      col += 8u;
      const bool wrap = col >= C;
      col -= wrap ? C : 0u;
      row += wrap ? 1u : 0u;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = j < n ? (a[j] * b[j]) * gv[j] : 0.0f;
    return;
  }
  int64_t e[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) e[j] = e0 + (j < n ? 8 * j : 0);
  norm_x_any8<TG>(t, e, hp, x);
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = j < n ? x[j] : 0.0f;
}

// Replays chain c over segment seg from s, equal to the reference's serial fmaf loop bit for bit (one
// wavefront).  Lane l holds the chain's elements 8l .. 8l + 7 of the segment.  A round takes every
// remaining element's increment under s's binade, a saturating prefix sum of them in element order,
// and the first element that is a tie or whose prefix takes the chain out of the binade; the
// elements before it are one integer add, that element is one fmaf, and the next round starts after
// it.  A finite chain only grows, so the rounds are the segment's binade crossings and special
// elements, plus one.  An infinite chain changes only at a NaN element; a NaN chain not at all.
template <typename TG>
__device__ float norm_replay(const DevTensor& t, int c, int64_t seg, float s, const Hp& hp) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t main = t.N - (t.N & 7);
  const int64_t f0 = seg * kNormSegElems;
  const int cnt = int(min(int64_t(kNormChainSeg), (main - f0) / 8));  // at least 1
  // this lane's elements; a lane wholly past the segment's end reads the segment's first ones and counts for nothing
  const int mine = min(max(cnt - lane * 8, 0), 8);
  float x[8];
  norm_x_chain8<TG>(t, f0 + 64 * int64_t(mine > 0 ? lane : 0) + c, mine, hp, x);
  if (s == 0.0f) {
    // A chain's first segment crosses a binade every few elements, and its early increments keep many
    // fractional bits, so ties are common too: instead of a round per crossing or tie, its elements are
    // applied one by one (the reference's own loop), each broadcast from its lane.  Elements past the
    // segment's end are 0, and fmaf(0, 0, s) is s, so the loop needs no branch.
#pragma unroll 1
    for (int l = 0; l < kWave; l += 2) {  // (unrolled whole, the loop's code takes longer to fetch than to run)
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const float xk = norm_lane(x[k & 7], l + (k >> 3));
        s = fmaf(xk, xk, s);
      }
    }
    return s;
  }
  int pos = 0;  // the elements before pos are applied
  while (pos < cnt) {  // uniform
    if (!(s <= 0x1.fffffep127f)) {
      if (s != s) break;
      uint32_t nanm = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = lane * 8 + j;
        nanm |= (k >= pos && k < cnt && x[j] != x[j]) ? (1u << j) : 0u;
      }
      const uint64_t bal = __ballot(nanm != 0);
      if (bal != 0) {
        const int fl = __builtin_ctzll(bal);
        const int jj = int(norm_lane(uint32_t(__builtin_ctz(nanm | 0x100u)), fl));
        float xe = x[0];
#pragma unroll
        for (int j = 1; j < 8; ++j) xe = jj == j ? x[j] : xe;
        xe = norm_lane(xe, fl);
        s = fmaf(xe, xe, s);
      }
      break;
    }
    const int E = norm_binade(s);
    const uint32_t m = norm_mant(s, E);
    const uint32_t room = kNormFull - m;  // an increment prefix that reaches this leaves the binade
    // this lane's increments as prefixes, from the pair of sums of the records (NormAcc); the first tie or
    // departure from the binade within the lane is an event, after which its prefixes mean nothing
    const uint32_t bits = uint32_t(E + 127) << 23;
    float even = __uint_as_float(bits), odd = __uint_as_float(bits + 1u);
    uint32_t incl[8], evm = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float xj = lane * 8 + j >= pos ? x[j] : 0.0f;  // (elements past the segment's end are 0)
      even = fmaf(xj, xj, even);
      odd = fmaf(xj, xj, odd);
      incl[j] = __float_as_uint(even) - bits;
      evm |= (incl[j] >= (1u << 23) || __float_as_uint(odd) - bits != incl[j] + 1u) ? (1u << j) : 0u;
    }
    const uint32_t winc = norm_wave_scan(min(incl[7], kNormSat));  // inclusive scan of the lanes' runs
    const uint32_t excl = norm_wave_prev(winc);
#pragma unroll
    for (int j = 0; j < 8; ++j) evm |= excl + min(incl[j], kNormSat) >= room ? (1u << j) : 0u;
    const uint64_t bal = __ballot(evm != 0);
    if (bal == 0) {
      s = norm_value(m + norm_lane(winc, kWave - 1), E);  // below room
      break;
    }
    const int fl = __builtin_ctzll(bal);
    const int j0 = __builtin_ctz(evm | 0x100u);  // this lane's first event (8: none)
    uint32_t before = excl;                      // the increments before that event, on lane fl
    float xe = x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
      before = j0 == j ? excl + incl[j - 1] : before;
      xe = j0 == j ? x[j] : xe;
    }
    const int jj = int(norm_lane(uint32_t(j0), fl));
    before = norm_lane(before, fl);
    xe = norm_lane(xe, fl);
    s = fmaf(xe, xe, norm_value(m + before, E));
    pos = fl * 8 + jj + 1;
  }
  return s;
}

// The increment of a segment's record for a chain in binade E, or kNormSat when the record does not
// cover E.  With s = +inf (E = 128), a segment needs its replay only if it may hold a NaN: an
// exception, which saturates both sums.
__device__ __forceinline__ uint32_t norm_rec_add(uint32_t w0, uint32_t wa, uint32_t wb, int E) {
  const int Ea = int(w0 & 511u) - 256;
  const bool two = (w0 & kRecTwo) != 0;
  const uint32_t fin = E == Ea ? wa : ((two && E == Ea + 1) ? wb : kNormSat);
  const uint32_t inf = (wa >= kNormFull && (!two || wb >= kNormFull)) ? kNormSat : 0u;
  return E == 128 ? inf : fin;
}

constexpr int kNormWalkThreads = kWave;  // one wavefront per chain

// One wavefront per (tensor, chain).  A batch loads the records of kWave * kNormWalkSegs segments, a
// run of kNormWalkSegs per lane.  Then, from the chain's position: every lane sums its records under
// the chain's binade, a scan over the lanes finds the first segment whose record does not cover the
// binade or takes the chain out of it, every segment before it is skipped with its integer sum, that
// segment is replayed, and the scan resumes after it with the records already loaded.
template <typename TG>
__global__ __launch_bounds__(kNormWalkThreads) void k_norm_walk(const DevTensor* __restrict__ T,
                                                                const int32_t* __restrict__ tids,
                                                                const int64_t* __restrict__ wstart, int ntens, Hp hp) {
  const int lane = threadIdx.x;
  const int64_t total = wstart[ntens];
  // Workgroup w runs on XCD w % 8 (the dispatcher deals a launch's workgroups to the eight XCDs in
  // turn).  The items, eight per tensor (its chains), go to the XCDs in eight contiguous ranges, so
  // that a tensor's chains share one XCD's L2: they mostly replay the same segments at about the same
  // time, and each replay reads the cache lines that hold all eight chains' elements.
  const int64_t per = total % kXcds == 0 ? total / kXcds : 0;
  for (int64_t w = blockIdx.x; w < total; w += gridDim.x) {
    const int64_t item = per > 0 ? (w % kXcds) * per + w / kXcds : w;
    const int slot = find_slot(wstart, ntens, item);
    const DevTensor& t = T[tids[slot]];
    const int c = int(item - wstart[slot]);
    const int64_t nseg = t.nseg;
    const CAME8_GLOBAL uint32_t* __restrict__ W0 = gbl(t.nrec + c * nseg);
    const CAME8_GLOBAL uint32_t* __restrict__ WA = gbl(t.nrec + (8 + c) * nseg);
    const CAME8_GLOBAL uint32_t* __restrict__ WB = gbl(t.nrec + (16 + c) * nseg);
    // the first segment is replayed from zero without reading its record (a tensor of one segment forms
    // none)
    float s = nseg > 0 ? norm_replay<TG>(t, c, 0, 0.0f, hp) : 0.0f;
    int64_t seg = 1;
    while (seg < nseg && s == s) {  // a NaN chain stays NaN
      // the batch starts at a multiple of kNormWalkSegs; its segments before seg count for nothing
      const int64_t bstart = seg & ~int64_t(kNormWalkSegs - 1);
      const int64_t base = bstart + int64_t(lane) * kNormWalkSegs;
      const int64_t bend = min(nseg, bstart + int64_t(kWave) * kNormWalkSegs);
      uint32_t r0[kNormWalkSegs], ra[kNormWalkSegs], rb[kNormWalkSegs];
      if (base + kNormWalkSegs <= nseg) {  // consecutive records of each array: 4-dword loads
#pragma unroll
        for (int q = 0; q < kNormWalkSegs / 4; ++q) {
          const u32x4u a0 = *reinterpret_cast<const CAME8_GLOBAL u32x4u*>(W0 + base + 4 * q);
          const u32x4u aa = *reinterpret_cast<const CAME8_GLOBAL u32x4u*>(WA + base + 4 * q);
          const u32x4u ab = *reinterpret_cast<const CAME8_GLOBAL u32x4u*>(WB + base + 4 * q);
          r0[4 * q] = a0.x; r0[4 * q + 1] = a0.y; r0[4 * q + 2] = a0.z; r0[4 * q + 3] = a0.w;
          ra[4 * q] = aa.x; ra[4 * q + 1] = aa.y; ra[4 * q + 2] = aa.z; ra[4 * q + 3] = aa.w;
          rb[4 * q] = ab.x; rb[4 * q + 1] = ab.y; rb[4 * q + 2] = ab.z; rb[4 * q + 3] = ab.w;
        }
      } else {  // the array's end: clamped loads (the records past it count for nothing)
#pragma unroll
        for (int j = 0; j < kNormWalkSegs; ++j) {
          const int64_t k = min(base + j, nseg - 1);
          r0[j] = W0[k];
          ra[j] = WA[k];
          rb[j] = WB[k];
        }
      }
      while (seg < bend && s == s) {  // the segments [seg, bend) of this batch
        const bool inf = !(s <= 0x1.fffffep127f);
        const int E = inf ? 128 : norm_binade(s);
        const uint32_t m = inf ? 0u : norm_mant(s, E);
        const uint32_t room = kNormFull - m;  // the chain leaves its binade once its increments reach this
        // this lane's run: the sum of its records from seg on, up to the first one that stops the chain
        uint32_t add[kNormWalkSegs], run = 0;
        bool stop = false;
#pragma unroll
        for (int j = 0; j < kNormWalkSegs; ++j) {
          add[j] = norm_rec_add(r0[j], ra[j], rb[j], E);
          if (base + j >= seg && base + j < bend && !stop) {
            if (add[j] >= kNormSat) stop = true;
            else run = sat_add(run, add[j]);
          }
        }
        // inclusive scan of the runs over the lanes (saturating sums, in lane order)
        const uint32_t incl = norm_wave_scan(run);
        const uint32_t excl = norm_wave_prev(incl);  // exact while the chain has not left its binade
        const uint32_t tot = norm_lane(incl, kWave - 1);
        // the first lane whose run is cut short or takes the chain out of its binade
        const uint64_t bal = __ballot(stop || sat_add(excl, run) >= room);
        if (bal == 0) {
          if (!inf) s = norm_value(m + tot, E);  // tot < room
          seg = bend;
          break;
        }
        const int first = __builtin_ctzll(bal);
        uint32_t acc = excl;
        int64_t k = max(base, seg);
#pragma unroll
        for (int j = 0; j < kNormWalkSegs; ++j) {
          if (k == base + j && k < bend && add[j] < kNormSat && acc + add[j] < room) {
            acc += add[j];
            k = base + j + 1;
          }
        }
        const uint32_t mm = m + norm_lane(acc, first);
        const int64_t ks = int64_t(norm_lane(uint32_t(k), first)) | (int64_t(norm_lane(uint32_t(uint64_t(k) >> 32), first)) << 32);
        s = norm_replay<TG>(t, c, ks, inf ? s : norm_value(mm, E), hp);
        seg = ks + 1;
      }
    }
    if (lane == 0) t.nchain[c] = s;
  }
}

// The eight accumulators added left to right, then the N % 8 tail elements in torch's order (a block
// of four rounded squares added one at a time when four or more remain, then the rest as fused
// multiply-adds), sqrt, and the clip divisor.  A thread per tensor.
template <typename TG>
__global__ __launch_bounds__(kThreads) void k_norm_final(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                         int ntens, Hp hp) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k >= ntens) return;
  const DevTensor& t = T[tids[k]];
  float b = t.nchain[0];
  for (int j = 1; j < 8; ++j) b = b + t.nchain[j];
  int64_t d = t.N - (t.N & 7);
  if (t.N - d >= 4) {
    for (const int64_t e = d + 4; d < e; ++d) {
      const float u = u_at<TG>(t, d, hp);
      const float uu = u * u;  // rounded on its own (the build does not contract)
      b = b + uu;
    }
  }
  for (; d < t.N; ++d) {
    const float u = u_at<TG>(t, d, hp);
    b = fmaf(u, u, b);
  }
  const float c = clip_from_norm(sqrtf(b), t.N, hp);
  t.clip[0] = c;
  t.clip[1] = rcp_for_div(c);
}

// ---------------------------------------------------------------------------
// small tensors: the whole step in one workgroup
// ---------------------------------------------------------------------------
// A 1-D tensor or a matrix (prefix 1) of at most kLargeElems elements with at most kSmallStates rows and columns takes
// one workgroup for all of its step: the passes above are a dozen dependent launches of a few microseconds each, which
// is all the time a small tensor takes (a 96x200 layer, a 16x1280 adapter: 5 to 15 us a launch, 150 us a step).  The
// update (then u - m, then m) stays in LDS, where the sums over rows and columns and the eight serial chains of the clip
// norm read it; a matrix's momentum is formed twice, as in the passes, since LDS holds one float an element.  The
// arithmetic is that of the passes.  What bounds it is latency: the chains (4.6 ns an element of one), a memory round
// trip per eight elements of a thread and operand, and the sums.  Two sizes: 256 threads for up to kSmallElems elements,
// several workgroups a CU, and 1024 threads, whose LDS may fill a CU.  A step of 96x200, 96, 10x96 and 10: 161 us in
// twelve launches, 61 in this one; 192 adapters of 16x640 to 16x2048: 333 us in 17, 95 in this one.
constexpr int kSmallThreads = 256, kLargeThreads = 1024;
constexpr int kSmallElems = 2048, kLargeElems = 32768;
constexpr int64_t kSmallStates = 2560;  // rows + columns: two floats each beside kLargeElems floats of LDS
// LDS of a workgroup of nt threads for tensors of up to n elements and s states
constexpr size_t small_lds(int nt, int64_t n, int64_t s) { return size_t(nt) * 8 + size_t(n) * 4 + size_t(s) * 8; }

// Sums over the rows and the columns of val(e)^2 of an R x C matrix, in fp64 and a fixed order; row(r, s) and
// col(j, s) are each called by one thread.  Four values at a time, so that their loads overlap (past the end: a value
// that exists, counted as zero).  dsum: NT doubles of LDS.  Every thread calls it; it synchronises before the columns
// are finished, not after.
template <typename Val>
__device__ __forceinline__ double small_sum4(Val val, int e0, int step, int n) {  // n values from e0, step apart
  double s = 0.0;
#pragma unroll 1
  for (int i = 0; i < n; i += 4) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = val(e0 + min(i + k, n - 1) * step);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double d = i + k < n ? double(v[k]) : 0.0;
      s = fma(d, d, s);
    }
  }
  return s;
}
template <int NT, typename Val, typename RowFn, typename ColFn>
__device__ __forceinline__ void small_sums(Val val, int R, int C, double* dsum, RowFn row, ColFn col) {
  const int tid = threadIdx.x;
  int lg = 0;  // 2^lg lanes of a row: about four values each
  while (lg < 6 && (4 << lg) < C) ++lg;
  const int G = 1 << lg, li = tid & (G - 1);
  for (int r0 = 0; r0 < R; r0 += NT >> lg) {  // uniform
    const int r = r0 + (tid >> lg);
    double s = 0.0;
    if (r < R && li < C) s = small_sum4(val, r * C + li, G, (C - li + G - 1) >> lg);
    for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, kWave);
    if (r < R && li == 0) row(r, s);
  }
  if (C >= NT) {
    for (int j = tid; j < C; j += NT) col(j, small_sum4(val, j, C, R));
    __syncthreads();
  } else {
    const int H = min(kWave, NT / C);  // threads of a column, every H-th row each
    const int h = tid / C, j = tid - h * C;
    if (h < H) dsum[tid] = h < R ? small_sum4(val, h * C + j, H * C, (R - h + H - 1) / H) : 0.0;
    __syncthreads();
    if (tid < C) {
      double s = dsum[tid];
      for (int k = 1; k < H; ++k) s += dsum[k * C + tid];
      col(tid, s);
    }
  }
}

// Codes and scales of n values in LDS, a wavefront per block of B (any size; a short block is zero padded).  A lane
// holds its first four values of a block (all of them up to B = 256).
template <bool SIGNED, int NW>
__device__ __forceinline__ void small_quant(const float* x, int n, int B, void* q, float* a) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nb = (n - 1) / B + 1;  // n >= 1; n + B may be past 2^31
  CAME8_GLOBAL uint8_t* qb = gbl(static_cast<uint8_t*>(q));
#pragma unroll 1
  for (int blk = wid; blk < nb; blk += NW) {
    const int i0 = blk * B, i1 = min(i0 + B, n);
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = x[min(i0 + lane + k * kWave, i1 - 1)];  // past the end: the last one again
    float mx = nan_max(nan_max(quant_val<SIGNED>(v[0]), quant_val<SIGNED>(v[1])),
                       nan_max(quant_val<SIGNED>(v[2]), quant_val<SIGNED>(v[3])));
    if (!SIGNED && i1 - i0 < B) mx = nan_max(mx, 0.0f);
    for (int i = i0 + lane + 4 * kWave; i < i1; i += kWave) mx = nan_max(mx, quant_val<SIGNED>(x[i]));
    const float raw = group_max<64>(mx), am = fix_absmax(raw), rcp = rcp_for_div(am);
    const bool fast = rcp == rcp && raw == raw;
    uint32_t c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = quant_code<SIGNED>(v[k], am, rcp, fast);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (i0 + lane + k * kWave < i1) qb[i0 + lane + k * kWave] = uint8_t(c[k]);
    for (int i = i0 + lane + 4 * kWave; i < i1; i += kWave) qb[i] = uint8_t(quant_code<SIGNED>(x[i], am, rcp, fast));
    if (lane == 0) a[blk] = am;
  }
}

// sum over the workgroup of one double a thread, in a fixed order (every thread gets it; synchronises)
template <int NT>
__device__ __forceinline__ double small_total(double v, double* dsum) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  v = wave_sum(v);
  __syncthreads();  // dsum's readers are done
  if (lane == 0) dsum[wid] = v;
  __syncthreads();
  double s = dsum[0];
#pragma unroll
  for (int k = 1; k < NT / kWave; ++k) s += dsum[k];
  return s;
}

// This thread's elements e = tid, tid + NT, ... of an R x C matrix (or a row of C), U at a time: load(e, k) of all U,
// then calc(row, col, k) of all, then store(e, k) of those that exist (the others are the last element again).
template <int NT, int U, typename Load, typename Calc, typename Store>
__device__ __forceinline__ void small_each(int N, int R, int C, Load load, Calc calc, Store store) {
  const int tid = threadIdx.x;
  int row = tid / C, col = tid - row * C;
  const int dq = NT / C, dr = NT - dq * C;  // the next element's row and column follow from this one's
#pragma unroll 1
  for (int e0 = tid; e0 < N; e0 += U * NT) {
#pragma unroll
    for (int k = 0; k < U; ++k) load(uint32_t(min(e0 + k * NT, N - 1)), k);
#pragma unroll
    for (int k = 0; k < U; ++k) {
      calc(min(row, R - 1), col, k);
      row += dq;
      col += dr;
      const bool wrap = col >= C;
      col -= wrap ? C : 0;
      row += wrap ? 1 : 0;
    }
#pragma unroll
    for (int k = 0; k < U; ++k)
      if (e0 + k * NT < N) store(uint32_t(e0 + k * NT), k);
  }
}

template <typename TP, typename TG, int NT>
__global__ __launch_bounds__(NT) void k_small_step(const DevTensor* __restrict__ T, const int32_t* __restrict__ tids,
                                                   int ntens, int exact_norm, Hp hp) {
  using GS = typename TG::storage;
  using PS = typename TP::storage;
  extern __shared__ double small_mem[];
  __shared__ float clip_s;
  constexpr int NW = NT / kWave;
  constexpr int U = 8;  // elements a thread loads together
  const int tid = threadIdx.x, lane = tid & 63;
  for (int item = blockIdx.x; item < ntens; item += gridDim.x) {
    const DevTensor& t = T[tids[item]];
    const bool fact = t.factored != 0, f32 = t.fp32st != 0;
    const int N = int(t.N), R = int(t.R), C = int(t.C);
    double* dsum = small_mem;
    float* x = reinterpret_cast<float*>(small_mem + NT);  // N
    float* fac = x + N;                                   // row factors r_i [R], column factors c_j [C]
    float* stv = fac + (fact ? R + C : 0);                // the new states, alike; then rr_i, cr_j
    const CAME8_GLOBAL GS* __restrict__ g = gbl(static_cast<const GS*>(t.g));
    const CAME8_GLOBAL float* m32 = gbl(static_cast<const float*>(st_m(t)));
    const CAME8_GLOBAL int8_t* mq = gbl(static_cast<const int8_t*>(t.mq));
    const CAME8_GLOBAL float* ma = gbl(static_cast<const float*>(t.ma));
    const CAME8_GLOBAL float* v32 = gbl(static_cast<const float*>(st_sq_row(t)));
    const CAME8_GLOBAL uint8_t* vq = gbl(static_cast<const uint8_t*>(t.rq));
    const CAME8_GLOBAL float* va = gbl(static_cast<const float*>(t.ra));
    // e / B for e < 2^15: the quotient of e + 1/2 is at least 1 / (2B) from a whole number, its error below 2^-8 / B
    const float invB = 1.0f / float(hp.B);
    auto blk = [&](uint32_t e) __attribute__((always_inline)) { return uint32_t((float(e) + 0.5f) * invB); };
    // the old momentum of element e of the 8-bit states (no branch, which would make several elements' loads wait for
    // each other: an infinite or NaN scale / 127 is itself)
    auto m_q8 = [&](uint32_t e) __attribute__((always_inline)) {
      const float a = ma[blk(e)];
      return float(mq[e]) * (fabsf(a) <= 0x1.fffffep127f ? div_fast(a, kSignedQ, kRcpSignedQ) : a);
    };
    // the row and column states (RES: of the residual) from the sums of the squares in x: the new states into stv and
    // to memory (codes and scales, or fp32 states), factors into fac (RES: over the states in stv).  Ends synchronised.
    auto states = [&](auto RES) __attribute__((always_inline)) {
      constexpr bool kRes = decltype(RES)::value;
      const float beta = kRes ? hp.b3 : hp.b2, alpha = kRes ? hp.a3 : hp.a2;
      const double eps = double(kRes ? hp.eps1 : hp.eps0);
      const float fC = float(C), fR = float(R), invC = 1.0f / fC;
      float* rst = kRes ? t.ra : st_sq_row(t);  // fp32 states
      float* cst = kRes ? t.ca : st_sq_col(t);
      uint8_t* rq = t.rq + (kRes ? R : 0);
      uint8_t* cq = t.cq + (kRes ? C : 0);
      float* ra = t.ra + (kRes ? t.nbr : 0);
      float* ca = t.ca + (kRes ? t.nbc : 0);
      double rs = 0.0;
      small_sums<NT>([&](int e) { return x[e]; }, R, C, dsum, [&](int r, double s) {
        const float old = f32 ? rst[r] : deq_u8(rq[r], ra[blk_of(r, hp)]);
        const float tot = float(s + double(C) * eps);
        const float v = fmaf(kRes ? tot / fC : tot * invC, alpha, old * beta);
        stv[r] = v;
        rs += v;
      }, [&](int j, double s) {
        const float old = f32 ? cst[j] : deq_u8(cq[j], ca[blk_of(j, hp)]);
        stv[R + j] = clamp_min_tiny(fmaf(float(s + double(R) * eps) / fR, alpha, old * beta));
      });
      const float mean = row_mean_of_sum(t, small_total<NT>(rs, dsum));  // synchronises: stv is whole
      if constexpr (!kRes)
        for (int r = tid; r < R + C; r += NT) fac[r] = rsqrt_ref(r < R ? stv[r] / mean : stv[r]);
      if (f32) {
        for (int r = tid; r < R; r += NT) rst[r] = stv[r];
        for (int j = tid; j < C; j += NT) cst[j] = stv[R + j];
      } else {  // (every old code was read before the barriers above)
        small_quant<false, NW>(stv, R, hp.B, rq, ra);
        small_quant<false, NW>(stv + R, C, hp.B, cq, ca);
      }
      __syncthreads();
      if constexpr (kRes) {
        for (int r = tid; r < R + C; r += NT) stv[r] = rsqrt_ref(r < R ? stv[r] / mean : stv[r]);
        __syncthreads();
      }
    };
    // ---- the update, into x ----
    float gv[U], vo[U];
    auto load_v = [&](uint32_t e, int k) __attribute__((always_inline)) {  // a 1-D tensor's gradient and old second moment
      gv[k] = TG::load(g[e]);
      vo[k] = f32 ? v32[e] : deq_u8(vq[e], va[blk(e)]);
    };
    if (fact) {
      small_each<NT, U>(N, R, C, [&](uint32_t e, int k) { gv[k] = TG::load(g[e]); }, [](int, int, int) {},
                        [&](uint32_t e, int k) { x[e] = gv[k]; });
      __syncthreads();
      states(std::false_type{});
      small_each<NT, U>(N, R, C, [&](uint32_t e, int k) { gv[k] = x[e]; },
                        [&](int row, int col, int k) { gv[k] = (fac[row] * fac[R + col]) * gv[k]; },
                        [&](uint32_t e, int k) { x[e] = gv[k]; });
    } else {
      small_each<NT, U>(N, 1, N, load_v, [&](int, int, int k) { gv[k] = rsqrt_ref(vec_v_from(gv[k], vo[k], hp)) * gv[k]; },
                        [&](uint32_t e, int k) { x[e] = gv[k]; });
    }
    __syncthreads();
    // ---- the clip divisor ----
    float norm = 0.0f;
    if (exact_norm) {
      double s = 0.0;
      for (int e = tid; e < N; e += NT) s = fma(double(x[e]), double(x[e]), s);
      norm = float(sqrt(small_total<NT>(s, dsum)));
    } else if (tid < kWave) {  // lane c < 8: chain c; then the chains and the tail in the reference's order (k_norm_final)
      const int n8 = N >> 3;
      const float* xc = x + (lane & 7);
      float acc = 0.0f;
      // 16 elements load while the 16 before them are added
      auto load16 = [&](float (&y)[16], int i) __attribute__((always_inline)) {
        const int j = i + 16 <= n8 ? i : 0;  // past the end: unused
#pragma unroll
        for (int k = 0; k < 16; ++k) y[k] = xc[(j + k) * 8];
        __builtin_amdgcn_sched_barrier(0);
      };
      auto add16 = [&](const float (&y)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = fmaf(y[k], y[k], acc);
        __builtin_amdgcn_sched_barrier(0);
      };
      int i = 0;
      if (n8 >= 16) {
        float y[16], z[16];
        load16(y, 0);
#pragma unroll 1
        for (; i + 32 <= n8; i += 32) {
          load16(z, i + 16);
          add16(y);
          load16(y, i + 32);
          add16(z);
        }
        if (i + 16 <= n8) {
          add16(y);
          i += 16;
        }
      }
      for (; i < n8; ++i) acc = fmaf(xc[i * 8], xc[i * 8], acc);
      float b = norm_lane(acc, 0);
#pragma unroll
      for (int k = 1; k < 8; ++k) b = b + norm_lane(acc, k);
      int d = n8 * 8;
      if (N - d >= 4) {
        for (const int e = d + 4; d < e; ++d) {
          const float sq = x[d] * x[d];
          b = b + sq;
        }
      }
      for (; d < N; ++d) b = fmaf(x[d], x[d], b);
      norm = sqrtf(b);
    }
    if (tid == 0) {
      const float c = clip_from_norm(norm, t.N, hp);
      clip_s = c;
      t.clip[0] = c;
      t.clip[1] = rcp_for_div(c);
    }
    __syncthreads();
    const float clip = clip_s;
    // ---- the momentum: a vector's into x; of a matrix d = u - m for the residual's sums, and again for the write ----
    const bool h16 = !fact && !f32 && (hp.fp16u || t.fp16u);
    auto m_new = [&](float w, float mo) { return fmaf(w, hp.a1, mo * hp.b1); };
    float mo[U];
    small_each<NT, U>(N, 1, N, [&](uint32_t e, int k) {
      mo[k] = f32 ? m32[e] : m_q8(e);
      gv[k] = x[e];
    }, [&](int, int, int k) {
      const float w = (h16 ? round_f16(gv[k]) : gv[k]) / clip;
      const float m = m_new(w, mo[k]);
      gv[k] = fact ? w - m : m;
    }, [&](uint32_t e, int k) { x[e] = gv[k]; });
    __syncthreads();
    if (fact) states(std::true_type{});
    // ---- the parameter; the momentum into x ----
    {
      CAME8_GLOBAL PS* p = gbl(static_cast<PS*>(t.p));
      float po[U];
      if (fact) {
        small_each<NT, U>(N, R, C, [&](uint32_t e, int k) {
          gv[k] = TG::load(g[e]);
          po[k] = TP::load(p[e]);
          mo[k] = f32 ? m32[e] : m_q8(e);
        }, [&](int row, int col, int k) {
          gv[k] = m_new(((fac[row] * fac[R + col]) * gv[k]) / clip, mo[k]);
          po[k] = param_update<TP>(po[k], (stv[row] * stv[R + col]) * gv[k], hp);
        }, [&](uint32_t e, int k) {
          p[e] = TP::store(po[k]);
          x[e] = gv[k];
        });
      } else {
        small_each<NT, U>(N, 1, N, [&](uint32_t e, int k) {
          po[k] = TP::load(p[e]);
          gv[k] = x[e];
        }, [&](int, int, int k) { po[k] = param_update<TP>(po[k], gv[k], hp); }, [&](uint32_t e, int k) { p[e] = TP::store(po[k]); });
      }
    }
    __syncthreads();
    if (f32) {
      for (int e = tid; e < N; e += NT) st_m(t)[e] = x[e];
    } else {
      small_quant<true, NW>(x, N, hp.B, t.mq, t.ma);
    }
    if (!fact) {  // the second moment, formed again from the old one
      __syncthreads();
      small_each<NT, U>(N, 1, N, load_v, [&](int, int, int k) { gv[k] = vec_v_from(gv[k], vo[k], hp); }, [&](uint32_t e, int k) {
        if (f32) st_sq_row(t)[e] = gv[k];
        else x[e] = gv[k];
      });
      __syncthreads();
      if (!f32) small_quant<false, NW>(x, N, hp.B, t.rq, t.ra);
    }
    __syncthreads();  // the LDS is used again
  }
}

}  // namespace came8
