// bsattn_prefill.hip -- gfx950 (CDNA4) dense causal attention of a prefill
// chunk over a block-sparse cache (16-bit or affine-quantized).
//
// Built with -fno-honor-nans -mno-amdgpu-ieee: the scores are MFMA results
// (never signalling NaNs), so max trees compile to v_max3_f32 without the
// operand quieting IEEE mode asks for.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

// (the shared header's NaN-aware helpers are not used here)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wnan-infinity-disabled"
#include "bsattn_device.h"
#pragma clang diagnostic pop

namespace bsattn {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

template <int DT>
__device__ __forceinline__ f32x16 mfma32x32x16(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (DT == 0)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

typedef int16_t i16x2 __attribute__((ext_vector_type(2)));

// all bits of the 16-bit elements whose magnitude bits are `lim` or more
__device__ __forceinline__ u32x4 at_least16(u32x4 w, uint32_t lim) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t mag = w[k] & 0x7FFF7FFFu;
    const i16x2 l = {(int16_t)lim, (int16_t)lim};
    const i16x2 below = (__builtin_bit_cast(i16x2, mag) - l) >> 15;  // the difference's sign
    w[k] = ~__builtin_bit_cast(uint32_t, below);
  }
  return w;
}

// a workgroup barrier that orders LDS only: the global loads of later units
// stay in flight across it
__device__ __forceinline__ void unit_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// x of the lane 32 places away (the other half of a column's tokens)
__device__ __forceinline__ float pair_max(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

constexpr int kPfWaves = 8;           // waves per workgroup (half as many for few tiles: prefill_width)
constexpr int kPfCols = 32;           // MFMA columns per wave
constexpr int kPfSplits = 16;         // most parts a tile's tokens are split into
constexpr float kNoMax = -3.0e38f;    // running maximum of a column that has seen nothing

// one wave's share of a 32-token unit, as loaded: F of its 8 K and of its 8 V
// fragments (16 bytes a lane), or their codes and one token's scales
template <int KB, int F>
struct Staged {
  uint32_t k[F][KB / 4], v[F][KB / 4];
  u32x4 e;
};
template <int F>
struct Staged<0, F> {
  u32x4 k[F], v[F];
};

// ---------------------------------------------------------------------------
// dense causal attention for the last L tokens of each sequence (a prefill
// chunk whose keys / values were appended): query token i of a sequence
// holding T tokens sits at position T - L + i and attends to tokens
// [0, T - L + i] (the causal mask BaseKVCache.makeMask gives for n > 1).
// A wave owns 32 MFMA columns, each a (query token, q head) pair (32 / G
// tokens x the G heads of kv head h); the workgroup's W waves take
// consecutive tokens of one (sequence, kv head) and walk its tokens in units
// of 32, with an online softmax per column:
//   S^T[token][col] = K[token] . Q[col]        (A = K rows, B = Q^T)
//   O^T[dim][col]  += V^T[dim] . P^T[col]      (A = V^T, B = P^T)
// with v_mfma_f32_32x32x16.  S^T row r of a unit is its token
// 16 (r / 16) + 8 (r / 4 % 2) + 4 (r / 8 % 2) + r % 4, so that a lane's
// accumulator entries 8 kk .. 8 kk + 7 are tokens 16 kk + 8 (lane / 32) .. + 7
// of its column: the P^T operand of k-step kk, with no shuffles, against the
// V fragments as they are stored.  K fragments are read from LDS by row in
// the same way (16 bytes a lane from the fragment that holds them).
//
// The unit pipeline (one workgroup barrier per two units).  In step u a wave
//  - computes S of unit u + 1 (K from LDS) while it turns S of unit u into P,
//    then O += V P of unit u: products that depend on nothing in the
//    softmax, for the matrix cores to run beside it;
//  - writes its fragments of unit u + 3, which it loaded two steps ago, to
//    LDS and loads those of unit u + 5.
// The barrier ends the odd steps.  Between two of them (steps u and u + 1, u
// even) the waves read K of u + 1 and u + 2 and write u + 3 and u + 4: four
// slots; they read V of u and u + 1, keep that of u + 2 and write the same
// two: eight slots, by the unit's low bits.  What bounds it: the power that
// MFMAs and LDS reads take together (the clock falls to ~2.0 GHz), LDS reads
// (16 KiB a wave and unit) and the VALU work of a wave's softmax between its
// MFMAs (16 x 32 cycles a wave and unit, two waves per SIMD): ~70 VALU a unit
// and 16 exp2, 20 more for bf16 V.  Four waves of 64 columns, which halve the
// LDS reads and leave one wave per SIMD, took 2575 us where this took 2198.
//
// V of a bf16 cache is converted to fp16 on its way to LDS (exact for
// |v| < 65520 down to the fp16 normal range) for an fp16 PV product without
// the hi / lo split of P.  A value fp16 cannot take is left out there and the
// unit noted; the noted units are gone through once more after the last one,
// for those values alone, in bf16 with P as hi + lo from the cache's own
// fragments.  So are infinities and NaN of any cache's V in units that some
// columns do not see: a later token's reach no earlier query.
// Codes of an affine cache (KB = 4 / 8 bits, fp16 q / out) are dequantized on
// the way, as fp16 values fl16(scale * code + bias) (one packed fused
// multiply-add per pair, so each is the correctly rounded value).
//
// The workgroups of one (sequence, kv head, part) read the same units, so the
// flat workgroup index is remapped to give them consecutive indices within
// one XCD (workgroups are dealt to the 8 XCDs in turn): they then share that
// XCD's L2 instead of fetching every unit into all eight.  The tiles with the
// most tokens come first.
// nsplit > 1: each tile's units are cut into nsplit runs, whose unnormalised
// (o, m, l) go to po / pml for k_prefill_combine.
// The loop's counters, page lookup and addresses are scalar: workgroup indexes
// that come from divisions, and bounds made from them, pass through uniform(),
// or the compiler keeps them in vector registers and 64-bit vector products
// at every unit.
// Measured, 512-token chunks at 32k tokens, Hq 32, Hkv 8, with vector counters
// and a barrier at every unit -> with scalar ones and a barrier at every
// second unit -> now (no flags in the loop, nothing spilled): 8 sequences,
// bf16 2388 -> 2215 -> 2133 us (1022 TFLOP/s), int4 2494 -> 2391 -> 2373 us;
// one sequence, split in 4, 362 -> 297 -> 283 us; a prompt of 8191 fp16 tokens
// 575 -> 585 -> 562 us (16x16x32 MFMAs in 4-wave workgroups, one unit ahead:
// 2838, 2985, 1124 and 685 us).
// grid (ceil(L / (32 W / G)) * Hkv * n * nsplit), W = 8 or 4 waves
// ---------------------------------------------------------------------------
template <int DT, int KB, int W>
__global__ __launch_bounds__(64 * kPfWaves) void k_prefill(Geometry geo, SeqBatch sb, int L, int lg, int gx,
                                                          int nsplit, const uint16_t* __restrict__ q,
                                                          float sl2, uint16_t* __restrict__ out,
                                                          float* __restrict__ po, float* __restrict__ pml) {
  static_assert(KB == 0 || DT == 0, "quantized caches: fp16");
  // the running maximum a column's weights are taken against is raised only
  // when a unit's maximum exceeds it by more than 2^kLazy: the weights then
  // stay below 2^kLazy, and the rescaling of O^T (a pass over its registers)
  // is skipped for most units; O^T / l is unchanged by the choice
  constexpr float kLazy = 8.f;
  constexpr bool CV = KB == 0 && DT == 1;
  constexpr int F = 8 / W;  // K, and V, fragments of a unit that a wave loads: wave + W i
  using St = Staged<KB, F>;
  __shared__ __align__(16) u32x4 s_k[4][8 * 64], s_v[8][8 * 64];
  __shared__ __align__(16) u32x4 s_ent[KB ? W : 1][KB ? 32 : 1];  // each wave's copy of a unit's scales / biases
  // units whose V holds an element that is left to the end, bit x - odd0.  A
  // bf16 cache: any unit (tables are at most 12288 blocks wide).  Otherwise
  // those that only some columns see, at most 9: a word per wave, its own
  constexpr int ODDW = CV ? 2 * 12288 / 32 + 1 : W;
  __shared__ uint32_t s_odd[ODDW];
  __shared__ int s_anyodd;  // (CV) whether there are any
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 31, hh = lane >> 5;
  // XCD-grouped workgroup order (a bijection on [0, total))
  const int total = gridDim.x, flat = blockIdx.x, even = total & ~7;
  const int lid = flat < even ? (flat & 7) * (even >> 3) + (flat >> 3) : flat;
  const int run_of = uniform(lid / gx), tile = gx - 1 - (lid - run_of * gx);
  const int pair = uniform(run_of / nsplit), part = run_of - pair * nsplit;
  const int bi = uniform(pair / geo.hkv), h = pair - bi * geo.hkv;
  const int qpw = kPfCols >> lg;            // query tokens per wave
  const int twg = tile * W * qpw;           // the workgroup's first query token
  const bool active = uniform(twg + wave * qpw < L);
  const int seq = uniform(sb.ids[bi]);
  const int T = uniform(geo.meta[seq]);
  const int head = (h << lg) + (col & ((1 << lg) - 1));
  const int tq = twg + wave * qpw + (col >> lg);
  // scores are taken as (K . Q') * |sl2| with Q' = Q * sign(sl2): the sign
  // flip is exact, and a positive factor lets the block maximum be found on
  // the raw products.  A padding column (no query token) has Q = 0, sees
  // every token and is not stored.
  const uint32_t qflip = sl2 < 0.f ? 0x80008000u : 0u;
  const float sc = fabsf(sl2);
  const int pos = tq < L ? T - L + tq : T;
  u32x4 qf[8];
  {
    const uint16_t* src = q + q_row(sb, bi, head) + (size_t)min(tq, L - 1) * kHeadDim + 8 * hh;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = tq < L ? *(const u32x4*)(src + 16 * s) ^ qflip : u32x4{0u, 0u, 0u, 0u};
  }
  const int ksh = geo.tb == 64 ? 1 : 0;  // log2 of the units of a block
  const int last = T - L + min(L - 1, twg + W * qpw - 1);  // the workgroup's last position
  const int nunit = last / 32 + 1;
  // (at most 24576 units, of 12288 blocks, in at most 16 parts; kept in scalar
  // registers, so that the loop's counters, page lookups and addresses are
  // scalar too)
  const int ua = uniform((int)((uint32_t)nunit * part / nsplit)), ub = uniform((int)((uint32_t)nunit * (part + 1) / nsplit));
  // units below nfull are whole and visible to every column of the workgroup
  const int nfull = uniform(min((T - L + twg + 1) / 32, ub));
  const int odd0 = CV ? ua : nfull;
  // magnitude bits of infinity, and of the elements left to the end (bf16: from 65536)
  constexpr uint32_t INF = DT == 0 ? 0x7C00u : 0x7F80u, ODD = CV ? 0x4780u : INF;

  // --- units from memory: this wave's fragments, in the slab's own order
  const int32_t* bt = block_table(geo, seq);
  const int lastblk = last / geo.tb;
  int pbase = ua >> ksh;  // lane i of pagev: page of block pbase + i
  int pagev = bt[min(pbase + lane, lastblk)];
  const uint32_t lane16 = 16 * (threadIdx.x & 63);
  auto load = [&](int x, St& st) __attribute__((always_inline)) {
    x = max(min(x, ub - 1), ua);
    const int blk = x >> ksh, sub = x & ((1 << ksh) - 1);
    if (blk >= pbase + 64) {
      pbase = blk;
      pagev = bt[min(pbase + lane, lastblk)];
      __builtin_amdgcn_s_waitcnt(0x0F70);  // here, every 64 blocks, and not at each use of pagev
    }
    const int page = __builtin_amdgcn_readlane(pagev, blk - pbase);
    const uint8_t* slab = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes;
    const uint8_t *ks = slab + geo.k_off, *vs = slab + geo.v_off;
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const int f = wave + W * i;
      if constexpr (KB == 0) {
        st.k[i] = *(const u32x4*)(ks + (8 * sub + f) * 1024 + lane16);
        st.v[i] = *(const u32x4*)(vs + ((f << ksh) + sub) * 1024 + lane16);
      } else if constexpr (KB == 4) {
        st.k[i][0] = *(const uint32_t*)(ks + (2 * sub + (f >> 2)) * 1024 + 4 * (f & 3) + lane16);
        st.v[i][0] = *(const uint32_t*)(vs + (((f >> 2) << ksh) + sub) * 1024 + 4 * (f & 3) + lane16);
      } else {
        const uint2 a = *(const uint2*)(ks + (4 * sub + (f >> 1)) * 1024 + 8 * (f & 1) + lane16);
        const uint2 b = *(const uint2*)(vs + (((f >> 1) << ksh) + sub) * 1024 + 8 * (f & 1) + lane16);
        st.k[i][0] = a.x;
        st.k[i][1] = a.y;
        st.v[i][0] = b.x;
        st.v[i][1] = b.y;
      }
    }
    if constexpr (KB != 0) {
      const int x32 = lane & 31;
      st.e = *(const u32x4*)(slab + geo.sb_off + (((x32 >> 3) * (geo.tb >> 2)) + 8 * sub + (x32 & 7)) * 16);
    }
  };
  // f16 pairs (s * c + b): c from the f16 values OFF + c / INV_UNIT exactly
  [[maybe_unused]] auto deq = [&](u32x4 hv, const uint32_t* sp, const uint32_t* bp) __attribute__((always_inline)) {
    using QC = QCode<KB ? KB : 4>;
    const f16x2 unit2 = {(_Float16)QC::INV_UNIT, (_Float16)QC::INV_UNIT};
    const f16x2 off2 = {(_Float16)(-QC::OFF * QC::INV_UNIT), (_Float16)(-QC::OFF * QC::INV_UNIT)};
    u32x4 o4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // (a vector element is copied out first: __builtin_bit_cast of
      // hv[k] itself reads element 0 with this compiler)
      const uint32_t w = hv[k];
      const f16x2 c = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, w), unit2, off2);
      o4[k] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, sp[k]), c,
                                                                    __builtin_bit_cast(f16x2, bp[k])));
    }
    return o4;
  };
  [[maybe_unused]] auto codes = [&](const uint32_t* w) __attribute__((always_inline)) {
    if constexpr (KB == 4) return nib_to_f16(w[0]);
    else return byte_to_f16(w[0], w[1]);
  };
  // w without the elements that are left to the end, with the unit noted when
  // there are any
  auto drop = [&](int r, u32x4 w) __attribute__((always_inline)) {
    u16x2 big = {0, 0};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t mag = w[k] & 0x7FFF7FFFu;
      big = __builtin_elementwise_max(big, __builtin_bit_cast(u16x2, mag));
    }
    constexpr uint32_t UP = 0x10001u * (0x8000u - ODD);  // carries ODD and more into the sign bits
    if (__builtin_amdgcn_ballot_w64(((__builtin_bit_cast(uint32_t, big) + UP) & 0x80008000u) != 0u) != 0) {
      w &= ~at_least16(w, ODD);
      const int at = ua + r - odd0;
      if (lane == 0) {
        if constexpr (CV) {
          atomicOr(&s_odd[min(at >> 5, ODDW - 1)], 1u << (at & 31));
          s_anyodd = 1;
        } else {
          s_odd[wave] |= 1u << (at & 31);
        }
      }
    }
    return w;
  };
  // --- and into LDS, as 16-bit fragments; r: the unit's index from ua
  auto stage = [&](int r, const St& st, auto mask_tag, auto raw_tag) __attribute__((always_inline)) {
    constexpr bool RAW = decltype(raw_tag)::value;
    if constexpr (KB != 0) {
      // the unit's scale / bias entries through this wave's own LDS rows
      // (a wave's LDS accesses complete in order)
      s_ent[wave][lane & 31] = st.e;
      wave_lds_order();
    }
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const int f = wave + W * i;
      u32x4 kw, vw;
      if constexpr (KB == 0) {
        kw = st.k[i];
        vw = st.v[i];
        if constexpr (CV) {
          if constexpr (!RAW) vw = drop(r, vw);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t x = vw[k];
            vw[k] = cvt_pk<0>(__uint_as_float(x << 16), __uint_as_float(x & 0xFFFF0000u));
          }
        }
      } else {
        const uint32_t* ent = (const uint32_t*)s_ent[wave];
        {
          // row m of QK key tile t is token 8 (m / 4) + 4 t + m % 4 of the unit
          const int t = f >> 2, m = lane & 15;
          const int x = 8 * (m >> 2) + 4 * t + (m & 3);
          const uint32_t sel = (f & 2) ? 0x03020302u : 0x01000100u;  // dim group of k-step f & 3
          const uint32_t s2 = __builtin_amdgcn_perm(ent[4 * x], ent[4 * x], sel);
          const uint32_t b2 = __builtin_amdgcn_perm(ent[4 * x + 1], ent[4 * x + 1], sel);
          const uint32_t sp[4] = {s2, s2, s2, s2}, bp[4] = {b2, b2, b2, b2};
          kw = deq(codes(st.k[i]), sp, bp);
        }
        {
          // (v scale, v bias) of tokens 8 g + 2 k, 8 g + 2 k + 1 as f16 pairs
          const int g = lane >> 4;
          uint32_t sp[4], bp[4];
          const uint32_t sel = (f >> 2) ? 0x07060302u : 0x05040100u;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint2 e0 = *(const uint2*)(ent + 4 * (8 * g + 2 * k) + 2), e1 = *(const uint2*)(ent + 4 * (8 * g + 2 * k + 1) + 2);
            sp[k] = __builtin_amdgcn_perm(e1.x, e0.x, sel);
            bp[k] = __builtin_amdgcn_perm(e1.y, e0.y, sel);
          }
          vw = deq(codes(st.v[i]), sp, bp);
        }
      }
      if constexpr (decltype(mask_tag)::value) {
        // V of tokens past the sequence end (stale page data) is zeroed
        const int valid = T - 32 * (ua + r), g = lane >> 4;
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int tk = 8 * g + 2 * jj;
          vw[jj] &= (tk < valid ? 0x0000FFFFu : 0u) | (tk + 1 < valid ? 0xFFFF0000u : 0u);
        }
        if constexpr (!CV && !RAW)
          if (ua + r >= nfull) vw = drop(r, vw);
      }
      s_k[r & 3][f * 64 + lane] = kw;
      s_v[r & 7][f * 64 + lane] = vw;
    }
    if constexpr (KB != 0) wave_lds_order();
  };

  // --- this wave's columns
  float m = kNoMax, l = 0.f, thr = -INFINITY, lm = -INFINITY;
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
  // lane offsets (16-byte entries) of the K and V operands in a slot
  const int kl = ((col >> 3) & 1) * 256 + 8 * (col >> 4) + 4 * ((col >> 2) & 1) + (col & 3) + 16 * hh;
  const int vl = (col >> 4) * 64 + (col & 15) + 16 * hh;
  auto scores = [&](int r) __attribute__((always_inline)) {  // S^T of unit ua + r
    const u32x4* kp = s_k[r & 3] + kl;
    f32x16 a;
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) a = mfma32x32x16<DT>(kp[32 * s], qf[s], a);
    return a;
  };
  // the largest score of this lane's tokens, masked past the column's position
  auto lane_max = [&](f32x16& a, int r, auto mask_tag) __attribute__((always_inline)) {
    if constexpr (decltype(mask_tag)::value) {
      const int lim = pos - 32 * (ua + r) - 8 * hh;
#pragma unroll
      for (int i = 0; i < 16; ++i) a[i] = 16 * (i >> 3) + (i & 7) <= lim ? a[i] : -INFINITY;
    }
    float x = fmaxf(fmaxf(a[0], a[1]), a[2]), y = fmaxf(fmaxf(a[3], a[4]), a[5]);
    x = fmaxf(fmaxf(x, a[6]), a[7]);
    y = fmaxf(fmaxf(y, a[8]), a[9]);
    x = fmaxf(fmaxf(x, a[10]), a[11]);
    y = fmaxf(fmaxf(y, a[12]), a[13]);
    x = fmaxf(fmaxf(x, a[14]), a[15]);
    return fmaxf(x, y);
  };
  // step r: `cur` holds S of unit r, `nxt` takes that of unit r + 1.  MASK:
  // the units up to r + 4 may be partial, or not visible to every column.
  // (The two score tiles and the two staged units stay in their registers: the
  // steps come in pairs that name them the other way round.  Swapping them
  // instead made the masked steps spill, and wait for the loads in flight.)
  auto step = [&](int r, f32x16& cur, f32x16& nxt, St& st, auto act, auto mask_tag, bool sync)
      __attribute__((always_inline)) {
    constexpr bool ACT = decltype(act)::value;
    if constexpr (ACT) {
      // the column's maximum is needed only when some lane's scores pass the
      // raising threshold thr = (m + kLazy) / sc
      if (__builtin_amdgcn_ballot_w64(lm > thr)) {
        const float bm = pair_max(lm) * sc;
        const bool raise = bm > m + kLazy;
        const float mn = raise ? bm : m;
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        l *= alpha;
        m = mn;
        thr = (mn + kLazy) / sc;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
      }
    }
    stage(r + 3, st, mask_tag, std::false_type{});
    load(ua + r + 5, st);
    if constexpr (ACT) {
      nxt = scores(r + 1);
#pragma unroll
      for (int i = 0; i < 16; ++i) cur[i] = __builtin_amdgcn_exp2f(fmaf(cur[i], sc, -m));
      float ps = cur[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) ps += cur[i];
      l += ps;  // this lane's tokens; the column's halves are summed at the end
      const u32x4* vp = s_v[r & 7] + vl;
      u32x4 pf[2];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) pf[kk][jj] = cvt_pk<0>(cur[8 * kk + 2 * jj], cur[8 * kk + 2 * jj + 1]);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) o[dt] = mfma32x32x16<0>(vp[dt * 128 + kk * 32], pf[kk], o[dt]);
      lm = lane_max(nxt, r + 1, mask_tag);
    }
    if (sync) unit_barrier();
  };

  St st0, st1;
  f32x16 sa, sb2;
  load(ua, st0);
  load(ua + 1, st1);
  if constexpr (CV) {
    for (int i = threadIdx.x; i < ODDW; i += 64 * W) s_odd[i] = 0u;
    if (threadIdx.x == 0) s_anyodd = 0;
    unit_barrier();
  } else {
    if (lane == 0) s_odd[wave] = 0u;
  }
  stage(0, st0, std::true_type{}, std::false_type{});
  load(ua + 2, st0);
  stage(1, st1, std::true_type{}, std::false_type{});
  load(ua + 4, st1);
  stage(2, st0, std::true_type{}, std::false_type{});
  load(ua + 3, st0);
  unit_barrier();
  if (active) {
    sa = scores(0);
    lm = lane_max(sa, 0, std::true_type{});
  }
  unit_barrier();
  // every wave takes ub - ua steps (a barrier after every second one); a wave
  // past the last query token only loads and stages.  The steps whose units
  // (up to r + 4) are whole and visible to every column come first, in pairs.
  auto run = [&](auto act) __attribute__((always_inline)) {
    const int n = ub - ua, plain = nfull - ua - 4;  // pairs r, r + 1 with r + 4 < nfull - ua
    int r = 0;
#pragma unroll 1
    for (; r < plain; r += 2) {
      step(r, sa, sb2, st0, act, std::false_type{}, false);
      step(r + 1, sb2, sa, st1, act, std::false_type{}, true);
    }
#pragma unroll 1
    for (; r < n; r += 2) {
      step(r, sa, sb2, st0, act, std::true_type{}, false);
      if (r + 1 == n) break;
      step(r + 1, sb2, sa, st1, act, std::true_type{}, true);
    }
  };
  if (active) run(std::true_type{});
  else run(std::false_type{});
  // The noted units once more, for the elements left out.  Infinities and NaN
  // are added token by token, to the columns that see the token: a product
  // would bring 0 * inf to the others (and, with P as hi + lo, inf - inf).
  unit_barrier();
  uint32_t odd_word = 0u;  // (bits of units odd0 ..)
  if constexpr (CV) odd_word = s_anyodd;
  else
#pragma unroll
    for (int w = 0; w < W; ++w) odd_word |= s_odd[w];
  odd_word = (uint32_t)uniform((int)odd_word);
  if (odd_word != 0u) {
    auto next = [&](int x) __attribute__((always_inline)) {  // the first noted unit from x on, or ub
#pragma unroll 1
      for (; x < ub; ++x) {
        const int at = x - odd0;
        if ((CV ? (uint32_t)uniform((int)s_odd[at >> 5]) : odd_word) >> (at & 31) & 1u) break;
      }
      return x;
    };
    int x = next(odd0);
    pbase = min(x, ub - 1) >> ksh;
    pagev = bt[min(pbase + lane, lastblk)];
    load(x, st0);
#pragma unroll 1
    while (x < ub) {
      const int r = x - ua, at = x;
      // the unit's V as it is stored: a bf16 cache's own, or the 16-bit tile
      const uint8_t* vs = (const uint8_t*)s_v[r & 7];
      int tile16 = 1024;  // bytes from one 16-dim tile to the next
      [[maybe_unused]] u32x4 vf[CV ? 2 : 1][CV ? 4 : 1];
      if constexpr (CV) {
        const int page = __builtin_amdgcn_readlane(pagev, (x >> ksh) - pbase);
        vs = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes + geo.v_off + (x & ((1 << ksh) - 1)) * 1024;
        tile16 = 1024 << ksh;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int dt = 0; dt < 4; ++dt)
            vf[kk][dt] = *(const u32x4*)(vs + (2 * dt + (col >> 4)) * tile16 + ((col & 15) + 16 * (2 * kk + hh)) * 16);
      }
      unit_barrier();
      stage(r, st0, std::true_type{}, std::true_type{});
      x = next(x + 1);
      load(x, st0);
      unit_barrier();
      if (!active) continue;
      sa = scores(r);
      if (at >= nfull) lane_max(sa, r, std::true_type{});
#pragma unroll
      for (int i = 0; i < 16; ++i) sa[i] = __builtin_amdgcn_exp2f(fmaf(sa[i], sc, -m));
      if constexpr (CV) {
        const int valid = T - 32 * at;
        u16x2 top = {0, 0};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            u32x4& v = vf[kk][dt];
            v &= at_least16(v, ODD);
            if (valid < 32)  // (stale page data)
#pragma unroll
              for (int jj = 0; jj < 4; ++jj) {
                const int tk = 8 * (2 * kk + hh) + 2 * jj;
                v[jj] &= (tk < valid ? 0x0000FFFFu : 0u) | (tk + 1 < valid ? 0xFFFF0000u : 0u);
              }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t mag = v[k] & 0x7FFF7FFFu;
              top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, mag));
            }
          }
        const bool each =
            __builtin_amdgcn_ballot_w64(((__builtin_bit_cast(uint32_t, top) + 0x10001u * (0x8000u - INF)) & 0x80008000u) != 0u) != 0;
        if (each)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) vf[kk][dt] &= ~at_least16(vf[kk][dt], INF);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          u32x4 ph, pl;
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const float p0 = sa[8 * kk + 2 * jj], p1 = sa[8 * kk + 2 * jj + 1];
            const uint32_t w = cvt_pk<1>(p0, p1);
            ph[jj] = w;
            pl[jj] = cvt_pk<1>(p0 - __uint_as_float(w << 16), p1 - __uint_as_float(w & 0xFFFF0000u));
          }
#pragma unroll
          for (int dt = 0; dt < 4; ++dt) {
            o[dt] = mfma32x32x16<1>(vf[kk][dt], ph, o[dt]);
            o[dt] = mfma32x32x16<1>(vf[kk][dt], pl, o[dt]);
          }
        }
        if (!each) continue;
      }
      const int lim = pos - 32 * at;
#pragma unroll 1
      for (int t = 0; t < 32; ++t) {
        const int own = 8 * (t >> 4) + (t & 7);  // entry of token t in the lanes of half t / 8 % 2
        float p = sa[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) p = i == own ? sa[i] : p;
        p = __shfl(p, col + 32 * ((t >> 3) & 1), 64);
        const uint8_t* vt = vs + 256 * (t >> 3) + 2 * (t & 7) + 64 * hh;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const uint32_t w = *(const uint16_t*)(vt + (2 * dt + (i >> 3)) * tile16 + 128 * ((i >> 2) & 1) + 16 * (i & 3));
            if (t <= lim && (w & 0x7FFFu) >= INF) o[dt][i] = fmaf(p, to_f32<DT>((uint16_t)w), o[dt][i]);
          }
      }
    }
  }
  if (!active) return;
  // O^T: entry i of a lane is dim 32 dt + 8 (i / 4) + 4 hh + i % 4 of its column
  const float lt = pair_sum(l);
  if (tq >= L) return;
  if (nsplit == 1) {
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    uint16_t* dst = out + q_row(sb, bi, head) + (size_t)tq * kHeadDim + 4 * hh;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *(uint2*)(dst + 32 * dt + 8 * i) = make_uint2(pack2<DT>(o[dt][4 * i] * inv, o[dt][4 * i + 1] * inv),
                                                     pack2<DT>(o[dt][4 * i + 2] * inv, o[dt][4 * i + 3] * inv));
  } else {
    const size_t rows = (size_t)sb.n * geo.hq * L;
    const size_t row = part * rows + ((size_t)bi * geo.hq + head) * L + tq;
    float* dst = po + row * kHeadDim + 4 * hh;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *(f32x4*)(dst + 32 * dt + 8 * i) = f32x4{o[dt][4 * i], o[dt][4 * i + 1], o[dt][4 * i + 2], o[dt][4 * i + 3]};
    if (hh == 0) *(float2*)(pml + 2 * row) = make_float2(m, lt);
  }
}

// merges the parts of each output row: 32 threads a row, 4 dims each
template <int DT>
__global__ __launch_bounds__(256) void k_prefill_combine(int rows, int nsplit, const float* __restrict__ po,
                                                        const float* __restrict__ pml,
                                                        uint16_t* __restrict__ out) {
  const int row = blockIdx.x * 8 + (threadIdx.x >> 5), c = threadIdx.x & 31;
  if (row >= rows) return;
  float M = kNoMax;
  for (int p = 0; p < nsplit; ++p) M = fmaxf(M, pml[2 * ((size_t)p * rows + row)]);
  float l = 0.f;
  f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int p = 0; p < nsplit; ++p) {
    const size_t at = (size_t)p * rows + row;
    const float2 ml = *(const float2*)(pml + 2 * at);
    const f32x4 x = *(const f32x4*)(po + at * kHeadDim + 4 * c);
    const float w = __builtin_amdgcn_exp2f(ml.x - M);
    l += w * ml.y;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] += w * x[i];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  *(uint2*)(out + (size_t)row * kHeadDim + 4 * c) =
      make_uint2(pack2<DT>(a[0] * inv, a[1] * inv), pack2<DT>(a[2] * inv, a[3] * inv));
}

// tiles of whole workgroups (kPfWaves waves)
static int64_t prefill_tiles(const Geometry& g, int n, int L) {
  return (int64_t)((L * g.group + kPfWaves * kPfCols - 1) / (kPfWaves * kPfCols)) * g.hkv * n;
}

// Parts for n sequences of at most `tokens` tokens: the number with the least
// rounds of workgroups (one per CU at a time) times the units a round takes,
// where a split adds the merge.  A chunk whose tiles fill the CUs once or a
// whole number of times is not split (8 sequences of 512 tokens: 512 tiles);
// one sequence's 64 tiles are split in 4 (1109 us with one workgroup of 128
// columns a tile, unsplit; 294 us).
int prefill_splits(const Geometry& g, int n, int L, int tokens) {
  if (g.cus <= 0) return 1;
  const int64_t tiles = prefill_tiles(g, n, L);
  const int64_t rows = (int64_t)n * g.hq * L;
  const int units = (tokens + 31) / 32;
  int best = 1;
  double cost = 0.0;
  for (int s = 1; s <= kPfSplits; ++s) {
    if (s > 1 && (rows * s > kPrefillRows || units < 8 * s)) break;
    // rounds of workgroups, each the units of its part and about 4 more for its start and end
    const double c = (double)((tiles * s + g.cus - 1) / g.cus) * ((double)units / s + 4.0) +
                     (s > 1 ? 8.0 + (double)rows * s * 4e-4 : 0.0);
    if (s == 1 || c < 0.97 * cost) {
      best = s;
      cost = c;
    }
  }
  return best;
}

template <int DT, int KB, int W>
static hipError_t prefill_dispatch(const Geometry& g, const SeqBatch& b, int L, int nsplit, const uint16_t* q, float sl2,
                                   uint16_t* out, float* ws, hipEvent_t done, hipStream_t s, Timing* prof) {
  const int lg = __builtin_ctz((unsigned)g.group);
  const int per_wg = (W * kPfCols) >> lg;
  const int gx = (L + per_wg - 1) / per_wg;
  const int rows = b.n * g.hq * L;
  float* pml = ws ? ws + (size_t)nsplit * rows * kHeadDim : nullptr;
  launch(k_prefill<DT, KB, W>, dim3((unsigned)gx * g.hkv * b.n * nsplit), dim3(64 * W), 0, s, prof, kProfPrefill, g,
         b, L, lg, gx, nsplit, q, sl2, out, ws, pml);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || nsplit == 1) return e;
  const dim3 grid((rows + 7) / 8), blk(256);
  const float *po = ws, *ml = pml;
  if (done && !prof)  // (the event is the dispatch's own: no packet of its own behind it)
    hipExtLaunchKernelGGL(k_prefill_combine<DT>, grid, blk, 0u, s, nullptr, done, 0u, rows, nsplit, po, ml, out);
  else
    launch(k_prefill_combine<DT>, grid, blk, 0, s, prof, kProfCombine, rows, nsplit, po, ml, out);
  e = hipGetLastError();
  if (e == hipSuccess && done && prof) e = hipEventRecord(done, s);
  return e;
}

// Workgroups of 4 waves (half a tile) where those of all tiles and parts still
// fit the CUs at once: a wave then has a SIMD to itself, and a unit takes it
// little more than half as long.  One fp16 prompt of 200 tokens, Hq 32, Hkv 8:
// 17.0 us with 8 waves (32 workgroups), 12.7 with 4 (56); of 600 26.1 and
// 20.5, of 1000 (256 workgroups of 4) 35.3 and 28.9.  With more, the second
// round costs more than that: 1500 tokens take 47 us with 8 waves.
template <int DT, int KB>
static hipError_t prefill_width(const Geometry& g, const SeqBatch& b, int L, int nsplit, const uint16_t* q, float sl2,
                                uint16_t* out, float* ws, hipEvent_t done, hipStream_t s, Timing* prof) {
  if (2 * prefill_tiles(g, b.n, L) * nsplit <= g.cus)
    return prefill_dispatch<DT, KB, kPfWaves / 2>(g, b, L, nsplit, q, sl2, out, ws, done, s, prof);
  return prefill_dispatch<DT, KB, kPfWaves>(g, b, L, nsplit, q, sl2, out, ws, done, s, prof);
}

hipError_t launch_prefill(const Geometry& g, const SeqBatch& b, int L, int nsplit, const void* q, float scale,
                          void* out, float* ws, hipEvent_t done, hipStream_t s, Timing* prof) {
  const float sl2 = scale * 1.4426950408889634f;
  const uint16_t* qq = (const uint16_t*)q;
  uint16_t* oo = (uint16_t*)out;
  if (g.kv_bits == 4) return prefill_width<0, 4>(g, b, L, nsplit, qq, sl2, oo, ws, done, s, prof);
  if (g.kv_bits == 8) return prefill_width<0, 8>(g, b, L, nsplit, qq, sl2, oo, ws, done, s, prof);
  if (g.dtype == 0) return prefill_width<0, 0>(g, b, L, nsplit, qq, sl2, oo, ws, done, s, prof);
  return prefill_width<1, 0>(g, b, L, nsplit, qq, sl2, oo, ws, done, s, prof);
}

}  // namespace bsattn
