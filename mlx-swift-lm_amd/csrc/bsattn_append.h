// bsattn_append.h -- device code of the appends shared by the append kernels
// and the kernels that append as part of another launch: one token into a
// 16-bit or affine-quantized slab, with the summary of the block it fills.
#pragma once

#include "bsattn_device.h"

namespace bsattn {

__device__ __forceinline__ float h2f(uint32_t bits16) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}
__device__ __forceinline__ float lo_f(uint32_t w) { return h2f(w & 0xFFFFu); }
__device__ __forceinline__ float hi_f(uint32_t w) { return h2f(w >> 16); }

// One token of entry bi (row bi of k / v [n][Hkv][D]) into a 16-bit slab by a
// 256-thread workgroup, lanes 0..15 with 8 dims each.  A token that fills its
// block also writes the block's summary: the keys of the block's other tokens
// (written by earlier launches) are requested first, all at once and without
// a branch (token indices clamped; at most four keys per thread), pass
// through LDS with the new key from the registers of the lanes that store it,
// and 16 lanes fold them in token order.
template <int DT>
__device__ __forceinline__ void append_token(const Geometry& geo, int seq, int bi, int h, int pos, int page,
                                             const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                             u32x4 (*s_blk)[16]) {
  const int tg = threadIdx.x >> 4, c = threadIdx.x & 15;
  const int blk = pos / geo.tb, slot = pos - blk * geo.tb;
  const bool fills = slot == geo.tb - 1;
  u32x4 pre[4];
  if (fills) {
    const uint16_t* Kt =
        (const uint16_t*)(geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes + geo.k_off);
#pragma unroll
    for (int i = 0; i < 4; ++i) pre[i] = *(const u32x4*)(Kt + k_elem(min(tg + 16 * i, geo.tb - 2), 8 * c));
  }
  u32x4 kr = u32x4{0u, 0u, 0u, 0u};
  if (tg == 0) {
    const size_t src = ((size_t)bi * geo.hkv + h) * kHeadDim + 8 * c;
    kr = *(const u32x4*)(k + src);
    const u32x4 vr = *(const u32x4*)(v + src);
    put_token(geo, page, h, slot, c, kr, vr);
  }
  if (!fills) return;
  // keys 0 .. Tb-2 (loaded above); key Tb-1 is kr of tg 0
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (tg + 16 * i < geo.tb - 1) s_blk[tg + 16 * i][c] = pre[i];
  if (tg == 0) s_blk[geo.tb - 1][c] = kr;
  __syncthreads();
  if (tg != 0) return;
  *(u32x4*)(summary_row(geo, seq, h, blk) + 8 * c) = fold_block<DT>(s_blk, geo.tb, c);
}

// ---------------------------------------------------------------------------
// quantize 8 consecutive dims of one row (lane c of the 16 lanes holding the
// row; lanes c & ~7 .. +7 hold one 64-dim group) by mlx's affine rule, in
// fp32 with correctly rounded divisions:
//   scale = max((max - min) / (2^b - 1), 1e-7), negated unless
//   |min| > |max|; edge = min if |min| > |max| else max;
//   q0 = rint(edge / scale); q0 != 0: scale = edge / q0, bias = edge;
//   q0 == 0 (an all-zero group): bias = 0;
//   code = clamp(rint((x - bias) / scale), 0, 2^b - 1) from the fp32 scale
//   and bias, which are stored rounded to fp16.
// (Signed zeros cannot matter: q0 == 0 only when edge is a zero, and then
// bias is +0.)
// ---------------------------------------------------------------------------
template <int KB>
__device__ __forceinline__ void quantize8(const u32x4 raw, uint32_t (&codes)[8], uint16_t& scale_out,
                                          uint16_t& bias_out) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (e & 1) ? hi_f(raw[e >> 1]) : lo_f(raw[e >> 1]);
  float mn = x[0], mx = x[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) {
    mn = fminf(mn, x[e]);
    mx = fmaxf(mx, x[e]);
  }
#pragma unroll
  for (int off = 1; off < 8; off <<= 1) {
    mn = fminf(mn, __shfl_xor(mn, off, 64));
    mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  }
  constexpr float nbins = (float)((1 << KB) - 1);
  float scale = fmaxf(__fdiv_rn(__fsub_rn(mx, mn), nbins), (float)1e-7);
  const bool side = fabsf(mn) > fabsf(mx);
  scale = side ? scale : -scale;
  const float edge = side ? mn : mx;
  const float q0 = __builtin_rintf(__fdiv_rn(edge, scale));
  float bias = 0.0f;
  if (q0 != 0.0f) {
    scale = __fdiv_rn(edge, q0);
    bias = edge;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float qv = __builtin_rintf(__fdiv_rn(__fsub_rn(x[e], bias), scale));
    qv = qv < 0.0f ? 0.0f : qv;
    qv = qv > nbins ? nbins : qv;
    codes[e] = (uint8_t)qv;
  }
  scale_out = __builtin_bit_cast(uint16_t, (_Float16)scale);
  bias_out = __builtin_bit_cast(uint16_t, (_Float16)bias);
}

// dim d of a quantized block's summary, from its K codes Kc and scales /
// biases Sb (slab layout): sequential fp32 fold of the dequantized keys
// fmaf(scale, code, bias) from token 0, times 1/tb, to fp16
template <int KB>
__device__ __forceinline__ uint16_t fold_block_q(const uint8_t* Kc, const uint16_t* Sb, int tb, int d) {
  const int grp = d >> 6;
  float acc = 0.0f;
#pragma unroll 8
  for (int t = 0; t < tb; ++t) {
    int sh;
    const int code = (Kc[kq_byte(KB, t, d, &sh)] >> sh) & ((1 << KB) - 1);
    const uint16_t* f = Sb + 8 * sb_entry(tb, t);
    const float w = __builtin_fmaf(h2f(f[grp]), (float)code, h2f(f[2 + grp]));
    acc = (t == 0) ? w : __fadd_rn(acc, w);
  }
  return __builtin_bit_cast(uint16_t, (_Float16)__fmul_rn(acc, 1.0f / (float)tb));
}

// LDS of a one-token append workgroup (256 threads): the keys of the block
// it fills ([token][8-dim chunk]; quantized: its code tile, at most 8 KiB,
// then its scales / biases)
struct AppendLds {
  u32x4 blk[64][16];
};

// ---------------------------------------------------------------------------
// One token into a quantized slab by a 256-thread workgroup: wave 0 quantizes
// it (lanes 0..15 the key, 16..31 the value, 8 dims each) and stores it; a
// V code shares its byte (int4) or word with its neighbours' tokens, so its
// old byte is read with the token.  When the token fills its block, the
// block's other codes and scales are requested first of all, pass through LDS
// with the token's own, and 128 threads fold them into the block's summary.
// A launch of its own per step for this (behind one for the metadata, and
// before one for the summary) cost two kernel boundaries and more: it is run
// by workgroups of the scoring launch, which reads nothing that it writes.
// ---------------------------------------------------------------------------
template <int KB>
__device__ __forceinline__ void append_token_q(const Geometry& geo, int seq, int bi, int h, int pos, int page,
                                               const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                               AppendLds& lds) {
  constexpr int NPRE = KB / 4;  // 16-byte pieces of a 64-token code tile per thread
  const int tid = threadIdx.x, c = tid & 15;
  const bool val = (tid & 16) != 0;
  const int blk = pos / geo.tb, slot = pos - blk * geo.tb;
  uint8_t* slab = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes;
  uint8_t* Kc = slab + geo.k_off;
  uint8_t* Vc = slab + geo.v_off;
  u32x4* Sb = (u32x4*)(slab + geo.sb_off);
  const bool fills = slot == geo.tb - 1;
  const int pieces = geo.tb * KB;  // of this cache's code tile
  u32x4 pre[NPRE], psb = u32x4{0u, 0u, 0u, 0u};
  if (fills) {
#pragma unroll
    for (int i = 0; i < NPRE; ++i) pre[i] = ((const u32x4*)Kc)[min(tid + 256 * i, pieces - 1)];
    psb = Sb[min(tid, geo.tb - 1)];
  }
  uint32_t codes[8];
  uint16_t sc = 0, bs = 0;
  u32x4 entry = u32x4{0u, 0u, 0u, 0u};
  if (tid < 64) {  // wave 0, whole (lanes 32.. repeat lanes 0..31 and store nothing)
    const size_t src = ((size_t)bi * geo.hkv + h) * kHeadDim + 8 * c;
    const u32x4 raw = *(const u32x4*)((val ? v : k) + src);
    uint8_t old[8];
    if constexpr (KB == 4) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        int sh;
        old[e] = Vc[vq_byte(KB, geo.tb, slot, 8 * c + e, &sh)];
      }
    }
    quantize8<KB>(raw, codes, sc, bs);
    const uint32_t sbw = (uint32_t)sc | ((uint32_t)bs << 16);
    // groups 0 and 1 of the key sit in lanes 0 and 8, of the value in 16 and 24
    const uint32_t k0 = (uint32_t)__builtin_amdgcn_readlane((int)sbw, 0);
    const uint32_t k1 = (uint32_t)__builtin_amdgcn_readlane((int)sbw, 8);
    const uint32_t v0 = (uint32_t)__builtin_amdgcn_readlane((int)sbw, 16);
    const uint32_t v1 = (uint32_t)__builtin_amdgcn_readlane((int)sbw, 24);
    entry = u32x4{(k0 & 0xFFFFu) | (k1 << 16), (k0 >> 16) | (k1 & 0xFFFF0000u), (v0 & 0xFFFFu) | (v1 << 16),
                  (v0 >> 16) | (v1 & 0xFFFF0000u)};
    if (tid < 32 && val) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        int sh;
        uint8_t* dst = Vc + vq_byte(KB, geo.tb, slot, 8 * c + e, &sh);
        if constexpr (KB == 4) *dst = (uint8_t)((old[e] & (0xF0u >> sh)) | (codes[e] << sh));
        else *dst = (uint8_t)codes[e];
      }
    }
    if (tid == 0) Sb[sb_entry(geo.tb, slot)] = entry;
  }
  // the key's codes of lane c: one word (int4) or two (int8) of the tile
  uint32_t w0 = 0u, w1 = 0u;
  int sh;
  const int kat = kq_byte(KB, slot, 8 * c, &sh);
  if (tid < 16) {
    if constexpr (KB == 4) {
#pragma unroll
      for (int e = 0; e < 8; ++e) w0 |= codes[e] << (4 * q_nib(e));
      *(uint32_t*)(Kc + kat) = w0;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w0 |= codes[e] << (8 * e);
        w1 |= codes[4 + e] << (8 * e);
      }
      *(uint2*)(Kc + kat) = make_uint2(w0, w1);
    }
  }
  if (!fills) return;
  uint8_t* lc = (uint8_t*)lds.blk;
  u32x4* ls = (u32x4*)(lc + 64 * kHeadDim * KB / 8);
#pragma unroll
  for (int i = 0; i < NPRE; ++i)
    if (tid + 256 * i < pieces) ((u32x4*)lc)[tid + 256 * i] = pre[i];
  if (tid < geo.tb) ls[tid] = psb;
  __syncthreads();
  if (tid < 16) {
    *(uint32_t*)(lc + kat) = w0;
    if constexpr (KB == 8) *(uint32_t*)(lc + kat + 4) = w1;
    if (tid == 0) ls[sb_entry(geo.tb, slot)] = entry;
  }
  __syncthreads();
  if (tid < kHeadDim)
    summary_row(geo, seq, h, blk)[tid] = fold_block_q<KB>(lc, (const uint16_t*)ls, geo.tb, tid);
}

// The append part of a decode step's scoring launch: entry bi's token to kv
// head h by one 256-thread workgroup, and the step's metadata patches by the
// workgroup of (0, 0), for the launches that follow.  Nothing in the same
// launch reads what it writes: the append takes its position and page from
// the arguments, the scoring its lengths from sb, and the block that a token
// completes is the newest block, which is forced (recent >= 1), never scored.
template <int DT>
__device__ __forceinline__ void append_step_body(const Geometry& geo, const SeqBatch& sb, const StepAppend& ap,
                                                 int h, int bi, AppendLds& lds) {
  if (h == 0 && bi == 0 && (int)threadIdx.x < ap.pb.n) geo.meta[ap.pb.idx[threadIdx.x]] = ap.pb.val[threadIdx.x];
  const int seq = sb.ids[bi], pos = sb.len[bi] - 1, page = ap.sp.page[bi];
  if constexpr (DT == 0) {
    if (geo.kv_bits == 4) {
      append_token_q<4>(geo, seq, bi, h, pos, page, ap.k, ap.v, lds);
      return;
    }
    if (geo.kv_bits == 8) {
      append_token_q<8>(geo, seq, bi, h, pos, page, ap.k, ap.v, lds);
      return;
    }
  }
  append_token<DT>(geo, seq, bi, h, pos, page, ap.k, ap.v, lds.blk);
}

}  // namespace bsattn
