// bsattn_blocks.hip -- appends and exports of many tokens, by whole blocks.
//
// A workgroup moves one (block, kv head) slab between the token-major arrays
// of the API ([n][Hkv][tokens][D]) and the fragment-major tiles of the cache:
// one wave per 32-token segment and tile (TB / 32 waves for V, as many for
// K), every load of a wave issued before its first wait.  A K fragment is
// 16-byte pieces of token rows, so K moves with no exchange: the lane that
// owns a piece of the fragment loads it from its row (64 bytes of 16 rows
// per instruction).  V is transposed: thread (g, c) holds 8 tokens x 8 dims,
// exchanges them in registers (one v_perm per word) and reaches the
// fragments' lane order through LDS, so that pool and arrays are both read
// and written in runs of at least 64 bytes.
//
// Bound by HBM.  Export and reload of 32k tokens x 8 kv heads of bf16 K and V
// (134 MB read and written by each): 187 -> 123 us, 4.4 TB/s, where one lane
// per 16-byte piece stored or loaded the 8 elements of V one by one (77-79 us
// each way) and a launch after it read the keys again for the summaries
// (17 us).  A prompt of 8191 fp16 tokens, appended and attended: 607 -> 583 us.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "bsattn_append.h"
#include "bsattn_device.h"

namespace bsattn {

// 8 x 8 transpose of 16-bit elements: word i of out[e] is element e of rows
// 2 i and 2 i + 1
__device__ __forceinline__ void transpose8x8(const u32x4 (&row)[8], u32x4 (&out)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[e][i] = __builtin_amdgcn_perm(row[2 * i + 1][e >> 1], row[2 * i][e >> 1], (e & 1) ? 0x07060302u : 0x05040100u);
}

// Place of the 16-byte piece (dim tile dt, lane 16 g + n) of a V segment in
// its LDS exchange buffer: the low lane bits are rotated by dt, so that
// neither side of the exchange meets more bank conflicts than its bytes do.
__device__ __forceinline__ int v_place(int dt, int lane) { return dt * 64 + (lane ^ dt); }

// token of its 32-token segment that K fragment (tile parity tl) of lane row m holds
__device__ __forceinline__ int k_seg_tok(int tl, int m) { return 8 * (m >> 2) + 4 * tl + (m & 3); }

// physical page of the x-th block that entry bi's append touches
__device__ __forceinline__ int append_page(const Geometry& geo, const AppendPages& pg, int seq, int bi, int x, int blk) {
  return pg.given ? pg.page[pg.off[bi] + x] : block_table(geo, seq)[blk];
}

// ---------------------------------------------------------------------------
// append of L tokens per sequence to a 16-bit cache, with the summaries of
// the blocks it fills: the block's keys pass through LDS (those of tokens
// appended earlier come from the tile) and 64 lanes fold two dims each in
// token order.  A V piece of 8 tokens that is only partly new is merged with
// the tile's.  When the host has passed the touched blocks' pages, workgroup
// (0, 0, 0) applies the metadata patches for the launches that follow (nothing
// here reads the metadata then).  grid (blocks touched, Hkv, n)
// ---------------------------------------------------------------------------
template <int DT, int TB>
__global__ __launch_bounds__(4 * TB) void k_append_blocks(Geometry geo, AppendBatch ab, AppendPages pg,
                                                          PatchBatch pb, const uint16_t* __restrict__ k,
                                                          const uint16_t* __restrict__ v) {
  constexpr int SEG = TB / 32;  // 32-token segments of a block
  __shared__ u32x4 s_v[SEG][512];
  __shared__ u32x4 s_k[TB][17];  // a padded row per token
  const int x = blockIdx.x, h = blockIdx.y, bi = blockIdx.z;
  if (x == 0 && h == 0 && bi == 0)
    for (int i = threadIdx.x; i < pb.n; i += 4 * TB) geo.meta[pb.idx[i]] = pb.val[i];
  const int old = ab.old_len[bi], end = old + ab.L;
  const int blk = old / TB + x;
  if (blk * TB >= end) return;
  const int seq = ab.seq[bi];
  const int page = append_page(geo, pg, seq, bi, x, blk);
  const bool fills = (blk + 1) * TB <= end;
  uint8_t* slab = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes;
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int seg = wave % SEG;
  const int seg0 = blk * TB + 32 * seg;  // the segment's first position
  const int64_t row0 = ((int64_t)bi * geo.hkv + h) * ab.L - old;  // row of position p: row0 + p
  if (wave < SEG) {
    if (seg0 < end && seg0 + 32 > old) {
      const int g = lane >> 4, c = lane & 15;
      const int p0 = seg0 + 8 * g;
      u32x4 row[8], out[8];
  #pragma unroll
      for (int i = 0; i < 8; ++i)  // positions that are not appended read a neighbour's row
        row[i] = *(const u32x4*)(v + (row0 + min(max(p0 + i, old), end - 1)) * kHeadDim + 8 * c);
      transpose8x8(row, out);
  #pragma unroll
      for (int e = 0; e < 8; ++e) s_v[seg][v_place(c >> 1, 16 * g + 8 * (c & 1) + e)] = out[e];
      wave_lds_order();
      u32x4* Vf = (u32x4*)(slab + geo.v_off) + seg * 64 + lane;
      if (seg0 >= old && seg0 + 32 <= end) {
  #pragma unroll
        for (int dt = 0; dt < 8; ++dt) Vf[dt * SEG * 64] = s_v[seg][v_place(dt, lane)];
      } else if (p0 < end && p0 + 8 > old) {
        u32x4 m;  // halfwords of the appended tokens
  #pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = p0 + 2 * i;
          m[i] = (p >= old && p < end ? 0x0000FFFFu : 0u) | (p + 1 >= old && p + 1 < end ? 0xFFFF0000u : 0u);
        }
  #pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          const u32x4 w = s_v[seg][v_place(dt, lane)], was = Vf[dt * SEG * 64];
          Vf[dt * SEG * 64] = (w & m) | (was & ~m);
        }
      }
    }
  } else {
    const int m = lane & 15, g = lane >> 4;
    u32x4* Kf = (u32x4*)(slab + geo.k_off) + seg * 8 * 64 + lane;
    u32x4 kr[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      const int p = seg0 + k_seg_tok(f >> 2, m);
      const u32x4* src = p >= old && p < end ? (const u32x4*)(k + (row0 + p) * kHeadDim + 32 * (f & 3) + 8 * g)
                                             : Kf + f * 64;
      kr[f] = *src;
    }
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      const int t = k_seg_tok(f >> 2, m), p = seg0 + t;
      if (p >= old && p < end) Kf[f * 64] = kr[f];
      if (fills) s_k[32 * seg + t][4 * (f & 3) + g] = kr[f];
    }
  }
  if (!fills) return;
  __syncthreads();
  if (threadIdx.x < 64) {
    // dims 2 t and 2 t + 1: sequential fp32 fold from token 0, times 1/Tb, in
    // the cache's type (the order of fold_block)
    auto dims = [&](int t) { return ((const uint32_t*)s_k[t])[threadIdx.x]; };
    uint32_t w = dims(0);
    float a = to_f32<DT>((uint16_t)w), b = to_f32<DT>((uint16_t)(w >> 16));
#pragma unroll 16
    for (int t = 1; t < TB; ++t) {
      w = dims(t);
      a = __fadd_rn(a, to_f32<DT>((uint16_t)w));
      b = __fadd_rn(b, to_f32<DT>((uint16_t)(w >> 16)));
    }
    constexpr float inv = 1.0f / (float)TB;
    ((uint32_t*)summary_row(geo, seq, h, blk))[threadIdx.x] = pack2<DT>(__fmul_rn(a, inv), __fmul_rn(b, inv));
  }
}

// ---------------------------------------------------------------------------
// export: pages -> [n, Hkv, T, D], the same exchange backwards.
// grid (ceil(T / TB), Hkv, n)
// ---------------------------------------------------------------------------
template <int TB>
__global__ __launch_bounds__(4 * TB) void k_export_blocks(Geometry geo, SeqBatch sb, int T, uint16_t* __restrict__ ko,
                                                          uint16_t* __restrict__ vo) {
  constexpr int SEG = TB / 32;
  __shared__ u32x4 s_v[SEG][512];
  const int blk = blockIdx.x, h = blockIdx.y, bi = blockIdx.z;
  const int page = block_table(geo, sb.ids[bi])[blk];
  const uint8_t* slab = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes;
  const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int seg = wave % SEG;
  const int seg0 = blk * TB + 32 * seg;
  const size_t row0 = ((size_t)bi * geo.hkv + h) * T + seg0;
  if (seg0 >= T) return;
  if (wave < SEG) {
    const u32x4* Vf = (const u32x4*)(slab + geo.v_off) + seg * 64 + lane;
    u32x4 vr[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) vr[dt] = Vf[dt * SEG * 64];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) s_v[seg][v_place(dt, lane)] = vr[dt];
    wave_lds_order();
    const int g = lane >> 4, c = lane & 15;
    u32x4 in[8], row[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) in[e] = s_v[seg][v_place(c >> 1, 16 * g + 8 * (c & 1) + e)];
    transpose8x8(in, row);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (seg0 + 8 * g + i < T) *(u32x4*)(vo + (row0 + 8 * g + i) * kHeadDim + 8 * c) = row[i];
  } else {
    const int m = lane & 15, g = lane >> 4;
    const u32x4* Kf = (const u32x4*)(slab + geo.k_off) + seg * 8 * 64 + lane;
    u32x4 kr[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) kr[f] = Kf[f * 64];
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      const int t = k_seg_tok(f >> 2, m);
      if (seg0 + t < T) *(u32x4*)(ko + (row0 + t) * kHeadDim + 32 * (f & 3) + 8 * g) = kr[f];
    }
  }
}

// ---------------------------------------------------------------------------
// quantized caches.  A token's codes travel as its row's MLX words (element i
// in bits b * i up): thread (g, c) holds the KB / 4 words of dims 8c .. 8c+7
// of the 8 tokens 8 g .. of its segment.
// ---------------------------------------------------------------------------
// 4 x 4 transpose of bytes: byte j of out[i] is byte i of r_j
__device__ __forceinline__ void transpose4x4(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t (&out)[4]) {
  const uint32_t a = __builtin_amdgcn_perm(r1, r0, 0x05010400u), b = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
  const uint32_t c = __builtin_amdgcn_perm(r3, r2, 0x05010400u), d = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
  out[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
  out[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
  out[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
  out[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// 8 x 8 transpose of nibbles: nibble p of out[d] is nibble d of in[p]
__device__ __forceinline__ void transpose_nibbles(const uint32_t (&in)[8], uint32_t (&out)[8]) {
  constexpr uint32_t M = 0x0F0F0F0Fu;
  uint32_t lo[4], hi[4], t[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    lo[j] = (in[2 * j] & M) | ((in[2 * j + 1] & M) << 4);
    hi[j] = ((in[2 * j] >> 4) & M) | (in[2 * j + 1] & ~M);
  }
  transpose4x4(lo[0], lo[1], lo[2], lo[3], t);
#pragma unroll
  for (int b = 0; b < 4; ++b) out[2 * b] = t[b];
  transpose4x4(hi[0], hi[1], hi[2], hi[3], t);
#pragma unroll
  for (int b = 0; b < 4; ++b) out[2 * b + 1] = t[b];
}

// the element of an int4 word in nibble p (the inverse of q_nib)
__host__ __device__ constexpr int nib_elem(int p) { return p < 4 ? 2 * p : 2 * p - 7; }

// MLX int4 word (element e in nibble e) <-> tile word (element e in nibble q_nib(e))
__device__ __forceinline__ uint32_t to_tile_word(uint32_t w) {
  auto even = [](uint32_t x) {  // nibbles 0, 2, 4, 6 into the low 16 bits
    x &= 0x0F0F0F0Fu;
    x = (x | (x >> 4)) & 0x00FF00FFu;
    return (x | (x >> 8)) & 0xFFFFu;
  };
  return even(w) | (even(w >> 4) << 16);
}
__device__ __forceinline__ uint32_t from_tile_word(uint32_t w) {
  auto spread = [](uint32_t x) {
    x = (x | (x << 8)) & 0x00FF00FFu;
    return (x | (x << 4)) & 0x0F0F0F0Fu;
  };
  return spread(w & 0xFFFFu) | (spread(w >> 16) << 4);
}

// tokens' words w -> for each dim e the codes of its 8 tokens as the V tile
// stores them, and back (the exchange is its own inverse)
template <int KB>
__device__ __forceinline__ void transpose_codes(const uint32_t (&w)[8][KB / 4], uint32_t (&out)[8][KB / 4],
                                                bool to_tile) {
  if constexpr (KB == 4) {
    uint32_t in[8], o[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) in[p] = w[to_tile ? nib_elem(p) : p][0];
    transpose_nibbles(in, o);
#pragma unroll
    for (int p = 0; p < 8; ++p) out[to_tile ? p : nib_elem(p)][0] = o[p];
  } else {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        uint32_t t[4];
        transpose4x4(w[4 * q][half], w[4 * q + 1][half], w[4 * q + 2][half], w[4 * q + 3][half], t);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[4 * half + i][q] = t[i];
      }
  }
}

// Place of V fragment f's 16-byte piece of lane `lane` in a segment's LDS
// exchange buffer (low lane bits rotated as in v_place), and the fragment,
// lane and word of thread (g, c)'s dim 8 c + e in it.
template <int KB>
__device__ __forceinline__ int vq_place(int f, int lane) {
  return f * 64 + (lane ^ (KB == 8 ? f + 4 * ((lane >> 4) & 1) : (lane >> 4) + 4 * f));
}
template <int KB>
__device__ __forceinline__ uint32_t* vq_words(u32x4* buf, int g, int c, int e) {
  constexpr int DPF = QCode<KB>::DPF;  // 16-dim tiles per fragment
  const int dt = c >> 1;
  return (uint32_t*)(buf + vq_place<KB>(dt / DPF, 16 * g + 8 * (c & 1) + e)) + (dt % DPF) * (KB / 4);
}

// the arrays of a quantized append or export, 16-bit or in the MLX layout
struct QuantSrc {
  const uint16_t *k16, *v16;
  const uint32_t *kw, *vw;
  const uint16_t *ks, *kb, *vs, *vb;
};
struct QuantDst {
  uint32_t *kw, *vw;
  uint16_t *ks, *kb, *vs, *vb;
};

// ---------------------------------------------------------------------------
// append of L tokens per sequence to a quantized cache (16-bit tokens
// quantized here, or codes), with the summaries of the blocks it fills.  K
// codes are brought into the tile's order in LDS, which is also what the
// summary's fold reads.  grid (blocks touched, Hkv, n)
// ---------------------------------------------------------------------------
template <int KB, int TB, bool QUANTIZE>
__global__ __launch_bounds__(4 * TB) void k_append_blocks_q(Geometry geo, AppendBatch ab, AppendPages pg,
                                                            PatchBatch pb, QuantSrc src) {
  constexpr int SEG = TB / 32, W = KB / 4, WPR = QCode<KB>::WPR;
  constexpr int NVF = KB / 2;      // V fragments of a segment
  constexpr int KF = KB / 4;       // K fragments of a 16-token tile
  __shared__ u32x4 s_v[SEG][NVF * 64];
  __shared__ u32x4 s_k[TB * KB];   // the K code tile
  __shared__ u32x4 s_sb[TB];       // scales / biases, by sb_entry
  const int x = blockIdx.x, h = blockIdx.y, bi = blockIdx.z;
  if (x == 0 && h == 0 && bi == 0)
    for (int i = threadIdx.x; i < pb.n; i += 4 * TB) geo.meta[pb.idx[i]] = pb.val[i];
  const int old = ab.old_len[bi], end = old + ab.L;
  const int blk = old / TB + x;
  if (blk * TB >= end) return;
  const int seq = ab.seq[bi];
  const int page = append_page(geo, pg, seq, bi, x, blk);
  const bool fills = (blk + 1) * TB <= end;
  uint8_t* slab = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes;
  u32x4* Sb = (u32x4*)(slab + geo.sb_off);
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63;
  const int seg = wave % SEG;
  const bool is_v = wave < SEG;
  const int seg0 = blk * TB + 32 * seg;
  const int64_t row0 = ((int64_t)bi * geo.hkv + h) * ab.L - old;  // row of position p: row0 + p
  auto appended = [&](int p) { return p >= old && p < end; };
  if (seg0 < end && seg0 + 32 > old) {
    const int g = lane >> 4, c = lane & 15;
    const int p0 = seg0 + 8 * g;
    uint32_t w[8][W];
    if constexpr (QUANTIZE) {
      u32x4 raw[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)  // positions that are not appended read a neighbour's row
        raw[i] = *(const u32x4*)((is_v ? src.v16 : src.k16) + (row0 + min(max(p0 + i, old), end - 1)) * kHeadDim + 8 * c);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint32_t codes[8];
        uint16_t sc, bs;
        quantize8<KB>(raw[i], codes, sc, bs);
#pragma unroll
        for (int j = 0; j < W; ++j) w[i][j] = 0u;
#pragma unroll
        for (int e = 0; e < 8; ++e) w[i][e * KB / 32] |= codes[e] << (e * KB % 32);
        if ((c & 7) == 0 && appended(p0 + i)) {
          uint16_t* f = (uint16_t*)(s_sb + sb_entry(TB, 32 * seg + 8 * g + i)) + (is_v ? 4 : 0) + (c >> 3);
          f[0] = sc;
          f[2] = bs;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t* r = (is_v ? src.vw : src.kw) + (row0 + min(max(p0 + i, old), end - 1)) * WPR + W * c;
#pragma unroll
        for (int j = 0; j < W; ++j) w[i][j] = r[j];
      }
    }
    if (is_v) {
      uint32_t o[8][W];
      transpose_codes<KB>(w, o, true);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint32_t* d = vq_words<KB>(s_v[seg], g, c, e);
#pragma unroll
        for (int j = 0; j < W; ++j) d[j] = o[e][j];
      }
      wave_lds_order();
      u32x4* Vf = (u32x4*)(slab + geo.v_off) + seg * 64 + lane;
      if (seg0 >= old && seg0 + 32 <= end) {
#pragma unroll
        for (int f = 0; f < NVF; ++f) Vf[f * SEG * 64] = s_v[seg][vq_place<KB>(f, lane)];
      } else if (p0 < end && p0 + 8 > old) {
        u32x4 m;  // codes of the appended tokens
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          m[q] = 0u;
          if constexpr (KB == 4) {
#pragma unroll
            for (int e = 0; e < 8; ++e) m[q] |= appended(p0 + e) ? 0xFu << (4 * q_nib(e)) : 0u;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) m[q] |= appended(p0 + 4 * (q & 1) + e) ? 0xFFu << (8 * e) : 0u;
          }
        }
#pragma unroll
        for (int f = 0; f < NVF; ++f) {
          const u32x4 n = s_v[seg][vq_place<KB>(f, lane)], was = Vf[f * SEG * 64];
          Vf[f * SEG * 64] = (n & m) | (was & ~m);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        int sh;
        uint32_t* d = (uint32_t*)((uint8_t*)s_k + kq_byte(KB, 32 * seg + 8 * g + i, 8 * c, &sh));
        if constexpr (KB == 4) d[0] = to_tile_word(w[i][0]);
        else {
          d[0] = w[i][0];
          d[1] = w[i][1];
        }
      }
    }
  }
  if (!is_v) {
    wave_lds_order();
    u32x4* Kf = (u32x4*)(slab + geo.k_off);
#pragma unroll
    for (int j = 0; j < 2 * KF; ++j) {
      const int at = (seg * 2 * KF + j) * 64 + lane;
      if (appended(seg0 + k_seg_tok(j / KF, lane & 15))) Kf[at] = s_k[at];
      else if (fills) s_k[at] = Kf[at];
    }
  }
  const int tok = tid, pt = blk * TB + tok;  // threads 0 .. TB-1: one token's scales / biases
  const int at = tid < TB ? sb_entry(TB, tok) : 0;
  if (tid < TB) {
    if (!appended(pt)) {
      if (fills) s_sb[at] = Sb[at];
    } else if constexpr (!QUANTIZE) {
      const int64_t r = 2 * (row0 + pt);
      auto pair = [&](const uint16_t* a) { return (uint32_t)a[r] | ((uint32_t)a[r + 1] << 16); };
      const u32x4 f = u32x4{pair(src.ks), pair(src.kb), pair(src.vs), pair(src.vb)};
      s_sb[at] = f;
      Sb[at] = f;
    }
  }
  if (!QUANTIZE && !fills) return;
  __syncthreads();
  if constexpr (QUANTIZE)
    if (tid < TB && appended(pt)) Sb[at] = s_sb[at];
  if (fills && tid < kHeadDim)
    summary_row(geo, seq, h, blk)[tid] = fold_block_q<KB>((const uint8_t*)s_k, (const uint16_t*)s_sb, TB, tid);
}

// ---------------------------------------------------------------------------
// export in the MLX layout: kw / vw [n, Hkv, T, D*b/32] uint32 (LSB first),
// scales / biases [n, Hkv, T, D/64] fp16.  grid (ceil(T / TB), Hkv, n)
// ---------------------------------------------------------------------------
template <int KB, int TB>
__global__ __launch_bounds__(4 * TB) void k_export_blocks_q(Geometry geo, SeqBatch sb, int T, QuantDst dst) {
  constexpr int SEG = TB / 32, W = KB / 4, WPR = QCode<KB>::WPR;
  constexpr int NF = KB / 2;  // fragments of a segment, K or V
  __shared__ u32x4 s_v[SEG][NF * 64];
  __shared__ u32x4 s_k[TB * KB];
  const int blk = blockIdx.x, h = blockIdx.y, bi = blockIdx.z;
  const int page = block_table(geo, sb.ids[bi])[blk];
  const uint8_t* slab = geo.pool + ((size_t)page * geo.hkv + h) * geo.slab_bytes;
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63;
  const int seg = wave % SEG;
  const bool is_v = wave < SEG;
  const size_t row0 = ((size_t)bi * geo.hkv + h) * T + blk * TB;  // row of the block's token 0
  const int left = T - blk * TB;                                  // tokens from it on
  if (tid < TB && tid < left) {
    const u32x4 f = ((const u32x4*)(slab + geo.sb_off))[sb_entry(TB, tid)];
    const size_t r = 2 * (row0 + tid);
    auto put = [&](uint16_t* a, uint32_t p) {
      a[r] = (uint16_t)p;
      a[r + 1] = (uint16_t)(p >> 16);
    };
    put(dst.ks, f[0]);
    put(dst.kb, f[1]);
    put(dst.vs, f[2]);
    put(dst.vb, f[3]);
  }
  if (32 * seg >= left) return;
  const int g = lane >> 4, c = lane & 15;
  uint32_t w[8][W];
  u32x4 r[NF];
  if (is_v) {
    const u32x4* Vf = (const u32x4*)(slab + geo.v_off) + seg * 64 + lane;
#pragma unroll
    for (int f = 0; f < NF; ++f) r[f] = Vf[f * SEG * 64];
#pragma unroll
    for (int f = 0; f < NF; ++f) s_v[seg][vq_place<KB>(f, lane)] = r[f];
    wave_lds_order();
    uint32_t in[8][W];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t* d = vq_words<KB>(s_v[seg], g, c, e);
#pragma unroll
      for (int j = 0; j < W; ++j) in[e][j] = d[j];
    }
    transpose_codes<KB>(in, w, false);
  } else {
    const u32x4* Kf = (const u32x4*)(slab + geo.k_off) + seg * NF * 64 + lane;
#pragma unroll
    for (int f = 0; f < NF; ++f) r[f] = Kf[f * 64];
#pragma unroll
    for (int f = 0; f < NF; ++f) s_k[(seg * NF + f) * 64 + lane] = r[f];
    wave_lds_order();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      int sh;
      const uint32_t* d = (const uint32_t*)((const uint8_t*)s_k + kq_byte(KB, 32 * seg + 8 * g + i, 8 * c, &sh));
      if constexpr (KB == 4) w[i][0] = from_tile_word(d[0]);
      else {
        w[i][0] = d[0];
        w[i][1] = d[1];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int t = 32 * seg + 8 * g + i;
    uint32_t* o = (is_v ? dst.vw : dst.kw) + (row0 + t) * WPR + W * c;
    if (t < left)
#pragma unroll
      for (int j = 0; j < W; ++j) o[j] = w[i][j];
  }
}

// ===========================================================================
// launchers
// ===========================================================================
hipError_t launch_append(const Geometry& g, const AppendBatch& ab, const AppendPages& pg, const PatchBatch& pb,
                         int blocks, const void* k, const void* v, hipStream_t s, Timing* prof) {
  const dim3 grid(blocks, g.hkv, ab.n);
  const uint16_t *kk = (const uint16_t*)k, *vv = (const uint16_t*)v;
  const int kind = kProfAppend;
  if (g.tb == 64) {
    if (g.dtype == 0) launch(k_append_blocks<0, 64>, grid, dim3(256), 0, s, prof, kind, g, ab, pg, pb, kk, vv);
    else launch(k_append_blocks<1, 64>, grid, dim3(256), 0, s, prof, kind, g, ab, pg, pb, kk, vv);
  } else {
    if (g.dtype == 0) launch(k_append_blocks<0, 32>, grid, dim3(128), 0, s, prof, kind, g, ab, pg, pb, kk, vv);
    else launch(k_append_blocks<1, 32>, grid, dim3(128), 0, s, prof, kind, g, ab, pg, pb, kk, vv);
  }
  return hipGetLastError();
}

hipError_t launch_export(const Geometry& g, const SeqBatch& b, int T, void* k_out, void* v_out,
                         hipStream_t s) {
  const dim3 grid((T + g.tb - 1) / g.tb, g.hkv, b.n);
  if (g.tb == 64)
    hipLaunchKernelGGL(k_export_blocks<64>, grid, dim3(256), 0, s, g, b, T, (uint16_t*)k_out, (uint16_t*)v_out);
  else
    hipLaunchKernelGGL(k_export_blocks<32>, grid, dim3(128), 0, s, g, b, T, (uint16_t*)k_out, (uint16_t*)v_out);
  return hipGetLastError();
}

template <bool QUANTIZE>
static hipError_t append_q(const Geometry& g, const AppendBatch& ab, const AppendPages& pg, const PatchBatch& pb,
                           int blocks, const QuantSrc& src, hipStream_t s, Timing* prof) {
  const dim3 grid(blocks, g.hkv, ab.n);
  const int kind = kProfAppend;
  if (g.kv_bits == 4) {
    if (g.tb == 64) launch(k_append_blocks_q<4, 64, QUANTIZE>, grid, dim3(256), 0, s, prof, kind, g, ab, pg, pb, src);
    else launch(k_append_blocks_q<4, 32, QUANTIZE>, grid, dim3(128), 0, s, prof, kind, g, ab, pg, pb, src);
  } else {
    if (g.tb == 64) launch(k_append_blocks_q<8, 64, QUANTIZE>, grid, dim3(256), 0, s, prof, kind, g, ab, pg, pb, src);
    else launch(k_append_blocks_q<8, 32, QUANTIZE>, grid, dim3(128), 0, s, prof, kind, g, ab, pg, pb, src);
  }
  return hipGetLastError();
}

hipError_t launch_append_q16(const Geometry& g, const AppendBatch& ab, const AppendPages& pg, const PatchBatch& pb,
                             int blocks, const void* k, const void* v, hipStream_t s, Timing* prof) {
  QuantSrc src{};
  src.k16 = (const uint16_t*)k;
  src.v16 = (const uint16_t*)v;
  return append_q<true>(g, ab, pg, pb, blocks, src, s, prof);
}

hipError_t launch_append_quantized(const Geometry& g, const AppendBatch& ab, const AppendPages& pg,
                                   const PatchBatch& pb, int blocks, const uint32_t* kw, const void* ks,
                                   const void* kb, const uint32_t* vw, const void* vs, const void* vb,
                                   hipStream_t s, Timing* prof) {
  const QuantSrc src{nullptr, nullptr, kw, vw, (const uint16_t*)ks, (const uint16_t*)kb, (const uint16_t*)vs,
                     (const uint16_t*)vb};
  return append_q<false>(g, ab, pg, pb, blocks, src, s, prof);
}

hipError_t launch_export_quantized(const Geometry& g, const SeqBatch& b, int T, uint32_t* kw,
                                   void* ks, void* kb, uint32_t* vw, void* vs, void* vb,
                                   hipStream_t s) {
  const dim3 grid((T + g.tb - 1) / g.tb, g.hkv, b.n);
  const QuantDst dst{kw, vw, (uint16_t*)ks, (uint16_t*)kb, (uint16_t*)vs, (uint16_t*)vb};
  if (g.kv_bits == 4) {
    if (g.tb == 64) hipLaunchKernelGGL((k_export_blocks_q<4, 64>), grid, dim3(256), 0, s, g, b, T, dst);
    else hipLaunchKernelGGL((k_export_blocks_q<4, 32>), grid, dim3(128), 0, s, g, b, T, dst);
  } else {
    if (g.tb == 64) hipLaunchKernelGGL((k_export_blocks_q<8, 64>), grid, dim3(256), 0, s, g, b, T, dst);
    else hipLaunchKernelGGL((k_export_blocks_q<8, 32>), grid, dim3(128), 0, s, g, b, T, dst);
  }
  return hipGetLastError();
}

}  // namespace bsattn
