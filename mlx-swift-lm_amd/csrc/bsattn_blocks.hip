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

}  // namespace bsattn
