// Indexer stage-0 block scores on the matrix cores, and their training gradient (gfx950).
//
//   score[t, c] = max over keys j of block c with seg(t) <= j < ls(t) of q_t . k_j,
//   ls(t) = max(pos(t) - LW + 1, 0)      (dash_attention.py:801-835,
//                                         sparse_gather_triton.py:395-428)
//
//   blockmax_f32_kernel     inference: 128 query rows x up to 128 keys per work-group by
//                           fp32 matrix products, the bits of the row-by-row kernel
//   blockmax_split_kernel   training: fp32 keys -> three bf16 parts per key, in the LDS
//                           image of a 32-key tile
//   blockmax_mfma_kernel    training: 128 query rows x up to 1,024 keys per work-group by
//                           products of the bf16 parts
//   blockmax_bwd_q_kernel   dq of every row from the winning keys, and the bit mask of
//                           the (row, block) pairs with a gradient
//   blockmax_bwd_k_kernel   dk of every key from that mask; blockmax_bwd_sum_kernel adds
//                           its row ranges
//
// In training every fp32 operand is x = x_h + x_m + x_l (three round-to-nearest bf16 parts, 24
// significand bits), and q.k the fp32-accumulated sum of the six products x_i y_j with
// i + j <= 2; the dropped ones are below 2^-24 of the product.  Operands that are not
// finite, or beyond 2^60 (their products could overflow in another order), take a scalar
// fp32 dot product instead.
//
// The gradient of a maximum goes to the keys that attain it, in equal shares.  The forward
// pass keeps the winning key of every (row, block) in a byte; 255 stands for "no single
// winner" (none visible, a tie, or a value at the clamp), which the backward pass works
// out again from fp32 dot products.

#include "dash_common.h"

#include <limits.h>

#include <type_traits>

namespace dash {

constexpr int kBmTile = 32;                       // keys per tile
constexpr int kBmPlane = kBmTile * 128;           // elements of one part of a tile
constexpr int kBmTileBytes = 3 * kBmPlane * 2;    // 24 KB
constexpr int kBmRows = 128;                      // query rows per work-group
constexpr int kBmMaxChunk = 1024;                 // keys per work-group, at most
constexpr int kBmMaxBlocks = kBmMaxChunk / 32;    // blocks per work-group, at most
constexpr int kBmF32Chunk = 128;                  // keys per work-group of the fp32 kernel, at most
constexpr int kBmSlow = 255;                      // no single winning key
constexpr int kBmRange = 4096;                    // query rows per dk work-group
constexpr float kBmWide = 1.152921504606847e18f;  // 2^60

typedef __attribute__((address_space(3))) void lds_void;

struct BlockMaxArgs {
  const float* q; int64_t q_sb, q_st;
  const float* k; int64_t k_sb, k_st;
  const int32_t* pos; const int32_t* seg; int64_t ps_sb;
  const char* planes;          // [B, ntiles] tiles of kBmTileBytes
  const int32_t* wide;         // [B, ntiles] tile holds operands for the scalar path
  int B, C, Sk, bs, lw, nblk, mode;
  int ntiles;                  // nblk * bs / 32
  int chunk_tiles;             // tiles per work-group (whole blocks)
  float* out; int64_t o_sb, o_sc;
  uint8_t* arg;                // [B, C, nblk] winning key within its block, or null
};

__device__ __forceinline__ bool bm_wide(float x) { return !(fabsf(x) <= kBmWide); }

__device__ __forceinline__ void bm_split3(float x, __bf16& h, __bf16& m, __bf16& l) {
  h = (__bf16)x;
  const float r1 = x - (float)h;
  m = (__bf16)r1;
  l = (__bf16)(r1 - (float)m);
}

// The fp32 matrix product adds its two k values one after the other, each as a fused
// multiply-add, so 64 of them over a row's dims in order leave the sum that the FMA loop of
// the row-by-row kernel (blockmax_kernel) forms, with its infinities, NaNs and subnormal
// values.  A row's scores are the same bits whichever kernel takes it, in a prompt, a chunk
// or a decode step, and rows whose scores all but tie route alike.  (The products of bf16
// parts below sum in another order: with them a prompt of 2,730 tokens routed some rows to
// another block than its chunks did.)
// Each wavefront keeps its 32 rows in 64 registers (lane (n, hl): dims 2 i + hl of row n);
// S^T = K Q^T gives lane l the scores of query l % 32, so the maximum over a block's keys is
// per lane, with one exchange between the wave's halves.  Key tiles stream through two 16 KB
// stages by direct loads.  Bound by the matrix products, 4,096 cycles per wavefront and tile
// (1,536 with bf16 parts, which need the keys split first), at half their rate.  In blocks of
// 32, 2,730 rows and keys take 26.9 us (row by row 93.9, bf16 parts 24.2), 8,301 133.3 (bf16 parts
// 85.6), 2,730 rows of 27,300 keys 206.9 (753.7, 138.9), one row of 2,730 keys 7.3 (16.0, 15.8).
__global__ __launch_bounds__(256, 3) void blockmax_f32_kernel(BlockMaxArgs a) {
  __shared__ __attribute__((aligned(16))) float s0[kBmTile * 128];
  __shared__ __attribute__((aligned(16))) float s1[kBmTile * 128];
  __shared__ float sOut[4][32][kBmF32Chunk / 32 + 1];
  __shared__ int sHi[4];
  const int b = blockIdx.z, r0 = blockIdx.x * kBmRows;
  const int tid = threadIdx.x, lane = wave_lane(), wv = tid / kWave;
  const int n = lane & 31, hl = lane >> 5;
  const int tpb = a.bs / kBmTile;
  const int T0 = blockIdx.y * a.chunk_tiles;
  const int Tend = min(T0 + a.chunk_tiles, a.ntiles);
  const int c0 = T0 / tpb, nb = (Tend - T0) / tpb;        // this chunk's blocks
  const float empty = a.mode == 1 ? -INFINITY : kScoreNeg;

  const int rw = r0 + wv * 32;                            // the wavefront's first row
  const bool rok = rw + n < a.C;
  const int rc = min(rw + n, a.C - 1);
  // visible keys [lo, hi)
  const int64_t ls = (int64_t)a.pos[(int64_t)b * a.ps_sb + rc] - a.lw + 1;
  const int hi = (int)(ls < 0 ? 0 : (ls < a.Sk ? ls : a.Sk));
  const int lo = a.seg ? a.seg[(int64_t)b * a.ps_sb + rc] : 0;
  int w_hi = rok ? hi : 0;
#pragma unroll
  for (int m = 16; m >= 1; m >>= 1) w_hi = max(w_hi, __shfl_xor(w_hi, m, kWave));
  w_hi = __builtin_amdgcn_readfirstlane(w_hi);            // most keys any of its rows sees
  if (lane == 0) sHi[wv] = w_hi;
  for (int e = lane; e < 32 * nb; e += kWave) sOut[wv][e / nb][e % nb] = empty;
  __syncthreads();
  const int g_hi = max(max(sHi[0], sHi[1]), max(sHi[2], sHi[3]));
  // tiles with a visible key, in whole blocks
  int T1 = (g_hi + kBmTile - 1) / kBmTile;
  T1 = min((T1 + tpb - 1) / tpb * tpb, Tend);

  if (T0 < T1) {
    const float* qr = a.q + (int64_t)b * a.q_sb + (int64_t)rc * a.q_st;
    float q[64];
#pragma unroll
    for (int c = 0; c < 32; ++c) {
      const float4 x = *(const float4*)(qr + 4 * c);
      q[2 * c] = hl ? x.y : x.x;
      q[2 * c + 1] = hl ? x.w : x.z;
    }
    const float* kb = a.k + (int64_t)b * a.k_sb;
    // 16-byte chunk c of key row r at slot c ^ r of its 512 bytes; rows past the keys
    // repeat the last one
    auto fetch = [&](float* s, int T) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int pr = 4 * u + wv, r = 2 * pr + hl;
        const float* src = kb + (int64_t)min(T * kBmTile + r, a.Sk - 1) * a.k_st + ((n ^ r) << 2);
        __builtin_amdgcn_global_load_lds((const void*)src, (lds_void*)(s + pr * 256), 16, 0, 0);
      }
    };
    float best = -INFINITY;                // the block's maximum over this lane's keys
    auto step = [&](int T, auto par) {
      constexpr int P = decltype(par)::value;
      const float* const sc = P == 0 ? s0 : s1;
      float* const sn = P == 0 ? s1 : s0;
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();                     // tile T landed; every wavefront left T - 1
      if (T + 1 < T1) fetch(sn, T + 1);
      const int j0 = T * kBmTile;
      if (j0 < w_hi) {
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int c = 0; c < 32; ++c) {
          const float4 x = *(const float4*)(sc + n * 128 + ((c ^ n) << 2));
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(hl ? x.y : x.x, q[2 * c], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(hl ? x.w : x.z, q[2 * c + 1], acc, 0, 0, 0);
        }
        // register i: key j0 + 8 (i / 4) + 4 hl + i % 4
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = j0 + 8 * (i >> 2) + 4 * hl + (i & 3);
          float v = acc[i];
          if (a.mode == 0) v = fminf(fmaxf(v, -kActClamp), kActClamp);
          best = fmaxf(best, (j >= lo && j < hi) ? v : -INFINITY);
        }
      }
      if ((T + 1) % tpb == 0) {            // the block is complete
        const float m = fmaxf(best, __shfl_xor(best, 32, kWave));
        if (hl == 0) sOut[wv][n][T / tpb - c0] = m == -INFINITY ? empty : m;
        best = -INFINITY;
      }
    };
    fetch(s0, T0);
    for (int T = T0; T < T1; T += 2) {
      step(T, std::integral_constant<int, 0>{});
      if (T + 1 < T1) step(T + 1, std::integral_constant<int, 1>{});
    }
  }
  __syncthreads();
  for (int e = lane; e < 32 * nb; e += kWave) {
    const int rr = e / nb, cc = e % nb;
    if (rw + rr < a.C)
      a.out[(int64_t)b * a.o_sb + (int64_t)(rw + rr) * a.o_sc + c0 + cc] = sOut[wv][rr][cc];
  }
}

// One work-group per 32-key tile.  16-byte chunk c (8 dims) of key row n sits in slot
// c ^ (n % 16) of its 256-byte row, so that the 32 lanes of an operand read (32 rows, one
// chunk) cover the LDS banks evenly.
__global__ __launch_bounds__(256) void blockmax_split_kernel(const float* __restrict__ k,
                                                             int64_t k_sb, int64_t k_st, int Sk,
                                                             int ntiles, char* __restrict__ planes,
                                                             int32_t* __restrict__ wide) {
  const int tile = blockIdx.x, b = blockIdx.y;
  bf16* const p = (bf16*)(planes + ((int64_t)b * ntiles + tile) * kBmTileBytes);
  const int n = threadIdx.x >> 3, c0 = (threadIdx.x & 7) * 2;    // row, two chunks
  const int j = tile * kBmTile + n;
  float4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (j < Sk) {
    const float* r = k + (int64_t)b * k_sb + (int64_t)j * k_st + c0 * 8;
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *(const float4*)(r + 4 * u);
  }
  bool w = false;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const float xs[8] = {v[2 * c].x, v[2 * c].y, v[2 * c].z, v[2 * c].w,
                         v[2 * c + 1].x, v[2 * c + 1].y, v[2 * c + 1].z, v[2 * c + 1].w};
    bf16x8 h, m, l;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      w |= bm_wide(xs[e]);
      __bf16 a, d, f;
      bm_split3(xs[e], a, d, f);
      h[e] = a; m[e] = d; l[e] = f;
    }
    const int off = n * 128 + (((c0 + c) ^ (n & 15)) << 3);
    *(bf16x8*)(p + off) = h;
    *(bf16x8*)(p + kBmPlane + off) = m;
    *(bf16x8*)(p + 2 * kBmPlane + off) = l;
  }
  const int any = __syncthreads_or(w);
  if (threadIdx.x == 0) wide[(int64_t)b * ntiles + tile] = any;
}

// What bounds it: 48 MFMAs of 32 cycles per wavefront and tile (six products of 8 k-steps)
// against 24 KB of LDS operand reads, so the matrix cores; the keys are split once by the
// kernel above instead of once per row tile.  Each wavefront keeps its 32 rows' three parts
// in 96 registers; S^T = K Q^T gives lane l the scores of query l % 32, so the maximum over
// a block's keys is per lane, with one exchange between the wave's halves.  Tiles stream
// through two 24 KB stages by direct loads (two work-groups per CU).
template <bool ARG>
__global__ __launch_bounds__(256, 2) void blockmax_mfma_kernel(BlockMaxArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 s0[3 * kBmPlane];
  __shared__ __attribute__((aligned(16))) bf16 s1[3 * kBmPlane];
  __shared__ float sOut[4][32][kBmMaxBlocks + 1];
  __shared__ uint8_t sArg[4][32][kBmMaxBlocks + 4];
  __shared__ int sHi[4];
  const int b = blockIdx.z, r0 = blockIdx.x * kBmRows;
  const int tid = threadIdx.x, lane = wave_lane(), wv = tid / kWave;
  const int n = lane & 31, hl = lane >> 5;
  const int tpb = a.bs / kBmTile;
  const int T0 = blockIdx.y * a.chunk_tiles;
  const int Tend = min(T0 + a.chunk_tiles, a.ntiles);
  const int c0 = T0 / tpb, nb = (Tend - T0) / tpb;        // this chunk's blocks
  const float empty = a.mode == 1 ? -INFINITY : kScoreNeg;

  const int rw = r0 + wv * 32;                            // the wavefront's first row
  const int r = rw + n;
  const bool rok = r < a.C;
  const int rc = min(r, a.C - 1);
  const int p = a.pos[(int64_t)b * a.ps_sb + rc];
  // visible keys [lo, hi)
  const int64_t ls = (int64_t)p - a.lw + 1;
  const int hi = (int)(ls < 0 ? 0 : (ls < a.Sk ? ls : a.Sk));
  const int lo = a.seg ? a.seg[(int64_t)b * a.ps_sb + rc] : 0;
  int w_hi = rok ? hi : 0, w_lo = rok ? lo : INT_MIN, w_min = rok ? hi : INT_MAX;
#pragma unroll
  for (int m = 16; m >= 1; m >>= 1) {
    w_hi = max(w_hi, __shfl_xor(w_hi, m, kWave));
    w_lo = max(w_lo, __shfl_xor(w_lo, m, kWave));
    w_min = min(w_min, __shfl_xor(w_min, m, kWave));
  }
  w_hi = __builtin_amdgcn_readfirstlane(w_hi);            // most keys any of its rows sees
  w_lo = __builtin_amdgcn_readfirstlane(w_lo);
  w_min = __builtin_amdgcn_readfirstlane(w_min);
  if (lane == 0) sHi[wv] = w_hi;
  for (int e = lane; e < 32 * nb; e += kWave) {
    sOut[wv][e / nb][e % nb] = empty;
    if (ARG) sArg[wv][e / nb][e % nb] = (uint8_t)kBmSlow;
  }
  __syncthreads();
  const int g_hi = max(max(sHi[0], sHi[1]), max(sHi[2], sHi[3]));
  // tiles with a visible key, in whole blocks
  int T1 = (g_hi + kBmTile - 1) / kBmTile;
  T1 = min((T1 + tpb - 1) / tpb * tpb, Tend);

  if (T0 < T1) {
    // this row's 128 dims in three parts: lane (n, hl) holds dims 16 kk + 8 hl .. +7
    const float* qr = a.q + (int64_t)b * a.q_sb + (int64_t)rc * a.q_st + 8 * hl;
    bf16x8 qh[8], qm[8], ql[8];
    bool qwide = false;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const float4 x = *(const float4*)(qr + 16 * kk), y = *(const float4*)(qr + 16 * kk + 4);
      const float xs[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        qwide |= bm_wide(xs[e]);
        __bf16 h, m, l;
        bm_split3(xs[e], h, m, l);
        qh[kk][e] = h; qm[kk][e] = m; ql[kk][e] = l;
      }
    }
    const char* tiles = a.planes + (int64_t)b * a.ntiles * kBmTileBytes;
    // bit T - T0: the tile's scores come from the scalar path
    const bool twide = T0 + lane < T1 && a.wide[(int64_t)b * a.ntiles + T0 + lane] != 0;
    const uint32_t wide = __any(qwide) ? ~0u : (uint32_t)__ballot(twide);
    auto fetch = [&](bf16* s, int T) {
      const char* src = tiles + (int64_t)T * kBmTileBytes + wv * 6144 + lane * 16;
#pragma unroll
      for (int u = 0; u < 6; ++u)
        __builtin_amdgcn_global_load_lds((const void*)(src + u * 1024),
                                         (lds_void*)((char*)s + wv * 6144 + u * 1024), 16, 0, 0);
    };
    const uint32_t koff = (uint32_t)(n * 256) | (uint32_t)((hl << 4) ^ ((n & 15) << 4));
    // the block's running maximum over this lane's keys, its key and how often it occurs
    float best = -INFINITY;
    int barg = 0, bcnt = 0;
    auto step = [&](int T, auto par) {
      constexpr int P = decltype(par)::value;
      bf16* const sc = P == 0 ? s0 : s1;
      bf16* const sn = P == 0 ? s1 : s0;
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();                     // tile T landed; every wavefront left T - 1
      if (T + 1 < T1) fetch(sn, T + 1);
      const int j0 = T * kBmTile;
      if (j0 < w_hi) {
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
        uint32_t ko = koff;
        asm volatile("" : "+v"(ko));
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          const char* pr = (const char*)sc + (ko ^ (uint32_t)(kk << 5));
          const bf16x8 kh = *(const bf16x8*)pr;
          const bf16x8 km = *(const bf16x8*)(pr + 2 * kBmPlane);
          const bf16x8 kl = *(const bf16x8*)(pr + 4 * kBmPlane);
          // smallest terms first
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kl, qh[kk], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, ql[kk], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(km, qm[kk], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(km, qh[kk], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, qm[kk], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, qh[kk], acc, 0, 0, 0);
        }
        // register i: key j0 + 8 (i / 4) + 4 hl + i % 4
        if ((wide >> (T - T0)) & 1u) {
          const float* q1 = a.q + (int64_t)b * a.q_sb + (int64_t)rc * a.q_st;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int j = min(j0 + 8 * (i >> 2) + 4 * hl + (i & 3), a.Sk - 1);
            const float* k1 = a.k + (int64_t)b * a.k_sb + (int64_t)j * a.k_st;
            float s = 0.f;
            for (int d = 0; d < 128; ++d) s = fmaf(q1[d], k1[d], s);
            // a NaN score counts as the lower clamp (mode 0), not at all (mode 1), or makes
            // the block's score NaN (mode 2: carried as +inf, which the clamp excludes)
            if (a.mode == 1)
              s = fmaxf(s, -INFINITY);
            else if (a.mode == 2 && s != s)
              s = INFINITY;
            else
              s = fminf(fmaxf(s, -kActClamp), kActClamp);
            acc[i] = s;
          }
        }
        if (j0 + kBmTile > w_min || w_lo > j0) {           // some row does not see all of it
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int j = j0 + 8 * (i >> 2) + 4 * hl + (i & 3);
            acc[i] = (j >= lo && j < hi) ? acc[i] : -INFINITY;
          }
        }
        float m = acc[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) m = fmaxf(m, acc[i]);
        if (ARG) {
          int cnt = 0, arg = 0;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const bool e = acc[i] == m;
            cnt += e;
            arg = e ? 8 * (i >> 2) + (i & 3) : arg;
          }
          arg += (T % tpb) * kBmTile + 4 * hl;
          if (m > best) {
            barg = arg;
            bcnt = cnt;
          } else if (m == best) {
            bcnt += cnt;
          }
        }
        best = fmaxf(best, m);
      }
      if ((T + 1) % tpb == 0) {            // the block is complete
        const float ob = __shfl_xor(best, 32, kWave);
        const float m = fmaxf(best, ob);
        const int col = T / tpb - c0;
        if (ARG) {
          const int oa = __shfl_xor(barg, 32, kWave), oc = __shfl_xor(bcnt, 32, kWave);
          const int cnt = (best == m ? bcnt : 0) + (ob == m ? oc : 0);
          const int arg = best == m ? barg : oa;
          const bool one = cnt == 1 && m > -INFINITY && (a.mode == 1 || fabsf(m) < kActClamp);
          if (hl == 0) sArg[wv][n][col] = (uint8_t)(one ? arg : kBmSlow);
        }
        if (hl == 0)
          sOut[wv][n][col] = m == -INFINITY ? empty
                             : a.mode == 1 ? m
                             : m == INFINITY && a.mode == 2 ? __builtin_nanf("")
                                           : fminf(fmaxf(m, -kActClamp), kActClamp);
        best = -INFINITY;
        barg = bcnt = 0;
      }
    };
    fetch(s0, T0);
    for (int T = T0; T < T1; T += 2) {
      step(T, std::integral_constant<int, 0>{});
      if (T + 1 < T1) step(T + 1, std::integral_constant<int, 1>{});
    }
  }
  __syncthreads();
  for (int e = lane; e < 32 * nb; e += kWave) {
    const int rr = e / nb, cc = e % nb;
    if (rw + rr < a.C) {
      a.out[(int64_t)b * a.o_sb + (int64_t)(rw + rr) * a.o_sc + c0 + cc] = sOut[wv][rr][cc];
      if (ARG) a.arg[((int64_t)b * a.C + rw + rr) * a.nblk + c0 + cc] = sArg[wv][rr][cc];
    }
  }
}

// ---------------------------------------------------------------------------
// Backward
// ---------------------------------------------------------------------------
struct BlockMaxBwdArgs {
  const float* q; int64_t q_sb, q_st;
  const float* k; int64_t k_sb, k_st;
  const int32_t* pos; int64_t ps_sb;
  const uint8_t* arg;          // [B, C, nblk]
  const float* g; int64_t g_sb, g_sc;
  float* dq; float* dk;        // [B, C, 128], [B, Sk, 128] contiguous
  int B, C, Sk, bs, lw, nblk;
  int nwords;                  // 64-block words of the mask
  uint64_t* mask;              // [B, nwords, C]
  int nrange;                  // row ranges of kBmRange rows
  float* part;                 // [nrange, B, Sk, 128] (nrange > 1)
  int32_t* used;               // [nrange, B, nblk] (nrange > 1)
};

// The keys of block c that attain the maximum of row r, as a wavefront: each lane takes
// keys c bs + lane (+ 64); returns the share of the gradient per key (0: none) and in
// hit[u] whether this lane's key u takes part.  A key beyond the clamp attains it but
// passes no gradient.
__device__ __forceinline__ float bm_ties(const BlockMaxBwdArgs& a, int b, int r, int c, float g,
                                         bool (&hit)[2]) {
  const int lane = wave_lane();
  const int64_t ls = (int64_t)a.pos[(int64_t)b * a.ps_sb + r] - a.lw + 1;
  const int hi = (int)(ls < 0 ? 0 : (ls < a.Sk ? ls : a.Sk));
  const float* q = a.q + (int64_t)b * a.q_sb + (int64_t)r * a.q_st;
  float raw[2], val[2];
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int o = lane + 64 * u, j = c * a.bs + o;
    raw[u] = 0.f;
    val[u] = -INFINITY;
    if (o < a.bs && j < hi) {
      const float* k = a.k + (int64_t)b * a.k_sb + (int64_t)j * a.k_st;
      float s = 0.f;
      for (int d = 0; d < 128; ++d) s = fmaf(q[d], k[d], s);
      raw[u] = s;
      val[u] = fminf(fmaxf(s, -kActClamp), kActClamp);
    }
    m = fmaxf(m, val[u]);
  }
  m = wave_max(m);
  int cnt = 0;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const bool e = m > -INFINITY && val[u] == m;
    cnt += __popcll(__ballot(e));
    hit[u] = e && fabsf(raw[u]) <= kActClamp;   // never a NaN
  }
  return cnt > 0 ? g / (float)cnt : 0.f;
}

// One wavefront per row.  The gradient is zero outside the entmax support, so a row has
// tens of nonzero entries of its nblk: they are found 64 at a time by ballot, and each
// adds its share of the winning key's 512-byte row (two dims per lane).  Bound by the
// reads of g and arg, 5 B per (row, block).
__global__ __launch_bounds__(256) void blockmax_bwd_q_kernel(BlockMaxBwdArgs a) {
  const int b = blockIdx.y, r = blockIdx.x * 4 + threadIdx.x / kWave;
  if (r >= a.C) return;
  const int lane = wave_lane();
  const float* gr = a.g + (int64_t)b * a.g_sb + (int64_t)r * a.g_sc;
  const uint8_t* ar = a.arg + ((int64_t)b * a.C + r) * a.nblk;
  const float* kb = a.k + (int64_t)b * a.k_sb + 2 * lane;
  float2 acc = make_float2(0.f, 0.f);
  for (int w = 0; w < a.nwords; ++w) {
    const int c = w * 64 + lane;
    const float g = c < a.nblk ? gr[c] : 0.f;
    const int arg = c < a.nblk ? ar[c] : 0;
    const uint64_t nz = __ballot(g != 0.f);
    const uint64_t slow = nz & __ballot(arg == kBmSlow);
    if (lane == 0) a.mask[((int64_t)b * a.nwords + w) * a.C + r] = nz;
    uint64_t todo = nz & ~slow;
    while (todo) {                         // four rows in flight
      float gu[4];
      float2 x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int f = todo ? __builtin_ctzll(todo) : 0;
        gu[u] = todo ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(g), f)) : 0.f;
        const int j = (w * 64 + f) * a.bs + __builtin_amdgcn_readlane(arg, f);
        x[u] = make_float2(0.f, 0.f);
        if (todo) x[u] = *(const float2*)(kb + (int64_t)j * a.k_st);
        todo &= todo - 1;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc.x = fmaf(gu[u], x[u].x, acc.x);
        acc.y = fmaf(gu[u], x[u].y, acc.y);
      }
    }
    uint64_t rest = slow;
    while (rest) {
      const int f = __builtin_ctzll(rest);
      rest &= rest - 1;
      const int cb = w * 64 + f;
      bool hit[2];
      const float share =
          bm_ties(a, b, r, cb, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(g), f)), hit);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint64_t keys = __ballot(hit[u]);
        while (keys) {
          const int64_t j = (int64_t)cb * a.bs + 64 * u + __builtin_ctzll(keys);
          keys &= keys - 1;
          const float2 x = *(const float2*)(kb + j * a.k_st);
          acc.x = fmaf(share, x.x, acc.x);
          acc.y = fmaf(share, x.y, acc.y);
        }
      }
    }
  }
  *(float2*)(a.dq + ((int64_t)b * a.C + r) * 128 + 2 * lane) = acc;
}

// One work-group per (key block, range of kBmRange rows, sequence).  Each wavefront walks
// its share of the range's rows in order (64 mask words per load, one bit each), keeps the
// block's dk in LDS (two dims per lane) and adds g q_t to the winning key's row; the
// wavefronts' sums are then added in a fixed order, so dk is the same on every run.  Bound
// by the latency of the q rows (four in flight per wavefront).
template <int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void blockmax_bwd_k_kernel(BlockMaxBwdArgs a) {
  extern __shared__ __attribute__((aligned(16))) float sAcc[];   // [WAVES][bs][128]
  __shared__ int sUsed;
  const int c = blockIdx.x, rg = blockIdx.y, b = blockIdx.z;
  const int lane = wave_lane(), wv = threadIdx.x / kWave;
  float* const acc = sAcc + (int64_t)wv * a.bs * 128;
  for (int e = lane; e < a.bs * 32; e += kWave)
    ((float4*)acc)[e] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (threadIdx.x == 0) sUsed = 0;
  __syncthreads();
  const int per = kBmRange / WAVES;
  const int t0 = rg * kBmRange + wv * per, t1 = min(t0 + per, a.C);
  const uint64_t* mw = a.mask + ((int64_t)b * a.nwords + (c >> 6)) * a.C;
  const uint64_t bit = 1ull << (c & 63);
  const float* qb = a.q + (int64_t)b * a.q_sb + 2 * lane;
  bool any = false;
  auto add = [&](int key, float w, const float2& x) {
    float2* p = (float2*)(acc + key * 128 + 2 * lane);
    float2 y = *p;
    y.x = fmaf(w, x.x, y.x);
    y.y = fmaf(w, x.y, y.y);
    *p = y;
  };
  for (int t = t0; t < t1; t += kWave) {
    const int r = t + lane;
    const bool on = r < t1 && (mw[r] & bit);
    uint64_t todo = __ballot(on);
    if (!todo) continue;
    any = true;
    const float g = on ? a.g[(int64_t)b * a.g_sb + (int64_t)r * a.g_sc + c] : 0.f;
    const int arg = on ? a.arg[((int64_t)b * a.C + r) * a.nblk + c] : 0;
    const uint64_t slow = __ballot(on && arg == kBmSlow);
    todo &= ~slow;
    while (todo) {                         // four rows in flight
      float gu[4];
      int ku[4];
      float2 x[4];
      bool in[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        in[u] = todo != 0;
        const int f = in[u] ? __builtin_ctzll(todo) : 0;
        gu[u] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(g), f));
        ku[u] = __builtin_amdgcn_readlane(arg, f);
        x[u] = make_float2(0.f, 0.f);
        if (in[u]) x[u] = *(const float2*)(qb + (int64_t)(t + f) * a.q_st);
        todo &= todo - 1;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (in[u]) add(ku[u], gu[u], x[u]);
    }
    uint64_t rest = slow;
    while (rest) {
      const int f = __builtin_ctzll(rest);
      rest &= rest - 1;
      bool hit[2];
      const float share = bm_ties(
          a, b, t + f, c, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(g), f)), hit);
      const float2 x = *(const float2*)(qb + (int64_t)(t + f) * a.q_st);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint64_t keys = __ballot(hit[u]);
        while (keys) {
          add(64 * u + __builtin_ctzll(keys), share, x);
          keys &= keys - 1;
        }
      }
    }
  }
  if (any && lane == 0) sUsed = 1;
  __syncthreads();
  if (a.nrange > 1) {
    const int64_t cell = ((int64_t)rg * a.B + b) * a.nblk + c;
    if (threadIdx.x == 0) a.used[cell] = sUsed;
    if (!sUsed) return;
  }
  float* const dst = a.nrange > 1 ? a.part + ((int64_t)rg * a.B + b) * a.Sk * 128
                                  : a.dk + (int64_t)b * a.Sk * 128;
  const int nkeys = min(a.bs, a.Sk - c * a.bs);
  for (int e = threadIdx.x; e < nkeys * 32; e += WAVES * kWave) {
    float4 s = ((const float4*)sAcc)[e];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      const float4 y = ((const float4*)(sAcc + (int64_t)w * a.bs * 128))[e];
      s.x += y.x; s.y += y.y; s.z += y.z; s.w += y.w;
    }
    ((float4*)(dst + (int64_t)c * a.bs * 128))[e] = s;
  }
}

// dk = the sum of the row ranges' parts, in range order: 32 lanes per key row.
__global__ __launch_bounds__(256) void blockmax_bwd_sum_kernel(BlockMaxBwdArgs a) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = e >> 5;
  if (row >= (int64_t)a.B * a.Sk) return;
  const int b = (int)(row / a.Sk), j = (int)(row % a.Sk);
  const int c = j / a.bs;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int rg = 0; rg < a.nrange; ++rg) {
    if (c >= a.nblk || !a.used[((int64_t)rg * a.B + b) * a.nblk + c]) continue;
    const float4 y = ((const float4*)a.part)[(int64_t)rg * a.B * a.Sk * 32 + e];
    s.x += y.x; s.y += y.y; s.z += y.z; s.w += y.w;
  }
  ((float4*)a.dk)[e] = s;
}

static bool bm_supported(int d, int bs) {
  return d == 128 && (bs == 32 || bs == 64 || bs == 96 || bs == 128);
}
static bool bm_rows_ok(const void* p, int64_t sb, int64_t st) {
  return (uintptr_t)p % 16 == 0 && sb % 4 == 0 && st % 4 == 0;
}
static int bm_status() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? kOk : (int)e;
}

}  // namespace dash

extern "C" int dash_block_max_fused_workspace_size(int B, int block_size, int nblk,
                                                   int64_t* bytes) {
  using namespace dash;
  if (!bytes || B < 0 || nblk < 0) return kErrInvalid;
  if (!bm_supported(128, block_size)) return kErrUnsupported;
  const int64_t nt = (int64_t)nblk * (block_size / kBmTile);
  *bytes = (int64_t)B * nt * (kBmTileBytes + 4);
  return kOk;
}

extern "C" int dash_block_max_fused(const float* q, int64_t q_sb, int64_t q_st, int C,
                                    const int32_t* pos, const int32_t* seg, int64_t ps_sb,
                                    const float* k, int64_t k_sb, int64_t k_st, int Sk, int B,
                                    int d, int block_size, int local_window, int nblk, int mode,
                                    float* out, int64_t o_sb, int64_t o_sc, uint8_t* arg, void* ws,
                                    int64_t ws_bytes, void* stream) {
  using namespace dash;
  if (!q || !pos || !k || !out || B < 0 || C < 0 || nblk < 0 || Sk < 0) return kErrInvalid;
  if (mode < 0 || mode > 2) return kErrInvalid;
  if (!bm_supported(d, block_size) || !bm_rows_ok(q, q_sb, q_st) || !bm_rows_ok(k, k_sb, k_st) ||
      B > 65535)
    return kErrUnsupported;
  const int tpb = block_size / kBmTile, nt = nblk * tpb, rt = (C + kBmRows - 1) / kBmRows;
  BlockMaxArgs a{};
  a.q = q; a.q_sb = q_sb; a.q_st = q_st; a.k = k; a.k_sb = k_sb; a.k_st = k_st;
  a.pos = pos; a.seg = seg; a.ps_sb = ps_sb;
  a.B = B; a.C = C; a.Sk = Sk; a.bs = block_size; a.lw = std::max(1, local_window);
  a.nblk = nblk; a.mode = mode; a.ntiles = nt;
  a.out = out; a.o_sb = o_sb; a.o_sc = o_sc; a.arg = arg;
  hipStream_t st = (hipStream_t)stream;
  // keys per work-group: as many as let the rows' reads serve many keys, halved while the
  // grid holds too few work-groups
  auto blocks_per_group = [&](int most, int least, int64_t groups) {
    int keys = most;
    while (keys > least && (int64_t)rt * B * ((nt * kBmTile + keys - 1) / keys) < groups) keys /= 2;
    return std::max(1, keys / block_size);
  };
  if (mode != 2 && !arg) {
    if (B == 0 || C == 0 || nblk == 0) return kOk;
    // blocks of 32: 1,000 rows and keys 10.1 us with 32 keys (21.2 with 128), 2,730 26.9 with 64
    // (30.6 with 32, 31.8 with 128), 8,301 133.3 with 128 (140.7 with 64, 189.8 with 1,024)
    const int bpc = blocks_per_group(kBmF32Chunk, 32, 512);
    a.chunk_tiles = bpc * tpb;
    blockmax_f32_kernel<<<dim3(rt, (nblk + bpc - 1) / bpc, B), 256, 0, st>>>(a);
    return bm_status();
  }
  if (!ws) return kErrInvalid;
  if ((uintptr_t)ws % 16 != 0) return kErrUnsupported;
  int64_t need = 0;
  dash_block_max_fused_workspace_size(B, block_size, nblk, &need);
  if (ws_bytes < need) return kErrWorkspace;
  if (B == 0 || C == 0 || nblk == 0) return kOk;
  char* const planes = (char*)ws;
  int32_t* const wide = (int32_t*)(planes + (int64_t)B * nt * kBmTileBytes);
  blockmax_split_kernel<<<dim3(nt, B), 256, 0, st>>>(k, k_sb, k_st, Sk, nt, planes, wide);
  // scores leave in 64-byte or longer pieces with 1,024 keys
  const int bpc = blocks_per_group(kBmMaxChunk, 256, 512);
  a.planes = planes; a.wide = wide; a.chunk_tiles = bpc * tpb;
  const dim3 grid(rt, (nblk + bpc - 1) / bpc, B);
  if (arg)
    blockmax_mfma_kernel<true><<<grid, 256, 0, st>>>(a);
  else
    blockmax_mfma_kernel<false><<<grid, 256, 0, st>>>(a);
  return bm_status();
}

// Pieces of the backward workspace: mask, then (more than one row range) the ranges' dk and
// their use flags.
static void bm_bwd_layout(int B, int C, int Sk, int nblk, int64_t* mask, int64_t* part,
                          int64_t* used) {
  using namespace dash;
  const int64_t nr = (C + kBmRange - 1) / kBmRange;
  *mask = ((int64_t)B * ((nblk + 63) / 64) * C * 8 + 15) / 16 * 16;
  *part = nr > 1 ? nr * B * Sk * 128 * 4 : 0;
  *used = nr > 1 ? nr * B * nblk * 4 : 0;
}

extern "C" int dash_block_max_backward_workspace_size(int B, int C, int Sk, int nblk,
                                                      int64_t* bytes) {
  using namespace dash;
  if (!bytes || B < 0 || C < 0 || Sk < 0 || nblk < 0) return kErrInvalid;
  int64_t m, p, u;
  bm_bwd_layout(B, C, Sk, nblk, &m, &p, &u);
  *bytes = m + p + u;
  return kOk;
}

extern "C" int dash_block_max_backward(const float* q, int64_t q_sb, int64_t q_st, int C,
                                       const int32_t* pos, int64_t ps_sb, const float* k,
                                       int64_t k_sb, int64_t k_st, int Sk, int B, int d,
                                       int block_size, int local_window, int nblk,
                                       const uint8_t* arg, const float* g, int64_t g_sb,
                                       int64_t g_sc, float* dq, float* dk, void* ws,
                                       int64_t ws_bytes, void* stream) {
  using namespace dash;
  if (!q || !pos || !k || !arg || !g || !dq || !dk || !ws || B < 0 || C < 0 || nblk < 0 || Sk < 0)
    return kErrInvalid;
  if (!bm_supported(d, block_size) || !bm_rows_ok(q, q_sb, q_st) || !bm_rows_ok(k, k_sb, k_st) ||
      (uintptr_t)ws % 16 != 0 || (uintptr_t)dq % 16 != 0 || (uintptr_t)dk % 16 != 0 || B > 65535)
    return kErrUnsupported;
  // every key belongs to a block (the rows of other keys would stay unwritten)
  if ((int64_t)nblk * block_size < Sk || (int64_t)(nblk - 1) * block_size >= Sk) return kErrUnsupported;
  int64_t mb, pb, ub;
  bm_bwd_layout(B, C, Sk, nblk, &mb, &pb, &ub);
  if (ws_bytes < mb + pb + ub) return kErrWorkspace;
  if (B == 0 || C == 0 || nblk == 0) return kOk;
  const int nr = (C + kBmRange - 1) / kBmRange;
  BlockMaxBwdArgs a{q, q_sb, q_st, k, k_sb, k_st, pos, ps_sb, arg, g, g_sb, g_sc, dq, dk, B, C, Sk,
                    block_size, std::max(1, local_window), nblk, (nblk + 63) / 64, (uint64_t*)ws, nr,
                    (float*)((char*)ws + mb), (int32_t*)((char*)ws + mb + pb)};
  hipStream_t st = (hipStream_t)stream;
  blockmax_bwd_q_kernel<<<dim3((C + 3) / 4, B), 256, 0, st>>>(a);
  const dim3 grid(nblk, nr, B);
  const size_t per_wave = (size_t)block_size * 128 * 4;
  if (block_size <= 32)                    // 64 KB of sums: two work-groups per CU
    blockmax_bwd_k_kernel<4><<<grid, 256, 4 * per_wave, st>>>(a);
  else if (block_size <= 64)
    blockmax_bwd_k_kernel<2><<<grid, 128, 2 * per_wave, st>>>(a);
  else
    blockmax_bwd_k_kernel<1><<<grid, 64, per_wave, st>>>(a);
  if (nr > 1)
    blockmax_bwd_sum_kernel<<<dim3((unsigned)(((int64_t)B * Sk * 32 + 255) / 256)), 256, 0, st>>>(a);
  return bm_status();
}
