// Extend attention over a paged cache: the query rows of request b are the positions
// ctx[b] + t of a cached sequence of klen[b] keys (unlimited_ocr_v2_backend.py:1302-1335),
// each attending its window and its routed blocks like a decode query.  Included by
// dash_prefill.hip, whose plan, scan and scatter kernels it uses.
//
//   plan, scan, scatter      every routed (row, slot) pair grouped by key block, chunks of
//                            256 pairs (no dense blocks)
//   extend_routed_kernel     one work-group per chunk and head: the block's K and V in LDS,
//                            32 gathered queries per wavefront and round
//   extend_window_kernel     128 rows of one request and head over their window band
//   extend_merge_kernel      per (row, head) the window's and the slots' partials
//
// One query at a time (dash_attn_decode) every key row comes from the L2 once per query and
// the products run on the vector units: 6,816 us for 5,021 rows of 10 heads, window 512, 16
// routed blocks of 64.  Grouped by block a key row is read once per 256 pairs and the
// products run on the matrix cores, 380 us with the plan; what bounds it now is the traffic
// of the pairs' partials (512 B written and read per pair and head).
//
// Precision is that of the decode kernels: fp32 scores, weights, sums and partials.  A
// weight enters the bf16 matrix product as three bf16 parts (24 significand bits), so it
// is not rounded.  A row's result does not depend on the rows it shares a tile or chunk
// with: window items start at multiples of 64 keys, a pair's partial involves its own block
// only, and the partials are added in slot order.  Masked keys add exact zeros where V is
// finite; the window kernel gives a V value that is not to the rows that see its key, and a
// routed block's reach the rows that name the block, as in the row-by-row kernels.
#pragma once

namespace dash {

struct ExtendArgs {
  PrefillArgs p;               // k_st / v_st: token strides within a page; k_sb / v_sb unused
  const int32_t* table; int64_t table_stride;   // pages of one block
  int64_t k_sp, v_sp;          // page strides
  int64_t T;                   // query rows
  float* part_o;               // [T, H, K, 128] routed partials, not normalised
  float2* part_ml;             // [T, H, K] base-2 reference and weight sum
  float* win_o;                // [T, H, 128] window partials
  float2* win_ml;              // [T, H]
  void* out; int out_bf16; int64_t o_st, o_sh;
};

// The three bf16 parts of eight weights (round to nearest; their sum is the fp32 value).
__device__ __forceinline__ void ext_split3(const float (&x)[8], bf16x8& h, bf16x8& m, bf16x8& l) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bf16 a = (bf16)x[e];
    const float r = x[e] - (float)a;
    const bf16 b = (bf16)r;
    h[e] = a;
    m[e] = b;
    l[e] = (bf16)(r - (float)b);
  }
}

// acc_o[dt] += V^T P^T over keys kbase .. kbase+15 of a swizzled V stage (see pv_at), P in
// three parts, smallest first.
__device__ __forceinline__ void ext_pv(const bf16* sVs, uint32_t vl, int kbase, const bf16x8& ph,
                                       const bf16x8& pm, const bf16x8& pl, floatx16 (&acc_o)[4]) {
  bf16x8 vop[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
    const char* p = (const char*)sVs + kbase * 256 + (vl ^ (uint32_t)(dt << 6));
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_short4*)(__attribute__((address_space(3))) void*)p);
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_short4*)(__attribute__((address_space(3))) void*)(p + 2048));
    const bf16x4 l4 = __builtin_bit_cast(bf16x4, lo);
    const bf16x4 h4 = __builtin_bit_cast(bf16x4, hi);
#pragma unroll
    for (int e = 0; e < 4; ++e) { vop[dt][e] = l4[e]; vop[dt][e + 4] = h4[e]; }
  }
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vop[dt], pl, acc_o[dt], 0, 0, 0);
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vop[dt], pm, acc_o[dt], 0, 0, 0);
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vop[dt], ph, acc_o[dt], 0, 0, 0);
}

// acc_o[dt] += V^T P^T over the 64 keys of a swizzled V stage, P in three parts.  The item's
// products sum from zero, smallest parts first, before they meet the row's total: 12 roundings
// at the item's size and one at the total's, instead of 12 at the total's.
__device__ __forceinline__ void ext_pv_item(const bf16* sVs, uint32_t vl, const bf16x8 (&ph)[4],
                                            const bf16x8 (&pm)[4], const bf16x8 (&pl)[4],
                                            floatx16 (&acc_o)[4]) {
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
    bf16x8 vop[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const char* p = (const char*)sVs + ks * 16 * 256 + (vl ^ (uint32_t)(dt << 6));
      const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_short4*)(__attribute__((address_space(3))) void*)p);
      const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_short4*)(__attribute__((address_space(3))) void*)(p + 2048));
      const bf16x4 l4 = __builtin_bit_cast(bf16x4, lo);
      const bf16x4 h4 = __builtin_bit_cast(bf16x4, hi);
#pragma unroll
      for (int e = 0; e < 4; ++e) { vop[ks][e] = l4[e]; vop[ks][e + 4] = h4[e]; }
    }
    floatx16 t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vop[ks], pl[ks], t, 0, 0, 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vop[ks], pm[ks], t, 0, 0, 0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vop[ks], ph[ks], t, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_o[dt][r] += t[r];
  }
}

// Direct loads of keys j0 .. j0+63 (j0 a multiple of 32, j0 < klen) of one head into a
// swizzled stage by 4 wavefronts: row 16 u + 4 wv + lane / 16.  Rows past the last key
// repeat it, so that no unused row of the cache is read; the 16 rows of a group lie in one
// page (blocks are 32 keys or multiples of 64).  SWZ: 0 the K swizzle, 1 the V swizzle.
template <int SWZ>
__device__ __forceinline__ void ext_fetch(bf16* sX, const bf16* xb, const int32_t* tr, int64_t x_sp,
                                          int64_t x_st, int bs, int j0, int klen, int wv, int lane) {
  const int r0 = 4 * wv + (lane >> 4);
  const int slot = SWZ ? v_slot(r0, lane & 15) : k_slot(r0, lane & 15);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int blk = min(j0 + 16 * u, klen - 1) / bs;
    const int row = min(j0 + 16 * u + r0, klen - 1) - blk * bs;
    const bf16* src = xb + (int64_t)tr[blk] * x_sp + (int64_t)row * x_st + slot * 8;
    __builtin_amdgcn_global_load_lds((const void*)src,
                                     (__attribute__((address_space(3))) void*)(sX + (4 * u + wv) * 4 * 128),
                                     16, 0, 0);
  }
}

// V values that are not finite would reach every row of an item through its products with
// masked weights.  In a stage, just landed, each wavefront clears them in the rows it loaded
// and returns the mask of the keys that hold any (its bit 4 u + i: row 16 u + 4 wv + i).
__device__ __forceinline__ uint32_t ext_clear_rows(bf16* sX, int wv, int lane) {
  uint32_t keys = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    uint4* p = (uint4*)(sX + (4 * u + wv) * 4 * 128) + lane;
    uint4 x = *p;
    bool bad = false;
    auto fix = [&](uint32_t& w) {
      if ((w & 0x7f80u) == 0x7f80u) { w &= 0xffff0000u; bad = true; }
      if ((w & 0x7f800000u) == 0x7f800000u) { w &= 0xffffu; bad = true; }
    };
    fix(x.x); fix(x.y); fix(x.z); fix(x.w);
    if (bad) *p = x;
    const uint64_t m = __ballot(bad);
#pragma unroll
    for (int i = 0; i < 4; ++i) keys |= ((m >> (16 * i)) & 0xffffu) ? 1u << (4 * u + i) : 0u;
  }
  return keys;
}

// Bound by the matrix cores' chain per item (16 products of S^T, 48 of the three-part
// P V) against the softmax's VALU work of the same 64 keys; K and V of the next item are
// fetched meanwhile, two work-groups per CU.  Where a work-group's result is not finite it
// walks its band again, an item at a time, with V's finite values in the products, and adds
// the others to the rows that see them.
__global__ __launch_bounds__(256, 2) void extend_window_kernel(ExtendArgs a) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) bf16 sK0[64 * D];
  __shared__ __attribute__((aligned(16))) bf16 sK1[64 * D];
  __shared__ __attribute__((aligned(16))) bf16 sV0[64 * D];
  __shared__ __attribute__((aligned(16))) bf16 sV1[64 * D];
  __shared__ uint32_t sBad[4];             // keys of an item with values that are not finite
  const PrefillArgs& p = a.p;
  const int lid = xcd_logical_id(blockIdx.x, gridDim.x);
  const int g = lid % p.ntv, h = lid / p.ntv;
  if (g >= p.tile_pref[p.B]) return;
  const int b = p.tile_doc[g];
  const int t0 = (g - p.tile_pref[b]) * kPfTQ;
  const int len = seq_len(p, b), klen = key_len(p, b);
  const int tid = threadIdx.x, lane = wave_lane(), wv = tid / kWave;
  const int hl = lane >> 5, n = lane & 31;
  const int64_t r0 = row0(p, b);
  const int tq = t0 + wv * 32 + n;
  const bool qvalid = tq < len;
  const int tqc = min(tq, len - 1);
  const bf16* qb = p.q + (r0 + tqc) * p.q_st + (int64_t)h * p.q_sh;
  bf16x8 qop[D / 16];
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) qop[kk] = *(const bf16x8*)(qb + kk * 16 + hl * 8);

  const int qp = q_pos_of(p, b, tqc, klen);
  // first window key; a row at no position sees none
  const int q_lo = qp >= 0 ? max(qp - p.lw + 1, 0) : 0x40000000;
  const int qfirst = q_pos_of(p, b, t0, klen);
  const int qlast = q_pos_of(p, b, min(t0 + kPfTQ - 1, len - 1), klen);
  const int j_first = max(qfirst - p.lw + 1, 0) / 64 * 64;
  const int n_items = qlast >= 0 ? qlast / 64 - j_first / 64 + 1 : 0;

  floatx16 acc_o[D / 32];
  float m_run, l_run;
  auto reset = [&] {
    m_run = -INFINITY;
    l_run = 0.f;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc_o[dt][r] = 0.f;
  };
  const int32_t* tr = a.table + (int64_t)b * a.table_stride;
  const bf16* kb = p.k + (int64_t)h * p.k_sh;
  const bf16* vb = p.v + (int64_t)h * p.v_sh;
  const uint32_t kl0 = k_lane_off(n, hl), vl0 = v_lane_off(lane);
  const float csc = p.scale_log2e;

  // the item of keys j0 .. j0 + 63 in stage pair P
  auto item = [&](int j0, auto par) __attribute__((always_inline)) {
    constexpr int P = decltype(par)::value;
    bf16* const sKc = P == 0 ? sK0 : sK1;
    bf16* const sVc = P == 0 ? sV0 : sV1;
    if (!__any(qvalid && q_lo <= j0 + 63 && qp >= j0)) return;
    uint32_t kl = kl0, vl = vl0;
    asm volatile("" : "+v"(kl), "+v"(vl));
    floatx16 s[2];
    float mraw = -INFINITY;
    const int kq = j0 + 4 * hl - q_lo;
    const uint32_t span = qp >= 0 ? (uint32_t)(qp - q_lo) : 0u;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[hf][r] = 0.f;
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk)
        s[hf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_frag_at(sKc, kl, hf, kk), qop[kk], s[hf],
                                                        0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t d = (uint32_t)(kq + 32 * hf + 8 * (r >> 2) + (r & 3));
        s[hf][r] = d <= span ? s[hf][r] : -INFINITY;
        mraw = fmaxf(mraw, s[hf][r]);
      }
    }
    // the reference moves only when a row's maximum exceeds it by more than 8
    const float mloc = xor32_max(mraw * csc);
    const bool up = mloc > m_run + 8.f;
    if (__any(up)) {
      const float alpha = up ? fast_exp2(m_run - mloc) : 1.f;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc_o[dt][r] *= alpha;
      m_run = up ? mloc : m_run;
    }
    const float off = m_run == -INFINITY ? 0.f : -m_run;
    bf16x8 ph[4], pm[4], pl[4];
    float l_item = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = fast_exp2(fmaf(s[ks >> 1][8 * (ks & 1) + e], csc, off));
      l_item += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
      ext_split3(x, ph[ks], pm[ks], pl[ks]);
    }
    l_run += l_item;
    ext_pv_item(sVc, vl, ph, pm, pl, acc_o);
  };
  auto step = [&](int it, auto par) __attribute__((always_inline)) {
    constexpr int P = decltype(par)::value;
    bf16* const sKn = P == 0 ? sK1 : sK0;
    bf16* const sVn = P == 0 ? sV1 : sV0;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();                       // item it landed; every wavefront left it - 1
    const int j0 = j_first + it * 64;
    if (it + 1 < n_items) {
      ext_fetch<0>(sKn, kb, tr, a.k_sp, p.k_st, p.bs, j0 + 64, klen, wv, lane);
      ext_fetch<1>(sVn, vb, tr, a.v_sp, p.v_st, p.bs, j0 + 64, klen, wv, lane);
    }
    item(j0, par);
  };
  reset();
  if (n_items > 0) {
    ext_fetch<0>(sK0, kb, tr, a.k_sp, p.k_st, p.bs, j_first, klen, wv, lane);
    ext_fetch<1>(sV0, vb, tr, a.v_sp, p.v_st, p.bs, j_first, klen, wv, lane);
  }
  for (int it = 0; it < n_items; it += 2) {
    step(it, std::integral_constant<int, 0>{});
    if (it + 1 < n_items) step(it + 1, std::integral_constant<int, 1>{});
  }
  float z = 0.f;                           // NaN where a value is not finite
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) z = fmaf(acc_o[dt][r], 0.f, z);
  if (__syncthreads_or(z != 0.f)) {
    reset();
    for (int it = 0; it < n_items; ++it) {
      const int j0 = j_first + it * 64;
      __syncthreads();                     // every wavefront left the stages
      ext_fetch<0>(sK0, kb, tr, a.k_sp, p.k_st, p.bs, j0, klen, wv, lane);
      ext_fetch<1>(sV0, vb, tr, a.v_sp, p.v_st, p.bs, j0, klen, wv, lane);
      __builtin_amdgcn_s_waitcnt(0);
      const uint32_t bad = ext_clear_rows(sV0, wv, lane);
      if (lane == 0) sBad[wv] = bad;
      __syncthreads();
      item(j0, std::integral_constant<int, 0>{});
      for (int w = 0; w < 4; ++w)
        for (uint32_t todo = sBad[w]; todo; todo &= todo - 1) {
          const int i = __builtin_ctz(todo), key = j0 + 16 * (i >> 2) + 4 * w + (i & 3);
          if (key >= klen) continue;       // a repeated row
          const bool sees = key >= q_lo && key <= qp;
          const int blk = key / p.bs;
          const bf16* vr = vb + (int64_t)tr[blk] * a.v_sp + (int64_t)(key - blk * p.bs) * p.v_st + 4 * hl;
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const bf16x4 x = *(const bf16x4*)(vr + 32 * dt + 8 * q);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float f = (float)x[e];
                if (sees && !(fabsf(f) <= 3.402823466e38f)) acc_o[dt][4 * q + e] += f;
              }
            }
        }
    }
  }
  const float l_tot = xor32_sum(l_run);
  if (qvalid) {
    const int64_t row = (r0 + tq) * p.H + h;
    float* wo = a.win_o + row * D + 4 * hl;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(float4*)(wo + dt * 32 + 8 * q) = make_float4(acc_o[dt][4 * q], acc_o[dt][4 * q + 1],
                                                       acc_o[dt][4 * q + 2], acc_o[dt][4 * q + 3]);
    if (hl == 0) a.win_ml[row] = make_float2(m_run, l_tot);
  }
}

// Bound by the partials it writes (512 B per pair and head; 411 MB in 192 us at 5,021 rows,
// 16 slots, 10 heads).  A pair's partial goes to its place in [row, head, slot] order, so
// that the merge reads a row's slots in one piece: rows are 512 B, whole lines wherever they
// lie.  They leave through LDS, eight rows at a time, two rows per store instruction.  Eight
// wavefronts of one round of 32 pairs in 128 registers (four wavefronts of two rounds, which
// hold both rounds' queries, took 196 registers and 233 us).
__global__ __launch_bounds__(512, 4) void extend_routed_kernel(ExtendArgs a) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) bf16 sKs[kPfIT * D];
  __shared__ __attribute__((aligned(16))) bf16 sVs[kPfIT * D];
  __shared__ __attribute__((aligned(16))) bf16 sTr[8 * 16 * D];   // 4 KB per wavefront
  const PrefillArgs& p = a.p;
  // real chunks first, as prefill_sparse_kernel maps its grid
  const int nreal = p.H * p.chunk_pref[p.B];
  if ((int)blockIdx.x >= nreal) return;
  const int lid = xcd_logical_id(blockIdx.x, nreal);
  int b = 0;
  {
    int hi = p.B;
    while (hi - b > 1) {
      const int mid = (b + hi) >> 1;
      if (p.H * p.chunk_pref[mid] <= lid) b = mid; else hi = mid;
    }
  }
  const int pb = p.chunk_pref[b], nc = p.chunk_pref[b + 1] - pb;
  const int hc = lid - p.H * pb;
  const int h = hc / nc, ch = hc % nc;
  const int tid = threadIdx.x, lane = wave_lane(), wv = tid / kWave;
  const int hl = lane >> 5, n = lane & 31;
  const int32_t* rec = p.chunk_rec + ((int64_t)b * p.chunk_cap + ch) * kRec;
  const int c = rec[0], npairs = rec[1];
  const int pid_first = rec[kRecHead];
  const int pid_raw = rec[kRecHead + wv * 32 + n];
  const int len = seq_len(p, b), klen = key_len(p, b);
  const int64_t r0 = row0(p, b);
  const int32_t* tr = a.table + (int64_t)b * a.table_stride;
  const int kfirst = c * p.bs;
  {
    // wavefronts 0-3 load K, 4-7 V
    const int kend = min(klen, kfirst + p.bs);
    if (wv < 4)
      ext_fetch<0>(sKs, p.k + (int64_t)h * p.k_sh, tr, a.k_sp, p.k_st, p.bs, kfirst, kend, wv, lane);
    else
      ext_fetch<1>(sVs, p.v + (int64_t)h * p.v_sh, tr, a.v_sp, p.v_st, p.bs, kfirst, kend, wv - 4, lane);
  }
  // this wavefront's 32 pairs; lanes past the count repeat the chunk's first pair
  const bool active = wv * 32 + n < npairs;
  const int pid = min(max(active ? pid_raw : pid_first, 0), len * p.K - 1);
  const int t = pid / p.K;
  const bf16* qb = p.q + r0 * p.q_st + (int64_t)h * p.q_sh;
  bf16x8 qrow[D / 16];
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const int tk = __shfl(t, 4 * kk + (lane >> 4), kWave);
    qrow[kk] = *(const bf16x8*)(qb + (int64_t)tk * p.q_st + (lane & 15) * 8);
  }
  const float bl = p.bias[r0 * p.K + pid] * 1.4426950408889634f;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (wv * 32 >= npairs) return;           // no barrier from here on

  bf16* const st = sTr + wv * 16 * D;
  const uint32_t kl0 = k_lane_off(n, hl), vl0 = v_lane_off(lane);
  const float csc = p.scale_log2e;
  bf16x8 qop[D / 16];
#pragma unroll
  for (int piece = 0; piece < 2; ++piece) {
#pragma unroll
    for (int kk = 4 * piece; kk < 4 * piece + 4; ++kk) {
      const int rr = 4 * (kk - 4 * piece) + (lane >> 4);
      *(bf16x8*)(st + (rr * 16 + ((lane & 15) ^ rr)) * 8) = qrow[kk];
    }
    wave_lds_sync();
    if ((n >> 4) == piece) {
      const int rr = n & 15;
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk)
        qop[kk] = *(const bf16x8*)(st + (rr * 16 + ((2 * kk + hl) ^ rr)) * 8);
    }
    wave_lds_sync();
  }
  // keys below the window of this pair's query
  const int hi = min(q_pos_of(p, b, t, klen) - p.lw + 1, min(klen, kfirst + p.bs)) - 1;
  const int last = active ? hi - kfirst - 4 * hl : -1;
  floatx16 s[2];
  float mraw = -INFINITY;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s[hf][r] = 0.f;
    if (32 * hf >= p.bs) continue;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
      s[hf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_frag_at(sKs, kl0, hf, kk), qop[kk], s[hf],
                                                      0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[hf][r] = 32 * hf + 8 * (r >> 2) + (r & 3) <= last ? s[hf][r] : -INFINITY;
      mraw = fmaxf(mraw, s[hf][r]);
    }
  }
  const float m = xor32_max(fmaf(mraw, csc, bl));
  const float off = bl - (m == -INFINITY ? 0.f : m);
  floatx16 acc_o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_o[dt][r] = 0.f;
  float lsum = 0.f;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    if (32 * hf >= p.bs) continue;
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[e] = fast_exp2(fmaf(s[hf][8 * jj + e], csc, off));
        lsum += x[e];
      }
      bf16x8 ph, pm, pl;
      ext_split3(x, ph, pm, pl);
      ext_pv(sVs, vl0, 32 * hf + 16 * jj, ph, pm, pl, acc_o);
    }
  }
  const float l_tot = xor32_sum(lsum);
  // this pair's partial among the request's: (row, head, slot), in 32 bits
  const int pair = t * p.H * p.K + (pid - t * p.K);
  float* const po = a.part_o + (r0 * p.H + h) * p.K * D;
  if (active && hl == 0) a.part_ml[(r0 * p.H + h) * p.K + pair] = make_float2(m, l_tot);
  // 16-byte chunk c of row r at slot c ^ (r % 8) of its 512 bytes
  float* const stf = (float*)st;
#pragma unroll
  for (int piece = 0; piece < 4; ++piece) {
    if ((n >> 3) == piece) {
      const int rr = n & 7;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(float4*)(stf + rr * D + (((dt * 8 + 2 * q + hl) ^ rr) << 2)) =
              make_float4(acc_o[dt][4 * q], acc_o[dt][4 * q + 1], acc_o[dt][4 * q + 2],
                          acc_o[dt][4 * q + 3]);
    }
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int rr = 2 * k + hl;
      const int src = 8 * piece + rr;      // the pair whose row this half of the wave writes
      const int pw = __shfl(pair, src, kWave);
      if (wv * 32 + src < npairs)
        *(float4*)(po + (int64_t)pw * D + n * 4) = *(const float4*)(stf + rr * D + ((n ^ rr) << 2));
    }
    wave_lds_sync();
  }
}

// One wavefront per (row, head): the window's partial and the row's routed ones (lane s
// holds the weight of slot s), two dims per lane.  Bound by reading the partials, 512 B per
// slot; sixteen slots are in flight at a time.
__global__ __launch_bounds__(256) void extend_merge_kernel(ExtendArgs a) {
  constexpr int D = 128;
  const PrefillArgs& p = a.p;
  const int64_t item = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
  if (item >= a.T * p.H) return;
  const int lane = wave_lane();
  const int64_t row = item / p.H;
  const int h = (int)(item % p.H);
  const bool on = lane < p.K && p.kind[row * p.K + lane] == 2;
  const uint64_t live = __ballot(on);
  const float2 ml = on ? a.part_ml[item * p.K + lane] : make_float2(-INFINITY, 0.f);
  const float2 wm = a.win_ml[item];
  const float2 wo = *(const float2*)(a.win_o + item * D + 2 * lane);
  const float* po = a.part_o + item * p.K * D + 2 * lane;
  const float M = fmaxf(wave_max(ml.x), wm.x);
  const float Mu = M == -INFINITY ? 0.f : M;
  const float w = on ? fast_exp2(ml.x - Mu) : 0.f;
  const float ww = fast_exp2(wm.x - Mu);
  const float L = wave_sum(ml.y * w) + wm.y * ww;
  float2 acc = make_float2(wo.x * ww, wo.y * ww);
  uint64_t todo = live;
  while (todo) {
    float2 x[16];
    float u[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int s = todo ? __builtin_ctzll(todo) : 0;
      u[i] = todo ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), s)) : 0.f;
      x[i] = make_float2(0.f, 0.f);
      if (todo) x[i] = *(const float2*)(po + s * D);
      todo &= todo - 1;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      acc.x = fmaf(u[i], x[i].x, acc.x);
      acc.y = fmaf(u[i], x[i].y, acc.y);
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const int64_t off = row * a.o_st + (int64_t)h * a.o_sh + 2 * lane;
  if (a.out_bf16) {
    bf16x2 r;
    r[0] = (bf16)(acc.x * inv);
    r[1] = (bf16)(acc.y * inv);
    *(bf16x2*)((bf16*)a.out + off) = r;
  } else {
    *(float2*)((float*)a.out + off) = make_float2(acc.x * inv, acc.y * inv);
  }
}

// Workspace pieces (256-byte aligned): the block counters, arrival and error words and the
// slot kinds (cleared together), the plan, the partials.
struct ExtendLayout {
  int64_t count, done, err, kind, clear_end, tbase, bch, nchunks, cpref, rec, tpref, tdoc, po, pml,
      wo, wml, total;
  int chunk_cap, ntiles_cap, ntv;
};

inline ExtendLayout extend_layout(int B, int H, int S_q, int64_t T, int K, int nblk_cap) {
  constexpr int64_t D = 128;
  ExtendLayout L;
  // full chunks, and one partly filled per block that a row names
  L.chunk_cap = (int)((int64_t)S_q * K / kPfCH + std::min<int64_t>(nblk_cap, (int64_t)S_q * K) + 1);
  L.ntiles_cap = (S_q + kPfTQ - 1) / kPfTQ;
  L.ntv = (int)((T + (int64_t)(kPfTQ - 1) * B) / kPfTQ) + 1;
  const int64_t nbc = (int64_t)B * nblk_cap;
  int64_t o = 0;
  auto align = [](int64_t x) { return (x + 255) / 256 * 256; };
  L.count = o; o += nbc * 4;
  L.done = o; o += 4;
  L.err = o; o += 4;
  L.kind = o = (o + 15) / 16 * 16; o += T * K;
  L.clear_end = (o + 3) / 4 * 4; o = align(o);
  L.tbase = o; o = align(o + nbc * L.ntiles_cap * 4);
  L.bch = o; o = align(o + nbc * 4);
  L.nchunks = o; o = align(o + (int64_t)B * 4);
  L.cpref = o; o = align(o + (int64_t)(B + 1) * 4);
  L.rec = o; o = align(o + (int64_t)B * L.chunk_cap * kRec * 4);
  L.tpref = o; o = align(o + (int64_t)(B + 1) * 4);
  L.tdoc = o; o = align(o + (int64_t)L.ntv * 4);
  L.po = o; o = align(o + T * H * K * D * 4);
  L.pml = o; o = align(o + T * H * K * 8);
  L.wo = o; o = align(o + T * H * D * 4);
  L.wml = o; o = align(o + T * H * 8);
  L.total = o;
  return L;
}

}  // namespace dash

extern "C" int dash_attn_extend_workspace_size(int B, int H, int max_query_len, int64_t T, int K,
                                               int nblk, int64_t* bytes) {
  using namespace dash;
  if (!bytes || B < 0 || H <= 0 || max_query_len < 0 || T < 0 || K < 0 || nblk < 0)
    return kErrInvalid;
  *bytes = extend_layout(B, H, max_query_len, T, K, nblk).total;
  return kOk;
}

extern "C" int dash_attn_extend(
    const void* q, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sh, int64_t k_st,
    int64_t k_sp, const void* v, int64_t v_sh, int64_t v_st, int64_t v_sp,
    const int32_t* block_table, int64_t table_stride, const int32_t* seq_lens,
    const int32_t* context_lens, const int32_t* cu_seqlens_q, const int32_t* idx,
    const uint8_t* valid, const float* bias, int K, void* out, int out_bf16, int64_t o_st,
    int64_t o_sh, int B, int H, int64_t T, int max_query_len, int nblk, int D, int block_size,
    int local_window, float scale, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace dash;
  if (!q || !k || !v || !out || !block_table || !seq_lens || !context_lens || !cu_seqlens_q ||
      B < 0 || H <= 0 || T < 0 || max_query_len < 0 || nblk < 0 || K < 0 || local_window < 1)
    return kErrInvalid;
  if (K > 0 && (!idx || !bias)) return kErrInvalid;
  if (D != 128 || (block_size != 32 && block_size != 64) || K > kPfMaxSlots || nblk > kPfMaxBlocks ||
      !(scale > 0.f) || B > 65535)
    return kErrUnsupported;
  const int64_t strides[] = {q_st, q_sh, k_sh, k_st, k_sp, v_sh, v_st, v_sp};
  for (int64_t s : strides)
    if (s % 8 != 0) return kErrUnsupported;
  const void* ptrs[] = {q, k, v};
  for (const void* x : ptrs)
    if ((uintptr_t)x % 16 != 0) return kErrUnsupported;
  if ((uintptr_t)out % 8 != 0 || o_st % 2 != 0 || o_sh % 2 != 0) return kErrUnsupported;
  if (B == 0 || T == 0) return kOk;
  if (max_query_len == 0 || nblk == 0) return kErrInvalid;
  const ExtendLayout L = extend_layout(B, H, max_query_len, T, K, nblk);
  if (!workspace || workspace_bytes < L.total || (uintptr_t)workspace % 256 != 0)
    return kErrWorkspace;
  // grids and row ids in 32 bits
  if (T * H * std::max(K, 1) > INT32_MAX || (int64_t)L.chunk_cap * H * B > INT32_MAX ||
      (int64_t)L.ntv * H > INT32_MAX || (T * H + 3) / 4 > INT32_MAX)
    return kErrUnsupported;
  char* w = (char*)workspace;
  ExtendArgs a = {};
  PrefillArgs& p = a.p;
  p.q = (const bf16*)q; p.k = (const bf16*)k; p.v = (const bf16*)v;
  p.q_st = q_st; p.q_sh = q_sh; p.k_sh = k_sh; p.k_st = k_st; p.v_sh = v_sh; p.v_st = v_st;
  p.idx = idx; p.valid = valid; p.bias = bias; p.K = K;
  p.cu = cu_seqlens_q;
  p.slots_vec = slots_vectorizable(K, idx, valid, bias);
  p.S = max_query_len; p.H = H; p.bs = block_size; p.lw = local_window; p.nblk_cap = nblk; p.B = B;
  p.scale_log2e = scale * 1.4426950408889634f;
  p.ntiles = L.ntiles_cap;
  p.kind = (uint8_t*)(w + L.kind);
  p.dense_threshold = kPfTQ + 1;           // every routed pair block-major
  p.blk_count = (int32_t*)(w + L.count);
  p.tile_base = (int32_t*)(w + L.tbase);
  p.ntiles_cap = L.ntiles_cap;
  p.blk_chunk = (int32_t*)(w + L.bch);
  p.num_chunks = (int32_t*)(w + L.nchunks);
  p.chunk_pref = (int32_t*)(w + L.cpref);
  p.done = (int32_t*)(w + L.done);
  p.err = (int32_t*)(w + L.err);
  p.chunk_rec = (int32_t*)(w + L.rec);
  p.chunk_cap = L.chunk_cap;
  p.spos = nullptr;
  p.ppos = INT64_MAX;
  p.tile_pref = (int32_t*)(w + L.tpref);
  p.tile_doc = (int32_t*)(w + L.tdoc);
  p.ntv = L.ntv;
  p.ctx = context_lens; p.klen = seq_lens; p.key_cap = nblk * block_size;
  a.table = block_table; a.table_stride = table_stride;
  a.k_sp = k_sp; a.v_sp = v_sp; a.T = T;
  a.part_o = (float*)(w + L.po); a.part_ml = (float2*)(w + L.pml);
  a.win_o = (float*)(w + L.wo); a.win_ml = (float2*)(w + L.wml);
  a.out = out; a.out_bf16 = out_bf16; a.o_st = o_st; a.o_sh = o_sh;
  hipStream_t st = (hipStream_t)stream;
  const int nclear = (int)((L.clear_end - L.count) / 4);
  hipLaunchKernelGGL(prefill_clear_kernel, dim3((nclear + 255) / 256), dim3(256), 0, st, p.blk_count,
                     nclear);
  if (K > 0) launch_plan(p, L.ntiles_cap, st);
  hipLaunchKernelGGL(prefill_scan_kernel, dim3(B), dim3(1024), 0, st, p);
  if (K > 0) {
    hipLaunchKernelGGL(prefill_scatter_kernel, dim3(L.ntiles_cap, B), dim3(kPfTQ), 0, st, p);
    hipLaunchKernelGGL(extend_routed_kernel, dim3(L.chunk_cap * H * B), dim3(512), 0, st, a);
  }
  hipLaunchKernelGGL(extend_window_kernel, dim3(L.ntv * H), dim3(256), 0, st, a);
  hipLaunchKernelGGL(extend_merge_kernel, dim3((unsigned)((T * H + 3) / 4)), dim3(256), 0, st, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? kOk : (int)e;
}
