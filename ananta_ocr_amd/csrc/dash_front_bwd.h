// Gradients of the training router front end (included by dash_prefill.hip, whose stage
// helpers it uses): index q/k projections p = hs W^T of bf16 hidden states with nan_to_num,
// Gemma RMSNorm, RoPE and the finiteness guards (dash_attention.py:680-700, 808-821).
//
//   front_bwd_rows_kernel    d idx_q, d idx_k -> d p (bf16) and the norm weights' gradients
//   front_bwd_w_kernel       d W = d p^T hs over a range of rows
//   front_bwd_sum_kernel     the ranges' shares of d W and of the norm weights
//   front_bwd_h_kernel       d hs = d p W, zero where hs is not finite
//
// As tensor ops the front end's forward and backward took some 70 launches and 1.5 ms of a
// 27,300-token training step (hidden 1,280), two thirds of it elementwise passes over the
// hidden states and weight-gradient products on 34 work-groups.
#pragma once

namespace dash {

constexpr int kFbD = 128;                 // index dim
constexpr int kFbRows = 64;               // rows of a d W step
constexpr int kFbCols = 128;              // hidden columns of a work-group's tile

struct FrontBwdArgs {
  const bf16* proj;            // [T, 256] projections, q then k, as the linear layers give them
  const float* gq; const float* gk;   // [T, 128]
  const float* nq; const float* nk;   // norm weights
  const void* cos; const void* sin; int cs_bf16; int64_t cs_sb, cs_st;
  int64_t T; int S, hid;
  float eps;
  const bf16* hs; int64_t hs_st;      // [T, hid]
  const bf16* wq; const bf16* wk;     // [128, hid]
  bf16* dproj;                 // [T, 256]
  float* npart; int nwg;       // [nwg, 256] norm weight shares
  float* wpart; int nrange, range;    // [nrange, 256, hid]; rows per range
  bf16* dwq; bf16* dwk;        // [128, hid], or null
  float* dnq; float* dnk;      // [128]
  bf16* dhs;                   // [T, hid], or null
};

__device__ __forceinline__ bool fb_finite(float x) { return fabsf(x) <= 3.402823466e38f; }
// non-finite -> 0, clamped (dash_attention.py:607-613)
__device__ __forceinline__ float fb_grad(float g) {
  return fb_finite(g) ? fminf(fmaxf(g, -kGradClamp), kGradClamp) : 0.f;
}
// nan_to_num(nan/inf -> 0) of the two bf16 halves of a word
__device__ __forceinline__ uint32_t fb_sanitize2(uint32_t x) {
  const uint32_t l = ((x & 0x7f80u) == 0x7f80u) ? 0u : (x & 0xffffu);
  const uint32_t h = ((x & 0x7f800000u) == 0x7f800000u) ? 0u : (x & 0xffff0000u);
  return l | h;
}

// One wavefront per (row, side), lane l dims 2 l and 2 l + 1, as router_qk_kernel; the
// forward's intermediate values are formed again from the projection.  A wavefront walks
// many rows of one side and keeps its share of the norm weight's gradient in registers.
// Bound by its 1.5 KB a row.
__global__ __launch_bounds__(256) void front_bwd_rows_kernel(FrontBwdArgs a) {
  __shared__ float2 sW[4][kWave];
  const int lane = wave_lane(), wv = threadIdx.x / kWave, i0 = 2 * lane;
  const int side = wv & 1;
  const float2 nw = *(const float2*)((side ? a.nk : a.nq) + i0);
  const float w0 = 1.0f + nw.x, w1 = 1.0f + nw.y;
  const float* gp = side ? a.gk : a.gq;
  float2 dw = make_float2(0.f, 0.f);
  for (int64_t row = (int64_t)blockIdx.x * 2 + (wv >> 1); row < a.T; row += (int64_t)gridDim.x * 2) {
    const bf16x2 pv = *(const bf16x2*)(a.proj + row * 256 + side * kFbD + i0);
    const float2 gv = *(const float2*)(gp + row * kFbD + i0);
    const float p0 = (float)pv[0], p1 = (float)pv[1];
    const float x0 = fb_finite(p0) ? p0 : 0.f, x1 = fb_finite(p1) ? p1 : 0.f;
    const float r = rsqrtf(wave_sum(x0 * x0 + x1 * x1) * (1.0f / kFbD) + a.eps);
    const float a0 = x0 * r, a1 = x1 * r;
    const float c0 = fminf(fmaxf(a0, -kActClamp), kActClamp), c1 = fminf(fmaxf(a1, -kActClamp), kActClamp);
    const float b0 = c0 * w0, b1 = c1 * w1;
    float g0 = fb_grad(gv.x), g1 = fb_grad(gv.y);
    if (a.cos) {
      const int64_t o = (row / a.S) * a.cs_sb + (row % a.S) * a.cs_st + i0;
      float co0, co1, si0, si1;
      if (a.cs_bf16) {
        const bf16x2 cv = *(const bf16x2*)((const bf16*)a.cos + o);
        const bf16x2 sv = *(const bf16x2*)((const bf16*)a.sin + o);
        co0 = (float)cv[0]; co1 = (float)cv[1]; si0 = (float)sv[0]; si1 = (float)sv[1];
      } else {
        const float2 cv = *(const float2*)((const float*)a.cos + o);
        const float2 sv = *(const float2*)((const float*)a.sin + o);
        co0 = cv.x; co1 = cv.y; si0 = sv.x; si1 = sv.y;
      }
      // out_i = y_i cos_i + h_i sin_i with h_i = -y_{i+64} (i < 64) or y_{i-64}; no
      // gradient where the output is not finite (only cos or sin can make it so)
      const float y0 = fminf(fmaxf(b0, -kActClamp), kActClamp), y1 = fminf(fmaxf(b1, -kActClamp), kActClamp);
      const float q0 = __shfl_xor(y0, 32, kWave), q1 = __shfl_xor(y1, 32, kWave);
      const float sg = lane < 32 ? -1.f : 1.f;
      if (!fb_finite(y0 * co0 + sg * q0 * si0)) g0 = 0.f;
      if (!fb_finite(y1 * co1 + sg * q1 * si1)) g1 = 0.f;
      const float t0 = __shfl_xor(g0 * si0, 32, kWave), t1 = __shfl_xor(g1 * si1, 32, kWave);
      g0 = g0 * co0 - sg * t0;
      g1 = g1 * co1 - sg * t1;
    }
    if (fabsf(b0) > kActClamp) g0 = 0.f;
    if (fabsf(b1) > kActClamp) g1 = 0.f;
    dw.x = fmaf(g0, c0, dw.x);
    dw.y = fmaf(g1, c1, dw.y);
    float d0 = fabsf(a0) > kActClamp ? 0.f : g0 * w0, d1 = fabsf(a1) > kActClamp ? 0.f : g1 * w1;
    const float dot = wave_sum(d0 * x0 + d1 * x1) * (1.0f / kFbD) * r * r;
    d0 = r * (d0 - x0 * dot);
    d1 = r * (d1 - x1 * dot);
    bf16x2 out;
    out[0] = (bf16)(fb_finite(p0) ? d0 : 0.f);
    out[1] = (bf16)(fb_finite(p1) ? d1 : 0.f);
    *(bf16x2*)(a.dproj + row * 256 + side * kFbD + i0) = out;
  }
  sW[wv][lane] = dw;
  __syncthreads();
  if (wv < 2) {
    const float2 o = sW[wv + 2][lane];
    *(float2*)(a.npart + (int64_t)blockIdx.x * 256 + side * kFbD + i0) = make_float2(dw.x + o.x, dw.y + o.y);
  }
}

// d W tile of a row range: 256 dims x 128 hidden columns, 64 rows a step.  Both operands run
// over the rows, so both are read from row-major stages by transposing reads: d p straight
// into LDS, hs through registers, where it loses its non-finite values and the rows past the
// end.  Wavefront w owns dims 64 w .. + 63.  Bound by its reads of d p (every column tile
// reads all of it, from the L2) and of hs; two to three work-groups per CU.
__global__ __launch_bounds__(256, 2) void front_bwd_w_kernel(FrontBwdArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 sA[2][kFbRows * 128];
  __shared__ __attribute__((aligned(16))) bf16 sB[kFbRows * 128];
  const int tid = threadIdx.x, lane = wave_lane(), wv = tid / kWave;
  const int col0 = blockIdx.x * kFbCols;
  const int64_t t_lo = (int64_t)blockIdx.y * a.range, t_hi = min(t_lo + a.range, a.T);
  floatx16 acc[2][4];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[m][n][i] = 0.f;
  // hs: thread's 16-byte chunk of rows r + 16 u
  const int hr = tid >> 4, hc = tid & 15;
  uint4 hv[4];
  auto load_h = [&](int64_t t0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t t = t0 + hr + 16 * u;
      hv[u] = make_uint4(0u, 0u, 0u, 0u);
      if (t < t_hi) hv[u] = *(const uint4*)(a.hs + t * a.hs_st + col0 + hc * 8);
    }
  };
  load_h(t_lo);
  for (int64_t t0 = t_lo; t0 < t_hi; t0 += kFbRows) {
    __syncthreads();                       // every wavefront is done with the stages
#pragma unroll
    for (int s = 0; s < 2; ++s)
      stage_rows(sA[s], wv, lane, [&](int r) { return a.dproj + min(t0 + r, a.T - 1) * 256 + s * kFbD; });
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = hr + 16 * u;
      const uint4 v = make_uint4(fb_sanitize2(hv[u].x), fb_sanitize2(hv[u].y), fb_sanitize2(hv[u].z),
                                 fb_sanitize2(hv[u].w));
      *(uint4*)(sB + r * 128 + (hc ^ bw_swz(r & 15)) * 8) = v;
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t0 + kFbRows < t_hi) load_h(t0 + kFbRows);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      bf16x8 fa[2], fb[4];
#pragma unroll
      for (int m = 0; m < 2; ++m) fa[m] = tr_frag_k(sA[wv >> 1], 16 * ks, 2 * (wv & 1) + m, lane);
#pragma unroll
      for (int n = 0; n < 4; ++n) fb[n] = tr_frag_k(sB, 16 * ks, n, lane);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[m], fb[n], acc[m][n], 0, 0, 0);
    }
  }
  // lane = hidden column, register i: dim 8 (i / 4) + 4 (lane / 32) + i % 4 of the tile
  float* const o = a.wpart + (int64_t)blockIdx.y * 256 * a.hid + col0 + (lane & 31);
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int dim = 64 * wv + 32 * m + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        o[(int64_t)dim * a.hid + 32 * n] = acc[m][n][i];
      }
}

// Sums the ranges' shares of d W (four columns per thread) and, in the work-groups past
// them, the norm weights' shares, in a fixed order.
__global__ __launch_bounds__(256) void front_bwd_sum_kernel(FrontBwdArgs a, int wgroups) {
  if ((int)blockIdx.x >= wgroups) {
    // 16 threads per norm weight
    const int d = ((int)blockIdx.x - wgroups) * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15;
    float s = 0.f;
    for (int w = sub; w < a.nwg; w += 16) s += a.npart[(int64_t)w * 256 + d];
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) s += __shfl_xor(s, m, kWave);
    if (sub == 0) (d < kFbD ? a.dnq : a.dnk)[d & 127] = s;
    return;
  }
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (e >= (int64_t)256 * a.hid) return;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int r = 0; r < a.nrange; ++r) {
    const float4 x = *(const float4*)(a.wpart + (int64_t)r * 256 * a.hid + e);
    s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
  }
  const int64_t half = (int64_t)kFbD * a.hid;
  bf16x4 w;
  w[0] = (bf16)s.x; w[1] = (bf16)s.y; w[2] = (bf16)s.z; w[3] = (bf16)s.w;
  bf16* const o = e < half ? a.dwq : a.dwk;
  if (o) *(bf16x4*)(o + (e < half ? e : e - half)) = w;
}

// d hs tile of 128 rows x 128 hidden columns over the 256 dims, one side (128 dims) at a
// time: d p rows and W rows in LDS, W by transposing reads.  Wavefront (rw, cw) owns rows
// 64 rw .. and columns 64 cw ..  The tile leaves through LDS in whole 256-byte row pieces,
// with the hidden states' non-finite positions cleared.  Bound by reading hs and writing
// d hs.
__global__ __launch_bounds__(256, 2) void front_bwd_h_kernel(FrontBwdArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 sP[2][64 * 128];    // d p rows
  __shared__ __attribute__((aligned(16))) bf16 sW[2][64 * 128];    // W dims 64 s ..
  const int tid = threadIdx.x, lane = wave_lane(), wv = tid / kWave;
  const int hl = lane >> 5, n = lane & 31;
  const int rw = wv & 1, cw = wv >> 1;
  const int ncol = a.hid / kFbCols;
  const int col0 = (blockIdx.x % ncol) * kFbCols;
  const int64_t t0 = (int64_t)(blockIdx.x / ncol) * 128;
  floatx16 acc[2][2];                      // [column tile][row tile]
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[c][r][i] = 0.f;
  for (int side = 0; side < 2; ++side) {
    const bf16* w = side ? a.wk : a.wq;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      stage_rows(sP[s], wv, lane,
                 [&](int r) { return a.dproj + min(t0 + 64 * s + r, a.T - 1) * 256 + side * kFbD; });
      stage_rows(sW[s], wv, lane, [&](int r) { return w + (int64_t)(64 * s + r) * a.hid + col0; });
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      // k order of the transposing reads: dims 16 ks + 8 (e / 4) + 4 hl + e % 4
      bf16x8 fa[2], fp[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) fa[c] = tr_frag_k(sW[ks >> 2], 16 * (ks & 3), 2 * cw + c, lane);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const bf16* row = sP[rw] + (32 * r + n) * 128;
        const int sw = bw_swz(n & 15);
        const bf16x4 lo = *(const bf16x4*)(row + ((2 * ks) ^ sw) * 8 + 4 * hl);
        const bf16x4 hi = *(const bf16x4*)(row + ((2 * ks + 1) ^ sw) * 8 + 4 * hl);
#pragma unroll
        for (int e = 0; e < 4; ++e) { fp[r][e] = lo[e]; fp[r][e + 4] = hi[e]; }
      }
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r)
          acc[c][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[c], fp[r], acc[c][r], 0, 0, 0);
    }
  }
  __syncthreads();
  // rows 64 rw + 32 r + n, columns 64 cw + 32 c + 8 g + 4 hl .. + 3 into sP (64 rows each)
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (bf16)acc[c][r][4 * g + e];
        *(bf16x4*)(sP[rw] + (32 * r + n) * 128 + ((8 * cw + 4 * c + g) ^ (n & 15)) * 8 + 4 * hl) = v;
      }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int r = 16 * u + (tid >> 4), c = tid & 15;
    const int64_t t = t0 + r;
    if (t < a.T) {
      uint4 v = *(const uint4*)(sP[r >> 6] + (r & 63) * 128 + (c ^ (r & 15)) * 8);
      const uint4 h = *(const uint4*)(a.hs + t * a.hs_st + col0 + c * 8);
      // the mask of a word: halves that are finite
      auto keep = [](uint32_t x) {
        return (((x & 0x7f80u) == 0x7f80u) ? 0u : 0xffffu) |
               (((x & 0x7f800000u) == 0x7f800000u) ? 0u : 0xffff0000u);
      };
      v.x &= keep(h.x); v.y &= keep(h.y); v.z &= keep(h.z); v.w &= keep(h.w);
      *(uint4*)(a.dhs + t * a.hid + col0 + c * 8) = v;
    }
  }
}

struct FrontBwdLayout {
  int64_t dproj, npart, wpart, total;
  int nwg, nrange, range;
};
inline FrontBwdLayout front_bwd_layout(int64_t T, int hid) {
  FrontBwdLayout L;
  // 16 rows a wavefront at most until the grid holds 1,024 work-groups
  L.nwg = (int)std::min<int64_t>(std::max<int64_t>((T + 15) / 16, 1), 1024);
  // at most 32 ranges (their shares are written and read once), of at least 4 steps
  const int64_t steps = (T + kFbRows - 1) / kFbRows;
  const int64_t per = std::max<int64_t>(4, (steps + 31) / 32);
  L.range = (int)(per * kFbRows);
  L.nrange = (int)std::max<int64_t>(1, (steps + per - 1) / per);
  int64_t o = 0;
  L.dproj = o; o = align256(o + T * 256 * 2);
  L.npart = o; o = align256(o + (int64_t)L.nwg * 256 * 4);
  L.wpart = o; o = align256(o + (int64_t)L.nrange * 256 * hid * 4);
  L.total = o;
  return L;
}

}  // namespace dash

extern "C" int dash_router_front_backward_workspace_size(int64_t T, int hidden, int64_t* bytes) {
  using namespace dash;
  if (!bytes || T < 0 || hidden <= 0) return kErrInvalid;
  *bytes = front_bwd_layout(T, hidden).total;
  return kOk;
}

extern "C" int dash_router_front_backward(
    const void* proj, const float* d_iq, const float* d_ik, const float* wq_norm,
    const float* wk_norm, float eps, const void* cos, const void* sin, int cs_bf16, int64_t cs_sb,
    int64_t cs_st, int B, int S, int hidden, const void* hs, int64_t hs_st, const void* w_q,
    const void* w_k, void* dw_q, void* dw_k, float* dwq_norm, float* dwk_norm, void* dhs,
    void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace dash;
  if (!proj || !d_iq || !d_ik || !wq_norm || !wk_norm || !hs || !w_q || !w_k || !dwq_norm ||
      !dwk_norm || B < 0 || S < 0 || hidden <= 0 || (cos == nullptr) != (sin == nullptr))
    return kErrInvalid;
  if (hidden % kFbCols != 0 || hs_st % 8 != 0) return kErrUnsupported;
  const void* p16[] = {hs, w_q, w_k, proj, d_iq, d_ik};
  for (const void* p : p16)
    if ((uintptr_t)p % 16 != 0) return kErrUnsupported;
  if ((uintptr_t)wq_norm % 8 != 0 || (uintptr_t)wk_norm % 8 != 0 || (uintptr_t)dhs % 16 != 0 ||
      (uintptr_t)dw_q % 8 != 0 || (uintptr_t)dw_k % 8 != 0)
    return kErrUnsupported;
  const int cs = cs_bf16 ? 2 : 4;
  if (cos && ((uintptr_t)cos % (2 * cs) != 0 || (uintptr_t)sin % (2 * cs) != 0 || cs_sb % 2 != 0 ||
              cs_st % 2 != 0))
    return kErrUnsupported;
  const int64_t T = (int64_t)B * S;
  if (T == 0) return kErrUnsupported;
  const FrontBwdLayout L = front_bwd_layout(T, hidden);
  if (!workspace || workspace_bytes < L.total || (uintptr_t)workspace % 256 != 0)
    return kErrWorkspace;
  const int64_t htiles = (T + 127) / 128 * (hidden / kFbCols);
  if (htiles > INT32_MAX) return kErrUnsupported;
  char* w = (char*)workspace;
  FrontBwdArgs a = {};
  a.proj = (const bf16*)proj; a.gq = d_iq; a.gk = d_ik; a.nq = wq_norm; a.nk = wk_norm;
  a.cos = cos; a.sin = sin; a.cs_bf16 = cs_bf16; a.cs_sb = cs_sb; a.cs_st = cs_st;
  a.T = T; a.S = S; a.hid = hidden; a.eps = eps;
  a.hs = (const bf16*)hs; a.hs_st = hs_st; a.wq = (const bf16*)w_q; a.wk = (const bf16*)w_k;
  a.dproj = (bf16*)(w + L.dproj);
  a.npart = (float*)(w + L.npart); a.nwg = L.nwg;
  a.wpart = (float*)(w + L.wpart); a.nrange = L.nrange; a.range = L.range;
  a.dwq = (bf16*)dw_q; a.dwk = (bf16*)dw_k; a.dnq = dwq_norm; a.dnk = dwk_norm;
  a.dhs = (bf16*)dhs;
  hipStream_t st = (hipStream_t)stream;
  const bool want_w = dw_q || dw_k;
  hipLaunchKernelGGL(front_bwd_rows_kernel, dim3(L.nwg), dim3(256), 0, st, a);
  if (want_w)
    hipLaunchKernelGGL(front_bwd_w_kernel, dim3(hidden / kFbCols, L.nrange), dim3(256), 0, st, a);
  const int wgroups = want_w ? (int)(((int64_t)64 * hidden + 255) / 256) : 0;
  hipLaunchKernelGGL(front_bwd_sum_kernel, dim3(wgroups + 16), dim3(256), 0, st, a, wgroups);
  if (dhs) hipLaunchKernelGGL(front_bwd_h_kernel, dim3((unsigned)htiles), dim3(256), 0, st, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? kOk : (int)e;
}
